// Photometric loss of the training loop and its gradient w.r.t. the rendered ray colours:
//   L = (1 - lambda) * mean|x - y| + lambda * (1 - mean SSIM(x, y))
// with SSIM over an 11x11 Gaussian window (sigma 1.5), zero padding, C1 = 0.01^2, C2 = 0.03^2
// (reference utils/loss_utils.py:17-64, used at scripts/train.py:110-112 with lambda = 0.2), and
// the supersampling reduction in front of it (utils/general_utils.py:489-502): the image pixel
// (x, y) is the mean of the fx*fy rays (x*fx + i, y*fy + j) of a row-major (H*fy) x (W*fx) grid.
//
// SSIM gradient in closed form.  Per pixel q, with mu1 = w*x, mu2 = w*y, E11 = w*x^2,
// E22 = w*y^2, E12 = w*xy (w the window, * the zero-padded "same" correlation):
//   A1 = 2 mu1 mu2 + C1, A2 = 2 (E12 - mu1 mu2) + C2, B1 = mu1^2 + mu2^2 + C1,
//   B2 = (E11 - mu1^2) + (E22 - mu2^2) + C2, s = A1 A2 / (B1 B2)
//   Gm  = ds/dmu1 = (2 mu2 (A2 - A1) - 2 mu1 s (B2 - B1)) / (B1 B2)
//   G11 = ds/dE11 = -s / B2,   G12 = ds/dE12 = 2 A1 / (B1 B2)
// and, the window being symmetric, d(mean s)/dx(p) = (w*Gm + 2 x w*G11 + y w*G12)(p) / N.
// Every convolution is separable (the window is the outer product of the 1-D Gaussian).  Two launches,
// each over 32x16-pixel tiles with all three channels: k_ssim holds a tile's images with their
// 5-pixel rim in LDS, runs the horizontal and the vertical 11-tap pass there and writes the three
// gradient maps; k_grad does the same with those.  What bounds them is HBM traffic, 11 planes moved
// (2 images, 3 maps out; 3 maps, 2 images in, 1 out) instead of the 36 of one launch per pass:
// 242 -> 91 us for the loss and its gradient at 1237x822 (k_ssim 46, k_grad 38).

#include <hip/hip_runtime.h>

#include "rg_internal.h"

namespace rg {
namespace {

constexpr int kLB = 256;
constexpr int kHalf = 5;
constexpr int kTX = 32, kTY = 16;                             // a tile
constexpr int kPX = kTX + 2 * kHalf, kPY = kTY + 2 * kHalf;  // with its rim
constexpr int kRun = 4;                                       // outputs of one thread along x

struct Win {
    float w[2 * kHalf + 1];
};

// The image's pixel (x, y): the mean of its fx*fy rays of the row-major (H*fy) x (W*fx) grid.
__device__ __forceinline__ void ray_mean(const float* __restrict__ rays, int W, int x, int y, int fx, int fy, float* v) {
    const int64_t RW = (int64_t)W * fx;
    float s[3] = {0.0f, 0.0f, 0.0f};
    for (int j = 0; j < fy; ++j)
        for (int i = 0; i < fx; ++i) {
            const int64_t r = ((int64_t)y * fy + j) * RW + (int64_t)x * fx + i;
            s[0] += rays[3 * r];
            s[1] += rays[3 * r + 1];
            s[2] += rays[3 * r + 2];
        }
    const float inv = 1.0f / (float)(fx * fy);
    for (int c = 0; c < 3; ++c) v[c] = s[c] * inv;
}

// Horizontal pass over the tile's rows with their rim: `K` moments of each pixel (vals), kRun outputs a
// thread so that a run's pixels are read once.  A tap outside the image adds zero.
template <int K, typename F>
__device__ __forceinline__ void pass_x(const Win& win, F&& vals, float (*h)[kPY][kTX + 1]) {
    for (int i = threadIdx.x; i < kPY * (kTX / kRun); i += kLB) {
        const int y = i / (kTX / kRun), x0 = (i % (kTX / kRun)) * kRun;
        float acc[K][kRun];
#pragma unroll
        for (int k = 0; k < K; ++k)
#pragma unroll
            for (int o = 0; o < kRun; ++o) acc[k][o] = 0.0f;
#pragma unroll
        for (int t = 0; t < kRun + 2 * kHalf; ++t) {
            float v[K];
            vals(y, x0 + t, v);
#pragma unroll
            for (int o = 0; o < kRun; ++o) {
                if (t - o < 0 || t - o > 2 * kHalf) continue;
                const float wk = win.w[t - o];
#pragma unroll
                for (int k = 0; k < K; ++k) acc[k][o] += wk * v[k];
            }
        }
#pragma unroll
        for (int k = 0; k < K; ++k)
#pragma unroll
            for (int o = 0; o < kRun; ++o) h[k][y][x0 + o] = acc[k][o];
    }
}

// Vertical pass at tile pixel (x, y): its K sums.
template <int K>
__device__ __forceinline__ void pass_y(const Win& win, float (*h)[kPY][kTX + 1], int x, int y, float* acc) {
#pragma unroll
    for (int k = 0; k < K; ++k) acc[k] = 0.0f;
#pragma unroll
    for (int t = 0; t <= 2 * kHalf; ++t)
#pragma unroll
        for (int k = 0; k < K; ++k) acc[k] += win.w[t] * h[k][y + t][x];
}

// SSIM and its three gradient maps, and the tile's sums of SSIM and |x - y| (double, so the mean does
// not depend on the tiles' rounding).
__global__ void __launch_bounds__(kLB) k_ssim(const float* __restrict__ rays, const float* __restrict__ target, int W, int H,
                                              int fx, int fy, Win win, float* __restrict__ gmap,
                                              double* __restrict__ partial) {
    __shared__ float X[3][kPY][kPX], Y[3][kPY][kPX];
    __shared__ float h[5][kPY][kTX + 1];
    __shared__ double red[2][kLB / 64];
    const int64_t HW = (int64_t)W * H, S = 3 * HW;
    const int bx = blockIdx.x * kTX, by = blockIdx.y * kTY;
    for (int i = threadIdx.x; i < kPY * kPX; i += kLB) {
        const int py = i / kPX, px = i % kPX, x = bx + px - kHalf, y = by + py - kHalf;
        float v[3] = {0.0f, 0.0f, 0.0f}, t[3] = {0.0f, 0.0f, 0.0f};
        if (x >= 0 && x < W && y >= 0 && y < H) {
            ray_mean(rays, W, x, y, fx, fy, v);
            for (int c = 0; c < 3; ++c) t[c] = target[c * HW + (int64_t)y * W + x];
        }
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            X[c][py][px] = v[c];
            Y[c][py][px] = t[c];
        }
    }
    double s_sum = 0.0, l1_sum = 0.0;
    for (int c = 0; c < 3; ++c) {
        __syncthreads();
        pass_x<5>(win, [&](int y, int x, float* v) {
            const float a = X[c][y][x], b = Y[c][y][x];
            v[0] = a;
            v[1] = b;
            v[2] = a * a;
            v[3] = b * b;
            v[4] = a * b;
        }, h);
        __syncthreads();
        for (int i = threadIdx.x; i < kTX * kTY; i += kLB) {
            const int tx = i % kTX, ty = i / kTX, x = bx + tx, y = by + ty;
            if (x >= W || y >= H) continue;
            float m[5];
            pass_y<5>(win, h, tx, ty, m);
            const float mu1 = m[0], mu2 = m[1], e11 = m[2], e22 = m[3], e12 = m[4];
            const float C1 = 0.0001f, C2 = 0.0009f;
            const float mu12 = mu1 * mu2;
            const float A1 = 2.0f * mu12 + C1;
            const float A2 = 2.0f * (e12 - mu12) + C2;
            const float B1 = mu1 * mu1 + mu2 * mu2 + C1;
            const float B2 = (e11 - mu1 * mu1) + (e22 - mu2 * mu2) + C2;
            const float den = B1 * B2;
            const float s = (A1 * A2) / den;
            const int64_t o = c * HW + (int64_t)y * W + x;
            gmap[o] = (2.0f * mu2 * (A2 - A1) - 2.0f * mu1 * s * (B2 - B1)) / den;
            gmap[S + o] = -s / B2;
            gmap[2 * S + o] = 2.0f * A1 / den;
            s_sum += (double)s;
            l1_sum += (double)fabsf(X[c][ty + kHalf][tx + kHalf] - Y[c][ty + kHalf][tx + kHalf]);
        }
    }
    for (int o = 32; o > 0; o >>= 1) {
        s_sum += __shfl_xor(s_sum, o, 64);
        l1_sum += __shfl_xor(l1_sum, o, 64);
    }
    if ((threadIdx.x & 63) == 0) {
        red[0][threadIdx.x >> 6] = s_sum;
        red[1][threadIdx.x >> 6] = l1_sum;
    }
    __syncthreads();
    if (threadIdx.x < 2) {
        double v = 0.0;
        for (int k = 0; k < kLB / 64; ++k) v += red[threadIdx.x][k];
        partial[2 * ((int64_t)blockIdx.y * gridDim.x + blockIdx.x) + threadIdx.x] = v;
    }
}

// The gradient maps through the window, gradient assembly and scatter to the supersampled rays.
__global__ void __launch_bounds__(kLB) k_grad(const float* __restrict__ gmap, const float* __restrict__ rays,
                                              const float* __restrict__ target, int W, int H, int fx, int fy, Win win,
                                              float lambda, float* __restrict__ dl_rays) {
    __shared__ float M[3][kPY][kPX];
    __shared__ float h[3][kPY][kTX + 1];
    const int64_t HW = (int64_t)W * H, S = 3 * HW;
    const int bx = blockIdx.x * kTX, by = blockIdx.y * kTY;
    constexpr int N = kTX * kTY / kLB;  // pixels of a thread
    float g[N][3], xv[N][3];
#pragma unroll
    for (int k = 0; k < N; ++k) {
        const int i = threadIdx.x + k * kLB, x = bx + i % kTX, y = by + i / kTX;
        if (x < W && y < H) ray_mean(rays, W, x, y, fx, fy, xv[k]);
    }
    const float invN = 1.0f / (float)S;
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        __syncthreads();
        for (int i = threadIdx.x; i < kPY * kPX; i += kLB) {
            const int py = i / kPX, px = i % kPX, x = bx + px - kHalf, y = by + py - kHalf;
            const bool in = x >= 0 && x < W && y >= 0 && y < H;
            const int64_t o = c * HW + (int64_t)y * W + x;
            for (int m = 0; m < 3; ++m) M[m][py][px] = in ? gmap[m * S + o] : 0.0f;
        }
        __syncthreads();
        pass_x<3>(win, [&](int y, int x, float* v) {
            for (int m = 0; m < 3; ++m) v[m] = M[m][y][x];
        }, h);
        __syncthreads();
#pragma unroll
        for (int k = 0; k < N; ++k) {
            const int i = threadIdx.x + k * kLB, tx = i % kTX, ty = i / kTX, x = bx + tx, y = by + ty;
            if (x >= W || y >= H) continue;
            float m[3];
            pass_y<3>(win, h, tx, ty, m);
            const float yv = target[c * HW + (int64_t)y * W + x];
            const float ds = (m[0] + 2.0f * xv[k][c] * m[1] + yv * m[2]) * invN;
            const float e = xv[k][c] - yv;
            const float dl1 = (e > 0.0f ? invN : (e < 0.0f ? -invN : 0.0f));
            g[k][c] = ((1.0f - lambda) * dl1 - lambda * ds) / (float)(fx * fy);
        }
    }
    const int64_t RW = (int64_t)W * fx;
#pragma unroll
    for (int k = 0; k < N; ++k) {
        const int i = threadIdx.x + k * kLB, x = bx + i % kTX, y = by + i / kTX;
        if (x >= W || y >= H) continue;
        for (int j = 0; j < fy; ++j)
            for (int q = 0; q < fx; ++q) {
                const int64_t r = ((int64_t)y * fy + j) * RW + (int64_t)x * fx + q;
                for (int c = 0; c < 3; ++c) dl_rays[3 * r + c] = g[k][c];
            }
    }
}

__global__ void k_loss_final(const double* __restrict__ partial, int nb, int64_t N, float lambda,
                             float* __restrict__ loss, float* __restrict__ parts) {
    __shared__ double red[2][kLB];
    double s = 0.0, l = 0.0;
    for (int i = threadIdx.x; i < nb; i += kLB) {
        s += partial[2 * i];
        l += partial[2 * i + 1];
    }
    red[0][threadIdx.x] = s;
    red[1][threadIdx.x] = l;
    __syncthreads();
    for (int off = kLB / 2; off > 0; off >>= 1) {
        if ((int)threadIdx.x < off) {
            red[0][threadIdx.x] += red[0][threadIdx.x + off];
            red[1][threadIdx.x] += red[1][threadIdx.x + off];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        const double ssim = red[0][0] / (double)N, l1 = red[1][0] / (double)N;
        loss[0] = (float)((1.0 - lambda) * l1 + lambda * (1.0 - ssim));
        if (parts) {
            parts[0] = (float)l1;
            parts[1] = (float)ssim;
        }
    }
}

}  // namespace

int64_t loss_workspace_bytes(int W, int H) {
    const int64_t tiles = (int64_t)((W + kTX - 1) / kTX) * ((H + kTY - 1) / kTY);
    // gradient maps (3), tile partials
    return (int64_t)sizeof(float) * 9 * (int64_t)W * H + (int64_t)sizeof(double) * 2 * tiles + 256;
}

hipError_t launch_loss_l1_ssim(const float* rays, const float* target, int W, int H, int fx, int fy,
                               const float* window11, float lambda, float* loss, float* parts, float* dl_rays,
                               void* ws, hipStream_t s) {
    const int64_t S = 3 * (int64_t)W * H;
    Win win;
    for (int k = 0; k < 2 * kHalf + 1; ++k) win.w[k] = window11[k];
    float* gm = static_cast<float*>(ws);
    uintptr_t pa = reinterpret_cast<uintptr_t>(gm + 3 * S);
    pa = (pa + 255) & ~(uintptr_t)255;
    double* partial = reinterpret_cast<double*>(pa);
    const dim3 tiles((W + kTX - 1) / kTX, (H + kTY - 1) / kTY);
    hipLaunchKernelGGL(k_ssim, tiles, dim3(kLB), 0, s, rays, target, W, H, fx, fy, win, gm, partial);
    hipLaunchKernelGGL(k_loss_final, dim3(1), dim3(kLB), 0, s, partial, (int)(tiles.x * tiles.y), S, lambda, loss, parts);
    if (dl_rays)
        hipLaunchKernelGGL(k_grad, tiles, dim3(kLB), 0, s, gm, rays, target, W, H, fx, fy, win, lambda, dl_rays);
    return hipGetLastError();
}

}  // namespace rg
