// Device code shared by the ray kernels (the per-ray slab stepper in trace.hip and the tile kernels
// in tile.hip): sampling and compositing of one slab, the backward's per-sample coefficients and
// gradient moments, the wave-merged gradient scatter, work items, records and work queues.
#pragma once

#include <hip/hip_runtime.h>

#include "rg_device.h"
#include "rg_internal.h"

namespace rg {

constexpr int kGradVals = 14;

enum CounterIdx { C_K = 0, C_P = 1, C_OVF = 2, C_FALLBACK = 3, C_GATHER = 4, C_LOSS = 6, C_REC_WORDS = 8,
                  C_REC_FULL = 9, C_DROP = 10, C_BAD = 11, C_LOSS64 = 14 };

struct RayOut {
    float C[3];
    float depth;
    float T;
};

// Rays whose view or pixel index is out of range (skipped), and gradient records or replayed hits
// skipped by a bounds check (an internal error: every parity test asserts none), go straight to
// their device counters with an atomic on those rare paths, so they cost no registers.
struct Counters {
    unsigned int K = 0, P = 0, ovf = 0, fallback = 0, gathers = 0, rec_words = 0, rec_full = 0;
};

__device__ __forceinline__ void count_drop(unsigned long long* drops) { atomicAdd(drops, 1ull); }

// FP32 gradient add (device scope, relaxed: the result is read by a later kernel).
__device__ __forceinline__ void gadd(float* p, float v) {
    __hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Address of gradient value k (0..13) of a slot: 0-2 d mu, 3 d sigma, 4-6 d s, 7-10 d q in the
// slot's accumulator record (offsets 0-6, 8-11), 11-13 the view's colour gradient.
__device__ __forceinline__ float* grad_addr(const DevGrad& gr, int n, int slot, int view, int k) {
    if (k < 11) return gr.acc + (size_t)kAccStride * slot + (k < 7 ? k : k + 1);
    return reinterpret_cast<float*>(gr.drgb + (size_t)view * n + slot) + (k - 11);
}

__device__ __forceinline__ void load_rec(const float4* __restrict__ geo, int s, float4& g0, float4& g1, float4& g2,
                                         float4& g3) {
    g0 = geo[4 * s];
    g1 = geo[4 * s + 1];
    g2 = geo[4 * s + 2];
    g3 = geo[4 * s + 3];
}

// The Gaussian's weight along the ray, exp(-(A + Cq tau^2)), as one native exp2 with -log2(e)
// folded into the per-hit terms; every pass (forward, backward buffers, gradients) evaluates it
// the same way, so they agree bit for bit.  Weights that small enough to flush to zero are far
// below the sample threshold.
struct WExp {
    float a, c;  // -A log2(e), -Cq log2(e)
};

__device__ __forceinline__ WExp wexp(const Isect& I) {
    constexpr float kLog2e = 1.4426950408889634f;
    return WExp{-I.A * kLog2e, -I.Cq * kLog2e};
}

__device__ __forceinline__ float weight(const WExp& k, float tau) {
    return __builtin_amdgcn_exp2f(fmaf(k.c, tau * tau, k.a));  // explicit fma: same rounding in every pass
}

// Accumulate one hit's contribution to the slab's sample buffers (computeBufferForward,
// forward/gaussians_aabb.cu:437-498).
template <int SPB, bool RNG>
__device__ __forceinline__ void accum_hit(const Isect& I, float sigma, float4 col, float tb, unsigned int seed,
                                          const DevParams& p, float* sig, float* cr, float* cg, float* cb) {
    unsigned int st = seed;
    const WExp k = wexp(I);
#pragma unroll
    for (int i = 0; i < SPB; ++i) {
        if (SPB > 8 && i >= p.spb) break;
        const float t = sample_t(tb, i, p.dt, RNG ? p.rnd_sample : 0, st);
        const float sw = sigma * weight(k, t - I.tc);
        // a sample at or below the threshold adds exact zeros (no branch per sample)
        const float m = sw > p.sigma_thr ? sw : 0.0f;
        sig[i] += m;
        cr[i] += m * col.x;
        cg[i] += m * col.y;
        cb[i] += m * col.z;
    }
}

// Opacity of one sample, 1 - exp(-sigma dt) (forward/gaussians_aabb.cu:509), with the native
// exp2 (1 ulp) and the native reciprocal for the colour below: the forward's compositing and the
// backward's coefficients use the same two, so the backward retraces the forward's transmittance.
__device__ __forceinline__ float sample_alpha(float s, float dt) {
    constexpr float kNegLog2e = -1.4426950408889634f;
    return 1.0f - __builtin_amdgcn_exp2f(s * (dt * kNegLog2e));
}

// colorBlending (forward/gaussians_aabb.cu:500-519) + depth (cuda_gui/gaussians_aabb.cu:415) where it is
// asked for.
template <int SPB, bool RNG>
__device__ __forceinline__ void composite(const float* sig, const float* cr, const float* cg, const float* cb, float tb,
                                          unsigned int seed, const DevParams& p, bool depth, RayOut& o) {
    unsigned int st = seed;
    float ta[SPB];
#pragma unroll
    for (int i = 0; i < SPB; ++i) {
        if (SPB > 8 && i >= p.spb) break;
        const float s = sig[i];
        const float alpha = sample_alpha(s, p.dt);
        // colour = sums / sigma: one reciprocal per sample (a sample without hits has zero sums)
        const float inv = __builtin_amdgcn_rcpf(fmaxf(s, 0x1p-126f));
        const float r = cr[i] * inv, g = cg[i] * inv, b = cb[i] * inv;
        ta[i] = o.T * alpha;
        o.C[0] += ta[i] * r;
        o.C[1] += ta[i] * g;
        o.C[2] += ta[i] * b;
        o.T *= 1.0f - alpha;
    }
    if (!depth) return;
#pragma unroll
    for (int i = 0; i < SPB; ++i) {
        if (SPB > 8 && i >= p.spb) break;
        o.depth += ta[i] * sample_t(tb, i, p.dt, RNG ? p.rnd_sample : 0, st);
    }
}

// Thresholded densities of one hit at the slab's samples (accum_hit's m).
template <int SPB, bool RNG>
__device__ __forceinline__ void sample_densities(const Isect& I, float sigma, float tb, unsigned int seed,
                                                 const DevParams& p, float* m) {
    unsigned int st = seed;
    const WExp k = wexp(I);
#pragma unroll
    for (int i = 0; i < SPB; ++i) {
        if (SPB > 8 && i >= p.spb) break;
        const float t = sample_t(tb, i, p.dt, RNG ? p.rnd_sample : 0, st);
        const float sw = sigma * weight(k, t - I.tc);
        m[i] = sw > p.sigma_thr ? sw : 0.0f;
    }
}

// Adds a hit's densities and their colour's projection F = dLdC . c on dL/dC to the slab's sums: of the
// colour the backward needs no more.
template <int SPB>
__device__ __forceinline__ void accum_densities(const float* m, float F, const DevParams& p, float* sig, float* ep) {
#pragma unroll
    for (int i = 0; i < SPB; ++i) {
        if (SPB > 8 && i >= p.spb) break;
        sig[i] += m[i];
        ep[i] += m[i] * F;
    }
}

__device__ __forceinline__ float project_color(const float* dL, float4 c) {
    return dL[0] * c.x + dL[1] * c.y + dL[2] * c.z;
}

// Per-sample backward coefficients of one slab, from its sums: overwrites (sig, ep) with
// (G_i, Bq_i) and advances T and the projected colour remainder Dr = dLdC . Crem past the
// slab (Crem_i: the ray's colour not yet composited before sample i; only its projection on
// dLdC enters the coefficients, so one scalar is carried instead of three).
//   A_i  = dt * dLdC . (T_i c^_i - Crem_i) = dt * (T_i E_i - Dr_i)   (dcolor_dsigma_aux, backward :706)
//   Bq_i = T_i alpha_i / sigma_i                (0 when sigma_i == 0)
//   E_i  = dLdC . c^_i = (dLdC . sums_i) / sigma_i
//   G_i  = A_i - Bq_i E_i, so that a hit of colour c weighs sample i by phi_i = G_i + Bq_i (dLdC . c)
template <int SPB>
__device__ __forceinline__ void slab_coeffs(float* sig, float* ep, const DevParams& p, float& T, float& Dr) {
#pragma unroll
    for (int i = 0; i < SPB; ++i) {
        if (SPB > 8 && i >= p.spb) break;
        const float s = sig[i];
        const float alpha = sample_alpha(s, p.dt);
        // the forward's colour is sums / sigma (composite); only its projection E on dLdC enters
        const float inv = s > 0.0f ? __builtin_amdgcn_rcpf(s) : 0.0f;
        const float E = ep[i] * inv;
        const float A = p.dt * (T * E - Dr);
        const float ta = T * alpha;
        const float Bq = ta * inv;
        Dr -= ta * E;
        T *= 1.0f - alpha;
        sig[i] = A - Bq * E;
        ep[i] = Bq;
    }
}

// D' = M' d, as the predicate forms it (exact FP32).
__device__ __forceinline__ void ray_in_ellipsoid(const float4 g1, const float4 g2, const float4 g3, const Ray& r, float* D) {
#pragma clang fp contract(off)
    D[0] = (g1.x * r.dx + g1.y * r.dy) + g1.z * r.dz;
    D[1] = (g2.x * r.dx + g2.y * r.dy) + g2.z * r.dz;
    D[2] = (g3.x * r.dx + g3.y * r.dy) + g3.z * r.dz;
}

// Gradient moments of one (slab, hit) for one ray.  Over the slab's samples the hit contributes
// four sums of its densities m = sigma w (S0 = sum m phi, T1 = sum m phi tau, T2 = sum m phi tau^2,
// Sc = sum m Bq; tau = t - t_c, phi = G + Bq F with F = dLdC . colour; G, Bq from slab_coeffs).
// Every gradient of the Gaussian is linear in the ray-dependent moments
//   Gy'   = P S0 + D T1                                     (3)
//   Y'    = P P^T S0 + (P D^T + D P^T) T1 + D D^T T2         (6, symmetric)
//   S0 / sigma, and dL_c Sc                                 (1 + 3)
// (P, D the ray's ellipsoid-space offset at t_c and direction, the ones that the densities come from:
// another evaluation of P, as good by itself, costs the gradients 1.2 to 1.5 times their error)
// with coefficients that depend on the Gaussian alone, so the wave sums these 13 moments over its
// lanes and expand the sum once per Gaussian (expand_grad) instead of once per lane.
constexpr int kMoments = 13;

// The moments of a ray from its four sums.
__device__ __forceinline__ void ray_moments(const float* P, const float* D, float sigma, float S0, float T1, float T2,
                                            float Sc, const float* dL, float* v) {
    float W[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        v[a] = P[a] * S0 + D[a] * T1;
        W[a] = P[a] * T1 + D[a] * T2;
    }
    // with U = Gy' and W = P T1 + D T2: Y'_ab = P_a U_b + D_a W_b; (0,0) (1,1) (2,2) (0,1) (0,2) (1,2)
    const int ya[6] = {0, 1, 2, 0, 0, 1}, yb[6] = {0, 1, 2, 1, 2, 2};
#pragma unroll
    for (int k = 0; k < 6; ++k) v[3 + k] = P[ya[k]] * v[yb[k]] + D[ya[k]] * W[yb[k]];
    v[9] = S0 * __builtin_amdgcn_rcpf(sigma);
    v[10] = dL[0] * Sc;
    v[11] = dL[1] * Sc;
    v[12] = dL[2] * Sc;
}

template <int SPB, bool RNG>
__device__ __forceinline__ void grad_moments(const float* P, const float* D, float sigma, const float* m, float tc, float F,
                                             float tb, unsigned int seed, const DevParams& p, const float* Gq,
                                             const float* Bq, const float* dL, float* v) {
    float S0 = 0.0f, T1 = 0.0f, T2 = 0.0f, Sc = 0.0f;
    unsigned int st = seed;
#pragma unroll
    for (int i = 0; i < SPB; ++i) {
        if (SPB > 8 && i >= p.spb) break;
        const float tau = sample_t(tb, i, p.dt, RNG ? p.rnd_sample : 0, st) - tc;
        const float wp = m[i] * (Gq[i] + Bq[i] * F);
        S0 += wp;
        T1 += wp * tau;
        T2 += wp * (tau * tau);
        Sc += m[i] * Bq[i];
    }
    ray_moments(P, D, sigma, S0, T1, T2, Sc, dL, v);
}

// The 14 gradient values of one Gaussian from its summed moments m (grad_moments):
// v = (d mu[3], d sigma, d s[3], d q[4] (w,x,y,z), d rgb[3]), with the Gaussian's record rows of
// M' (g1..g3), scales s and delta (brec[0]), quaternion (brec[1]); y = d (P + tau D) in the
// unenlarged ellipsoid frame, so Gy = d Gy', Y = d^2 Y'.
__device__ __forceinline__ void expand_grad(const float* mo, float4 g1, float4 g2, float4 g3, float4 b0, float4 q,
                                            float* v) {
    const float d = b0.w, d2 = d * d;
    const float Gy[3] = {d * mo[0], d * mo[1], d * mo[2]};
    const float Y[3][3] = {{d2 * mo[3], d2 * mo[6], d2 * mo[7]},
                           {d2 * mo[6], d2 * mo[4], d2 * mo[8]},
                           {d2 * mo[7], d2 * mo[8], d2 * mo[5]}};
    const float m[3][3] = {{g1.x, g1.y, g1.z}, {g2.x, g2.y, g2.z}, {g3.x, g3.y, g3.z}};  // rows of M'
    const float s[3] = {b0.x, b0.y, b0.z};
    float dcol[3][3];
#pragma unroll
    for (int c = 0; c < 3; ++c) v[c] = d * (m[0][c] * Gy[0] + m[1][c] * Gy[1] + m[2][c] * Gy[2]);
    // reciprocal scales: native reciprocal (1 ulp), well inside the gradients' tolerance
    const float is[3] = {__builtin_amdgcn_rcpf(s[0]), __builtin_amdgcn_rcpf(s[1]), __builtin_amdgcn_rcpf(s[2])};
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const float f = -d * is[k];
#pragma unroll
        for (int c = 0; c < 3; ++c)
            dcol[k][c] = f * (s[0] * s[0] * Y[0][k] * m[0][c] + s[1] * s[1] * Y[1][k] * m[1][c] +
                              s[2] * s[2] * Y[2][k] * m[2][c]);
    }
    // quaternion chain (backward/gaussians_aabb.cu:747-763), q = (r, i, j, k) = (w, x, y, z)
    const float r = q.x, qi = q.y, qj = q.z, qk = q.w;
    const float* c0 = dcol[0];
    const float* c1 = dcol[1];
    const float* c2 = dcol[2];
    v[3] = mo[9];
    v[4] = Y[0][0] * is[0];
    v[5] = Y[1][1] * is[1];
    v[6] = Y[2][2] * is[2];
    v[7] = 2.0f * (qk * c0[1] - qj * c0[2] - qk * c1[0] + qi * c1[2] + qj * c2[0] - qi * c2[1]);
    v[8] = 2.0f * (qj * c0[1] + qk * c0[2] + qj * c1[0] + r * c1[2] + qk * c2[0] - r * c2[1]) -
           4.0f * qi * (c1[1] + c2[2]);
    v[9] = 2.0f * (qi * c0[1] - r * c0[2] + qi * c1[0] + qk * c1[2] + r * c2[0] + qk * c2[1]) -
           4.0f * qj * (c0[0] + c2[2]);
    v[10] = 2.0f * (r * c0[1] + qi * c0[2] - r * c1[0] + qj * c1[2] + qi * c2[0] + qj * c2[1]) -
            4.0f * qk * (c0[0] + c1[1]);
    v[11] = mo[10];
    v[12] = mo[11];
    v[13] = mo[12];
}

// Staging area of the wave-merged gradient sums in LDS.  Global atomics are issued in bursts of
// kStage records: every vector memory operation of a wave completes in order, so an atomic
// issued between two loads makes the wave wait for its round trip at the next load; a burst
// pays that wait once per kStage records instead of once per record.
constexpr int kStage = 16;
struct GradStage {
    float val[kStage][16];
    int slot[kStage];
    int view[kStage];
};

// The records staged: their number and, in lane e, the key (view * n + slot) of record e, -1 past the last.
struct Staged {
    int n = 0;
    int key = -1;
};

// Issues the first cnt staged records: four records per instruction (lanes 16e..16e+13).  The
// records were written by other lanes: the workgroup is one wavefront, and the barriers order
// the LDS writes before these reads and these reads before the next records' writes.
__device__ __forceinline__ void stage_flush(GradStage& G, Staged& st, const DevScene& sc, const DevGrad& gr,
                                            int lane, unsigned long long* drops) {
    const int cnt = st.n;
    __syncthreads();
    // lane e decodes record e's key and expands its summed moments into its 14 gradient values,
    // in place
    if (lane < cnt) {
        const int key = st.key;
        const int view = key / sc.n;
        const int slot = key - view * sc.n;
        G.slot[lane] = slot;
        G.view[lane] = view;
        if ((unsigned)slot < (unsigned)sc.n) {
            float mo[kMoments], v[kGradVals];
#pragma unroll
            for (int k = 0; k < kMoments; ++k) mo[k] = G.val[lane][k];
            const float4 g1 = sc.geo[4 * slot + 1], g2 = sc.geo[4 * slot + 2], g3 = sc.geo[4 * slot + 3];
            expand_grad(mo, g1, g2, g3, sc.brec[2 * slot], sc.brec[2 * slot + 1], v);
#pragma unroll
            for (int k = 0; k < kGradVals; ++k) G.val[lane][k] = v[k];
        }
    }
    __syncthreads();
    const int j = lane & 15;
    for (int e0 = 0; e0 < cnt; e0 += 4) {
        const int e = e0 + (lane >> 4);
        if (e < cnt && j < kGradVals) {
            const int slot = G.slot[e], view = G.view[e];
            if ((unsigned)slot < (unsigned)sc.n && (unsigned)view < (unsigned)gr.num_views)
                gadd(grad_addr(gr, sc.n, slot, view, j), G.val[e][j]);
            else if (j == 0)
                count_drop(drops);  // never expected: counted so that tests see it
        }
    }
    __syncthreads();
    st = Staged();
}

// Wave-wide sum of the 13 gradient moments of one Gaussian (all lanes hold a contribution, zero
// for lanes without one), added to the staged record of its key view * n + slot or appended as one
// (decoded, expanded and flushed when the area is full): a Gaussian that the wavefront meets in several
// slabs in turn costs one expansion and one set of atomics, and its sum fewer roundings.  Against a
// record per event: backward 138.7 -> 134.8 ms at 1M Gaussians, the gradients' error against sums in 64 bits
// 2.9e-6 -> 1.6e-6.  The sums are formed by a
// reduce-scatter: the lanes below 32 keep values 0..7 and add the upper lanes' copies of them,
// the upper lanes values 8..15 (v_permlane32_swap); then the same over row pairs
// (v_permlane16_swap), over lane bit 3 (DPP row rotation by 8) and bit 2 (DPP half-row mirror:
// the partner differs in bits 2..0, and the quad sum below covers bits 1..0); after that lane l
// holds value bitrev4(l >> 2) summed over its quad's partners, and two DPP steps complete the sum
// over the quad.  No LDS traffic.  Called by all 64 lanes together.
__device__ __forceinline__ void grad_scatter_wave(const float* v, int key, const DevScene& sc,
                                                  const DevGrad& gr, int lane, GradStage& G, Staged& st,
                                                  unsigned long long* drops) {
    float a[16], b[8], c[4], d[2];
#pragma unroll
    for (int k = 0; k < 16; ++k) a[k] = k < kMoments ? v[k] : 0.0f;
#pragma unroll
    for (int j = 0; j < 8; ++j) b[j] = pair_add32(a[j], a[j + 8]);
#pragma unroll
    for (int j = 0; j < 4; ++j) c[j] = pair_add16(b[j], b[j + 4]);
    const bool up8 = (lane & 8) != 0;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const float keep = up8 ? c[j + 2] : c[j];
        const float send = up8 ? c[j] : c[j + 2];
        d[j] = keep + dpp_f<kDppRor8>(send);
    }
    const bool up4 = (lane & 4) != 0;
    float x = (up4 ? d[1] : d[0]) + dpp_f<kDppHalfMirror>(up4 ? d[0] : d[1]);
    x += dpp_f<kDppXor2>(x);
    x += dpp_f<kDppXor1>(x);
    const int idx = ((lane >> 5) & 1) * 8 + ((lane >> 4) & 1) * 4 + ((lane >> 3) & 1) * 2 + ((lane >> 2) & 1);
    const unsigned long long same = __builtin_amdgcn_ballot_w64(st.key == key);
    if (same != 0ULL) {
        if ((lane & 3) == 0) atomicAdd(&G.val[__builtin_ctzll(same)][idx], x);
        return;
    }
    if ((lane & 3) == 0) G.val[st.n][idx] = x;
    if (lane == st.n) st.key = key;
    if (++st.n == kStage) stage_flush(G, st, sc, gr, lane, drops);
}

__device__ __forceinline__ int wave_lane() { return threadIdx.x & (kWave - 1); }

// LBVH traversal of the lanes executing the call: wave-uniform packet walk or per-lane walk.
template <typename F>
__device__ __forceinline__ void trav(const DevParams& p, const DevScene& sc, const Ray& ray, float ta, float tb,
                                     F&& on_leaf) {
    if (p.packet) traverse_packet(sc.nodes, sc.total_nodes, true, ray, ta, tb, on_leaf);
    else traverse(sc.nodes, sc.total_nodes, ray, ta, tb, on_leaf);
}

// Layout: the R rays of a wavefront (DevParams::rays_per_wave) share one region of R * words per ray;
// sector c of the ray in lane l sits at (c * R + l) * 8 words.  The rays of a wavefront thus write
// neighbouring sectors (no stride that would send every lane to one memory channel).
struct Rec {
    unsigned int* w = nullptr;  // sector 0 of this ray; nullptr: off
    int stride = 8 * kWave;     // words from one of its sectors to the next
    int pos = 0;                // next word (a multiple of 8)
    int end = 0;                // capacity (recording) or words recorded (replay)
    bool full = false;          // recording ran out of space
};

// Region of wavefront `wave` (groups of 64 items cut into 64 / rays_per_wave wavefronts each).
__device__ __forceinline__ unsigned int* rec_region(const DevParams& p, int64_t wave) {
    return p.rec + wave * ((int64_t)p.rays_per_wave * p.rec_words);
}

__device__ __forceinline__ unsigned int* rec_at(const Rec& rc, int w) { return rc.w + (w >> 3) * rc.stride + (w & 7); }

__device__ __forceinline__ int rec_len(int cnt) { return (2 + cnt + 7) & ~7; }

typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

struct RayRef {
    int view;
    int pixel;
    int64_t out;  // output row
    bool active;
};

// Tile-ordered enumeration for the implicit full-view mode: work item w -> pixel.
__device__ __forceinline__ bool tile_pixel(int64_t w, int width, int height, int& pixel) {
    const int64_t tile = w >> 6;
    const int lane = (int)(w & 63);
    const int tiles_x = (width + 7) >> 3;
    const int tx = (int)(tile % tiles_x), ty = (int)(tile / tiles_x);
    const int px = tx * 8 + (lane & 7), py = ty * 8 + (lane >> 3);
    if (px >= width || py >= height) return false;
    pixel = py * width + px;
    return true;
}

__device__ __forceinline__ void flush_counters(const Counters& c, DevStats st) {
    // wave-level reduction, one atomic per counter per wave
    unsigned int v[7] = {c.K, c.P, c.ovf, c.fallback, c.gathers, c.rec_words, c.rec_full};
    const int idx[7] = {C_K, C_P, C_OVF, C_FALLBACK, C_GATHER, C_REC_WORDS, C_REC_FULL};
#pragma unroll
    for (int k = 0; k < 7; ++k) {
        unsigned int x = v[k];
        for (int o = 32; o > 0; o >>= 1) x += __shfl_xor(x, o, 64);
        v[k] = x;
    }
    if (wave_lane() == 0) {
#pragma unroll
        for (int k = 0; k < 7; ++k)
            if (v[k]) atomicAdd(&st.c[idx[k]], (unsigned long long)v[k]);
    }
}

// Item of lane `lane` of wavefront `wave`, -1 for a lane without one.  With 64 rays per wavefront the
// items are consecutive (8x8 tiles of a view); with fewer, each group of 64 items is cut along the
// Z-curve of its 8x8 tile, so that 16 rays are a 4x4 block and 4 rays a 2x2 block.
__device__ __forceinline__ int64_t wave_item(const DevParams& p, int64_t wave, int lane) {
    if (p.rays_per_wave == kWave) return wave * kWave + lane;
    if (lane >= p.rays_per_wave) return -1;
    const int64_t i = wave * p.rays_per_wave + lane;
    const int z = (int)(i & 63);
    const int x = (z & 1) | ((z >> 1) & 2) | ((z >> 2) & 4), y = ((z >> 1) & 1) | ((z >> 2) & 2) | ((z >> 3) & 4);
    return (i & ~(int64_t)63) + 8 * y + x;
}

// rec_len of a ray in a wavefront's tile record: its 16-byte cells (at most 2^24), whether it is that of
// a split wavefront, the ray's beam in it, kTileRecord.
constexpr int kTileRecord = 0x40000000, kTileGroupShift = 28, kTileSplit = 1 << 27, kTileCells = kTileSplit - 1;

// Starts a ray: clears its output; false when the ray has no slab to process (it misses the scene
// box, or its first slab is below half an ulp of t).
__device__ __forceinline__ bool forward_begin(const DevParams& p, const Ray& ray, RayOut& o) {
    o.C[0] = o.C[1] = o.C[2] = 0.0f;
    o.depth = 0.0f;
    o.T = 1.0f;
    return ray.tenter < ray.texit && add_exact(ray.tenter, p.dt * (float)p.spb) > ray.tenter;
}

enum RayStatus { RAY_NONE = 0, RAY_OK = 1, RAY_BAD = 2 };

// Work item -> (view, pixel, output row).  RAY_NONE: past the end of the job, or a padding item
// of the implicit single-view mode (whose items are enumerated in 8x8 tiles, num_items being the
// padded tile count * 64).  RAY_BAD: a listed view or pixel index outside the views set by
// rg_set_views; such a ray is skipped (its output row reads NaN) and counted.
__device__ __forceinline__ int resolve(const RayJob& job, int64_t w, RayRef& q) {
    q.view = job.view;
    q.pixel = 0;
    q.out = w;
    q.active = false;
    if (job.ray_view || job.pixels) {
        if (w >= job.num_rays) return RAY_NONE;
        if (job.ray_view) {
            q.view = job.ray_view[w];
            q.pixel = job.ray_pixel[w];
        } else {
            q.pixel = job.pixels[w];
        }
        if ((unsigned)q.view >= (unsigned)job.num_views) return RAY_BAD;
        const rg_camera& cam = job.cams[q.view];
        if (q.pixel < 0 || (int64_t)q.pixel >= (int64_t)cam.width * cam.height) return RAY_BAD;
        q.active = true;
        return RAY_OK;
    }
    if (w >= job.num_rays) return RAY_NONE;
    const rg_camera& cam = job.cams[job.view];
    int pixel;
    if (!tile_pixel(w, cam.width, cam.height, pixel)) return RAY_NONE;
    q.pixel = pixel;
    q.out = pixel;
    q.active = true;
    return RAY_OK;
}

// Writes a finished ray's colour (with the background behind its remaining transmittance),
// depth and opacity, and closes its hit-list records.
template <int RM>
__device__ __forceinline__ void forward_finish(const DevParams& p, const RayRef& q, int64_t item, const RayOut& o, const Rec& rc,
                                               Counters& ctr, float* __restrict__ out_rgb, float* __restrict__ out_depth,
                                               float* __restrict__ out_opac) {
    if constexpr (RM == 1) {
        p.rec_len[item] = rc.pos | (rc.full ? (int)0x80000000u : 0);
        p.rec_id[item] = make_int2(q.view, q.pixel);  // the backward replays only the same ray
        ctr.rec_full += rc.full ? 1u : 0u;
    }
    out_rgb[3 * q.out + 0] = o.C[0] + o.T * p.bg;
    out_rgb[3 * q.out + 1] = o.C[1] + o.T * p.bg;
    out_rgb[3 * q.out + 2] = o.C[2] + o.T * p.bg;
    if (out_depth) out_depth[q.out] = o.depth;
    if (out_opac) out_opac[q.out] = 1.0f - o.T;
}

// A ray whose view or pixel index is out of range: NaN outputs, no records, counted.
template <int RM>
__device__ __forceinline__ void forward_bad(const DevParams& p, const RayRef& q, int64_t item, DevStats st,
                                            float* __restrict__ out_rgb, float* __restrict__ out_depth,
                                            float* __restrict__ out_opac) {
    atomicAdd(&st.c[C_BAD], 1ull);
    const float nan = __builtin_nanf("");
    out_rgb[3 * q.out + 0] = nan;
    out_rgb[3 * q.out + 1] = nan;
    out_rgb[3 * q.out + 2] = nan;
    if (out_depth) out_depth[q.out] = nan;
    if (out_opac) out_opac[q.out] = nan;
    if constexpr (RM == 1) {
        p.rec_len[item] = 0;
        p.rec_id[item] = make_int2(-1, -1);
    }
}

// XCD-aware block order: consecutive work blocks land on the same XCD's L2.
__device__ __forceinline__ int64_t block_item(int64_t b, int64_t nblocks) {
    const int64_t per = (nblocks + 7) >> 3;
    const int64_t xcd = b & 7, k = b >> 3;
    return xcd * per + k;
}

// One lane's ray of a backward pass.
struct BwdRay {
    bool active = false;
    Ray ray = {};
    unsigned int seed = 0u;
    float dL[3] = {0.0f, 0.0f, 0.0f};
    float Cf[3] = {0.0f, 0.0f, 0.0f};
    int view = 0;
    int tile = -1;       // the ray's beam in its wavefront's tile record (-1: none)
    bool trunc = false;  // the record holds its hits up to some depth only
    Rec rc;
};

// Sets up work item `item` of a backward: its rendered colour, dL/dC (given, or formed from the
// per-pixel loss against target, whose value is added to loss), its hit-list records when they
// were written for this same ray, and the ray itself.  A ray with zero dL/dC stays inactive.
template <bool RNG, int RM>
__device__ __forceinline__ void backward_setup(const DevScene& sc, const DevParams& p, const RayJob& job, int64_t wave,
                                               int lane, int64_t item, const float* __restrict__ ray_colors,
                                               const float* __restrict__ dLdC, const float* __restrict__ target,
                                               int loss_kind, DevStats st, BwdRay& b, float& loss, bool split = false,
                                               bool lead = true) {
    RayRef q;
    const int rs = resolve(job, item, q);
    if (rs == RAY_BAD && lead) atomicAdd(&st.c[C_BAD], 1ull);
    if (rs != RAY_OK) return;
    b.Cf[0] = ray_colors[3 * q.out];
    b.Cf[1] = ray_colors[3 * q.out + 1];
    b.Cf[2] = ray_colors[3 * q.out + 2];
    if (target) {
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            const float e = b.Cf[c] - target[3 * q.out + c];
            if (loss_kind == 1) {
                loss += fabsf(e);
                b.dL[c] = e > 0.0f ? 1.0f : (e < 0.0f ? -1.0f : 0.0f);
            } else {
                loss += e * e;
                b.dL[c] = 2.0f * e;
            }
        }
    } else {
        b.dL[0] = dLdC[3 * q.out];
        b.dL[1] = dLdC[3 * q.out + 1];
        b.dL[2] = dLdC[3 * q.out + 2];
    }
    if (b.dL[0] == 0.0f && b.dL[1] == 0.0f && b.dL[2] == 0.0f) return;
    b.active = true;
    b.view = q.view;
    if constexpr (RM == 2) {
        // records of this item are replayed only when the forward wrote them for the same
        // (view, pixel); otherwise the ray walks the tree
        const int2 id = p.rec_id[item];
        if (id.x == q.view && id.y == q.pixel) {
            const int len = p.rec_len[item];
            if (len & kTileRecord) {
                // the record of the whole wavefront is no use to a part of it, nor the other way round
                if (((len & kTileSplit) != 0) == split) b.tile = (len >> kTileGroupShift) & 3;
                b.trunc = len < 0;
                b.rc.end = min(len & kTileCells, (p.rays_per_wave * p.rec_words) >> 2);
            } else {
                b.rc.w = rec_region(p, wave) + 8 * lane;
                b.rc.stride = 8 * p.rays_per_wave;
                b.rc.end = min(len & 0x7fffffff, p.rec_words);
            }
        }
    }
    const rg_camera cam = job.cams[q.view];
    b.seed = RNG ? tea4(p.iteration, (unsigned int)q.pixel) : 0u;
    b.ray = make_ray(cam, q.pixel, sc.box, p.t_near, p.t_far, RNG ? p.jitter : 0, &b.seed);
}

// Adds the wavefront's loss to the loss counters: whole wavefronts in 32 bits, the many small terms
// of narrow ones in 64, where the order of their additions does not show (k_loss_out adds the two).
__device__ __forceinline__ void add_loss(const DevParams& p, float loss, int lane, DevStats st) {
    const float ls = wave_sum64(loss);
    if (lane != 0 || ls == 0.0f) return;
    if (p.rays_per_wave == kWave) atomicAdd(reinterpret_cast<float*>(&st.c[C_LOSS]), ls);
    else atomicAdd(reinterpret_cast<double*>(&st.c[C_LOSS64]), (double)ls);
}

// ------------------------------------------------------------------ persistent kernels --------
//
// The same per-ray work as k_forward / k_backward, but launched as as many wavefronts as the GPU
// holds at once, each taking p.ray_chunk work items (whole 8x8 tiles) at a time from a device work
// queue until every queue is empty.  The items are cut into 8 contiguous bands, one per XCD (a
// wavefront's XCD is its block index mod 8: blocks are dispatched round-robin over the XCDs), so
// each XCD's L2 sees a compact part of the scene as with the grid launch; a wavefront whose band is
// exhausted takes chunks from the other bands (work stealing), so no XCD idles while another still
// has rays -- the grid launch's static bands (one view per XCD on the 8-view workload) leave the
// XCDs with the cheaper views idle at the end.

// Next chunk [lo, hi) of work items for a wavefront on XCD x: its own band's queue first, then the
// other bands' in turn.  spent: bands this wavefront found exhausted.  Called by all active lanes
// together; the results are wave-uniform.
__device__ __forceinline__ bool take_chunk(const DevParams& p, int64_t num_items, int x, int64_t& lo, int64_t& hi,
                                           unsigned int& spent) {
    const int64_t tiles = (num_items + kWave - 1) / kWave;
    const int64_t band = ((tiles + 7) / 8) * kWave;  // items per band, whole tiles
    const bool leader = (int)threadIdx.x == __ffsll((long long)__ballot(1)) - 1;
    for (int j = 0; j < 8; ++j) {
        const int b = (x + j) & 7;
        if (spent & (1u << b)) continue;
        const int64_t start = (int64_t)b * band;
        const int64_t len = min(band, num_items - start);
        if (len <= 0) {
            spent |= 1u << b;
            continue;
        }
        unsigned long long got = 0ull;
        if (leader) got = atomicAdd(&p.queue[b], (unsigned long long)p.ray_chunk);
        const unsigned int glo = __builtin_amdgcn_readfirstlane((unsigned int)(got & 0xffffffffull));
        const unsigned int ghi = __builtin_amdgcn_readfirstlane((unsigned int)(got >> 32));
        const int64_t g = (int64_t)(((unsigned long long)ghi << 32) | glo);
        if (g < len) {
            lo = start + g;
            hi = start + min(g + (int64_t)p.ray_chunk, len);
            return true;
        }
        spent |= 1u << b;
    }
    return false;
}

// Lanes of mask below this lane.
__device__ __forceinline__ int lanes_below(unsigned long long mask) {
    return __builtin_amdgcn_mbcnt_hi((unsigned int)(mask >> 32), __builtin_amdgcn_mbcnt_lo((unsigned int)mask, 0u));
}

// Wavefronts of a job (groups of 64 items, each cut into 64 / rays_per_wave).
inline int64_t num_waves(const DevParams& p, int64_t items) {
    return (items + kWave - 1) / kWave * (kWave / p.rays_per_wave);
}

}  // namespace rg
