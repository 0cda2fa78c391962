// Beam gathers: the candidates of a whole wavefront's rays (an 8x8 pixel tile) from one tree walk.
//
// The rays of a tile share their origin and differ little in direction, so the Gaussians that any
// of them can meet inside a depth range are found once for the tile, 64 tree nodes at a time (one
// per lane) against the beam that holds all its rays, instead of one node at a time against 64
// rays.  The candidates then go through the exact per-ray predicate in slot order, so which
// Gaussians a ray hits, and the order it sums them in, do not depend on how they were found: the
// beam tests only have to be conservative.
//
// What bounds it: with one node per step the walks took 34.6k node visits of about 25 vector
// instructions per tile on the 1M-Gaussian workload (8.13M rays), 40 % of the forward's instructions,
// most of the rest being per-slab walks of dense stretches; with 64 nodes per step a tile gathers 16
// times, and its time goes to the predicate of 2000 candidates (1220 of them hit by 35 lanes on
// average).  Forward 224 -> 119 ms, and backward 204 -> 167 ms from the events it leaves.
#pragma once

#include "rg_device.h"

namespace rg {

constexpr int kTileCand = 256;   // candidates of one gathered depth range (4 per lane)
constexpr int kTileStack = 512;  // pending tree nodes of a gather

struct TileLds {
    int stack[kTileStack];
    int slot[kTileCand];
    float z0[kTileCand], z1[kTileCand];  // depth range in which the beam can meet the candidate
};

__device__ __forceinline__ float wave_max64f(float v) { return -wave_min64f(-v); }

__device__ __forceinline__ float uniform_f(float v) {
    return __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(v)));
}

// Lanes of mask below this lane.
__device__ __forceinline__ int mask_rank(unsigned long long mask) {
    return __builtin_amdgcn_mbcnt_hi((unsigned int)(mask >> 32), __builtin_amdgcn_mbcnt_lo((unsigned int)mask, 0u));
}

// The rays o + t d, t >= 0, whose directions lie within [dmin, dmax] per component and within eps of
// dc (wave-uniform).
struct Beam {
    float o[3];
    float dc[3];
    float eps;
    float rmin[3], rmax[3];  // 1 / dmin, 1 / dmax
};

// Beam of the lanes with act (at least one; they share their origin).  Called by all 64 lanes.
__device__ __forceinline__ Beam make_beam(bool act, const Ray& r) {
    Beam b;
    const int first = __ffsll((long long)__ballot(act)) - 1;
    b.o[0] = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(r.ox), first));
    b.o[1] = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(r.oy), first));
    b.o[2] = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(r.oz), first));
    const float d[3] = {r.dx, r.dy, r.dz};
    float dev = 0.0f;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        float lo = uniform_f(wave_min64f(act ? d[a] : INFINITY));
        float hi = uniform_f(wave_max64f(act ? d[a] : -INFINITY));
        b.dc[a] = 0.5f * (lo + hi);
        const float e = act ? d[a] - b.dc[a] : 0.0f;
        dev += e * e;
        // widened past the rounding of the tests below, and away from zero
        lo -= 1e-6f;
        hi += 1e-6f;
        if (fabsf(lo) < 1e-9f) lo = -1e-9f;
        if (fabsf(hi) < 1e-9f) hi = 1e-9f;
        b.rmin[a] = 1.0f / lo;
        b.rmax[a] = 1.0f / hi;
    }
    b.eps = uniform_f(wave_max64f(__builtin_sqrtf(dev))) * 1.0001f + 1e-6f;
    return b;
}

// Whether the beam can meet the box within the depths [s0, s1]: per axis, o + t dmin <= hi and
// o + t dmax >= lo.  The boxes carry their own padding against rounding (k_preprocess).  An empty
// box (lo = +inf, hi = -inf) fails; a NaN passes.
__device__ __forceinline__ bool beam_box(const Beam& b, const float4 lo, const float4 hi, float s0, float s1) {
    float tn = s0, tf = s1;
    const float L[3] = {lo.x, lo.y, lo.z}, H[3] = {hi.x, hi.y, hi.z};
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        const float th = (H[a] - b.o[a]) * b.rmin[a];
        const float tl = (L[a] - b.o[a]) * b.rmax[a];
        const bool up = b.rmin[a] > 0.0f, vp = b.rmax[a] > 0.0f;
        tf = fminf(tf, up ? th : INFINITY);
        tn = fmaxf(tn, up ? -INFINITY : th);
        tn = fmaxf(tn, vp ? tl : -INFINITY);
        tf = fminf(tf, vp ? INFINITY : tl);
    }
    return !(tn > tf * 1.00001f);
}

// Whether some ray of the beam can meet the Gaussian's bounding ellipsoid within [s0, s1], and the
// depths [z0, z1] at which it can.  With the ellipsoid's unit-sphere map M', a ray within eps of
// the centre line is within t eps |M'| of it at depth t in that map, so it meets the unit sphere
// only where the centre line is inside the sphere of radius 1 + t eps |M'|, and t is at most the
// distance to the ellipsoid's far side.  The radius is padded far beyond the rounding of the predicate and of this test, which grow with |M'O|.
__device__ __forceinline__ bool beam_ellipsoid(const Beam& b, const float4 g0, const float4 g1, const float4 g2,
                                               const float4 g3, float s0, float s1, float& z0, float& z1) {
    const float Ox = b.o[0] - g0.x, Oy = b.o[1] - g0.y, Oz = b.o[2] - g0.z;
    const float P0 = g1.x * Ox + g1.y * Oy + g1.z * Oz;
    const float P1 = g2.x * Ox + g2.y * Oy + g2.z * Oz;
    const float P2 = g3.x * Ox + g3.y * Oy + g3.z * Oz;
    const float D0 = g1.x * b.dc[0] + g1.y * b.dc[1] + g1.z * b.dc[2];
    const float D1 = g2.x * b.dc[0] + g2.y * b.dc[1] + g2.z * b.dc[2];
    const float D2 = g3.x * b.dc[0] + g3.y * b.dc[1] + g3.z * b.dc[2];
    const float n1 = g1.x * g1.x + g1.y * g1.y + g1.z * g1.z;
    const float n2 = g2.x * g2.x + g2.y * g2.y + g2.z * g2.z;
    const float n3 = g3.x * g3.x + g3.y * g3.y + g3.z * g3.z;
    // largest and smallest |M' x|^2 / |x|^2 (Gershgorin: exact for the orthogonal rows of a unit
    // quaternion, a bound for any other)
    const float x12 = fabsf(g1.x * g2.x + g1.y * g2.y + g1.z * g2.z);
    const float x13 = fabsf(g1.x * g3.x + g1.y * g3.y + g1.z * g3.z);
    const float x23 = fabsf(g2.x * g3.x + g2.y * g3.y + g2.z * g3.z);
    const float nmax = fmaxf(n1 + x12 + x13, fmaxf(n2 + x12 + x23, n3 + x13 + x23));
    const float nmin = fminf(n1 - x12 - x13, fminf(n2 - x12 - x23, n3 - x13 - x23));
    const float far = __builtin_sqrtf(Ox * Ox + Oy * Oy + Oz * Oz) + 1.0f / __builtin_sqrtf(fmaxf(nmin, 0.0f));
    const float opp = P0 * P0 + P1 * P1 + P2 * P2;
    const float inv = 1.0f / (D0 * D0 + D1 * D1 + D2 * D2);
    const float tc = -(P0 * D0 + P1 * D1 + P2 * D2) * inv;
    const float Q0 = P0 + tc * D0, Q1 = P1 + tc * D1, Q2 = P2 + tc * D2;
    const float pp = Q0 * Q0 + Q1 * Q1 + Q2 * Q2;
    const float reach = fminf(far * 1.001f, s1 * 1.001f) * b.eps * __builtin_sqrtf(nmax);
    const float R = 1.002f + reach * 1.002f + 3e-5f * __builtin_sqrtf(opp);
    const float q = (R * R - pp) * inv;
    if (!(g1.w > 0.0f) || q < 0.0f) return false;
    const float half = __builtin_sqrtf(q);
    const float pad = 1e-5f * (fabsf(tc) + half) + 1e-6f;
    z0 = tc - half - pad;
    z1 = tc + half + pad;
    if (!(z0 <= z1)) {  // NaN: no bound
        z0 = -INFINITY;
        z1 = INFINITY;
    }
    return !(z0 > s1) && !(z1 < s0);
}

// Gathers the beam's candidates within [s0, s1] into W, sorted by slot; returns their number, or -1
// when they do not fit.  Called by all 64 lanes; wave-uniform result.
__device__ __forceinline__ int beam_gather(const float4* __restrict__ nodes, const float4* __restrict__ geo, int total,
                                           const Beam& b, float s0, float s1, TileLds& W, int lane) {
    if (total <= 0) return 0;
    if (lane == 0) W.stack[0] = 0;
    int sp = 1, cnt = 0;
    __syncthreads();
    while (sp > 0) {
        // each of the p nodes taken puts at most two in its place
        const int p = min(min(sp, 64), kTileStack - sp);
        if (p <= 0) return -1;
        int node = lane < p ? W.stack[sp - 1 - lane] : total;
        sp -= p;
        __syncthreads();
        bool inner = false, keep = false;
        int right = 0, slot = 0;
        float z0 = 0.0f, z1 = 0.0f;
        if ((unsigned)node < (unsigned)total) {
            const float4 lo = nodes[2 * node], hi = nodes[2 * node + 1];
            if (beam_box(b, lo, hi, s0, s1)) {
                slot = __float_as_int(hi.w);
                if (slot < 0) {
                    right = ~slot;
                    inner = right > node;  // links only lead forward: the walk ends
                } else if (slot < ((total + 1) >> 1)) {
                    keep = beam_ellipsoid(b, geo[4 * slot], geo[4 * slot + 1], geo[4 * slot + 2], geo[4 * slot + 3],
                                          s0, s1, z0, z1);
                }
            }
        }
        const unsigned long long mi = __ballot(inner), mk = __ballot(keep);
        const int nk = __popcll(mk);
        if (cnt + nk > kTileCand) return -1;
        if (inner) {
            const int at = sp + 2 * mask_rank(mi);
            W.stack[at] = right;
            W.stack[at + 1] = node + 1;
        }
        if (keep) {
            const int at = cnt + mask_rank(mk);
            W.slot[at] = slot;
            W.z0[at] = z0;
            W.z1[at] = z1;
        }
        sp += 2 * __popcll(mi);
        cnt += nk;
        __syncthreads();
    }
    // by slot: each candidate's rank is the number of smaller slots
    constexpr int C = kTileCand / 64;
    int s[C], rank[C];
    float a0[C], a1[C];
#pragma unroll
    for (int j = 0; j < C; ++j) {
        const int i = 64 * j + lane;
        s[j] = i < cnt ? W.slot[i] : 0x7fffffff;
        a0[j] = W.z0[i];
        a1[j] = W.z1[i];
        rank[j] = 0;
    }
#pragma unroll
    for (int jj = 0; jj < C; ++jj) {
        const int lim = min(64, cnt - 64 * jj);
        for (int i = 0; i < lim; ++i) {
            const int v = __builtin_amdgcn_readlane(s[jj], i);
#pragma unroll
            for (int j = 0; j < C; ++j)
                if (64 * j < cnt) rank[j] += v < s[j] ? 1 : 0;
        }
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < C; ++j)
        if (64 * j + lane < cnt) {
            W.slot[rank[j]] = s[j];
            W.z0[rank[j]] = a0[j];
            W.z1[rank[j]] = a1[j];
        }
    __syncthreads();
    return cnt;
}

// A record or colour read at a wave-uniform index, as scalar loads.
__device__ __forceinline__ float4 ld_uniform(const float4* __restrict__ p, int64_t i) {
    const node_f32x4 v = ((const const_node_f32x4*)p)[i];
    return make_float4(v.x, v.y, v.z, v.w);
}

}  // namespace rg
