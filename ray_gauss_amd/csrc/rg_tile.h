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
// times, and its time goes to the predicate of its candidates, the 8 samples of 1220 events (35 lanes
// hit on average) and the gathers.  Forward 224 -> 119.7 ms, and backward 204 -> 167 ms from the events it
// leaves; with the candidates' terms in the list, the shorter roots and the tighter beams 99.2 ms; with
// leaves tested 64 at a time, ranges that shrink while they are gathered and rounds of several lists 87.9.
// With cheaper rounds and merged gradient records 83.7 and 134.7 ms: 477k and 660k vector instructions a
// tile, one every 3.4 and 3.9 cycles.
#pragma once

#include "rg_device.h"

namespace rg {

constexpr int kTileCand = 256;   // candidates of one gathered depth range (4 per lane)
constexpr int kTileStack = 384;  // pending tree nodes of a gather
constexpr int kTileReserve = 128;  // of them for the depth of the tree

// The rays o + t d, t >= 0, whose directions lie within [dmin, dmax] per component and within eps of
// dc + a u + b v with |a|, |b| <= 1 (wave-uniform).
struct Beam {
    float o[3];
    float dc[3];
    float u[3], v[3];
    float eps;
    float rmin[3], rmax[3];  // 1 / dmin, 1 / dmax
    int cuts;                // halvings of the leaves that a round's gathers may make
};

// A slab's samples in wavefronts that hold one in each lane (spread), exchanged between a ray's eight lanes.
struct SpreadLds {
    float alpha[kWave], rest[kWave];
    float v[4][kWave];
};

struct TileLds {
    union {
        int stack[kTileStack];  // during a gather
        SpreadLds spread;       // after the round's hits
    };
    int slot[kTileCand];                 // 2 slot + 1 where the terms are out of inv_sqrt_exact's range
    float4 oc[kTileCand];                // the predicate's O' = M' (o - mu) and c = |O'|^2 - 1
    float z0[kTileCand], z1[kTileCand];  // depth range in which the beam can meet the candidate
    int leaf[2 * kWave], leaf_slot[2 * kWave];  // leaves (nodes) whose box the beam meets, not tested yet
    Beam beam;                           // of the gathers: kept here, not in registers between them
};

__device__ __forceinline__ float wave_max64f(float v) { return -wave_min64f(-v); }

__device__ __forceinline__ float uniform_f(float v) {
    return __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(v)));
}

// Lanes of mask below this lane.
__device__ __forceinline__ int mask_rank(unsigned long long mask) {
    return __builtin_amdgcn_mbcnt_hi((unsigned int)(mask >> 32), __builtin_amdgcn_mbcnt_lo((unsigned int)mask, 0u));
}

// Beam of the lanes with act (at least one; they share their origin).  axis is the direction its
// sides should follow (the image's rows: the beam of a block of pixels is then little larger than the
// block).  Called by all 64 lanes.
__device__ __forceinline__ void make_beam(bool act, const Ray& r, const float* axis, TileLds& W, int lane) {
    Beam b;
    const int first = __ffsll((long long)__ballot(act)) - 1;
    b.o[0] = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(r.ox), first));
    b.o[1] = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(r.oy), first));
    b.o[2] = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(r.oz), first));
    const float d[3] = {r.dx, r.dy, r.dz};
    float e[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        float lo = uniform_f(wave_min64f(act ? d[a] : INFINITY));
        float hi = uniform_f(wave_max64f(act ? d[a] : -INFINITY));
        b.dc[a] = 0.5f * (lo + hi);
        e[a] = act ? d[a] - b.dc[a] : 0.0f;
        // widened past the rounding of the tests below, and away from zero
        lo -= 1e-6f;
        hi += 1e-6f;
        if (fabsf(lo) < 1e-9f) lo = -1e-9f;
        if (fabsf(hi) < 1e-9f) hi = 1e-9f;
        b.rmin[a] = 1.0f / lo;
        b.rmax[a] = 1.0f / hi;
    }
    // unit vectors u along the axis across dc, v across both; any others, or none, would do
    const float dd = b.dc[0] * b.dc[0] + b.dc[1] * b.dc[1] + b.dc[2] * b.dc[2];
    const float k = (axis[0] * b.dc[0] + axis[1] * b.dc[1] + axis[2] * b.dc[2]) / dd;
    float u[3], v[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) u[a] = axis[a] - k * b.dc[a];
    const float il = 1.0f / __builtin_sqrtf(u[0] * u[0] + u[1] * u[1] + u[2] * u[2]);
    const float jl = il / __builtin_sqrtf(dd);
    const bool none = !(il < 1e6f) || !(jl < 1e6f);
    v[0] = none ? 0.0f : (b.dc[1] * u[2] - b.dc[2] * u[1]) * jl;
    v[1] = none ? 0.0f : (b.dc[2] * u[0] - b.dc[0] * u[2]) * jl;
    v[2] = none ? 0.0f : (b.dc[0] * u[1] - b.dc[1] * u[0]) * jl;
#pragma unroll
    for (int a = 0; a < 3; ++a) u[a] = none ? 0.0f : u[a] * il;
    const float eu = e[0] * u[0] + e[1] * u[1] + e[2] * u[2], ev = e[0] * v[0] + e[1] * v[1] + e[2] * v[2];
    const float hu = uniform_f(wave_max64f(fabsf(eu))), hv = uniform_f(wave_max64f(fabsf(ev)));
    float dev = 0.0f;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        const float f = e[a] - eu * u[a] - ev * v[a];
        dev += f * f;
        b.u[a] = u[a] * hu;
        b.v[a] = v[a] * hv;
    }
    b.eps = wave_max64f(__builtin_sqrtf(dev)) * 1.0001f + 1e-6f;
    // A round whose candidates take several lists evaluates all of them; one that walks the tree, those in
    // the boxes that its rays meet, which are fewer where 64 rays are scattered over a wide beam.  Forward of
    // random rays in blocks of 8 / 32 / 64 / 128 of 1024 pixels (widths 0.006, 0.023, 0.045, 0.09) at 1M Gaussians,
    // several lists: 4.86 / 27.2 / 103 / 498 ms, at most two: 6.55 / 26.2 / 56 / 77.
    b.cuts = fmaxf(hu, hv) < 0.0125f ? 0x7fffffff : 1;
    __syncthreads();
    if (lane == 0) W.beam = b;
    __syncthreads();
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
// depths [z0, z1] at which it can; odd: |D'|^2 may be out of inv_sqrt_exact's range.  In the
// ellipsoid's unit-sphere map M' the ray is P + t (D + a U + b V + e), with D, U, V the images of dc, u,
// v and |e| <= er = eps |M'|, and t is at most the distance to the ellipsoid's far side.  Across D, along
// the unit vector n from the centre to the centre line's closest point Q, the ray is at least
// pm = |Q| - t (|U.n| + |V.n| + er) away: it meets the unit sphere only if pm <= 1, and then only where
// its component along D is at most sqrt(1 - pm^2).  The radius is padded far beyond the rounding
// of the predicate and of this test, which grow with |P|.
// A sphere of radius 1 + t eps |M'| around the centre line, with the beam's whole radius as eps, is 40
// instructions less, but a third of the candidates it leaves were met by no ray of the round.
__device__ __forceinline__ bool beam_ellipsoid(const Beam& b, const float4 g0, const float4 g1, const float4 g2,
                                               const float4 g3, float s0, float s1, float& z0, float& z1, bool& odd) {
    const float Ox = b.o[0] - g0.x, Oy = b.o[1] - g0.y, Oz = b.o[2] - g0.z;
    auto row = [](const float4 g, const float* x) { return g.x * x[0] + g.y * x[1] + g.z * x[2]; };
    const float O[3] = {Ox, Oy, Oz};
    const float P0 = row(g1, O), P1 = row(g2, O), P2 = row(g3, O);
    const float D0 = row(g1, b.dc), D1 = row(g2, b.dc), D2 = row(g3, b.dc);
    const float U0 = row(g1, b.u), U1 = row(g2, b.u), U2 = row(g3, b.u);
    const float V0 = row(g1, b.v), V1 = row(g2, b.v), V2 = row(g3, b.v);
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
    odd = !(nmin > 0x1p-58f && nmax < 0x1p60f);
    const float far = __builtin_sqrtf(Ox * Ox + Oy * Oy + Oz * Oz) + 1.0f / __builtin_sqrtf(fmaxf(nmin, 0.0f));
    const float opp = P0 * P0 + P1 * P1 + P2 * P2;
    const float inv = 1.0f / (D0 * D0 + D1 * D1 + D2 * D2);
    const float tc = -(P0 * D0 + P1 * D1 + P2 * D2) * inv;
    const float Q0 = P0 + tc * D0, Q1 = P1 + tc * D1, Q2 = P2 + tc * D2;
    const float q = __builtin_sqrtf(Q0 * Q0 + Q1 * Q1 + Q2 * Q2);
    const float reach = fminf(far, s1) * 1.002f;
    const float er = b.eps * __builtin_sqrtf(nmax);
    const float wn = (fabsf(U0 * Q0 + U1 * Q1 + U2 * Q2) + fabsf(V0 * Q0 + V1 * Q1 + V2 * Q2)) / fmaxf(q, 1e-20f);
    const float wd = (fabsf(U0 * D0 + U1 * D1 + U2 * D2) + fabsf(V0 * D0 + V1 * D1 + V2 * D2)) * inv;
    const float R = 1.002f + 3e-5f * __builtin_sqrtf(opp);
    const float pm = fmaxf(q - reach * (wn + er), 0.0f);
    if (!(g1.w > 0.0f) || pm > R) return false;
    const float half = __builtin_sqrtf((R * R - pm * pm) * inv) + reach * (wd + er * __builtin_sqrtf(inv));
    const float pad = 1e-5f * (fabsf(tc) + half) + 1e-6f;
    z0 = tc - half - pad;
    z1 = tc + half + pad;
    if (!(z0 <= z1)) {  // NaN: no bound
        z0 = -INFINITY;
        z1 = INFINITY;
    }
    return !(z0 > s1) && !(z1 < s0);
}

// O' and c of the predicate, with isect_terms' operations.
__device__ __forceinline__ float4 origin_terms(const Beam& b, const float4 g0, const float4 g1, const float4 g2,
                                               const float4 g3) {
#pragma clang fp contract(off)
    const float Ox = b.o[0] - g0.x, Oy = b.o[1] - g0.y, Oz = b.o[2] - g0.z;
    const float Op0 = (g1.x * Ox + g1.y * Oy) + g1.z * Oz;
    const float Op1 = (g2.x * Ox + g2.y * Oy) + g2.z * Oz;
    const float Op2 = (g3.x * Ox + g3.y * Oy) + g3.z * Oz;
    return make_float4(Op0, Op1, Op2, ((Op0 * Op0 + Op1 * Op1) + Op2 * Op2) - 1.0f);
}

// The gathered depth range of a marching tile (wave-uniform).
struct TileWalk {
    float s1 = 0.0f;       // end of the range
    int m = 1;             // its length in slabs
    int cnt = 0;           // candidates in the list
    int first = 0, limit = 0;  // nodes whose leaves it covers
    int cuts = 0;            // halvings of the leaves that the round may still make
    int skip = 0, back = 0;  // rounds to walk before the next gather, and after the last one that failed
    bool valid = false;
    bool direct = false;   // the round's candidates do not fit: it walks the tree itself
};

// End of a range of m slabs that covers the round [tlag, whi].
__device__ __forceinline__ float range_end(int m, float tlag, float whi, float slab) {
    return m > 1 ? fmaxf(tlag + (float)(m + 1) * slab, whi) : whi;
}

// Ranks of the list's keys (W.slot), four per lane.
constexpr int kCandLane = kTileCand / kWave;
__device__ __forceinline__ void rank_keys(const TileLds& W, int cnt, int lane, unsigned int* key, int* rank) {
#pragma unroll
    for (int j = 0; j < kCandLane; ++j) {
        key[j] = kWave * j + lane < cnt ? (unsigned int)W.slot[kWave * j + lane] : 0xffffffffu;
        rank[j] = 0;
    }
#pragma unroll
    for (int jj = 0; jj < kCandLane; ++jj) {
        const int lim = min(kWave, cnt - kWave * jj);
        for (int i = 0; i < lim; ++i) {
            const unsigned int v = __builtin_amdgcn_readlane(key[jj], i);
#pragma unroll
            for (int j = 0; j < kCandLane; ++j)
                if (kWave * j < cnt) rank[j] += v < key[j] ? 1 : 0;
        }
    }
}

// Keeps the candidates with z0 <= s1 and key < limit; returns their number.
__device__ __forceinline__ int drop_candidates(TileLds& W, int cnt, float s1, unsigned int limit, int lane) {
    int n = 0;
#pragma unroll
    for (int j = 0; j < kCandLane; ++j) {
        const int i = kWave * j + lane;
        const unsigned int key = W.slot[i];
        const float z0 = W.z0[i], z1 = W.z1[i];
        const bool keep = i < cnt && !(z0 > s1) && key < limit;
        const unsigned long long mk = __builtin_amdgcn_ballot_w64(keep);
        const int at = n + mask_rank(mk);
        __syncthreads();
        if (keep) {
            W.slot[at] = key;
            W.z0[at] = z0;
            W.z1[at] = z1;
        }
        n += __popcll(mk);
        __syncthreads();
    }
    return n;
}

// Gathers the candidates of W's beam within [tlag, w.s1] (a range of w.m slabs) and the leaves
// from w.first on into W, sorted by slot, and sets w.cnt.  When they do not fit, the range is halved, down to the round
// [tlag, whi], and then with split, as often as the beam allows, the leaves to the lower half of those found
// (w.limit); what was found stays where it still belongs.  Returns false when they do not fit all the same.  64 nodes are taken
// at a time from the top of a stack, and the leaves among them are tested 64 at a time too: the test is
// most of a gather's arithmetic (230 of 300 instructions), and few of the 64 nodes are leaves.  Testing
// them as they came, starting again with half the range and walking the tree for each round whose
// candidates do not fit took 100 us a gather and 10 walks in the dearest tile of 300k Gaussians: forward
// 17.3 -> 15.9 ms there, 99.2 -> 87.9 ms at 1M, 2.22 -> 1.55 ms on one view of 100k.
// Called by all 64 lanes; wave-uniform result.
__device__ __forceinline__ bool beam_gather(const float4* __restrict__ nodes, const float4* __restrict__ geo, int total,
                                            TileWalk& w, float tlag, float whi, float slab, bool split, TileLds& W,
                                            int lane) {
    w.cnt = 0;
    w.limit = total;
    if (total <= 0) return true;
    const Beam& b = W.beam;
    const int n = (total + 1) >> 1;
    if (lane == 0) W.stack[0] = 0;
    int sp = 1, queue = 0;
    __syncthreads();
    if (w.first == 0) w.cuts = split ? b.cuts : 0;
    while (sp > 0 || queue > 0) {
        // the next nodes and, once there are 64, leaves; each of the p nodes puts at most two in its
        // place, and a nearly full stack is walked in depth
        const int take = queue >= kWave || sp == 0 ? min(queue, kWave) : 0;
        if (sp >= kTileStack) return false;
        const int p = min(min(sp, kWave), max(kTileStack - kTileReserve - sp, 1));
        queue -= take;
        sp -= p;
        const int node = lane < p ? W.stack[sp + p - 1 - lane] : total;
        const int tested = lane < take ? W.leaf[queue + lane] : total;
        const int slot = lane < take ? W.leaf_slot[queue + lane] : 0;
        __syncthreads();
        float4 lo = {}, hi = {}, g0 = {}, g1 = {}, g2 = {}, g3 = {};
        if ((unsigned)node < (unsigned)w.limit) {
            lo = nodes[2 * (int64_t)node];
            hi = nodes[2 * (int64_t)node + 1];
        }
        if (tested < w.limit) {
            const float4* g = geo + 4 * (int64_t)slot;
            g0 = g[0], g1 = g[1], g2 = g[2], g3 = g[3];
        }
        if (p > 0) {
            bool left = false, right = false, leaf = false;
            int child = 0;
            const int link = __float_as_int(hi.w);
            if ((unsigned)node < (unsigned)w.limit && beam_box(b, lo, hi, tlag, w.s1)) {
                if (link < 0) {
                    child = ~link;
                    const int end = __float_as_int(lo.w);
                    // links only lead forward: the walk ends
                    left = child > node && child > w.first;
                    right = child > node && child < w.limit && end > w.first;
                } else {
                    leaf = link < n && node >= w.first;
                }
            }
            const unsigned long long ml = __builtin_amdgcn_ballot_w64(left), mr = __builtin_amdgcn_ballot_w64(right),
                                     mq = __builtin_amdgcn_ballot_w64(leaf);
            if (right) W.stack[sp + mask_rank(mr)] = child;
            sp += __popcll(mr);
            if (left) W.stack[sp + mask_rank(ml)] = node + 1;
            sp += __popcll(ml);
            if (leaf) {
                const int at = queue + mask_rank(mq);
                W.leaf[at] = node;
                W.leaf_slot[at] = link;
            }
            queue += __popcll(mq);
        }
        if (take > 0) {
            bool odd = false;
            float z0 = 0.0f, z1 = 0.0f;
            bool keep = tested < w.limit && beam_ellipsoid(b, g0, g1, g2, g3, tlag, w.s1, z0, z1, odd);
            unsigned long long mk = __builtin_amdgcn_ballot_w64(keep);
            while (w.cnt + __popcll(mk) > kTileCand) {
                if (w.m > 1) {
                    w.m >>= 1;
                    w.s1 = range_end(w.m, tlag, whi, slab);
                } else if (w.cuts > 0) {
                    --w.cuts;
                    unsigned int key[kCandLane];
                    int rank[kCandLane];
                    rank_keys(W, w.cnt, lane, key, rank);
#pragma unroll
                    for (int j = 0; j < kCandLane; ++j) {
                        const unsigned long long mid = __builtin_amdgcn_ballot_w64(rank[j] == w.cnt / 2 && kWave * j + lane < w.cnt);
                        if (mid != 0ULL) w.limit = (unsigned int)__builtin_amdgcn_readlane(key[j], __builtin_ctzll(mid)) >> 1;
                    }
                } else {
                    return false;
                }
                w.cnt = drop_candidates(W, w.cnt, w.s1, 2u * w.limit, lane);
                keep = keep && !(z0 > w.s1) && tested < w.limit;
                mk = __builtin_amdgcn_ballot_w64(keep);
            }
            if (keep) {
                const int at = w.cnt + mask_rank(mk);
                W.slot[at] = (int)(2u * tested + (odd ? 1u : 0u));
                W.z0[at] = z0;
                W.z1[at] = z1;
            }
            w.cnt += __popcll(mk);
        }
        __syncthreads();
    }
    // by slot, whose order is that of the leaves' nodes
    unsigned int key[kCandLane];
    int rank[kCandLane];
    float a0[kCandLane], a1[kCandLane];
#pragma unroll
    for (int j = 0; j < kCandLane; ++j) {
        a0[j] = W.z0[kWave * j + lane];
        a1[j] = W.z1[kWave * j + lane];
    }
    rank_keys(W, w.cnt, lane, key, rank);
    __syncthreads();
#pragma unroll
    for (int j = 0; j < kCandLane; ++j)
        if (kWave * j + lane < w.cnt) {
            const int slot = __float_as_int(nodes[(int64_t)(key[j] | 1u)].w);
            const float4* g = geo + 4 * (int64_t)slot;
            W.slot[rank[j]] = 2 * slot + (int)(key[j] & 1u);
            W.z0[rank[j]] = a0[j];
            W.z1[rank[j]] = a1[j];
            W.oc[rank[j]] = origin_terms(b, g[0], g[1], g[2], g[3]);
        }
    __syncthreads();
    return true;
}

// A record or colour read at a wave-uniform index, as scalar loads.
__device__ __forceinline__ float4 ld_uniform(const float4* __restrict__ p, int64_t i) {
    const node_f32x4 v = ((const const_node_f32x4*)p)[i];
    return make_float4(v.x, v.y, v.z, v.w);
}

// The exact predicate and hit test of a listed candidate within [tmin, tmax] (0 <= tmin), for the lanes
// with cond; with the results of intersect and overlaps, and I as they leave it but for A and P,
// which refine_sampling sets.  The roots are formed with the native square root and reciprocal, each
// within one ulp, and thus within 1e-6 of themselves; where that could decide a comparison, they are
// formed again with the exact operations.  With O' and c from the list about 80 instructions instead of
// the 140 of intersect (2000 such evaluations per tile at 1M Gaussians: forward 119.7 -> 99.2 ms,
// together with the tighter beams).
__device__ __forceinline__ bool listed_hit(const float4 oc, const float4 g1, const float4 g2, const float4 g3, const Ray& r,
                                           float tmin, float tmax, bool cond, Isect& I) {
#pragma clang fp contract(off)
    const float Dp0 = (g1.x * r.dx + g1.y * r.dy) + g1.z * r.dz;
    const float Dp1 = (g2.x * r.dx + g2.y * r.dy) + g2.z * r.dz;
    const float Dp2 = (g3.x * r.dx + g3.y * r.dy) + g3.z * r.dz;
    const float ddp = (Dp0 * Dp0 + Dp1 * Dp1) + Dp2 * Dp2;
    const float l = inv_sqrt_exact<false>(ddp);
    const float Dh0 = Dp0 * l, Dh1 = Dp1 * l, Dh2 = Dp2 * l;
    const float b = -((oc.x * Dh0 + oc.y * Dh1) + oc.z * Dh2);
    const float P0 = oc.x + b * Dh0, P1 = oc.y + b * Dh1, P2 = oc.z + b * Dh2;
    const float pp = (P0 * P0 + P1 * P1) + P2 * P2;
    const float disc = 1.0f - pp;
    const bool in = cond && disc > 1e-7f;
    if (__builtin_amdgcn_ballot_w64(in) == 0ULL) return false;
    I.tc = b * l;
    I.Cq = g1.w * ddp;
    I.Dx = Dp0;
    I.Dy = Dp1;
    I.Dz = Dp2;
    I.l = l;
    const float sd = __builtin_amdgcn_sqrtf(disc);
    const float q = (b > 0.0f) ? b + sd : b - sd;
    I.r1 = (oc.w * __builtin_amdgcn_rcpf(q)) * l;
    I.r2 = q * l;
    const float lo = fmaxf(tmin, I.r1), hi = fminf(tmax, I.r2);
    const float margin = 2e-6f * (fabsf(lo) + fabsf(hi));
    const bool clear = fabsf(hi - lo) > margin && fabsf(I.r1 - tmin) > margin;
    if (__builtin_amdgcn_ballot_w64(in && !clear) != 0ULL) {
        const float sx = __builtin_sqrtf(disc);
        const float qx = (b > 0.0f) ? b + sx : b - sx;
        I.r1 = (oc.w / qx) * l;
        I.r2 = qx * l;
        return in && overlaps(tmin, tmax, I.r1, I.r2);
    }
    return in && lo <= hi;
}

}  // namespace rg
