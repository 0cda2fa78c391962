// Tile kernels: the forward and backward of wavefronts whose rays form narrow beams.
//
// A wavefront whose rays form a narrow beam (8x8 tiles of a view, subsets of them) marches as one:
// in each round the lanes near the laggard (tile_window) process one slab each, and the
// candidates whose depth range meets the round's come from one list for all lanes (beam_gather),
// taken in slot order.  A candidate's record is read once for the wavefront, through scalar loads,
// and every lane applies the exact predicate to it; the slabs a ray processes, the hits it sums in
// each and their order are those of the per-ray slab stepper (trace.hip).

#include <hip/hip_runtime.h>

#include <climits>

#include "rg_device.h"
#include "rg_internal.h"
#include "rg_tile.h"
#include "rg_trace.h"

namespace rg {
namespace {

constexpr int kMaxSeg = 4096;

constexpr float kTileSync = 0.75f;  // lanes within this many slabs of the laggard step together
// A wavefront's rays make up at most kTileGroups beams, each of one view and within the spread
// (per direction component, from its first ray; 8x8 pixels of a 1000-pixel, 40-degree view are 0.006)
// kTileSpread and sqrt(kTileDensity / n); other wavefronts go to the slab stepper.  A beam's
// candidates grow with the Gaussians and with the square of its width, its rays' own hits do not.
// Measured on 64 random rays of a block of S pixels out of 1024 (train step, every wavefront's rays in the
// stepper / as tiles with bounds 0.2 and 3000): 1M Gaussians S = 32 102 / 45 ms, 64 177 / 151, 128 (spread 0.09)
// 283 / 242, 256 (up to four beams) 323 / 380; 300k S = 128 115 / 43, 256 130 / 51; 20k 256 10.4 / 7.6, 1024
// 7.0 / 19.6; with the bounds below 45, 151, 246, 361; 43, 82; 10.9, 4.1.  Several beams: a list of 8x8 tiles
// with ragged edges has wavefronts that hold the end of one row of tiles and the start of the next (one beam each; in
// the stepper the 1 % of such wavefronts took 10 of 290 ms at 1M Gaussians).
constexpr float kTileSpread = 0.1f, kTileDensity = 2000.0f;
constexpr int kTileGroups = 4;
// Where more than one in kHalfShare of a job's wavefronts (of kSampled looked at) are no beams, only those of
// half these widths march as tiles: the others are beams by chance, each as dear as the widest allowed, and
// the launch lasts as long as they do before the stepper begins.  Rays as above, up to four beams a wavefront,
// train step of 4096 wavefronts (all in the stepper / all beams as tiles / this rule): 300k S = 256 154 / 205 /
// 125 ms, 100k 256 62.9 / 39.0 / 38.4, 100k 512 45.1 / 69.4 / 44.2, 20k larger Gaussians 256 32.9 / 35.9 / 35.5,
// 512 43.7 / 76.0 / 41.5; of 1024 wavefronts 1M 256 321 / 350 / 135.
constexpr int kSampled = 1024, kHalfShare = 8;
// Rounds that are walked after gathers that failed, before the next gather, at most (1, 3, 7, ...): in a dense
// stretch the next round's candidates do not fit either.  300k S = 128, 4096 wavefronts 92.7 -> 86.5 ms, 100k S = 256
// 45.9 -> 39.0.
constexpr int kMaxSkip = 15;

// Whether the job's wavefronts are held to beams of half the widths (k_tile_sample).
__device__ __forceinline__ bool half_beams(const DevParams& p) {
    return p.sample_wide && *p.sample_wide > (unsigned long long)p.sample_limit;
}

// Assigns the lanes with act to beams (group 0 .. kTileGroups - 1); false when they make up more.
__device__ __forceinline__ bool tile_groups(const DevScene& sc, bool half, bool act, int view, const Ray& r, int& group) {
    float limit = fminf(kTileSpread, __builtin_sqrtf(kTileDensity / (float)sc.n));
    if (half) limit *= 0.5f;
    group = -1;
    unsigned long long rem = __ballot(act);
    for (int k = 0; k < kTileGroups && rem != 0ULL; ++k) {
        const int f = __ffsll((long long)rem) - 1;
        const float x = fabsf(r.dx - __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(r.dx), f)));
        const float y = fabsf(r.dy - __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(r.dy), f)));
        const float z = fabsf(r.dz - __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(r.dz), f)));
        const bool in = ((rem >> threadIdx.x) & 1ULL) != 0ULL && view == __builtin_amdgcn_readlane(view, f);
        const bool mine = in && x <= limit && y <= limit && z <= limit;
        if (mine) group = k;
        const unsigned long long m = __ballot(mine);
        if (m == 0ULL) return false;  // a NaN direction
        rem &= ~m;
    }
    return rem == 0ULL;
}

// Makes the list cover the round [tlag, whi]: all of it, or with split at least its first leaves.  The
// range's length doubles while the list is mostly empty and halves while it is nearly full.
__device__ __forceinline__ void tile_list(TileWalk& w, const DevScene& sc, float tlag, float whi, float slab, bool split,
                                          TileLds& W, int lane, bool alive, Counters& ctr) {
    if (w.valid && !(whi > w.s1)) return;
    if (w.valid && 4 * w.cnt < kTileCand) w.m = min(w.m * 2, kMaxSeg);
    else if (w.valid && 4 * w.cnt > 3 * kTileCand) w.m = max(w.m >> 1, 1);
    w.valid = true;
    if (w.skip > 0) {
        --w.skip;
        w.direct = true;
        w.cnt = 0;
        return;
    }
    w.s1 = range_end(w.m, tlag, whi, slab);
    w.direct = !beam_gather(sc.nodes, sc.geo, sc.total_nodes, w, tlag, whi, slab, split, W, lane);
    if (w.direct) w.cnt = 0;
    w.back = w.direct ? min(2 * w.back + 1, kMaxSkip) : 0;
    w.skip = w.back;
    if (alive) ctr.gathers++;
}

// Whether a lane at depth tb takes part in the round whose laggard is at tlag <= tb; the laggard always does
// (at depths where a slab is less than an ulp of t, tlag + kTileSync * slab may round to tlag).
__device__ __forceinline__ bool in_round(float tb, float tlag, float slab) { return tb - tlag < kTileSync * slab; }

// The lanes of the next round: its depths [tlag, whi] and whether this lane takes part.
__device__ __forceinline__ bool tile_window(bool alive, float tb, float slab, float& tlag, float& whi) {
    // depths are not negative: their order is that of their bits
    const int bits = __float_as_int(tb);
    tlag = __int_as_float(__builtin_amdgcn_readfirstlane(wave_min64(alive ? bits : 0x7f800000)));
    const bool part = alive && in_round(tb, tlag, slab);
    whi = add_exact(__int_as_float(__builtin_amdgcn_readfirstlane(~wave_min64(part ? ~bits : INT_MAX))), slab);
    return part;
}

// Chunk j of the list: this lane's entry of W.slot and the lanes whose candidate meets [wlo, whi].
__device__ __forceinline__ unsigned long long tile_chunk(const TileLds& W, int cnt, int j, int lane, float wlo, float whi,
                                                         int& slot) {
    const int i = 64 * j + lane;
    const bool in = i < cnt;
    slot = in ? W.slot[i] : 0;
    return __builtin_amdgcn_ballot_w64(in && !(W.z0[i] > whi) && !(W.z1[i] < wlo));
}

// After a round without candidates: every lane steps over the slabs that end before the next
// candidate's depths (or the end of the list).
__device__ __forceinline__ void tile_jump(const TileWalk& w, const TileLds& W, int lane, float whi, float slab, bool alive,
                                          const Ray& ray, float& tb) {
    float next = w.s1;
    for (int i = lane; i < w.cnt; i += kWave)
        if (W.z0[i] > whi) next = fminf(next, W.z0[i]);
    next = uniform_f(wave_min64f(next));
    while (alive) {
        const float nt = add_exact(tb, slab);
        if (!(tb < ray.texit) || !(fminf(ray.texit, nt) < next) || !(nt > tb)) break;
        tb = nt;
    }
}

// Record of a tile: 16-byte cells in the space of its rays' hit-list records.  Per round with hits a
// header (depth of the laggard, number of events, view, beam) followed by its events (slot, lanes that
// hit it: low word, high word, 0).  A lane's slab of a round is the first at or beyond the header's
// depth.  One lane stores each cell: eight share a cache line, which leaves L2 once.
struct TileRec {
    u32x4* cells = nullptr;
    int pos = 0, cap = 0;  // cells of whole rounds written, cells there are
    bool full = false;     // a round did not fit: nothing is recorded from it on
    int n = 0;             // events of the current round
};

__device__ __forceinline__ void tile_rec_event(TileRec& r, int slot, unsigned long long hits, int lane) {
    ++r.n;
    if (r.pos + r.n >= r.cap) r.full = true;
    if (lane == 0 && !r.full)
        r.cells[r.pos + r.n] = u32x4{(unsigned int)slot, (unsigned int)hits, (unsigned int)(hits >> 32), 0u};
}

__device__ __forceinline__ void tile_rec_round(TileRec& r, float tlag, int view, int group, int lane) {
    if (r.n > 0 && !r.full) {
        if (lane == 0) 
            r.cells[r.pos] = u32x4{__float_as_uint(tlag), (unsigned int)r.n, (unsigned int)view, (unsigned int)group};
        r.pos += 1 + r.n;
    }
    r.n = 0;
}

// Spread wavefronts: at most eight rays, each in eight lanes, one sample of the slab per lane (lane = 8 ray +
// sample).  An event then takes the arithmetic of one sample instead of eight, and a lane sums its sample over
// the events in their order, as elsewhere.  They are the wavefronts of small jobs and the parts of split
// ones: fewer than the GPU holds, and each nearly alone on its SIMD, where the length of its chain of
// instructions is its time.  One 64x64 view of 4096 Gaussians: forward 158 -> 137 us, backward 185 -> 150;
// 30k Gaussians with random samples (parts of 32-ray wavefronts) 384 -> 362 and 465 -> 399.

// Depth of the lane's sample.
template <bool RNG>
__device__ __forceinline__ float spread_t(float tb, int i, unsigned int seed, const DevParams& p) {
    unsigned int st = seed;
    if (!RNG || p.rnd_sample != 1) return sample_t(tb, i, p.dt, RNG ? p.rnd_sample : 0, st);
    float t = 0.0f;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        const float tk = sample_t(tb, k, p.dt, p.rnd_sample, st);
        t = k == i ? tk : t;
    }
    return t;
}

// Density of a hit at the lane's sample, zero at or below thr.
__device__ __forceinline__ float spread_density(const Isect& I, float sigma, float t, float thr) {
    const float sw = sigma * weight(wexp(I), t - I.tc);
    return sw > thr ? sw : 0.0f;
}

// composite over the eight lanes of a ray: T, which all have, and in each lane one of the colours' or the
// depth's sums (lane & 3), in the order of the samples.
__device__ __forceinline__ void spread_composite(float sig, float cr, float cg, float cb, float t, const DevParams& p,
                                                 SpreadLds& X, int lane, float& T, float& sum) {
    const float alpha = sample_alpha(sig, p.dt);
    const float inv = __builtin_amdgcn_rcpf(fmaxf(sig, 0x1p-126f));
    X.alpha[lane] = alpha;
    X.rest[lane] = 1.0f - alpha;
    X.v[0][lane] = cr * inv;
    X.v[1][lane] = cg * inv;
    X.v[2][lane] = cb * inv;
    X.v[3][lane] = t;
    __builtin_amdgcn_wave_barrier();
    const int first = lane & 56, c = lane & 3;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        const float ta = T * X.alpha[first + j];
        sum += ta * X.v[c][first + j];
        T *= X.rest[first + j];
    }
    __builtin_amdgcn_wave_barrier();
}

// slab_coeffs for the lane's sample: overwrites (sig, ep) with its (G, Bq).
__device__ __forceinline__ void spread_coeffs(float& sig, float& ep, const DevParams& p, SpreadLds& X, int lane, float& T,
                                              float& Dr) {
    const float alpha = sample_alpha(sig, p.dt);
    const float inv = sig > 0.0f ? __builtin_amdgcn_rcpf(sig) : 0.0f;
    const float E = ep * inv;
    X.alpha[lane] = alpha;
    X.rest[lane] = 1.0f - alpha;
    X.v[0][lane] = E;
    __builtin_amdgcn_wave_barrier();
    const int first = lane & 56;
    float Ti = T, Di = Dr;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        Ti = (lane & 7) == j ? T : Ti;
        Di = (lane & 7) == j ? Dr : Di;
        Dr -= T * X.alpha[first + j] * X.v[0][first + j];
        T *= X.rest[first + j];
    }
    __builtin_amdgcn_wave_barrier();
    const float Bq = Ti * alpha * inv;
    sig = p.dt * (Ti * E - Di) - Bq * E;
    ep = Bq;
}

// Forward of the lanes with act, which share their view, as one beam.  Called by all 64 lanes.
template <int SPB, bool RNG, int RM, bool SPREAD>
__device__ __forceinline__ void forward_tile(const DevScene& sc, const DevParams& p, bool act, const Ray& ray,
                                             unsigned int& seed, int view, const float* cam_u, int group, int hit_depth,
                                             bool want_depth, TileLds& W, int lane,
                                             Counters& ctr, RayOut& o, TileRec& rc) {
    const float slab = p.dt * (float)p.spb;
    const float4* __restrict__ rgbv = sc.rgb + (size_t)view * sc.n;
    make_beam(act, ray, cam_u, W, lane);
    TileWalk w;
    w.m = p.seg_slabs;
    bool alive = act && o.T > p.t_eps;
    float tb = ray.tenter;
    // sums of a round that goes on with another list, in memory: few do, and the registers are the gather's
    constexpr int NS = SPREAD ? 1 : SPB;  // samples of a lane
    float held_sums[4 * NS];
    __attribute__((address_space(5))) volatile float* held = (__attribute__((address_space(5))) volatile float*)held_sums;
    int nh = 0;
    bool any = false;  // the round has candidates
    while (__ballot(alive) != 0ULL) {
        float tlag, whi;
        const bool part = tile_window(alive, tb, slab, tlag, whi);
        tile_list(w, sc, tlag, whi, slab, true, W, lane, alive, ctr);
        const float tmin = fmaxf(ray.tenter, tb), tmax = fminf(ray.texit, add_exact(tb, slab));
        float sig[NS], cr[NS], cg[NS], cb[NS];
#pragma unroll
        for (int i = 0; i < NS; ++i) sig[i] = cr[i] = cg[i] = cb[i] = 0.0f;
        if (w.first > 0) {
#pragma unroll
            for (int i = 0; i < NS; ++i) {
                sig[i] = held[4 * i];
                cr[i] = held[4 * i + 1];
                cg[i] = held[4 * i + 2];
                cb[i] = held[4 * i + 3];
            }
        } else {
            nh = 0;
            any = false;
        }
        const float ts = SPREAD ? spread_t<RNG>(tb, lane & 7, seed, p) : 0.0f;
        // at: the candidate's place in the list, or -1
        auto eval = [&](int slot, int at, bool cond) {
            const float4 g0 = ld_uniform(sc.geo, 4 * (int64_t)slot), g1 = ld_uniform(sc.geo, 4 * (int64_t)slot + 1),
                         g2 = ld_uniform(sc.geo, 4 * (int64_t)slot + 2), g3 = ld_uniform(sc.geo, 4 * (int64_t)slot + 3);
            Isect I;
            bool hit;
            if (at >= 0) hit = listed_hit(W.oc[at], g1, g2, g3, ray, tmin, tmax, cond, I);
            else hit = cond && intersect(g0, g1, g2, g3, ray, I) && overlaps(tmin, tmax, I.r1, I.r2);
            const unsigned long long hits = __builtin_amdgcn_ballot_w64(hit);
            if (hits == 0ULL) return;
            if constexpr (RM == 1) {
                if (!rc.full) tile_rec_event(rc, slot, hits, lane);
            }
            if (hit) {
                refine_sampling(g0, g1, g2, g3, ray, I);
                if constexpr (SPREAD) {
                    const float4 col = ld_uniform(rgbv, slot);
                    const float m = spread_density(I, g0.w, ts, p.sigma_thr);
                    sig[0] += m;
                    cr[0] += m * col.x;
                    cg[0] += m * col.y;
                    cb[0] += m * col.z;
                } else {
                    accum_hit<SPB, RNG>(I, g0.w, ld_uniform(rgbv, slot), tb, seed, p, sig, cr, cg, cb);
                }
                if (tb == ray.tenter || I.r1 > tmin) ctr.P++;
                ++nh;
            }
        };
        any |= w.direct;
        for (int j = 0; kWave * j < w.cnt; ++j) {
            int sl;
            unsigned long long m = tile_chunk(W, w.cnt, j, lane, tlag, whi, sl);
            any |= m != 0ULL;
            while (m != 0ULL) {
                const int i = __builtin_ctzll(m);
                const int code = __builtin_amdgcn_readlane(sl, i);
                m &= m - 1ULL;
                eval(code >> 1, (code & 1) ? -1 : kWave * j + i, part);
            }
        }
        if (w.direct) {
            const float ix = 1.0f / ray.dx, iy = 1.0f / ray.dy, iz = 1.0f / ray.dz;
            for (int idx = w.first; idx < sc.total_nodes;) {
                idx = __builtin_amdgcn_readfirstlane(idx);
                const float4 lo = ld_node(sc.nodes, 2 * idx), hi = ld_node(sc.nodes, 2 * idx + 1);
                const int miss = __float_as_int(lo.w), leaf = __float_as_int(hi.w);
                if (miss <= idx || leaf >= sc.n) break;  // malformed link: never loop
                const bool h = part && box_hit(lo, hi, ray, ix, iy, iz, tmin, tmax);
                const bool met = __ballot(h) != 0ULL;
                if (met && leaf >= 0) eval(leaf, -1, h);
                idx = met && leaf < 0 ? idx + 1 : miss;
            }
            w.valid = false;
        } else if (w.limit < sc.total_nodes) {  // the round goes on with its other leaves
#pragma unroll
            for (int i = 0; i < NS; ++i) {
                held[4 * i] = sig[i];
                held[4 * i + 1] = cr[i];
                held[4 * i + 2] = cg[i];
                held[4 * i + 3] = cb[i];
            }
            w.first = w.limit;
            w.valid = false;
            continue;
        }
        if (w.first > 0) {
            w.first = 0;
            w.valid = false;
        }
        if constexpr (RM == 1) {
            if (!rc.full) tile_rec_round(rc, tlag, view, group, lane);
        }
        if (part) {
            if (nh > 0) {
                ctr.K += nh;
                if (p.max_hits > 0 && nh > p.max_hits) ctr.ovf++;
                if (nh > hit_depth) ctr.fallback++;
                if constexpr (SPREAD) spread_composite(sig[0], cr[0], cg[0], cb[0], ts, p, W.spread, lane, o.T, o.C[0]);
                else composite<SPB, RNG>(sig, cr, cg, cb, tb, seed, p, want_depth, o);
                if (RNG && p.rnd_sample == 1) seed = skip_draws(seed, p.spb);  // the slab's draws are spent
            }
            const float nt = add_exact(tb, slab);
            alive = nt > tb && nt < ray.texit && o.T > p.t_eps;
            tb = nt;
        }
        if (!any && p.fwd_jump) {
            tile_jump(w, W, lane, whi, slab, alive, ray, tb);
            alive = alive && tb < ray.texit;
        }
    }
}

// The events of a round whose sample densities the first pass leaves in LDS for the second, which then
// needs neither the predicate's terms nor the weights again: the arithmetic of an event is what
// bounds the backward (about 250 vector instructions in the first pass and 340 in the second, 1220
// events per tile at 1M Gaussians).  Four of them with the staging area are the LDS that three
// wavefronts per SIMD leave to each (160 KB / 12); most rounds have no more.  Measured on a training
// pass: 165 -> 146 ms at 1M Gaussians (8 views of 1237x822), 23.2 -> 21.5 ms at 300k, 231 -> 191 us at
// 4096 with one 64x64 view.
constexpr int kKept = 4;
struct KeptEvents {
    float4 m[kKept][2][kWave];  // thresholded density sigma w of the 8 samples
    float4 ptc[kKept][kWave];   // the offset P and t_c
};

// The same of a spread wavefront, behind the exchange area, which lies where a walked tile's does.
constexpr int kKeptSpread = 8;
struct KeptSpread {
    SpreadLds X;
    float m[kKeptSpread][kWave];
    float4 ptc[kKeptSpread][kWave];
};

// A walked tile holds its candidates, a replayed one its round's kept events.
union BwdLds {
    TileLds W;
    KeptEvents K;
    KeptSpread S;
};
static_assert(sizeof(KeptSpread) <= sizeof(KeptEvents) && sizeof(TileLds) <= sizeof(KeptEvents), "LDS of a backward");

// Backward of the lanes with act, called by all 64 lanes.  In each round the wavefront has a list
// of events -- a Gaussian and the lanes that hit it in their slab of the round -- which it goes
// through twice: to recompute the slabs' sample buffers and from them the per-sample coefficients,
// and to sum each Gaussian's gradient moments over its lanes.  The events come from the forward's
// record of the tile (cells; lanes take part with their beam in it, tile, -1: none), and for the lanes with
// walk, once it ends, from the tile's own gathers.
template <int SPB, bool RNG, bool SPREAD>
__device__ __forceinline__ void backward_tile(const DevScene& sc, const DevParams& p, const rg_camera* cams, bool act, const Ray& ray,
                                              unsigned int seed, int view, const float* Cfwd, const float* dL,
                                              const u32x4* __restrict__ cells, int num_cells, int tile, bool walk,
                                              BwdLds& S, GradStage& G, int lane, const DevGrad& gr, Counters& ctr,
                                              unsigned long long* drops) {
    const float slab = p.dt * (float)p.spb;
    TileLds& W = S.W;
    Staged staged;
    bool alive = act && (ray.tenter < ray.texit) && (add_exact(ray.tenter, slab) > ray.tenter) && 1.0f > p.t_eps;
    float T = 1.0f;
    float Dr = dL[0] * Cfwd[0] + dL[1] * Cfwd[1] + dL[2] * Cfwd[2];  // dLdC . (colour not yet composited)
    float tb = ray.tenter;
    // events of the current batch, one per lane (in the record's case a window of its cells)
    int ev_slot = 0, ev_lo = 0, ev_hi = 0, ev_beam = 0;
    int wbase = -kWave;  // first cell of the window
    auto window = [&](int first) {
        wbase = first;
        const int i = first + lane;
        u32x4 c = {0u, 0u, 0u, 0u};
        if (i < num_cells) c = __builtin_nontemporal_load(cells + i);
        ev_slot = (int)c.x;
        ev_lo = (int)c.y;
        ev_hi = (int)c.z;
        ev_beam = (int)c.w;
    };
    int pos = 0;
    unsigned long long todo = 0ULL;  // lanes of the beam being walked
    int gview = 0, group = -1;
    TileWalk w;
    while (true) {
        const bool replay = pos < num_cells;
        float tlag = 0.0f, whi = 0.0f;
        int total = 0, first = 0;  // events of the round (replay), lane of the first one
        bool part;
        if (replay) {
            if (pos - wbase >= kWave) window(pos);
            first = pos - wbase;
            total = __builtin_amdgcn_readlane(ev_lo, first);
            if (first + 1 + total > kWave && first > 0) {
                window(pos);
                first = 0;
            }
            tlag = __uint_as_float((unsigned int)__builtin_amdgcn_readlane(ev_slot, first));
            gview = __builtin_amdgcn_readlane(ev_hi, first);
            const bool mine = tile == __builtin_amdgcn_readlane(ev_beam, first);
            ++first;
            if (total <= 0 || total >= num_cells - pos) {  // never expected: end of the record
                pos = num_cells;
                continue;
            }
            while (alive && mine && tb < tlag) {
                const float nt = add_exact(tb, slab);
                if (!(nt > tb) || !(nt < ray.texit)) alive = false;
                else tb = nt;
            }
            part = alive && mine && in_round(tb, tlag, slab);
        } else {
            if ((__ballot(alive && walk) & todo) == 0ULL) {  // the next beam
                if (group < 0) {
                    int g = 0;
                    if (!tile_groups(sc, half_beams(p), alive && walk, view, ray, g)) g = view;  // (left to this kernel: one view)
                    group = alive && walk ? g : INT_MAX;
                }
                const unsigned long long rem = __ballot(alive && walk);
                if (rem == 0ULL) break;
                const int f = __ffsll((long long)rem) - 1;
                gview = __builtin_amdgcn_readlane(view, f);
                todo = __ballot(alive && walk && group == __builtin_amdgcn_readlane(group, f));
                make_beam(((todo >> lane) & 1ULL) != 0ULL, ray, cams[gview].u, W, lane);
                w = TileWalk();
                w.m = p.seg_slabs;
            }
            const bool mine = alive && ((todo >> lane) & 1ULL) != 0ULL;
            part = tile_window(mine, tb, slab, tlag, whi);
            tile_list(w, sc, tlag, whi, slab, false, W, lane, mine, ctr);
        }
        const float4* __restrict__ rgbv = sc.rgb + (size_t)gview * sc.n;
        const int key_base = gview * sc.n;
        const float tmin = fmaxf(ray.tenter, tb), tmax = fminf(ray.texit, add_exact(tb, slab));
        const unsigned int cur_seed = seed;
        // the density sums and the projected colour sums, then the coefficients G_i, Bq_i
        constexpr int NS = SPREAD ? 1 : SPB;  // samples of a lane
        float sig[NS], ep[NS];
#pragma unroll
        for (int i = 0; i < NS; ++i) sig[i] = ep[i] = 0.0f;
        const float ts = SPREAD ? spread_t<RNG>(tb, lane & 7, seed, p) : 0.0f;
        int nh = 0;
        bool any = false, one = false;  // the round has candidates; its events fit one batch
        int ne = 0;
        // goes through the round's events in order: fn(number in the round, slot, lane hit it)
        auto each_event = [&](bool again, auto&& fn) {
            // the enumeration of a walked round, resumed batch by batch
            int j = -1, sl = 0, idx = 0;
            unsigned long long m = 0ULL;
            for (int done = 0;;) {
                bool last;
                if (replay) {
                    if (done > 0 || (again && total >= kWave)) {  // a long round's later batches
                        window(pos + 1 + done);
                        first = 0;
                    }
                    ne = min(total - done, kWave - first);
                    last = done + ne >= total;
                } else if (again && one) {
                    last = true;
                } else {
                    ne = 0;
                    last = false;
                    while (ne < kWave) {
                        int slot;
                        bool cond = part;
                        if (w.direct) {
                            if (idx >= sc.total_nodes) {
                                last = true;
                                break;
                            }
                            idx = __builtin_amdgcn_readfirstlane(idx);
                            const float4 lo = ld_node(sc.nodes, 2 * idx), hi = ld_node(sc.nodes, 2 * idx + 1);
                            const int miss = __float_as_int(lo.w);
                            slot = __float_as_int(hi.w);
                            if (miss <= idx || slot >= sc.n) {  // malformed link: never loop
                                last = true;
                                break;
                            }
                            cond = part && box_hit(lo, hi, ray, 1.0f / ray.dx, 1.0f / ray.dy, 1.0f / ray.dz, tmin, tmax);
                            const bool met = __ballot(cond) != 0ULL;
                            idx = met && slot < 0 ? idx + 1 : miss;
                            if (!met || slot < 0) continue;
                            any = true;
                        } else {
                            if (m == 0ULL) {
                                if (kWave * (++j) >= w.cnt) {
                                    last = true;
                                    break;
                                }
                                m = tile_chunk(W, w.cnt, j, lane, tlag, whi, sl);
                                any |= m != 0ULL;
                                continue;
                            }
                            slot = __builtin_amdgcn_readlane(sl, __builtin_ctzll(m)) >> 1;
                            m &= m - 1ULL;
                        }
                        const float4 g0 = ld_uniform(sc.geo, 4 * (int64_t)slot), g1 = ld_uniform(sc.geo, 4 * (int64_t)slot + 1),
                                     g2 = ld_uniform(sc.geo, 4 * (int64_t)slot + 2),
                                     g3 = ld_uniform(sc.geo, 4 * (int64_t)slot + 3);
                        Isect I;
                        const bool hit = cond && intersect(g0, g1, g2, g3, ray, I) && overlaps(tmin, tmax, I.r1, I.r2);
                        const unsigned long long hits = __ballot(hit);
                        if (hits == 0ULL) continue;
                        const bool at = lane == ne;
                        ev_slot = at ? slot : ev_slot;
                        ev_lo = at ? (int)(unsigned int)hits : ev_lo;
                        ev_hi = at ? (int)(unsigned int)(hits >> 32) : ev_hi;
                        ++ne;
                    }
                    first = 0;
                    if (!again && done == 0) one = last;
                }
                for (int e = first; e < first + ne; ++e) {
                    const int slot = __builtin_amdgcn_readlane(ev_slot, e);
                    const unsigned long long hits =
                        (unsigned long long)(unsigned int)__builtin_amdgcn_readlane(ev_lo, e) |
                        (unsigned long long)(unsigned int)__builtin_amdgcn_readlane(ev_hi, e) << 32;
                    const bool in = part && ((hits >> lane) & 1ULL) != 0ULL;
                    if (__builtin_amdgcn_ballot_w64(in) == 0ULL) continue;
                    if ((unsigned)slot >= (unsigned)sc.n) {
                        if (lane == 0 && !again) count_drop(drops);
                        continue;
                    }
                    fn(done + e - first, slot, in);
                }
                done += ne;
                if (last) break;
            }
        };
        // densities of a hit: it passed the exact test, so only its sampling terms are computed
        auto densities = [&](const float4 g0, const float4 g1, const float4 g2, const float4 g3, float* md) -> float4 {
            Isect I;
            float bq, cq;
            isect_terms(g0, g1, g2, g3, ray, I, bq, cq);
            refine_sampling(g0, g1, g2, g3, ray, I);
            if constexpr (SPREAD) md[0] = spread_density(I, g0.w, ts, p.sigma_thr);
            else sample_densities<SPB, RNG>(I, g0.w, tb, cur_seed, p, md);
            return make_float4(I.Px, I.Py, I.Pz, I.tc);
        };
        each_event(false, [&](int number, int slot, bool in) {
            const float4 g0 = ld_uniform(sc.geo, 4 * (int64_t)slot), g1 = ld_uniform(sc.geo, 4 * (int64_t)slot + 1),
                         g2 = ld_uniform(sc.geo, 4 * (int64_t)slot + 2), g3 = ld_uniform(sc.geo, 4 * (int64_t)slot + 3);
            const float4 col = ld_uniform(rgbv, slot);
            if (!in) return;
            float md[NS];
            const float4 ptc = densities(g0, g1, g2, g3, md);
            if constexpr (SPREAD) {
                sig[0] += md[0];
                ep[0] += md[0] * project_color(dL, col);
                if (replay && number < kKeptSpread) {
                    S.S.m[number][lane] = md[0];
                    S.S.ptc[number][lane] = ptc;
                }
            } else {
                accum_densities<SPB>(md, project_color(dL, col), p, sig, ep);
            }
            if constexpr (SPB == 8 && !SPREAD) {
                if (replay && number < kKept) {
                    S.K.m[number][0][lane] = make_float4(md[0], md[1], md[2], md[3]);
                    S.K.m[number][1][lane] = make_float4(md[4], md[5], md[6], md[7]);
                    S.K.ptc[number][lane] = ptc;
                }
            }
            ++nh;
        });
        if (nh > 0) {
            if constexpr (SPREAD) spread_coeffs(sig[0], ep[0], p, W.spread, lane, T, Dr);
            else slab_coeffs<SPB>(sig, ep, p, T, Dr);
            if (RNG && p.rnd_sample == 1) seed = skip_draws(seed, p.spb);  // the slab's draws are spent
        }
        if (__builtin_amdgcn_ballot_w64(nh > 0) != 0ULL) {
            each_event(true, [&](int number, int slot, bool in) {
                const float4 g0 = ld_uniform(sc.geo, 4 * (int64_t)slot), g1 = ld_uniform(sc.geo, 4 * (int64_t)slot + 1),
                             g2 = ld_uniform(sc.geo, 4 * (int64_t)slot + 2), g3 = ld_uniform(sc.geo, 4 * (int64_t)slot + 3);
                const float4 col = ld_uniform(rgbv, slot);
                float v[kMoments];
#pragma unroll
                for (int k = 0; k < kMoments; ++k) v[k] = 0.0f;
                if (in) {
                    float md[NS];
                    float4 ptc;
                    if (SPB == 8 && replay && number < (SPREAD ? kKeptSpread : kKept)) {
                        if constexpr (SPREAD) {
                            md[0] = S.S.m[number][lane];
                            ptc = S.S.ptc[number][lane];
                        } else if constexpr (SPB == 8) {
                            const float4 a = S.K.m[number][0][lane], b = S.K.m[number][1][lane];
                            md[0] = a.x, md[1] = a.y, md[2] = a.z, md[3] = a.w;
                            md[4] = b.x, md[5] = b.y, md[6] = b.z, md[7] = b.w;
                            ptc = S.K.ptc[number][lane];
                        }
                    } else {
                        ptc = densities(g0, g1, g2, g3, md);
                    }
                    const float P[3] = {ptc.x, ptc.y, ptc.z};
                    float D[3];
                    ray_in_ellipsoid(g1, g2, g3, ray, D);
                    if constexpr (SPREAD) {
                        const float tau = ts - ptc.w;
                        const float wp = md[0] * (sig[0] + ep[0] * project_color(dL, col));
                        ray_moments(P, D, g0.w, wp, wp * tau, wp * (tau * tau), md[0] * ep[0], dL, v);
                    } else {
                        grad_moments<SPB, RNG>(P, D, g0.w, md, ptc.w, project_color(dL, col), tb, cur_seed, p, sig, ep, dL, v);
                    }
                }
                grad_scatter_wave(v, key_base + slot, sc, gr, lane, G, staged, drops);
            });
        }
        if (replay) pos += 1 + total;
        if (part) {
            const float nt = add_exact(tb, slab);
            alive = nt > tb && nt < ray.texit && T > p.t_eps;
            tb = nt;
        }
        if (!replay) {
            if (w.direct) w.valid = false;
            else if (!any) {
                const bool mine = alive && ((todo >> lane) & 1ULL) != 0ULL;
                tile_jump(w, W, lane, whi, slab, mine, ray, tb);
                alive = alive && tb < ray.texit;
            }
        }
    }
    stage_flush(G, staged, sc, gr, lane, drops);
}

// ------------------------------------------------------------------ order --------------------
//
// The wavefronts of a job cost from a few to hundreds of times their mean (a blob's core against its
// rim), and a launch lasts as long as its dearest ones, which sit next to each other in the image:
// on one view of 100k Gaussians the 10000 wavefronts of a forward took 530 us on average and the
// last of them 6 ms, 5.65 ms for what 4096 resident wavefronts could do in 1.3.  So the dear ones
// start first.  What a wavefront costs is estimated in the forward from the Gaussians' means around
// its pixels, counted on a coarse grid of each view, and known in the backward from its record.
constexpr int kGrid = 128;              // cells of a view along each axis
constexpr int kSplats = 1 << 20;        // Gaussians counted at most (every k-th of more)
constexpr int kOrderBuckets = 32;       // half octaves of the weight
constexpr int kOrderBlock = 1024;
// A wavefront that costs more than an even share of the launch ends after the others however early it
// starts, so it is split into quarters of its rays (narrower beams: each takes about half its time; in
// eighths, spread ones, the parts of 64 rays cost more together than they shorten: 1.10 ms instead of 0.99).  A
// backward takes the forward's parts with its records.  The weights exaggerate: with shares 0.5 / 1 / 2 / 4 / none
// (times an even one) a forward of one view of 100k Gaussians in blobs took 0.99 / 1.02 / 0.99 / 1.30 /
// 1.55 ms, its backward 1.18 / 1.19 / 1.10 / 1.28 / 1.54, one at four times the slabs 1.61 / 1.72 / 1.83 / 2.72 / 3.26,
// and an unbounded view of 1M, whose wavefronts are even, 12.5 / 10.7 / 9.98 / 10.0 / 10.0.  Ray lists, which
// may have wavefronts that are no beams, are not split.
constexpr float kSplitShare = 2.0f;
constexpr int kSplitPart = 8;
// Rays of a part of a split wavefront: a quarter, but no fewer than a spread one holds.
__host__ __device__ inline int split_rays(const DevParams& p) { return max(p.rays_per_wave / 4, min(p.rays_per_wave, 8)); }


__global__ void __launch_bounds__(256) k_tile_splat(int n, int stride, const float4* __restrict__ geo,
                                                    const rg_camera* __restrict__ cams, int first_view,
                                                    unsigned int* __restrict__ grid) {
    const int64_t i = ((int64_t)blockIdx.x * 256 + threadIdx.x) * stride;
    if (i >= n) return;
    const rg_camera& c = cams[first_view + blockIdx.y];
    const float4 g = geo[4 * i];
    const float dx = g.x - c.eye[0], dy = g.y - c.eye[1], dz = g.z - c.eye[2];
    const float z = dx * c.w[0] + dy * c.w[1] + dz * c.w[2];
    const float x = (dx * c.u[0] + dy * c.u[1] + dz * c.u[2]) / (c.tanx * z);
    const float y = (dx * c.v[0] + dy * c.v[1] + dz * c.v[2]) / (c.tany * z);
    if (!(z > 0.0f) || !(fabsf(x) < 1.0f) || !(fabsf(y) < 1.0f)) return;
    const int cx = min((int)((x + 1.0f) * (0.5f * kGrid)), kGrid - 1), cy = min((int)((y + 1.0f) * (0.5f * kGrid)), kGrid - 1);
    atomicAdd(&grid[((int)blockIdx.y * kGrid + cy) * kGrid + cx], 1u);
}

// Bucket of each wavefront's weight: the count of the 3x3 cells around its first ray, or (grid ==
// nullptr) the cells of its record.
__global__ void __launch_bounds__(256) k_tile_weight(DevParams p, RayJob job, int64_t num_items, int first_view, int waves,
                                                     const unsigned int* __restrict__ grid,
                                                     unsigned char* __restrict__ bucket, int* __restrict__ hist) {
    __shared__ int cnt[kOrderBuckets];
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (threadIdx.x < kOrderBuckets) cnt[threadIdx.x] = 0;
    __syncthreads();
    unsigned int w = 0u;
    bool cut = false;
    RayRef q;
    const int64_t item = i < waves ? wave_item(p, i, 0) : num_items;
    if (item < num_items && resolve(job, item, q) == RAY_OK) {
        if (grid) {
            const rg_camera& c = job.cams[q.view];
            const int cx = (int)((int64_t)(q.pixel % c.width) * kGrid / c.width);
            const int cy = (int)((int64_t)(q.pixel / c.width) * kGrid / c.height);
            const unsigned int* g = grid + (int64_t)(q.view - first_view) * kGrid * kGrid;
            for (int y = max(cy - 1, 0); y <= min(cy + 1, kGrid - 1); ++y)
                for (int x = max(cx - 1, 0); x <= min(cx + 1, kGrid - 1); ++x) w += g[y * kGrid + x];
        } else {
            const int len = p.rec_len[item];
            if (len & kTileRecord) {
                w = (unsigned int)len & kTileCells;
                cut = (len & kTileSplit) != 0;
            }
        }
    }
    // twice the exponent plus the leading bit of the mantissa; bucket 0 the heaviest, and of records those
    // of split wavefronts
    const int b = cut ? 0 : max(kOrderBuckets - 1 - min((__float_as_int((float)(w + 1u)) >> 22) - 2 * 127, kOrderBuckets - 1),
                                grid ? 0 : 1);
    if (i < waves) {
        bucket[i] = (unsigned char)b;
        atomicAdd(&cnt[b], 1);
    }
    __syncthreads();
    if (threadIdx.x < kOrderBuckets && cnt[threadIdx.x] > 0) atomicAdd(&hist[threadIdx.x], cnt[threadIdx.x]);
}

// The heaviest buckets whose wavefronts are split: those with more than kSplitShare of an even share of
// the whole weight, as long as they are at most 1 / kSplitPart of the wavefronts.
__device__ __forceinline__ int split_buckets(const int* hist, int waves, int slots) {
    float total = 0.0f;
    for (int k = 0; k < kOrderBuckets; ++k) total += (float)hist[k] * __builtin_amdgcn_exp2f(-0.5f * (float)k);
    int n = 0, tiles = 0;
    for (; n < kOrderBuckets; ++n) {
        tiles += hist[n];
        if (tiles > waves / kSplitPart) break;
        if (!(__builtin_amdgcn_exp2f(-0.5f * (float)n) * (float)slots > kSplitShare * total)) break;
    }
    return n;
}

// The wavefronts by falling weight, near their own order within a bucket (hist: the buckets' sizes, then
// their cursors), as 16 wave, or for each part k of a split one 16 wave + 2 k + 1, and -1 in the rest of
// the list; clears the grid for the next job.  split: the number of heaviest buckets that are split, -1: by
// their weight.
__global__ void __launch_bounds__(kOrderBlock) k_tile_order(int waves, const unsigned char* __restrict__ bucket,
                                                            int* __restrict__ hist, int* __restrict__ order, int entries,
                                                            int split, int parts, int slots, unsigned int* grid,
                                                            int cells) {
    __shared__ int cnt[kOrderBuckets], at[kOrderBuckets], num_split, end;
    const int t = threadIdx.x, i = blockIdx.x * kOrderBlock + t;
    if (t < kOrderBuckets) cnt[t] = 0;
    for (int k = i; k < cells; k += gridDim.x * kOrderBlock) grid[k] = 0u;
    __syncthreads();
    const int b = i < waves ? bucket[i] : -1;
    int rank = 0;
    for (unsigned long long rem = __ballot(b >= 0); rem != 0ULL;) {
        const int v = __builtin_amdgcn_readlane(b, __ffsll((long long)rem) - 1);
        const unsigned long long m = __ballot(b == v);
        int first = 0;
        if ((t & 63) == 0) first = atomicAdd(&cnt[v], __popcll(m));
        first = __builtin_amdgcn_readfirstlane(first);
        if (b == v) rank = first + mask_rank(m);
        rem &= ~m;
    }
    __syncthreads();
    if (t < kOrderBuckets) {
        int n = split >= 0 ? split : split_buckets(hist, waves, slots);
        if (split == 1 && hist[0] > waves / kSplitPart) n = 0;  // never expected: not this job's records
        int start = 0;
        for (int k = 0; k < t; ++k) start += hist[k] * (k < n ? parts : 1);
        if (cnt[t] > 0) at[t] = start + atomicAdd(&hist[kOrderBuckets + t], cnt[t]) * (t < n ? parts : 1);
        if (t == 0) num_split = n;
        if (t == kOrderBuckets - 1) end = start + hist[t] * (t < n ? parts : 1);
    }
    __syncthreads();
    if (b >= num_split) order[at[b] + rank] = 16 * i;
    else if (b >= 0)
        for (int k = 0; k < parts; ++k) order[at[b] + parts * rank + k] = 16 * i + 2 * k + 1;
    for (int k = end + i; k < entries; k += gridDim.x * kOrderBlock) order[k] = -1;
}

// ------------------------------------------------------------------ kernels ------------------

// Wavefront of a block, -1 past the last: runs of `chunk` go to one XCD (blocks are dispatched
// round-robin over the eight), so that its L2 serves a compact part of the scene, and the runs in
// turn to all of them, so that no XCD is left with the cheaper ones.  A part of a split wavefront is a
// wavefront of split_rays rays (split).
__device__ __forceinline__ int64_t tile_wave(DevParams& p, int64_t b, int chunk, int waves, bool& split) {
    const int64_t k = b >> 3;
    const int64_t i = ((k / chunk) * 8 + (b & 7)) * chunk + k % chunk;
    split = false;
    if (i >= waves) return -1;
    if (!p.order) return i;
    const int code = p.order[i];
    if (code < 0) return -1;
    split = (code & 1) != 0;
    if (!split) return code >> 4;
    const int parts = p.rays_per_wave / split_rays(p);
    p.rays_per_wave = split_rays(p);
    return (int64_t)(code >> 4) * parts + ((code >> 1) & 7);
}

// Leaves the lanes with mine to the slab stepper.
template <bool SPREAD>
__device__ __forceinline__ void tile_leave(const DevParams& p, int64_t wave, bool mine, int lane) {
    unsigned long long m = __ballot(mine);
    if (SPREAD) {  // in the stepper a lane has a ray
        unsigned long long rays = 0ULL;
        for (int r = 0; r < 8; ++r) rays |= ((m >> (8 * r)) & 1ULL) << r;
        m = rays;
    }
    if (lane == 0)
        p.wide[atomicAdd(p.wide_count, 1ull)] = make_int4((int)wave, (int)(unsigned int)m, (int)(unsigned int)(m >> 32), 0);
}

template <int SPB, bool RNG, int RM, bool SPREAD>
__device__ __forceinline__ void forward_wave(const DevScene& sc, const DevParams& p, const RayJob& job, int64_t num_items,
                                             int64_t wave, bool split, int hit_depth, float* __restrict__ out_rgb,
                                             float* __restrict__ out_depth, float* __restrict__ out_opac, DevStats st,
                                             TileLds& W, int lane) {
    const bool lead = !SPREAD || (lane & 7) == 0;  // of the ray's lanes
    const int64_t item = wave_item(p, wave, SPREAD ? lane >> 3 : lane);
    const bool in = item >= 0 && item < num_items;
    Counters ctr;
    RayRef q;
    q.view = -1;
    const int rs = in ? resolve(job, item, q) : (int)RAY_NONE;
    Ray ray = {};
    unsigned int seed = 0u;
    RayOut o;
    bool alive = false;
    if (rs == RAY_OK) {
        const rg_camera cam = job.cams[q.view];
        seed = RNG ? tea4(p.iteration, (unsigned int)q.pixel) : 0u;
        ray = make_ray(cam, q.pixel, sc.box, p.t_near, p.t_far, RNG ? p.jitter : 0, &seed);
        alive = forward_begin(p, ray, o);
    }
    int group = 0;  // one view, all of it narrow
    if (p.wide && !tile_groups(sc, half_beams(p), alive, q.view, ray, group)) {
        tile_leave<SPREAD>(p, wave, in, lane);
        return;
    }
    Rec rc;
    TileRec tr;
    if constexpr (RM == 1) {
        tr.cells = reinterpret_cast<u32x4*>(rec_region(p, wave));
        tr.cap = (p.rays_per_wave * p.rec_words) >> 2;
    }
    for (int g = 0; g < kTileGroups; ++g) {
        const bool mine = alive && group == g;
        const unsigned long long m = __ballot(mine);
        if (m == 0ULL) break;
        const int view = __builtin_amdgcn_readlane(q.view, __ffsll((long long)m) - 1);
        forward_tile<SPB, RNG, RM, SPREAD>(sc, p, mine, ray, seed, view, job.cams[view].u, g, hit_depth,
                                           out_depth != nullptr, W, lane, ctr, o, tr);
        if (mine) rc.full = tr.full;
    }
    if constexpr (SPREAD) {  // the sums of the ray's lanes
        const float sum = o.C[0];
        for (int c = 0; c < 3; ++c) o.C[c] = __shfl(sum, (lane & 56) + c);
        o.depth = __shfl(sum, (lane & 56) + 3);
    }
    if constexpr (RM == 1) {
        rc.pos = tr.pos | (max(group, 0) << kTileGroupShift) | kTileRecord | (split ? kTileSplit : 0);
        if (lane == 0) ctr.rec_words += 4 * tr.pos;
        if (rs == RAY_NONE && in && lead) {  // padding: no records
            p.rec_len[item] = 0;
            p.rec_id[item] = make_int2(-1, -1);
        }
    }
    if (rs == RAY_OK && lead) forward_finish<RM>(p, q, item, o, rc, ctr, out_rgb, out_depth, out_opac);
    if (rs == RAY_BAD && lead) forward_bad<RM>(p, q, item, st, out_rgb, out_depth, out_opac);
    if (!lead) ctr = Counters();
    flush_counters(ctr, st);
}

template <int SPB, bool RNG, int RM>
__global__ void __launch_bounds__(kWave) __attribute__((amdgpu_waves_per_eu(SPB == 8 ? 4 : 3)))
k_tile_forward(DevScene sc, DevParams p, RayJob job, int64_t num_items, int waves, int chunk, int hit_depth,
               float* __restrict__ out_rgb, float* __restrict__ out_depth, float* __restrict__ out_opac, DevStats st) {
    __shared__ TileLds W;
    bool split;
    const int64_t wave = tile_wave(p, blockIdx.x, chunk, waves, split);
    if (wave < 0) return;
    if constexpr (SPB == 8) {
        if (p.rays_per_wave <= 8) {
            forward_wave<SPB, RNG, RM, true>(sc, p, job, num_items, wave, split, hit_depth, out_rgb, out_depth, out_opac, st,
                                             W, threadIdx.x);
            return;
        }
    }
    forward_wave<SPB, RNG, RM, false>(sc, p, job, num_items, wave, split, hit_depth, out_rgb, out_depth, out_opac, st, W,
                                      threadIdx.x);
}

template <int SPB, bool RNG, int RM, bool SPREAD>
__device__ __forceinline__ void backward_wave(const DevScene& sc, const DevParams& p, const RayJob& job, int64_t num_items,
                                              int64_t wave, bool split, const float* __restrict__ ray_colors,
                                              const float* __restrict__ dLdC, const float* __restrict__ target,
                                              int loss_kind, int count_stats, const DevGrad& gr, DevStats st, BwdLds& S,
                                              GradStage& G, int lane) {
    const bool lead = !SPREAD || (lane & 7) == 0;  // of the ray's lanes
    const int64_t item = wave_item(p, wave, SPREAD ? lane >> 3 : lane);
    const bool in = item >= 0 && item < num_items;
    Counters ctr;
    float loss = 0.0f;
    BwdRay b;
    if (in) backward_setup<RNG, RM>(sc, p, job, wave, lane, item, ray_colors, dLdC, target, loss_kind, st, b, loss, split, lead);
    if (target) add_loss(p, lead ? loss : 0.0f, lane, st);
    // the rays whose tile the forward recorded, and the others if they can go as a tile too
    const unsigned long long recorded = RM == 2 ? __ballot(b.active && b.tile >= 0) : 0ULL;
    const bool rest = b.active && b.tile < 0;
    int group;
    const bool leave = p.wide && __ballot(rest) != 0ULL &&
                       (__ballot(rest && b.rc.w) != 0ULL || !tile_groups(sc, half_beams(p), rest, b.view, b.ray, group));
    if (leave) tile_leave<SPREAD>(p, wave, rest, lane);
    int num_cells = 0;
    if (recorded != 0ULL) num_cells = __builtin_amdgcn_readlane(b.rc.end, __ffsll((long long)recorded) - 1);
    const u32x4* cells = RM == 2 ? reinterpret_cast<const u32x4*>(rec_region(p, wave)) : nullptr;
    backward_tile<SPB, RNG, SPREAD>(sc, p, job.cams, b.active && !(leave && rest), b.ray, b.seed, b.view, b.Cf, b.dL, cells,
                                    num_cells, b.tile, rest || b.trunc, S, G, lane, gr, ctr, st.c + C_DROP);
    if (!lead) ctr = Counters();
    if (count_stats) flush_counters(ctr, st);
}

template <int SPB, bool RNG, int RM>
__global__ void __launch_bounds__(kWave) __attribute__((amdgpu_waves_per_eu(3)))
k_tile_backward(DevScene sc, DevParams p, RayJob job, int64_t num_items, int waves, int chunk, const float* __restrict__ ray_colors,
                const float* __restrict__ dLdC, const float* __restrict__ target, int loss_kind, int count_stats,
                DevGrad gr, DevStats st) {
    __shared__ BwdLds S;
    __shared__ GradStage G;
    bool split;
    const int64_t wave = tile_wave(p, blockIdx.x, chunk, waves, split);
    if (wave < 0) return;
    if constexpr (SPB == 8) {
        if (p.rays_per_wave <= 8) {
            backward_wave<SPB, RNG, RM, true>(sc, p, job, num_items, wave, split, ray_colors, dLdC, target, loss_kind,
                                              count_stats, gr, st, S, G, threadIdx.x);
            return;
        }
    }
    backward_wave<SPB, RNG, RM, false>(sc, p, job, num_items, wave, split, ray_colors, dLdC, target, loss_kind, count_stats,
                                       gr, st, S, G, threadIdx.x);
}

// Counts the wavefronts that are no beams, every stride-th of the job looked at.
__global__ void __launch_bounds__(kWave) k_tile_sample(DevScene sc, DevParams p, RayJob job, int64_t num_items, int stride,
                                                       unsigned long long* count) {
    const int lane = threadIdx.x;
    const int64_t item = wave_item(p, (int64_t)blockIdx.x * stride, lane);
    RayRef q;
    q.view = -1;
    Ray ray = {};
    bool alive = false;
    if (item >= 0 && item < num_items && resolve(job, item, q) == RAY_OK) {
        const rg_camera cam = job.cams[q.view];
        unsigned int seed = p.jitter ? tea4(p.iteration, (unsigned int)q.pixel) : 0u;
        ray = make_ray(cam, q.pixel, sc.box, p.t_near, p.t_far, p.jitter, &seed);
        RayOut o;
        alive = forward_begin(p, ray, o);
    }
    int group;
    if (!tile_groups(sc, false, alive, q.view, ray, group) && lane == 0) atomicAdd(count, 1ull);
}

// Counts for half_beams.  Not in the smallest jobs (4 rays a wavefront), where each wavefront's march is short
// either way and the launch would show, nor before a replay, which takes the forward's beams.
void launch_sample(const DevScene& sc, DevParams& p, const RayJob& job, unsigned long long* count, hipStream_t s) {
    if (!p.wide || p.rays_per_wave <= 4 || p.rec_mode == 2) return;
    const int64_t waves = num_waves(p, job.num_rays);
    const int64_t stride = (waves + kSampled - 1) / kSampled;
    const int64_t samples = (waves + stride - 1) / stride;
    hipLaunchKernelGGL(k_tile_sample, dim3((unsigned)samples), dim3(kWave), 0, s, sc, p, job, job.num_rays, (int)stride, count);
    p.sample_wide = count;
    p.sample_limit = (int)(samples / kHalfShare);
}

// Launch of a tile kernel over all wavefronts of a job.
template <typename K, typename... A>
void launch_tiles(K kernel, const DevScene& sc, const DevParams& p, const RayJob& job, hipStream_t s, A... args) {
    const int64_t waves = p.order && !p.wide ? order_entries(num_waves(p, job.num_rays)) : num_waves(p, job.num_rays);
    // 64 wavefronts of the image's own order, at least 8 runs for each XCD; 8 of the ordered ones
    const int chunk = p.order ? 8 : (int)(waves < 8 * 8 * 64 ? (waves + 63) / 64 : 64);
    const int64_t nb = (waves + 8 * chunk - 1) / (8 * chunk) * (8 * chunk);
    hipLaunchKernelGGL(kernel, dim3((unsigned)nb), dim3(kWave), 0, s, sc, p, job, job.num_rays, (int)waves, chunk, args...);
}

// Fills p.order (dear wavefronts first): from the Gaussians' means (forward), or the records.
void launch_order(const DevScene& sc, const DevParams& p, const RayJob& job, bool records, int slots,
                  unsigned long long* counters, hipStream_t s) {
    int* hist = reinterpret_cast<int*>(counters);
    const int waves = (int)num_waves(p, job.num_rays);
    const int first = job.ray_view ? 0 : job.view, views = job.ray_view ? job.num_views : 1;
    const int64_t stride = ((int64_t)sc.n * views + kSplats) / kSplats;
    const int64_t count = (sc.n + stride - 1) / stride;
    if (!records && count > 0)
        hipLaunchKernelGGL(k_tile_splat, dim3((unsigned)((count + 255) / 256), views), dim3(256), 0, s, sc.n, (int)stride,
                           sc.geo, job.cams, first, p.order_grid);
    hipLaunchKernelGGL(k_tile_weight, dim3((waves + 255) / 256), dim3(256), 0, s, p, job, job.num_rays, first, waves,
                       records ? nullptr : p.order_grid, p.order_bucket, hist);
    hipLaunchKernelGGL(k_tile_order, dim3((waves + kOrderBlock - 1) / kOrderBlock), dim3(kOrderBlock), 0, s, waves,
                       p.order_bucket, hist, p.order, (int)(p.wide ? waves : order_entries(waves)),
                       p.wide || p.rays_per_wave <= split_rays(p) ? 0 : records ? 1 : -1,
                       p.rays_per_wave / split_rays(p), slots, p.order_grid, records ? 0 : views * kGrid * kGrid);
}

// Specialised on SPB (8 samples per slab, or any number up to 16), on whether the random generator is used and on the
// record mode.
#define RG_TILE_DISPATCH(RMV, RMON, KERNEL, ...)                                                       \
    do {                                                                                               \
        const bool rng = p.jitter || p.rnd_sample;                                                     \
        if (p.spb == 8) {                                                                              \
            if (rng) launch_tiles(RMV ? KERNEL<8, true, RMON> : KERNEL<8, true, 0>, __VA_ARGS__);      \
            else launch_tiles(RMV ? KERNEL<8, false, RMON> : KERNEL<8, false, 0>, __VA_ARGS__);        \
        } else {                                                                                       \
            if (rng) launch_tiles(RMV ? KERNEL<16, true, RMON> : KERNEL<16, true, 0>, __VA_ARGS__);    \
            else launch_tiles(RMV ? KERNEL<16, false, RMON> : KERNEL<16, false, 0>, __VA_ARGS__);      \
        }                                                                                              \
    } while (0)

}  // namespace

// The stepper takes all rays where its own options are asked for (per-lane walks, refilled lanes) and
// below depth zero, where a beam's bounds do not hold.
bool takes_tiles(const DevParams& p) {
    return p.packet && p.t_near >= 0.0f && !(p.ray_chunk > 0 && p.refill_lanes > 0);
}

// Small jobs spread their rays over more wavefronts: with fewer than the GPU holds (4 on each of its
// 1024 SIMDs) the slowest wavefront is the launch, and a narrower beam has fewer candidates.  Beyond
// that narrow wavefronts only repeat work.  Drop-in training step with 4 / 8 / 16 / 32 / 64 rays (us; - : not
// measured): 64 tiles of 4k Gaussians 490 / 583 / - / - / -, 256 of 20k 750 / 968 / 1550 / - / -, 529 of 20k
// 796 / 855 / 938 / - / -, 1024 of 30k in blobs 1115 / 1061 / 956 / - / -, unbounded 1934 / 1333 / 1261 / - / -,
// 2025 - / 1178 / 1016 / 958 / - and - / 1950 / 1490 / 1327 / -, 3025 of 50k - / 1646 / 1337 / 1257 / - and - / 3154 /
// 2196 / 1720 / -; before the spread wavefronts, 2555 tiles 3370 / 2340 / 2130 / 2250 / 3320, 3750 tiles 29.3 / 18.8 /
// 13.2 / 11.3 / 9.9 ms.
int rays_per_wave(int64_t num_items) {
    const int64_t tiles = (num_items + kWave - 1) / kWave;
    return tiles <= 576 ? 4 : tiles <= 1024 ? 16 : tiles <= 3072 ? 32 : 64;
}

int64_t order_entries(int64_t waves) { return waves + 3 * (waves / kSplitPart); }

int64_t order_grid_cells(int views) { return (int64_t)views * kGrid * kGrid; }

// A block's rays differ by at most eight pixel steps of the image plane along each axis; their unit
// directions differ by no more, the plane's nearest point being w at a right angle.
bool view_is_narrow(const rg_camera& cam, int64_t n) {
    auto dot = [](const float* a, const float* b) { return (double)a[0] * b[0] + (double)a[1] * b[1] + (double)a[2] * b[2]; };
    const double uw = dot(cam.u, cam.w), vw = dot(cam.v, cam.w), ww = dot(cam.w, cam.w);
    const double uu = dot(cam.u, cam.u), vv = dot(cam.v, cam.v);
    if (!(ww > 0.0) || !(uw * uw <= 1e-8 * uu * ww) || !(vw * vw <= 1e-8 * vv * ww)) return false;
    const double dx = 16.0 * fabs((double)cam.tanx) / cam.width, dy = 16.0 * fabs((double)cam.tany) / cam.height;
    const double spread = 1.01 * sqrt((dx * dx * uu + dy * dy * vv) / ww);
    return spread < kTileSpread && (double)n * spread * spread < kTileDensity;
}

hipError_t launch_forward(const DevScene& sc, const DevParams& p0, const RayJob& job, int hit_depth, float* out_rgb,
                          float* out_depth, float* out_opacity, DevStats st, hipStream_t s) {
    if (job.num_rays <= 0) return hipSuccess;
    DevParams p = p0;
    p.wide_count = st.c + 80;
    if (p.tiles) {
        launch_sample(sc, p, job, st.c + 84, s);
        if (p.order) launch_order(sc, p, job, false, 4096, st.c + 16, s);
        RG_TILE_DISPATCH(p.rec_mode == 1, 1, k_tile_forward, sc, p, job, s, hit_depth, out_rgb, out_depth, out_opacity, st);
        if (!p.wide) return hipGetLastError();
    }
    return launch_forward_steps(sc, p, job, hit_depth, out_rgb, out_depth, out_opacity, st, s);
}

hipError_t launch_backward(const DevScene& sc, const DevParams& p0, const RayJob& job, int hit_depth,
                           const float* ray_colors, const float* dLdC, const float* target, int loss_kind,
                           int count_stats, DevGrad gr, DevStats st, hipStream_t s) {
    if (job.num_rays <= 0) return hipSuccess;
    DevParams p = p0;
    p.wide_count = st.c + 82;
    if (p.tiles) {
        launch_sample(sc, p, job, st.c + 85, s);
        if (p.order) launch_order(sc, p, job, p.rec_mode == 2, 3072, st.c + 48, s);
        RG_TILE_DISPATCH(p.rec_mode == 2, 2, k_tile_backward, sc, p, job, s, ray_colors, dLdC, target, loss_kind, count_stats,
                         gr, st);
        if (!p.wide) return hipGetLastError();
    }
    return launch_backward_steps(sc, p, job, hit_depth, ray_colors, dLdC, target, loss_kind, count_stats, gr, st, s);
}

}  // namespace rg
