// Ray kernels of the gfx950 ray caster: forward render, recompute-based backward (optionally
// forming a per-pixel loss gradient itself), and the hit-set export used for verification.
//
// Per ray (one lane), the reference's per-slab loop (cuda_train/forward/gaussians_aabb.cu:521-612,
// backward/gaussians_aabb.cu:505-775) is kept exactly -- slab grid tb accumulated in FP32 from
// tenter, 8-sample buffers, thresholded density sums, per-slab transmittance exit -- but the hit
// sets are found differently: instead of one BVH traversal per slab, one traversal gathers every
// bounding-ellipsoid interval [r1, r2] overlapping a SEGMENT of m slabs into a per-lane list in
// LDS (capacity hit_depth); each slab's hit set is then {entries: max(tmin,r1) <= min(tmax,r2)},
// the reference's own predicate.  m adapts to the list fill (doubling across empty space,
// halving on overflow); a slab whose own hit set exceeds the list is processed by a per-slab
// traversal that accumulates on the fly (no storage).  Forward and backward step through slabs
// with the same SegState machine, so both make identical segment decisions and sum each slab in
// the same order (the traversal's DFS order, which is increasing slot: slots are numbered in the
// tree's depth-first leaf order by either builder).
//
// Sampling uses the closed form of the Gaussian along the ray: with the predicate's quantities
// (t_c = b l, P = O' + b D^, D' = M' d, h = ln|sigma/thr|),
//     0.5 |M (o + t d - mu)|^2 = h |P|^2 + h |D'|^2 (t - t_c)^2,
// so each (sample, hit) costs one FMA pair and one exp.  The backward accumulates, per
// (slab, hit), four scalars (sum m phi, sum m phi tau, sum m phi tau^2, sum m B; m = sigma w) and
// expands them into the 14 parameter gradients of backward/gaussians_aabb.cu:700-763.
//
// Gradient scatter is wave-cooperative: every lane's list is sorted by slot, so after each
// lane has prepared one slab, the 64 lanes (an 8x8 pixel tile) walk the union of their hit sets in
// increasing slot order (a wave-wide min per step); the lanes holding the current Gaussian compute
// their contributions together, and the wave sums them and issues the 14 atomic adds as one
// 14-lane instruction.

#include <hip/hip_runtime.h>

#include <climits>

#include "rg_device.h"
#include "rg_internal.h"
#include "rg_trace.h"

namespace rg {
namespace {

constexpr int kMaxSeg = 4096;

// Per-lane interval list in LDS, [entry][lane] so lanes access consecutive words: the Gaussian's
// slot, its predicate interval and its sampling quadratic (t_c, A, Cq) from the gather.
template <int CAP>
struct IList {
    int g[CAP][kWave];
    float r1[CAP][kWave];
    float r2[CAP][kWave];
};

// Bit e set for the list entries (e < cnt) whose interval meets the slab [tmin, tmax]: the
// lanes then loop over their own hits only (in increasing entry = slot order), so a wave
// iterates max-over-lanes(hits) times instead of max-over-lanes(cnt).
//
// Every listed interval met its gathered segment, so r1 <= r2 (or one of them is NaN), and every
// slab has tmin <= tmax; for such operands overlaps(tmin, tmax, r1, r2) is !(r1 > tmax) and
// !(r2 < tmin), NaN ends included (overlaps() lets fmaxf / fminf drop a NaN).  That form needs
// no NaN-quieting max/min and no branch per entry: the loop ends at the longest list among the
// lanes executing the call (a ballot, which counts only those lanes), and each lane masks off the
// entries past its own count.
template <int CAP>
__device__ __forceinline__ unsigned int slab_mask(const IList<CAP>& L, int cnt, float tmin, float tmax, int lane) {
    unsigned int m = 0u;
#pragma unroll
    for (int e = 0; e < CAP; ++e) {
        if (__builtin_amdgcn_ballot_w64(e < cnt) == 0ULL) break;
        const bool in = (e < cnt) & !(L.r1[e][lane] > tmax) & !(L.r2[e][lane] < tmin);
        m |= in ? 1u << e : 0u;
    }
    return m;
}

// Sampling terms of a listed hit, recomputed from the Gaussian's record (a list entry keeps only
// the slot and the interval, 12 bytes, so the list holds twice the entries in the same LDS).
// The same operations as the predicate's give the same values; the roots are skipped.
__device__ __forceinline__ Isect entry_hit(const DevScene& sc, const Ray& ray, int slot, float r1, float r2,
                                           float& sigma) {
    float4 g0, g1, g2, g3;
    load_rec(sc.geo, slot, g0, g1, g2, g3);
    Isect I;
    float b, c;
    isect_terms(g0, g1, g2, g3, ray, I, b, c);  // the interval is the entry's: no roots needed
    I.r1 = r1;
    I.r2 = r2;
    refine_sampling(g0, g1, g2, g3, ray, I);
    sigma = g0.w;
    return I;
}

// Writes list entry e of the lane from Gaussian `slot` (false when the ray misses its ellipsoid).
template <int CAP>
__device__ __forceinline__ bool load_entry(const DevScene& sc, const Ray& ray, int slot, IList<CAP>& L, int e,
                                           int lane) {
    float4 g0, g1, g2, g3;
    load_rec(sc.geo, slot, g0, g1, g2, g3);
    Isect I;
    if (!intersect(g0, g1, g2, g3, ray, I)) return false;
    L.g[e][lane] = slot;
    L.r1[e][lane] = I.r1;
    L.r2[e][lane] = I.r2;
    return true;
}

// Gathers the intervals overlapping [ta, tb] of the Gaussians with slot > after into the lane's
// list; returns the count, or CAP + 1 on overflow (the list then holds the first CAP).  Entries
// come out in DFS order of the tree = increasing slot.
template <int CAP>
__device__ __forceinline__ int gather(const DevScene& sc, const DevParams& p, const Ray& ray, float ta, float tb,
                                      IList<CAP>& L, int lane, int after = -1) {
    int cnt = 0;
    trav(p, sc, ray, ta, tb, [&](int slot) -> bool {
        if (slot <= after) return true;
        float4 g0, g1, g2, g3;
        load_rec(sc.geo, slot, g0, g1, g2, g3);
        Isect I;
        if (!intersect(g0, g1, g2, g3, ray, I)) return true;
        if (!overlaps(ta, tb, I.r1, I.r2)) return true;
        if (cnt >= CAP) {
            cnt = CAP + 1;
            return false;
        }
        L.g[cnt][lane] = slot;
        L.r1[cnt][lane] = I.r1;
        L.r2[cnt][lane] = I.r2;
        ++cnt;
        return true;
    });
    return cnt;
}

// ------------------------------------------------------------------ slab stepper -------------
//
// The reference's slab loop, with hit sets served from gathered segments.  next_slab() returns
// the next slab to process (tb, tmin, tmax) in either list mode (s.cnt entries in the lane's
// list) or direct mode (the slab's hit set overflows the list: per-slab traversal); empty
// segments are skipped without returning.  advance_slab() moves past the slab just processed.

struct SegState {
    float tb;       // start of the current slab (reference tbuffer)
    int k;          // index of that slab along the ray
    float seg_hi;   // end of the gathered segment
    float seg_lo;   // start of the gathered segment
    int m;          // segment length in slabs for the next gather
    int cnt;        // entries in the lane's list
    bool valid;     // list holds the current segment
    bool direct;    // current slab is processed by per-slab traversal
    int dpos;       // replay of a direct slab: first word of its recorded hit list
    int dcnt;       //   and its length (-1: no recorded list, traverse)
    bool dense;     // the last direct slab held more hits than the list: walk the next one too
    int knext;      // replay: slab index of the next record not yet taken (INT_MAX: none)
};

__device__ __forceinline__ void seg_init(SegState& s, const Ray& ray, const DevParams& p) {
    s.tb = ray.tenter;
    s.k = 0;
    s.seg_hi = ray.tenter;
    s.seg_lo = ray.tenter;
    s.m = p.seg_slabs;
    s.cnt = 0;
    s.valid = false;
    s.direct = false;
    s.dpos = 0;
    s.dcnt = -1;
    s.dense = false;
    s.knext = INT_MAX;
}

// ------------------------------------------------------------------ hit-list records ---------
//
// The forward records, per ray, every list it gathered and every slab it served by per-slab
// traversal; the backward over the same rays replays them instead of walking the LBVH.  Each
// record carries the index of the slab where the forward gathered it, and the backward takes
// every record that starts at or before its current slab, so it holds the forward's list for
// every slab: the same Gaussians in the same order.  A ray whose records end before its backward
// does (space ran out, or the backward goes further) continues with its own gathers from there.
// A record is a whole number of 32-byte sectors written by full 16-byte stores (a partly written
// sector costs a read-modify-write in the memory):
//   word 0: bit 31 set, bit 30 direct slab, bits 29..24 list count, bits 21..0 slab index
//   word 1: list record: end of the gathered segment (float bits);
//           direct slab: number of hits recorded after it (kRecNoList: none, the slab is walked)
//   words 2..: the list's slots, or the direct slab's hits in traversal order, zero padded
constexpr unsigned int kRecOn = 0x80000000u, kRecDirect = 0x40000000u, kRecNoList = 0xffffffffu;
constexpr int kRecMaxSlab = (1 << 22) - 1;
constexpr int kRecMaxDirect = 256;  // longest recorded hit list of a direct slab

template <int CAP>
__device__ __forceinline__ void record(Rec& rc, int k, bool direct, float hi, const IList<CAP>& L, int cnt,
                                       int lane) {
    if (!rc.w || rc.full) return;
    const int len = rec_len(cnt);
    if (k > kRecMaxSlab || rc.pos + len > rc.end) {
        rc.full = true;
        return;
    }
    const unsigned int h0 = kRecOn | (direct ? kRecDirect : 0u) | ((unsigned int)cnt << 24) | (unsigned int)k;
    for (int c = 0; c < len; c += 4) {
        unsigned int v[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int e = c + j - 2;
            v[j] = c + j == 0 ? h0 : c + j == 1 ? __float_as_uint(hi) : (e < cnt ? (unsigned int)L.g[e][lane] : 0u);
        }
        // streaming stores: the records are read once, by the next kernel, and must not evict
        // the tree and Gaussian records the traversal keeps in L2
        const u32x4 q = {v[0], v[1], v[2], v[3]};
        __builtin_nontemporal_store(q, reinterpret_cast<u32x4*>(rec_at(rc, rc.pos + c)));
    }
    rc.pos += len;
}

// Direct slab (forward): the record is opened before the slab's traversal, its hits appended as
// the traversal reaches them, and closed with their count (a list that does not fit is dropped:
// the backward then walks that slab).
__device__ __forceinline__ int rec_direct_open(Rec& rc) {
    if (!rc.w || rc.full) return -1;
    if (rc.pos + 8 > rc.end) {
        rc.full = true;
        return -1;
    }
    return rc.pos;
}

__device__ __forceinline__ void rec_direct_push(const Rec& rc, int start, int n, int slot) {
    const int w = start + 2 + n;
    if (start >= 0 && n < kRecMaxDirect && w < rc.end) *rec_at(rc, w) = (unsigned int)slot;
}

__device__ __forceinline__ void rec_direct_close(Rec& rc, int start, int n, int k) {
    if (start < 0) return;
    const bool listed = n <= kRecMaxDirect && start + rec_len(n) <= rc.end && k <= kRecMaxSlab;
    *rec_at(rc, start) = kRecOn | kRecDirect | (unsigned int)min(k, kRecMaxSlab);
    *rec_at(rc, start + 1) = listed ? (unsigned int)n : kRecNoList;
    rc.pos = start + (listed ? rec_len(n) : 8);
}

// Replay: takes every record that starts at or before the current slab.  Anything that does not
// fit the lane's list or does not reproduce (never expected) ends the replay.
template <int CAP>
__device__ __forceinline__ void take_records(SegState& s, const DevScene& sc, const Ray& ray, IList<CAP>& L,
                                             int lane, Rec& rc) {
    s.knext = INT_MAX;
    while (rc.pos + 8 <= rc.end) {
        const u32x4 h = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(rec_at(rc, rc.pos)));
        if (!(h.x & kRecOn)) {
            rc.w = nullptr;
            s.valid = false;
            return;
        }
        if ((int)(h.x & (unsigned int)kRecMaxSlab) > s.k) {
            s.knext = (int)(h.x & (unsigned int)kRecMaxSlab);
            return;
        }
        const int cnt = (int)((h.x >> 24) & 63u);
        const int len = rec_len(cnt);
        if (h.x & kRecDirect) {
            s.direct = true;
            s.cnt = 0;
            s.valid = true;
            const unsigned int n = h.y;
            if (n != kRecNoList && n <= (unsigned int)kRecMaxDirect && rc.pos + rec_len((int)n) <= rc.end) {
                s.dpos = rc.pos + 2;
                s.dcnt = (int)n;
                rc.pos += rec_len((int)n);
            } else {
                s.dcnt = -1;
                rc.pos += 8;
            }
            continue;
        }
        bool ok = cnt <= CAP && rc.pos + len <= rc.end;
        for (int e = 0; ok && e < cnt; ++e) {
            const int slot = (int)__builtin_nontemporal_load(rec_at(rc, rc.pos + 2 + e));
            ok = slot >= 0 && slot < sc.n && load_entry<CAP>(sc, ray, slot, L, e, lane);
        }
        if (!ok) {
            rc.w = nullptr;
            s.valid = false;
            return;
        }
        s.direct = false;
        s.cnt = cnt;
        s.seg_hi = __uint_as_float(h.y);
        s.valid = true;
        rc.pos += len;
    }
}

template <int CAP, int RM>
__device__ __forceinline__ bool next_slab(SegState& s, const DevScene& sc, const DevParams& p, const Ray& ray,
                                          IList<CAP>& L, int lane, Counters& ctr, float& tmin, float& tmax, Rec& rc) {
    const float slab = p.dt * (float)p.spb;
    while (true) {
        if (!(s.tb < ray.texit)) return false;
        if constexpr (RM == 2) {
            if (rc.w) {
                take_records<CAP>(s, sc, ray, L, lane, rc);
                if (!s.valid) rc.w = nullptr;  // no record holds this slab: own gathers from here on
            }
        }
        if (!s.valid && s.dense) {
            // inside a dense stretch (the last slab needed its own walk): a gather would most
            // likely overflow too, so the slab is walked without trying it
            ctr.fallback++;
            s.direct = true;
            s.cnt = 0;
            s.dcnt = -1;
            s.valid = true;
        }
        if (!s.valid) {
            s.seg_hi = fminf(ray.texit, s.tb + (float)s.m * slab);
            s.seg_lo = s.tb;
            const int cnt = gather<CAP>(sc, p, ray, s.tb, s.seg_hi, L, lane);
            ctr.gathers++;
            if (cnt > CAP) {
                // shorter segments down to two slabs; a single slab is walked rather than
                // gathered (one traversal either way, and the walk needs no list)
                if (s.m > 2) {
                    s.m >>= 1;
                    continue;
                }
                ctr.fallback++;
                s.direct = true;
                s.cnt = 0;
                s.dcnt = -1;  // recorded (with its hits) by the forward's traversal of the slab
            } else {
                s.direct = false;
                s.cnt = cnt;
                if constexpr (RM == 1) record<CAP>(rc, s.k, false, s.seg_hi, L, cnt, lane);
            }
            s.valid = true;
        }
        tmax = fminf(ray.texit, add_exact(s.tb, slab));
        if (!s.direct) {
            if (tmax > s.seg_hi) {  // segment done: adapt its length to the list fill, gather the next
                if (s.cnt == 0 || 4 * s.cnt < CAP) s.m = min(s.m * 2, kMaxSeg);
                else if (4 * s.cnt > 3 * CAP) s.m = max(s.m >> 1, 1);
                s.valid = false;
                continue;
            }
            if (s.cnt == 0) {  // empty segment: its slabs have no hits
                const float nt = add_exact(s.tb, slab);
                if (!(nt > s.tb)) return false;
                s.tb = nt;
                ++s.k;
                continue;
            }
        }
        tmin = fmaxf(ray.tenter, s.tb);
        return true;
    }
}

// Whether the lane's next slab needs a new gather because its list is spent (a lane crossing an
// empty segment does not count: it only steps to the segment end).
__device__ __forceinline__ bool needs_gather(const SegState& s, const Ray& ray, const DevParams& p) {
    const float slab = p.dt * (float)p.spb;
    return !s.valid || (!s.direct && s.cnt > 0 && fminf(ray.texit, add_exact(s.tb, slab)) > s.seg_hi);
}

// Wave-synchronous gathers: when one lane executing the call must gather, all of them gather
// anew from their current slab, so that one packet traversal serves every lane.  The gathered
// lists hold the same hit sets, so the result does not change.  Lanes replaying recorded lists
// (own = false) neither gather nor ask others to.
__device__ __forceinline__ void sync_gathers(SegState& s, const Ray& ray, const DevParams& p, bool own = true) {
    const bool need = own && needs_gather(s, ray, p);
    // a lane that has used up less than half of its segment keeps its list for a later round
    const bool fresh = s.valid && !s.direct && s.cnt > 0 && 2.0f * (s.tb - s.seg_lo) < s.seg_hi - s.seg_lo;
    if (__ballot(need) != 0ULL && own && (need || !fresh)) s.valid = false;
}

__device__ __forceinline__ bool advance_slab(SegState& s, const DevParams& p) {
    const float nt = add_exact(s.tb, p.dt * (float)p.spb);
    if (s.direct) {
        s.direct = false;
        s.valid = false;
    }
    if (!(nt > s.tb)) return false;  // slab below half an ulp of t: no progress possible
    s.tb = nt;
    ++s.k;
    return true;
}

// ------------------------------------------------------------------ per-ray bodies -----------

// Wavefront-wide step over slabs without hits, after a round in which no lane had one: the lanes
// stepping through a list (step) advance together over the slabs empty for them, up to the
// wavefront's earliest possible next hit -- the smallest start (or the segment end) among the list
// entries that have not ended before each lane's slab; lanes that cannot step bound it by their
// slab (bound_tb).  Every slab passed ends before that point, so none overlaps an entry: the slabs
// with hits and their order are unchanged, and the lanes stay in step in depth.  A replaying lane
// stops at the slab of its next record (knext), which it takes there.  Called by all 64 lanes.
template <int CAP>
__device__ __forceinline__ void jump_empty(SegState& s, const Ray& ray, const DevParams& p, const IList<CAP>& L,
                                           int lane, bool step, bool bound_tb, int knext) {
    float bound = bound_tb ? s.tb : INFINITY;
    if (step) {
        bound = s.seg_hi;
        for (int e = 0; e < s.cnt; ++e)
            if (!(L.r2[e][lane] < s.tb)) bound = fminf(bound, fmaxf(L.r1[e][lane], s.tb));
    }
    const float tstar = wave_min64f(bound);
    if (step && tstar < INFINITY) {
        const float slab = p.dt * (float)p.spb;
        while (s.k < knext) {
            const float nt = add_exact(s.tb, slab);
            if (!(fminf(ray.texit, nt) < tstar) || !(nt > s.tb)) break;
            s.tb = nt;
            ++s.k;
        }
    }
}

// One slab of the forward (the reference's raygen loop body, forward/gaussians_aabb.cu:546-606):
// the next slab with hits, its sample buffers, compositing.  Returns false when the ray is done.
template <int SPB, int CAP, bool RNG, int RM>
__device__ __forceinline__ bool forward_step(const DevScene& sc, const DevParams& p, const Ray& ray,
                                             unsigned int& seed, const float4* __restrict__ rgbv, IList<CAP>& L,
                                             int lane, Counters& ctr, RayOut& o, Rec& rc, SegState& s,
                                             bool* hit = nullptr) {
    if (!(o.T > p.t_eps)) return false;
    const float first_tb = ray.tenter;
    sync_gathers(s, ray, p);
    float tmin, tmax;
    if (!next_slab<CAP, RM>(s, sc, p, ray, L, lane, ctr, tmin, tmax, rc)) return false;
    const float tb = s.tb;
    float sig[SPB], cr[SPB], cg[SPB], cb[SPB];
#pragma unroll
    for (int i = 0; i < SPB; ++i) sig[i] = cr[i] = cg[i] = cb[i] = 0.0f;
    int nh = 0;
    auto eval_hit = [&](int slot, const Isect& I, float sigma) {
        accum_hit<SPB, RNG>(I, sigma, rgbv[slot], tb, seed, p, sig, cr, cg, cb);
        if (tb == first_tb || I.r1 > tmin) ctr.P++;
        ++nh;
    };
    if (s.direct) {
        int rstart = -1;
        if constexpr (RM == 1) rstart = rec_direct_open(rc);
        trav(p, sc, ray, tmin, tmax, [&](int slot) -> bool {
            float4 g0, g1, g2, g3;
            load_rec(sc.geo, slot, g0, g1, g2, g3);
            Isect I;
            if (!intersect(g0, g1, g2, g3, ray, I)) return true;
            if (!overlaps(tmin, tmax, I.r1, I.r2)) return true;
            refine_sampling(g0, g1, g2, g3, ray, I);
            if constexpr (RM == 1) rec_direct_push(rc, rstart, nh, slot);
            eval_hit(slot, I, g0.w);
            return true;
        });
        if constexpr (RM == 1) rec_direct_close(rc, rstart, nh, s.k);
        s.dense = nh > CAP;
    } else {
        unsigned int m = slab_mask<CAP>(L, s.cnt, tmin, tmax, lane);
        while (m != 0u) {
            const int e = __builtin_ctz(m);
            m &= m - 1u;
            const int slot = L.g[e][lane];
            float sigma;
            const Isect I = entry_hit(sc, ray, slot, L.r1[e][lane], L.r2[e][lane], sigma);
            eval_hit(slot, I, sigma);
        }
    }
    ctr.K += nh;
    if (hit) *hit = nh > 0;
    if (p.max_hits > 0 && nh > p.max_hits) ctr.ovf++;
    if (nh > 0) {
        composite<SPB, RNG>(sig, cr, cg, cb, tb, seed, p, true, o);
        if (RNG && p.rnd_sample == 1) seed = skip_draws(seed, p.spb);  // the slab's draws are spent
    }
    return advance_slab(s, p);
}

template <int SPB, int CAP, bool RNG, int RM>
__device__ void forward_ray(const DevScene& sc, const DevParams& p, const Ray& ray, unsigned int seed,
                            const float4* __restrict__ rgbv, IList<CAP>& L, int lane, Counters& ctr, RayOut& o,
                            Rec& rc) {
    SegState s;
    bool alive = forward_begin(p, ray, o);
    seg_init(s, ray, p);
    bool jump = false;
    while (__ballot(alive) != 0ULL) {
        if (jump) jump_empty<CAP>(s, ray, p, L, lane, alive && s.valid && !s.direct, alive, INT_MAX);
        bool hit = false;
        if (alive) alive = forward_step<SPB, CAP, RNG, RM>(sc, p, ray, seed, rgbv, L, lane, ctr, o, rc, s, &hit);
        jump = p.fwd_jump && __ballot(hit) == 0ULL;
    }
}

// Scatter of the slabs whose hit set overflowed the list (lanes with dsc), called by all 64
// lanes together: a packet traversal over the lanes' slab intervals; at each leaf the lanes whose
// slab holds the Gaussian compute its gradient contribution and the wave sums them into one
// staged record per view (as in the list scatter), instead of 14 atomics per lane and hit.
template <int SPB, bool RNG>
__device__ void direct_scatter_wave(const DevScene& sc, const DevParams& p, bool dsc, const Ray& ray,
                                    const float4* __restrict__ rgbv, float cur_tb, unsigned int cur_seed,
                                    float cur_tmin, float cur_tmax,
                                    const float* Gq, const float* Bq, const float* dL, GradStage& G,
                                    Staged& st, int lane, const DevGrad& gr, int view, unsigned long long* drops) {
    const float ix = 1.0f / ray.dx, iy = 1.0f / ray.dy, iz = 1.0f / ray.dz;
    const int total = sc.total_nodes;
    bool live = dsc;
    int idx = 0;
    while (idx < total && __ballot(live) != 0ULL) {
        idx = __builtin_amdgcn_readfirstlane(idx);
        const float4 lo = ld_node(sc.nodes, 2 * idx);
        const float4 hi = ld_node(sc.nodes, 2 * idx + 1);
        const int miss = __float_as_int(lo.w);
        const int leaf = __float_as_int(hi.w);
        if (miss <= idx) break;  // malformed link (uniform): never loop
        const bool h = live && box_hit(lo, hi, ray, ix, iy, iz, cur_tmin, cur_tmax);
        if (__ballot(h) == 0ULL) {
            idx = miss;
            continue;
        }
        if (leaf < 0) {
            idx = idx + 1;
            continue;
        }
        if (leaf >= sc.n) break;  // malformed leaf index (uniform)
        float v[kMoments];
#pragma unroll
        for (int k = 0; k < kMoments; ++k) v[k] = 0.0f;
        bool c = false;
        if (h) {
            float4 g0, g1, g2, g3;
            load_rec(sc.geo, leaf, g0, g1, g2, g3);
            Isect I;
            if (intersect(g0, g1, g2, g3, ray, I) && overlaps(cur_tmin, cur_tmax, I.r1, I.r2)) {
                refine_sampling(g0, g1, g2, g3, ray, I);
                float md[SPB];
                sample_densities<SPB, RNG>(I, g0.w, cur_tb, cur_seed, p, md);
                const float P[3] = {I.Px, I.Py, I.Pz}, D[3] = {I.Dx, I.Dy, I.Dz};
                grad_moments<SPB, RNG>(P, D, g0.w, md, I.tc, project_color(dL, rgbv[leaf]), cur_tb, cur_seed, p, Gq, Bq,
                                       dL, v);
                c = true;
            }
        }
        unsigned long long rem = __ballot(c);
        while (rem != 0ULL) {  // one record per view among the contributing lanes (normally one)
            const int vw = __builtin_amdgcn_readlane(view, __ffsll((long long)rem) - 1);
            const bool mine = c && view == vw;
            float w[kMoments];
#pragma unroll
            for (int k = 0; k < kMoments; ++k) w[k] = mine ? v[k] : 0.0f;
            grad_scatter_wave(w, vw * sc.n + leaf, sc, gr, lane, G, st, drops);
            rem &= ~__ballot(mine);
        }
        idx = miss;
    }
}

// Backward of one ray per lane, called by all 64 lanes of the wave together (inactive lanes pass
// active = false).  Each outer iteration every live lane prepares its next slab that has hits
// (recomputed buffers, per-sample coefficients, T and the colour remainder advanced); then the
// wave walks the union of the prepared slabs' hits in increasing (view, slot) order and scatters
// one summed contribution per Gaussian.  Slabs served by per-slab traversal scatter per lane.
template <int SPB, int CAP, bool RNG, int RM>
__device__ void backward_wave(const DevScene& sc, const DevParams& p, bool active, const Ray& ray, unsigned int seed,
                              const float4* __restrict__ rgbv, const float* Cfwd, const float* dL, IList<CAP>& L,
                              GradStage& G, int lane, const DevGrad& gr, int view, Counters& ctr, Rec& rc,
                              unsigned long long* drops) {
    Staged st;  // records in the staging area
    bool alive = active && (ray.tenter < ray.texit) && (add_exact(ray.tenter, p.dt * (float)p.spb) > ray.tenter);
    float T = 1.0f;
    float Dr = dL[0] * Cfwd[0] + dL[1] * Cfwd[1] + dL[2] * Cfwd[2];  // dLdC . (colour not yet composited)
    SegState s;
    seg_init(s, ray, p);
    const int key_base = view * sc.n;
    // lanes within p.bwd_window slabs of the laggard step together (half a slab at 1M Gaussians:
    // 4 % faster than one, the same as a quarter; one slab 12 % faster on a 300k-Gaussian batch)
    const float window = p.bwd_window * p.dt * (float)p.spb;
    bool pend = false;  // next_slab() has produced a slab not yet processed
    bool jump = false;  // the last round found no hit in any lane's slab (jump_empty)
    float tmin = 0.0f, tmax = 0.0f;
    while (__ballot(alive) != 0ULL) {
        if (jump)
            jump_empty<CAP>(s, ray, p, L, lane, alive && !pend && s.valid && !s.direct, alive, rc.w ? s.knext : INT_MAX);
        // prepared slab: list mode (has: cur_cnt list entries) or per-slab traversal (dsc)
        bool has = false, dsc = false, prepped = false;
        float cur_tb = 0.0f, cur_tmin = 0.0f, cur_tmax = 0.0f;
        unsigned int cur_seed = 0u;
        int cur_cnt = 0;
        bool cur_dlist = false;  // the entries are a direct slab's recorded hits (all in the slab)
        int cur_dpos = 0;
        unsigned int cur_m = 0u;  // list mode: the entries in the slab (slab_mask), not yet scattered
        // the prepared slab's density and projected colour sums; after slab_coeffs the per-sample
        // backward coefficients G_i, Bq_i read by the scatter below
        float sig[SPB], ep[SPB];
        if (alive && !pend) {
            if (!(T > p.t_eps)) {
                alive = false;
            } else {
                sync_gathers(s, ray, p, rc.w == nullptr);
                if (!next_slab<CAP, RM>(s, sc, p, ray, L, lane, ctr, tmin, tmax, rc)) alive = false;
                else pend = true;
            }
        }
        // depth synchronisation: the wave's merged scatter only pays off when the lanes' current
        // slabs are at similar depth (similar Gaussians), so lanes ahead of the laggard wait
        const float tsync = wave_min64f(alive && pend ? s.tb : INFINITY);
        if (alive && pend && s.tb <= tsync + window) {
            pend = false;
            prepped = true;
            {
                const float tb = s.tb;
#pragma unroll
                for (int i = 0; i < SPB; ++i) sig[i] = ep[i] = 0.0f;
                int nh = 0;
                auto add_hit = [&](const Isect& I, float sigma, int slot) {
                    float md[SPB];
                    sample_densities<SPB, RNG>(I, sigma, tb, seed, p, md);
                    accum_densities<SPB>(md, project_color(dL, rgbv[slot]), p, sig, ep);
                    ++nh;
                };
                auto direct_hit = [&](int slot) -> bool {
                    float4 g0, g1, g2, g3;
                    load_rec(sc.geo, slot, g0, g1, g2, g3);
                    Isect I;
                    if (!intersect(g0, g1, g2, g3, ray, I)) return true;
                    if (!overlaps(tmin, tmax, I.r1, I.r2)) return true;
                    refine_sampling(g0, g1, g2, g3, ray, I);
                    add_hit(I, g0.w, slot);
                    return true;
                };
                if (s.direct && RM == 2 && s.dcnt >= 0) {
                    // the forward's hits of this slab: they passed the exact test in the forward over
                    // this same ray (the token, the handle's generation and the row's (view, pixel)
                    // are checked), so only their sampling terms are computed, as for list entries
                    for (int i = 0; i < s.dcnt; ++i) {
                        const int slot = (int)*rec_at(rc, s.dpos + i);
                        if ((unsigned)slot < (unsigned)sc.n) {
                            float sigma;
                            const Isect I = entry_hit(sc, ray, slot, 0.0f, 0.0f, sigma);
                            add_hit(I, sigma, slot);
                        } else {
                            count_drop(drops);
                        }
                    }
                    s.dense = nh > CAP;
                } else if (s.direct) {
                    trav(p, sc, ray, tmin, tmax, direct_hit);
                    s.dense = nh > CAP;
                } else {
                    unsigned int m = slab_mask<CAP>(L, s.cnt, tmin, tmax, lane);
                    cur_m = m;
                    while (m != 0u) {
                        const int e = __builtin_ctz(m);
                        m &= m - 1u;
                        const int slot = L.g[e][lane];
                        float sigma;
                        const Isect I = entry_hit(sc, ray, slot, L.r1[e][lane], L.r2[e][lane], sigma);
                        add_hit(I, sigma, slot);
                    }
                }
                if (nh > 0) {
                    slab_coeffs<SPB>(sig, ep, p, T, Dr);
                    cur_tb = tb;
                    cur_seed = seed;
                    cur_tmin = tmin;
                    cur_tmax = tmax;
                    if (RNG && p.rnd_sample == 1) seed = skip_draws(seed, p.spb);  // the slab's draws are spent
                    if (s.direct && RM == 2 && s.dcnt >= 0) {
                        has = true;
                        cur_dlist = true;
                        cur_dpos = s.dpos;
                        cur_cnt = s.dcnt;
                    } else if (s.direct) {
                        dsc = true;
                    } else {
                        has = true;
                        cur_cnt = s.cnt;
                    }
                }
                if (!advance_slab(s, p)) alive = false;
            }
        }
        jump = __ballot(prepped) != 0ULL && __ballot(has || dsc) == 0ULL;
        // converged: slabs whose hit set overflowed the list scatter from a packet traversal
        if (__ballot(dsc) != 0ULL)
            direct_scatter_wave<SPB, RNG>(sc, p, dsc, ray, rgbv, cur_tb, cur_seed, cur_tmin, cur_tmax, sig, ep, dL, G,
                                     st, lane, gr, view, drops);
        // wave-merged scatter over the prepared slabs' list hits.  A lane's key (view * n + slot of
        // its next hit; INT_MAX when it has none) changes only when its hit is scattered, and the
        // following hit's slot is loaded ahead of that hit's arithmetic.
        int e = 0;
        auto dlist_key = [&]() -> int {
            while (e < cur_cnt) {
                const int sl = (int)*rec_at(rc, cur_dpos + e);
                if ((unsigned)sl < (unsigned)sc.n) return key_base + sl;
                ++e;  // an out-of-range slot was counted when the slab was prepared
            }
            return INT_MAX;
        };
        int my = INT_MAX;
        if (has && cur_dlist) my = dlist_key();
        else if (has && cur_m != 0u) my = key_base + L.g[__builtin_ctz(cur_m)][lane];  // slot order
        while (true) {
            const int mn = wave_min64(my);
            if (mn == INT_MAX) break;
            const bool act = (my == mn);
            float v[kMoments];
#pragma unroll
            for (int k = 0; k < kMoments; ++k) v[k] = 0.0f;
            if (act) {
                const int slot = mn - key_base;
                int nxt = -1;
                if (cur_dlist) {
                    if (e + 1 < cur_cnt) nxt = (int)*rec_at(rc, cur_dpos + e + 1);
                } else {
                    cur_m &= cur_m - 1u;
                    if (cur_m != 0u) nxt = L.g[__builtin_ctz(cur_m)][lane];
                }
                float4 g0, g1, g2, g3;
                load_rec(sc.geo, slot, g0, g1, g2, g3);
                Isect I;
                // a list entry or a recorded direct hit passed the exact test when it was gathered
                // or recorded, so only its sampling terms are computed (the same values, without the
                // roots)
                {
                    float b, c;
                    isect_terms(g0, g1, g2, g3, ray, I, b, c);
                    refine_sampling(g0, g1, g2, g3, ray, I);
                    float md[SPB];
                    sample_densities<SPB, RNG>(I, g0.w, cur_tb, cur_seed, p, md);
                    const float P[3] = {I.Px, I.Py, I.Pz}, D[3] = {I.Dx, I.Dy, I.Dz};
                    grad_moments<SPB, RNG>(P, D, g0.w, md, I.tc, project_color(dL, rgbv[slot]), cur_tb, cur_seed, p, sig,
                                           ep, dL, v);
                }
                if (cur_dlist) {
                    ++e;
                    my = (unsigned)nxt < (unsigned)sc.n ? key_base + nxt : dlist_key();
                } else {
                    my = cur_m != 0u ? key_base + nxt : INT_MAX;
                }
            }
            grad_scatter_wave(v, mn, sc, gr, lane, G, st, drops);
        }
    }
    stage_flush(G, st, sc, gr, lane, drops);
}

// Parts, of at least 4 rays, that each of the nw wavefronts left by the tile kernels is cut into: as many as
// the GPU holds at once, since with fewer the slowest wavefront is the launch.  64 random rays of a block of
// 128 of 1024 pixels, 4096 wavefronts of which every fifth or so is left, 300k Gaussians: train step 158 -> 104 ms.
// More parts than that only repeat work: 64 rays of 512-pixel blocks at 20k 41.9 -> 54.6 ms with four times as many.
__device__ __forceinline__ int wide_parts(const DevParams& p, int64_t nw) {
    int parts = 1;
    while (8 * parts <= p.rays_per_wave && 2 * parts * nw <= kWideBlocks) parts *= 2;
    return parts;
}

// The wavefront whose part a block takes next, as its place in p.wide (-1: none is left), and this lane's
// place among its rays (rays_per_wave: none).
__device__ __forceinline__ int64_t next_wide(const DevParams& p, int64_t nw, int parts, int lane, int& ray) {
    int i = 0;
    if (lane == 0) i = (int)atomicAdd(p.wide_count + 1, 1ull);
    i = __builtin_amdgcn_readfirstlane(i);
    if (i >= nw * parts) return -1;
    const int rays = p.rays_per_wave / parts;
    ray = lane < rays ? (i % parts) * rays + lane : p.rays_per_wave;
    return i / parts;
}

// Renders the work items below `end` of wavefront `wave`, one per lane (lane_ray: its place in the wavefront).
template <int SPB, int CAP, bool RNG, int RM>
__device__ __forceinline__ void forward_items(const DevScene& sc, const DevParams& p, const RayJob& job, int64_t wave,
                                              int64_t end, IList<CAP>& L, int lane, int lane_ray, float* __restrict__ out_rgb,
                                              float* __restrict__ out_depth, float* __restrict__ out_opac, DevStats st) {
    Counters ctr;
    RayRef q;
    const int64_t item = lane_ray < p.rays_per_wave ? wave_item(p, wave, lane_ray) : -1;
    const bool in = item >= 0 && item < end;
    const int rs = in ? resolve(job, item, q) : (int)RAY_NONE;
    if (rs == RAY_BAD) {
        forward_bad<RM>(p, q, item, st, out_rgb, out_depth, out_opac);
    } else if (rs == RAY_OK) {
        const rg_camera cam = job.cams[q.view];
        unsigned int seed = RNG ? tea4(p.iteration, (unsigned int)q.pixel) : 0u;
        const Ray ray = make_ray(cam, q.pixel, sc.box, p.t_near, p.t_far, RNG ? p.jitter : 0, &seed);
        RayOut o;
        Rec rc;
        if constexpr (RM == 1) {
            rc.w = rec_region(p, wave) + 8 * lane_ray;
            rc.stride = 8 * p.rays_per_wave;
            rc.end = p.rec_words;
        }
        forward_ray<SPB, CAP, RNG, RM>(sc, p, ray, seed, sc.rgb + (size_t)q.view * sc.n, L, lane, ctr, o, rc);
        if constexpr (RM == 1) ctr.rec_words += rc.pos;
        forward_finish<RM>(p, q, item, o, rc, ctr, out_rgb, out_depth, out_opac);
    } else if (RM == 1 && in) {
        p.rec_id[item] = make_int2(-1, -1);  // padding: no records
    }
    flush_counters(ctr, st);
}

// The wavefront of each block, or (p.wide) the wavefronts that the tile kernel left to the stepper.
template <int SPB, int CAP, bool RNG, int RM>
__global__ void __launch_bounds__(kWave) __attribute__((amdgpu_waves_per_eu(SPB == 8 ? 4 : 3))) k_forward(DevScene sc, DevParams p, RayJob job, int64_t num_items,
                                                   float* __restrict__ out_rgb, float* __restrict__ out_depth,
                                                   float* __restrict__ out_opac, DevStats st) {
    __shared__ IList<CAP> L;
    const int lane = threadIdx.x;
    const int64_t nw = p.wide ? (int64_t)*p.wide_count : 1;
    const int parts = p.wide ? wide_parts(p, nw) : 1;
    while (nw > 0) {
        int64_t wave = block_item(blockIdx.x, gridDim.x);
        int ray = lane;
        if (p.wide) {
            const int64_t i = next_wide(p, nw, parts, lane, ray);
            if (i < 0) return;
            wave = p.wide[i].x;
        }
        forward_items<SPB, CAP, RNG, RM>(sc, p, job, wave, num_items, L, lane, ray, out_rgb, out_depth, out_opac, st);
        if (!p.wide) return;
    }
}

// Backward of the work items below `end` of wavefront `wave`, one per lane (lane_ray); lanes: those that take part
// (the rest were done by the tile kernel, with the loss and the bad rays of all of them).
template <int SPB, int CAP, bool RNG, int RM>
__device__ __forceinline__ void backward_items(const DevScene& sc, const DevParams& p, const RayJob& job, int64_t wave,
                                               int64_t end, unsigned long long lanes, IList<CAP>& L, GradStage& G, int lane,
                                               int lane_ray, const float* __restrict__ ray_colors, const float* __restrict__ dLdC,
                                               const float* __restrict__ target, int loss_kind, int count_stats,
                                               const DevGrad& gr, DevStats st) {
    Counters ctr;
    float loss = 0.0f;
    BwdRay b;
    const int64_t item = lane_ray < p.rays_per_wave ? wave_item(p, wave, lane_ray) : -1;
    if (item >= 0 && item < end && ((lanes >> lane_ray) & 1ULL))
        backward_setup<RNG, RM>(sc, p, job, wave, lane_ray, item, ray_colors, dLdC, target, loss_kind, st, b, loss);
    backward_wave<SPB, CAP, RNG, RM>(sc, p, b.active, b.ray, b.seed, sc.rgb + (size_t)b.view * sc.n, b.Cf, b.dL, L, G,
                                     lane, gr, b.view, ctr, b.rc, st.c + C_DROP);
    if (count_stats) flush_counters(ctr, st);
    if (target && !p.wide) add_loss(p, loss, lane, st);
}

// Backward over a batch.  dL/dC comes from dLdC, or -- with target != nullptr -- from the
// per-pixel loss of the rendered colours against target (loss_kind 0: L2 sum (C-t)^2, 1: L1
// sum |C-t|), whose value is summed into the loss counter.  count_stats = 0 leaves the
// traversal counters to the forward of the same step.
template <int SPB, int CAP, bool RNG, int RM>
__global__ void __launch_bounds__(kWave) __attribute__((amdgpu_waves_per_eu(3))) k_backward(DevScene sc, DevParams p, RayJob job, int64_t num_items,
                                                    const float* __restrict__ ray_colors, const float* __restrict__ dLdC,
                                                    const float* __restrict__ target, int loss_kind, int count_stats,
                                                    DevGrad gr, DevStats st) {
    __shared__ IList<CAP> L;
    __shared__ GradStage G;
    const int lane = threadIdx.x;
    const int64_t nw = p.wide ? (int64_t)*p.wide_count : 1;
    const int parts = p.wide ? wide_parts(p, nw) : 1;
    while (nw > 0) {
        int64_t wave = block_item(blockIdx.x, gridDim.x);
        int ray = lane;
        unsigned long long lanes = ~0ULL;
        if (p.wide) {
            const int64_t i = next_wide(p, nw, parts, lane, ray);
            if (i < 0) return;
            const int4 w = p.wide[i];
            wave = w.x;
            lanes = (unsigned long long)(unsigned int)w.y | (unsigned long long)(unsigned int)w.z << 32;
        }
        backward_items<SPB, CAP, RNG, RM>(sc, p, job, wave, num_items, lanes, L, G, lane, ray, ray_colors, dLdC, target,
                                          loss_kind, count_stats, gr, st);
        if (!p.wide) return;
    }
}

// Persistent forward over whole tiles: each wavefront takes chunks from the queues and renders
// them one tile (64 rays, one per lane) at a time, exactly as k_forward renders its tile.
template <int SPB, int CAP, bool RNG, int RM>
__global__ void __launch_bounds__(kWave) __attribute__((amdgpu_waves_per_eu(SPB == 8 ? 4 : 3)))
k_forward_pq(DevScene sc, DevParams p, RayJob job, int64_t num_items, float* __restrict__ out_rgb,
             float* __restrict__ out_depth, float* __restrict__ out_opac, DevStats st) {
    __shared__ IList<CAP> L;
    const int lane = threadIdx.x;
    int64_t lo = 0, hi = 0;
    unsigned int spent = 0u;
    while (take_chunk(p, num_items, blockIdx.x & 7, lo, hi, spent))
        for (int64_t base = lo; base < hi; base += kWave)  // counters are flushed per tile
            forward_items<SPB, CAP, RNG, RM>(sc, p, job, base / kWave, hi, L, lane, lane, out_rgb, out_depth, out_opac, st);
}

// Persistent forward that refills idle lanes (refill_lanes = k, 0 < k < 64): as soon as k lanes
// are done they take the next rays of the chunk (and further chunks).  A lane's ray advances one
// slab per wave step (forward_step), but a refilled lane starts at the scene box while the others
// are deeper in, so the wavefront's lanes no longer query similar ray segments and its packet
// traversals visit the union of two depth ranges: measured slower than whole tiles on the
// 1M-Gaussian workload, kept as a tuning option.
template <int SPB, int CAP, bool RNG, int RM>
__global__ void __launch_bounds__(kWave) __attribute__((amdgpu_waves_per_eu(SPB == 8 ? 4 : 3)))
k_forward_refill(DevScene sc, DevParams p, RayJob job, int64_t num_items, float* __restrict__ out_rgb,
                 float* __restrict__ out_depth, float* __restrict__ out_opac, DevStats st) {
    __shared__ IList<CAP> L;
    const int lane = threadIdx.x;
    const int xcd = blockIdx.x & 7;
    const int refill = p.refill_lanes;
    Counters ctr;
    int64_t clo = 0, chi = 0;  // items of the current chunk not yet handed out (wave-uniform)
    unsigned int spent = 0u;
    bool more = true;          // the queues may hold more items (wave-uniform)
    bool alive = false;        // this lane holds a ray that is not done
    RayRef q;
    q.view = 0;
    q.pixel = 0;
    q.out = 0;
    q.active = false;
    Ray ray = {};
    unsigned int seed = 0u;
    SegState s;
    seg_init(s, ray, p);
    RayOut o;
    o.C[0] = o.C[1] = o.C[2] = 0.0f;
    o.depth = 0.0f;
    o.T = 1.0f;
    Rec rc;
    int64_t item = 0;
    while (true) {
        if (more && __popcll(__ballot(!alive)) >= refill) {
            // hand the next items to the idle lanes, taking chunks from the queues as needed
            bool need = !alive;
            while (true) {
                const unsigned long long nm = __ballot(need);
                if (nm == 0ull) break;
                if (clo >= chi && !take_chunk(p, num_items, xcd, clo, chi, spent)) {
                    more = false;
                    break;
                }
                const int64_t avail = chi - clo;
                const int rank = lanes_below(nm);
                if (need && rank < avail) {
                    need = false;
                    item = clo + rank;
                    const int rs = resolve(job, item, q);
                    if (rs == RAY_OK) {
                        const rg_camera cam = job.cams[q.view];
                        seed = RNG ? tea4(p.iteration, (unsigned int)q.pixel) : 0u;
                        ray = make_ray(cam, q.pixel, sc.box, p.t_near, p.t_far, RNG ? p.jitter : 0, &seed);
                        if constexpr (RM == 1) {
                            rc.w = rec_region(p, item / kWave) + 8 * (item % kWave);
                            rc.pos = 0;
                            rc.end = p.rec_words;
                            rc.full = false;
                        }
                        alive = forward_begin(p, ray, o);
                        seg_init(s, ray, p);
                        if (!alive) forward_finish<RM>(p, q, item, o, rc, ctr, out_rgb, out_depth, out_opac);
                    } else if (rs == RAY_BAD) {
                        forward_bad<RM>(p, q, item, st, out_rgb, out_depth, out_opac);
                    }
                }
                clo += min((int64_t)__popcll(nm), avail);
            }
        }
        if (__ballot(alive) == 0ull) {
            if (!more) break;
            continue;
        }
        if (alive && !forward_step<SPB, CAP, RNG, RM>(sc, p, ray, seed, sc.rgb + (size_t)q.view * sc.n, L, lane, ctr, o,
                                                      rc, s)) {
            if constexpr (RM == 1) ctr.rec_words += rc.pos;
            forward_finish<RM>(p, q, item, o, rc, ctr, out_rgb, out_depth, out_opac);
            alive = false;
        }
    }
    flush_counters(ctr, st);
}

// Persistent backward: each wavefront takes chunks of whole tiles from the queues and runs the
// depth-synchronised, wave-merged backward on one tile (64 rays) at a time.
template <int SPB, int CAP, bool RNG, int RM>
__global__ void __launch_bounds__(kWave) __attribute__((amdgpu_waves_per_eu(3)))
k_backward_pq(DevScene sc, DevParams p, RayJob job, int64_t num_items, const float* __restrict__ ray_colors,
              const float* __restrict__ dLdC, const float* __restrict__ target, int loss_kind, int count_stats,
              DevGrad gr, DevStats st) {
    __shared__ IList<CAP> L;
    __shared__ GradStage G;
    const int lane = threadIdx.x;
    const int xcd = blockIdx.x & 7;
    int64_t lo = 0, hi = 0;
    unsigned int spent = 0u;
    while (take_chunk(p, num_items, xcd, lo, hi, spent))
        for (int64_t base = lo; base < hi; base += kWave)  // counters are flushed per tile
            backward_items<SPB, CAP, RNG, RM>(sc, p, job, base / kWave, hi, ~0ULL, L, G, lane, lane, ray_colors, dLdC, target,
                                              loss_kind, count_stats, gr, st);
}

__global__ void k_reset_queue(unsigned long long* q) {
    if (threadIdx.x < 8) q[threadIdx.x] = 0ull;
}

// Verification: per-slab hit sets from the same traversal + predicate (every slab to texit).
__global__ void __launch_bounds__(kWave) k_debug_hits(DevScene sc, DevParams p, RayJob job, int max_slabs,
                                                      int max_pairs, int32_t* pairs, int64_t* counts, float* ro,
                                                      float* rd, float* te, float* tx) {
    const int64_t r = (int64_t)blockIdx.x * kWave + threadIdx.x;
    if (r >= job.num_rays) return;
    RayRef q;
    if (job.pixels || job.ray_view) {
        if (resolve(job, r, q) != RAY_OK) {
            counts[r] = 0;
            return;
        }
    } else {  // no pixel list: ray r is pixel r (row-major)
        q.view = job.view;
        q.pixel = (int)r;
    }
    const rg_camera cam = job.cams[q.view];
    unsigned int seed = tea4(p.iteration, (unsigned int)q.pixel);
    const Ray ray = make_ray(cam, q.pixel, sc.box, p.t_near, p.t_far, p.jitter, &seed);
    ro[3 * r] = ray.ox;
    ro[3 * r + 1] = ray.oy;
    ro[3 * r + 2] = ray.oz;
    rd[3 * r] = ray.dx;
    rd[3 * r + 1] = ray.dy;
    rd[3 * r + 2] = ray.dz;
    te[r] = ray.tenter;
    tx[r] = ray.texit;
    int64_t n = 0;
    if (ray.tenter < ray.texit) {
        const float slab = p.dt * (float)p.spb;
        float tb = ray.tenter;
        for (int s = 0; s < max_slabs && tb < ray.texit; ++s) {
            const float tmin = fmaxf(ray.tenter, tb);
            const float tmax = fminf(ray.texit, add_exact(tb, slab));
            if (tmax > ray.tenter) {
                trav(p, sc, ray, tmin, tmax, [&](int slot) -> bool {
                    float4 g0, g1, g2, g3;
                    load_rec(sc.geo, slot, g0, g1, g2, g3);
                    Isect I;
                    if (intersect(g0, g1, g2, g3, ray, I) && overlaps(tmin, tmax, I.r1, I.r2)) {
                        if (n < max_pairs) {
                            pairs[(r * max_pairs + n) * 2] = s;
                            pairs[(r * max_pairs + n) * 2 + 1] = sc.perm[slot];
                        }
                        ++n;
                    }
                    return true;
                });
            }
            const float nt = add_exact(tb, slab);
            if (!(nt > tb)) break;
            tb = nt;
        }
    }
    counts[r] = n;
}

__global__ void k_reset_counters(unsigned long long* c) {
    if (threadIdx.x < kCounters) c[threadIdx.x] = 0;
}

__global__ void k_loss_out(const unsigned long long* c, float* out) {
    if (threadIdx.x == 0)
        *out = (float)((double)*reinterpret_cast<const float*>(&c[C_LOSS]) + *reinterpret_cast<const double*>(&c[C_LOSS64]));
}

}  // namespace

// In the implicit single-view mode RayJob.num_rays carries the padded 8x8-tile item count.
#define RG_DISPATCH_CAP(SPBC, RNGC, RMC, CAPV, KERNEL, ...)                                                       \
    do {                                                                                                             \
        if (CAPV <= 8) hipLaunchKernelGGL((KERNEL<SPBC, 8, RNGC, RMC>), __VA_ARGS__);                                \
        else if (CAPV <= 16) hipLaunchKernelGGL((KERNEL<SPBC, 16, RNGC, RMC>), __VA_ARGS__);                         \
        else hipLaunchKernelGGL((KERNEL<SPBC, 32, RNGC, RMC>), __VA_ARGS__);                                         \
    } while (0)
#define RG_DISPATCH_CAP6(SPBC, RNGC, RMC, CAPV, KERNEL, ...)                                                      \
    do {                                                                                                             \
        if (CAPV <= 6) hipLaunchKernelGGL((KERNEL<SPBC, 6, RNGC, RMC>), __VA_ARGS__);                                \
        else if (CAPV <= 12) hipLaunchKernelGGL((KERNEL<SPBC, 12, RNGC, RMC>), __VA_ARGS__);                         \
        else if (CAPV <= 16) hipLaunchKernelGGL((KERNEL<SPBC, 16, RNGC, RMC>), __VA_ARGS__);                         \
        else hipLaunchKernelGGL((KERNEL<SPBC, 32, RNGC, RMC>), __VA_ARGS__);                                         \
    } while (0)
// Kernels are specialised on SPB (8 samples per slab, or any number up to 16), the list capacity, on whether the
// random generator is used at all (jitter or rnd_sample), which costs registers, and on the
// hit-list record mode (RMV: 0 none, or the kernel's recording / replaying mode), so that kernels
// without records carry none of their code.
#define RG_DISPATCH_ANY(CAPMACRO, SPBV, CAPV, RNGV, RMV, RMON, KERNEL, ...)                                         \
    do {                                                                                                             \
        if (RMV) {                                                                                                   \
            if (SPBV == 8) {                                                                                         \
                if (RNGV) CAPMACRO(8, true, RMON, CAPV, KERNEL, __VA_ARGS__);                                        \
                else CAPMACRO(8, false, RMON, CAPV, KERNEL, __VA_ARGS__);                                            \
            } else {                                                                                                 \
                if (RNGV) CAPMACRO(16, true, RMON, CAPV, KERNEL, __VA_ARGS__);                                       \
                else CAPMACRO(16, false, RMON, CAPV, KERNEL, __VA_ARGS__);                                           \
            }                                                                                                        \
        } else {                                                                                                     \
            if (SPBV == 8) {                                                                                         \
                if (RNGV) CAPMACRO(8, true, 0, CAPV, KERNEL, __VA_ARGS__);                                           \
                else CAPMACRO(8, false, 0, CAPV, KERNEL, __VA_ARGS__);                                               \
            } else {                                                                                                 \
                if (RNGV) CAPMACRO(16, true, 0, CAPV, KERNEL, __VA_ARGS__);                                          \
                else CAPMACRO(16, false, 0, CAPV, KERNEL, __VA_ARGS__);                                              \
            }                                                                                                        \
        }                                                                                                            \
    } while (0)
#define RG_DISPATCH(SPBV, CAPV, RNGV, RMV, ...) RG_DISPATCH_ANY(RG_DISPATCH_CAP, SPBV, CAPV, RNGV, RMV, 2, __VA_ARGS__)
#define RG_DISPATCH_FWD(SPBV, CAPV, RNGV, RMV, ...) \
    RG_DISPATCH_ANY(RG_DISPATCH_CAP6, SPBV, CAPV, RNGV, RMV, 1, __VA_ARGS__)

hipError_t launch_loss_out(DevStats st, float* out, hipStream_t s) {
    hipLaunchKernelGGL(k_loss_out, dim3(1), dim3(64), 0, s, st.c, out);
    return hipGetLastError();
}

hipError_t launch_reset_counters(DevStats st, hipStream_t s) {
    hipLaunchKernelGGL(k_reset_counters, dim3(1), dim3(128), 0, s, st.c);
    return hipGetLastError();
}

// Number of wavefronts a persistent kernel is launched with: as many as the GPU holds at once
// (occupancy x CUs, a multiple of 8 so that every XCD gets the same number), and no more than
// there are chunks of work.
template <typename K>
static int64_t persistent_grid(K kernel, int64_t chunks) {
    int dev = 0, cus = 0, per_cu = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
        cus = 256;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, reinterpret_cast<const void*>(kernel), kWave, 0) !=
            hipSuccess ||
        per_cu <= 0)
        per_cu = 1;
    const int64_t resident = (int64_t)cus * per_cu;
    int64_t g = chunks < resident ? chunks : resident;
    g = ((g + 7) / 8) * 8;
    return g > 0 ? g : 8;
}

template <typename K, typename... A>
static void launch_persistent(K kernel, int64_t items, const DevParams& p, hipStream_t s, A... args) {
    const int64_t chunks = (items + p.ray_chunk - 1) / p.ray_chunk;
    hipLaunchKernelGGL(k_reset_queue, dim3(1), dim3(64), 0, s, p.queue);
    hipLaunchKernelGGL(kernel, dim3((unsigned)persistent_grid(kernel, chunks)), dim3(kWave), 0, s, args...);
}

#define RG_PQ_CAP(SPBC, RNGC, RMC, CAPV, KERNEL, ...)                                                           \
    do {                                                                                                             \
        if (CAPV <= 8) launch_persistent(KERNEL<SPBC, 8, RNGC, RMC>, __VA_ARGS__);                                  \
        else if (CAPV <= 16) launch_persistent(KERNEL<SPBC, 16, RNGC, RMC>, __VA_ARGS__);                           \
        else launch_persistent(KERNEL<SPBC, 32, RNGC, RMC>, __VA_ARGS__);                                           \
    } while (0)
#define RG_PQ_CAP6(SPBC, RNGC, RMC, CAPV, KERNEL, ...)                                                          \
    do {                                                                                                             \
        if (CAPV <= 6) launch_persistent(KERNEL<SPBC, 6, RNGC, RMC>, __VA_ARGS__);                                  \
        else if (CAPV <= 12) launch_persistent(KERNEL<SPBC, 12, RNGC, RMC>, __VA_ARGS__);                           \
        else if (CAPV <= 16) launch_persistent(KERNEL<SPBC, 16, RNGC, RMC>, __VA_ARGS__);                           \
        else launch_persistent(KERNEL<SPBC, 32, RNGC, RMC>, __VA_ARGS__);                                           \
    } while (0)

// Blocks of a stepper launch: one per wavefront, or as many as take the tile kernel's leftovers in
// turn (their number is known on the device alone; none is the common case).
static unsigned int step_blocks(const DevParams& p, int64_t items) {
    const int64_t nb = num_waves(p, items) * (p.wide ? (p.rays_per_wave + 3) / 4 : 1);
    return (unsigned int)(p.wide ? (nb < kWideBlocks ? nb : kWideBlocks) : ((nb + 7) / 8) * 8);
}

hipError_t launch_forward_steps(const DevScene& sc, const DevParams& p, const RayJob& job, int hit_depth, float* out_rgb,
                                float* out_depth, float* out_opacity, DevStats st, hipStream_t s) {
    const int64_t items = job.num_rays;  // already the padded item count in implicit mode
    if (items <= 0) return hipSuccess;
    const bool rng = p.jitter || p.rnd_sample;
    if (p.ray_chunk > 0 && !p.wide && p.refill_lanes > 0 && p.refill_lanes < kWave) {
        RG_DISPATCH_ANY(RG_PQ_CAP6, p.spb == 8 ? 8 : 16, hit_depth, rng, p.rec_mode == 1, 1, k_forward_refill, items, p,
                        s, sc, p, job, items, out_rgb, out_depth, out_opacity, st);
        return hipGetLastError();
    }
    if (p.ray_chunk > 0 && !p.wide) {
        RG_DISPATCH_ANY(RG_PQ_CAP6, p.spb == 8 ? 8 : 16, hit_depth, rng, p.rec_mode == 1, 1, k_forward_pq, items, p, s,
                        sc, p, job, items, out_rgb, out_depth, out_opacity, st);
        return hipGetLastError();
    }
    RG_DISPATCH_FWD(p.spb == 8 ? 8 : 16, hit_depth, rng, p.rec_mode == 1, k_forward, dim3(step_blocks(p, items)), dim3(kWave),
                    0, s, sc, p, job, items, out_rgb, out_depth, out_opacity, st);
    return hipGetLastError();
}

hipError_t launch_backward_steps(const DevScene& sc, const DevParams& p, const RayJob& job, int hit_depth,
                                 const float* ray_colors, const float* dLdC, const float* target, int loss_kind,
                                 int count_stats, DevGrad gr, DevStats st, hipStream_t s) {
    const int64_t items = job.num_rays;
    if (items <= 0) return hipSuccess;
    const bool rng = p.jitter || p.rnd_sample;
    if (p.ray_chunk > 0 && !p.wide) {
        RG_DISPATCH_ANY(RG_PQ_CAP, p.spb == 8 ? 8 : 16, hit_depth, rng, p.rec_mode == 2, 2, k_backward_pq, items, p, s,
                        sc, p, job, items, ray_colors, dLdC, target, loss_kind, count_stats, gr, st);
        return hipGetLastError();
    }
    RG_DISPATCH(p.spb == 8 ? 8 : 16, hit_depth, rng, p.rec_mode == 2, k_backward, dim3(step_blocks(p, items)), dim3(kWave), 0, s,
                sc, p, job, items, ray_colors, dLdC, target, loss_kind, count_stats, gr, st);
    return hipGetLastError();
}

hipError_t launch_debug_hits(const DevScene& sc, const DevParams& p, const RayJob& job, int max_slabs, int max_pairs,
                             int32_t* pairs, int64_t* counts, float* ro, float* rd, float* te, float* tx,
                             hipStream_t s) {
    if (job.num_rays <= 0) return hipSuccess;
    const int64_t nb = (job.num_rays + kWave - 1) / kWave;
    hipLaunchKernelGGL(k_debug_hits, dim3((unsigned)nb), dim3(kWave), 0, s, sc, p, job, max_slabs, max_pairs, pairs,
                       counts, ro, rd, te, tx);
    return hipGetLastError();
}

}  // namespace rg
