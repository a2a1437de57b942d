// engine_scene.hip -- SCENE engine: one workgroup runs a whole scene.
//
// A persistent kernel takes scenes from a work queue (largest first).  For
// each scene the workgroup keeps positions and previous positions in LDS
// when both fit the LDS budget, positions alone when only they fit, or works
// from global memory; it runs all updates and substeps of the launch with
// workgroup barriers between dependent phases (src/solver.rs:106-116):
//
//   links     dependency layers streamed from global memory, a barrier
//             between layers (src/solver.rs:143-153)
//   circles   exact replay of the (i, j) lexicographic pair sweep
//             (src/solver.rs:168-177) from per-circle candidate lists: a
//             round runs every pair whose earlier pairs (sharing a circle)
//             are done; a sweep stands when no pair missing from the lists
//             can have touched at its turn, else it is undone and rerun with
//             new lists (circle_sweep)
//   bodies    EXT4 static colliders, bounds, Verlet
//             (src/solver.rs:155-165, 118-128)
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <cstring>
#include <memory>
#include <mutex>
#include <vector>

#include "../../include/bendy2d.h"
#include "common.h"
#include "engine.h"
#include "bodies.h"
#include "kernels.h"
#include "pack.h"
#include "scene_pack.h"

namespace bd {

// Orders one wavefront's memory operations between its lanes: a wavefront's
// LDS and vector memory instructions execute in order, so keeping the
// compiler from moving them across this point is all that is needed.
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// A pointer into LDS, typed as such: the low 32 bits of a generic LDS address
// are its LDS offset.  Accesses through it are LDS instructions, where a
// generic pointer takes flat ones (slower, and counted against both the LDS
// and the vector-memory wait counters).
#define BD_LDS __attribute__((address_space(3)))
template <typename T>
__device__ __forceinline__ BD_LDS T *to_lds(T *p) {
    return (BD_LDS T *)(uint32_t)(uint64_t)p;
}


template <int WG>
__device__ __forceinline__ float wg_max(float v, float *s_red) {
    for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o, 64));
    const int wave = threadIdx.x >> 6;
    __syncthreads();
    if ((threadIdx.x & 63) == 0) s_red[wave] = v;
    __syncthreads();
    float m = s_red[0];
#pragma unroll 2
    for (int w = 1; w < WG / 64; w++) m = fmaxf(m, s_red[w]);
    return uni(m);
}

// inclusive prefix sum over the lanes of the wavefront, all lanes active
// (ROCm's device library: a row-shift and row-broadcast sequence)
extern "C" __device__ uint32_t __ockl_wfscan_add_u32(uint32_t, bool);

// Exclusive scan of a[0..n) into out[0..n] (out[n] the total) in global memory by
// one workgroup; out may be a.
template <int WG>
__device__ void wg_scan_global(const uint32_t *a, uint32_t *out, uint32_t n, uint32_t *s_wave) {
    uint32_t carry = 0;
    // The wave index is uniform and the lane scan takes no lane masks: the
    // loops over the waves below are scalar loops, and no per-lane compare
    // stays live for the whole kernel.
    const int lane = threadIdx.x & 63;
    const uint32_t wave = uni(threadIdx.x >> 6);
    for (uint32_t base = 0; base < n; base += WG * 4) {
        uint32_t i0 = base + threadIdx.x * 4;
        uint32_t v[4], local = 0;
        for (int k = 0; k < 4; k++) { v[k] = (i0 + k < n) ? a[i0 + k] : 0u; local += v[k]; }
        const uint32_t inc = __ockl_wfscan_add_u32(local, true);
        __syncthreads();
        if (lane == 63) s_wave[wave] = inc;
        __syncthreads();
        uint32_t woff = 0, total = 0;
#pragma unroll 1
        for (uint32_t w = 0; w < wave; w++) woff += s_wave[w];
        total = woff;
#pragma unroll 1
        for (uint32_t w = wave; w < WG / 64; w++) total += s_wave[w];
        uint32_t run = carry + woff + inc - local;
        for (int k = 0; k < 4; k++) {
            if (i0 + k < n) out[i0 + k] = run;
            run += v[k];
        }
        carry += total;
    }
    if (threadIdx.x == 0) out[n] = carry;
    __syncthreads();
}

// Upper bound on how far a circle can have been from its list-build position
// `r0` during a sweep that started at `p` and took it at most `path` away from
// `p` (its largest excursion, see below).  A circle at a non-finite position
// takes part in no pair (every comparison with it is false), so it cannot
// invalidate the list; one whose list-build position was non-finite but is
// finite now forces a rebuild.
//
// The bound is taken relative to a common shift u of the whole scene: for a
// pair, |(p_i - r_i) - (p_j - r_j)| <= |p_i - r_i - u| + |p_j - r_j - u| for
// any fixed u, so bulk motion (a falling body) does not count.
__device__ __forceinline__ float moved_bound(float2 p, float2 r0, float2 u, float path) {
    if (!(fabsf(p.x) <= 3.0e38f) || !(fabsf(p.y) <= 3.0e38f)) return 0.0f;
    if (!(fabsf(r0.x) <= 3.0e38f) || !(fabsf(r0.y) <= 3.0e38f)) return INFINITY;
    float dx = (p.x - r0.x) - u.x, dy = (p.y - r0.y) - u.y;
    float v = sqrtf(dx * dx + dy * dy) + path;
    return v == v ? v : INFINITY;
}


__device__ __forceinline__ int scell(float x, double inv_h) {
    double c = floor((double)x * inv_h);
    if (!(c > -1073741824.0)) c = -1073741824.0;
    if (c > 1073741824.0) c = 1073741824.0;
    return (int)c;
}

// The circle-pair workspace of a scene, in its chunk (layout: cc_layout).
struct CCWork {
    float2 *ref, *save;
    float *path, *skin, *need;
    uint32_t *cnt, *off;
    uint16_t *cand;
    float2 *traj;  // per list entry: the circle's position after that pair ran
    uint32_t *head, *stamp, *wl, *key;
    float4 *rec;  // circles in bucket order: x, y, radius + skin, index (| kOutlierBit)
    uint32_t *start, *fill, *items;
};

constexpr uint32_t kOutlierBit = 0x80000000u;

constexpr uint32_t kOutCap = 512;   // circles with an outlying skin, per list build
constexpr uint32_t kMidList = 256;  // longer candidate lists are sorted by the whole workgroup
constexpr uint32_t kSlot = 24;      // normal partners kept from the counting pass (more are gathered again)
static_assert(2 * kSlot <= 8 * kCandCap, "count-pass slots must fit in the trajectory array");
constexpr uint32_t kNone = 0xffffffffu;
// sweeps with at least this many candidate pairs park previous positions (or
// positions) in global memory to hold their round state in LDS
constexpr uint32_t kParkPairs = 32;
// Failed attempts at a sweep after which it runs sequentially instead.
constexpr int kFallbackAttempt = 4;
// Sweeps after such a fallback that run sequentially without trying lists.
constexpr uint32_t kFallbackStreak = 16;
// A circle has drifted once it is further than this fraction of its skin from
// its list-build position (relative to a common shift of the scene): the
// fraction that a valid sweep may use.  A list is rebuilt before a sweep when
// more than kDriftedBase + Nc / kDriftedShare circles have, or one of those has
// come into reach of a circle it does not list; else the sweep's check looks at
// each of them on its own.  A few circles shot out of a
// collider or a pile move by more than any skin every substep, and brought a new
// list each time (20 to 320 us, against about 1 us a circle for the check).
constexpr float kDriftRebuild = 0.8f;
// With fewer than kDriftedLeast circles a list costs no more than one check (10 us)
// and saves the checks of the sweeps that follow (a dropped 12 x 12 body, 14
// updates, eight of them: 5 to 36 % shorter; at 361 circles as often longer).
constexpr uint32_t kDriftedBase = 8u, kDriftedShare = 64u, kDriftedLeast = 256u;

// FbGrid: bucket heads (u16, tmask + 1 of them, 0xffff for an empty bucket),
// per-circle next links (u16) and a candidate buffer of cap entries (u16): in
// LDS when the scene leaves room, else in the workspace.  A circle's bucket
// is always that of its current position, so it is not stored.
struct FbGrid {
    uint16_t *head;
    uint16_t *next, *cand;
    uint32_t tmask, cap;
};

struct CCShared {
    CCWork work;
    uint16_t out[kOutCap];   // outlier circles of the current list
    uint32_t hist[33];       // skins by log2(skin / base)
    uint32_t nout;
    uint32_t nmid, nlong;    // candidate lists sorted by a wavefront / by the workgroup
    uint32_t nact;           // slots of the sweep's active lists handed out (see prune_lists)
    uint32_t nnear, stalled; // circles beyond their active margins; a list left unfinished
    const uint16_t *act;     // the sweep's active lists (LDS or workspace)
    uint32_t halt;           // the scene's time budget for this launch is spent
    float4 red4[32];         // the wavefronts' drift boxes and sums (see drift_box)
    uint32_t cnt3[3];        // worklist lengths, rotating (see the round loop)
    uint32_t poly_last[3];   // polygon pairs: see poly_pair_loop
    // LDS the sequential fallback may use for its grid: the scene's previous
    // positions when they are held in LDS (parked in q_global meanwhile), or
    // what the positions leave of the launch's LDS
    struct Fallback {
        uint8_t *lds;
        uint32_t lds_bytes, nq;
        float2 *q_lds, *q_global;
        float2 *p_global;  // positions' global copy when they are in LDS without prev (MODE 1)
    } fb;
    uint32_t free_off, free_bytes;  // dynamic LDS past what the scene keeps there
    FbGrid grid;             // the fallback's grid (see sequential_sweep)
    uint32_t fb_streak;      // sweeps left that go straight to the fallback
    // the scene's schedule between sweeps: its base skin, whether the candidate
    // list holds, that list's pairs, the sweeps since it was built, its outlier
    // threshold and its smallest skin.  Written by lane 0 at the end of a sweep,
    // read at the start of the next (barriers lie between).
    struct Steer {
        float skin;
        uint32_t list_valid, pairs, since_build;
        float s_cell, smin;
        uint32_t level;   // of the active margins' base (see kActiveBase)
        uint32_t clean;   // sweeps since a margin was too small
        uint32_t heat;    // second runs of late (see kHeatMiss)
    } cs;
    // statistics of the scene during a launch, written by lane 0 only (in LDS
    // rather than in every lane's registers)
    struct Counts {
        uint32_t rounds, redos, rebuilds, kept, unchecked, n_out, n_far, max_list, fallbacks;
        float smax;
        uint64_t t_build, t_count, t_lists, t_sort, t_links, t_sweep, t_bodies;
    } cnt;
};

// minimum and sum over the active lanes of the wavefront (ROCm's device library)
extern "C" __device__ float __ockl_wfred_min_f32(float);
extern "C" __device__ float __ockl_wfred_add_f32(float);

// Drift of the circles from their list-build positions: a common shift u of the
// scene, and a bound no finite displacement is further from u than (infinite
// when some circle has a finite position but a non-finite list-build one).
// Every thread gets the workgroup's result.  With MEAN u is the mean
// displacement: one circle shot out of a pile must not shift all others.
// Without, u is the centre of the displacements' box, which is enough to see
// that nobody drifted far, and is asked every substep of a body in flight: the
// box takes four lane reductions (minima of the bounds and the negated bounds)
// and one barrier (640 flying bodies: the sweep phase 2.1 times shorter than
// with nine values through LDS-routed shuffles).  Barriers lie between two calls of
// one form, after which its slots are free again; circle_sweep may ask with MEAN
// right after quiet_sweep has asked without, so that one takes the worklists' space.
struct Drift {
    float ux, uy, box;
};

template <int WG, bool MEAN>
__device__ __forceinline__ Drift drift_box(const float2 *P, uint32_t Np, uint32_t Nc, const float2 *ref_,
                                           float4 *red4) {
    BD_GLOBAL const uint64_t *const ref = to_global((const uint64_t *)ref_);
    float4 v = make_float4(INFINITY, INFINITY, INFINITY, INFINITY);
    float sx = 0.0f, sy = 0.0f, n = 0.0f;
#pragma unroll 2
    for (uint32_t c = threadIdx.x; c < Nc; c += WG) {
        const float2 p = P[Np + c];
        const uint64_t rb = ref[c];
        const float dx = p.x - __uint_as_float((uint32_t)rb), dy = p.y - __uint_as_float((uint32_t)(rb >> 32));
        // a circle at a non-finite position touches nothing and does not count
        if (fabsf(p.x) <= 3.0e38f && fabsf(p.y) <= 3.0e38f) {
            const bool ok = fabsf(dx) <= 3.0e38f && fabsf(dy) <= 3.0e38f;
            v.x = fminf(v.x, ok ? dx : -INFINITY);
            v.y = fminf(v.y, ok ? -dx : -INFINITY);
            v.z = fminf(v.z, dy);
            v.w = fminf(v.w, -dy);
            if (MEAN && ok) { sx += dx; sy += dy; n += 1.0f; }
        }
    }
    auto reduce = [&]() {
        v.x = __ockl_wfred_min_f32(v.x);
        v.y = __ockl_wfred_min_f32(v.y);
        v.z = __ockl_wfred_min_f32(v.z);
        v.w = __ockl_wfred_min_f32(v.w);
        if constexpr (MEAN) {
            sx = __ockl_wfred_add_f32(sx);
            sy = __ockl_wfred_add_f32(sy);
            n = __ockl_wfred_add_f32(n);
        }
    };
    reduce();
    if constexpr (WG > 64) {
        const uint32_t lane = threadIdx.x & 63u;
        if (lane == 0u) {
            red4[threadIdx.x >> 6] = v;
            if constexpr (MEAN) red4[16u + (threadIdx.x >> 6)] = make_float4(sx, sy, n, 0.0f);
        }
        __syncthreads();
        v = red4[lane & (WG / 64u - 1u)];
        if constexpr (MEAN) {
            const float4 t = red4[16u + (lane & (WG / 64u - 1u))];
            const bool once = lane < WG / 64u;  // each wavefront's sums once
            sx = once ? t.x : 0.0f;
            sy = once ? t.y : 0.0f;
            n = once ? t.z : 0.0f;
        }
        reduce();
    }
    const float x0 = uni(v.x), x1 = -uni(v.y), y0 = uni(v.z), y1 = -uni(v.w);
    if (!(x0 <= x1)) return Drift{0.0f, 0.0f, x0 == INFINITY ? 0.0f : INFINITY};  // no finite circle, or not ok
    float ux = 0.5f * (x0 + x1), uy = 0.5f * (y0 + y1), bx = 0.5f * (x1 - x0), by = 0.5f * (y1 - y0);
    if constexpr (MEAN) {
        if (uni(n) > 0.0f) {
            ux = uni(sx) / uni(n);
            uy = uni(sy) / uni(n);
            bx = fmaxf(fabsf(x0 - ux), fabsf(x1 - ux));
            by = fmaxf(fabsf(y0 - uy), fabsf(y1 - uy));
        }
    }
    const float box = sqrtf(bx * bx + by * by);
    return Drift{ux, uy, box == box ? box : INFINITY};
}

// An upper bound of the drift as a fraction of the smallest skin, with a margin
// for the rounding of the box.
__device__ __forceinline__ float drift_share(float box, float smin) { return (box * 1.0001f) / (smin * 0.9999f); }

typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

// The candidate grid's buckets.  Cell (x, y) goes to bucket (x + y stride) mod T
// with stride about 0.618 T: the cells of a row are consecutive buckets, so a row
// of neighbouring cells is one run of records, and the rows start evenly spread
// over the table.  Three neighbouring rows of three cells share no bucket
// (T >= 32: the starts of rows 1 and 2 apart are at least 3 buckets away).  With
// a hash per cell each of the 9 cells cost two loads and its records a cache line
// of their own, also where neighbours in space are neighbours in memory.  A list
// build, in all: 10,000 circles of a soft body 213 -> 91 us, a gas of 16,000
// 660 -> 318, one of 2,000 with 319 outliers 384 -> 110.
// T is the power of two at or above the circle count where the counters of that
// many buckets fit the LDS beside the positions (grid_buckets), else half of it:
// circles per bucket hardly change the time (its records are one run), counters
// in LDS do.
struct CCGrid {
    uint32_t T, stride, Nc;
    double inv_h;
    const uint32_t *start;  // first record of each bucket, start[T] = Nc (workspace)
};

__device__ __forceinline__ uint32_t grid_buckets(uint32_t Np, uint32_t Nc, uint32_t T) {
    const uint32_t half = T >> 1;
    return half >= 32u && 8u * (Np + Nc) + 2u * half > 136u * 1024u ? half >> 1 : half;
}

__device__ __forceinline__ CCGrid cc_grid(uint32_t Np, uint32_t Nc, uint32_t table, double h, const uint32_t *start) {
    const uint32_t T = grid_buckets(Np, Nc, table);
    return CCGrid{T, (uint32_t)((float)T * 0.618034f) | 1u, Nc, 1.0 / h, start};
}

__device__ __forceinline__ uint32_t grid_bucket(const CCGrid &g, uint32_t cx, uint32_t cy) {
    return (cx + cy * g.stride) & (g.T - 1u);
}

// The records of the n cells from (cx, cy) on along its row: first record and
// count; the run goes on at record 0 after the last one.  start(k) is the first
// record of bucket k, k <= T.  (Records of other cells in these buckets are among
// them; with n >= T they are all records.)
template <typename F>
__device__ __forceinline__ uint32_t grid_row(const CCGrid &g, uint32_t cx, uint32_t cy, uint32_t n, F start,
                                             uint32_t &first) {
    if (n >= g.T) { first = 0u; return g.Nc; }
    const uint32_t b = grid_bucket(g, cx, cy), e = b + n;
    const bool wrap = e > g.T;
    const uint32_t s0 = start(b), s1 = start(wrap ? e - g.T : e);
    first = s0;
    return wrap ? g.Nc - s0 + s1 : s1 - s0;
}

// The buckets' first records: 16-bit in LDS while a list is built (when they
// fit), and 32-bit in the workspace.
template <bool LDS>
struct GridStart;
template <>
struct GridStart<true> {
    BD_LDS const uint16_t *p;
    __device__ __forceinline__ uint32_t operator()(uint32_t k) const { return p[k]; }
};
template <>
struct GridStart<false> {
    BD_GLOBAL const uint32_t *p;
    __device__ __forceinline__ uint32_t operator()(uint32_t k) const { return p[k]; }
};
template <bool LDS>
__device__ __forceinline__ GridStart<LDS> grid_start(const uint32_t *global, uint32_t lds_off) {
    extern __shared__ float2 s_dyn[];
    if constexpr (LDS) return {to_lds((const uint16_t *)((const uint8_t *)s_dyn + lds_off))};
    else return {to_global(global)};
}

// Candidate pairs are the pairs closer than (r_c + skin_c) + (r_o + skin_o)
// when the list is built.  A normal circle (skin <= s_cell) finds its normal
// partners in the 3x3 cells of size h = 2 (r_max + s_cell) around it: three runs
// of records (a record from another cell in those buckets is still a true
// partner when it passes the distance test, and it is in one run only).  An
// outlier (larger skin) finds all its partners itself and writes itself into its
// normal partners' lists too, so normal circles never search far.  The first
// `cap` partners go to out; the count is returned in full.
template <bool LDS>
__device__ __noinline__ uint32_t gather_normal(uint32_t c, const CCWork &w, CCGrid g, uint32_t lds_off,
                                               float2 p, float ec, uint16_t *out_, uint32_t cap) {
    const GridStart<LDS> start = grid_start<LDS>(w.start, lds_off);
    BD_GLOBAL const f32x4 *const rec = to_global((const f32x4 *)w.rec);
    BD_GLOBAL uint16_t *const out = (BD_GLOBAL uint16_t *)(uint64_t)out_;  // (each lane its own)
    const uint32_t Nc = uni(g.Nc);
    const uint32_t cx = (uint32_t)scell(p.x, g.inv_h) - 1u, cy = (uint32_t)scell(p.y, g.inv_h);
    uint32_t s0[3], pre1, pre2, total;
    if (g.T < 32u) {
        s0[0] = s0[1] = s0[2] = 0u;
        pre1 = pre2 = total = Nc;  // a table too small for separate rows: every record
    } else {
        pre1 = grid_row(g, cx, cy - 1u, 3u, start, s0[0]);
        pre2 = pre1 + grid_row(g, cx, cy, 3u, start, s0[1]);
        total = pre2 + grid_row(g, cx, cy + 1u, 3u, start, s0[2]);
    }
    constexpr uint32_t kU = 4;
    uint32_t n = 0;
#pragma unroll 1
    for (uint32_t t0 = 0; t0 < total; t0 += kU) {
        f32x4 r[kU];
#pragma unroll
        for (uint32_t u = 0; u < kU; u++) {
            const uint32_t t = min(t0 + u, total - 1u);
            uint32_t s = t < pre1 ? s0[0] + t : t < pre2 ? s0[1] + (t - pre1) : s0[2] + (t - pre2);
            if (s >= Nc) s -= Nc;
            r[u] = rec[s];
        }
#pragma unroll
        for (uint32_t u = 0; u < kU; u++) {
            const uint32_t o = __float_as_uint(r[u].w);
            // an outlier lists its pairs itself
            if (t0 + u >= total || o == c || (o & kOutlierBit)) continue;
            float ex = p.x - r[u].x, ey = p.y - r[u].y;
            float lim = ec + r[u].z;
            if (ex * ex + ey * ey < lim * lim) {
                if (n < cap) out[n] = (uint16_t)o;
                n++;
            }
        }
    }
    return n;
}

// Outliers' partners.  A near outlier (its normal partners lie within 8
// cells) has those cells scanned: the (outlier, row of cells) items of all near
// outliers are spread over the workgroup's threads when the outliers fit one
// stage, else 16 lanes take one outlier at a time.  A far one is searched
// by the whole workgroup over every circle, and pairs of two outliers by all pairs among
// the outliers.  An outlier-normal pair is found once, by the outlier, and
// goes into both lists; an outlier-outlier pair is found once per direction
// (the test is symmetric) and goes into the first one's list.  MODE 0 counts
// into cnt, MODE 1 appends at the lists' cursors.  stage: WG / 2 entries of
// LDS scratch.  Returns the far outliers.
template <int WG, int MODE, bool LDS>
__device__ __noinline__ uint32_t gather_outliers(const CCWork &w, CCGrid g, uint32_t lds_off, const float *crad,
                                    const uint16_t *outs, uint32_t n_out_, float rmax, float s_cell, double h,
                                    uint32_t *cursor, float4 *stage, uint32_t *s_wave) {
    const uint32_t n_out = uni(n_out_), Nc = uni(g.Nc);
    const GridStart<LDS> start = grid_start<LDS>(w.start, lds_off);
    BD_GLOBAL const f32x4 *const rec = to_global((const f32x4 *)w.rec);
    const double inv_h = g.inv_h;
    auto add = [&](uint32_t c, uint32_t o) {
        if (MODE == 0) atomicAdd(&w.cnt[c], 1u);
        else w.cand[atomicAdd(&cursor[c], 1u)] = (uint16_t)o;
    };
    auto reach_of = [&](float ec) { return ((double)ec + (double)rmax + (double)s_cell) / h; };
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    // the outliers' positions and reaches in LDS (stage), WG / 2 at a time
    constexpr uint32_t kStage = WG / 2;
    auto stage_tile = [&](uint32_t t0, uint32_t tn) {
        __syncthreads();  // the previous tile is no longer read
        for (uint32_t k = threadIdx.x; k < tn; k += WG) {
            const uint32_t o = outs[t0 + k];
            const float2 po = w.ref[o];
            stage[k] = make_float4(po.x, po.y, crad[o] + w.skin[o], 0.0f);
        }
        __syncthreads();
    };
    const bool one_tile = n_out <= kStage;
    // the rows a near outlier scans: 2R + 1 of as many cells, R = ceil(reach)
    auto near_side = [&](float ec) -> uint32_t {
        const double reach = reach_of(ec);
        return reach <= 8.0 ? 2u * (uint32_t)(int)ceil(reach) + 1u : 0u;
    };
    // row q of the outlier's cells
    auto scan_row = [&](uint32_t c, float2 p, float ec, uint32_t side, uint32_t q) {
        const uint32_t cx = (uint32_t)scell(p.x, inv_h) - (side >> 1), cy = (uint32_t)scell(p.y, inv_h) - (side >> 1) + q;
        uint32_t s0;
        const uint32_t len = grid_row(g, cx, cy, side, start, s0);
        constexpr uint32_t kU = 4;
#pragma unroll 1
        for (uint32_t t0 = 0; t0 < len; t0 += kU) {
            f32x4 r[kU];
#pragma unroll
            for (uint32_t u = 0; u < kU; u++) {
                uint32_t s = s0 + min(t0 + u, len - 1u);
                if (s >= Nc) s -= Nc;
                r[u] = rec[s];
            }
#pragma unroll
            for (uint32_t u = 0; u < kU; u++) {
                const uint32_t o = __float_as_uint(r[u].w);
                float ex = p.x - r[u].x, ey = p.y - r[u].y;
                float lim = ec + r[u].z;
                if (t0 + u >= len || (o & kOutlierBit) || !(ex * ex + ey * ey < lim * lim)) continue;  // outliers: below
                // found in the row of its own cell only (other rows may hold the same buckets)
                if ((uint32_t)scell(r[u].y, inv_h) != cy || (uint32_t)scell(r[u].x, inv_h) - cx >= side) continue;
                add(c, o);
                add(o, c);
            }
        }
    };
    if (one_tile && n_out) {
        stage_tile(0u, n_out);
        // every (near outlier, row) item across the workgroup: each outlier's
        // first item (an exclusive prefix over the outliers' row counts) goes
        // in its stage entry's w, and a thread takes a contiguous run of items,
        // finding its first outlier by bisection
        const uint32_t t = threadIdx.x;
        const uint32_t rows = t < n_out ? near_side(stage[t].z) : 0u;
        const uint32_t inc = __ockl_wfscan_add_u32(rows, true);
        if (lane == 63u) s_wave[wave] = inc;
        __syncthreads();
        const uint32_t uw = uni(wave);
        uint32_t below = 0, items = 0;
#pragma unroll 1
        for (uint32_t v = 0; v < uw; v++) below += s_wave[v];
        items = below;
#pragma unroll 1
        for (uint32_t v = uw; v < WG / 64; v++) items += s_wave[v];
        if (t < n_out) stage[t].w = __uint_as_float(below + inc - rows);
        __syncthreads();
        const uint32_t per = (items + WG - 1) / WG;
        uint32_t i = t * per;
        const uint32_t i1 = min(items, i + per);
        if (i < i1) {
            // the last outlier whose first item is at or before i (one with no
            // rows shares its first item with the next, and is passed over)
            uint32_t lo = 0, hi = n_out;
            while (hi - lo > 1u) {
                const uint32_t mid = (lo + hi) >> 1;
                if (__float_as_uint(stage[mid].w) <= i) lo = mid; else hi = mid;
            }
            uint32_t k = lo;
            float4 e = stage[k];
            uint32_t side = near_side(e.z), q = i - __float_as_uint(e.w);
#pragma unroll 1
            for (; i < i1; i++) {
                if (q == side) {
                    // the next outlier with rows
                    do {
                        e = stage[++k];
                        side = near_side(e.z);
                    } while (side == 0u && k + 1u < n_out);
                    q = 0;
                }
                scan_row(outs[k], make_float2(e.x, e.y), e.z, side, q);
                q++;
            }
        }
    }
    // more outliers than one stage holds: 16 lanes an outlier, over its rows
    for (uint32_t k = threadIdx.x >> 4; k < n_out && !one_tile; k += WG / 16) {
        const uint32_t c = outs[k];
        const float ec = crad[c] + w.skin[c];
        const uint32_t side = near_side(ec);
        for (uint32_t q = lane & 15u; q < side; q += 16u) scan_row(c, w.ref[c], ec, side, q);
    }
    uint32_t n_far = 0;
    // every wavefront finds the far ones, 64 outliers at a time (one after the
    // other they cost a dependent load and a division each: 0.4 us, for each of
    // up to kOutCap outliers and twice a list)
    for (uint32_t k0 = 0; k0 < n_out; k0 += 64u) {
        const uint32_t k = k0 + lane;
        bool is_far = false;
        if (k < n_out) is_far = near_side(one_tile ? stage[k].z : crad[outs[k]] + w.skin[outs[k]]) == 0u;
        for (uint64_t m = __ballot(is_far); m; m &= m - 1u) {
            n_far++;
            const uint32_t c = uni((uint32_t)outs[k0 + (uint32_t)__ffsll((unsigned long long)m) - 1u]);
            const float2 p = w.ref[c];
            const float ec = crad[c] + w.skin[c];
            for (uint32_t s = threadIdx.x; s < Nc; s += WG) {
                const float4 r = w.rec[s];
                const uint32_t o = __float_as_uint(r.w);
                if (o & kOutlierBit) continue;
                float ex = p.x - r.x, ey = p.y - r.y;
                float lim = ec + r.z;
                if (ex * ex + ey * ey < lim * lim) { add(c, o); add(o, c); }
            }
        }
    }
    // outlier pairs: a wavefront takes outlier a, its lanes the staged ones
    for (uint32_t t0 = 0; t0 < n_out; t0 += kStage) {
        const uint32_t tn = min(kStage, n_out - t0);
        if (!one_tile) stage_tile(t0, tn);
        for (uint32_t a = wave; a < n_out; a += WG / 64) {
            const uint32_t c = outs[a];
            float2 p;
            float ec;
            if (one_tile) {
                const float4 e = stage[a];
                p = make_float2(e.x, e.y);
                ec = e.z;
            } else {
                p = w.ref[c];
                ec = crad[c] + w.skin[c];
            }
            for (uint32_t k = lane; k < tn; k += 64) {
                if (t0 + k == a) continue;
                const float4 q = stage[k];
                float ex = p.x - q.x, ey = p.y - q.y;
                float lim = ec + q.z;
                if (ex * ex + ey * ey < lim * lim) add(c, outs[t0 + k]);
            }
        }
    }
    return n_far;
}

// Ascending sort of a list of at most K < 65536 entries by one thread: a
// bitonic network over registers (K a power of two), padding sorting last.
template <int K>
__device__ __forceinline__ void sort_in_registers(uint16_t *my, uint32_t n) {
    uint32_t v[K];
#pragma unroll
    for (int i = 0; i < K; i++) v[i] = i < (int)n ? (uint32_t)my[i] : 0xffffffffu;
#pragma unroll
    for (int k = 2; k <= K; k <<= 1)
#pragma unroll
        for (int j = k >> 1; j > 0; j >>= 1)
#pragma unroll
            for (int i = 0; i < K; i++) {
                const int l = i ^ j;
                if (l > i) {
                    const uint32_t a = v[i], b = v[l];
                    const bool up = (i & k) == 0;
                    v[i] = up ? min(a, b) : max(a, b);
                    v[l] = up ? max(a, b) : min(a, b);
                }
            }
#pragma unroll
    for (int i = 0; i < K; i++)
        if (i < (int)n) my[i] = (uint16_t)v[i];
}

// Ascending sort of a list of at most kMidList distinct entries by one
// wavefront: each lane ranks its entries against the whole list, then writes
// them to their ranks.  Every lane runs the rank loop to the end (the trip
// count is uniform) before any lane stores, so no entry is overwritten while
// it is still being read.
__device__ __forceinline__ void sort_by_wave(uint16_t *my, uint32_t n) {
    constexpr int M = kMidList / 64;
    const uint32_t lane = threadIdx.x & 63u;
    uint32_t v[M], r[M];
#pragma unroll
    for (int m = 0; m < M; m++) {
        const uint32_t k = lane + 64u * m;
        v[m] = k < n ? (uint32_t)my[k] : 0xffffffffu;
        r[m] = 0u;
    }
#pragma unroll 8
    for (uint32_t j = 0; j < n; j++) {
        const uint32_t x = my[j];
#pragma unroll
        for (int m = 0; m < M; m++) r[m] += x < v[m] ? 1u : 0u;
    }
#pragma unroll
    for (int m = 0; m < M; m++)
        if (lane + 64u * m < n) my[r[m]] = (uint16_t)v[m];
}

// Cell size of the candidate grid: twice the largest radius plus the skin of
// normal circles, so a normal pair lies in neighbouring cells.
__device__ __forceinline__ double cell_size(float rmax, float s_cell) {
    return 2.0 * ((double)rmax + (double)s_cell) * 1.001 + 1e-30;
}

// Position of x in c's active list, or where it would go; found tells whether
// the list holds it.
__device__ __forceinline__ uint32_t list_rank(const CCWork &w, const uint16_t *act, uint32_t c, uint32_t x,
                                              bool &found) {
    const uint16_t *my = act + w.items[c];
    uint32_t lo = 0, hi = w.key[c];
    while (lo < hi) {
        const uint32_t mid = (lo + hi) >> 1;
        const uint32_t v = my[mid];
        if (v == x) { found = true; return mid; }
        if (v < x) lo = mid + 1; else hi = mid;
    }
    found = false;
    return lo;
}

// Whether x is in c's candidate list.
__device__ __forceinline__ bool is_candidate(const CCWork &w, uint32_t c, uint32_t x) {
    const uint16_t *my = w.cand + w.off[c];
    uint32_t lo = 0, hi = w.cnt[c];
    while (lo < hi) {
        const uint32_t mid = (lo + hi) >> 1, v = my[mid];
        if (v == x) return true;
        if (v < x) lo = mid + 1; else hi = mid;
    }
    return false;
}

// Whether the pair (c, x), missing from the active lists, would have
// overlapped when the reference tests it.  Its turn comes after the pairs of
// c with smaller partners and those of x with smaller partners (the
// reference's (i, j) order), so each circle is where the sweep left it after
// that prefix of its own list: exactly, as long as no other missing pair
// touched first, which this same test covers for every missing pair.  The
// overlap test is Circle::solve_circle's (src/circle.rs:32-35) on those
// positions, so a pair it clears was a no-op in the reference too.
__device__ __forceinline__ bool missed_pair_touches(const CCWork &w, const uint16_t *act, const float *crad,
                                                    uint32_t c, uint32_t x) {
    bool found = false;
    const uint32_t kc = list_rank(w, act, c, x, found);
    if (found) return false;  // on the list: run in order by the sweep
    const uint32_t kx = list_rank(w, act, x, c, found);
    const float2 pc = kc ? w.traj[w.items[c] + kc - 1] : w.save[c];
    const float2 px = kx ? w.traj[w.items[x] + kx - 1] : w.save[x];
    const bool c_first = c < x;
    const float2 pi = c_first ? pc : px, pj = c_first ? px : pc;
    const float ri = crad[c_first ? c : x], rj = crad[c_first ? x : c];
    float dx = pi.x - pj.x, dy = pi.y - pj.y;
    float q = dx * dx + dy * dy;
    float rs = ri + rj;
    return q < rs * rs;
}

// A sweep in which some circles moved further than 0.8 of their skins is
// still exact when no pair missing from the lists touched at its turn.  Pairs
// of two circles within their skins stayed apart by construction; this looks
// at every pair with a circle beyond its skin (`over`, with -v in vb; the
// others hold v <= vmax, v being a circle's bound on its distance from its
// list-build position, relative to the common shift u, over the whole sweep).
// During the sweep such a circle c was within path_c of its start, and a circle
// x within its skin within v_x of where it was listed, shifted by u: if the two
// are more than r_c + r_x + path_c + v_x apart there, they stayed apart; the
// rest get the exact test above.  So only the cells around c's start are
// searched, however far c has come since the list was built.
//
// With few overruns (at most kOutCap, listed in LDS) pairs of two overrun
// circles are tested all against all and the grid scan skips them; with more
// (listed in the workspace; only right after a list build, when every circle's
// start is its listed position) the grid scan covers them too, vmax then being
// the largest bound of any circle, and a pair of two overruns is tested from
// both ends.
template <int WG, typename Idx>
__device__ __noinline__ int overruns_check(const CCWork &w, const uint16_t *act, const float *crad, const float *vb, const Idx *over,
                              uint32_t n_over, float vmax, float2 u, float rmax, double h, CCGrid g,
                              float *s_red, bool scan_overruns) {
    const GridStart<false> start{to_global(g.start)};
    const uint32_t Nc = uni(g.Nc);
    // rounding margin: a fifth of the overrun circle's skin (the margin the
    // skin test leaves too) plus about 80 ulps of the coordinates
    auto margin = [&](float2 p, float sk) { return 0.2f * sk + 1e-5f * (fabsf(p.x) + fabsf(p.y) + 1.0f); };
    auto apart = [&](float2 p, float2 q, float lim) {
        float dx = p.x - q.x, dy = p.y - q.y;
        return !(sqrtf(dx * dx + dy * dy) <= lim);  // NaN: a non-finite circle touches nothing
    };
    float bad = 0.0f, far = 0.0f;
    // 16 lanes a circle, over the rows of its cells
    for (uint32_t k = threadIdx.x >> 4; k < n_over; k += WG / 16) {
        const uint32_t c = over[k];
        float2 p = w.save[c];
        if (!(fabsf(p.x) <= 3.0e38f) || !(fabsf(p.y) <= 3.0e38f)) continue;  // touches nothing
        p.x = p.x - u.x; p.y = p.y - u.y;
        const float rc = crad[c], vc = w.path[c], mc = margin(p, fminf(w.skin[c], rmax)) + 1e-5f * (fabsf(u.x) + fabsf(u.y));
        const double reach = ((double)rc + (double)vc + (double)mc + (double)rmax + (double)vmax) / h;
        if (!(reach <= 8.0)) { far = 1.0f; continue; }
        const uint32_t R = (uint32_t)(int)ceil(reach), side = 2u * R + 1u;
        const uint32_t cx = (uint32_t)scell(p.x, g.inv_h) - R, cy = (uint32_t)scell(p.y, g.inv_h) - R;
        for (uint32_t q = threadIdx.x & 15u; q < side; q += 16u) {
            uint32_t s0;
            const uint32_t len = grid_row(g, cx, cy + q, side, start, s0);
            for (uint32_t t = 0; t < len; t++) {
                const float4 r = w.rec[s0 + t < Nc ? s0 + t : s0 + t - Nc];
                const uint32_t x = __float_as_uint(r.w) & ~kOutlierBit;
                float vx = vb[x];
                if (x == c) continue;
                if (!(vx >= 0.0f)) {  // beyond its skin: below, or here when overruns are scanned
                    if (!scan_overruns) continue;
                    vx = -vx;
                }
                if (apart(p, make_float2(r.x, r.y), ((rc + crad[x]) + (vc + vx)) + mc)) continue;
                if (missed_pair_touches(w, act, crad, c, x)) bad = fmaxf(bad, is_candidate(w, c, x) ? 1.0f : 2.0f);
            }
        }
    }
    if (!scan_overruns)
    for (uint32_t q = threadIdx.x; q < n_over * n_over; q += WG) {
        const uint32_t a = q / n_over, b = q - a * n_over;
        if (a >= b) continue;
        const uint32_t c = over[a], o = over[b];
        const float lim = ((crad[c] + crad[o]) + (w.path[c] + w.path[o])) * (1.0f + 0x1p-16f);
        if (apart(w.save[c], w.save[o], lim)) continue;
        if (missed_pair_touches(w, act, crad, c, o)) bad = fmaxf(bad, is_candidate(w, c, o) ? 1.0f : 2.0f);
    }
    // 0: every missing pair stayed apart; 1: one touched, but only candidates
    // that the active lists left out; 2: one that the candidate lists do not
    // hold; 3: an overrun too far to search (the sweep is redone without knowing)
    return (int)wg_max<WG>(fmaxf(bad, 3.0f * far), s_red);
}

// A sweep in which some circles (near, listed in fill) moved further than 0.8 of
// their active margins, but within their skins, is still exact when none of
// their candidates left out of the active lists touched at its turn.  A pair
// further apart at the sweep's start than the radii and both excursions stayed
// apart; the rest get the exact test.  Returns 0, or 1 if one touched.
template <int WG>
__device__ __noinline__ int near_check(const CCWork &w, const uint16_t *act, const float *crad, uint32_t n_near,
                                       float *s_red) {
    float bad = 0.0f;
    for (uint32_t k = threadIdx.x; k < n_near; k += WG) {
        const uint32_t c = w.fill[k], o0 = w.off[c], n = w.cnt[c];
        const float2 p = w.save[c];
        const float rc = crad[c], vc = w.path[c];
        for (uint32_t e = 0; e < n; e++) {
            const uint32_t x = w.cand[o0 + e];
            const float2 q = w.save[x];
            const float dx = p.x - q.x, dy = p.y - q.y;
            // a relative margin far above the rounding of these few operations
            const float lim = ((rc + crad[x]) + (vc + w.path[x])) * (1.0f + 0x1p-16f);
            if (!(sqrtf(dx * dx + dy * dy) <= lim)) continue;  // NaN: a non-finite circle touches nothing
            if (missed_pair_touches(w, act, crad, c, x)) bad = 1.0f;
        }
    }
    return (int)wg_max<WG>(bad, s_red);
}

// Whether one of the circles that drifted beyond their skins (`over`, nd of them,
// with -v in vb; the others hold v <= vmax) is now, before the sweep, in reach of
// a circle that its candidate list does not hold, reach being that of the active
// lists (radii and margins).  Such a pair would most likely touch and cost a
// second run of the sweep; a new list beforehand costs less.
template <int WG>
__device__ __noinline__ bool drifted_meet(const float2 *P, uint32_t Np, const CCWork &w, const float *crad,
                                          const float *vb, const uint16_t *over, uint32_t nd, float vmax, float2 u,
                                          float mbase, float rmax, double h, CCGrid g, float *s_red) {
    const GridStart<false> start{to_global(g.start)};
    const uint32_t Nc = uni(g.Nc), lane = threadIdx.x & 15u;
    float met = 0.0f;
    auto meets = [&](uint32_t c, float2 p, float ec, uint32_t x) {
        const float2 q = P[Np + x];
        const float dx = p.x - q.x, dy = p.y - q.y, lim = ec + (crad[x] + fmaxf(mbase, w.need[x]));
        return dx * dx + dy * dy < lim * lim && !is_candidate(w, c, x);
    };
    for (uint32_t k = threadIdx.x >> 4; k < nd; k += WG / 16) {
        const uint32_t c = over[k];
        const float2 p = P[Np + c];
        const float mc = fmaxf(mbase, w.need[c]), ec = crad[c] + mc;
        const float2 pu = make_float2(p.x - u.x, p.y - u.y);
        const double reach = ((double)ec + (double)rmax + (double)mbase + (double)vmax) / h;
        if (!(reach <= 8.0)) { met = 1.0f; continue; }
        const uint32_t R = (uint32_t)(int)ceil(reach), side = 2u * R + 1u;
        const uint32_t cx = (uint32_t)scell(pu.x, g.inv_h) - R, cy = (uint32_t)scell(pu.y, g.inv_h) - R;
        for (uint32_t q = lane; q < side; q += 16u) {
            uint32_t s0;
            const uint32_t len = grid_row(g, cx, cy + q, side, start, s0);
            for (uint32_t t = 0; t < len; t++) {
                const uint32_t x = __float_as_uint(w.rec[s0 + t < Nc ? s0 + t : s0 + t - Nc].w) & ~kOutlierBit;
                if (x != c && vb[x] >= 0.0f && meets(c, p, ec, x)) met = 1.0f;
            }
        }
        for (uint32_t j = lane; j < nd; j += 16u)
            if (j != k && meets(c, p, ec, over[j])) met = 1.0f;
    }
    return wg_max<WG>(met, s_red) > 0.0f;
}

// Sequential fallback of the circle-pair sweep, for a sweep whose candidate
// lists keep failing (circles pushed far within the sweep, lists beyond the
// workspace): the reference's (i, j) loop (src/solver.rs:168-177) row by
// row, which needs no list made in advance.  Run by the first wavefront
// alone; the caller holds the others at a barrier.
//
// The circles sit in a hashed grid of cell size h = 2 r_max + M, each in
// the bucket of the cell its current position is in (a push that moves a
// circle to another bucket moves it in the grid).  Row i gathers every
// j > i closer than r_i + r_j + M to circle i (nine lanes walk the nine
// buckets of the 3x3 cells around it).  The lanes hold the candidates and
// their positions in registers (a candidate does not move before its turn);
// the next pair of the row is the smallest candidate above the last one
// that overlaps circle i where it is now (a wavefront minimum), since the
// reference's test is false, and the pair a no-op, for every j in between.
// One lane runs that pair.  Only circle i moves within its row
// besides each partner at its own turn, so the gather is complete while
// circle i stays within M/2 of where it was gathered from; when it moves
// further the rest of the row is gathered again, with a margin one cell
// wider each time (up to two cells, over 5x5 and then 7x7 cells), so a
// circle pushed far within its row is gathered again only a few times.
// The halved margin leaves room for f32 rounding of the distance tests.
//
constexpr uint32_t kNone16 = 0xffffu;

// minimum over the active lanes of the wavefront (ROCm's device library)
extern "C" __device__ uint32_t __ockl_wfred_min_u32(uint32_t);

template <int WG>
__device__ __noinline__ void sequential_sweep(float2 *P, uint32_t Np, uint32_t Nc, const float *crad, bool uni_r,
                                              float runi, float rmax, const FbGrid *gp, uint32_t *s_fb) {
    const FbGrid g = *gp;
    const uint32_t lane = threadIdx.x & 63u;
    const float rm = fmaxf(rmax, 1e-3f);
    const float M = 0.5f * rm;
    const double hd = 2.0 * (double)rm + (double)M;
    const double inv_h = 1.0 / hd;
    const float hstep = 0.999f * (float)hd;
    uint16_t *const head = g.head;
    uint16_t *const next = g.next, *const cand = g.cand;
    const uint32_t tmask = g.tmask;
    auto radius = [=](uint32_t c) { return uni_r ? runi : crad[c]; };
    auto finite2 = [](float2 p) { return fabsf(p.x) <= 3.0e38f && fabsf(p.y) <= 3.0e38f; };
    auto bucket = [=](float2 p) {
        return finite2(p) ? (cell_hash(scell(p.x, inv_h), scell(p.y, inv_h)) & tmask) : kNone;
    };
    auto wave_sync = []() { __threadfence_block(); __builtin_amdgcn_wave_barrier(); };
    auto link = [=](uint32_t c, uint32_t k) {  // c into bucket k (lane 0 alone)
        next[c] = head[k];
        head[k] = (uint16_t)c;
    };
    auto unlink = [=](uint32_t c, uint32_t k) {  // c out of bucket k (lane 0 alone; lists are acyclic)
        uint32_t x = head[k];
        if (x == c) {
            head[k] = next[c];
        } else {
#pragma unroll 1
            for (uint32_t guard = 0; x != kNone16 && guard < Nc; guard++) {
                const uint32_t y = next[x];
                if (y == c) { next[x] = next[c]; break; }
                x = y;
            }
        }
    };
    // heads are u16, two to a 32-bit word: a circle goes in by compare-and-swap
    // on its bucket's word (each attempt that fails saw another lane succeed)
    uint32_t *const head32 = (uint32_t *)head;
#pragma unroll 1
    for (uint32_t b = lane; b <= tmask / 2u; b += 64) head32[b] = 0xffffffffu;
    wave_sync();
#pragma unroll 1
    for (uint32_t c = lane; c < Nc; c += 64) {
        const uint32_t k = bucket(P[Np + c]);
        if (k != kNone) {
            const uint32_t sh = 16u * (k & 1u);
            uint32_t old = head32[k >> 1], seen;
            do {
                seen = old;
                next[c] = (uint16_t)(seen >> sh);
                old = atomicCAS(&head32[k >> 1], seen, (seen & ~(0xffffu << sh)) | (c << sh));
            } while (old != seen);
        }
    }
    wave_sync();
#pragma unroll 1
    for (uint32_t i = 0; i + 1 < Nc; i++) {
        if (!finite2(P[Np + i])) continue;  // touches nothing (every comparison with it is false)
        const float ri = radius(i);
        uint32_t jlast = i, level = 0, lcap = 2;
        // a pass runs a pair or ends the row, except a wider gather that
        // found too many candidates, which the next pass redoes one cell
        // narrower (the row's widest from then on)
#pragma unroll 1
        for (uint32_t pass = 0; pass < 2u * Nc + 2u; pass++) {
            const float2 base = P[Np + i];
            // margin of this gather: M, and one cell more for each gather of
            // the row that circle i outran; the cells within R of its own
            // hold every circle within reach (R cells apart is more than R h)
            const float Ml = M + (float)level * hstep;
            const int R = (int)level + 1, side = 2 * R + 1;
            if (lane == 0) s_fb[0] = 0u;
            wave_sync();
            // gather: lane q walks the bucket of cell q of the side x side
            // block (a bucket two cells share is walked twice; its circles are
            // then listed twice, which changes no pair's turn)
            const int cx0 = scell(base.x, inv_h), cy0 = scell(base.y, inv_h);
            if (lane < (uint32_t)(side * side)) {
                const uint32_t kk =
                    cell_hash(cx0 + (int)(lane % (uint32_t)side) - R, cy0 + (int)(lane / (uint32_t)side) - R) & tmask;
                uint32_t j = head[kk];
#pragma unroll 1
                for (uint32_t guard = 0; j != kNone16 && guard < Nc; guard++) {
                    const uint32_t nx = next[j];
                    if (j > jlast) {
                        const float2 pj = P[Np + j];
                        const float dx = base.x - pj.x, dy = base.y - pj.y, lim = (ri + radius(j)) + Ml;
                        if (dx * dx + dy * dy < lim * lim) {
                            const uint32_t at = atomicAdd(&s_fb[0], 1u);
                            if (at < g.cap) cand[at] = (uint16_t)j;
                        }
                    }
                    j = nx;
                }
            }
            wave_sync();
            const uint32_t n = s_fb[0];
            const bool fits = n <= g.cap && n <= kMidList;
            if (!fits && level > 0u) {
                lcap = level - 1u;
                level = lcap;
                continue;
            }
            if (fits) {
                constexpr int KM = kMidList / 64;
                uint32_t v[KM];
                float2 pv[KM];
                float rv[KM];
#pragma unroll
                for (int m = 0; m < KM; m++) {
                    const uint32_t k = lane + 64u * m;
                    v[m] = k < n ? (uint32_t)cand[k] : kNone;
                    pv[m] = make_float2(0.0f, 0.0f);
                    rv[m] = 0.0f;
                    if (v[m] != kNone) { pv[m] = P[Np + v[m]]; rv[m] = ri + radius(v[m]); }
                }
                uint32_t again = 0u;
#pragma unroll 1
                for (;;) {
                    const float2 a = P[Np + i];
                    uint32_t best = kNone;
#pragma unroll
                    for (int m = 0; m < KM; m++) {
                        const float dx = a.x - pv[m].x, dy = a.y - pv[m].y;
                        if (v[m] != kNone && v[m] > jlast && dx * dx + dy * dy < rv[m] * rv[m]) best = min(best, v[m]);
                    }
                    const uint32_t j = __ockl_wfred_min_u32(best);
                    if (j == kNone) break;  // the row is done
                    if (lane == 0) {
                        float2 ai = a;
                        const float2 b0 = P[Np + j];
                        float2 b = b0;
                        float qi, qj;
                        uint32_t moved = 0u;
                        if (solve_circle_pair(ai.x, ai.y, b.x, b.y, ri, radius(j), qi, qj)) {
                            P[Np + i] = ai;
                            P[Np + j] = b;
                            const uint32_t ob = bucket(b0), nb = bucket(b);  // b0 is finite: it was gathered
                            if (nb != ob) {
                                unlink(j, ob);
                                if (nb != kNone) link(j, nb);
                            }
                            const float gx = ai.x - base.x, gy = ai.y - base.y;
                            moved = !(gx * gx + gy * gy <= 0.25f * Ml * Ml) ? 1u : 0u;
                        }
                        s_fb[1] = moved;
                    }
                    wave_sync();
                    jlast = j;
                    if (s_fb[1]) { again = 1u; break; }
                }
                if (!again) break;  // the row is done
                level = min(level + 1u, lcap);
                continue;           // gather the rest of the row again
            }
            wave_sync();
            if (lane == 0) {
                uint32_t again = 0u;
                float2 a = P[Np + i];
#pragma unroll 1
                for (uint32_t k = 0; k < n; k++) {
                    uint32_t j;
                    {
                        // too many to rank: the next j above jlast within reach,
                        // by walking the block's buckets again (lane 0 alone)
                        j = kNone;
#pragma unroll 1
                        for (int q = 0; q < side * side; q++) {
                            const uint32_t kq = cell_hash(cx0 + q % side - R, cy0 + q / side - R) & tmask;
                            uint32_t x = head[kq];
#pragma unroll 1
                            for (uint32_t guard = 0; x != kNone16 && guard < Nc; guard++) {
                                const uint32_t nx = next[x];
                                if (x > jlast && x < j) {
                                    const float2 px = P[Np + x];
                                    const float dx = base.x - px.x, dy = base.y - px.y;
                                    const float lim = (ri + radius(x)) + Ml;
                                    if (dx * dx + dy * dy < lim * lim) j = x;
                                }
                                x = nx;
                            }
                        }
                        if (j == kNone) break;
                    }
                    jlast = j;
                    const float2 b0 = P[Np + j];
                    float2 b = b0;
                    float qi, qj;
                    if (solve_circle_pair(a.x, a.y, b.x, b.y, ri, radius(j), qi, qj)) {
                        P[Np + i] = a;
                        P[Np + j] = b;
                        const uint32_t ob = bucket(b0), nb = bucket(b);  // b0 is finite: it was gathered
                        if (nb != ob) {
                            unlink(j, ob);
                            if (nb != kNone) link(j, nb);
                        }
                        const float gx = a.x - base.x, gy = a.y - base.y;
                        if (!(gx * gx + gy * gy <= 0.25f * Ml * Ml)) { again = 1u; break; }
                    }
                }
                s_fb[1] = again;
                s_fb[2] = jlast;
            }
            wave_sync();
            jlast = s_fb[2];
            if (!s_fb[1]) break;
            level = min(level + 1u, lcap);
        }
    }
    wave_sync();
}

// The sequential sweep for the whole workgroup: the first wavefront runs it,
// then every circle's skin need follows from how far the sweep moved it, and
// the lists are marked stale.  Its grid goes into LDS when the scene leaves
// room there (previous positions held in LDS are parked in global memory
// for the sweep), else into the circle-pair workspace.
template <int WG>
__device__ __forceinline__ void fallback_sweep(float2 *P, uint32_t Np, uint32_t Nc, const float *crad, bool uni_r,
                                               float runi, float rmax, uint32_t T, const CCWork &w, CCShared *sh) {
    const int tid = threadIdx.x;
    const CCShared::Fallback fb = sh->fb;
    for (uint32_t c = tid; c < Nc; c += WG) w.save[c] = P[Np + c];
    if (fb.q_lds)
        for (uint32_t j = tid; j < fb.nq; j += WG) fb.q_global[j] = fb.q_lds[j];
    __syncthreads();
    // heads 2 B per bucket, next links 2 B per circle, 256 candidates
    FbGrid &g = sh->grid;
    const uint64_t fixed = 2ull * Nc + 2ull * kMidList;
    uint32_t tb = 0;
    if (fixed + 2ull * 64 <= fb.lds_bytes) {
        tb = 64;
        while (tb < 32768u && tb < 2 * Nc && fixed + 2ull * 2 * tb <= fb.lds_bytes) tb <<= 1;
    }
    if (tb) {
        uint8_t *at = fb.lds;
        g.head = (uint16_t *)at; at += 2ull * tb;
        g.next = (uint16_t *)at; at += 2ull * Nc;
        g.cand = (uint16_t *)at;
        g.tmask = tb - 1;
        g.cap = kMidList;
    } else {
        // workspace: 2T heads (in start's T + 1 words), next links in key,
        // candidates in stamp
        g.head = (uint16_t *)w.start;
        g.next = (uint16_t *)w.key;
        g.cand = (uint16_t *)w.stamp;
        g.tmask = 2 * T - 1;
        g.cap = 2 * Nc;
    }
    __syncthreads();  // the grid's description, written by every thread alike, before the first wavefront reads it
    if (tid < 64) sequential_sweep<WG>(P, Np, Nc, crad, uni_r, runi, rmax, &sh->grid, sh->cnt3);
    __syncthreads();
    if (fb.q_lds)
        for (uint32_t j = tid; j < fb.nq; j += WG) fb.q_lds[j] = fb.q_global[j];
    for (uint32_t c = tid; c < Nc; c += WG) {
        const float2 p = P[Np + c], q = w.save[c];
        const float dx = p.x - q.x, dy = p.y - q.y;
        const float d = sqrtf(dx * dx + dy * dy) * (1.0f + 0x1p-20f);
        w.need[c] = (d <= 3.0e38f) ? fmaxf(1.5f * d, 0.75f * w.need[c]) : 0.0f;
    }
    if (tid == 0) {
        sh->cnt.fallbacks++;
        sh->cs.list_valid = 0u;
        // a base skin driven below its floor by lists that did not fit starts
        // over from the usual one
        sh->cs.skin = fmaxf(sh->cs.skin, 0.05f * fmaxf(rmax, 1e-3f));
    }
    __syncthreads();
}

// The sweep's active lists: of each circle's candidates those that can touch
// it during this sweep.  Circle c has a margin m_c = max(base, need_c) for its
// pushes in one sweep, and (c, o) is active when the two are now closer than
// (r_c + m_c) + (r_o + m_o); both ends find it, since the test is symmetric.  A
// candidate left out was further apart than the radii and both margins, so it
// stays a no-op while its circles keep within them (near_check looks at those
// that do not).  The candidate skins, sized to last many sweeps, are far larger
// than one sweep's pushes: on a soft body in contact most candidates are the
// lattice neighbours, which never touch, and each would lengthen the chain of
// rounds.  A 100 x 100 body piling up ran 390 rounds a sweep over every
// candidate and runs 18 over the active ones (sweeps 0.49 -> 0.066 ms).
//
// The lists keep the candidates' order, each followed by kNone16.  A wavefront
// takes the room for its 64 lists with one atomic, in any order.  items[c] and
// key[c] get list c's place and length, st[c] its round state (see rounds_core).
// Returns the slots used; with more than cap of them nothing past cap is
// written, and the caller chooses another place.
// The base margin, in units of the largest radius, at level 0; each level
// doubles it.  A sweep that had to run again because a circle within its skin met a
// pair beyond its margin raises the scene's level by two, kLevelClean sweeps without
// one lower it: a
// settling pile stays at level 0 (its rounds grow with the margins), a hot gas,
// whose first contacts push circles by most of a radius, at the top (its rounds
// are few: 16,000 circles ran every sweep twice at level 0).  Circles beyond their
// skins meet such pairs too, a few in a pile that is being hit, where a second run of
// the sweep costs less than the level, but every third sweep in a gas that falls into
// a heap: they raise it once the second runs come closer together than the sweeps
// that heat takes to cool (16,000 circles falling, 320 sweeps: 111 second runs and
// 4.02 ms an update without, 8 and 3.55 with).  All of it is
// kept between launches: counted anew in each, a launch of fewer than kLevelClean
// sweeps could only raise the level (4,096 soft bodies piled up, 8 sweeps a launch:
// 6.0e6 rounds and 26.0 ms an update, 3.6e6 and 23.7 with the count kept).  A level
// given up too soon costs a second run of the sweep, one kept too long longer rounds
// (those bodies, and batches of 96 piles from their first contact, 8 updates each: 32
// clean sweeps 23.6 and 15.10 ms, 48 24.0 and 15.06, 64 23.7 and 14.95; piles settling
// for 30 updates 48.5, 48.8 and 49.3, 52.7 at a level that never falls).
constexpr float kActiveBase = 0.05f;
constexpr uint32_t kLevels = 4u, kLevelClean = 64u;
constexpr uint32_t kHeatMiss = 5u, kHeatRaise = 13u;  // one off a clean sweep
static_assert(kLevels < 8u && kLevelClean <= 128u && kHeatRaise <= 16u, "kept between launches in 3, 7 and 4 bits");
constexpr uint32_t kCurMask = 0x00ffffffu;
constexpr uint32_t kStamp8 = 0xffu;
static_assert(kCandCap * 65536ull <= kCurMask + 1ull, "a list cursor must fit 24 bits");

template <int WG, typename STP, typename LSP>
__device__ __forceinline__ uint32_t prune_lists(const float2 *Pc, uint32_t Nc, const float *crad, bool uni_r,
                                                float runi, float mbase, float mscale, const CCWork &w, CCShared *sh,
                                                STP st, LSP list, uint32_t cap) {
    const uint32_t lane = threadIdx.x & 63u;
    BD_GLOBAL const float *const need = to_global((const float *)w.need);
    BD_GLOBAL const float *const rad = to_global(crad);
    BD_GLOBAL const uint16_t *const cand = to_global((const uint16_t *)w.cand);
    if (threadIdx.x == 0) sh->nact = 0u;
    __syncthreads();
#pragma unroll 1
    for (uint32_t c0 = threadIdx.x - lane; c0 < Nc; c0 += WG) {
        const uint32_t c = c0 + lane;
        uint32_t n = 0, len = 0, o0 = 0;
        uint32_t mask = 0;
        float2 p = make_float2(0.0f, 0.0f);
        float ec = 0.0f;
        auto active = [&](uint32_t o) {
            const float2 q = Pc[o];
            const float eo = (uni_r ? runi : rad[o]) + mscale * fmaxf(mbase, need[o]);
            const float dx = p.x - q.x, dy = p.y - q.y, lim = ec + eo;
            return dx * dx + dy * dy < lim * lim;
        };
        if (c < Nc) {
            p = Pc[c];
            w.save[c] = p;
            n = w.cnt[c];
            o0 = w.off[c];
            ec = (uni_r ? runi : rad[c]) + mscale * fmaxf(mbase, need[c]);
#pragma unroll 1
            for (uint32_t k = 0; k < n; k += 4u) {
                // four candidates at a time (the last one again past the end)
                uint32_t o[4];
#pragma unroll
                for (uint32_t u = 0; u < 4u; u++) o[u] = cand[o0 + min(k + u, n - 1u)];
#pragma unroll
                for (uint32_t u = 0; u < 4u; u++) {
                    const bool on = k + u < n && active(o[u]);
                    if (on && k + u < 32u) mask |= 1u << (k + u);
                    len += on ? 1u : 0u;
                }
            }
        }
        // room for the wavefront's lists, and a terminator for each that is not empty
        const uint32_t want = len ? len + 1u : 0u;
        const uint32_t inc = __ockl_wfscan_add_u32(want, true);
        uint32_t base = 0;
        if (lane == 63u) base = inc ? atomicAdd(&sh->nact, inc) : 0u;
        base = __builtin_amdgcn_readlane(base, 63);
        const uint32_t at = base + inc - want;
        if (c < Nc) {
            w.items[c] = len ? at : 0u;
            w.key[c] = len;
            uint32_t n1 = kNone16, n2 = kNone16;
            if (len && at + want <= cap) {
                uint32_t j = 0;
                auto put = [&](uint32_t o) {
                    if (j == 0u) n1 = o;
                    if (j == 1u) n2 = o;
                    list[at + j] = (uint16_t)o;
                    j++;
                };
                if (n <= 32u) {
#pragma unroll 1
                    for (uint32_t m = mask; m; m &= m - 1u) put(cand[o0 + (uint32_t)__ffs(m) - 1u]);
                } else {
#pragma unroll 1
                    for (uint32_t k = 0; k < n; k++) {
                        const uint32_t o = cand[o0 + k];
                        if (active(o)) put(o);
                    }
                }
                list[at + j] = (uint16_t)kNone16;
            }
            st[c] = (uint64_t)((len ? at : 0u) | (kStamp8 << 24)) | ((uint64_t)(n1 | (n2 << 16)) << 32);
        }
    }
    __syncthreads();
    return uni(sh->nact);
}

// The rounds of one sweep over its active lists.  Per circle 64 bits of state
// (st): its cursor in the lists (24 bits) with the round in which it last moved
// (8 bits, kStamp8 for none), its next partner and the partner after that (16
// bits each, kNone16 for none).  Pair (x, y) is ready exactly when each is the
// other's next partner.
//
// A round is a chain of dependent accesses: the pair, its circles' states and
// positions, the states of their new partners, the slots of the pairs that
// became ready.  With the lists in LDS (LL) a circle's partner after next is
// read and stored at once; with lists in global memory that load is issued
// after the pair is solved and before its stores (vector memory operations
// complete in order, stores included) and waited for at the end of the round.
// Rounds with at most 64 ready pairs run on the first wavefront alone, without
// workgroup barriers, and hand out worklist slots by ballots instead of
// atomics; the solve overlaps the readiness reads, which need no position
// (1.1 -> 0.5 us a round with the lists in LDS).
template <int WG, bool LL, typename PCP, typename STP, typename LSP>
__device__ __forceinline__ void rounds_core(PCP Pc, uint32_t Nc, const float *crad_, bool uni_r, float runi,
                                            CCShared *sh, uint32_t *s_wl_, STP st, LSP list) {
    const int tid = threadIdx.x;
    const CCWork &ww = sh->work;
    BD_GLOBAL const uint32_t *const aoff = to_global((const uint32_t *)ww.items);
    BD_GLOBAL float *const path = to_global(ww.path);
    BD_GLOBAL const uint64_t *const save = to_global((const uint64_t *)ww.save);  // f32x2 as their bits
    BD_GLOBAL uint64_t *const traj = to_global((uint64_t *)ww.traj);
    auto bits = [](float2 v) { return (uint64_t)__float_as_uint(v.x) | ((uint64_t)__float_as_uint(v.y) << 32); };
    auto f32x2 = [](uint64_t b) { return make_float2(__uint_as_float((uint32_t)b), __uint_as_float((uint32_t)(b >> 32))); };
    auto next = [](uint64_t s) { return (uint32_t)(s >> 32) & 0xffffu; };
    BD_GLOBAL const float *const crad = to_global(crad_);
    // worklists: the first WG ready pairs of a round in LDS (s_wl, two
    // buffers of WG), the rest in HBM at the same index
    BD_LDS uint32_t *const s_wl = to_lds(s_wl_);
    BD_GLOBAL uint32_t *const gwl[2] = {to_global(ww.wl), to_global(ww.wl) + (Nc / 2 + 1)};
    auto wl_put = [&](uint32_t b, uint32_t i, uint32_t v) {
        if (i < (uint32_t)WG) s_wl[b * WG + i] = v; else gwl[b][i] = v;
    };
    auto wl_get = [&](uint32_t b, uint32_t i) { return i < (uint32_t)WG ? s_wl[b * WG + i] : gwl[b][i]; };
    // the partner after the next one's successor is at cursor + 2, where there
    // is a successor (its list goes on to the terminator at least)
    auto after = [&](uint32_t u, uint32_t x) { return list[x == kNone16 ? u : u + 2u]; };
    auto state = [](uint32_t u, uint32_t r8, uint32_t x, uint32_t y) {
        return (uint64_t)(u | (r8 << 24)) | ((uint64_t)(x | (y << 16)) << 32);
    };
    auto ready = [](uint32_t x, uint32_t y, uint64_t sy, uint32_t r8) {
        // y's next partner is x; when both moved the smaller one adds the pair
        return y != kNone16 && ((uint32_t)(sy >> 32) & 0xffffu) == x && !(((uint32_t)sy >> 24) == r8 && y < x);
    };
    auto pair_of = [](uint32_t x, uint32_t y) { return x < y ? x | (y << 16) : y | (x << 16); };
    if (tid == 0) { sh->cnt3[0] = 0u; sh->cnt3[1] = 0u; sh->cnt3[2] = 0u; sh->stalled = 0u; }
    __syncthreads();
#pragma unroll 1
    for (uint32_t c = tid; c < Nc; c += WG) {
        const uint32_t o = next(st[c]);
        if (o != kNone16 && c < o && next(st[o]) == c) wl_put(0, atomicAdd(&sh->cnt3[0], 1u), c | (o << 16));
    }
    __syncthreads();
    uint32_t n = uni(sh->cnt3[0]);
    uint32_t r = 0, r8 = 0;
    // every 255 rounds: no stamp may match a round number about to recur
    auto clear_stamps = [&](uint32_t first, uint32_t stride) {
#pragma unroll 1
        for (uint32_t c = first; c < Nc; c += stride) st[c] = st[c] | ((uint64_t)kStamp8 << 24);
    };
    __shared__ uint32_t s_rr[3];
    auto wave_rounds = [&]() {
        const uint32_t lane = threadIdx.x & 63u;
        const uint32_t r0 = r;
#pragma unroll 1
        do {
            const uint32_t cb = r & 1u, nb = cb ^ 1u;
            const bool first = lane < n;
            uint32_t c = 0, o = 0, xc = kNone16, xo = kNone16, uc = 0, uo = 0;
            uint64_t qc = 0, qo = 0;
            float2 pi = make_float2(0.0f, 0.0f), pj = pi;
            uint16_t fyc = 0, fyo = 0;
            if (first) {
                const uint32_t pr = s_wl[cb * WG + lane];
                c = pr & 0xffffu;
                o = pr >> 16;
                const uint64_t sc = st[c], so = st[o];
                pi = f32x2(Pc[c]);
                pj = f32x2(Pc[o]);
                uc = (uint32_t)sc & kCurMask;
                uo = (uint32_t)so & kCurMask;
                xc = (uint32_t)(sc >> 48);
                xo = (uint32_t)(so >> 48);
                uint32_t yc = kNone16, yo = kNone16;
                if constexpr (LL) {
                    const uint32_t lc = after(uc, xc), lo = after(uo, xo);
                    yc = xc == kNone16 ? kNone16 : lc;
                    yo = xo == kNone16 ? kNone16 : lo;
                }
                st[c] = state(uc + 1u, r8, xc, yc);
                st[o] = state(uo + 1u, r8, xo, yo);
            }
            wave_sync();
            if (first) {
                qc = st[xc == kNone16 ? c : xc];
                qo = st[xo == kNone16 ? o : xo];
                float qi = 0.0f, qj = 0.0f;
                const float rc = uni_r ? runi : crad[c], ro = uni_r ? runi : crad[o];
                const bool touch = solve_circle_pair(pi.x, pi.y, pj.x, pj.y, rc, ro, qi, qj);
                if constexpr (!LL) {
                    __builtin_amdgcn_sched_barrier(0);
                    fyc = after(uc, xc);
                    fyo = after(uo, xo);
                    __builtin_amdgcn_sched_barrier(0);
                }
                if (touch) {
                    Pc[c] = bits(pi);
                    Pc[o] = bits(pj);
                }
                // each circle's position after each of its pairs, in list order:
                // its excursion from the sweep's start is taken from these
                traj[uc] = bits(pi);
                traj[uo] = bits(pj);
            }
            const bool a0 = first && ready(c, xc, qc, r8), a1 = first && ready(o, xo, qo, r8);
            const uint64_t b0 = __ballot(a0), b1 = __ballot(a1);
            const uint32_t n0 = (uint32_t)__popcll(b0);
            if (a0) wl_put(nb, __builtin_amdgcn_mbcnt_hi((uint32_t)(b0 >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)b0, 0u)),
                           pair_of(c, xc));
            if (a1) wl_put(nb, n0 + __builtin_amdgcn_mbcnt_hi((uint32_t)(b1 >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)b1, 0u)),
                           pair_of(o, xo));
            if constexpr (!LL) {
                if (first) {
                    if (xc != kNone16) st[c] = state(uc + 1u, r8, xc, fyc);
                    if (xo != kNone16) st[o] = state(uo + 1u, r8, xo, fyo);
                }
            }
            wave_sync();
            n = n0 + (uint32_t)__popcll(b1);
            if (++r8 == kStamp8) {
                clear_stamps(lane, 64u);
                wave_sync();
                r8 = 0u;
            }
            r++;
        } while (n > 0 && n <= 64u);
        if (lane == 0) {
            sh->cnt.rounds += r - r0;
            sh->cnt3[0] = 0u; sh->cnt3[1] = 0u; sh->cnt3[2] = 0u;
            s_rr[0] = r; s_rr[1] = r8; s_rr[2] = n;
        }
    };
#pragma unroll 1
    while (n > 0) {
        if (n <= 64u) {
            if (tid < 64) wave_rounds();
            __syncthreads();
            r = uni(s_rr[0]);
            r8 = uni(s_rr[1]);
            n = uni(s_rr[2]);
            __syncthreads();  // s_rr is read before a later pass of the first wavefront writes it
            continue;
        }
        const uint32_t cb = r & 1u, nb = cb ^ 1u;
        if (tid == 0) sh->cnt3[(r + 2) % 3] = 0u;  // read at the end of round r-1, two barriers ago
        // the pairs: solve, step both cursors
#pragma unroll 1
        for (uint32_t k = tid; k < n; k += WG) {
            const uint32_t pr = wl_get(cb, k), c = pr & 0xffffu, o = pr >> 16;
            const uint64_t sc = st[c], so = st[o];
            float2 pi = f32x2(Pc[c]), pj = f32x2(Pc[o]);
            const uint32_t uc = (uint32_t)sc & kCurMask, uo = (uint32_t)so & kCurMask;
            const uint32_t xc = (uint32_t)(sc >> 48), xo = (uint32_t)(so >> 48);
            const uint32_t lc = after(uc, xc), lo = after(uo, xo);
            float qi = 0.0f, qj = 0.0f;
            const float rc = uni_r ? runi : crad[c], ro = uni_r ? runi : crad[o];
            if (solve_circle_pair(pi.x, pi.y, pj.x, pj.y, rc, ro, qi, qj)) {
                Pc[c] = bits(pi);
                Pc[o] = bits(pj);
            }
            st[c] = state(uc + 1u, r8, xc, xc == kNone16 ? kNone16 : lc);
            st[o] = state(uo + 1u, r8, xo, xo == kNone16 ? kNone16 : lo);
            traj[uc] = bits(pi);
            traj[uo] = bits(pj);
        }
        __syncthreads();
        // pairs completed by a circle that moved
#pragma unroll 1
        for (uint32_t k = tid; k < n; k += WG) {
            const uint32_t pr = wl_get(cb, k);
#pragma unroll 1
            for (int e = 0; e < 2; e++) {
                const uint32_t x = e ? pr >> 16 : pr & 0xffffu, y = next(st[x]);
                if (ready(x, y, st[y == kNone16 ? x : y], r8))
                    wl_put(nb, atomicAdd(&sh->cnt3[(r + 1) % 3], 1u), pair_of(x, y));
            }
        }
        __syncthreads();
        n = uni(sh->cnt3[(r + 1) % 3]);
        if (tid == 0) sh->cnt.rounds++;
        if (++r8 == kStamp8) {
            clear_stamps(tid, WG);
            __syncthreads();
            r8 = 0u;
        }
        r++;
    }
    // each circle's largest excursion from its start position (the running
    // maximum over its positions after its pairs, in their order: a pair that
    // did not touch repeats the position before it); every list must be done
#pragma unroll 1
    for (uint32_t c = tid; c < Nc; c += WG) {
        const uint64_t s = st[c];
        const uint32_t o0 = aoff[c], u1 = (uint32_t)s & kCurMask;
        if (next(s) != kNone16) sh->stalled = 1u;
        const float2 sv = f32x2(save[c]);
        float pth = 0.0f;
#pragma unroll 4
        for (uint32_t u = o0; u < u1; u++) {
            const float2 q = f32x2(traj[u]);
            pth = excursion(pth, q.x, q.y, sv.x, sv.y);
        }
        path[c] = pth;
    }
}

// The active lists and rounds of one sweep, out of line: the sweep's list
// builds and the kernel's link and body phases keep their registers.  The round
// state (8 bytes a circle) sits in the LDS the scene leaves free, or, for a
// sweep with enough candidate pairs to pay for two copies, in place of the
// circles' previous positions (held in LDS, unused by the sweep) or of their
// positions (the rounds then work on the global copy), parked in global memory
// meanwhile; else in the workspace (head, stamp).  The lists go into the LDS
// still free when they fit, else behind the trajectories in the workspace.  The
// code is instantiated for each placement, so LDS is addressed as LDS.  Parked
// positions go back at the end; the lists stay for the checks.  Returns the
// active list slots, 0 when no pair is active (nothing has run then), kNone
// when the workspace cannot hold the lists.
template <int WG>
__device__ __noinline__ uint32_t sweep_rounds(float2 *P, uint32_t Np, uint32_t Nc, const float *crad, bool uni_r,
                                              float runi, float mbase, float mscale, CCShared *sh, uint32_t *s_wl,
                                              uint32_t pairs) {
    extern __shared__ float2 s_dyn[];
    const int tid = threadIdx.x;
    const CCWork &w = sh->work;
    const CCShared::Fallback &fb = sh->fb;
    float2 *Pc = P + Np, *pl = nullptr, *pg = nullptr;
    uint32_t st_off = kNone, l_off = sh->free_off, l_bytes = sh->free_bytes;
    if (l_bytes >= 8u * Nc) {
        st_off = l_off;
        l_off += 8u * Nc;
        l_bytes -= 8u * Nc;
    } else if (pairs >= kParkPairs) {
        if (fb.q_lds) {
            pl = fb.q_lds + Np;
            pg = fb.q_global + Np;
        } else if (fb.p_global) {
            pl = P + Np;
            pg = fb.p_global + Np;
            Pc = pg;
        }
        if (pl) {
#pragma unroll 1
            for (uint32_t c = tid; c < Nc; c += WG) pg[c] = pl[c];
            __syncthreads();
            st_off = (uint32_t)((uint8_t *)pl - (uint8_t *)s_dyn);
        }
    }
    // the positions as 64-bit words, typed by where they are (LDS, or global
    // memory for a scene without them in LDS or with them parked): a generic
    // LDS address carries the LDS aperture in its high half
    const bool pc_lds = ((uint64_t)Pc >> 32) == ((uint64_t)s_dyn >> 32);
    uint32_t total = 0;
    // lists behind the trajectories (8 bytes a slot): at most gcap slots
    const uint32_t gcap = (uint32_t)(8ull * kCandCap * Nc / 10u);
    uint16_t *glist = nullptr;
    auto place = [&](uint32_t slots) { glist = (uint16_t *)(w.traj + slots); };
    auto run = [&](auto st) {
        // in LDS when they fit (the first pass finds out), else in the workspace
        total = prune_lists<WG>(Pc, Nc, crad, uni_r, runi, mbase, mscale, w, sh, st,
                                to_lds((uint16_t *)((uint8_t *)s_dyn + l_off)), l_bytes / 2u);
        if (total == 0u) return;
        const bool ll = total <= l_bytes / 2u;
        if (ll) {
            if (tid == 0) sh->act = (const uint16_t *)((uint8_t *)s_dyn + l_off);
            if (pc_lds)
                rounds_core<WG, true>(to_lds((uint64_t *)Pc), Nc, crad, uni_r, runi, sh, s_wl, st,
                                      to_lds((const uint16_t *)((uint8_t *)s_dyn + l_off)));
            else
                rounds_core<WG, true>(to_global((uint64_t *)Pc), Nc, crad, uni_r, runi, sh, s_wl, st,
                                      to_lds((const uint16_t *)((uint8_t *)s_dyn + l_off)));
            return;
        }
        if (total > gcap) { total = kNone; return; }
        place(total);
        __syncthreads();
        prune_lists<WG>(Pc, Nc, crad, uni_r, runi, mbase, mscale, w, sh, st, to_global(glist), total);
        if (tid == 0) sh->act = glist;
        if (pc_lds)
            rounds_core<WG, false>(to_lds((uint64_t *)Pc), Nc, crad, uni_r, runi, sh, s_wl, st,
                                   to_global((const uint16_t *)glist));
        else
            rounds_core<WG, false>(to_global((uint64_t *)Pc), Nc, crad, uni_r, runi, sh, s_wl, st,
                                   to_global((const uint16_t *)glist));
    };
    if (st_off != kNone) run(to_lds((uint64_t *)((uint8_t *)s_dyn + st_off)));
    else run(to_global((uint64_t *)w.head));
    __syncthreads();  // the state has been read for the last time; act and stalled are set
    if (pl) {
#pragma unroll 1
        for (uint32_t c = tid; c < Nc; c += WG) pl[c] = pg[c];
        __syncthreads();
    }
    return total;
}

// Ascending partner order (the reference's pair order) for every candidate
// list: short lists by their thread, longer ones by a wavefront, the longest by
// the workgroup (queued at the two ends of wl).  Returns the longest list.
template <int WG>
__device__ __noinline__ uint32_t sort_lists(uint32_t Nc_, CCShared *sh, float *s_red) {
    const int tid = threadIdx.x;
    const uint32_t Nc = uni(Nc_);
    const CCWork &w = sh->work;
    if (tid == 0) { sh->nmid = 0u; sh->nlong = 0u; }
    __syncthreads();
    const uint32_t wl_end = 2u * (Nc / 2u + 1u) - 1u;
    uint32_t longest = 0;
    for (uint32_t c = tid; c < Nc; c += WG) {
        uint16_t *my = w.cand + w.off[c];
        const uint32_t n = w.cnt[c];
        longest = max(longest, n);
        if (n <= 1u) continue;
        if (n <= 8u) sort_in_registers<8>(my, n);
        else if (WG < 1024 && n <= 16u) sort_in_registers<16>(my, n);
        // 32 registers more than a 1,024-lane workgroup's 128 allow
        // without spilling: there such lists go to a wavefront
        else if (WG < 1024 && n <= 32u) sort_in_registers<(WG < 1024 ? 32 : 16)>(my, n);
        else if (n <= kMidList) w.wl[atomicAdd(&sh->nmid, 1u)] = c;
        else w.wl[wl_end - atomicAdd(&sh->nlong, 1u)] = c;
    }
    __syncthreads();
    const uint32_t nmid = uni(sh->nmid), nlong = uni(sh->nlong);
    for (uint32_t q = tid >> 6; q < nmid; q += WG / 64) {
        const uint32_t c = w.wl[q];
        sort_by_wave(w.cand + w.off[c], w.cnt[c]);
    }
    for (uint32_t q = 0; q < nlong; q++) {
        const uint32_t c = w.wl[wl_end - q], n = w.cnt[c];
        uint16_t *my = w.cand + w.off[c];
        for (uint32_t k = tid; k < n; k += WG) w.items[k] = my[k];
        __syncthreads();
        // partners are distinct, so the ranks are a permutation of [0, n)
        for (uint32_t k = tid; k < n; k += WG) {
            const uint32_t v = w.items[k];
            uint32_t rank = 0;
            for (uint32_t j2 = 0; j2 < n; j2++) rank += w.items[j2] < v ? 1u : 0u;
            my[rank] = (uint16_t)v;
        }
        __syncthreads();
    }
    __syncthreads();
    return (uint32_t)wg_max<WG>((float)longest, s_red);
}

// The circles' records in bucket order (rec, start), their positions now in ref.
// The counters are in LDS: 16 bits each, two to a word, so a circle's rank in its
// bucket comes back from the count itself (kept with the bucket in key).
template <int WG>
__device__ __noinline__ void grid_in_lds(const float2 *P, uint32_t Np_, const float *crad, CCGrid g, float s_cell,
                                         uint32_t lds_off_, const CCWork &w, uint32_t *s_wave) {
    extern __shared__ float2 s_dyn[];
    const uint32_t tid = threadIdx.x, Np = uni(Np_), Nc = uni(g.Nc), T = uni(g.T);
    BD_LDS uint32_t *const word = to_lds((uint32_t *)((uint8_t *)s_dyn + uni(lds_off_)));
    BD_LDS uint16_t *const half = (BD_LDS uint16_t *)word;
    BD_GLOBAL u32x2 *const start = to_global((u32x2 *)w.start);
    BD_GLOBAL f32x2 *const ref = to_global((f32x2 *)w.ref);
    BD_GLOBAL uint32_t *const key = to_global(w.key);
    BD_GLOBAL const float *const skin = to_global((const float *)w.skin), *const rad = to_global(crad);
    BD_GLOBAL f32x4 *const rec = to_global((f32x4 *)w.rec);
    const uint32_t words = T >> 1;  // (T is even)
    for (uint32_t b = tid; b < words; b += WG) word[b] = 0u;
    __syncthreads();
#pragma unroll 2
    for (uint32_t c = tid; c < Nc; c += WG) {
        const float2 p = P[Np + c];
        ref[c] = f32x2{p.x, p.y};
        const uint32_t kk = grid_bucket(g, (uint32_t)scell(p.x, g.inv_h), (uint32_t)scell(p.y, g.inv_h));
        const uint32_t sft = (kk & 1u) * 16u;
        const uint32_t old = __hip_atomic_fetch_add(word + (kk >> 1), 1u << sft, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        key[c] = kk | ((old >> sft) & 0xffffu) << 16;
    }
    __syncthreads();
    // exclusive scan: a lane takes a run of words
    const uint32_t per = (words + WG - 1u) / WG, w0 = min(words, tid * per), w1 = min(words, w0 + per);
    uint32_t sum = 0;
    for (uint32_t i = w0; i < w1; i++) {
        const uint32_t v = word[i];
        sum += (v & 0xffffu) + (v >> 16);
    }
    const uint32_t inc = __ockl_wfscan_add_u32(sum, true), wave = uni(tid >> 6);
    if ((tid & 63u) == 63u) s_wave[wave] = inc;
    __syncthreads();
    uint32_t run = inc - sum;
#pragma unroll 1
    for (uint32_t v = 0; v < wave; v++) run += s_wave[v];
    for (uint32_t i = w0; i < w1; i++) {
        const uint32_t v = word[i], mid = run + (v & 0xffffu);
        word[i] = run | mid << 16;
        start[i] = u32x2{run, mid};
        run = mid + (v >> 16);
    }
    if (tid == 0) {
        half[T] = (uint16_t)Nc;
        w.start[T] = Nc;
    }
    __syncthreads();
#pragma unroll 2
    for (uint32_t c = tid; c < Nc; c += WG) {
        const uint32_t k = key[c];
        const f32x2 p = ref[c];
        const float sk = skin[c];
        rec[half[k & 0xffffu] + (k >> 16)] =
            f32x4{p.x, p.y, rad[c] + sk, __uint_as_float(c | (sk > s_cell ? kOutlierBit : 0u))};
    }
    __syncthreads();
}

// The same with the counters in the workspace (start, fill).
template <int WG>
__device__ __noinline__ void grid_in_memory(const float2 *P, uint32_t Np_, const float *crad, CCGrid g,
                                            float s_cell, const CCWork &w, uint32_t *s_wave) {
    const uint32_t tid = threadIdx.x, Np = uni(Np_), Nc = uni(g.Nc), T = uni(g.T);
    for (uint32_t b = tid; b < T; b += WG) { w.start[b] = 0u; w.fill[b] = 0u; }
    __syncthreads();
    for (uint32_t c = tid; c < Nc; c += WG) {
        const float2 p = P[Np + c];
        w.ref[c] = p;
        const uint32_t kk = grid_bucket(g, (uint32_t)scell(p.x, g.inv_h), (uint32_t)scell(p.y, g.inv_h));
        w.key[c] = kk;
        atomicAdd(&w.start[kk], 1u);
    }
    __syncthreads();
    wg_scan_global<WG>(w.start, w.start, T, s_wave);  // bucket k = [start[k], start[k+1])
    for (uint32_t c = tid; c < Nc; c += WG) {
        const uint32_t kk = w.key[c];
        const float2 p = w.ref[c];
        const float sk = w.skin[c];
        w.rec[w.start[kk] + atomicAdd(&w.fill[kk], 1u)] =
            make_float4(p.x, p.y, crad[c] + sk, __uint_as_float(c | (sk > s_cell ? kOutlierBit : 0u)));
    }
    __syncthreads();
}

// A new candidate list for the circles where they are now.  The schedule's state
// (skins, thresholds, pair count) goes to cs.  Returns 0, 1 when the list does
// not fit the workspace (the skins have been reduced: try again), 2 when not
// even the smallest skins fit.
template <int WG>
__device__ __noinline__ uint32_t build_lists(const float2 *P, uint32_t Np_, uint32_t Nc_, const float *crad,
                                             float rmax_, uint32_t T_, CCShared *sh, float *s_red, uint32_t *s_u32,
                                             uint32_t *s_wl) {
    const int tid = threadIdx.x;
    const uint32_t Np = uni(Np_), Nc = uni(Nc_), T = uni(T_);
    const float rmax = uni(rmax_);
    const CCWork &w = sh->work;
    float sbase = uni(sh->cs.skin);
    const uint32_t since_build = uni(sh->cs.since_build);
    __syncthreads();  // cs has been read: lane 0 writes it below
    if (tid == 0) sh->cnt.rebuilds++;
    const uint64_t tb0 = wall_clock64();
    // per-circle skins: the base, or what the circle's recent sweeps pushed it;
    // s_cell: the skin at most kOutCap circles exceed (log2 histogram)
    if (tid <= 32) sh->hist[tid] = 0u;
    __syncthreads();
    float smax = 0.0f, nsmin = -INFINITY;
    for (uint32_t c = tid; c < Nc; c += WG) {
        float sk = fmaxf(sbase, w.need[c]);
        w.skin[c] = sk;
        smax = fmaxf(smax, sk);
        nsmin = fmaxf(nsmin, -sk);
        if (sk > sbase)
            atomicAdd(&sh->hist[sk <= 3.0e38f ? min(32, 1 + (int)floorf(log2f(sk / sbase))) : 32], 1u);
    }
    smax = wg_max<WG>(smax, s_red);
    const float smin = -wg_max<WG>(nsmin, s_red);
    int B = 0;
    {
        uint32_t above = 0;
        for (int b = 32; b >= 1; b--) {
            if (above + sh->hist[b] > kOutCap) { B = b; break; }
            above += sh->hist[b];
        }
    }
    const float s_cell = uni(fminf(smax, sbase * exp2f((float)B)));
    if (tid == 0) sh->nout = 0u;
    __syncthreads();
    for (uint32_t c = tid; c < Nc; c += WG)
        if (w.skin[c] > s_cell) sh->out[atomicAdd(&sh->nout, 1u)] = (uint16_t)c;
    __syncthreads();
    const uint32_t n_out = uni(sh->nout);
    const double h = cell_size(rmax, s_cell);
    const CCGrid g = cc_grid(Np, Nc, T, h, w.start);
    const uint32_t lds_off = sh->free_off;
    // the buckets' counters in the free LDS when they fit (two to a word, and one
    // more for the end)
    const bool in_lds = 2u * g.T + 4u <= sh->free_bytes && Nc < 65536u;
    if (in_lds) grid_in_lds<WG>(P, Np, crad, g, s_cell, lds_off, w, s_u32);
    else grid_in_memory<WG>(P, Np, crad, g, s_cell, w, s_u32);
    // counts: normal circles gather their normal partners into a slot of
    // kSlot entries (in traj, free until the sweep) and keep the count in
    // stamp; then outliers add themselves to their partners' counts
    uint16_t *const slot = (uint16_t *)w.traj;
    auto gather = [&](uint32_t c, uint16_t *out, uint32_t cap) {
        const float2 p = w.ref[c];
        const float ec = crad[c] + w.skin[c];
        return in_lds ? gather_normal<true>(c, w, g, lds_off, p, ec, out, cap)
                      : gather_normal<false>(c, w, g, lds_off, p, ec, out, cap);
    };
    for (uint32_t c = tid; c < Nc; c += WG) {
        const uint32_t n = w.skin[c] > s_cell ? 0u : gather(c, slot + (size_t)c * kSlot, kSlot);
        w.cnt[c] = n;
        w.stamp[c] = n;
    }
    __syncthreads();
    uint32_t n_far = 0u;
    if (n_out) {
        n_far = in_lds ? gather_outliers<WG, 0, true>(w, g, lds_off, crad, sh->out, n_out, rmax, s_cell, h, nullptr,
                                                      (float4 *)s_wl, s_u32)
                       : gather_outliers<WG, 0, false>(w, g, lds_off, crad, sh->out, n_out, rmax, s_cell, h, nullptr,
                                                       (float4 *)s_wl, s_u32);
        __syncthreads();
    }
    const uint64_t tb1 = wall_clock64();
    wg_scan_global<WG>(w.cnt, w.off, Nc, s_u32);
    const uint32_t total = uni(w.off[Nc]);
    // (one slot a circle stays for the active lists' terminators)
    if (total > (kCandCap - 1u) * Nc) {
        // more candidates than the workspace holds: first the outlying
        // skins come down to the outlier threshold (they list the most
        // partners), and only with no outliers left the base skin
        // shrinks; the skins the other circles showed they need stay
        __syncthreads();
        if (n_out) {
            for (uint32_t c = tid; c < Nc; c += WG) w.need[c] = fminf(w.need[c], 0.5f * s_cell);
        } else {
            sbase = 0.7f * sbase;
            for (uint32_t c = tid; c < Nc; c += WG) w.need[c] = fminf(w.need[c], sbase);
        }
        if (tid == 0) sh->cs.skin = sbase;
        return sbase < 1e-4f * fmaxf(rmax, 1e-3f) ? 2u : 1u;
    }
    // lists: normal partners first (from the slot, or gathered again when
    // they did not fit it), outliers append at a cursor (in head)
    for (uint32_t c = tid; c < Nc; c += WG) {
        uint32_t own = 0;
        if (w.skin[c] <= s_cell) {
            own = w.stamp[c];
            uint16_t *dst = w.cand + w.off[c];
            if (own <= kSlot) {
                const uint16_t *src = slot + (size_t)c * kSlot;
                for (uint32_t i = 0; i < own; i++) dst[i] = src[i];
            } else {
                gather(c, dst, own);
            }
        }
        w.head[c] = w.off[c] + own;
    }
    __syncthreads();
    if (n_out) {
        if (in_lds)
            gather_outliers<WG, 1, true>(w, g, lds_off, crad, sh->out, n_out, rmax, s_cell, h, w.head, (float4 *)s_wl,
                                         s_u32);
        else
            gather_outliers<WG, 1, false>(w, g, lds_off, crad, sh->out, n_out, rmax, s_cell, h, w.head, (float4 *)s_wl,
                                          s_u32);
        __syncthreads();
    }
    const uint64_t tb2 = wall_clock64();
    const uint32_t max_list = uni(sort_lists<WG>(Nc, sh, s_red));
    // base skin: rebuilds every few sweeps cost more than larger lists
    if (since_build < 4) sbase = fminf(1.25f * sbase, 0.5f * fmaxf(rmax, 1e-3f));
    else if (since_build > 32) sbase = fmaxf(0.8f * sbase, 0.05f * fmaxf(rmax, 1e-3f));
    const uint64_t tb3 = wall_clock64();
    if (tid == 0) {
        sh->cs = CCShared::Steer{sbase, 1u, total / 2, 0u, s_cell, smin, sh->cs.level, sh->cs.clean, sh->cs.heat};
        sh->cnt.n_out = n_out;
        sh->cnt.n_far = n_far;
        sh->cnt.smax = smax;
        sh->cnt.max_list = max_list;
        sh->cnt.t_build += tb3 - tb0;
        sh->cnt.t_count += tb1 - tb0;
        sh->cnt.t_lists += tb2 - tb1;
        sh->cnt.t_sort += tb3 - tb2;
    }
    return 0u;
}

// One circle-pair sweep of a scene (src/solver.rs:168-177), exact: of the
// candidate pairs those that can touch this time (prune_lists) run in rounds;
// pair (c, o), c < o, is ready when o is the smallest unprocessed partner of c
// and c that of o, so every earlier pair (in the reference's (i, j) order)
// sharing c or o has run.  Ready pairs share no circle.  After a round only
// circles that moved can complete a new ready pair, so each round looks at
// those alone (a worklist).  The sweep is valid when no circle's pushes took
// it beyond 0.8 of its active margin, nor beyond 0.8 of its skin since the
// candidate list was built (relative to a common shift of the scene): a pair not run
// started further apart than the sum of the two radii and margins, so it cannot
// have overlapped.  When some circles went further, near_check and
// overruns_check look at every pair of theirs that was not run; only if one of
// them touched is the sweep undone and rerun, first with wider active margins,
// then with a new candidate list and larger skins for the circles that moved.
// The list is rebuilt before a sweep when more circles than kDriftedBase +
// Nc / kDriftedShare (any, in scenes of fewer than kDriftedLeast) have drifted more
// than kDriftRebuild of their skins since it was built, or one of those has come into
// reach of a circle that it does not list.
// Returns the new error state (0 = fine).
template <int WG>
__device__ __noinline__ uint32_t circle_sweep(float2 *P, uint32_t Np_, uint32_t Nc_, const float *crad, bool uni_r_,
                                              float runi_, float rmax_, uint32_t T_, CCShared *sh, float *s_red,
                                              uint32_t *s_u32, uint32_t *s_wl) {
    const int tid = threadIdx.x;
    // arguments arrive in vector registers: the uniform ones back to scalars
    const uint32_t Np = uni(Np_), Nc = uni(Nc_), T = uni(T_);
    const bool uni_r = uni((uint32_t)uni_r_) != 0u;
    const float runi = uni(runi_), rmax = uni(rmax_);
    const CCWork &w = sh->work;
    CCShared::Steer &cs = sh->cs;  // written by lane 0, read after a barrier
    uint32_t widen = 0u;  // attempts of this sweep that left a touching pair out of the active lists
    // a scene whose lists just failed goes on without them for a few sweeps
    bool fallback = false;
    for (int attempt = uni(sh->fb_streak) != 0u ? kFallbackAttempt : 0;; attempt++) {
        if (fallback || attempt >= kFallbackAttempt) {
            // the lists keep failing: the sequential sweep, from the sweep's
            // start positions (P holds them: every redo restores them)
            fallback_sweep<WG>(P, Np, Nc, crad, uni_r, runi, rmax, T, w, sh);
            if (tid == 0) sh->fb_streak = sh->fb_streak ? sh->fb_streak - 1u : kFallbackStreak;
            __syncthreads();
            return 0u;
        }
        const float mbase = kActiveBase * (float)(1u << uni(cs.level)) * fmaxf(rmax, 1e-3f);
        bool rebuild = uni(cs.list_valid) == 0u;
        uint32_t drifted = 0u;  // circles beyond their skins before the sweep
        float2 u = make_float2(0.0f, 0.0f);
        if (!rebuild) {
            // drift since the list was built, relative to a common shift u, as a
            // fraction of each circle's skin (at most box / smallest skin, with
            // a margin for rounding, when the displacements' bounding box is
            // small; else each circle is measured)
            const Drift dr = drift_box<WG, true>(P, Np, Nc, w.ref, sh->red4);
            u = make_float2(dr.ux, dr.uy);
            if (!(drift_share(dr.box, uni(cs.smin)) <= kDriftRebuild)) {
                if (tid == 0) sh->nout = 0u;
                __syncthreads();
                float *vb = (float *)w.stamp;
                float vmax = 0.0f;
                for (uint32_t c = tid; c < Nc; c += WG) {
                    const float v = moved_bound(P[Np + c], w.ref[c], u, 0.0f);
                    const bool in = v <= kDriftRebuild * w.skin[c];
                    vb[c] = in ? v : -v;
                    if (in) {
                        vmax = fmaxf(vmax, v);
                    } else {
                        const uint32_t k = atomicAdd(&sh->nout, 1u);
                        if (k < kOutCap) sh->out[k] = (uint16_t)c;
                    }
                }
                vmax = wg_max<WG>(vmax, s_red);
                drifted = uni(sh->nout);
                rebuild = drifted > (Nc < kDriftedLeast ? 0u : min(kDriftedBase + Nc / kDriftedShare, kOutCap));
                if (drifted && !rebuild) {
                    const double h = cell_size(rmax, uni(cs.s_cell));
                    rebuild = drifted_meet<WG>(P, Np, w, crad, vb, sh->out, drifted, vmax, u, mbase, rmax, h,
                                               cc_grid(Np, Nc, T, h, w.start), s_red);
                }
            }
            // no candidate pair at all and every circle within its skin: no
            // pair can overlap during the sweep, which therefore changes nothing
            if (!rebuild && drifted == 0u && uni(cs.pairs) == 0u) {
                if (tid == 0) cs.since_build++;
                return 0u;
            }
        }
        if (rebuild) {
            if (tid == 0) cs.list_valid = 0u;
            const uint32_t rc = uni(build_lists<WG>(P, Np, Nc, crad, rmax, T, sh, s_red, s_u32, s_wl));
            __syncthreads();
            if (rc) {
                if (rc == 2u) fallback = true;
                continue;
            }
            u = make_float2(0.0f, 0.0f);
            drifted = 0u;
        }
        // ---- sweep: the active pairs in rounds
        // a redo widens the margins, then takes every candidate
        const float mscale = widen == 0u ? 1.0f : widen == 1u ? 4.0f : INFINITY;
        const uint32_t pairs = uni(cs.pairs);
        const uint32_t active =
            pairs || drifted ? uni(sweep_rounds<WG>(P, Np, Nc, crad, uni_r, runi, mbase, mscale, sh, s_wl, pairs)) : 0u;
        if (active == kNone) {
            // more pairs in reach of each other than the workspace holds
            if (widen == 0u) fallback = true;
            widen = 0u;
            if (tid == 0) cs.list_valid = 0u;
            __syncthreads();
            continue;
        }
        if (active == 0u && drifted == 0u) {
            // no pair can touch, and nothing has moved: the skins hold (the
            // drift since the list was built is within kDriftRebuild of them)
            for (uint32_t c = tid; c < Nc; c += WG) w.need[c] = 0.75f * w.need[c];
            if (tid == 0) cs.since_build++;
            return 0u;
        }
        // every list must be exhausted (a schedule that stalls is an error);
        // circles beyond 0.8 of their skin go to out[] (free after list builds)
        // and vb (stamp, free after the rounds) gets each circle's bound v,
        // negated for those
        // (the worklist array, free after the rounds, lists every overrun
        // circle when there are more than kOutCap); circles within their skin
        // but beyond 0.8 of their active margin go to fill (free after list
        // builds)
        float vmax = 0.0f, vall = 0.0f;
        float *vb = (float *)w.stamp;
        if (tid == 0) { sh->nout = 0u; sh->nnear = 0u; if (!active) sh->stalled = 0u; }
        __syncthreads();
        for (uint32_t c = tid; c < Nc; c += WG) {
            float pth = w.path[c];
            if (!active) w.path[c] = pth = 0.0f;  // no round has run
            const float nd = w.need[c];
            float v = moved_bound(w.save[c], w.ref[c], u, pth);
            // the sweep's own pushes, decaying slowly so circles in lasting contact keep their skin
            w.need[c] = (pth <= 3.0e38f) ? fmaxf(1.5f * pth, 0.75f * nd) : 0.0f;
            if (v <= 0.8f * w.skin[c]) {
                vmax = fmaxf(vmax, v);
                vb[c] = v;
                if (!(pth <= 0.8f * (mscale * fmaxf(mbase, nd)))) w.fill[atomicAdd(&sh->nnear, 1u)] = c;
            } else {
                vb[c] = -v;
                vall = fmaxf(vall, v);
                uint32_t k = atomicAdd(&sh->nout, 1u);
                if (k < kOutCap) sh->out[k] = (uint16_t)c;
                w.wl[k] = c;
            }
        }
        if (uni(sh->stalled)) return 3u;
        vmax = wg_max<WG>(vmax, s_red);  // (its barriers cover the lists above)
        const uint32_t n_over = uni(sh->nout), n_near = uni(sh->nnear);
        const uint16_t *const act = sh->act;
        int check = 0;
        if (n_near) check = near_check<WG>(w, act, crad, n_near, s_red);
        const bool missed_near = check != 0;
        if (check == 0 && n_over) {
            const double h = cell_size(rmax, uni(cs.s_cell));  // the grid of the list build
            const CCGrid g = cc_grid(Np, Nc, T, h, w.start);
            if (n_over > kOutCap && !rebuild) {
                check = 3;  // too many to tell with an old list
            } else if (n_over > kOutCap) {
                vall = fmaxf(wg_max<WG>(vall, s_red), vmax);
                check = overruns_check<WG>(w, act, crad, vb, w.wl, n_over, vall, u, rmax, h, g, s_red, true);
            } else {
                check = overruns_check<WG>(w, act, crad, vb, sh->out, n_over, vmax, u, rmax, h, g, s_red, false);
            }
        }
        if (check == 0) {
            if (tid == 0) {
                cs.since_build++;
                if (n_over) sh->cnt.kept++;
                if (widen == 0u) {
                    if (cs.heat) cs.heat--;
                    if (++cs.clean >= kLevelClean) {
                        cs.clean = 0u;
                        if (cs.level) cs.level--;
                    }
                }
            }
            return 0u;
        }
        if (check == 3 && tid == 0) sh->cnt.unchecked++;
        // undo; the next attempt has the margins (and skins) the circles showed
        // they need
        for (uint32_t c = tid; c < Nc; c += WG) P[Np + c] = w.save[c];
        const bool same_list = check == 1 && widen < 2u;
        if (tid == 0) {
            sh->cnt.redos++;
            if (!same_list) cs.list_valid = 0u;
            if (check == 1 && !missed_near && widen == 0u) cs.heat += kHeatMiss;
            if (missed_near || cs.heat >= kHeatRaise) {
                cs.clean = cs.heat = 0u;
                if (widen == 0u) cs.level = min(cs.level + 2u, kLevels);
            }
        }
        __syncthreads();
        if (same_list) attempt--;
        widen++;
    }
}

// Whether a sweep has nothing to do: no candidate pair, and no circle drifted so
// far that there could be one.  This is every sweep of bodies in flight, so it
// is asked before circle_sweep is called (a call saves and restores registers).
template <int WG>
__device__ __forceinline__ bool quiet_sweep(const float2 *P, uint32_t Np, uint32_t Nc, CCShared *sh, uint32_t *s_wl) {
    if (uni(sh->cs.list_valid) == 0u || uni(sh->cs.pairs) != 0u || uni(sh->fb_streak) != 0u) return false;
    const Drift dr = drift_box<WG, false>(P, Np, Nc, sh->work.ref, (float4 *)s_wl);
    if (!(drift_share(dr.box, uni(sh->cs.smin)) <= kDriftRebuild)) return false;
    if (threadIdx.x == 0) sh->cs.since_build++;
    return true;
}

// Polygon pairs of one scene (see run_scene), kept out of line: a rare phase
// whose registers need not weigh on the rest of the kernel.
template <int WG>
__device__ __noinline__ void poly_pairs(float2 *P, const uint4 *ptab, const float2 *ctr, uint32_t npoly,
                                        uint32_t *poly_last) {
    extern __shared__ float2 s_dyn[];
    if (((uint64_t)P >> 32) == ((uint64_t)s_dyn >> 32))
        poly_pair_loop<WG>(to_lds((uint64_t *)P), ptab, ctr, uni(npoly), poly_last);
    else
        poly_pair_loop<WG>((uint64_t *)P, ptab, ctr, uni(npoly), poly_last);
}

// ---------------------------------------------------------------------------
// The link and body phases, out of line: each keeps its own few registers
// (inlined, they shared the scene loop's, and its spills sat in their loops),
// and positions and records are addressed by where they are, LDS or global
// memory (through generic pointers, a record's flat load also held up the
// waits for LDS).
// ---------------------------------------------------------------------------

// What the two phases need to know about the bodies: all of them circles of one
// radius, all of them particles, or any mix.
constexpr uint32_t kBodiesCircles = 0u, kBodiesParticles = 1u, kBodiesMixed = 2u;

// `iters` link sweeps, layer by layer with a barrier after each layer.  A layer
// is a chain of LDS accesses and one link's arithmetic behind that barrier, so
// everything else is taken out of it: a thread's first record of the next layer
// (of the next sweep's first layer at the end of one) loads while it solves the
// current layer's, its further records one ahead, and the layer bounds sit in
// one register, a bound to a lane (past 63 layers they come through the scalar
// cache).  The 32 x 32 cloth (64 layers a substep, 512 lanes): 0.50 -> 0.34 us a
// layer, of which 0.20 are the issue of about 55 vector instructions by two
// wavefronts to a SIMD.
template <int WG, uint32_t KIND, bool HELD, bool LDS, typename PP, typename LP>
__device__ __forceinline__ void link_layers(PP P, LP lk, const uint32_t *loff, uint32_t depth, uint32_t nlinks,
                                            uint32_t iters, uint32_t Np, uint32_t NpNc, BD_GLOBAL const float *crad,
                                            float r2u, float scaleu, bool uni_r) {
    const uint32_t tid = threadIdx.x;
    BD_CONST const uint32_t *const kloff = to_const(loff);
    const uint32_t held = HELD ? to_global(loff)[min(tid & 63u, depth)] : 0u;
    auto bound = [&](uint32_t L) { return HELD ? (uint32_t)__builtin_amdgcn_readlane(held, L) : kloff[L]; };
    auto f32x2 = [](uint64_t b) { return make_float2(__uint_as_float((uint32_t)b), __uint_as_float((uint32_t)(b >> 32))); };
    auto bits = [](float2 v) { return (uint64_t)__float_as_uint(v.x) | ((uint64_t)__float_as_uint(v.y) << 32); };
    auto solve = [&](uint64_t rec) {
        const uint32_t ab = (uint32_t)rec;
        const float t = __uint_as_float((uint32_t)(rec >> 32));
        constexpr uint32_t kIdx = KIND == kBodiesCircles ? 0xffffu : 0x7fffu;  // circles have no pins
        const uint32_t a = ab & kIdx, b = (ab >> 16) & kIdx;
        float2 A = f32x2(P[a]), B = f32x2(P[b]);
        const float dx = A.x - B.x, dy = A.y - B.y;
        float dist, nx, ny;
        length_and_unit(dx, dy, dx * dx + dy * dy, dist, nx, ny);
        const float e = dist - t;
        nx = nx * e;
        ny = ny * e;
        if (KIND == kBodiesCircles) {
            const float cx = (nx * scaleu) * r2u, cy = (ny * scaleu) * r2u;
            A.x = A.x - cx; A.y = A.y - cy;
            B.x = B.x + cx; B.y = B.y + cy;
        } else if (KIND == kBodiesMixed && a >= Np && a < NpNc) {
            float ra2 = r2u, rb2 = r2u, scale = scaleu;
            if (!uni_r) {
                const float ra = crad[a - Np], rb = crad[b - Np];
                ra2 = ra * ra; rb2 = rb * rb;
                scale = 1.0f / (ra2 + rb2);
            }
            A.x = A.x - (nx * scale) * rb2; A.y = A.y - (ny * scale) * rb2;
            B.x = B.x + (nx * scale) * ra2; B.y = B.y + (ny * scale) * ra2;
        } else {
            float cx = nx * 0.5f, cy = ny * 0.5f;
            // a free end beside a pinned one takes the whole correction (a
            // wavefront without pinned ends passes this by)
            const bool pa = (ab & kScenePinBit) != 0u, pb = (ab & (kScenePinBit << 16)) != 0u;
            if (__builtin_expect(__ballot((ab & ((kScenePinBit << 16) | kScenePinBit)) != 0u) != 0ull, 0)) {
                const float2 a0 = A, b0 = B;
                if (pa || pb) { cx = nx; cy = ny; }
                A.x = A.x - cx; A.y = A.y - cy;
                B.x = B.x + cx; B.y = B.y + cy;
                if (pa) A = a0;
                if (pb) B = b0;
            } else {
                A.x = A.x - cx; A.y = A.y - cy;
                B.x = B.x + cx; B.y = B.y + cy;
            }
        }
        P[a] = bits(A);
        P[b] = bits(B);
    };
    // loads past a layer's end read the last record instead, unused
    auto load = [&](uint32_t l) { return lk[min(l, nlinks - 1u)]; };
    uint32_t b0 = 0u, b1 = bound(1);
    uint64_t first = load(tid);
    for (uint32_t it = 0; it < iters; it++) {
#pragma unroll 1
        for (uint32_t L = 0; L < depth; L++) {
            const uint64_t rec = first;
            uint32_t l = b0 + tid;
            const uint32_t lo = b0, hi = b1;
            const bool wrap = L + 1 == depth;
            b0 = wrap ? 0u : b1;
            b1 = bound(wrap ? 1u : L + 2u);
            first = load(b0 + tid);
            if (hi - lo <= (uint32_t)WG) {
                if (l < hi) solve(rec);
            } else {
                uint64_t cur = rec;
#pragma unroll 1
                for (uint32_t k = lo; k < hi; k += WG) {
                    const uint64_t nxt = load(l + WG);
                    if (l < hi) solve(cur);
                    cur = nxt;
                    l += WG;
                }
            }
            if (LDS) lds_barrier();
            else __syncthreads();
        }
    }
    // the caller goes on to global memory too
    if (LDS) __syncthreads();
}

template <int WG, int MODE>
__device__ __noinline__ void link_phase(const SceneDesc *dp, float2 *P_, const LinkS *s_links, uint32_t iters_,
                                        uint32_t kind_) {
    const SceneDesc &d = *(const SceneDesc *)to_const(dp);
    char *base = (char *)d.base;
    const uint32_t *loff = (const uint32_t *)(base + d.loff_off);
    BD_GLOBAL const float *const crad = to_global((const float *)(base + d.crad_off));
    const uint32_t iters = uni(iters_), kind = uni(kind_), depth = d.depth;
    if (depth == 0u) return;
    const bool uni_r = (d.flags & kFlagUniformR) != 0;
    const float r2u = d.runi * d.runi, scaleu = 1.0f / (r2u + r2u);
    auto run = [&](auto P, auto lk) {
        constexpr bool LDS = MODE >= 1;
        const uint32_t nl = d.L, Np = d.Np, NpNc = d.Np + d.Nc;
        if (depth >= 64u)
            link_layers<WG, kBodiesMixed, false, LDS>(P, lk, loff, depth, nl, iters, Np, NpNc, crad, r2u, scaleu, uni_r);
        else if (kind == kBodiesCircles)
            link_layers<WG, kBodiesCircles, true, LDS>(P, lk, loff, depth, nl, iters, Np, NpNc, crad, r2u, scaleu, uni_r);
        else if (kind == kBodiesParticles)
            link_layers<WG, kBodiesParticles, true, LDS>(P, lk, loff, depth, nl, iters, Np, NpNc, crad, r2u, scaleu, uni_r);
        else
            link_layers<WG, kBodiesMixed, true, LDS>(P, lk, loff, depth, nl, iters, Np, NpNc, crad, r2u, scaleu, uni_r);
    };
    BD_GLOBAL const uint64_t *const glinks = to_global((const uint64_t *)(base + d.links_off));
    if constexpr (MODE == 2) {
        // records staged behind the positions (nullptr: left in global memory)
        if (uni((uint32_t)(uint64_t)s_links) != 0u) run(to_lds((uint64_t *)P_), to_lds((const uint64_t *)s_links));
        else run(to_lds((uint64_t *)P_), glinks);
    } else if constexpr (MODE == 1) {
        run(to_lds((uint64_t *)P_), glinks);
    } else {
        run(to_global((uint64_t *)P_), glinks);
    }
}

// Bodies: static colliders -> bounds -> Verlet.  acc: the initial acc of circles
// and polygon points is pending (the first substep).
template <int WG, uint32_t KIND, typename PP, typename QP>
__device__ __forceinline__ void step_bodies(const SceneDesc &d, PP P, QP Q, bool acc) {
    const char *base = (const char *)d.base;
    BD_GLOBAL const float *const crad = to_global((const float *)(base + d.crad_off));
    BD_GLOBAL const uint32_t *const pinmask = to_global((const uint32_t *)(base + d.pin_off));
    BD_GLOBAL const uint32_t *const gstatic = to_global((const uint32_t *)(base + d.gst_off));
    BD_GLOBAL const uint64_t *const acc0 = to_global((const uint64_t *)(base + d.acc0_off));
    const uint32_t N = d.N, Np = d.Np, NpNc = d.Np + d.Nc, ncol = d.ncol;
    const bool uni_r = (d.flags & kFlagUniformR) != 0, pins = (d.flags & kFlagPins) != 0;
    const float runi = d.runi, delta = d.delta, gex = d.gex, gey = d.gey;
    const float lox = d.lox, loy = d.loy, hix = d.hix, hiy = d.hiy;
    auto f32x2 = [](uint64_t b) { return make_float2(__uint_as_float((uint32_t)b), __uint_as_float((uint32_t)(b >> 32))); };
    auto bits = [](float2 v) { return (uint64_t)__float_as_uint(v.x) | ((uint64_t)__float_as_uint(v.y) << 32); };
#pragma unroll 1
    for (uint32_t j = threadIdx.x; j < N; j += WG) {
        if (KIND != kBodiesCircles && pins && j < Np && ((pinmask[j >> 5] >> (j & 31)) & 1u)) continue;
        float2 p = f32x2(P[j]), q = f32x2(Q[j]);
        const bool circle = KIND == kBodiesCircles || (KIND == kBodiesMixed && j >= Np && j < NpNc);
        float r = 0.0f;
        if (KIND == kBodiesCircles) r = runi;
        else if (KIND == kBodiesMixed && circle) r = uni_r ? runi : crad[j - Np];
        static_colliders(p, r, ncol, base + d.hdr_off, base + d.geo_off, base + d.pl_off);
        float ax = gex, ay = gey;
        if (KIND == kBodiesCircles || circle) {
            circle_bounds_axis(p.x, q.x, lox, hix, r);
            circle_bounds_axis(p.y, q.y, loy, hiy, r);
        } else {
            bounds_axis(p.x, q.x, lox, hix);
            bounds_axis(p.y, q.y, loy, hiy);
        }
        bool integrate = true;
        if (KIND == kBodiesMixed && j >= NpNc)
            // a static polygon's points skip Polygon::update (src/polygon.rs:125-128)
            integrate = !((gstatic[(j - NpNc) >> 5] >> ((j - NpNc) & 31)) & 1u);
        if (acc && j >= Np) {
            const float2 a0 = f32x2(acc0[j - Np]);
            ax = a0.x + d.gx;
            ay = a0.y + d.gy;
        }
        if (integrate) verlet(p.x, p.y, q.x, q.y, ax, ay, delta);
        P[j] = bits(p);
        Q[j] = bits(q);
    }
}

template <int WG, int MODE>
__device__ __noinline__ void body_phase(const SceneDesc *dp, float2 *P_, float2 *Q_, uint32_t kind_, uint32_t acc_) {
    const SceneDesc &d = *(const SceneDesc *)to_const(dp);
    const uint32_t kind = uni(kind_);
    const bool acc = uni(acc_) != 0u;
    auto run = [&](auto P, auto Q) {
        if (kind == kBodiesCircles) step_bodies<WG, kBodiesCircles>(d, P, Q, acc);
        else if (kind == kBodiesParticles) step_bodies<WG, kBodiesParticles>(d, P, Q, acc);
        else step_bodies<WG, kBodiesMixed>(d, P, Q, acc);
    };
    if constexpr (MODE == 2) run(to_lds((uint64_t *)P_), to_lds((uint64_t *)Q_));
    else if constexpr (MODE == 1) run(to_lds((uint64_t *)P_), to_global((uint64_t *)Q_));
    else run(to_global((uint64_t *)P_), to_global((uint64_t *)Q_));
}

// One scene for `steps` updates.  MODE 2 keeps positions and previous
// positions in LDS (s_lds), MODE 1 positions only, MODE 0 works on the scene
// chunk in global memory.
template <int WG, int MODE, bool SEQ>
__device__ __forceinline__ void run_scene(const SceneDesc *__restrict__ dp, uint32_t steps, SceneState *st,
                                          float2 *s_lds, float *s_red, uint32_t *s_u32,
                                          CCShared *s_cc, uint32_t *s_wl, uint32_t lds_bytes) {
    // fields are read where used: the descriptor is uniform and read-only, so
    // they come through scalar loads instead of a private copy
    const SceneDesc &d = *dp;
    char *base = (char *)d.base;
    float2 *gpos = (float2 *)(base + d.pos_off);
    float2 *gprev = (float2 *)(base + d.prev_off);
    const float *crad = (const float *)(base + d.crad_off);
    const LinkS *links = (const LinkS *)(base + d.links_off);
    float2 *P, *Q;
    if constexpr (MODE >= 1) P = s_lds; else P = gpos;
    if constexpr (MODE == 2) Q = s_lds + d.N; else Q = gprev;
    const uint32_t N = d.N, Np = d.Np, Nc = d.Nc, npoly = d.P;
    const uint4 *ptab = (const uint4 *)(base + d.poly_off);
    float2 *ctr = (float2 *)(base + d.ctr_off);
    const int tid = threadIdx.x;
    const bool uni_r = (d.flags & kFlagUniformR) != 0;
    const float runi = d.runi;
    const uint32_t kind = N == Nc && uni_r ? kBodiesCircles : N == Np ? kBodiesParticles : kBodiesMixed;

    // load state into LDS; with positions and previous positions there, the
    // link records follow them when they fit too
    if constexpr (MODE >= 1) {
        for (uint32_t j = tid; j < N; j += WG) {
            P[j] = gpos[j];
            if constexpr (MODE == 2) Q[j] = gprev[j];
        }
    }
    const bool links_lds = MODE == 2 && 16ull * N + 8ull * d.L <= lds_bytes;
    LinkS *const s_links = (LinkS *)(s_lds + 2 * N);
    if (links_lds)
        for (uint32_t l = tid; l < d.L; l += WG) s_links[l] = links[l];
    if (tid == 0) {
        const uint32_t kept = MODE == 2 ? 16u * N + (links_lds ? 8u * d.L : 0u) : MODE == 1 ? 8u * N : 0u;
        s_cc->free_off = kept;
        s_cc->free_bytes = lds_bytes > kept ? lds_bytes - kept : 0u;
        CCShared::Fallback &f = s_cc->fb;
        if constexpr (MODE == 2) {
            f.lds = (uint8_t *)Q; f.lds_bytes = 8u * N; f.q_lds = Q; f.q_global = gprev; f.nq = N;
            f.p_global = nullptr;
        } else {
            const uint32_t used = MODE == 1 ? 8u * N : 0u;
            f.lds = (uint8_t *)(s_lds) + used; f.lds_bytes = lds_bytes > used ? lds_bytes - used : 0u;
            f.q_lds = nullptr; f.q_global = nullptr; f.nq = 0u;
            f.p_global = MODE == 1 ? gpos : nullptr;
        }
    }
    __syncthreads();

    // circle-pair workspace
    char *ws = d.ws_base ? (char *)d.ws_base : base + d.ws_off;
    const CCLayout cl = cc_layout(Nc, d.T);
    CCWork &w = s_cc->work;
    if (tid == 0) {
    w.ref = (float2 *)(ws + cl.ref); w.save = (float2 *)(ws + cl.save);
    w.path = (float *)(ws + cl.path); w.skin = (float *)(ws + cl.skin); w.need = (float *)(ws + cl.need);
    w.cnt = (uint32_t *)(ws + cl.cnt); w.off = (uint32_t *)(ws + cl.off); w.cand = (uint16_t *)(ws + cl.cand);
    w.traj = (float2 *)(ws + cl.traj);
    w.head = (uint32_t *)(ws + cl.head); w.stamp = (uint32_t *)(ws + cl.stamp); w.wl = (uint32_t *)(ws + cl.wl);
    w.key = (uint32_t *)(ws + cl.key); w.rec = (float4 *)(ws + cl.rec); w.start = (uint32_t *)(ws + cl.start);
    w.fill = (uint32_t *)(ws + cl.fill); w.items = (uint32_t *)(ws + cl.items);
    }
    __syncthreads();
    if (Nc >= 2 && !st->ws_ready) {
        for (uint32_t c = tid; c < Nc; c += WG) w.need[c] = 0.0f;
        __syncthreads();
    }

    uint32_t err = uni(st->err);
    if (tid == 0) {
        s_cc->cs = CCShared::Steer{st->skin, (uint32_t)st->list_valid & 1u, st->pairs, st->since_build, st->s_cell, st->smin,
                                   (uint32_t)st->list_valid >> 1 & 7u, (uint32_t)st->ws_ready >> 1,
                                   (uint32_t)st->list_valid >> 4};
        s_cc->fb_streak = 0u;
        CCShared::Counts &k = s_cc->cnt;
        k = CCShared::Counts{};
        k.n_out = st->n_out; k.n_far = st->n_far; k.max_list = st->max_list; k.smax = st->smax;
    }
    __syncthreads();
    bool acc = (d.flags & kFlagAcc) != 0;

    const uint64_t t_scene0 = wall_clock64();
    uint32_t ran = 0;
    // a scene stopped by its time budget inside an update resumes at the
    // substep after the last one it ran
    uint32_t sub0 = uni((uint32_t)st->sub_phase), resume = 0u;
    for (uint32_t step = 0; step < steps; step++) {
        for (uint32_t sub = sub0; sub < d.sub_steps; sub++) {
            // ---- links: dependency layers, k sweeps
            const uint64_t tl0 = wall_clock64();
            // polygon centres (Polygon::calc_center, src/polygon.rs:231-237) as
            // Polygon::solve_links computes them before the polygon's links in
            // the last sweep; no other link moves a polygon's points, so the
            // start of that sweep gives the same sums
            auto poly_centres = [&]() {
                for (uint32_t q = tid; q < npoly; q += WG) {
                    const uint4 r = ptab[q];
                    float sx = 0.0f, sy = 0.0f;
                    for (uint32_t i = 0; i < r.y; i++) {
                        const float2 v = P[r.x + i];
                        sx = sx + v.x; sy = sy + v.y;
                    }
                    const float n = (float)r.y;
                    ctr[q] = make_float2(sx / n, sy / n);
                }
                __syncthreads();
            };
            if (npoly) {
                if (d.link_iters > 1) link_phase<WG, MODE>(dp, P, links_lds ? s_links : nullptr, d.link_iters - 1, kind);
                poly_centres();
                link_phase<WG, MODE>(dp, P, links_lds ? s_links : nullptr, 1u, kind);
            } else if (d.depth) {
                link_phase<WG, MODE>(dp, P, links_lds ? s_links : nullptr, d.link_iters, kind);
            }
            if (tid == 0) s_cc->cnt.t_links += wall_clock64() - tl0;
            // ---- circle pairs
            if (Nc >= 2 && !err)
            {
                const uint64_t t0 = wall_clock64();
                if constexpr (SEQ)
                    fallback_sweep<WG>(P, Np, Nc, crad, uni_r, runi, d.rmax, d.T, w, s_cc);
                else if (!quiet_sweep<WG>(P, Np, Nc, s_cc, s_wl))
                    err = uni(circle_sweep<WG>(P, Np, Nc, crad, uni_r, runi, d.rmax, d.T, s_cc, s_red, s_u32, s_wl));
                if (tid == 0) s_cc->cnt.t_sweep += wall_clock64() - t0;
            }
            // ---- polygon pairs (src/solver.rs:178-187): Polygon::solve_polygon
            // (src/polygon.rs:142-162) pair by pair, edge by edge.  For one edge
            // the other polygon's points are independent (each reads the edge's
            // ends as they were when its turn came, its own position and the two
            // centres), so they run across the workgroup; the last point that
            // hits (highest index) decides where the edge's ends go.
            if (npoly >= 2) poly_pairs<WG>(P, ptab, ctr, npoly, s_cc->poly_last);
            // ---- bodies: colliders -> bounds -> Verlet
            const uint64_t tq0 = wall_clock64();
            body_phase<WG, MODE>(dp, P, Q, kind, acc ? 1u : 0u);
            acc = false;
            __syncthreads();
            if (tid == 0) s_cc->cnt.t_bodies += wall_clock64() - tq0;
            if (d.budget && sub + 1 < d.sub_steps) {
                // stop after a substep once the budget is spent: the state
                // between substeps is whole, and the next launch resumes
                // there (one clock read, shared, so the workgroup leaves
                // together)
                if (tid == 0) s_cc->halt = (wall_clock64() - t_scene0 > (uint64_t)d.budget) ? 1u : 0u;
                __syncthreads();
                if (uni(s_cc->halt)) { resume = sub + 1; break; }
            }
        }
        if (resume) break;
        sub0 = 0u;
        ran = step + 1;
        if (d.budget && ran < steps) {
            // stop after a whole update once the budget is spent
            if (tid == 0) s_cc->halt = (wall_clock64() - t_scene0 > (uint64_t)d.budget) ? 1u : 0u;
            __syncthreads();
            if (uni(s_cc->halt)) break;
        }
    }
    // write back
    if constexpr (MODE >= 1) {
        for (uint32_t j = tid; j < N; j += WG) {
            gpos[j] = P[j];
            if constexpr (MODE == 2) gprev[j] = Q[j];
        }
    }
    // statistics (uniform across the workgroup)
    __syncthreads();
    if (tid == 0) {
        const CCShared::Steer &cs = s_cc->cs;
        st->skin = cs.skin;
        st->list_valid = (uint8_t)((cs.list_valid ? 1u : 0u) | cs.level << 1 | cs.heat << 4);
        st->err = err;
        const CCShared::Counts &k = s_cc->cnt;
        st->rounds += k.rounds;
        st->redos += k.redos;
        st->rebuilds += k.rebuilds;
        st->pairs = cs.pairs;
        if (Nc >= 2) st->ws_ready = (uint8_t)(1u | (cs.clean << 1));
        st->t_links += k.t_links;
        st->t_build += k.t_build;
        st->t_sweep += k.t_sweep - k.t_build;
        st->t_bodies += k.t_bodies;
        st->since_build = cs.since_build;
        st->n_out = k.n_out;
        st->n_far = k.n_far;
        st->max_list = k.max_list;
        st->s_cell = cs.s_cell;
        st->smax = k.smax;
        st->smin = cs.smin;
        st->t_count += k.t_count;
        st->t_lists += k.t_lists;
        st->t_sort += k.t_sort;
        st->kept += k.kept;
        st->unchecked += k.unchecked;
        st->fallbacks += k.fallbacks;
        st->last_steps = ran;
        st->sub_phase = (uint16_t)resume;
    }
    __syncthreads();
}

template <int WG>
__global__ void __launch_bounds__(WG, WG == 1024 ? 4 : 3) k_scenes(const SceneDesc *__restrict__ descs, SceneState *states,
                                               const uint32_t *__restrict__ order, uint32_t n,
                                               uint32_t *queue, uint32_t lds_bytes, uint32_t launch_steps) {
    extern __shared__ float2 s_lds[];
    __shared__ float s_red[WG / 64];
    __shared__ uint32_t s_u32[WG / 64];
    __shared__ CCShared s_cc;
    __shared__ __align__(16) uint32_t s_wl[2 * WG];  // also float4 scratch of the list builds
    __shared__ uint32_t s_next;
    for (uint32_t turn = blockIdx.x;; turn += gridDim.x) {
        if (threadIdx.x == 0) s_next = queue ? atomicAdd(queue, 1u) : turn;
        __syncthreads();
        const uint32_t k = uni(s_next);
        __syncthreads();
        if (k >= n) break;
        const uint32_t si = uni(order[k]);
        const SceneDesc *__restrict__ d = descs + si;
        const uint32_t steps = d->steps < launch_steps ? d->steps : launch_steps;
        if (steps == 0 || d->N == 0) continue;
        if (d->flags & kFlagSequential)  // diagnostic: every sweep sequential, state in global memory
            run_scene<WG, 0, true>(d, steps, states + d->state_slot, s_lds, s_red, s_u32, &s_cc, s_wl,
                                   lds_bytes);
        else if (16ull * d->N <= lds_bytes)
            run_scene<WG, 2, false>(d, steps, states + d->state_slot, s_lds, s_red, s_u32, &s_cc, s_wl,
                                    lds_bytes);
        else if (8ull * d->N <= lds_bytes)
            run_scene<WG, 1, false>(d, steps, states + d->state_slot, s_lds, s_red, s_u32, &s_cc, s_wl,
                                    lds_bytes);
        else
            run_scene<WG, 0, false>(d, steps, states + d->state_slot, s_lds, s_red, s_u32, &s_cc, s_wl,
                                    lds_bytes);
    }
}

// ---------------------------------------------------------------------------
// Host side
// ---------------------------------------------------------------------------

template <int WG>
static void launch_variant(dim3 grid, size_t lds, hipStream_t s, const SceneDesc *d, SceneState *st,
                           const uint32_t *order, uint32_t n, uint32_t *queue, uint32_t steps) {
    hipLaunchKernelGGL((k_scenes<WG>), grid, dim3(WG), lds, s, d, st, order, n, queue, (uint32_t)lds, steps);
}

using LaunchFn = void (*)(dim3, size_t, hipStream_t, const SceneDesc *, SceneState *, const uint32_t *, uint32_t,
                          uint32_t *, uint32_t);

static const struct {
    int wg;
    LaunchFn fn;
    const void *kern;
} kVariants[] = {
    {64, launch_variant<64>, (const void *)k_scenes<64>},
    {128, launch_variant<128>, (const void *)k_scenes<128>},
    {256, launch_variant<256>, (const void *)k_scenes<256>},
    {512, launch_variant<512>, (const void *)k_scenes<512>},
    {1024, launch_variant<1024>, (const void *)k_scenes<1024>},
};
constexpr int kNumVariants = sizeof(kVariants) / sizeof(kVariants[0]);
constexpr size_t kMaxDynLds = 144 * 1024;

int scene_variant_count() { return kNumVariants; }
int scene_variant_wg(int v) { return kVariants[v].wg; }
size_t scene_max_lds() { return kMaxDynLds; }

int launch_scene_variant(int v, uint32_t blocks, size_t lds_bytes, hipStream_t stream, const SceneDesc *d,
                         SceneState *st, const uint32_t *order, uint32_t n, uint32_t *queue, uint32_t steps,
                         std::string &err) {
    if (lds_bytes > kMaxDynLds) lds_bytes = kMaxDynLds;
    kVariants[v].fn(dim3(blocks), lds_bytes, stream, d, st, order, n, queue, steps);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
        err = std::string("scene kernel launch: ") + hipGetErrorString(e);
        return BD_ERR_DEVICE;
    }
    return BD_OK;
}

// Allow every variant the full dynamic LDS budget (once per process, before
// any launch or graph capture).
int scene_kernels_init(std::string &err) {
    static std::once_flag once;
    static hipError_t result = hipSuccess;
    std::call_once(once, []() {
        for (int v = 0; v < kNumVariants; v++) {
            hipError_t e = hipFuncSetAttribute(kVariants[v].kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kMaxDynLds);
            if (e != hipSuccess) result = e;
        }
    });
    if (result != hipSuccess) {
        err = std::string("hipFuncSetAttribute: ") + hipGetErrorString(result);
        return BD_ERR_DEVICE;
    }
    return BD_OK;
}

int scene_blocks_per_cu(int v, size_t lds_bytes) {
    int nb = 0;
    if (lds_bytes > kMaxDynLds) lds_bytes = kMaxDynLds;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, kVariants[v].kern, kVariants[v].wg, lds_bytes) != hipSuccess)
        return 1;
    return nb > 0 ? nb : 1;
}

// Launch shape of a single scene on an otherwise idle device: about two bodies
// per lane; positions, previous positions and, when they fit, the link records
// in LDS, with room behind them for the circle-pair rounds' state (8 bytes a
// circle) and active lists (2 bytes an entry).  In a batch, where LDS decides how
// many scenes run at once, that is room for four entries a circle; a scene with
// the device to itself takes room for kAloneEntries: lists that do not fit are written
// a second time, into memory, and the rounds read them there (a gas of 2,000 circles
// that falls into a heap 702 us an update with room for four, 645 with sixteen; one
// of 1,000 with mixed radii 634 and 585).
void scene_launch_shape(const SceneDesc &d, uint32_t &wg, uint32_t &lds, uint32_t entries) {
    wg = 64;
    while (wg < 1024 && wg * 2 < d.N) wg <<= 1;
    const uint64_t bodies = 16ull * d.N, links = 8ull * d.L;
    const uint64_t rounds = d.Nc >= 2 ? (8ull + 2ull * entries) * d.Nc : 0ull;
    const uint64_t want = bodies + links <= kMaxDynLds ? bodies + links + rounds : bodies + rounds;
    lds = (uint32_t)std::min<uint64_t>(want, kMaxDynLds);
}

int variant_for_wg(int wg) {
    for (int v = 0; v < kNumVariants; v++)
        if (kVariants[v].wg == wg) return v;
    return -1;
}

// ---- scene images ----------------------------------------------------------

int build_scene_image(const HostScene &s, const Plan &p, SceneImage &img, std::string &err) {
    if (p.N > kSceneMaxPoints) { err = "scene too large for the SCENE engine"; return BD_ERR_CAPACITY; }
    SceneDesc &d = img.desc;
    std::memset(&d, 0, sizeof(d));
    d.N = p.N; d.Np = p.Np; d.Nc = p.Nc; d.Ng = p.Ng; d.depth = p.depth;
    d.P = (uint32_t)s.polys.size();
    d.L = (uint32_t)p.links.size();
    d.ncol = (uint32_t)s.cols.size();
    d.nplanes = (uint32_t)(s.planes.size() / 3);
    d.T = 0;
    if (d.Nc >= 2) { d.T = 1; while (d.T < 2 * d.Nc) d.T <<= 1; }
    uint64_t o = 0;
    d.pos_off = (uint32_t)o; o = align16(o + 8ull * d.N);
    d.prev_off = (uint32_t)o; o = align16(o + 8ull * d.N);
    d.crad_off = (uint32_t)o; o = align16(o + 4ull * d.Nc);
    d.acc0_off = (uint32_t)o; o = align16(o + 8ull * (d.Nc + d.Ng));
    d.pin_off = (uint32_t)o; o = align16(o + 4ull * ((d.Np + 31) / 32));
    d.loff_off = (uint32_t)o; o = align16(o + 4ull * (d.depth + 1));
    d.links_off = (uint32_t)o; o = align16(o + 8ull * d.L);
    d.hdr_off = (uint32_t)o; o = align16(o + 16ull * d.ncol);
    d.geo_off = (uint32_t)o; o = align16(o + 16ull * d.ncol);
    d.pl_off = (uint32_t)o; o = align16(o + 16ull * d.nplanes);
    d.poly_off = (uint32_t)o; o = align16(o + 16ull * d.P);
    d.ctr_off = (uint32_t)o; o = align16(o + 8ull * d.P);
    d.gst_off = (uint32_t)o; o = align16(o + 4ull * ((d.Ng + 31) / 32));
    img.init_bytes = o;  // everything above is initialised from the host
    d.ws_off = (uint32_t)o;
    d.ws_bytes = d.Nc >= 2 ? cc_layout(d.Nc, d.T).bytes : 0u;
    o = align16(o + d.ws_bytes);
    img.total_bytes = o;
    img.bytes.assign(img.init_bytes, 0);
    uint8_t *b = img.bytes.data();
    auto put = [&](uint32_t off, const void *src, size_t n) { if (n) std::memcpy(b + off, src, n); };
    std::vector<V2> pos(d.N), prev(d.N);
    for (uint32_t i = 0; i < d.Np; i++) { pos[i] = s.p_pos[i]; prev[i] = s.p_prev[i]; }
    for (uint32_t i = 0; i < d.Nc; i++) { pos[d.Np + i] = s.c_pos[i]; prev[d.Np + i] = s.c_prev[i]; }
    for (uint32_t i = 0; i < d.Ng; i++) { pos[d.Np + d.Nc + i] = s.g_pos[i]; prev[d.Np + d.Nc + i] = s.g_prev[i]; }
    put(d.pos_off, pos.data(), 8ull * d.N);
    put(d.prev_off, prev.data(), 8ull * d.N);
    put(d.crad_off, s.c_r.data(), 4ull * d.Nc);
    put(d.acc0_off, s.c_acc.data(), 8ull * d.Nc);
    put(d.acc0_off + 8ull * d.Nc, s.g_acc.data(), 8ull * d.Ng);
    {
        std::vector<uint4> tab(d.P);
        std::vector<float2> ctr(d.P);
        std::vector<uint32_t> mask((d.Ng + 31) / 32, 0u);
        for (uint32_t i = 0; i < d.P; i++) {
            const Poly &pg = s.polys[i];
            tab[i] = make_uint4(d.Np + d.Nc + pg.off, pg.n, pg.is_static ? 1u : 0u, 0u);
            ctr[i] = make_float2(pg.center.x, pg.center.y);
            if (pg.is_static)
                for (uint32_t k = pg.off; k < pg.off + pg.n; k++) mask[k >> 5] |= 1u << (k & 31);
        }
        put(d.poly_off, tab.data(), 16ull * d.P);
        put(d.ctr_off, ctr.data(), 8ull * d.P);
        put(d.gst_off, mask.data(), 4ull * mask.size());
    }
    bool pins = false;
    {
        std::vector<uint32_t> mask((d.Np + 31) / 32, 0u);
        for (uint32_t i = 0; i < d.Np; i++)
            if (s.p_pin[i]) { mask[i >> 5] |= 1u << (i & 31); pins = true; }
        put(d.pin_off, mask.data(), 4ull * mask.size());
    }
    put(d.loff_off, p.layer_off.data(), 4ull * (d.depth + 1));
    {
        std::vector<LinkS> ls(d.L);
        for (uint32_t i = 0; i < d.L; i++) {
            const Link12 &l = p.links[i];
            uint32_t a = l.a & kIndexMask, bb = l.b & kIndexMask;
            ls[i].a = (uint16_t)(a | ((l.a & kPinBit) ? kScenePinBit : 0u));
            ls[i].b = (uint16_t)(bb | ((l.b & kPinBit) ? kScenePinBit : 0u));
            ls[i].t = l.t;
        }
        put(d.links_off, ls.data(), 8ull * d.L);
    }
    {
        std::vector<int4> hdr(d.ncol);
        std::vector<float4> geo(d.ncol), pl(d.nplanes);
        for (uint32_t k = 0; k < d.ncol; k++) {
            const Collider &c = s.cols[k];
            hdr[k] = make_int4(c.kind, (int)c.plane_off, (int)c.nv, 0);
            geo[k] = make_float4(c.cx, c.cy, c.r, 0.0f);
        }
        for (uint32_t k = 0; k < d.nplanes; k++)
            pl[k] = make_float4(s.planes[3 * k], s.planes[3 * k + 1], s.planes[3 * k + 2], 0.0f);
        put(d.hdr_off, hdr.data(), 16ull * d.ncol);
        put(d.geo_off, geo.data(), 16ull * d.ncol);
        put(d.pl_off, pl.data(), 16ull * d.nplanes);
    }
    d.flags = pins ? kFlagPins : 0u;
    // diagnostic switch: every circle-pair sweep by the sequential fallback
    // (its results are the same; tests use it to run that path on any scene)
    if (const char *e = std::getenv("BD_SCENE_SEQUENTIAL_SWEEP"))
        if (e[0] == '1') d.flags |= kFlagSequential;
    img.acc_pending = s.any_initial_acc();
    d.rmax = 0.0f;
    for (float r : s.c_r) d.rmax = std::max(d.rmax, r);
    // one radius for every circle (same bits): the kernel reads it from the
    // descriptor instead of crad[]
    d.runi = 0.0f;
    if (!s.c_r.empty() &&
        std::all_of(s.c_r.begin(), s.c_r.end(), [&](float r) { return std::memcmp(&r, &s.c_r[0], 4) == 0; })) {
        d.flags |= kFlagUniformR;
        d.runi = s.c_r[0];
    }
    img.skin0 = std::max(0.25f * d.rmax, 0.025f);  // per circle: a pair's margin is the sum of both
    return BD_OK;
}

int import_scene_chunk(bd_solver *out, const SceneDesc &d, const uint8_t *chunk, uint64_t updates, std::string &err) {
    if (!d.P && !d.Ng)
        return solver_import_bodies(out, d.Np, d.Nc, chunk + d.pos_off, chunk + d.prev_off, updates, err);
    HostScene h;
    scene_chunk_to_host(d, chunk, h);
    return solver_import_state(out, h, updates, err);
}

void scene_chunk_to_host(const SceneDesc &d, const uint8_t *chunk, HostScene &h) {
    const float2 *pos = (const float2 *)(chunk + d.pos_off);
    const float2 *prev = (const float2 *)(chunk + d.prev_off);
    const float2 *ctr = (const float2 *)(chunk + d.ctr_off);
    const uint32_t NpNc = d.Np + d.Nc;
    h.p_pos.resize(d.Np); h.p_prev.resize(d.Np);
    h.c_pos.resize(d.Nc); h.c_prev.resize(d.Nc);
    h.g_pos.resize(d.Ng); h.g_prev.resize(d.Ng);
    for (uint32_t i = 0; i < d.N; i++) {
        V2 p{pos[i].x, pos[i].y}, q{prev[i].x, prev[i].y};
        if (i < d.Np) { h.p_pos[i] = p; h.p_prev[i] = q; }
        else if (i < NpNc) { h.c_pos[i - d.Np] = p; h.c_prev[i - d.Np] = q; }
        else { h.g_pos[i - NpNc] = p; h.g_prev[i - NpNc] = q; }
    }
    // the acc the bodies held when the chunk was built (the kernel reads it
    // on the first substep and never writes it)
    const float2 *acc0 = (const float2 *)(chunk + d.acc0_off);
    h.c_acc.resize(d.Nc);
    h.g_acc.resize(d.Ng);
    for (uint32_t i = 0; i < d.Nc; i++) h.c_acc[i] = V2{acc0[i].x, acc0[i].y};
    for (uint32_t i = 0; i < d.Ng; i++) h.g_acc[i] = V2{acc0[d.Nc + i].x, acc0[d.Nc + i].y};
    h.polys.assign(d.P, Poly{});
    for (uint32_t i = 0; i < d.P; i++) h.polys[i].center = V2{ctr[i].x, ctr[i].y};
    h.gravity = V2{d.gx, d.gy};
    h.sub_steps = d.sub_steps;
}

void set_scene_params(SceneDesc &d, const StepParams &sp, uint32_t steps, bool acc_pending) {
    d.steps = steps;
    d.sub_steps = sp.sub_steps;
    d.link_iters = sp.link_iters;
    d.delta = sp.delta;
    d.gex = sp.gex; d.gey = sp.gey; d.gx = sp.gx; d.gy = sp.gy;
    d.lox = sp.lox; d.loy = sp.loy; d.hix = sp.hix; d.hiy = sp.hiy;
    d.flags = (d.flags & ~kFlagAcc) | (acc_pending ? kFlagAcc : 0u);
}

// ---- single-scene engine ---------------------------------------------------

class SceneEngine : public Engine {
public:
    explicit SceneEngine(hipStream_t s) : stream_(s) {}
    ~SceneEngine() override {
        if (chunk_) (void)hipFree(chunk_);
        if (dev_) (void)hipFree(dev_);
    }
    int kind() const override { return BD_ENGINE_SCENE; }

    int upload(const HostScene &s, const Plan &p, std::string &err) override {
        SceneImage img;
        int rc = build_scene_image(s, p, img, err);
        if (rc) return rc;
        rc = scene_kernels_init(err);
        if (rc) return rc;
        if (chunk_) { (void)hipFree(chunk_); chunk_ = nullptr; }
        BD_HIP(hipMalloc((void **)&chunk_, std::max<uint64_t>(img.total_bytes, 16)));
        BD_HIP(hipMemcpyAsync(chunk_, img.bytes.data(), img.init_bytes, hipMemcpyHostToDevice, stream_));
        desc_ = img.desc;
        desc_.base = (uint64_t)(uintptr_t)chunk_;
        acc_pending_ = img.acc_pending;
        sent_ = false;
        if (!dev_) BD_HIP(hipMalloc((void **)&dev_, 512));
        SceneState st{};
        st.skin = img.skin0;
        BD_HIP(hipMemcpyAsync(state_ptr(), &st, sizeof(st), hipMemcpyHostToDevice, stream_));
        uint32_t wg;
        scene_launch_shape(desc_, wg, lds_bytes_, kAloneEntries);
        variant_ = variant_for_wg((int)wg);
        BD_HIP(hipStreamSynchronize(stream_));
        N_ = p.N; Np_ = p.Np; Nc_ = p.Nc; P_ = desc_.P;
        return BD_OK;
    }

    int update(const StepParams &sp, Stats &st, std::string &err) override {
        set_scene_params(desc_, sp, 1, acc_pending_ && sp.first_acc);
        acc_pending_ = false;
        // the descriptor goes to the device when the update's parameters changed
        // (each copy held up a frame by about 8 us)
        if (!sent_ || std::memcmp(host_blob_, &desc_, sizeof(desc_)) != 0) {
            sent_ = false;
            std::memset(host_blob_, 0, sizeof(host_blob_));
            std::memcpy(host_blob_, &desc_, sizeof(desc_));
            BD_HIP(hipMemcpyAsync(dev_, host_blob_, sizeof(host_blob_), hipMemcpyHostToDevice, stream_));
            sent_ = true;
        }
        int rc = launch_scene_variant(variant_, 1, lds_bytes_, stream_, (const SceneDesc *)dev_, state_ptr(),
                                      (const uint32_t *)(dev_ + 256), 1, nullptr, 1u, err);
        if (rc) return rc;
        st.launches++;
        st.substeps += sp.sub_steps;
        return BD_OK;
    }

    // pos[N], prev[N], the scene's SceneState, then the polygon centres
    static constexpr size_t kStateWords = (sizeof(SceneState) + sizeof(float2) - 1) / sizeof(float2);
    size_t state_count() const override { return 2ull * N_ + kStateWords + P_; }
    hipStream_t stream() const override { return stream_; }

    StateParts state_parts() override {
        StateParts s;
        s.add(chunk_ + desc_.pos_off, N_);
        s.add(chunk_ + desc_.prev_off, N_);
        s.add(state_ptr(), kStateWords);
        s.add(chunk_ + desc_.ctr_off, P_);
        return s;
    }

    int unpack(const float2 *src, HostScene &s, std::string &err) override {
        if (!host_shape_matches(s, Np_, Nc_, N_ - Np_ - Nc_, err) || s.polys.size() != P_) return BD_ERR_STATE;
        const float2 *pos = src, *prev = src + N_, *ctr = src + 2 * N_ + kStateWords;
        SceneState stt;
        std::memcpy(&stt, src + 2 * N_, sizeof(stt));
        const uint32_t NpNc = Np_ + Nc_;
        for (uint32_t i = 0; i < N_; i++) {
            V2 p{pos[i].x, pos[i].y}, q{prev[i].x, prev[i].y};
            if (i < Np_) { s.p_pos[i] = p; s.p_prev[i] = q; }
            else if (i < NpNc) { s.c_pos[i - Np_] = p; s.c_prev[i - Np_] = q; }
            else { s.g_pos[i - NpNc] = p; s.g_prev[i - NpNc] = q; }
        }
        // a static polygon keeps the centre of its last Polygon::solve_links
        // (the others' centres follow from prev on the host)
        for (uint32_t i = 0; i < P_; i++)
            if (s.polys[i].is_static) s.polys[i].center = V2{ctr[i].x, ctr[i].y};
        if (stt.err) {
            err = "circle pair schedule did not converge (kind " + std::to_string(stt.err) + ", skin " +
                  std::to_string(stt.skin) + ", rounds " + std::to_string(stt.rounds) + ", redos " +
                  std::to_string(stt.redos) + ", rebuilds " + std::to_string(stt.rebuilds) + ")";
            return BD_ERR_COLLISION;
        }
        return BD_OK;
    }

    int sync(std::string &err) override {
        BD_HIP(hipStreamSynchronize(stream_));
        return BD_OK;
    }

private:
    SceneState *state_ptr() { return (SceneState *)(dev_ + 384); }
    hipStream_t stream_;
    uint8_t *chunk_ = nullptr;
    uint8_t *dev_ = nullptr;  // [0,256) desc, [256,260) order, [384,512) state
    uint8_t host_blob_[260] = {};  // what dev_ begins with, when sent_
    bool sent_ = false;
    SceneDesc desc_{};
    bool acc_pending_ = false;
    int variant_ = 0;
    uint32_t lds_bytes_ = 0;
    uint32_t N_ = 0, Np_ = 0, Nc_ = 0, P_ = 0;
};

bool scene_engine_fits(const HostScene &s, const Plan &p) {
    (void)s;
    return p.N <= 16384 && p.N > 0;
}

Engine *make_scene_engine(hipStream_t s) { return new SceneEngine(s); }

}  // namespace bd
