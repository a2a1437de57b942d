// engine_global.hip -- GLOBAL engine: the whole device works on one scene.
//
// Per substep (src/solver.rs:110-114):
//   links      one launch per dependency layer (k_link_layer), k sweeps; the
//              layers reproduce the sequential Gauss-Seidel order exactly
//              (src/solver.rs:143-153)
//   circles    candidate pairs from a hierarchical hashed cell broadphase
//              (per-circle margins, counting sort that numbers the circles), the
//              connected components of the candidate graph (union-find), and an
//              exact replay of the reference's (i, j) lexicographic sweep
//              (src/solver.rs:168-177) per component: by lanes of a wavefront,
//              a circle to each, or by a workgroup in LDS or in global memory;
//              a sweep whose circles left their margins is checked pair by pair
//              at each skipped pair's turn and redone only if one met
//   polygons   one workgroup replays the polygon-pair loop (src/solver.rs:178-187)
//   per body   EXT4 static colliders (records through the scalar cache), bounds,
//              Verlet, fused in one streaming kernel (src/solver.rs:155-165, 118-128)
#include <hip/hip_runtime.h>

#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstring>
#include <type_traits>
#include <vector>

#include "../../include/bendy2d.h"
#include "common.h"
#include "engine.h"
#include "bodies.h"
#include "kernels.h"

namespace bd {

// ---------------------------------------------------------------------------
// Kernels
// ---------------------------------------------------------------------------

// One dependency layer of links: no two links of the layer share a point.
// Algorithmic traffic: 12 B record + 2 x 8 B reads + 2 x 8 B writes per link.
__global__ void __launch_bounds__(256) k_link_layer(float2 *__restrict__ pos, const Link12 *__restrict__ links,
                                                    uint32_t n, const float *__restrict__ crad, uint32_t cbase) {
    uint32_t i = blockIdx.x * 256u + threadIdx.x;
    if (i >= n) return;
    Link12 l = links[i];
    uint32_t a = l.a & kIndexMask, b = l.b & kIndexMask;
    float2 A = pos[a], B = pos[b];
    if (l.a & kCircleLinkBit) {
        solve_circle_link(A.x, A.y, B.x, B.y, l.t, crad[a - cbase], crad[b - cbase]);
    } else {
        solve_particle_link(A.x, A.y, B.x, B.y, l.t, (l.a & kPinBit) != 0, (l.b & kPinBit) != 0);
    }
    pos[a] = A;
    pos[b] = B;
}

// Polygon centres (Polygon::calc_center, src/polygon.rs:231-237): sequential
// f32 sum in point order, one thread per polygon.
__global__ void k_poly_centers(const float2 *__restrict__ pos, const uint2 *__restrict__ ptab, uint32_t P,
                               float2 *__restrict__ centers) {
    uint32_t p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= P) return;
    uint2 t = ptab[p];
    float sx = 0.0f, sy = 0.0f;
    for (uint32_t i = 0; i < t.y; i++) {
        float2 v = pos[t.x + i];
        sx = sx + v.x; sy = sy + v.y;
    }
    float n = (float)t.y;
    centers[p] = make_float2(sx / n, sy / n);
}

// Polygon pair loop in one workgroup.
__global__ void __launch_bounds__(256) k_poly_pairs(float2 *pos, const uint2 *__restrict__ ptab, uint32_t P,
                                                    const float2 *__restrict__ centers) {
    __shared__ uint32_t s_slot[3];
    poly_pair_loop<256>((uint64_t *)pos, ptab, centers, P, s_slot);
}

constexpr int kLevels = 12;  // of the circle-pair grid
// component queues: for 4, 16 and 64 lanes, a workgroup in LDS, one in memory
constexpr uint32_t kQueues = 5, kQueueLds = 3, kQueueBig = 4;
// Control words of a sweep (zeroed with the bucket counters, which follow them;
// the two at kCtlTotal are one 64-bit counter).
enum : uint32_t {
    kCtlTotal = 0, kCtlMask = 2, kCtlOver, kCtlBad, kCtlRounds, kCtlInf, kCtlMissed, kCtlQuiet, kCtlMembers, kCtlFull,
    kCtlQueue = 12, kCtlEmax = kCtlQueue + kQueues, kCtlWords = 32
};
static_assert(kCtlEmax + kLevels <= (int)kCtlWords, "control words");

// The sweep whose control words these are was carried out and missed no pair.
__device__ __forceinline__ bool sweep_stands(const uint32_t *ctl) {
    return !(ctl[kCtlFull] | ctl[kCtlBad] | ctl[kCtlInf] | ctl[kCtlMissed]);
}

// The control words to the host: 32 words over PCIe and then their number, which
// the host waits for.
__global__ void __launch_bounds__(64) k_cg_verdict(const uint32_t *__restrict__ ctl, uint32_t *host, uint32_t number) {
    if (threadIdx.x < kCtlWords) host[threadIdx.x] = ctl[threadIdx.x];
    __threadfence_system();
    __syncthreads();
    if (threadIdx.x == 0u) __hip_atomic_store(host + kCtlWords, number, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

// Fused per-body phase: EXT4 static colliders -> bounds -> Verlet.  With a verdict
// nothing happens unless that sweep stands.
__global__ void __launch_bounds__(256) k_bodies(float2 *__restrict__ pos, float2 *__restrict__ prev,
                                                const uint32_t *__restrict__ pinmask,
                                                const float *__restrict__ crad,
                                                const float2 *__restrict__ acc0,
                                                const uint8_t *__restrict__ gflags,
                                                const int4 *__restrict__ colhdr,
                                                const float4 *__restrict__ colgeo,
                                                const float4 *__restrict__ planes, BodyParams P,
                                                const uint32_t *__restrict__ verdict) {
    if (verdict && !sweep_stands(verdict)) return;  // uniform
    for (uint32_t u = blockIdx.x * blockDim.x + threadIdx.x; u < P.N; u += gridDim.x * blockDim.x) {
        float r = 0.0f;
        float ax = P.gex, ay = P.gey;
        bool circle = false, integrate = true;
        if (u < P.Np) {
            if (pinmask && ((pinmask[u >> 5] >> (u & 31)) & 1u)) continue;  // EXT3: pinned never moves
        } else if (u < P.Np + P.Nc) {
            circle = true;
            r = crad[u - P.Np];
            if (P.first_acc) { float2 a = acc0[u - P.Np]; ax = a.x + P.gx; ay = a.y + P.gy; }
        } else {
            integrate = (gflags[u - P.Np - P.Nc] & 1u) == 0;  // Polygon::update returns if static
            if (P.first_acc && integrate) { float2 a = acc0[u - P.Np]; ax = a.x + P.gx; ay = a.y + P.gy; }
        }
        float2 p = pos[u], q = prev[u];
        static_colliders(p, r, P.ncol, colhdr, colgeo, planes);
        if (circle) {
            circle_bounds_axis(p.x, q.x, P.lox, P.hix, r);
            circle_bounds_axis(p.y, q.y, P.loy, P.hiy, r);
        } else {
            bounds_axis(p.x, q.x, P.lox, P.hix);
            bounds_axis(p.y, q.y, P.loy, P.hiy);
        }
        if (integrate) verlet(p.x, p.y, q.x, q.y, ax, ay, P.dt);
        pos[u] = p;
        prev[u] = q;
    }
}

__global__ void k_zero_acc0(float2 *acc0, uint32_t n) {
    uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) acc0[i] = make_float2(0.0f, 0.0f);
}

// ---------------------------------------------------------------------------
// Circle-pair schedule kernels
// ---------------------------------------------------------------------------
//
// Every sweep builds candidate lists from the circles' positions at its
// start (save).  Circle i gets a margin m_i = max(s0, need_i), where need_i
// follows how far the circle's pushes took it from save in recent sweeps; its
// reach is r_i + m_i, and (i, j) is a candidate pair when
// |save_i - save_j| < reach_i + reach_j.  A pair left out can only meet during
// the sweep if e_i + e_j > m_i + m_j, e being each circle's largest distance
// from save during the sweep (excursion), so the sweep stands when every
// e_i <= 0.9 m_i.  Otherwise the pairs that the overrunning circles left out are
// checked at their turns (k_cg_verify), and only if one met is the sweep undone and
// run again with the larger needs.
//
// Margins can differ by orders of magnitude (a jammed ring of circles around a
// collider beside quiet gas), so the grid is hierarchical: circle i sits at
// level L_i, the smallest L with m_i <= lim_L = lim_0 4^L, in a grid of cell size
// h_L = 2 (rmax + lim_L) (x1.001); all levels share one table of T buckets, cell
// (x, y) of level L in bucket (x + y stride + L c) mod T with stride about
// 0.618 T: the cells of a row are consecutive buckets.  Circle i scans the levels
// L <= L_i over the cells that its reach plus level L's largest reach covers, and
// the levels above L_i over the 3x3 cells around its own cell there, a run of
// records per row.  Both sides of a pair find it, so each circle writes its own
// list without atomics.
//
// The counting sort that fills the buckets also numbers the circles: slot s is
// place s in bucket order, and every array of the sweep after the sort goes by
// slot.  The circles that a wavefront's 64 slots meet lie in a few runs of
// neighbouring slots, where by circle number every access took a cache line of
// its own (262,144 circles, 32 sweeps and the upload: 32.7 ms, 23.6 by slot; with
// what follows 13.2).
// Only the order of the pairs is by circle number: lists are sorted by it, and an
// entry holds the partner's slot and, in kLater, whether its number is larger.
//
// The sweep then runs per connected component of the candidate graph: pairs
// of different components share no circle, so they commute, and within one
// component the reference's (i, j) order (src/solver.rs:168-177) is kept by the
// round protocol: pair (i, j) runs once j is the next unprocessed partner of i and
// i the next of j.  Components of up to 4, 16 and 64 circles run in as many lanes
// of a wavefront, a circle to a lane; larger ones in a workgroup, in LDS or, above
// kLdsMembers circles, in global memory.
//
// The host waits once a sweep, for its verdict, and the device meanwhile runs what
// follows: the bodies, which look at the verdict themselves, and the zeroes of the
// next sweep's counters (a copy, a wait for the stream and then those two launches
// left the device idle: 20,011 circles, 8 updates with clone and readback 5.2 -> 4.2
// ms, 262,144 11.5 -> 10.8).  Lists are handed their space by
// one atomic per workgroup, out of what earlier sweeps needed (a sweep whose
// lists do not fit changes nothing and runs again with more), components
// likewise, and the check of overruns takes their number from device memory.
// Counters that many wavefronts add to are added to once a workgroup: 4,096
// atomics on one word take about 30 us (k_cg_check 34 -> 11 us).

constexpr uint32_t kSlotG = 16;  // candidates kept by the counting scan
constexpr uint32_t kLvlShift = 26;  // bucket record .w: circle | level << 26
constexpr uint32_t kIdxMaskG = (1u << kLvlShift) - 1u;
constexpr uint32_t kLater = 0x80000000u;   // list entry: the partner's number is larger
constexpr uint32_t kParent = 0x40000000u;  // list entry: the parent that the circle starts with (k_cg_union)
constexpr uint32_t kLaneList = 32;  // list entries of a circle that a lane holds
constexpr uint32_t kLdsMembers = 1024, kLdsEntries = 8192;
// A reach over more cells than kMaxScanCells in one level scans every circle.  One
// over more than kOwnScanCells (a circle above level 0; level 0 takes up to 3 x 3)
// is scanned by 16 lanes, kPieceCells cells of a row to each at a time: left to
// its own lane it held up the launch.
constexpr int64_t kMaxScanCells = 1024, kOwnScanCells = 32;
constexpr int kPieceCells = 4;
constexpr uint32_t kNoneG = 0xffffffffu;
constexpr int kCompWG = 256;
// Lanes that share a slot's edges in k_cg_union: an edge is a chain of a dozen
// dependent loads, and jammed circles have a dozen edges (one lane a slot 17.5 us
// with 20,011 circles and 25.0 with 262,144, four 8.9 and 19.1).
constexpr uint32_t kEdgeLanes = 4;
constexpr uint32_t kCheckPer = 4;  // slots a thread of k_cg_ranges and k_cg_check

// Per-sweep grid of every level, in device memory.
struct CGrid {
    double inv_h[kLevels];
    float lim[kLevels];        // largest margin of level L: lim_0 * 4^L
    float reach_max[kLevels];  // largest reach of level L: rmax + lim
};

__device__ __forceinline__ int cell_coord_d(double x, double inv_h) {
    double c = floor(x * inv_h);
    if (!(c > -1073741824.0)) c = -1073741824.0;
    if (c > 1073741824.0) c = 1073741824.0;
    return (int)c;
}

// Cell of a point for a cell size 1 / inv_h, clamped to +-2^30 so that huge
// or non-finite coordinates stay finite.
__device__ __forceinline__ int cell_coord(float x, double inv_h) { return cell_coord_d((double)x, inv_h); }

// Largest margin and inverse cell size of level L.
__device__ __forceinline__ float level_lim(float lim0, uint32_t L) { return ldexpf(lim0, 2 * (int)L); }
__device__ __forceinline__ double level_inv_h(float rmax, float lim) {
    return 1.0 / ((2.0 * (double)(rmax + lim)) * 1.001 + 1e-30);
}

// Margin of a circle that needs `need`, and its level.
__device__ __forceinline__ float level_margin(float s0, float lim0, float need, uint32_t &L) {
    const float m = fmaxf(s0, need);
    L = 0;
    while (L + 1 < (uint32_t)kLevels && m > level_lim(lim0, L)) L++;
    return fminf(m, level_lim(lim0, L));
}

struct Buckets {
    uint32_t nc, tmask, stride;
    const uint32_t *__restrict__ start;
    const float4 *__restrict__ rec;
};

__device__ __forceinline__ uint32_t bucket_of(uint32_t tmask, uint32_t stride, uint32_t L, int cx, int cy) {
    return ((uint32_t)cx + (uint32_t)cy * stride + L * 0x9e3779b9u) & tmask;
}

// Calls f(slot, record) for the records of level L in the cells x0 .. x1 of the
// rows y, y + step, ... <= y1.  A row's cells are one run of slots, going on at
// slot 0 after the last; three rows are looked up at a time and their runs read as
// one, kU records in flight (row by row every level cost three chains of dependent
// loads, for mostly empty runs).  near(record) is asked first: a run may hold
// other cells' and levels' records.
template <typename N, typename F>
__device__ __forceinline__ void scan_rows(const Buckets &b, uint32_t L, int x0, int x1, int y, int y1, int step,
                                          double ih, N near, F f) {
    const uint32_t nx = (uint32_t)(x1 - x0) + 1u, T = b.tmask + 1u;
    constexpr uint32_t kU = 4;
    for (; y <= y1; y += 3 * step) {
        uint32_t s0[3], len[3];
#pragma unroll
        for (int k = 0; k < 3; k++) {
            s0[k] = 0u;
            len[k] = 0u;
            if (y + k * step > y1) continue;
            len[k] = b.nc;  // (as many cells as buckets: all records)
            if (nx <= b.tmask) {
                const uint32_t at = bucket_of(b.tmask, b.stride, L, x0, y + k * step), e = at + nx;
                s0[k] = b.start[at];
                const uint32_t s1 = b.start[e > T ? e - T : e];
                len[k] = e > T ? b.nc - s0[k] + s1 : s1 - s0[k];
            }
        }
        const uint32_t p1 = len[0], p2 = p1 + len[1], total = p2 + len[2];
        for (uint32_t t0 = 0; t0 < total; t0 += kU) {
            float4 q[kU];
            uint32_t s[kU];
            int cy[kU];
#pragma unroll
            for (uint32_t u = 0; u < kU; u++) {
                const uint32_t t = min(t0 + u, total - 1u);
                s[u] = t < p1 ? s0[0] + t : t < p2 ? s0[1] + (t - p1) : s0[2] + (t - p2);
                cy[u] = t < p1 ? y : t < p2 ? y + step : y + 2 * step;
                if (s[u] >= b.nc) s[u] -= b.nc;
                q[u] = b.rec[s[u]];
            }
#pragma unroll
            for (uint32_t u = 0; u < kU; u++) {
                if (t0 + u >= total || !near(q[u])) continue;
                if ((__float_as_uint(q[u].w) >> kLvlShift) != L) continue;
                if (cell_coord(q[u].y, ih) != cy[u]) continue;
                const int cx = cell_coord(q[u].x, ih);
                if (cx < x0 || cx > x1) continue;
                f(s[u], q[u]);
            }
        }
    }
}

// The levels' grid, each circle's bucket and its rank there.  Thread t takes the
// circle that was in slot t in the sweep before: its neighbours in the wavefront
// then count into the same few cache lines of counters, and go to neighbouring
// slots in the scatter (by number each atomic was a request of its own).  The
// circles' needs are kept by that slot too.
__global__ void __launch_bounds__(256) k_cg_prep(const float2 *__restrict__ pos, uint32_t cbase,
                                                 const float *__restrict__ need, const uint32_t *__restrict__ order,
                                                 float s0, float lim0, float rmax, uint32_t nc, uint32_t tmask,
                                                 uint32_t stride, CGrid *__restrict__ g,
                                                 uint2 *__restrict__ key, uint32_t *__restrict__ count,
                                                 uint32_t *__restrict__ ctl) {
    const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t < (uint32_t)kLevels) {
        const float lim = level_lim(lim0, t);
        g->lim[t] = lim;
        g->reach_max[t] = rmax + lim;
        g->inv_h[t] = level_inv_h(rmax, lim);
    }
    uint32_t bit = 0;
    if (t < nc) {
        const uint32_t i = order[t];
        const float2 p = pos[cbase + i];
        uint32_t L;
        (void)level_margin(s0, lim0, need[t], L);
        const double ih = level_inv_h(rmax, level_lim(lim0, L));
        const uint32_t k = bucket_of(tmask, stride, L, cell_coord(p.x, ih), cell_coord(p.y, ih));
        key[t] = make_uint2(k, atomicAdd(&count[k], 1u));
        bit = 1u << L;
    }
    // occupied levels above 0 (level 0 counts as occupied): an atomic only where
    // a wavefront holds a level not yet seen in the word
    for (int o = 32; o > 0; o >>= 1) bit |= __shfl_xor(bit, o);
    bit &= ~1u;
    if ((threadIdx.x & 63u) == 0u && bit &&
        (bit & ~__hip_atomic_load(&ctl[kCtlMask], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)))
        atomicOr(&ctl[kCtlMask], bit);
}

// Each circle's record to its slot: position, reach, number and level in rec;
// radius, margin and need in aux.
__global__ void __launch_bounds__(256) k_cg_scatter(const float2 *__restrict__ pos, uint32_t cbase,
                                                    const float *__restrict__ crad, const float *__restrict__ need,
                                                    const uint32_t *__restrict__ order, float s0, float lim0,
                                                    const uint2 *__restrict__ key, uint32_t nc,
                                                    const uint32_t *__restrict__ start, float4 *__restrict__ rec,
                                                    float4 *__restrict__ aux) {
    const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= nc) return;
    const uint32_t i = order[t];
    const uint2 k = key[t];
    const uint32_t s = start[k.x] + k.y;
    const float2 p = pos[cbase + i];
    const float nd = need[t], r = crad[i];
    uint32_t L;
    const float m = level_margin(s0, lim0, nd, L);
    rec[s] = make_float4(p.x, p.y, r + m, __uint_as_float(i | (L << kLvlShift)));
    aux[s] = make_float4(r, m, nd, 0.0f);
}

template <typename T>
__device__ __forceinline__ void cswap(T &a, T &b) {
    const T lo = min(a, b), hi = max(a, b);
    a = lo; b = hi;
}

// Exclusive place of each thread's v among the workgroup's 256 threads; total is
// the sum (64-bit: lists can be as long as the scene).  s_sum: 4 words of LDS.
__device__ __forceinline__ uint64_t block_place(uint32_t v, uint64_t *s_sum, uint64_t &total) {
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    uint64_t inc = v;
    for (int o = 1; o < 64; o <<= 1) {
        const uint64_t t = __shfl_up(inc, o);
        if ((int)lane >= o) inc += t;
    }
    if (lane == 63u) s_sum[wave] = inc;
    __syncthreads();
    uint64_t base = 0;
    total = 0;
    for (uint32_t w = 0; w < 4u; w++) {
        if (w < wave) base += s_sum[w];
        total += s_sum[w];
    }
    return base + inc - v;
}

// Candidates of the circle in each slot (see above), in one go: count and keep
// the first kSlotG in LDS, take space for the workgroup's lists, write them
// sorted by circle number (longer ones from a second scan, through keys, the
// trajectories' space).  What the rest of the sweep starts from goes by the way:
// positions, excursions and parents (a circle hangs under the smallest slot of
// its list at once, which leaves the union a third of the edges).
__global__ void __launch_bounds__(256) k_cg_cand(Buckets bk, const CGrid *__restrict__ g, uint32_t cap,
                                                 uint32_t *__restrict__ cnt, uint32_t *__restrict__ off,
                                                 uint32_t *__restrict__ cand, uint64_t *__restrict__ keys,
                                                 uint32_t *__restrict__ par, uint32_t *__restrict__ csize,
                                                 float2 *__restrict__ spos, float *__restrict__ exc,
                                                 uint32_t *__restrict__ order, const float4 *__restrict__ aux,
                                                 float *__restrict__ need, uint32_t *__restrict__ ctl) {
    __shared__ uint64_t s_keep[kSlotG][256];
    __shared__ uint64_t s_sum[4], s_base;
    __shared__ uint32_t s_n[256], s_o[256], s_wide[256], s_nwide;
    const uint32_t tid = threadIdx.x, lane = tid & 63u, s = blockIdx.x * 256u + tid;
    const uint32_t mask = ctl[kCtlMask] | 1u;
    float4 r = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    bool on = false, wide = false;
    if (s < bk.nc) {
        r = bk.rec[s];
        spos[s] = make_float2(r.x, r.y);
        exc[s] = 0.0f;
        csize[s] = 0u;
        order[s] = __float_as_uint(r.w) & kIdxMaskG;
        need[s] = aux[s].z;
        // a circle at a non-finite position takes part in no pair
        on = fabsf(r.x) <= 3.0e38f && fabsf(r.y) <= 3.0e38f;
    }
    // the cells of level L within reach of a circle
    struct Span { int x0, x1, y0, y1; };
    auto span = [&](const float4 &c, uint32_t L, double ih) {
        const double R = ((double)c.z + (double)g->reach_max[L]) * (1.0 + 1e-6);
        return Span{cell_coord_d((double)c.x - R, ih), cell_coord_d((double)c.x + R, ih),
                    cell_coord_d((double)c.y - R, ih), cell_coord_d((double)c.y + R, ih)};
    };
    auto cells = [&](const float4 &c) {
        int64_t most = 0;
        for (uint32_t m = mask & ((2u << (__float_as_uint(c.w) >> kLvlShift)) - 1u); m; m &= m - 1u) {
            const uint32_t L = (uint32_t)__ffs(m) - 1u;
            const Span w = span(c, L, g->inv_h[L]);
            most = max(most, ((int64_t)w.x1 - w.x0 + 1) * ((int64_t)w.y1 - w.y0 + 1));
        }
        return most;
    };
    // f(key) for every candidate of the circle c in slot self: all of them, or with
    // SHARED those of the pieces that fall to this of 16 lanes
    auto gather = [&](const float4 &c, uint32_t self, auto shared, auto f) {
        constexpr bool kShared = decltype(shared)::value;
        auto near = [&](const float4 &q) {
            const float dx = c.x - q.x, dy = c.y - q.y, lim = c.z + q.z;
            return dx * dx + dy * dy < lim * lim;
        };
        auto found = [&](uint32_t t, const float4 &q) {
            if (t != self) f(((uint64_t)(__float_as_uint(q.w) & kIdxMaskG) << 32) | t);
        };
        if (kShared && cells(c) > kMaxScanCells) {
            for (uint32_t t = tid & 15u; t < bk.nc; t += 16u) {
                const float4 q = bk.rec[t];
                if (near(q)) found(t, q);
            }
            return;
        }
        const uint32_t low = (2u << (__float_as_uint(c.w) >> kLvlShift)) - 1u;  // levels up to its own
        for (uint32_t m = mask; m; m &= m - 1u) {
            const uint32_t L = (uint32_t)__ffs(m) - 1u;
            const double ih = g->inv_h[L];
            Span w;
            if ((low >> L) & 1u) w = span(c, L, ih);
            else {
                const int cx = cell_coord(c.x, ih), cy = cell_coord(c.y, ih);
                w = Span{cx - 1, cx + 1, cy - 1, cy + 1};
            }
            if constexpr (!kShared) {
                scan_rows(bk, L, w.x0, w.x1, w.y0, w.y1, 1, ih, near, found);
            } else {
                const uint32_t pieces = (uint32_t)(w.x1 - w.x0 + kPieceCells) / (uint32_t)kPieceCells;
                const uint32_t items = pieces * (uint32_t)(w.y1 - w.y0 + 1);
                for (uint32_t k = tid & 15u; k < items; k += 16u) {
                    const int x = w.x0 + (int)(k % pieces) * kPieceCells, y = w.y0 + (int)(k / pieces);
                    scan_rows(bk, L, x, min(x + kPieceCells - 1, w.x1), y, y, 1, ih, near, found);
                }
            }
        }
    };
    if (tid == 0u) s_nwide = 0u;
    __syncthreads();
    if (on && cells(r) > kOwnScanCells) {
        wide = true;
        s_wide[atomicAdd(&s_nwide, 1u)] = tid;
    }
    // 16 lanes for each circle with a wide scan: f(its thread, place, key)
    auto gather_wide = [&](auto f) {
        for (uint32_t k = tid >> 4; k < s_nwide; k += 16u) {
            const uint32_t st = s_wide[k], self = blockIdx.x * 256u + st;
            if (s_n[st] == kNoneG) continue;  // (nothing to do)
            gather(bk.rec[self], self, std::true_type{}, [&](uint64_t key) { f(st, atomicAdd(&s_n[st], 1u), key); });
        }
    };
    s_n[tid] = 0u;
    uint32_t n = 0;
    if (on && !wide)
        gather(r, s, std::false_type{}, [&](uint64_t key) {
            if (n < kSlotG) s_keep[n][tid] = key;
            n++;
        });
    __syncthreads();
    gather_wide([&](uint32_t st, uint32_t k, uint64_t key) {
        if (k < kSlotG) s_keep[k][st] = key;
    });
    __syncthreads();
    if (wide) n = s_n[tid];
    __syncthreads();
    s_n[tid] = n > kSlotG ? 0u : kNoneG;
    uint64_t total;
    const uint64_t at = block_place(n, s_sum, total);
    if (tid == 0u)
        s_base = total ? atomicAdd((unsigned long long *)&ctl[kCtlTotal], (unsigned long long)total) : 0ull;
    __syncthreads();
    const uint64_t base = s_base;
    if (base + total > cap) {  // uniform: nothing is replayed, the host makes room
        if (tid == 0u) ctl[kCtlFull] = 1u;
        return;
    }
    const uint32_t o0 = (uint32_t)(base + at);
    s_o[tid] = o0;
    __syncthreads();
    if (n > kSlotG && !wide) {
        uint32_t k = 0;
        gather(r, s, std::false_type{}, [&](uint64_t key) { keys[o0 + k++] = key; });
    }
    gather_wide([&](uint32_t st, uint32_t k, uint64_t key) {
        keys[s_o[st] + k] = key;
    });
    __syncthreads();
    // lists from a second scan: a wavefront each, U keys to a lane at a time, ranked
    // by number against all keys, 64 of them in a register that every lane's
    // comparison reads a lane of (a lane's own sort in memory was a chain of loads;
    // with 16 instead of 8 entries kept in LDS, which spares most lists the second
    // scan, this kernel took 20.0 us instead of 34.9 with 20,011 circles and 34.0
    // instead of 51.6 with 262,144).  The comparisons grow with the square of the
    // length: with 20,000 lists of 2,000 entries and one of 20,000 the scans and sorts
    // took 104 ms with a heap sort in a lane, 236 with a load for each key and list,
    // 113 like this; what the pairs of longer lists take grows as fast and is more.
    const uint32_t number = __float_as_uint(r.w) & kIdxMaskG;
    auto rank_list = [&](const uint64_t *k, uint32_t *to, uint32_t ln, uint32_t li, uint32_t least, auto per) {
        constexpr uint32_t U = decltype(per)::value;
        for (uint32_t x0 = 0; x0 < ln; x0 += 64u * U) {
            uint64_t key[U];
            uint32_t rank[U];
#pragma unroll
            for (uint32_t u = 0; u < U; u++) {
                key[u] = k[min(x0 + 64u * u + lane, ln - 1u)];
                rank[u] = 0u;
            }
            for (uint32_t y0 = 0; y0 < ln; y0 += 64u) {
                const uint32_t m = min(ln - y0, 64u);
                const uint32_t theirs = lane < m ? (uint32_t)(k[y0 + lane] >> 32) : kNoneG;
                for (uint32_t y = 0; y < m; y += 8u)
#pragma unroll
                    for (uint32_t v = 0; v < 8u; v++) {
                        const uint32_t one = __builtin_amdgcn_readlane(theirs, y + v);
#pragma unroll
                        for (uint32_t u = 0; u < U; u++) rank[u] += one < (uint32_t)(key[u] >> 32) ? 1u : 0u;
                    }
            }
#pragma unroll
            for (uint32_t u = 0; u < U; u++)
                if (x0 + 64u * u + lane < ln)
                    to[rank[u]] = (uint32_t)key[u] | ((uint32_t)(key[u] >> 32) > li ? kLater : 0u) |
                                  ((uint32_t)key[u] == least ? kParent : 0u);
        }
    };
    uint32_t low = s;
    for (uint64_t todo = __ballot(n > kSlotG); todo; todo &= todo - 1ull) {
        const int src = __ffsll((unsigned long long)todo) - 1;
        const uint32_t ln = (uint32_t)__shfl((int)n, src), lo0 = (uint32_t)__shfl((int)o0, src);
        const uint32_t li = (uint32_t)__shfl((int)number, src), self = s - lane + (uint32_t)src;
        const uint64_t *const k = keys + lo0;
        uint32_t least = self;
        for (uint32_t x = lane; x < ln; x += 64u) least = min(least, (uint32_t)k[x]);
        for (int o = 32; o > 0; o >>= 1) least = min(least, (uint32_t)__shfl_xor((int)least, o));
        if (ln <= 64u) rank_list(k, cand + lo0, ln, li, least, std::integral_constant<uint32_t, 1>{});
        else rank_list(k, cand + lo0, ln, li, least, std::integral_constant<uint32_t, 4>{});
        if ((int)lane == src) low = least;
    }
    if (s >= bk.nc) return;
    cnt[s] = n;
    off[s] = o0;
    auto entry = [&](uint64_t key) {
        return (uint32_t)key | ((uint32_t)(key >> 32) > number ? kLater : 0u) | ((uint32_t)key == low ? kParent : 0u);
    };
    // the kept ones by a sorting network of the size that the wavefront needs
    auto put = [&](auto size) {
        constexpr uint32_t K = decltype(size)::value;
        uint64_t v[K];
#pragma unroll
        for (uint32_t k = 0; k < K; k++) v[k] = k < n ? s_keep[k][tid] : ~0ull;
#pragma unroll
        for (uint32_t k = 2; k <= K; k <<= 1)
#pragma unroll
            for (uint32_t j = k >> 1; j > 0; j >>= 1)
#pragma unroll
                for (uint32_t x = 0; x < K; x++) {
                    const uint32_t l = x ^ j;
                    if (l > x) {
                        if ((x & k) == 0u) cswap(v[x], v[l]);
                        else cswap(v[l], v[x]);
                    }
                }
#pragma unroll
        for (uint32_t k = 0; k < K; k++)
            if (k < n) low = min(low, (uint32_t)v[k]);
#pragma unroll
        for (uint32_t k = 0; k < K; k++)
            if (k < n) cand[o0 + k] = entry(v[k]);
    };
    if (n <= kSlotG) {
        if (__ballot(n > 4u) == 0ull) put(std::integral_constant<uint32_t, 4>{});
        else if (__ballot(n > 8u) == 0ull) put(std::integral_constant<uint32_t, 8>{});
        else put(std::integral_constant<uint32_t, kSlotG>{});
    }
    par[s] = low;
}

// Union-find over the candidate graph, by slot.  parent[x] <= x always (a root is
// hooked under the smaller root), so every value ever read is an ancestor, also
// one that another XCD has replaced since: the walks may read it from the caches
// (their loads are of workgroup scope).  Hooking compares and swaps at device
// scope: a stale root fails there and gives its parent; a stale partner that is
// no root any more is still an ancestor to hang under, and smaller.
__device__ __forceinline__ uint32_t uf_load(const uint32_t *p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

__device__ uint32_t uf_find(uint32_t *par, uint32_t x) {
    for (;;) {
        const uint32_t p = uf_load(par + x);
        if (p == x) return x;
        const uint32_t g = uf_load(par + p);
        if (g == p) return p;
        __hip_atomic_store(par + x, g, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);  // path halving
        x = g;
    }
}

__global__ void __launch_bounds__(256) k_cg_union(const uint32_t *__restrict__ cnt, const uint32_t *__restrict__ off,
                                                  const uint32_t *__restrict__ cand, uint32_t nc, uint32_t *par,
                                                  const uint32_t *__restrict__ ctl) {
    const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x, i = t / kEdgeLanes;
    if (i >= nc || ctl[kCtlFull]) return;
    const uint32_t s0 = off[i], n = cnt[i];
    for (uint32_t s = t % kEdgeLanes; s < n; s += kEdgeLanes) {
        const uint32_t e = cand[s0 + s];
        uint32_t a = e & kIdxMaskG, b = i;
        if (a >= i || (e & kParent)) continue;  // each edge once, from its larger end
        for (;;) {
            a = uf_find(par, a);
            b = uf_find(par, b);
            if (a == b) break;
            if (a > b) { const uint32_t t = a; a = b; b = t; }
            const uint32_t old = atomicCAS(par + b, b, a);
            if (old == b) break;
            b = old;  // b was hooked meanwhile
        }
    }
}

// Component of each listed circle (its smallest slot), its place among the
// component's members, and the components' sizes.
__global__ void __launch_bounds__(256) k_cg_comp(const uint32_t *__restrict__ cnt, uint32_t nc, uint32_t *par,
                                                 uint32_t *__restrict__ root, uint32_t *__restrict__ place,
                                                 uint32_t *__restrict__ csize, const uint32_t *__restrict__ ctl) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nc || ctl[kCtlFull] || cnt[i] == 0u) return;
    const uint32_t r = uf_find(par, i);
    root[i] = r;
    place[i] = atomicAdd(&csize[r], 1u);
}

// Space for each component's members, and the queues by size, queue q at
// queues + q nc.  One atomic per workgroup and counter.
__global__ void __launch_bounds__(256) k_cg_ranges(const uint32_t *__restrict__ csize, uint32_t nc,
                                                   uint32_t *__restrict__ cstart, uint32_t *__restrict__ queues,
                                                   uint32_t *__restrict__ ctl) {
    __shared__ uint64_t s_sum[4];
    __shared__ uint32_t s_base[kQueues + 1], s_n[kQueues];
    const uint32_t tid = threadIdx.x;
    if (ctl[kCtlFull]) return;  // uniform
    if (tid < kQueues) s_n[tid] = 0u;
    __syncthreads();
    uint32_t n[kCheckPer], at[kCheckPer], sum = 0;
    auto queue_of = [](uint32_t m) {
        return m <= 4u ? 0u : m <= 16u ? 1u : m <= 64u ? 2u : m <= kLdsMembers ? kQueueLds : kQueueBig;
    };
#pragma unroll
    for (uint32_t u = 0; u < kCheckPer; u++) {
        const uint32_t i = (blockIdx.x * kCheckPer + u) * 256u + tid;
        n[u] = i < nc ? csize[i] : 0u;  // (0 but at roots)
        sum += n[u];
        if (n[u]) at[u] = atomicAdd(&s_n[queue_of(n[u])], 1u);
    }
    uint64_t total;
    uint32_t place = (uint32_t)block_place(sum, s_sum, total);
    if (tid <= kQueues) {
        const uint32_t add = tid < kQueues ? s_n[tid] : (uint32_t)total;
        s_base[tid] = add ? atomicAdd(&ctl[tid < kQueues ? kCtlQueue + tid : kCtlMembers], add) : 0u;
    }
    __syncthreads();
#pragma unroll
    for (uint32_t u = 0; u < kCheckPer; u++) {
        const uint32_t i = (blockIdx.x * kCheckPer + u) * 256u + tid;
        if (n[u] == 0u) continue;
        const uint32_t q = queue_of(n[u]);
        queues[(size_t)q * nc + s_base[q] + at[u]] = i;
        cstart[i] = s_base[kQueues] + place;
        place += n[u];
    }
}

// Members of each component, grouped at cstart[root].
__global__ void __launch_bounds__(256) k_cg_members(const uint32_t *__restrict__ cnt, const uint32_t *__restrict__ root,
                                                    const uint32_t *__restrict__ place,
                                                    const uint32_t *__restrict__ cstart, uint32_t nc,
                                                    uint32_t *__restrict__ members, const uint32_t *__restrict__ ctl) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nc || ctl[kCtlFull] || cnt[i] == 0u) return;
    members[cstart[root[i]] + place[i]] = i;
}

// The sweep's largest number of rounds: an atomic only for a new one (one for each
// of 14,000 components took 100 us).
__device__ __forceinline__ void note_rounds(uint32_t *ctl, uint32_t rounds) {
    if (rounds > __hip_atomic_load(&ctl[kCtlRounds], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
        atomicMax(&ctl[kCtlRounds], rounds);
}

// Components of at most W circles, W = 4, 16 or 64: W lanes of a wavefront each, a
// circle to a lane, its position in registers.  A round is: my next partner's next
// partner, and if that is me, its position, by lane permutes; both lanes of a pair
// then solve it alike and each keeps its own side.  Nothing is written between
// rounds but the trajectory.  (20,011 circles 28 -> 11 us, 262,144 72 -> 45 us
// against a wavefront with the state in LDS and a worklist for each component, and
// a serial replay by one lane for those of up to 4.)  The lists, as places in the component, are
// staged in LDS, each with a bit for a partner of larger number: such a pair's first
// end is the circle itself (the order shows in the sign of a zero).  A component with
// a longer list than kLaneList joins the queue of the LDS workgroups.
template <uint32_t W>
__device__ __forceinline__ void replay_lanes(uint32_t from, uint32_t step, const uint32_t *__restrict__ queue,
                                             uint32_t nq, float2 *__restrict__ P, const float4 *__restrict__ aux,
                                             const float4 *__restrict__ rec, float *__restrict__ exc,
                                             const uint32_t *__restrict__ cnt, const uint32_t *__restrict__ off,
                                             const uint32_t *__restrict__ cand, const uint32_t *__restrict__ csize,
                                             const uint32_t *__restrict__ cstart, const uint32_t *__restrict__ members,
                                             const uint32_t *__restrict__ place, uint32_t *__restrict__ lds_queue,
                                             float2 *__restrict__ traj, uint32_t *__restrict__ ctl,
                                             uint8_t (*s_list)[kLaneList + 4]) {
    constexpr uint32_t kNone8 = 0xffu, kLater8 = 0x40u;
    const uint32_t lane = threadIdx.x & 63u, k = lane & (W - 1u), base = lane & ~(W - 1u);
    uint32_t most = 0;
    for (uint32_t q0 = from; q0 < nq; q0 += step) {  // uniform per wavefront
        const uint32_t q = q0 + lane / W;
        uint32_t c = 0, m = 0, o = 0, r = 0;
        float2 p = make_float2(0.0f, 0.0f), p0 = p;
        float rad = 0.0f, e = 0.0f;
        bool on = false, fits = true;
        if (q < nq) {
            r = queue[q];
            on = k < csize[r];
            if (on) {
                c = members[cstart[r] + k];
                m = cnt[c];
                o = off[c];
                const float4 v = rec[c];
                p = p0 = make_float2(v.x, v.y);
                rad = aux[c].x;
                fits = m <= kLaneList;
            }
        }
        // (all lanes of the component take part, or none)
        const uint64_t group = (W == 64u ? ~0ull : ((1ull << (W & 63u)) - 1ull)) << base;
        if (__ballot(!fits) & group) {
            if (on && k == 0u) lds_queue[atomicAdd(&ctl[kCtlQueue + kQueueLds], 1u)] = r;
            on = false;
        }
        if (!on) m = 0u;
        constexpr uint32_t kU = 4;
        for (uint32_t t0 = 0; t0 < m; t0 += kU) {
            uint32_t v[kU];
#pragma unroll
            for (uint32_t u = 0; u < kU; u++) v[u] = cand[o + min(t0 + u, m - 1u)];
#pragma unroll
            for (uint32_t u = 0; u < kU; u++) v[u] = place[v[u] & kIdxMaskG] | (v[u] & kLater ? kLater8 : 0u);
#pragma unroll
            for (uint32_t u = 0; u < kU; u++) s_list[lane][t0 + u] = (uint8_t)v[u];  // (kU - 1 past the end at most)
        }
        if (m) s_list[lane][m] = (uint8_t)kNone8;
        uint32_t next = m ? s_list[lane][0] : kNone8, head = 0, rounds = 0;
        for (;; rounds++) {
            const int src = (int)(base + (next & (W - 1u)));
            const uint32_t theirs = (uint32_t)__shfl((int)next, src);
            const float2 pj = make_float2(__shfl(p.x, src), __shfl(p.y, src));
            const float rj = __shfl(rad, src);
            const bool first = (next & kLater8) != 0u;
            // (my partner's entry for me has the other bit; kNone8 is neither)
            const bool ready = next != kNone8 && theirs == (first ? k : k | kLater8);
            if (!__ballot(ready)) break;
            if (ready) {
                const uint32_t after = s_list[lane][head + 1u];
                float2 a = first ? p : pj, b = first ? pj : p;
                float qi = 0.0f, qj = 0.0f;
                if (solve_circle_pair(a.x, a.y, b.x, b.y, first ? rad : rj, first ? rj : rad, qi, qj)) {
                    p = first ? a : b;
                    e = excursion(e, p.x, p.y, p0.x, p0.y);
                }
                traj[o + head] = p;
                head++;
                next = after;
            }
        }
        if (on) {
            P[c] = p;
            exc[c] = e;
            if (head != m) atomicOr(&ctl[kCtlBad], 1u);
        }
        most = max(most, rounds);
    }
    if (lane == 0u && most) note_rounds(ctl, most);
}

// The components of up to 64 circles, largest first: the first workgroup past those
// of each queue.
struct LaneBlocks {
    uint32_t end64, end16, end4;
};

__global__ void __launch_bounds__(64) k_cg_lanes(float2 *__restrict__ P, const float4 *__restrict__ aux,
                                                 const float4 *__restrict__ rec, float *__restrict__ exc,
                                                 const uint32_t *__restrict__ cnt, const uint32_t *__restrict__ off,
                                                 const uint32_t *__restrict__ cand, const uint32_t *__restrict__ csize,
                                                 const uint32_t *__restrict__ cstart,
                                                 const uint32_t *__restrict__ members,
                                                 const uint32_t *__restrict__ place, uint32_t *__restrict__ queues,
                                                 uint32_t nc, LaneBlocks blk, float2 *__restrict__ traj,
                                                 uint32_t *__restrict__ ctl) {
    __shared__ uint8_t s_list[64][kLaneList + 4];
    if (ctl[kCtlFull]) return;  // uniform
    const uint32_t b = blockIdx.x;
    uint32_t *const lds_queue = queues + (size_t)kQueueLds * nc;
    if (b < blk.end64)
        replay_lanes<64>(b, blk.end64, queues + 2 * (size_t)nc, ctl[kCtlQueue + 2], P, aux, rec, exc, cnt, off, cand,
                         csize, cstart, members, place, lds_queue, traj, ctl, s_list);
    else if (b < blk.end16)
        replay_lanes<16>((b - blk.end64) * 4u, (blk.end16 - blk.end64) * 4u, queues + nc, ctl[kCtlQueue + 1], P, aux, rec,
                         exc, cnt, off, cand, csize, cstart, members, place, lds_queue, traj, ctl, s_list);
    else
        replay_lanes<4>((b - blk.end16) * 16u, (blk.end4 - blk.end16) * 16u, queues, ctl[kCtlQueue], P, aux, rec, exc,
                        cnt, off, cand, csize, cstart, members, place, lds_queue, traj, ctl, s_list);
}

// Components of 65 .. kLdsMembers circles, and smaller ones with long lists: a
// workgroup each, with the round protocol in LDS.  The members' positions, start
// positions, radii and excursions are staged into LDS and the lists remapped to
// local indices (a circle's place among the members, with kLater16 for a partner of
// larger number: the pair's first end is then the circle itself); the lists keep
// their order, which is all the protocol depends on.  Positions after each pair go to
// traj in global memory as in the other replays.  A component whose lists do
// not fit joins the queue of the global-memory workgroups.
__global__ void __launch_bounds__(256) k_cg_lds(float2 *__restrict__ P, const float4 *__restrict__ aux,
                                                const float4 *__restrict__ rec, float *__restrict__ exc,
                                                const uint32_t *__restrict__ cnt, const uint32_t *__restrict__ off,
                                                const uint32_t *__restrict__ cand, const uint32_t *__restrict__ csize,
                                                const uint32_t *__restrict__ cstart,
                                                const uint32_t *__restrict__ members,
                                                const uint32_t *__restrict__ place, uint32_t *__restrict__ queues,
                                                uint32_t nc, float2 *__restrict__ traj, uint32_t *__restrict__ ctl) {
    __shared__ float2 s_p[kLdsMembers], s_s[kLdsMembers];
    __shared__ float s_r[kLdsMembers], s_e[kLdsMembers];
    __shared__ uint32_t s_off[kLdsMembers];
    __shared__ uint16_t s_lb[kLdsMembers], s_cnt[kLdsMembers], s_head[kLdsMembers], s_nxp[kLdsMembers],
        s_stamp[kLdsMembers];
    __shared__ uint16_t s_list[kLdsEntries];
    __shared__ uint32_t s_wl[2][kLdsMembers / 2 + 1];
    __shared__ uint32_t s_n[3], s_bad;
    __shared__ uint64_t s_sum[4];
    constexpr uint16_t kNone16 = 0xffffu, kLater16 = 0x8000u;
    static_assert(kLdsMembers <= 0x7fffu, "a place and its flag in 16 bits");
    const uint32_t tid = threadIdx.x;
    // the pair that x's next entry y makes, its first end in the low half, once x is
    // the next partner of y too; 0 when it is not (no pair is: the ends differ)
    auto pair_of = [&](uint32_t x, uint32_t y) -> uint32_t {
        if (y == kNone16) return 0u;
        const uint32_t o = y & 0x7fffu;
        if (y & kLater16) return s_nxp[o] == x ? x | (o << 16) : 0u;
        return s_nxp[o] == (x | kLater16) ? o | (x << 16) : 0u;
    };
    if (ctl[kCtlFull]) return;  // uniform
    const uint32_t nmid = ctl[kCtlQueue + kQueueLds];
    const uint32_t *const queue = queues + (size_t)kQueueLds * nc;
    for (uint32_t q = blockIdx.x; q < nmid; q += gridDim.x) {  // uniform per workgroup
        const uint32_t r = queue[q], n = csize[r];
        const uint32_t *M = members + cstart[r];
        // stage; each thread takes consecutive members for the scan
        constexpr uint32_t kPer = kLdsMembers / 256u;
        uint32_t sum = 0;
        for (uint32_t u = 0; u < kPer; u++) {
            const uint32_t k = tid * kPer + u;
            if (k < n) {
                const uint32_t c = M[k];
                const float4 v = rec[c];
                s_p[k] = s_s[k] = make_float2(v.x, v.y);
                s_r[k] = aux[c].x;
                s_e[k] = 0.0f;
                s_off[k] = off[c];
                const uint32_t m = cnt[c];
                s_cnt[k] = (uint16_t)min(m, 0xffffu);
                sum += m;
            }
        }
        // exclusive list starts
        uint64_t total;
        uint32_t run = (uint32_t)block_place(sum, s_sum, total);
        if (total > kLdsEntries) {  // uniform: the lists do not fit
            if (tid == 0) queues[(size_t)kQueueBig * nc + atomicAdd(&ctl[kCtlQueue + kQueueBig], 1u)] = r;
            __syncthreads();
            continue;
        }
        for (uint32_t u = 0; u < kPer; u++) {
            const uint32_t k = tid * kPer + u;
            if (k < n) {
                s_lb[k] = (uint16_t)run;
                run += s_cnt[k];
            }
        }
        if (tid == 0) { s_n[0] = 0u; s_n[1] = 0u; s_n[2] = 0u; s_bad = 0u; }
        __syncthreads();
        // local lists
        for (uint32_t k = tid; k < n; k += 256u) {
            const uint32_t *src = cand + s_off[k];
            uint16_t *dst = s_list + s_lb[k];
            for (uint32_t e = 0, m = s_cnt[k]; e < m; e++)
                dst[e] = (uint16_t)(place[src[e] & kIdxMaskG] | (src[e] & kLater ? kLater16 : 0u));
        }
        __syncthreads();
        for (uint32_t k = tid; k < n; k += 256u) {
            s_head[k] = 0;
            s_nxp[k] = s_cnt[k] ? s_list[s_lb[k]] : kNone16;
            s_stamp[k] = kNone16;
        }
        __syncthreads();
        for (uint32_t k = tid; k < n; k += 256u) {
            const uint32_t y = s_nxp[k], pr = y & kLater16 ? pair_of(k, y) : 0u;  // each from its first end
            if (pr) s_wl[0][atomicAdd(&s_n[0], 1u)] = pr;
        }
        __syncthreads();
        uint32_t cur = s_n[0], rounds = 0;
        for (; cur > 0; rounds++) {
            const uint32_t cb = rounds & 1u, nb = cb ^ 1u;
            for (uint32_t k = tid; k < cur; k += 256u) {
                const uint32_t pr = s_wl[cb][k], c = pr & 0xffffu, o = pr >> 16;
                float2 pi = s_p[c], pj = s_p[o];
                const uint32_t hc = s_head[c], ho = s_head[o];
                const uint32_t xc = hc + 1u < s_cnt[c] ? s_list[s_lb[c] + hc + 1u] : kNone16;
                const uint32_t xo = ho + 1u < s_cnt[o] ? s_list[s_lb[o] + ho + 1u] : kNone16;
                float qi = 0.0f, qj = 0.0f;
                if (solve_circle_pair(pi.x, pi.y, pj.x, pj.y, s_r[c], s_r[o], qi, qj)) {
                    s_p[c] = pi;
                    s_p[o] = pj;
                    s_e[c] = excursion(s_e[c], pi.x, pi.y, s_s[c].x, s_s[c].y);
                    s_e[o] = excursion(s_e[o], pj.x, pj.y, s_s[o].x, s_s[o].y);
                }
                traj[s_off[c] + hc] = pi;
                traj[s_off[o] + ho] = pj;
                s_head[c] = (uint16_t)(hc + 1u);
                s_head[o] = (uint16_t)(ho + 1u);
                s_nxp[c] = (uint16_t)xc;
                s_nxp[o] = (uint16_t)xo;
                s_stamp[c] = (uint16_t)rounds;
                s_stamp[o] = (uint16_t)rounds;
            }
            if (tid == 0) s_n[(rounds + 2u) % 3u] = 0u;
            __syncthreads();
            for (uint32_t k = tid; k < cur; k += 256u) {
                const uint32_t pr = s_wl[cb][k];
                for (int e = 0; e < 2; e++) {
                    const uint32_t x = e ? pr >> 16 : pr & 0xffffu, y = s_nxp[x], np = pair_of(x, y);
                    // when both ends moved this round the first one adds the pair
                    if (np == 0u || (s_stamp[y & 0x7fffu] == (uint16_t)rounds && !(y & kLater16))) continue;
                    s_wl[nb][atomicAdd(&s_n[(rounds + 1u) % 3u], 1u)] = np;
                }
            }
            __syncthreads();
            cur = s_n[(rounds + 1u) % 3u];
        }
        for (uint32_t k = tid; k < n; k += 256u) {
            const uint32_t c = M[k];
            P[c] = s_p[k];
            exc[c] = s_e[k];
            if (s_head[k] != s_cnt[k]) s_bad = 1u;
        }
        __syncthreads();
        if (tid == 0) {
            if (s_bad) atomicOr(&ctl[kCtlBad], 1u);
            note_rounds(ctl, rounds);
        }
        __syncthreads();
    }
}

// A circle of a component that is replayed in memory: all that a pair reads and
// writes of it in half a cache line.  (Such a component's circles are met in no
// order of memory: as nine arrays, 150,000 circles of which 1 % are 8 times as large
// missed L2 530 million times in 16 sweeps of 124 ms; like this they take 86.)
struct __align__(64) CompCircle {
    float2 p, from;
    float rad, exc;
    uint32_t off, cnt, head, nxp, stamp;
};

// Components above kLdsMembers circles (or whose lists overflow LDS): one
// workgroup each, taken from a queue,
// with the round protocol.  head counts a circle's processed partners and nxp
// is the next one (kNoneG when done; with kLater when its number is larger, the
// circle then being the pair's first end), so (x, y) is ready exactly when
// x's nxp is y and y's is x.  Every round applies at least one pair, so the
// loop ends; a list left unfinished (a schedule that stalls) is reported.
// comp: a record a circle, or null until a scene has such a component; its sweep
// then changes nothing and runs again with them (a gas never does, and allocating
// them for a clone of 262,144 circles took 0.3 ms of its 11).
__global__ void __launch_bounds__(kCompWG) k_cg_comps(float2 *__restrict__ P, const float4 *__restrict__ aux,
                                                      const float4 *__restrict__ rec, float *__restrict__ exc,
                                                      const uint32_t *__restrict__ cnt,
                                                      const uint32_t *__restrict__ off,
                                                      const uint32_t *__restrict__ cand,
                                                      const uint32_t *__restrict__ csize,
                                                      const uint32_t *__restrict__ cstart,
                                                      const uint32_t *__restrict__ members,
                                                      const uint32_t *__restrict__ queues, uint32_t nc,
                                                      CompCircle *__restrict__ comp, uint2 *__restrict__ wl,
                                                      float2 *__restrict__ traj, uint32_t *__restrict__ ctl) {
    __shared__ uint32_t s_n[3], s_bad;
    const uint32_t tid = threadIdx.x;
    if (ctl[kCtlFull]) return;  // uniform
    const uint32_t nbig = ctl[kCtlQueue + kQueueBig];
    if (nbig != 0u && !comp) {  // uniform
        if (tid == 0u) ctl[kCtlFull] = 1u;
        return;
    }
    const uint32_t *const bigq = queues + (size_t)kQueueBig * nc;
    constexpr uint32_t kEntry = kIdxMaskG | kLater;
    // whether x is the next partner of its own next partner y
    auto mutual = [&](uint32_t x, uint32_t y) {
        return y != kNoneG && comp[y & kIdxMaskG].nxp == (y & kLater ? x : x | kLater);
    };
    for (uint32_t q = blockIdx.x; q < nbig; q += gridDim.x) {  // uniform per workgroup
        const uint32_t r = bigq[q], base = cstart[r], n = csize[r];
        const uint32_t *M = members + base;
        uint2 *const W[2] = {wl + base, wl + nc + base};
        for (uint32_t k = tid; k < n; k += kCompWG) {
            const uint32_t c = M[k], m = cnt[c], o = off[c];
            const float4 v = rec[c];
            const float2 p = make_float2(v.x, v.y);
            comp[c] = CompCircle{p, p, aux[c].x, 0.0f, o, m, 0u, m ? cand[o] & kEntry : kNoneG, kNoneG};
        }
        if (tid == 0) { s_n[0] = 0u; s_n[1] = 0u; s_n[2] = 0u; s_bad = 0u; }
        __syncthreads();
        for (uint32_t k = tid; k < n; k += kCompWG) {
            const uint32_t c = M[k], y = comp[c].nxp;
            if ((y & kLater) && mutual(c, y)) W[0][atomicAdd(&s_n[0], 1u)] = make_uint2(c, y & kIdxMaskG);
        }
        __syncthreads();
        uint32_t cur = s_n[0], rounds = 0;
        for (; cur > 0; rounds++) {
            const uint32_t now = rounds & 1u, nb = now ^ 1u;
            for (uint32_t k = tid; k < cur; k += kCompWG) {
                const uint2 pr = W[now][k];
                // (whole records: storing only what changed took 7 % longer)
                CompCircle a = comp[pr.x], b = comp[pr.y];
                const uint32_t ua = a.off + a.head++, ub = b.off + b.head++;
                a.nxp = a.head < a.cnt ? cand[ua + 1u] & kEntry : kNoneG;
                b.nxp = b.head < b.cnt ? cand[ub + 1u] & kEntry : kNoneG;
                a.stamp = b.stamp = rounds;
                float qi = 0.0f, qj = 0.0f;
                if (solve_circle_pair(a.p.x, a.p.y, b.p.x, b.p.y, a.rad, b.rad, qi, qj)) {
                    a.exc = excursion(a.exc, a.p.x, a.p.y, a.from.x, a.from.y);
                    b.exc = excursion(b.exc, b.p.x, b.p.y, b.from.x, b.from.y);
                }
                traj[ua] = a.p;
                traj[ub] = b.p;
                comp[pr.x] = a;
                comp[pr.y] = b;
            }
            if (tid == 0) s_n[(rounds + 2u) % 3u] = 0u;  // read two barriers ago
            __syncthreads();
            // pairs completed by a moved head; when both ends moved this round
            // the first one adds the pair
            for (uint32_t k = tid; k < cur; k += kCompWG) {
                const uint2 pr = W[now][k];
                for (int e = 0; e < 2; e++) {
                    const uint32_t x = e ? pr.y : pr.x, y = comp[x].nxp, o = y & kIdxMaskG;
                    const bool first = (y & kLater) != 0u;
                    if (!mutual(x, y) || (comp[o].stamp == rounds && !first)) continue;
                    W[nb][atomicAdd(&s_n[(rounds + 1u) % 3u], 1u)] = first ? make_uint2(x, o) : make_uint2(o, x);
                }
            }
            __syncthreads();
            cur = s_n[(rounds + 1u) % 3u];
        }
        for (uint32_t k = tid; k < n; k += kCompWG) {
            const uint32_t c = M[k];
            P[c] = comp[c].p;
            exc[c] = comp[c].exc;
            if (comp[c].head != comp[c].cnt) s_bad = 1u;
        }
        __syncthreads();
        if (tid == 0) {
            if (s_bad) atomicOr(&ctl[kCtlBad], 1u);
            note_rounds(ctl, rounds);
        }
        __syncthreads();  // s_n and s_bad are rewritten for the next component
    }
}

// Validity of the sweep, the circles' needs for the next one, and their positions
// back by circle number.  Circles that went further than 0.9 of their margin are
// queued in overq, and for each level the largest r + e among them goes to
// ctl[kCtlEmax + L] (as bits: positive floats order like their bit patterns).
// Atomics are taken once per workgroup, of kCheckPer slots a thread.
__global__ void __launch_bounds__(256) k_cg_check(const float *__restrict__ exc, const float4 *__restrict__ aux,
                                                  const float4 *__restrict__ rec, const float2 *__restrict__ spos,
                                                  const uint32_t *__restrict__ cnt, float *__restrict__ need, float s0,
                                                  uint32_t nc, float2 *__restrict__ pos, uint32_t cbase,
                                                  uint32_t *__restrict__ overq, uint32_t *__restrict__ ctl) {
    __shared__ uint32_t s_emax[kLevels], s_over, s_flags, s_base;
    const uint32_t tid = threadIdx.x;
    if (ctl[kCtlFull]) return;  // uniform: nothing was replayed
    if (tid < (uint32_t)kLevels) s_emax[tid] = 0u;
    if (tid == 0u) { s_over = 0u; s_flags = 0u; }
    __syncthreads();
    uint32_t at[kCheckPer];
#pragma unroll
    for (uint32_t u = 0; u < kCheckPer; u++) {
        const uint32_t s = (blockIdx.x * kCheckPer + u) * 256u + tid;
        at[u] = kNoneG;
        if (s >= nc) continue;
        const float4 a = aux[s], q = rec[s];
        const uint32_t i = __float_as_uint(q.w) & kIdxMaskG;
        const float e = exc[s];
        const bool over = !(e <= 0.9f * a.y), inf = !(e <= 3.0e38f);
        // jammed circles swing from sweep to sweep: the need keeps twice the
        // excursion and forgets slowly
        if (!inf) need[s] = fmaxf(2.0f * e, 0.9f * a.z);
        if (cnt[s]) pos[cbase + i] = spos[s];
        if (over) {
            at[u] = atomicAdd(&s_over, 1u);
            // (bit 1: a circle at the base margin overran)
            if (inf) atomicOr(&s_flags, 1u);
            else atomicMax(&s_emax[__float_as_uint(q.w) >> kLvlShift], __float_as_uint(a.x + e));
            if (!inf && a.y <= s0) atomicOr(&s_flags, 2u);
        }
    }
    __syncthreads();
    const uint32_t n = s_over;
    if (n == 0u) return;  // uniform
    if (tid == 0u) s_base = atomicAdd(&ctl[kCtlOver], n);
    if (tid == 1u && (s_flags & 1u)) atomicOr(&ctl[kCtlInf], 1u);
    if (tid == 2u && (s_flags & 2u)) atomicOr(&ctl[kCtlQuiet], 1u);
    if (tid < (uint32_t)kLevels && s_emax[tid]) atomicMax(&ctl[kCtlEmax + tid], s_emax[tid]);
    __syncthreads();
#pragma unroll
    for (uint32_t u = 0; u < kCheckPer; u++)
        if (at[u] != kNoneG) overq[s_base + at[u]] = (blockIdx.x * kCheckPer + u) * 256u + tid;
}

// Exact check of a sweep with overruns, one wavefront per overrunning circle.
// Pair (i, j) was skipped if j is not in i's list.  It cannot have met during
// the sweep if |save_i - save_j| >= (r_i + e_i) + (r_j + e_j), e being the
// excursions; a circle within its margin has r_j + e_j <= reach_j, so only
// pairs with an overrunning end can have met, and each overrunning circle
// scans every level L over (r_i + e_i) + max(largest reach of L, largest
// r + e of the overruns at L).  A skipped pair (a, b), a < b, that passes that
// test is tested at its own turn, as the reference would: a has then done its
// pairs with partners below b, b its pairs with partners below a, and traj
// holds each circle's position after each of its pairs.  If it overlapped
// there, the sweep is marked for a redo; otherwise skipping it changed nothing.
__global__ void __launch_bounds__(256) k_cg_verify(Buckets bk, const float4 *__restrict__ aux,
                                                   const float *__restrict__ exc, const CGrid *__restrict__ g,
                                                   const uint32_t *__restrict__ cnt, const uint32_t *__restrict__ off,
                                                   const uint32_t *__restrict__ cand,
                                                   const uint32_t *__restrict__ overq,
                                                   const float2 *__restrict__ traj, uint32_t *__restrict__ ctl) {
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t n_over = ctl[kCtlFull] ? 0u : ctl[kCtlOver];
    const uint32_t mask = ctl[kCtlMask] | 1u;
    auto number = [&](uint32_t s) { return __float_as_uint(bk.rec[s].w) & kIdxMaskG; };
    // entries of slot s's list with numbers below v
    auto rank = [&](uint32_t s, uint32_t v) {
        const uint32_t *l = cand + off[s];
        uint32_t lo = 0, hi = cnt[s];
        while (lo < hi) {
            const uint32_t mid = (lo + hi) >> 1;
            if (number(l[mid] & kIdxMaskG) < v) lo = mid + 1u; else hi = mid;
        }
        return lo;
    };
    bool missed = false;
    for (uint32_t k = (blockIdx.x * 256u + threadIdx.x) >> 6; k < n_over; k += gridDim.x * 4u) {  // uniform per wavefront
        const uint32_t i = overq[k];
        const float4 p = bk.rec[i];
        if (!(fabsf(p.x) <= 3.0e38f && fabsf(p.y) <= 3.0e38f)) continue;
        const float ai = aux[i].x + exc[i];
        const uint32_t ni = __float_as_uint(p.w) & kIdxMaskG;
        // a record's own reach covers r + e of a circle within its margin, the
        // level's largest r + e that of an overrun
        auto near = [&](const float4 &q, float emax) {
            const float lim = (ai + fmaxf(q.z, emax)) * (1.0f + 0x1p-15f);
            const float dx = p.x - q.x, dy = p.y - q.y;
            return dx * dx + dy * dy < lim * lim;
        };
        auto test = [&](uint32_t j, const float4 &q) {
            if (j == i) return;
            const float lim = (ai + (aux[j].x + exc[j])) * (1.0f + 0x1p-16f);
            const float dx = p.x - q.x, dy = p.y - q.y;
            const float d2 = dx * dx + dy * dy, reach = p.z + q.z;
            // within both reaches: listed (by this very test), and replayed in order
            if (!(d2 < lim * lim) || d2 < reach * reach) return;
            const uint32_t nj = __float_as_uint(q.w) & kIdxMaskG;
            const uint32_t ri = rank(i, nj), rj = rank(j, ni);
            const float2 pi = ri ? traj[off[i] + ri - 1u] : make_float2(p.x, p.y);
            const float2 pj = rj ? traj[off[j] + rj - 1u] : make_float2(q.x, q.y);
            const bool first = ni < nj;
            const float2 pa = first ? pi : pj, pb = first ? pj : pi;
            const float ex = pa.x - pb.x, ey = pa.y - pb.y;
            const float rs = first ? aux[i].x + aux[j].x : aux[j].x + aux[i].x;
            if (ex * ex + ey * ey < rs * rs) missed = true;
        };
        auto reach_at = [&](uint32_t L) {
            return ((double)ai + (double)fmaxf(g->reach_max[L], __uint_as_float(ctl[kCtlEmax + L]))) * (1.0 + 1e-4);
        };
        bool brute = false;
        for (uint32_t m = mask; m; m &= m - 1u) {
            const uint32_t L = (uint32_t)__ffs(m) - 1u;
            const double R = reach_at(L), ih = g->inv_h[L];
            const int64_t nx = (int64_t)cell_coord_d((double)p.x + R, ih) - cell_coord_d((double)p.x - R, ih) + 1;
            const int64_t ny = (int64_t)cell_coord_d((double)p.y + R, ih) - cell_coord_d((double)p.y - R, ih) + 1;
            if (nx * ny > kMaxScanCells || nx * ny > (int64_t)bk.tmask) brute = true;
        }
        if (brute) {
            for (uint32_t j = lane; j < bk.nc; j += 64u) test(j, bk.rec[j]);
            continue;
        }
        for (uint32_t m = mask; m; m &= m - 1u) {
            const uint32_t L = (uint32_t)__ffs(m) - 1u;
            const double R = reach_at(L), ih = g->inv_h[L];
            const float emax = __uint_as_float(ctl[kCtlEmax + L]);
            const int x0 = cell_coord_d((double)p.x - R, ih), x1 = cell_coord_d((double)p.x + R, ih);
            const int y0 = cell_coord_d((double)p.y - R, ih), y1 = cell_coord_d((double)p.y + R, ih);
            const uint32_t cells = (uint32_t)(x1 - x0) + 1u, T = bk.tmask + 1u;
            // a lane looks up a row's run of records; the records of up to 64 rows are
            // then spread over the lanes (a row, or a piece of one, to a lane left most
            // of them idle where a few cells hold thousands of records)
            for (int r0 = y0; r0 <= y1; r0 += 64) {
                uint32_t s0 = 0, len = 0;
                if (r0 + (int)lane <= y1) {
                    const uint32_t at = bucket_of(bk.tmask, bk.stride, L, x0, r0 + (int)lane), e = at + cells;
                    s0 = bk.start[at];
                    const uint32_t s1 = bk.start[e > T ? e - T : e];
                    len = e > T ? bk.nc - s0 + s1 : s1 - s0;
                }
                uint32_t end = len;
                for (int o = 1; o < 64; o <<= 1) {
                    const uint32_t v = (uint32_t)__shfl_up((int)end, o);
                    if ((int)lane >= o) end += v;
                }
                const uint32_t total = (uint32_t)__shfl((int)end, 63);
                for (uint32_t t0 = 0; t0 < total; t0 += 64u) {
                    const uint32_t t = min(t0 + lane, total - 1u);
                    uint32_t row = 0;  // the rows that end at t or before
                    for (uint32_t o = 32u; o > 0u; o >>= 1)
                        if ((uint32_t)__shfl((int)end, (int)(row + o - 1u)) <= t) row += o;
                    uint32_t s = (uint32_t)__shfl((int)s0, (int)row) + (t - (uint32_t)__shfl((int)(end - len), (int)row));
                    if (s >= bk.nc) s -= bk.nc;
                    const float4 q = bk.rec[s];
                    if (t0 + lane >= total || !near(q, emax)) continue;
                    if ((__float_as_uint(q.w) >> kLvlShift) != L || cell_coord(q.y, ih) != r0 + (int)row) continue;
                    const int cx = cell_coord(q.x, ih);
                    if (cx >= x0 && cx <= x1) test(s, q);
                }
            }
        }
    }
    if (missed) atomicOr(&ctl[kCtlMissed], 1u);
}

// The positions that the sweep started from, back by circle number.
__global__ void k_cc_restore(float2 *__restrict__ pos, uint32_t cbase, const float4 *__restrict__ rec, uint32_t nc) {
    const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= nc) return;
    const float4 q = rec[s];
    pos[cbase + (__float_as_uint(q.w) & kIdxMaskG)] = make_float2(q.x, q.y);
}

// ---------------------------------------------------------------------------
// Engine
// ---------------------------------------------------------------------------

class GlobalEngine : public Engine {
public:
    explicit GlobalEngine(hipStream_t s) : stream_(s) {}
    ~GlobalEngine() override {
        if (host_ctl_) (void)hipHostFree(host_ctl_);
    }
    int kind() const override { return BD_ENGINE_GLOBAL; }

    int upload(const HostScene &s, const Plan &p, std::string &err) override {
        Np_ = p.Np; Nc_ = p.Nc; Ng_ = p.Ng; N_ = p.N;
        P_ = (uint32_t)s.polys.size();
        layer_off_ = p.layer_off;
        depth_ = p.depth;
        std::vector<float2> pos(N_), prev(N_);
        auto put = [&](const std::vector<V2> &a, const std::vector<V2> &b, uint32_t base) {
            for (size_t i = 0; i < a.size(); i++) {
                pos[base + i] = make_float2(a[i].x, a[i].y);
                prev[base + i] = make_float2(b[i].x, b[i].y);
            }
        };
        put(s.p_pos, s.p_prev, 0);
        put(s.c_pos, s.c_prev, Np_);
        put(s.g_pos, s.g_prev, Np_ + Nc_);
        BD_HIP(pos_.alloc(std::max<size_t>(N_, 1)));
        BD_HIP(prev_.alloc(std::max<size_t>(N_, 1)));
        if (N_) {
            BD_HIP(hipMemcpyAsync(pos_.p, pos.data(), N_ * sizeof(float2), hipMemcpyHostToDevice, stream_));
            BD_HIP(hipMemcpyAsync(prev_.p, prev.data(), N_ * sizeof(float2), hipMemcpyHostToDevice, stream_));
        }
        // links
        BD_HIP(links_.alloc(std::max<size_t>(p.links.size(), 1)));
        if (!p.links.empty())
            BD_HIP(hipMemcpyAsync(links_.p, p.links.data(), p.links.size() * sizeof(Link12), hipMemcpyHostToDevice, stream_));
        // pins
        has_pins_ = s.any_pinned();
        if (has_pins_) {
            std::vector<uint32_t> mask((Np_ + 31) / 32, 0u);
            for (uint32_t i = 0; i < Np_; i++)
                if (s.p_pin[i]) mask[i >> 5] |= 1u << (i & 31);
            BD_HIP(pinmask_.alloc(mask.size()));
            BD_HIP(hipMemcpyAsync(pinmask_.p, mask.data(), mask.size() * 4, hipMemcpyHostToDevice, stream_));
        }
        // circle radii
        BD_HIP(crad_.alloc(std::max<size_t>(Nc_, 1)));
        if (Nc_) BD_HIP(hipMemcpyAsync(crad_.p, s.c_r.data(), Nc_ * 4, hipMemcpyHostToDevice, stream_));
        // initial acc of circles and polygon points
        if (Nc_ + Ng_) {
            std::vector<float2> acc(Nc_ + Ng_);
            for (uint32_t i = 0; i < Nc_; i++) acc[i] = make_float2(s.c_acc[i].x, s.c_acc[i].y);
            for (uint32_t i = 0; i < Ng_; i++) acc[Nc_ + i] = make_float2(s.g_acc[i].x, s.g_acc[i].y);
            BD_HIP(acc0_.alloc(acc.size()));
            BD_HIP(hipMemcpyAsync(acc0_.p, acc.data(), acc.size() * sizeof(float2), hipMemcpyHostToDevice, stream_));
        }
        // polygons
        if (P_) {
            std::vector<uint2> tab(P_);
            std::vector<uint8_t> flags(std::max<uint32_t>(Ng_, 1), 0);
            for (uint32_t i = 0; i < P_; i++) {
                tab[i] = make_uint2(Np_ + Nc_ + s.polys[i].off, s.polys[i].n);
                for (uint32_t k = 0; k < s.polys[i].n; k++) flags[s.polys[i].off + k] = s.polys[i].is_static ? 1 : 0;
            }
            BD_HIP(ptab_.alloc(P_));
            BD_HIP(centers_.alloc(P_));
            BD_HIP(gflags_.alloc(flags.size()));
            BD_HIP(hipMemcpyAsync(ptab_.p, tab.data(), P_ * sizeof(uint2), hipMemcpyHostToDevice, stream_));
            BD_HIP(hipMemcpyAsync(gflags_.p, flags.data(), flags.size(), hipMemcpyHostToDevice, stream_));
            std::vector<float2> c(P_);
            for (uint32_t i = 0; i < P_; i++) c[i] = make_float2(s.polys[i].center.x, s.polys[i].center.y);
            BD_HIP(hipMemcpyAsync(centers_.p, c.data(), P_ * sizeof(float2), hipMemcpyHostToDevice, stream_));
            static_poly_.clear();
            for (uint32_t i = 0; i < P_; i++)
                if (s.polys[i].is_static) static_poly_.push_back(i);
        }
        // static colliders
        ncol_ = (uint32_t)s.cols.size();
        nplanes_ = (uint32_t)(s.planes.size() / 3);
        if (ncol_) {
            std::vector<int4> hdr(ncol_);
            std::vector<float4> geo(ncol_);
            for (uint32_t k = 0; k < ncol_; k++) {
                const Collider &c = s.cols[k];
                hdr[k] = make_int4(c.kind, (int)c.plane_off, (int)c.nv, 0);
                geo[k] = make_float4(c.cx, c.cy, c.r, 0.0f);
            }
            std::vector<float4> pl(std::max<uint32_t>(nplanes_, 1));
            for (uint32_t k = 0; k < nplanes_; k++)
                pl[k] = make_float4(s.planes[3 * k], s.planes[3 * k + 1], s.planes[3 * k + 2], 0.0f);
            BD_HIP(colhdr_.alloc(ncol_));
            BD_HIP(colgeo_.alloc(ncol_));
            BD_HIP(planes_.alloc(pl.size()));
            BD_HIP(hipMemcpyAsync(colhdr_.p, hdr.data(), ncol_ * sizeof(int4), hipMemcpyHostToDevice, stream_));
            BD_HIP(hipMemcpyAsync(colgeo_.p, geo.data(), ncol_ * sizeof(float4), hipMemcpyHostToDevice, stream_));
            BD_HIP(hipMemcpyAsync(planes_.p, pl.data(), pl.size() * sizeof(float4), hipMemcpyHostToDevice, stream_));
        }
        if (!host_ctl_) BD_HIP(hipHostMalloc((void **)&host_ctl_, 64 * sizeof(uint32_t), hipHostMallocDefault));
        host_ctl_[kCtlWords] = verdict_ = 0u;
        zeroed_[0] = zeroed_[1] = false;
        rmax_ = 0.0f;
        for (float r : s.c_r) rmax_ = std::max(rmax_, r);
        if (Nc_ > kIdxMaskG) {
            err = "too many circles for one scene";
            return BD_ERR_ARG;
        }
        // per-circle margins start at the base margin
        s0_ = std::max(0.125f * rmax_, s0_min());
        clean_ = 0;
        BD_HIP(cg_need_.alloc(std::max<uint32_t>(Nc_, 1)));
        if (Nc_) BD_HIP(hipMemsetAsync(cg_need_.p, 0, Nc_ * sizeof(float), stream_));
        BD_HIP(cg_order_.alloc(std::max<uint32_t>(Nc_, 1)));
        std::vector<uint32_t> order(Nc_);
        for (uint32_t i = 0; i < Nc_; i++) order[i] = i;
        if (Nc_) BD_HIP(hipMemcpyAsync(cg_order_.p, order.data(), Nc_ * 4, hipMemcpyHostToDevice, stream_));
        // the upload copies read host vectors that die at return
        BD_HIP(hipStreamSynchronize(stream_));
        return BD_OK;
    }

    int update(const StepParams &sp, Stats &st, std::string &err) override {
        BodyParams bp;
        bp.dt = sp.delta; bp.gex = sp.gex; bp.gey = sp.gey; bp.gx = sp.gx; bp.gy = sp.gy;
        bp.lox = sp.lox; bp.loy = sp.loy; bp.hix = sp.hix; bp.hiy = sp.hiy;
        bp.N = N_; bp.Np = Np_; bp.Nc = Nc_;
        bp.ncol = ncol_;
        for (uint32_t step = 0; step < sp.sub_steps; step++) {
            bp.first_acc = (sp.first_acc && step == 0 && acc0_.p) ? 1u : 0u;
            // links, k sweeps; polygon centres before the last sweep
            for (uint32_t it = 0; it < sp.link_iters; it++) {
                if (P_ && it + 1 == sp.link_iters) {
                    hipLaunchKernelGGL(k_poly_centers, dim3((P_ + 255) / 256), dim3(256), 0, stream_, pos_.p, ptab_.p, P_, centers_.p);
                    st.launches++;
                }
                for (uint32_t d = 0; d < depth_; d++) {
                    uint32_t o = layer_off_[d], n = layer_off_[d + 1] - o;
                    hipLaunchKernelGGL(k_link_layer, dim3((n + 255) / 256), dim3(256), 0, stream_, pos_.p, links_.p + o, n, crad_.p, Np_);
                    st.launches++;
                }
            }
            if (P_ && sp.link_iters == 0) {
                hipLaunchKernelGGL(k_poly_centers, dim3((P_ + 255) / 256), dim3(256), 0, stream_, pos_.p, ptab_.p, P_, centers_.p);
                st.launches++;
            }
            if (Nc_ >= 2) {
                int rc = circles(st, err, P_ < 2 ? &bp : nullptr);
                if (rc) return rc;
                if (P_ < 2) {  // the bodies came with the sweep
                    st.substeps++;
                    continue;
                }
            }
            if (P_ >= 2) {
                hipLaunchKernelGGL(k_poly_pairs, dim3(1), dim3(256), 0, stream_, pos_.p, ptab_.p, P_, centers_.p);
                st.launches++;
            }
            if (N_) launch_bodies(bp, nullptr, st);
            st.substeps++;
        }
        if (sp.first_acc && acc0_.p) {
            uint32_t n = Nc_ + Ng_;
            hipLaunchKernelGGL(k_zero_acc0, dim3((n + 255) / 256), dim3(256), 0, stream_, acc0_.p, n);
            st.launches++;
        }
        BD_HIP(hipGetLastError());
        return BD_OK;
    }

    size_t state_count() const override { return 2ull * N_ + P_; }
    hipStream_t stream() const override { return stream_; }

    StateParts state_parts() override {
        StateParts s;
        s.add(pos_.p, N_);
        s.add(prev_.p, N_);
        s.add(centers_.p, P_);
        return s;
    }

    int unpack(const float2 *src, HostScene &s, std::string &err) override {
        if (!host_shape_matches(s, Np_, Nc_, Ng_, err)) return BD_ERR_STATE;
        const float2 *pos = src, *prev = src + N_, *centers = src + 2 * N_;
        auto get = [&](std::vector<V2> &a, std::vector<V2> &b, uint32_t base) {
            for (size_t i = 0; i < a.size(); i++) {
                a[i] = V2{pos[base + i].x, pos[base + i].y};
                b[i] = V2{prev[base + i].x, prev[base + i].y};
            }
        };
        get(s.p_pos, s.p_prev, 0);
        get(s.c_pos, s.c_prev, Np_);
        get(s.g_pos, s.g_prev, Np_ + Nc_);
        for (uint32_t p : static_poly_) s.polys[p].center = V2{centers[p].x, centers[p].y};
        return BD_OK;
    }

    int sync(std::string &err) override {
        BD_HIP(hipStreamSynchronize(stream_));
        return BD_OK;
    }

private:
    // Exact replay of the circle-pair sweep (see the circle-pair kernels): lists
    // from per-circle margins on the level grid, components, then the lane and
    // workgroup replays.  A sweep in which a circle that went further than 0.9 of
    // its margin met a pair that was left out is undone and run again with the
    // needs it showed.
    // With bodies, the per-body phase follows in the attempt that stands.
    int circles(Stats &st, std::string &err, const BodyParams *bodies) {
        const uint32_t nc = Nc_;
        const uint32_t nb = (nc + 255) / 256;
        uint32_t T = 1;
        while (T < nc) T <<= 1;
        const uint32_t tmask = T - 1, stride = (uint32_t)(0.618034 * (double)T) | 1u;
        // control words and bucket counters, zeroed by one fill per attempt (the
        // scan's last entry with them)
        const size_t zn = kCtlWords + (size_t)T + 1;
        const int rw = place_workspace(nc, T, zn, err);
        if (rw) return rw;
        if (!cand_cap_) cand_cap_ = std::max<uint64_t>(4ull * nc, 1024);
        for (int attempt = 0; attempt < 12; attempt++) {
            const uint32_t turn = turn_;
            uint32_t *const ctl = ws_.zero[turn], *const count = ctl + kCtlWords;
            BD_HIP(cc_cand_.alloc(cand_cap_));
            BD_HIP(cg_traj_.alloc(cand_cap_));
            // Level 0 takes margins up to 1.5 r_max, also while the base margin is
            // less: circles in lasting contact need more than the base, and on level
            // 1 each scans 5x5 cells of level 0 (limit s0 17.4 ms, 0.5 r_max 16.9, 1.0
            // to 2.0 16.4 for 262,144 circles).
            const float lim0 = std::max(s0_, 1.5f * rmax_);
            if (!zeroed_[turn]) fill_u32(ctl, zn, 0u, st);
            zeroed_[turn] = false;
            hipLaunchKernelGGL(k_cg_prep, dim3(nb), dim3(256), 0, stream_, pos_.p, Np_, cg_need_.p, cg_order_.p, s0_,
                               lim0, rmax_, nc,
                               tmask, stride, ws_.grid, ws_.key, count, ctl);
            st.launches++;
            int rc = exclusive_scan_u32(count, ws_.start, T + 1, stream_, scan_tmp_, st.launches, err);
            if (rc) return rc;
            hipLaunchKernelGGL(k_cg_scatter, dim3(nb), dim3(256), 0, stream_, pos_.p, Np_, crad_.p, cg_need_.p, cg_order_.p,
                               s0_, lim0, ws_.key, nc, ws_.start, ws_.rec, ws_.aux);
            const Buckets bk{nc, tmask, stride, ws_.start, ws_.rec};
            hipLaunchKernelGGL(k_cg_cand, dim3(nb), dim3(256), 0, stream_, bk, ws_.grid, (uint32_t)cand_cap_, ws_.cnt,
                               ws_.off, cc_cand_.p, (uint64_t *)cg_traj_.p, ws_.par, ws_.csize, ws_.spos,
                               ws_.exc, cg_order_.p, ws_.aux, cg_need_.p, ctl);
            hipLaunchKernelGGL(k_cg_union, dim3((unsigned)(((uint64_t)nc * kEdgeLanes + 255u) / 256u)), dim3(256), 0, stream_, ws_.cnt, ws_.off, cc_cand_.p, nc,
                               ws_.par, ctl);
            hipLaunchKernelGGL(k_cg_comp, dim3(nb), dim3(256), 0, stream_, ws_.cnt, nc, ws_.par, ws_.root,
                               ws_.place, ws_.csize, ctl);
            hipLaunchKernelGGL(k_cg_ranges, dim3((nb + kCheckPer - 1) / kCheckPer), dim3(256), 0, stream_, ws_.csize, nc, ws_.cstart,
                               ws_.queues, ctl);
            hipLaunchKernelGGL(k_cg_members, dim3(nb), dim3(256), 0, stream_, ws_.cnt, ws_.root, ws_.place,
                               ws_.cstart, nc, ws_.members, ctl);
            // (a component for W lanes has more than W / 4 circles, one for 4 at least two)
            LaneBlocks blk;
            blk.end64 = std::min<uint32_t>(kLaneGrid, nc / 17 + 1);
            blk.end16 = blk.end64 + std::min<uint32_t>(kLaneGrid, nc / 5 / 4 + 1);
            blk.end4 = blk.end16 + std::min<uint32_t>(kLaneGrid, nc / 2 / 16 + 1);
            hipLaunchKernelGGL(k_cg_lanes, dim3(blk.end4), dim3(64), 0, stream_, ws_.spos, ws_.aux, ws_.rec,
                               ws_.exc, ws_.cnt, ws_.off, cc_cand_.p, ws_.csize, ws_.cstart, ws_.members,
                               ws_.place, ws_.queues, nc, blk, cg_traj_.p, ctl);
            hipLaunchKernelGGL(k_cg_lds, dim3(std::min<uint32_t>(kLdsGrid, nc / 65 + 1)), dim3(256), 0, stream_,
                               ws_.spos, ws_.aux, ws_.rec, ws_.exc, ws_.cnt, ws_.off, cc_cand_.p,
                               ws_.csize, ws_.cstart, ws_.members, ws_.place, ws_.queues, nc, cg_traj_.p, ctl);
            hipLaunchKernelGGL(k_cg_comps, dim3(kCompGrid), dim3(kCompWG), 0, stream_, ws_.spos, ws_.aux, ws_.rec,
                               ws_.exc, ws_.cnt, ws_.off, cc_cand_.p, ws_.csize, ws_.cstart,
                               ws_.members, ws_.queues, nc, cg_comp_.n >= nc ? cg_comp_.p : nullptr,
                               ws_.wl, cg_traj_.p, ctl);
            hipLaunchKernelGGL(k_cg_check, dim3((nb + kCheckPer - 1) / kCheckPer), dim3(256), 0, stream_, ws_.exc,
                               ws_.aux, ws_.rec, ws_.spos, ws_.cnt, cg_need_.p, s0_, nc, pos_.p, Np_,
                               ws_.overq, ctl);
            hipLaunchKernelGGL(k_cg_verify, dim3(std::min<uint32_t>((nc + 3) / 4, kVerifyGrid)), dim3(256), 0, stream_, bk,
                               ws_.aux, ws_.exc, ws_.grid, ws_.cnt, ws_.off, cc_cand_.p, ws_.overq,
                               cg_traj_.p, ctl);
            hipLaunchKernelGGL(k_cg_verdict, dim3(1), dim3(64), 0, stream_, ctl, host_ctl_, ++verdict_);
            st.launches += 12;
            if (bodies) launch_bodies(*bodies, ctl, st);
            turn_ ^= 1u;
            fill_u32(ws_.zero[turn_], zn, 0u, st);
            BD_HIP(hipGetLastError());
            zeroed_[turn_] = true;
            rc = await_verdict(err);
            if (rc) return rc;
            uint64_t total;
            std::memcpy(&total, host_ctl_ + kCtlTotal, sizeof total);
            if (host_ctl_[kCtlFull]) {
                // nothing was replayed: the same attempt again, with room
                if (total > cand_cap_) {
                    if (total + total / 4 > 0xffffffffull) {
                        err = "too many candidate circle pairs";
                        return BD_ERR_CAPACITY;
                    }
                    cand_cap_ = total + total / 4;
                } else {
                    BD_HIP(cg_comp_.alloc(nc));
                }
                attempt--;
                continue;
            }
            st.cc_pairs = total / 2;
            st.cc_rounds += host_ctl_[kCtlRounds];
            if (host_ctl_[kCtlBad]) {
                err = "circle pair schedule stalled";
                return BD_ERR_COLLISION;
            }
            if (host_ctl_[kCtlInf]) {
                err = "circle pair sweep produced a non-finite push";
                return BD_ERR_COLLISION;
            }
            if (!host_ctl_[kCtlMissed]) {
                // quiet sweeps let the base margin shrink back
                if (++clean_ >= 16) {
                    s0_ = std::max(0.8f * s0_, s0_min());
                    clean_ = 0;
                }
                st.cc_margin = s0_;
                return BD_OK;
            }
            // a skipped pair may have met: undo, widen, redo
            st.cc_redos++;
            hipLaunchKernelGGL(k_cc_restore, dim3(nb), dim3(256), 0, stream_, pos_.p, Np_, ws_.rec, nc);
            st.launches++;
            clean_ = 0;
            // capped at 0.75 r_max: measured best over the gas box's run (0.25-1.0)
            if (host_ctl_[kCtlQuiet]) s0_ = std::min(1.5f * s0_, std::max(0.75f * rmax_, s0_min()));
        }
        err = "circle pair margin did not converge";
        return BD_ERR_COLLISION;
    }

    void launch_bodies(const BodyParams &bp, const uint32_t *verdict, Stats &st) {
        const uint32_t blocks = std::min<uint32_t>((N_ + 255) / 256, 65535u * 4);
        hipLaunchKernelGGL(k_bodies, dim3(blocks), dim3(256), 0, stream_, pos_.p, prev_.p,
                           has_pins_ ? pinmask_.p : nullptr, crad_.p, acc0_.p, gflags_.p, colhdr_.p, colgeo_.p,
                           planes_.p, bp, verdict);
        st.launches++;
    }

    // Waits for the last verdict: for its number at first, where a sweep takes some
    // hundred microseconds, then for the stream.
    int await_verdict(std::string &err) {
        auto here = [&]() { return __atomic_load_n(host_ctl_ + kCtlWords, __ATOMIC_ACQUIRE) == verdict_; };
        const auto until = std::chrono::steady_clock::now() + std::chrono::milliseconds(2);
        while (!here()) {
            if (std::chrono::steady_clock::now() < until) continue;
            BD_HIP(hipStreamSynchronize(stream_));
            if (here()) break;
            err = "circle pair sweep gave no verdict";
            return BD_ERR_DEVICE;
        }
        return BD_OK;
    }

    // The sweep's workspace, one allocation: 22 of them, and as many releases, took
    // 1.5 to 4 ms of a scene's life (a clone rolled out for 32 sweeps: 16 ms).
    struct Workspace {
        uint32_t *zero[2], *start, *cnt, *off, *par, *root, *place, *csize, *cstart, *members, *queues, *overq;
        float *exc;
        float2 *spos;
        float4 *rec, *aux;
        uint2 *key, *wl;
        CGrid *grid;
    };

    int place_workspace(uint32_t nc, uint32_t T, size_t zn, std::string &err) {
        size_t at = 0;
        auto take = [&](auto *&p, size_t count) {
            using V = std::remove_reference_t<decltype(*p)>;
            p = cg_arena_.p ? (V *)(cg_arena_.p + at) : nullptr;
            at += (count * sizeof(V) + 255) & ~(size_t)255;
        };
        auto all = [&]() {
            at = 0;
            take(ws_.zero[0], zn); take(ws_.zero[1], zn);
            take(ws_.grid, 1);
            take(ws_.key, nc); take(ws_.start, (size_t)T + 1); take(ws_.rec, nc); take(ws_.aux, nc);
            take(ws_.spos, nc); take(ws_.exc, nc); take(ws_.cnt, nc); take(ws_.off, nc);
            take(ws_.par, nc); take(ws_.root, nc); take(ws_.place, nc); take(ws_.csize, nc);
            take(ws_.cstart, nc); take(ws_.members, nc); take(ws_.queues, kQueues * (size_t)nc);
            take(ws_.overq, nc);
            take(ws_.wl, 2 * (size_t)nc);
        };
        all();
        BD_HIP(cg_arena_.alloc(at));
        all();
        return BD_OK;
    }

    float s0_min() const { return 0.05f * std::max(rmax_, 1e-3f); }

    void fill_u32(uint32_t *p, size_t n, uint32_t v, Stats &st) {
        launch_fill_u32(p, n, v, stream_);
        st.launches++;
    }

    static constexpr uint32_t kCompGrid = 256, kLdsGrid = 512, kLaneGrid = 8192, kVerifyGrid = 1024;
    hipStream_t stream_;
    uint32_t Np_ = 0, Nc_ = 0, Ng_ = 0, N_ = 0, P_ = 0, depth_ = 0, ncol_ = 0, nplanes_ = 0;
    bool has_pins_ = false;
    float rmax_ = 0.0f, s0_ = 0.0f;
    uint32_t clean_ = 0;
    std::vector<uint32_t> layer_off_;
    std::vector<uint32_t> static_poly_;
    DevBuf<float2> pos_, prev_, acc0_, centers_;
    DevBuf<Link12> links_;
    DevBuf<uint32_t> pinmask_;
    DevBuf<float> crad_;
    DevBuf<uint2> ptab_;
    DevBuf<uint8_t> gflags_;
    DevBuf<int4> colhdr_;
    DevBuf<float4> colgeo_, planes_;
    // circle schedule workspace
    DevBuf<uint8_t> cg_arena_;
    Workspace ws_;
    DevBuf<uint32_t> cc_cand_;
    DevBuf<CompCircle> cg_comp_;  // (from the first component that is replayed in memory on)
    DevBuf<float2> cg_traj_;
    // by slot of the last sweep: the circles (by number after an upload), their needs
    DevBuf<uint32_t> cg_order_;
    DevBuf<float> cg_need_;
    uint64_t cand_cap_ = 0;  // list entries there is room for
    ScanTemp scan_tmp_;
    // page-locked: the last verdict's words and its number
    uint32_t *host_ctl_ = nullptr, verdict_ = 0;
    // the counters alternate between sweeps; those of the next one are zeroed ahead
    uint32_t turn_ = 0;
    bool zeroed_[2] = {false, false};
};

Engine *make_global_engine(hipStream_t stream) { return new GlobalEngine(stream); }

}  // namespace bd
