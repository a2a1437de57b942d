// bodies.h -- the per-body phase shared by the engines: EXT4 static
// colliders, then bounds (src/solver.rs:155-165), then Verlet
// (src/solver.rs:118-128); and the edge-against-point push of soft polygons.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "common.h"

namespace bd {

// A value every lane of the workgroup holds alike, moved to a scalar register
// (the compiler cannot see that values read back from LDS are uniform).
__device__ __forceinline__ uint32_t uni(uint32_t v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ __forceinline__ float uni(float v) { return __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(v))); }

// A uniform pointer into global memory, typed as such, with its base read
// from the first lane: loads through it take a 32-bit offset beside a scalar
// base instead of a 64-bit flat address.
#define BD_GLOBAL __attribute__((address_space(1)))
template <typename T>
__device__ __forceinline__ BD_GLOBAL T *to_global(T *p) {
    const uint64_t a = (uint64_t)p;
    // each half through uni(), which returns it unsigned: the builtin's int,
    // widened directly, would carry bit 31 of the low half into the high one
    const uint64_t lo = uni((uint32_t)a);
    const uint64_t hi = uni((uint32_t)(a >> 32));
    return (BD_GLOBAL T *)((hi << 32) | lo);
}

// The same for read-only data read at uniform indices: typed as constant, it
// is read by scalar loads into scalar registers.
#define BD_CONST __attribute__((address_space(4)))
template <typename T>
__device__ __forceinline__ BD_CONST const T *to_const(const T *p) {
    const uint64_t a = (uint64_t)p;
    const uint64_t lo = uni((uint32_t)a);
    const uint64_t hi = uni((uint32_t)(a >> 32));
    return (BD_CONST const T *)((hi << 32) | lo);
}

struct BodyParams {
    float dt, gex, gey, gx, gy;
    float lox, loy, hix, hiy;
    uint32_t N, Np, Nc;
    uint32_t first_acc;
    uint32_t ncol;
};

// A convex polygon's planes (nx, ny, c) against a body of radius r.  The push
// uses the plane of largest signed distance, and only when that distance is
// below r; a plane at r or beyond already rules the push out, so the scan stops
// once it has for every lane (a NaN distance, first or later, never pushes
// either way).  plane(e): the e-th plane, e uniform; own(e): the same at a
// lane's own e.
template <typename F, typename G>
__device__ __forceinline__ void static_planes(float2 &p, float r, uint32_t n, F &&plane, G &&own) {
    float smax = 0.0f;
    uint32_t arg = 0xffffffffu;
    bool out = n == 0u;
#pragma unroll 1
    for (uint32_t e = 0; e < n; e++) {
        const auto w = plane(e);
        const float sd = (w.x * p.x + w.y * p.y) - w.z;
        out = out || sd >= r;
        if (arg == 0xffffffffu || sd > smax) { smax = sd; arg = e; }
        if (__ballot(!out) == 0ull) return;
    }
    if (!out && smax < r) {
        const auto w = own(arg);
        const float push = r - smax;
        p.x = p.x + w.x * push; p.y = p.y + w.y * push;
    }
}

typedef int I4 __attribute__((ext_vector_type(4)));
typedef float F4 __attribute__((ext_vector_type(4)));

// Static colliders in insertion order against a body of radius r (0 for
// particles and polygon points).  hdr: (kind, plane offset, planes, -);
// geo: circle (cx, cy, R, -); pl: polygon edge planes (nx, ny, c, -).  The
// records are uniform and come through the scalar cache into scalar registers
// (262,144 circles over 68 colliders: staged in LDS, two reads a collider for
// every wavefront, 19.9 us; from the scalar cache one by one, two dependent loads
// each, 21.6; four at a time 14.2.  48 flying bodies: a pass 5 % shorter).
// kU: how many at a time.  The tiled pass takes one: four held 87 scalar registers
// instead of 63 there, two of its workgroups no longer shared a CU, and a pass over
// 1,048,576 points took 18.2 us instead of 15.2.
template <uint32_t kU = 4u>
__device__ __forceinline__ void static_colliders(float2 &p, float r, uint32_t ncol, const void *hdr_, const void *geo_,
                                                 const void *pl_) {
    BD_CONST const I4 *const hdr = to_const((const I4 *)hdr_);
    BD_CONST const F4 *const geo = to_const((const F4 *)geo_);
    BD_CONST const F4 *const pl = to_const((const F4 *)pl_);
    BD_GLOBAL const F4 *const gpl = to_global((const F4 *)pl_);
    auto one = [&](const I4 &h, const F4 &g) {
        if (h.x == 0)
            static_circle(p.x, p.y, r, g.x, g.y, g.z);
        else
            static_planes(p, r, (uint32_t)h.z, [&](uint32_t e) -> F4 { return pl[h.y + e]; },
                          [&](uint32_t e) -> F4 { return gpl[h.y + e]; });
    };
    uint32_t k = 0;
#pragma unroll 1
    for (; kU > 1u && k + kU <= ncol; k += kU) {
        I4 h[kU];
        F4 g[kU];
#pragma unroll
        for (uint32_t u = 0; u < kU; u++) { h[u] = hdr[k + u]; g[u] = geo[k + u]; }
#pragma unroll
        for (uint32_t u = 0; u < kU; u++) one(h[u], g[u]);
    }
#pragma unroll 1
    for (; k < ncol; k++) {
        const I4 h = hdr[k];
        const F4 g = geo[k];
        one(h, g);
    }
}

// A particle (not pinned): colliders, bounds, Verlet with acc = 0 + g.
__device__ __forceinline__ void particle_body(float2 &p, float2 &q, const BodyParams &P, const int4 *hdr,
                                              const float4 *geo, const float4 *pl) {
    static_colliders<1u>(p, 0.0f, P.ncol, hdr, geo, pl);
    bounds_axis(p.x, q.x, P.lox, P.hix);
    bounds_axis(p.y, q.y, P.loy, P.hiy);
    verlet(p.x, p.y, q.x, q.y, P.gex, P.gey, P.dt);
}

// ---- soft polygons ----------------------------------------------------------

// common::line_intersection (src/common.rs:4-26)
__device__ __forceinline__ bool line_intersection(float2 p1, float2 p2, float2 p3, float2 p4, float2 &out) {
    float s1x = p2.x - p1.x, s1y = p2.y - p1.y;
    float s2x = p4.x - p3.x, s2y = p4.y - p3.y;
    float den = (-s2x) * s1y + s1x * s2y;
    float s = ((-s1y) * (p1.x - p3.x) + s1x * (p1.y - p3.y)) / den;
    float t = (s2x * (p1.y - p3.y) - s2y * (p1.x - p3.x)) / den;
    if (s >= 0.0f && s <= 1.0f && t >= 0.0f && t <= 1.0f) {
        out = make_float2(p1.x + (t * s1x), p1.y + (t * s1y));
        return true;
    }
    return false;
}

__device__ __forceinline__ float2 f2sub(float2 a, float2 b) { return make_float2(a.x - b.x, a.y - b.y); }
__device__ __forceinline__ float2 f2add(float2 a, float2 b) { return make_float2(a.x + b.x, a.y + b.y); }
__device__ __forceinline__ float2 f2mul(float2 a, float s) { return make_float2(a.x * s, a.y * s); }
__device__ __forceinline__ float f2dot(float2 a, float2 b) { return a.x * b.x + a.y * b.y; }
__device__ __forceinline__ float2 f2normalize(float2 a) {
    float n = sqrtf(f2dot(a, a));
    return make_float2(a.x / n, a.y / n);
}
__device__ __forceinline__ float f2mag(float2 a) { return sqrtf(f2dot(a, a)); }

// Polygon::resolve_line_intersection (src/polygon.rs:164-216)
__device__ __forceinline__ bool resolve_line(float2 self_center, float2 pa, float2 pb, float2 op, float2 other_center,
                             float2 &na, float2 &nb, float2 &no) {
    float2 inter;
    if (!line_intersection(pa, pb, op, other_center, inter)) return false;
    float2 nl = f2normalize(f2sub(pb, pa));                                    // :175
    float2 cp = f2mul(nl, f2dot(nl, f2sub(self_center, inter)) / f2dot(nl, nl));  // :177-179
    float2 nin = f2normalize(f2sub(self_center, f2add(inter, cp)));           // :181
    float da = f2mag(f2sub(inter, pa));                                       // :183
    float db = f2mag(f2sub(inter, pb));                                       // :184
    float dab = da + db;                                                      // :186
    float ia = db / dab, ib = da / dab;                                       // :188-189
    float2 diff = f2sub(inter, op);                                           // :191
    float2 ion = f2mul(nin, f2dot(nin, diff) / f2dot(nin, nin));             // :193-194
    float2 third = make_float2(ion.x / 3.0f, ion.y / 3.0f);                   // :196
    float2 line = f2mul(third, 2.0f);                                         // :198
    float2 da_v = f2mul(line, ia), db_v = f2mul(line, ib);                    // :200-201
    float2 ra = f2sub(pa, da_v), rb = f2sub(pb, db_v);                        // :203-204
    float2 ray_end = f2sub(op, f2mul(nin, 10000.0f));                         // :208
    float2 np;
    if (!line_intersection(pa, pb, op, ray_end, np)) return false;            // :206-213
    na = ra; nb = rb; no = np;
    return true;
}

// Polygon pair loop (src/solver.rs:178-187 -> Polygon::solve_polygon
// src/polygon.rs:142-162) by one workgroup.  Edges run in order; within an edge the
// other polygon's points are independent (each reads only the edge's ends as they
// were before it, its own position and the two centres), and the hit with the
// highest point index writes the ends ("last hit wins").  An edge that no point
// hits changes nothing, so a step tests as many edges as the lanes hold, against
// the positions as they are, and carries out the first that is hit; the edges
// behind it are tested again.  (Edge by edge, 5 polygons of 12 points took 240
// steps of two barriers, nearly all for nothing: an update 176 us, 46 now.)
// P holds positions as 64-bit words (in LDS or memory); tab[p].x, .y are a
// polygon's first point and point count; slot is 3 words of LDS.
template <int WG, typename WP, typename TAB>
__device__ __forceinline__ void poly_pair_loop(WP P, const TAB *tab, const float2 *ctr, uint32_t npoly,
                                               uint32_t *slot) {
    const uint32_t tid = threadIdx.x, lane = tid & 63u;
    auto get = [&](uint32_t i) {
        const uint64_t b = P[i];
        return make_float2(__uint_as_float((uint32_t)b), __uint_as_float((uint32_t)(b >> 32)));
    };
    auto put = [&](uint32_t i, float2 v) {
        P[i] = (uint64_t)__float_as_uint(v.x) | ((uint64_t)__float_as_uint(v.y) << 32);
    };
    // up to 64 polygons' table in registers, one to a lane
    const bool held = npoly <= 64u;
    const uint32_t hp = min(lane, npoly - 1u);
    const uint32_t h_at = tab[hp].x, h_n = tab[hp].y;
    const float2 h_c = ctr[hp];
    struct Poly { uint32_t at, n; float2 c; };
    auto poly = [&](uint32_t q) {
        Poly r;
        if (held) {
            r.at = __builtin_amdgcn_readlane(h_at, q);
            r.n = __builtin_amdgcn_readlane(h_n, q);
            r.c.x = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(h_c.x), q));
            r.c.y = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(h_c.y), q));
        } else {
            r.at = tab[q].x;
            r.n = tab[q].y;
            r.c = ctr[q];
        }
        return r;
    };
    if (tid < 3u) slot[tid] = 0u;
    __syncthreads();
    uint32_t turn = 0;  // slots rotate: the one after next is cleared behind a barrier
    auto winner = [&](uint32_t key) {
        uint32_t *const now = &slot[turn % 3u];
        if (key) atomicMax(now, key);
        __syncthreads();
        const uint32_t best = *now;
        if (tid == 0u) slot[(turn + 2u) % 3u] = 0u;
        turn++;
        return best;
    };
    for (uint32_t i = 0; i < npoly; i++)
        for (uint32_t j = i + 1; j < npoly; j++)
            for (uint32_t dir = 0; dir < 2u; dir++) {
                const Poly s = poly(dir ? j : i), o = poly(dir ? i : j);
                const uint32_t E = s.n, K = o.n;
                if (K == 0u) continue;
                if (K <= (uint32_t)WG && E < 65536u) {
                    const uint32_t per = (uint32_t)WG / K, le = tid / K, k = tid - le * K;
                    for (uint32_t e0 = 0; e0 < E;) {
                        const uint32_t e = e0 + le, ia = s.at + e, ib = s.at + (e + 1u == E ? 0u : e + 1u);
                        float2 a2, b2, o2;
                        const bool hit = le < per && e < E &&
                                         resolve_line(s.c, get(ia), get(ib), get(o.at + k), o.c, a2, b2, o2);
                        uint32_t first;  // the first edge that is hit
                        bool mine, last;
                        if constexpr (WG == 64) {
                            const uint64_t hits = __ballot(hit);
                            if (hits == 0ull) { e0 += per; continue; }
                            first = (uint32_t)__builtin_amdgcn_readlane(e, __ffsll((unsigned long long)hits) - 1);
                            mine = hit && e == first;
                            last = lane == 63u - (uint32_t)__clzll((long long)__ballot(mine));
                        } else {
                            const uint32_t key = hit ? (E - e) << 16 | (k + 1u) : 0u;
                            const uint32_t best = winner(key);
                            if (best == 0u) { e0 += per; continue; }
                            first = E - (best >> 16);
                            mine = hit && e == first;
                            last = key == best;
                        }
                        if (mine) put(o.at + k, o2);
                        if (last) { put(ia, a2); put(ib, b2); }
                        __syncthreads();
                        e0 = first + 1u;
                    }
                    continue;
                }
                for (uint32_t e = 0; e < E; e++) {
                    const uint32_t ia = s.at + e, ib = s.at + (e + 1u == E ? 0u : e + 1u);
                    const float2 pa = get(ia), pb = get(ib);
                    uint32_t mine = 0;
                    float2 na = pa, nb = pb;
                    for (uint32_t k = tid; k < K; k += WG) {
                        float2 a2, b2, o2;
                        if (resolve_line(s.c, pa, pb, get(o.at + k), o.c, a2, b2, o2)) {
                            put(o.at + k, o2);
                            na = a2; nb = b2; mine = k + 1u;
                        }
                    }
                    const uint32_t best = winner(mine);
                    if (mine && mine == best) { put(ia, na); put(ib, nb); }
                    __syncthreads();
                }
            }
}

}  // namespace bd
