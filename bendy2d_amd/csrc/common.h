// common.h -- records and arithmetic shared by the host runtime and every
// engine of the MI355X bendy2d solver step.
//
// The arithmetic helpers restate the reference's f32 expressions operation for
// operation (Rust evaluates left to right and never contracts a*b+c into an
// FMA); every translation unit that includes this file is compiled with
// -ffp-contract=off and without fast-math, and HIP's default correctly
// rounded sqrtf and division are kept.
#pragma once

#include <cstdint>
#include <cstddef>

#if defined(__HIPCC__)
#include <hip/hip_runtime.h>
#define BD_HD __host__ __device__ __forceinline__
#else
#define BD_HD inline
#endif

namespace bd {

struct V2 { float x, y; };

// Device link record, 12 bytes, sorted by dependency layer.
//   a: bits 0-29 point index, bit 30 = circle link (r^2-weighted law),
//      bit 31 = end a pinned.
//   b: bits 0-29 point index, bit 31 = end b pinned.
struct Link12 { uint32_t a, b; float t; };

constexpr uint32_t kIndexMask = 0x3fffffffu;
constexpr uint32_t kCircleLinkBit = 0x40000000u;
constexpr uint32_t kPinBit = 0x80000000u;
constexpr uint64_t kMaxPoints = (1ull << 30) - 1;

// n = sqrt(q) and the unit vector (dx / n, dy / n), each correctly rounded.
//
// The compiler's correctly rounded square root and two divisions are about 40
// vector instructions, three of them at a quarter of the rate, and the link
// layers are bound by issuing them.  On the device one reciprocal square root
// estimate serves all three (Markstein, IBM J. Res. Dev. 34, 1990): a coupled
// Newton step gives the root and its reciprocal y, the exact residual of the
// root rounds it correctly, a Newton step against the rounded root gives its
// reciprocal r, and each quotient is a product corrected by its exact residual.
// One ulp added to y in that step makes r come out right for the divisor whose
// significand is all ones, the one divisor such a quotient otherwise misses.
// Checked for an estimate up to 2 ulps off: every q in [1, 4) (so every
// significand and exponent parity) for n and r, and for every n that arises the
// dividends whose quotients lie nearest to the midpoint of two floats (1.6e9
// quotients, none wrong; all others are further from a midpoint than the error
// before the last rounding).  The range below keeps every intermediate normal;
// outside it, and for q of zero, infinity or NaN, the plain operations run.
// Dividends of zero are in the range, with their sign.
// Alone it took the 32 x 32 cloth from 301 to 293 us a frame and the 1024 x 1024
// cloth from 0.576 to 0.515 ms an update.
#if defined(__HIPCC__)
// The device form alone; false where its range does not hold (the results are
// then meaningless).
__device__ __forceinline__ bool length_and_unit_fast(float dx, float dy, float q, float &n, float &nx, float &ny) {
    const float y0 = __builtin_amdgcn_rsqf(q);
    const float g0 = q * y0, h = 0.5f * y0;
    const float t = __builtin_fmaf(-h, g0, 0.5f);
    const float y = __builtin_fmaf(y0, t, y0), g = __builtin_fmaf(g0, t, g0);
    const float d = __builtin_fmaf(-g, g, q);
    n = __builtin_fmaf(0.5f * d, y, g);
    const float e = __builtin_fmaf(-n, y, 1.0f);
    const float r = __builtin_fmaf(e, __uint_as_float(__float_as_uint(y) + 1u), y);
    const float ux = dx * r, uy = dy * r;
    const float rx = __builtin_fmaf(-ux, n, dx), ry = __builtin_fmaf(-uy, n, dy);
    // the corrected quotient of -0 is +0: the sign is the dividend's
    nx = __builtin_copysignf(__builtin_fmaf(rx, r, ux), dx);
    ny = __builtin_copysignf(__builtin_fmaf(ry, r, uy), dy);
    // |dx|, |dy| zero or at least 2^-55, q finite and at least 2^-56, in one
    // comparison: the bits without the sign, less one for the dividends (a zero
    // wraps to the top), plus one exponent for q (infinity and NaN wrap to the
    // bottom)
    const uint32_t bx = (__float_as_uint(dx) << 1) - 1u, by = (__float_as_uint(dy) << 1) - 1u;
    const uint32_t bq = (__float_as_uint(q) << 1) + 0x01000000u;
    return min(min(bx, by), bq) >= 0x47ffffffu;
}

// Barrier for a workgroup whose wavefronts exchange data through LDS alone:
// outstanding global loads (records on their way for the next layer) stay in
// flight across it, where __syncthreads waits for them.
__device__ __forceinline__ void lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}
#endif

BD_HD void length_and_unit(float dx, float dy, float q, float &n, float &nx, float &ny) {
#if defined(__HIP_DEVICE_COMPILE__)
    // the plain operations in a branch of their own, taken only by a wavefront
    // that has such a lane: a branch on each lane's range around both forms
    // cost more than the arithmetic it saved
    const bool fine = length_and_unit_fast(dx, dy, q, n, nx, ny);
    if (__builtin_expect(__ballot(!fine) != 0ull, 0)) {
        if (!fine) {
            n = sqrtf(q);
            nx = dx / n;
            ny = dy / n;
        }
    }
#else
    n = sqrtf(q);
    nx = dx / n;
    ny = dy / n;
#endif
}

// ParticleLink::solve (src/link.rs:18-27) with the pin extension: a pinned
// end does not move and the free end takes the whole correction; two free
// ends use the reference's 0.5 split.
BD_HD void solve_particle_link(float &ax, float &ay, float &bx, float &by, float t, bool pin_a, bool pin_b) {
    float dx = ax - bx, dy = ay - by, dist, nx, ny;
    length_and_unit(dx, dy, dx * dx + dy * dy, dist, nx, ny);
    float e = dist - t;
    if (!pin_a && !pin_b) {
        float cx = (nx * e) * 0.5f, cy = (ny * e) * 0.5f;
        ax = ax - cx; ay = ay - cy;
        bx = bx + cx; by = by + cy;
    } else if (!pin_a) {
        ax = ax - nx * e; ay = ay - ny * e;
    } else if (!pin_b) {
        bx = bx + nx * e; by = by + ny * e;
    }
}

// CircleLink::solve (src/link.rs:36-48).
BD_HD void solve_circle_link(float &ax, float &ay, float &bx, float &by, float t, float ra, float rb) {
    float dx = ax - bx, dy = ay - by, dist, nx, ny;
    length_and_unit(dx, dy, dx * dx + dy * dy, dist, nx, ny);
    float ra2 = ra * ra, rb2 = rb * rb;
    float scale = 1.0f / (ra2 + rb2);
    float e = dist - t;
    ax = ax - ((nx * e) * scale) * rb2; ay = ay - ((ny * e) * scale) * rb2;
    bx = bx + ((nx * e) * scale) * ra2; by = by + ((ny * e) * scale) * ra2;
}

// Circle::solve_circle (src/circle.rs:32-45).  Returns true when the pair
// overlapped; push_i / push_j receive the length of each circle's move.
BD_HD bool solve_circle_pair(float &ix, float &iy, float &jx, float &jy, float ri, float rj,
                             float &push_i, float &push_j) {
    float dx = ix - jx, dy = iy - jy;
    float q = dx * dx + dy * dy;
    float rs = ri + rj;
    if (q < rs * rs) {
        float n, nx, ny;
        length_and_unit(dx, dy, q, n, nx, ny);
        float ov = rs - n;
        float ri2 = ri * ri, rj2 = rj * rj;
        float scale = 1.0f / (ri2 + rj2);
        ix = ix + ((nx * scale) * ov) * rj2; iy = iy + ((ny * scale) * ov) * rj2;
        jx = jx - ((nx * scale) * ov) * ri2; jy = jy - ((ny * scale) * ov) * ri2;
        push_i = fabsf((scale * ov) * rj2);
        push_j = fabsf((scale * ov) * ri2);
        return true;
    }
    return false;
}

// Largest distance from a sweep's start position (sx, sy) reached so far,
// after a push moved the circle to (px, py).  The distance is rounded up by a
// relative 2^-20, far above float rounding, so the bound never falls below the
// truth.  A circle pushed back and forth keeps a small excursion where the sum
// of its pushes would grow without end.  A non-finite position leaves the
// bound unchanged: such a circle takes part in no pair.
BD_HD float excursion(float cur, float px, float py, float sx, float sy) {
    float dx = px - sx, dy = py - sy;
    float d = sqrtf(dx * dx + dy * dy) * (1.0f + 0x1p-20f);
    return fmaxf(cur, d);
}

// Particle::update (src/particle.rs:20-25): pos + vel + acc*dt*dt, acc = g
// (plus any initial acc on the first substep).
BD_HD void verlet(float &px, float &py, float &qx, float &qy, float ax, float ay, float dt) {
    float vx = px - qx, vy = py - qy;
    qx = px; qy = py;
    px = (px + vx) + ((ax * dt) * dt);
    py = (py + vy) + ((ay * dt) * dt);
}

// Particle::solve_bounds (src/particle.rs:27-46): lo/hi are bounds.pos and
// bounds.pos + bounds.size, per axis, if / else-if.
BD_HD void bounds_axis(float &p, float &q, float lo, float hi) {
    if (p < lo) {
        float v = q - p; q = lo - v; p = lo;
    } else if (p > hi) {
        float v = q - p; q = hi - v; p = hi;
    }
}

// Circle::solve_bounds (src/circle.rs:11-30): limits shifted by the radius,
// lo + r and (lo + size) - r.
BD_HD void circle_bounds_axis(float &p, float &q, float lo, float hi, float r) {
    float l = lo + r, h = hi - r;
    if (p < l) {
        float v = q - p; q = l - v; p = l;
    } else if (p > h) {
        float v = q - p; q = h - v; p = h;
    }
}

// EXT4 static circle collider: a body of radius r is pushed out of a fixed
// circle (cx, cy, R) by the whole overlap.  A body exactly at the centre is
// left in place.
BD_HD void static_circle(float &px, float &py, float r, float cx, float cy, float R) {
    float dx = px - cx, dy = py - cy;
    float q = dx * dx + dy * dy;
    float rs = r + R;
    if (q < rs * rs) {
        float d = sqrtf(q);
        if (d > 0.0f) {
            float nx = dx / d, ny = dy / d, ov = rs - d;
            px = px + nx * ov; py = py + ny * ov;
        }
    }
}

// Cell hashing for the circle-pair broadphase.
BD_HD uint32_t cell_hash(int32_t cx, int32_t cy) {
    return ((uint32_t)cx * 73856093u) ^ ((uint32_t)cy * 19349663u);
}

}  // namespace bd
