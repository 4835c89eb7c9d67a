// vrt_device.h — device-side pieces of the per-pixel path of
// src/fshader.glsl (castRay :59-129 and main :131-190) for gfx950.
//
// Every float operation below is one IEEE binary32 operation in the order
// the shader states it (the library is built with -ffp-contract=off, correctly
// rounded division and square root, denormals kept), so the hit index, face,
// shadow bits and step counts equal a literal scalar restatement of the
// shader.  The code is arranged for wave64 SIMT: one ray per lane, the axis
// choice as selects, the voxel index kept incrementally, and the shadow rays
// of a pixel cast one after another by the same lane.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <type_traits>

#include "vrt_internal.h"

namespace vrt {
namespace dev {

// GLSL int(float): truncation toward zero; out-of-range saturates, NaN -> 0.
// That is exactly what v_cvt_i32_f32 does, so it is issued directly (C++'s
// (int) of an out-of-range float is undefined and the guards would branch).
__device__ __forceinline__ int32_t f2i(float v) {
    int32_t r;
    asm("v_cvt_i32_f32 %0, %1" : "=v"(r) : "v"(v));
    return r;
}

// Largest integer not above v.
__device__ __forceinline__ int32_t floor_i(float v) {
    int32_t r;
    asm("v_cvt_flr_i32_f32 %0, %1" : "=v"(r) : "v"(v));
    return r;
}

// int(sign(v)) (src/fshader.glsl:71); sign(NaN) = 0.
__device__ __forceinline__ int32_t isign(float v) { return v > 0.0f ? 1 : (v < 0.0f ? -1 : 0); }

__device__ __forceinline__ float max0(float v) { return v > 0.0f ? v : 0.0f; }

// a / d rounded to nearest, given y = RN(1/d) (one IEEE division per ray) and
// dok = (2^-60 <= |d| <= 2^60).  Markstein's correction: q0 = RN(a*y),
// r = a - q0*d (exact, by FMA), q = RN(q0 + r*y) = RN(a/d).  With a and d
// in [2^-60, 2^60] every intermediate stays in the normal range, so each step
// is the same computation on the significands scaled by a power of two; the
// library's selftest checks all 2^23 x 2^23 significand pairs against IEEE
// division.  Any other input (zero, subnormal, huge, infinite, NaN) takes the
// IEEE division itself.
__device__ __forceinline__ float div_by(float a, float d, float y, bool dok) {
    const uint32_t ua = __float_as_uint(a) & 0x7fffffffu;
    const bool ok = dok & ((ua - 0x21800000u) <= (0x5d800000u - 0x21800000u));
    const float q0 = a * y;
    float q = __builtin_fmaf(__builtin_fmaf(-q0, d, a), y, q0);
    if (__builtin_expect(!ok, 0)) q = a / d;
    return q;
}

// The three quotients (cell boundary - position) / d of one intersect update
// share one range test and one fallback branch.  With |s| < 2^31 the cell
// int(s) does not saturate and every numerator is below 2^33 in magnitude, so
// only the lower end of the fast path's range is tested.  Larger numerators
// come only from a saturated cell (|s| >= 2^31 or infinite), which lies outside
// every grid: the ray's next step then leaves the grid and the quotients are
// never read.  A NaN numerator gives NaN on both paths.
__device__ __forceinline__ void div3_by(float ax, float ay, float az, float dx, float dy, float dz, float rx,
                                        float ry, float rz, bool dok, float& qx, float& qy, float& qz) {
    const float lo = fminf(fminf(fabsf(ax), fabsf(ay)), fabsf(az));
    const bool ok = dok & (lo >= 0x1p-60f);
    const float q0x = ax * rx, q0y = ay * ry, q0z = az * rz;
    qx = __builtin_fmaf(__builtin_fmaf(-q0x, dx, ax), rx, q0x);
    qy = __builtin_fmaf(__builtin_fmaf(-q0y, dy, ay), ry, q0y);
    qz = __builtin_fmaf(__builtin_fmaf(-q0z, dz, az), rz, q0z);
    if (__builtin_expect(!ok, 0)) {
        qx = ax / dx;
        qy = ay / dy;
        qz = az / dz;
    }
}

__device__ __forceinline__ bool div_range_ok(float d) {
    const uint32_t ud = __float_as_uint(d) & 0x7fffffffu;
    return (ud - 0x21800000u) <= (0x5d800000u - 0x21800000u);
}

// a / d for a = +0 or an integer in [1, 2^25] and d in [1, 2^24] with
// y = RN(1/d): the correction of div_by with every quantity normal (or +0),
// so no range test is needed.
__device__ __forceinline__ float div_small_int(float a, float d, float y) {
    const float q0 = a * y;
    return __builtin_fmaf(__builtin_fmaf(-q0, d, a), y, q0);
}

// RN(1/d): v_rcp_f32 (within one ulp) refined by one Newton step with FMAs,
// e = RN(1 - d*y0), y = RN(y0 + y0*e).  For |d| in [2^-60, 2^60] this equals
// IEEE division 1/d for every input: the library's reciprocal selftest
// compares the two for all 2^32 bit patterns.  rcp_fast is that form alone,
// for callers that test the range themselves; rcp_rn gives any other input
// the division itself.
__device__ __forceinline__ float rcp_fast(float d) {
    const float y0 = __builtin_amdgcn_rcpf(d);
    return __builtin_fmaf(__builtin_fmaf(-d, y0, 1.0f), y0, y0);
}
__device__ __forceinline__ float rcp_rn(float d) {
    float y = rcp_fast(d);
    if (__builtin_expect(!div_range_ok(d), 0)) y = 1.0f / d;
    return y;
}

// dot, length, normalize in GLM 1.0.0's order (func_geometric.inl:48-54,88;
// func_exponential.inl:136-139).
__device__ __forceinline__ float dot3(float ax, float ay, float az, float bx, float by, float bz) {
    float x = ax * bx;
    float y = ay * by;
    float z = az * bz;
    return (x + y) + z;
}

__device__ __forceinline__ uint8_t unorm8(float c) {
    float k = c > 0.0f ? (c < 1.0f ? c : 1.0f) : 0.0f;
    return (uint8_t)(int32_t)(k * 255.0f + 0.5f);
}

// Result of one castRay.
struct Hit {
    int64_t index;   // word index of the hit voxel in the padded render copy, or -1
    float pos[3];    // hitPos (valid on a hit)
    int32_t axis;    // axis of the step into the hit voxel (-1 on a miss)
    int32_t step;    // step on that axis
    int32_t word;    // the hit voxel's word
    uint32_t iters;  // loop iterations (stepCount increments)
};

// Clamps a cell coordinate to [-2, n + 1] (one v_med3_i32).  A walk indexes
// the padded copy only through this: a cell two or more outside the grid
// cannot enter it on the next step, and from -2 or n + 1 that step lands on a
// guard cell (kGuard = 3 of them on each side) whatever its direction, as it
// lands outside the grid from the true cell.
__device__ __forceinline__ int32_t clamp_cell(int32_t v, uint32_t n) {
    int32_t r;
    asm("v_med3_i32 %0, %1, -2, %2" : "=v"(r) : "v"(v), "s"((int32_t)n + 1));
    return r;
}

// Index arithmetic on the padded render copy, three forms: IdxB keeps the
// byte offset of the word (4 x index) in 32 bits when the copy is at most
// 2^32 bytes and 4 SX, 4 SXY < 2^23, so the gather adds it to the copy's base
// address in the load itself; Idx32 keeps the word index in 32 bits with
// signed 24-bit multiplies when the copy has at most 2^32 words and SX, SXY <
// 2^23; Idx64 otherwise.  make() takes clamped cells (clamp_cell), so every
// offset is non-negative and inside the copy, and y, z fit 24 bits.
// ref_index() turns the word index of an in-grid cell back into the
// reference's x + X*y + X*Y*z (src/fshader.glsl:36-39).
template <typename U>
__device__ __forceinline__ int64_t ref_index_of(const GridDesc& g, U L) {
    const U z = L / (U)g.SXY;
    const U r = L - z * (U)g.SXY;
    const U y = r / (U)g.SX;
    const U x = r - y * (U)g.SX;
    return (int64_t)x + (int64_t)g.X * (int64_t)y + (int64_t)g.XY * (int64_t)z;
}
struct IdxB {
    using T = uint32_t;  // byte offset
    __device__ __forceinline__ static T make(const GridDesc& g, int32_t x, int32_t y, int32_t z) {
        // a shift-add and two 24-bit multiply-adds
        uint32_t t = ((uint32_t)x << 2) + (uint32_t)g.origin * 4u;
        asm("v_mad_i32_i24 %0, %1, %2, %3" : "=v"(t) : "v"(y), "s"((int32_t)(g.SX * 4)), "v"(t));
        asm("v_mad_i32_i24 %0, %1, %2, %3" : "=v"(t) : "v"(z), "s"((int32_t)(g.SXY * 4)), "v"(t));
        return t;
    }
    // stride of a step on an axis
    __device__ __forceinline__ static T stride(const GridDesc& g, int32_t step, int axis) {
        return (uint32_t)step * (axis == 0 ? 4u : (axis == 1 ? g.SX * 4u : (uint32_t)g.SXY * 4u));
    }
    __device__ __forceinline__ static int32_t load(const int32_t* vox, T i) {
        return *(const int32_t*)((const char*)vox + i);
    }
    // i + c * stride, both factors within signed 24 bits
    __device__ __forceinline__ static T add(T i, int32_t c, int32_t stride) {
        asm("v_mad_i32_i24 %0, %1, %2, %3" : "=v"(i) : "v"(c), "v"(stride), "v"(i));
        return i;
    }
    __device__ __forceinline__ static int64_t word(T i) { return (int64_t)(i >> 2); }
    __device__ __forceinline__ static int64_t ref_index(const GridDesc& g, int64_t w) {
        return ref_index_of<uint32_t>(g, (uint32_t)w - (uint32_t)g.origin);
    }
};
struct Idx32 {
    using T = uint32_t;
    __device__ __forceinline__ static T make(const GridDesc& g, int32_t x, int32_t y, int32_t z) {
        uint32_t t = (uint32_t)x + (uint32_t)g.origin;
        asm("v_mad_i32_i24 %0, %1, %2, %3" : "=v"(t) : "v"(y), "s"((int32_t)g.SX), "v"(t));
        asm("v_mad_i32_i24 %0, %1, %2, %3" : "=v"(t) : "v"(z), "s"((int32_t)g.SXY), "v"(t));
        return t;
    }
    __device__ __forceinline__ static T stride(const GridDesc& g, int32_t step, int axis) {
        return (uint32_t)step * (axis == 0 ? 1u : (axis == 1 ? g.SX : (uint32_t)g.SXY));
    }
    __device__ __forceinline__ static int32_t load(const int32_t* vox, T i) { return vox[i]; }
    // i + c * stride, both factors within signed 24 bits
    __device__ __forceinline__ static T add(T i, int32_t c, int32_t stride) {
        asm("v_mad_i32_i24 %0, %1, %2, %3" : "=v"(i) : "v"(c), "v"(stride), "v"(i));
        return i;
    }
    __device__ __forceinline__ static int64_t word(T i) { return (int64_t)i; }
    __device__ __forceinline__ static int64_t ref_index(const GridDesc& g, int64_t w) {
        return ref_index_of<uint32_t>(g, (uint32_t)w - (uint32_t)g.origin);
    }
};
struct Idx64 {
    using T = uint64_t;
    __device__ __forceinline__ static T make(const GridDesc& g, int32_t x, int32_t y, int32_t z) {
        return g.origin + (uint64_t)(int64_t)x + (uint64_t)g.SX * (uint64_t)(int64_t)y +
               g.SXY * (uint64_t)(int64_t)z;
    }
    __device__ __forceinline__ static T stride(const GridDesc& g, int32_t step, int axis) {
        return (uint64_t)(int64_t)step * (axis == 0 ? 1u : (axis == 1 ? (uint64_t)g.SX : g.SXY));
    }
    __device__ __forceinline__ static int32_t load(const int32_t* vox, T i) { return vox[i]; }
    __device__ __forceinline__ static int64_t word(T i) { return (int64_t)i; }
    __device__ __forceinline__ static int64_t ref_index(const GridDesc& g, int64_t w) {
        return ref_index_of<uint64_t>(g, (uint64_t)w - g.origin);
    }
};

// castRay, src/fshader.glsl:59-129.  `lim` = min(float(dist), float(RENDER_DIST)):
// the loop test `t < dist && t < RENDER_DIST` of :83 is `t < lim` for any t.
// The walk reads the padded render copy and keeps only the word offset of
// the current cell, advanced by one step's stride per iteration; the cell
// coordinates are formed at the start and after each jump (clamp_cell), never
// per step.  A step off the grid (per-axis bounds, :42-45) lands on a guard
// cell, whose NaN jump ends the walk in that iteration with the result and
// iteration count of the reference's exit at :123-125.  The axis choice is
// computed with selects so the wave does not branch.
//
// ytop (shadow rays, and primary rays whose step count nothing shows): an
// upper bound on the y of every solid voxel, or INT32_MAX.  Let dy >= 0.  Every
// cell of a segment has y >= int(start.y), and a jump sets start.y += RN(dy * c)
// with c = the entry intersect plus the jump.  A negative entry intersect either belongs to an axis whose step
// leaves the grid (the walk ends before any jump), or comes from a zero
// direction component, which then makes c infinite or NaN at every jump from
// the first one on.  So after a jump that leaves int(start.y) > ytop with c
// finite and >= 0, every later jump keeps c >= 0, start.y never decreases,
// and no cell the walk can still reach is solid: the ray is a miss.  The loop
// stops there instead of walking on to the grid's edge or its budget; the
// result is the reference's, only the iteration count is smaller.  (A jump
// with c = -inf or NaN leaves int(start.y) at INT32_MIN or 0, where the test
// fires only if the grid has no solid voxel; c = +inf makes `travelled`
// infinite, which ends the walk at the next loop test anyway.)
// kAgain: where `again`, the walk is one that run_walk gave up, whose iterations
// are counted already up to there; h.iters leaves these out.
template <typename IX, bool kAgain>
__device__ __forceinline__ void walk_generic(const GridDesc& g, float sx, float sy, float sz, float dx, float dy,
                                             float dz, float lim, Hit& h, int32_t ytop, bool again) {
    using T = typename IX::T;
    const int32_t cx = f2i(sx), cy = f2i(sy), cz = f2i(sz);
    const int32_t stx = isign(dx), sty = isign(dy), stz = isign(dz);
    const int32_t fx = stx > 0, fy = sty > 0, fz = stz > 0;
    // The six reciprocals (the step sizes 1/|d + 1e-6| of :74-76 and 1/d for
    // the intersect quotients) share one range test: every |value| in
    // [2^-60, 2^60] takes rcp_rn's fast form, anything else (a zero, a
    // subnormal, a huge or infinite component) IEEE division for all six and
    // for the quotients.  A NaN component is NaN on either path.
    const float bx_ = fabsf(dx + 0.000001f), by_ = fabsf(dy + 0.000001f), bz_ = fabsf(dz + 0.000001f);
    const float lo = fminf(fminf(fminf(fabsf(dx), fabsf(dy)), fabsf(dz)), fminf(fminf(bx_, by_), bz_));
    const float hi = fmaxf(fmaxf(fmaxf(fabsf(dx), fabsf(dy)), fabsf(dz)), fmaxf(fmaxf(bx_, by_), bz_));
    const bool dok = (lo >= 0x1p-60f) & (hi <= 0x1p60f);
    float ddx, ddy, ddz, rx, ry, rz;
    if (__builtin_expect(dok, 1)) {
        ddx = rcp_fast(bx_);
        ddy = rcp_fast(by_);
        ddz = rcp_fast(bz_);
        rx = rcp_fast(dx);
        ry = rcp_fast(dy);
        rz = rcp_fast(dz);
    } else {
        ddx = 1.0f / bx_;
        ddy = 1.0f / by_;
        ddz = 1.0f / bz_;
        rx = 1.0f / dx;
        ry = 1.0f / dy;
        rz = 1.0f / dz;
    }
    float ix, iy, iz;
    div3_by((float)(cx + fx) - sx, (float)(cy + fy) - sy, (float)(cz + fz) - sz, dx, dy, dz, rx, ry, rz, dok, ix, iy,
            iz);
    const T sdx = IX::stride(g, stx, 0), sdy = IX::stride(g, sty, 1), sdz = IX::stride(g, stz, 2);
    T idx = IX::make(g, clamp_cell(cx, g.X), clamp_cell(cy, g.Y), clamp_cell(cz, g.Z));
    const int32_t* __restrict__ vox = g.vox;

    float trav = 0.0f;
    uint32_t iters = 0, counted = 0;
    int32_t axis = -1;
    int64_t result = -1;
    while (trav < lim) {
        iters++;
        trav += 1.0f;
        const bool bx = (ix < iy) & (ix < iz);
        const bool by = (iy < ix) & (iy < iz);
        const bool bz = !(bx | by);
        const T dsel = bx ? sdx : (by ? sdy : sdz);
        idx += dsel;
        const int32_t v = IX::load(vox, idx);
        // currentIntersect: the intersect of the axis just stepped, before its update
        const float cur = bx ? ix : (by ? iy : iz);
        if (v >= 0) {
            h.pos[0] = dx * cur + sx;
            h.pos[1] = dy * cur + sy;
            h.pos[2] = dz * cur + sz;
            axis = bx ? 0 : (by ? 1 : 2);
            result = IX::word(idx);
            h.word = v;
            break;
        }
        if (v != -1) {
            // the jump recomputes every intersect, so the step's update is skipped
            const float toJump = -__int_as_float(v);
            trav += toJump;
            const float c2 = cur + toJump;
            sx = dx * c2 + sx;
            sy = dy * c2 + sy;
            sz = dz * c2 + sz;
            const int32_t cx = f2i(sx), cy = f2i(sy), cz = f2i(sz);
            // A jump that leaves `travelled` at or past the budget (or NaN:
            // a guard cell) ends the walk at the loop test (:83); nothing the
            // jump recomputes is read after that.  One branch for that and
            // the cutoff.
            if (!(trav < lim) | (cy > ytop)) {
                // run_walk's last word, if in the caller's grid: both end here
                if (kAgain && again & (v == kGuardCorner)) counted = iters;
                break;
            }
            if constexpr (kAgain) {
                // where else run_walk ended: at a jump with a tiny fraction, or
                // in the step after a jump to below x = 0 or y = 0 (`again`
                // says that this step met the guard's corner: with both below
                // 0, or along the other axis, when this walk ends there too)
                const bool tiny = ((sx > 0.0f) & (sx < 0x1p-60f)) | ((sy > 0.0f) & (sy < 0x1p-60f)) |
                                  ((sz > 0.0f) & (sz < 0x1p-60f));
                const bool edge = (sx < 0.0f) | (sy < 0.0f);
                if (again & (tiny | edge)) {
                    counted = iters + (tiny ? 0 : 1);
                    again = false;
                }
            }
            div3_by((float)(cx + fx) - sx, (float)(cy + fy) - sy, (float)(cz + fz) - sz, dx, dy, dz, rx, ry, rz, dok,
                    ix, iy, iz);
            idx = IX::make(g, clamp_cell(cx, g.X), clamp_cell(cy, g.Y), clamp_cell(cz, g.Z));
        } else {
            // The axis just taken has step 0 (its direction component is +-0,
            // so its intersect is +-inf or NaN and adding its delta keeps it
            // so): the cell did not move, and every later iteration repeats
            // this one exactly -- same selection, same cell, same -1 word --
            // until the budget ends the walk as a miss.  Only the counters
            // advance, so they are advanced without the loads.  (The
            // reference's own light orbit keeps lightPos.z = X/2: a sun ray
            // from a hit on the plane z = X/2 has dir.z = +0 and a NaN z
            // intersect, so z is always the axis taken, and it sticks here
            // when its cell holds -1.)  The stride just added is 0 exactly
            // when that step is: a stride is the step times 1, SX or SXY,
            // nonzero in the index's width.
            if (dsel == 0) {
                while (trav < lim) {
                    iters++;
                    trav += 1.0f;
                }
                break;
            }
            ix = bx ? ix + ddx : ix;
            iy = by ? iy + ddy : iy;
            iz = bz ? iz + ddz : iz;
        }
    }
    h.index = result;
    h.axis = axis;
    h.step = axis == 0 ? stx : (axis == 1 ? sty : stz);
    h.iters = kAgain ? iters - counted : iters;
}

// The same walk for 32-bit indices (IdxB, Idx32), where it is bound by VALU
// issue: its loop is written out, with the arithmetic arranged so that a jump
// takes 35 VALU instructions instead of 41, a step 5 instead of 7, and an
// iteration 8 scalar ones where the compiler's loop has 24.  Against the
// compiler's loop, all else alike, 1920x1080 with sun and 16 lights: 152 -> 121
// us; 3840x2160 in the 8 GiB grid: 491 -> 407 us; 64 views in one launch: 7.64
// -> 6.25 ms; 320x180 (one walk's latency): 30.6 -> 26.3 us.
//
// Mirrored axes.  Negating a position and a direction component together
// negates every product and sum of the walk exactly (rounding to nearest is
// symmetric), so a ray is walked with each axis that it ascends negated: then
// it descends on all three, d' = -|d|.  Where c + f - s is the distance to the
// boundary ahead, |c + f - s| is the fraction of s' above its floor (one
// instruction for three), and the quotient by d is that fraction over |d|.  For
// an ascending axis s' = -s, floor(s') = -(int(s) + 1) unless s is whole.  The
// word index is base + sum of floor(s') times the step's negated stride; base
// takes up the 1.
//
// Which rays: those whose direction components lie in [2^-19, 2^6] in
// magnitude (kWide: from 2^-60, with 1e-6 added too) and whose start coordinates
// lie in [2^-20, 2^22] (start_walk).  On an
// ascending axis s then stays at least 2^-20, where the hardware's fraction is
// the rounded difference; on a descending one s may fall below 0 only on its
// way out of the grid (below).  Only the low end of a cell is clamped (lo:
// clamp_cell's -2 or n + 1, mirrored): a ray jumps from inside the grid,
// downward on every axis.  And |s'| stays below 2^31, where a cell would
// saturate and no bound on y (INT32_MAX) would become one: a jump goes less than
// 2^24 (the budget's limit) times 2^6 beyond a segment's steps, whose cells lie
// in a grid of less than 2^23 a side.
//
// After a jump a fraction may be below 2^-60, where the quotient's three
// instructions are not exact (label 6).  Where s is whole it is 0, and the
// shader's distance is 0 on a descending axis (the quotient -0) and 1 on an
// ascending one (the quotient RN(1/|d|)), whose cell is then one lower than
// floor(s') says.  A tiny fraction that is not 0 takes the ray to
// walk_generic.  (s beyond 2^23 is whole, and outside any grid with 32-bit
// indices.)
//
// Leaving through a low face.  For -1 < s < 0 the reference's cell is 0, with
// a negative intersect that its next step takes at once, out of the grid; here
// the cell is -1, from which any step meets a guard cell: a miss in the same
// iteration.  The two differ only if x and y are both on their way out with
// exactly equal intersects, for then the reference steps z.  Such a walk ends
// on a guard cell with x < 0 and y < 0, which hold kGuardCorner: the ray is
// then walked again by walk_generic.  (So are a few that end on one without
// such a tie, with the same result.)
//
// The loop: a lane that hits drops out with its state as it was before the
// step's update, so the axis, the intersect and the hit follow after the loop;
// one that ends as a miss holds a negative word.  Scalar masks nbx / nby: x / y
// is not the axis of this step, from the shader's strict comparisons; stp / jmp:
// the lanes that go on after a step through a -1 cell / that jump.  (A step of
// 0, which walk_generic looks for, needs a zero direction component.)  Every
// load is waited for in the block; a mask that a comparison writes goes through
// a scalar instruction, or two others, before a select reads it.
#define VRT_WALK(LOAD, COUNT, COUNTED)                                                                  \
    "s_mov_b64 %[ex], exec\n\t"                                                                         \
    "s_and_b64 exec, exec, %[alive]\n\t"                                                                \
    "s_cbranch_execz 9f\n\t"                                                                            \
    "1:\n\t"                                                                                            \
    "v_cmp_nlt_f32_e64 %[nbx], %[ix], %[iy]\n\t"                                                        \
    "v_cmp_nlt_f32_e64 %[ta], %[ix], %[iz]\n\t"                                                         \
    "v_cmp_nlt_f32_e64 %[nby], %[iy], %[ix]\n\t"                                                        \
    "v_cmp_nlt_f32_e64 vcc, %[iy], %[iz]\n\t"                                                           \
    "s_or_b64 %[nbx], %[nbx], %[ta]\n\t"                                                                \
    "s_or_b64 %[nby], %[nby], vcc\n\t"                                                                  \
    "v_cndmask_b32_e64 %[sel], %[nsty], %[nstz], %[nby]\n\t"                                            \
    "v_cndmask_b32_e64 %[sel], %[nstx], %[sel], %[nbx]\n\t"                                             \
    "v_sub_u32_e32 %[idx], %[idx], %[sel]\n\t"                                                          \
    LOAD                                                                                                \
    "v_add_f32_e32 %[trav], 1.0, %[trav]\n\t"                                                           \
    COUNT                                                                                               \
    "s_waitcnt vmcnt(0)\n\t"                                                                            \
    "v_cmp_gt_i32_e32 vcc, -1, %[word]\n\t" /* below -1: jumps */                                       \
    "s_andn2_b64 %[stp], exec, vcc\n\t"                                                                 \
    "s_cbranch_scc0 3f\n\t" /* every lane jumps */                                                      \
    "s_mov_b64 %[jmp], vcc\n\t"                                                                         \
    "v_cmp_eq_u32_e64 %[stp], -1, %[word]\n\t" /* the others are solid: done */                         \
    "s_andn2_b64 exec, %[stp], %[nbx]\n\t" /* a step through a -1 cell: its axis's intersect moves on */\
    "v_add_f32_e32 %[ix], %[ix], %[ddx]\n\t"                                                            \
    "s_and_b64 %[ta], %[stp], %[nbx]\n\t"                                                               \
    "s_andn2_b64 exec, %[ta], %[nby]\n\t"                                                               \
    "v_add_f32_e32 %[iy], %[iy], %[ddy]\n\t"                                                            \
    "s_and_b64 exec, %[ta], %[nby]\n\t"                                                                 \
    "v_add_f32_e32 %[iz], %[iz], %[ddz]\n\t"                                                            \
    "s_mov_b64 exec, %[stp]\n\t"                                                                        \
    "v_cmp_gt_f32_e64 %[stp], %[lim], %[trav]\n\t"                                                      \
    "s_mov_b64 exec, %[jmp]\n\t"                                                                        \
    "s_cbranch_execz 5f\n\t"                                                                            \
    "3:\n\t" /* a jump by the word's distance */                                                        \
    "v_cndmask_b32_e64 %[cur], %[iy], %[iz], %[nby]\n\t"                                                \
    "v_cndmask_b32_e64 %[cur], %[ix], %[cur], %[nbx]\n\t"                                               \
    "v_sub_f32_e32 %[trav], %[trav], %[word]\n\t"                                                       \
    "v_sub_f32_e32 %[cur], %[cur], %[word]\n\t"                                                         \
    "v_mul_f32_e32 %[t1], %[dy], %[cur]\n\t"                                                            \
    "v_mul_f32_e32 %[t0], %[dx], %[cur]\n\t"                                                            \
    "v_mul_f32_e32 %[t2], %[dz], %[cur]\n\t"                                                            \
    "v_add_f32_e32 %[sy], %[t1], %[sy]\n\t"                                                             \
    "v_add_f32_e32 %[sx], %[t0], %[sx]\n\t"                                                             \
    "v_add_f32_e32 %[sz], %[t2], %[sz]\n\t"                                                             \
    "v_cvt_flr_i32_f32_e32 %[t1], %[sy]\n\t"                                                            \
    "v_cmp_gt_f32_e32 vcc, %[lim], %[trav]\n\t"                                                         \
    "v_cmp_gt_f32_e64 %[ta], %[sy], %[tb]\n\t"                                                          \
    "s_and_b64 exec, vcc, %[ta]\n\t" /* out of budget, or above the solid top: a miss */                \
    "s_cbranch_execz 5f\n\t"                                                                            \
    "v_fract_f32_e32 %[ix], %[sx]\n\t"                                                                  \
    "v_fract_f32_e32 %[iy], %[sy]\n\t"                                                                  \
    "v_fract_f32_e32 %[iz], %[sz]\n\t"                                                                  \
    "v_cvt_flr_i32_f32_e32 %[t0], %[sx]\n\t"                                                            \
    "v_cvt_flr_i32_f32_e32 %[t2], %[sz]\n\t"                                                            \
    "v_min3_f32 %[cur], %[ix], %[iy], %[iz]\n\t"                                                        \
    "v_max_i32_e32 %[t0], %[t0], %[lox]\n\t"                                                            \
    "v_max_i32_e32 %[t1], %[t1], %[loy]\n\t"                                                            \
    "v_max_i32_e32 %[t2], %[t2], %[loz]\n\t"                                                            \
    "v_mad_i32_i24 %[idx], %[t0], %[nstx], %[base]\n\t"                                                 \
    "v_mad_i32_i24 %[idx], %[t1], %[nsty], %[idx]\n\t"                                                  \
    "v_mad_i32_i24 %[idx], %[t2], %[nstz], %[idx]\n\t"                                                  \
    "v_mul_f32_e32 %[t0], %[ix], %[rx]\n\t"                                                             \
    "v_mul_f32_e32 %[t1], %[iy], %[ry]\n\t"                                                             \
    "v_mul_f32_e32 %[t2], %[iz], %[rz]\n\t"                                                             \
    "v_fma_f32 %[ix], %[t0], %[dx], %[ix]\n\t"                                                          \
    "v_fma_f32 %[iy], %[t1], %[dy], %[iy]\n\t"                                                          \
    "v_fma_f32 %[iz], %[t2], %[dz], %[iz]\n\t"                                                          \
    "v_fma_f32 %[ix], %[ix], %[rx], %[t0]\n\t"                                                          \
    "v_fma_f32 %[iy], %[iy], %[ry], %[t1]\n\t"                                                          \
    "v_fma_f32 %[iz], %[iz], %[rz], %[t2]\n\t"                                                          \
    "v_cmp_nle_f32_e32 vcc, 0x21800000, %[cur]\n\t"                                                     \
    "s_cbranch_vccnz 6f\n\t"                                                                            \
    "5:\n\t"                                                                                            \
    "s_or_b64 exec, exec, %[stp]\n\t"                                                                   \
    "s_cbranch_execnz 1b\n\t"                                                                           \
    "s_branch 9f\n\t"                                                                                   \
    "6:\n\t" /* a fraction below 2^-60 */                                                               \
    "s_mov_b64 %[jmp], exec\n\t"                                                                        \
    "s_mov_b64 exec, vcc\n\t"                                                                           \
    "v_mov_b32_e32 %[idx], %[base]\n\t"                                                                 \
    "v_mov_b32_e32 %[cur], 0x80000000\n\t"                                                              \
    "v_fract_f32_e32 %[t0], %[sx]\n\t"                                                                  \
    "v_cvt_flr_i32_f32_e32 %[t1], %[sx]\n\t"                                                            \
    "v_cmp_eq_f32_e64 %[nbx], 0, %[t0]\n\t"                                                             \
    "v_cmp_gt_i32_e64 %[ta], 0, %[nstx]\n\t"                                                            \
    "v_cmp_gt_f32_e32 vcc, 0x21800000, %[t0]\n\t"                                                       \
    "s_andn2_b64 %[nby], vcc, %[nbx]\n\t" /* tiny, not whole: for the general walk */                   \
    "s_andn2_b64 %[jmp], %[jmp], %[nby]\n\t"                                                            \
    "v_mov_b32_e32 %[t2], 0xffc00001\n\t"                                                               \
    "v_cndmask_b32_e64 %[word], %[word], %[t2], %[nby]\n\t"                                             \
    "v_cndmask_b32_e64 %[ix], %[ix], %[cur], %[nbx]\n\t"                                                \
    "s_and_b64 %[ta], %[ta], %[nbx]\n\t"                                                                \
    "v_cndmask_b32_e64 %[ix], %[ix], %[rx], %[ta]\n\t"                                                  \
    "v_cndmask_b32_e64 %[t2], 0, 1, %[ta]\n\t"                                                          \
    "v_sub_u32_e32 %[t1], %[t1], %[t2]\n\t"                                                             \
    "v_max_i32_e32 %[t1], %[t1], %[lox]\n\t"                                                            \
    "v_mad_i32_i24 %[idx], %[t1], %[nstx], %[idx]\n\t"                                                  \
    "v_fract_f32_e32 %[t0], %[sy]\n\t"                                                                  \
    "v_cvt_flr_i32_f32_e32 %[t1], %[sy]\n\t"                                                            \
    "v_cmp_eq_f32_e64 %[nbx], 0, %[t0]\n\t"                                                             \
    "v_cmp_gt_i32_e64 %[ta], 0, %[nsty]\n\t"                                                            \
    "v_cmp_gt_f32_e32 vcc, 0x21800000, %[t0]\n\t"                                                       \
    "s_andn2_b64 %[nby], vcc, %[nbx]\n\t" /* tiny, not whole: for the general walk */                   \
    "s_andn2_b64 %[jmp], %[jmp], %[nby]\n\t"                                                            \
    "v_mov_b32_e32 %[t2], 0xffc00001\n\t"                                                               \
    "v_cndmask_b32_e64 %[word], %[word], %[t2], %[nby]\n\t"                                             \
    "v_cndmask_b32_e64 %[iy], %[iy], %[cur], %[nbx]\n\t"                                                \
    "s_and_b64 %[ta], %[ta], %[nbx]\n\t"                                                                \
    "v_cndmask_b32_e64 %[iy], %[iy], %[ry], %[ta]\n\t"                                                  \
    "v_cndmask_b32_e64 %[t2], 0, 1, %[ta]\n\t"                                                          \
    "v_sub_u32_e32 %[t1], %[t1], %[t2]\n\t"                                                             \
    "v_max_i32_e32 %[t1], %[t1], %[loy]\n\t"                                                            \
    "v_mad_i32_i24 %[idx], %[t1], %[nsty], %[idx]\n\t"                                                  \
    "v_fract_f32_e32 %[t0], %[sz]\n\t"                                                                  \
    "v_cvt_flr_i32_f32_e32 %[t1], %[sz]\n\t"                                                            \
    "v_cmp_eq_f32_e64 %[nbx], 0, %[t0]\n\t"                                                             \
    "v_cmp_gt_i32_e64 %[ta], 0, %[nstz]\n\t"                                                            \
    "v_cmp_gt_f32_e32 vcc, 0x21800000, %[t0]\n\t"                                                       \
    "s_andn2_b64 %[nby], vcc, %[nbx]\n\t" /* tiny, not whole: for the general walk */                   \
    "s_andn2_b64 %[jmp], %[jmp], %[nby]\n\t"                                                            \
    "v_mov_b32_e32 %[t2], 0xffc00001\n\t"                                                               \
    "v_cndmask_b32_e64 %[word], %[word], %[t2], %[nby]\n\t"                                             \
    "v_cndmask_b32_e64 %[iz], %[iz], %[cur], %[nbx]\n\t"                                                \
    "s_and_b64 %[ta], %[ta], %[nbx]\n\t"                                                                \
    "v_cndmask_b32_e64 %[iz], %[iz], %[rz], %[ta]\n\t"                                                  \
    "v_cndmask_b32_e64 %[t2], 0, 1, %[ta]\n\t"                                                          \
    "v_sub_u32_e32 %[t1], %[t1], %[t2]\n\t"                                                             \
    "v_max_i32_e32 %[t1], %[t1], %[loz]\n\t"                                                            \
    "v_mad_i32_i24 %[idx], %[t1], %[nstz], %[idx]\n\t"                                                  \
    "s_mov_b64 exec, %[jmp]\n\t"                                                                        \
    "s_branch 5b\n\t"                                                                                   \
    "9:\n\t"                                                                                            \
    "s_mov_b64 exec, %[ex]\n\t"                                                                         \
    COUNTED

static_assert((uint32_t)kGuardCorner == 0xffc00001u, "as written in the loop");

// Walk state of one lane; s, d, r mirrored as described above.
struct Walk {
    float sx, sy, sz, dx, dy, dz, rx, ry, rz, ddx, ddy, ddz, ix, iy, iz, trav;
    uint32_t idx, base, iters;
    int32_t nstx, nsty, nstz, lox, loy, loz, word;
    float tb;
};

#define VRT_WALK_OUT                                                                                            \
    [sx] "+&v"(w.sx), [sy] "+&v"(w.sy), [sz] "+&v"(w.sz), [ix] "+&v"(w.ix), [iy] "+&v"(w.iy),                   \
        [iz] "+&v"(w.iz), [trav] "+&v"(w.trav), [iters] "+&v"(w.iters), [word] "+&v"(w.word), [ex] "=&s"(ex),   \
        [nbx] "=&s"(nbx), [nby] "=&s"(nby), [stp] "=&s"(stp), [jmp] "=&s"(jmp), [ta] "=&s"(ta),                 \
        [cur] "=&v"(cur), [t0] "=&v"(t0), [t1] "=&v"(t1), [t2] "=&v"(t2), [sel] "=&v"(sel), [n] "+&s"(n),       \
        [k] "=&s"(k)
#define VRT_WALK_IN                                                                                             \
    [dx] "v"(w.dx), [dy] "v"(w.dy), [dz] "v"(w.dz), [rx] "v"(w.rx), [ry] "v"(w.ry), [rz] "v"(w.rz),             \
        [ddx] "v"(w.ddx), [ddy] "v"(w.ddy), [ddz] "v"(w.ddz), [nstx] "v"(w.nstx), [nsty] "v"(w.nsty),           \
        [nstz] "v"(w.nstz), [lox] "v"(w.lox), [loy] "v"(w.loy), [loz] "v"(w.loz), [base] "v"(w.base),           \
        [tb] "v"(w.tb), [vox] "s"(vox), [alive] "s"(alive), [lim] "v"(lim)
#define VRT_LOAD_B "global_load_dword %[word], %[idx], %[vox]\n\t"
// Word indices reach past 4 GiB: the address is 64 bits, from the index in the
// low half of a register pair whose high half is 0.
#define VRT_LOAD_32 "v_lshl_add_u64 %[addr], v[4:5], 2, %[vox]\n\tglobal_load_dword %[word], %[addr], off\n\t"
// Iterations per lane; or their sum over the wave, kept on the scalar unit and
// left in the first active lane (the others hold 0).
#define VRT_COUNT_LANES "v_add_u32_e32 %[iters], 1, %[iters]\n\t"
#define VRT_COUNT_WAVE "s_bcnt1_i32_b64 %[k], exec\n\ts_add_u32 %[n], %[n], %[k]\n\t"
#define VRT_COUNTED_WAVE \
    "s_ff1_i32_b64 %[k], exec\n\ts_mov_b32 m0, %[k]\n\ts_nop 0\n\tv_writelane_b32 %[iters], %[n], m0\n\t"

// Runs the loop for the lanes of `alive` until none is left.  kLanes: w.iters
// counts each lane's iterations; else the wave's sum ends in one lane.
template <bool kLanes>
__device__ __forceinline__ void run_walk(IdxB, const int32_t* vox, float lim, uint64_t alive, Walk& w) {
    uint64_t ex, nbx, nby, stp, jmp, ta;
    float cur, t0, t1, t2;
    int32_t sel;
    uint32_t n = 0, k;
    if constexpr (kLanes)
        asm volatile(VRT_WALK(VRT_LOAD_B, VRT_COUNT_LANES, "")
                     : VRT_WALK_OUT, [idx] "+&v"(w.idx)
                     : VRT_WALK_IN
                     : "vcc", "scc", "memory");
    else
        asm volatile(VRT_WALK(VRT_LOAD_B, VRT_COUNT_WAVE, VRT_COUNTED_WAVE)
                     : VRT_WALK_OUT, [idx] "+&v"(w.idx)
                     : VRT_WALK_IN
                     : "vcc", "scc", "m0", "memory");
}
template <bool kLanes>
__device__ __forceinline__ void run_walk(Idx32, const int32_t* vox, float lim, uint64_t alive, Walk& w) {
    uint64_t ex, nbx, nby, stp, jmp, ta;
    float cur, t0, t1, t2;
    int32_t sel;
    uint32_t n = 0, k;
    uint64_t addr;
    if constexpr (kLanes)
        asm volatile(VRT_WALK(VRT_LOAD_32, VRT_COUNT_LANES, "")
                     : VRT_WALK_OUT, [idx] "+&{v4}"(w.idx), [addr] "=&v"(addr)
                     : VRT_WALK_IN, [zero] "{v5}"(0u)
                     : "vcc", "scc", "memory");
    else
        asm volatile(VRT_WALK(VRT_LOAD_32, VRT_COUNT_WAVE, VRT_COUNTED_WAVE)
                     : VRT_WALK_OUT, [idx] "+&{v4}"(w.idx), [addr] "=&v"(addr)
                     : VRT_WALK_IN, [zero] "{v5}"(0u)
                     : "vcc", "scc", "m0", "memory");
}
#undef VRT_WALK
#undef VRT_WALK_OUT
#undef VRT_WALK_IN
#undef VRT_LOAD_B
#undef VRT_LOAD_32
#undef VRT_COUNT_LANES
#undef VRT_COUNT_WAVE
#undef VRT_COUNTED_WAVE

// The walk's state at a ray's start (arguments as cast_ray's), for rays that
// run_walk takes; false for any other.
//
// kWide (a frame's primary rays where the lanes count): a lane that goes to
// walk_generic makes its wave walk twice, one form after the other.  Along the
// horizon a component passes through 0 and a pixel in 700 lies below 2^-19: few,
// but in a frame's longest waves, which end it where it has few tiles or its
// rays run far.  Depth view, 1920x1080 in a 512x512x3700 grid: 399 us, from 2^-19
// 503; 960x540 261 and 374; 800x600 in a small world 2 to 3% less.  (Sending the
// whole wave to walk_generic instead: 402, 265 and 1% more everywhere.  Other rays
// do not gain: 16 views in one launch 1% slower, lists of few rays 3%.)
//
// The first cell and intersects.  From a hit: as after a jump, for a start
// inside the grid (any other takes walk_generic).  Else: the reference's
// formulas.  (The camera's distances to its cell's boundaries made with the
// frame instead of by every lane: no gain, small frames 2% slower.)
template <typename IX, bool kHit, bool kWide>
__device__ __forceinline__ bool start_walk(const GridDesc& g, float px, float py, float pz, float dx, float dy,
                                           float dz, Walk& w) {
    const float sx = kHit ? px + dx * 0.001f : px, sy = kHit ? py + dy * 0.001f : py,
                sz = kHit ? pz + dz * 0.001f : pz;
    const bool mx = dx > 0.0f, my = dy > 0.0f, mz = dz > 0.0f;
    w.sx = mx ? -sx : sx;
    w.sy = my ? -sy : sy;
    w.sz = mz ? -sz : sz;
    // |d| >= 2^-19 keeps |d + 1e-6| in range too; kWide tests both.  min and max
    // pass over a NaN; the comparisons of s (NaN where d is) or the sum do not.
    const float bx = fabsf(dx + 0.000001f), by = fabsf(dy + 0.000001f), bz = fabsf(dz + 0.000001f);
    float lo = fminf(fminf(fabsf(dx), fabsf(dy)), fabsf(dz));
    if constexpr (kWide) lo = fminf(lo, fminf(fminf(bx, by), bz));
    const float hi = fmaxf(fmaxf(fabsf(dx), fabsf(dy)), fabsf(dz));
    bool fast = (lo >= (kWide ? 0x1p-60f : 0x1p-19f)) & (hi <= 0x1p6f);
    if constexpr (kHit) {
        w.ix = __builtin_amdgcn_fractf(w.sx);
        w.iy = __builtin_amdgcn_fractf(w.sy);
        w.iz = __builtin_amdgcn_fractf(w.sz);
        fast &= (fminf(fminf(sx, sy), sz) >= 0x1p-20f) & (sx < g.FX) & (sy < g.FY) & (sz < g.FZ);
    } else {
        const float sum = ((dx + dy) + dz) + ((sx + sy) + sz);
        fast &= (fminf(fminf(sx, sy), sz) >= 0x1p-20f) & (fmaxf(fmaxf(sx, sy), sz) <= 0x1p22f) & (sum == sum);
    }
    if (!fast) return false;
    w.ddx = rcp_fast(bx);
    w.ddy = rcp_fast(by);
    w.ddz = rcp_fast(bz);
    w.rx = rcp_fast(fabsf(dx));
    w.ry = rcp_fast(fabsf(dy));
    w.rz = rcp_fast(fabsf(dz));
    w.dx = -fabsf(dx);
    w.dy = -fabsf(dy);
    w.dz = -fabsf(dz);
    w.nstx = (int32_t)IX::stride(g, mx ? -1 : 1, 0);
    w.nsty = (int32_t)IX::stride(g, my ? -1 : 1, 1);
    w.nstz = (int32_t)IX::stride(g, mz ? -1 : 1, 2);
    w.lox = mx ? -(int32_t)g.X - 2 : -2;
    w.loy = my ? -(int32_t)g.Y - 2 : -2;
    w.loz = mz ? -(int32_t)g.Z - 2 : -2;
    w.base = IX::make(g, 0, 0, 0) + (uint32_t)((mx ? w.nstx : 0) + (my ? w.nsty : 0) + (mz ? w.nstz : 0));
    if constexpr (kHit) {
        // u / |d| as after a jump: exact for u = 0 and u >= 2^-60
        auto quotient = [](float u, float d, float r) {
            const float q0 = u * r;
            return __builtin_fmaf(__builtin_fmaf(q0, d, u), r, q0);
        };
        w.idx = IX::add(w.base, floor_i(w.sx), w.nstx);
        w.idx = IX::add(w.idx, floor_i(w.sy), w.nsty);
        w.idx = IX::add(w.idx, floor_i(w.sz), w.nstz);
        // s >= 2^-20, so a fraction is 0 or at least 2^-43.  A whole s
        // on an ascending axis: the boundary ahead is 1 away, the
        // cell one lower than floor(s') says.  (Common: a face's
        // coordinate stays whole where d * 0.001 rounds away.)
        if (fminf(fminf(w.ix, w.iy), w.iz) == 0.0f) {
            const bool ax = mx & (w.ix == 0.0f), ay = my & (w.iy == 0.0f), az = mz & (w.iz == 0.0f);
            w.idx -= (uint32_t)((ax ? w.nstx : 0) + (ay ? w.nsty : 0) + (az ? w.nstz : 0));
            w.ix = ax ? 1.0f : w.ix;
            w.iy = ay ? 1.0f : w.iy;
            w.iz = az ? 1.0f : w.iz;
        }
        w.ix = quotient(w.ix, w.dx, w.rx);
        w.iy = quotient(w.iy, w.dy, w.ry);
        w.iz = quotient(w.iz, w.dz, w.rz);
    } else {
        const int32_t cx = f2i(sx), cy = f2i(sy), cz = f2i(sz);
        w.idx = IX::make(g, clamp_cell(cx, g.X), clamp_cell(cy, g.Y), clamp_cell(cz, g.Z));
        div3_by((float)(mx ? -cx - 1 : cx) - w.sx, (float)(my ? -cy - 1 : cy) - w.sy,
                (float)(mz ? -cz - 1 : cz) - w.sz, w.dx, w.dy, w.dz, -w.rx, -w.ry, -w.rz, true, w.ix, w.iy,
                w.iz);
    }
    w.trav = 0.0f;
    w.iters = 0;
    w.word = -1;
    return true;
}

// castRay, src/fshader.glsl:59-129 (see walk_generic for lim), from p, or with
// kHit from p + d * 0.001 (the shadow rays' start, :152, :165).  ytop: the cutoff's
// bound for a ray that does not head down (INT32_MAX: none).  What the
// walk does not need is recovered from its state afterwards (the direction and
// steps from d' and the strides, the start from p) rather than held in
// registers meanwhile.
//
// kLanes: h.iters is the ray's own iterations (a step map or the depth view
// shows them); else the lanes' h.iters only add up to the wave's.
template <typename IX, bool kHit, bool kLanes, bool kWide = false>
__device__ __forceinline__ void cast_ray(const GridDesc& g, float px, float py, float pz, float dx, float dy,
                                         float dz, float lim, Hit& h, int32_t ytop) {
    bool general = true, again = false;
    h.iters = 0;
    if constexpr (!std::is_same_v<IX, Idx64>) {
        Walk w;
        if (start_walk<IX, kHit, kWide>(g, px, py, pz, dx, dy, dz, w)) {
            w.tb = dy > 0.0f ? -1.0f - (float)ytop : -__builtin_inff();
            run_walk<kLanes>(IX{}, g.vox, lim, __ballot(0.0f < lim), w);
            auto flip = [](int32_t nst, float v) { return nst < 0 ? -v : v; };
            const bool bx = (w.ix < w.iy) & (w.ix < w.iz), by = (w.iy < w.ix) & (w.iy < w.iz);
            const float cur = bx ? w.ix : (by ? w.iy : w.iz);
            const bool hit = w.word >= 0;
            h.pos[0] = flip(w.nstx, w.dx * cur + w.sx);
            h.pos[1] = flip(w.nsty, w.dy * cur + w.sy);
            h.pos[2] = flip(w.nstz, w.dz * cur + w.sz);
            h.axis = hit ? (bx ? 0 : (by ? 1 : 2)) : -1;
            h.step = (bx ? w.nstx : (by ? w.nsty : w.nstz)) < 0 ? 1 : -1;
            h.index = hit ? IX::word(w.idx) : -1;
            h.word = w.word;
            general = again = w.word == kGuardCorner;
            dx = flip(w.nstx, w.dx);
            dy = flip(w.nsty, w.dy);
            dz = flip(w.nstz, w.dz);
            h.iters = w.iters;
        }
    }
    if (__builtin_expect(general, 0)) {
        const uint32_t sum = kLanes ? 0 : h.iters;  // of the wave's sum, what this lane holds
        walk_generic<IX, !kLanes && !std::is_same_v<IX, Idx64>>(
            g, kHit ? px + dx * 0.001f : px, kHit ? py + dy * 0.001f : py, kHit ? pz + dz * 0.001f : pz, dx, dy, dz, lim, h,
            dy >= 0.0f ? ytop : INT32_MAX, again);
        h.iters += sum;
    }
}

// main(), src/fshader.glsl:131-190, for the fragment at vPos = (vx, vy), pixel
// k of the target.  `top`: the grid's solid-top bound for shadow rays
// (INT32_MAX: none).  What the primary ray decides is stored before the shadow
// rays are walked, so it holds no registers meanwhile.  The hit's reference
// index (two integer divisions) is formed only when the target has a hit map.
// kLanes: see cast_ray.
template <typename IX, bool kLanes>
__device__ __forceinline__ void shade_pixel(const GridDesc& g, const FrameDesc& F, const vrt_target& t, int64_t k,
                                            float vx, float vy, int32_t top, uint32_t& rays, uint32_t& iters) {
    const vrt_frame& f = F.f;
    float col0 = 0.6f, col1 = 0.7f, col2 = 0.8f;

    // normalize(vec3(vPos.x*aspectRatio, vPos.y, focal)) (:136)
    const float ux = vx * f.aspect_ratio, uy = vy, uz = f.focal;
    const float un = rcp_rn(sqrtf(dot3(ux, uy, uz, ux, uy, uz)));
    const float rx = ux * un, ry = uy * un, rz = uz * un;
    // vec3(rotateMatrix * vec4(d, 0)) (:137), GLM's pairwise column sum
    const float* M = f.rotate_matrix;
    const float d0 = (M[0] * rx + M[4] * ry) + (M[8] * rz + M[12] * 0.0f);
    const float d1 = (M[1] * rx + M[5] * ry) + (M[9] * rz + M[13] * 0.0f);
    const float d2 = (M[2] * rx + M[6] * ry) + (M[10] * rz + M[14] * 0.0f);

    // The primary ray may take the cutoff when its step count is not an
    // output of this draw (no depth view, no step map): a ray that stops
    // there misses, as the reference's walk would.
    Hit h;
    cast_ray<IX, false, kLanes, kLanes>(g, f.cam_pos[0], f.cam_pos[1], f.cam_pos[2], d0, d1, d2, F.render_lim, h,
                        F.primary_cutoff != 0 ? top : INT32_MAX);
    iters = h.iters;
    uint32_t eval = 0, occ = 0;
    const bool hit = h.index != -1;
    const float hx = hit ? h.pos[0] : 0.0f, hy = hit ? h.pos[1] : 0.0f, hz = hit ? h.pos[2] : 0.0f;
    // firstHitNormal = -step on the axis of the last step
    const float nx = h.axis == 0 ? (float)(-h.step) : 0.0f;
    const float ny = h.axis == 1 ? (float)(-h.step) : 0.0f;
    const float nz = h.axis == 2 ? (float)(-h.step) : 0.0f;

    if (t.depth) {
        float depth = __builtin_inff();
        if (hit) {
            const float ex = hx - f.cam_pos[0], ey = hy - f.cam_pos[1], ez = hz - f.cam_pos[2];
            depth = sqrtf(dot3(ex, ey, ez, ex, ey, ez));
        }
        t.depth[k] = depth;
    }
    if (t.hit) t.hit[k] = hit ? IX::ref_index(g, h.index) : -1;
    if (t.face) t.face[k] = hit ? (uint8_t)(h.axis * 3 + (h.step + 1)) : (uint8_t)VRT_FACE_MISS;
    if (kLanes && t.steps) t.steps[k] = h.iters;

    if (kLanes && f.view_depth_field == 1) {
        const float s = div_small_int((float)h.iters, 100.0f, 1.0f / 100.0f);
        col0 = s;
        col1 = s;
        col2 = s;
    } else if (hit) {
        const int32_t vcol = h.word;
        // toLight = normalize(lightPos - firstHitPos) (:147)
        const float lx0 = f.light_pos[0] - hx, ly0 = f.light_pos[1] - hy, lz0 = f.light_pos[2] - hz;
        const float ln = rcp_rn(sqrtf(dot3(lx0, ly0, lz0, lx0, ly0, lz0)));
        const float tlx = lx0 * ln, tly = ly0 * ln, tlz = lz0 * ln;
        float m0 = 0.4f, m1 = 0.4f, m2 = 0.4f;  // AMBIENT

        // sun shadow (:152-156)
        {
            Hit s;
            cast_ray<IX, true, kLanes>(g, hx, hy, hz, tlx, tly, tlz, F.render_lim, s, top);
            iters += s.iters;
            eval |= 1u;
            if (s.index == -1) {
                const float add = 0.8f * max0(dot3(nx, ny, nz, tlx, tly, tlz));  // DIFFUSE
                m0 += add;
                m1 += add;
                m2 += add;
            } else {
                occ |= 1u;
            }
        }

        // local lights (:158-181).  The loop's first statement clamps to
        // MAX_OVERBRIGHT and leaves once every channel is >= 1.25; the
        // channels change only when a light adds to them, so the test is made
        // after each addition (and once for the sun) instead of on every
        // iteration, and the clamp is applied where the next iteration's test
        // would apply it: always after the sun, after light i only if i < 15
        // (no iteration follows the last).  Unplaced lights do nothing but
        // that test, so the loop visits the placed ones only.
        bool over = (m0 >= 1.25f) & (m1 >= 1.25f) & (m2 >= 1.25f);
        if (over) {
            m0 = 1.25f;
            m1 = 1.25f;
            m2 = 1.25f;
        }
        // The x distance alone rules most lights out for the whole wave: the
        // lights that it leaves to any lane, four at a time (their x and
        // bounds lie together, so a group waits for one scalar load; one light
        // after the other, each waiting for its own, took 3% of a frame with
        // 16 lights).
        uint32_t near = 0;
        for (int j = 0; j < VRT_MAX_LOCAL_LIGHTS && (F.light_valid >> j) != 0u; j += 4) {
#pragma unroll
            for (int i = 0; i < 4; i++)
                near |= __ballot(fabsf(F.light_x[j + i] - hx) <= F.light_axis_max[j + i]) != 0 ? 1u << (j + i) : 0u;
        }
        for (uint32_t rem = near & F.light_valid; rem != 0u; rem &= rem - 1u) {
            if (over) break;
            const int i = __builtin_ctz(rem);
            const vrt_local_light& L = f.lights[i];
            // length <= radius (:171), decided without the square root
            const float vx0 = L.pos[0] - hx, vy0 = L.pos[1] - hy, vz0 = L.pos[2] - hz;
            const float dd = dot3(vx0, vy0, vz0, vx0, vy0, vz0);
            if (!(dd <= F.light_dd_max[i])) continue;
            const float dist = sqrtf(dd);
            const float inv = rcp_rn(dist);
            const float ux1 = vx0 * inv, uy1 = vy0 * inv, uz1 = vz0 * inv;
            float lim = (float)f2i(dist + 1.0f);
            lim = lim < F.render_lim ? lim : F.render_lim;
            Hit s;
            cast_ray<IX, true, kLanes>(g, hx, hy, hz, ux1, uy1, uz1, lim, s, top);
            iters += s.iters;
            eval |= 2u << i;
            if (s.index == -1) {
                const float lam = max0(dot3(nx, ny, nz, ux1, uy1, uz1));
                const float fall = div_by(L.radius - dist, L.radius, F.light_rinv[i], div_range_ok(L.radius));
                m0 += L.rgb[0] * lam * fall;
                m1 += L.rgb[1] * lam * fall;
                m2 += L.rgb[2] * lam * fall;
                over = (m0 >= 1.25f) & (m1 >= 1.25f) & (m2 >= 1.25f);
                if (over & (i < VRT_MAX_LOCAL_LIGHTS - 1)) {
                    m0 = 1.25f;
                    m1 = 1.25f;
                    m2 = 1.25f;
                }
            } else {
                occ |= 2u << i;
            }
        }

        col0 = div_small_int((float)((vcol & 0x00FF0000) >> 16), 255.0f, 1.0f / 255.0f) * m0;
        col1 = div_small_int((float)((vcol & 0x0000FF00) >> 8), 255.0f, 1.0f / 255.0f) * m1;
        col2 = div_small_int((float)(vcol & 0x000000FF), 255.0f, 1.0f / 255.0f) * m2;
    }
    uint8_t* c = t.rgb + 3 * k;
    c[0] = unorm8(col0);
    c[1] = unorm8(col1);
    c[2] = unorm8(col2);
    if (t.shadow_eval) t.shadow_eval[k] = eval;
    if (t.shadow_occ) t.shadow_occ[k] = occ;
    rays = 1 + (uint32_t)__builtin_popcount(eval);
}

// vPos of pixel (px, row), row 0 at the top (GL rows count from the bottom):
// (2px+1)/W - 1 and (2py+1)/H - 1, the divisions through RN(1/W), RN(1/H).
__device__ __forceinline__ void pixel_vpos(int32_t W, int32_t H, float inv_w, float inv_h, int32_t px, int32_t row,
                                           float& vx, float& vy) {
    const int32_t py = H - 1 - row;
    vx = div_small_int((float)(2 * px + 1), (float)W, inv_w) - 1.0f;
    vy = div_small_int((float)(2 * py + 1), (float)H, inv_h) - 1.0f;
}

// Sum of a 32-bit value over a full wave (all 64 lanes active), on the scalar
// unit: prefix sums within each row of 16 lanes by DPP row shifts (zeros
// shifted in), then the row totals carried on by row broadcasts, so lane 63
// holds the total.  Six VALU adds instead of the lane-index arithmetic and
// LDS permutes of a shuffle tree.  The caller keeps the total below 2^32.
__device__ __forceinline__ uint32_t wave_sum_u32(uint32_t v) {
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x111, 0xf, 0xf, true);   // row_shr:1
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x112, 0xf, 0xf, true);   // row_shr:2
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x114, 0xf, 0xf, true);   // row_shr:4
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x118, 0xf, 0xf, true);   // row_shr:8
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x142, 0xa, 0xf, false);  // row_bcast:15, rows 1 and 3
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x143, 0xc, 0xf, false);  // row_bcast:31, rows 2 and 3
    return (uint32_t)__builtin_amdgcn_readlane((int)v, 63);
}

// The same for per-lane values below 2^58: the low 26 bits and the rest are
// summed apart (64 lanes of 26 bits stay below 2^32), then recombined.
__device__ __forceinline__ unsigned long long wave_sum_u58(unsigned long long v) {
    const uint32_t lo = wave_sum_u32((uint32_t)(v & 0x3ffffffull));
    const uint32_t hi = wave_sum_u32((uint32_t)(v >> 26));
    return (unsigned long long)lo + ((unsigned long long)hi << 26);
}

}  // namespace dev
}  // namespace vrt
