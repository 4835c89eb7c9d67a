// vrt_field.h — the depth field of a tile, 32 voxels per lane at a time.
//
// fixDepthField (src/render.cpp:226-253) gives an empty voxel the distance of
// the nearest solid one among the offsets (x, y, z) with x^2+y^2+z^2 <= 49,
// where distance is sqrt(a^2+b^2+c^2) of the offset with each component moved
// one step toward zero (the distance between the two unit cubes).  A solid at
// offset x along an axis is at |x|-1 there, and at 0 for x in {-1, 0, 1}: so
// with D the solidity dilated by one cell on every axis, the distance is the
// ordinary one from the voxel to the nearest cell of D.  The squared distance
// n = a^2+b^2+c^2 is then built up separably on bit masks, one bit per voxel
// along x: per row, X_a = the voxels with a cell of D at +-a along x; per
// (y, z), E_m = OR of X_a at +-b along y over a^2+b^2 = m; and last
// T_n = OR of E_m at +-c along z over m+c^2 = n.  No voxel scans a table, and
// 32 voxels share each operation.
//
// Which (a, b, c) count: those whose offsets lie inside the radius-7 ball,
// which are all with n <= 30 except (4, 3, 2) in any order (kClassOk below
// checks this against the ball).  n > 30 is none of the table's distances
// above -6.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <type_traits>

#include "vrt_internal.h"

namespace vrt {
namespace dev {

constexpr int kFieldReach = 5;  // largest component that counts (n <= 30)

constexpr bool class_432(int a, int b, int c) {
    return a + b + c == 9 && a * b * c == 24 && a * a + b * b + c * c == 29;
}

// Every class (a, b, c) below n = 36: all of its offsets are in the ball when
// it counts here, and none when it does not.  A zero component stands for
// offsets 0 and +-1, a > 0 for +-(a + 1).
constexpr bool classes_match_ball() {
    for (int a = 0; a <= 6; a++)
        for (int b = 0; b <= 6; b++)
            for (int c = 0; c <= 6; c++) {
                const int n = a * a + b * b + c * c;
                if (n >= 36) continue;
                const bool counts = n <= 30 && !class_432(a, b, c);
                const int lo = (a ? (a + 1) * (a + 1) : 0) + (b ? (b + 1) * (b + 1) : 0) + (c ? (c + 1) * (c + 1) : 0);
                const int hi = (a + 1) * (a + 1) + (b + 1) * (b + 1) + (c + 1) * (c + 1);
                const int R2 = VRT_DEPTH_FIELD_RADIUS * VRT_DEPTH_FIELD_RADIUS;
                if (counts ? hi > R2 : lo <= R2) return false;
            }
    return true;
}
static_assert(classes_match_ball(), "the distance classes are those of the radius-7 ball");

// The squared distances kept, nearest first: index 0 stands for n < 4 (the
// voxel's word is left as it was, :244-249), then each n with its own word
// (kFieldLevels of them, FieldWords), then kFieldNone: no class found, -6.
constexpr int kLevelN[kFieldLevels] = {4,  5,  6,  8,  9,  10, 11, 12, 13, 14, 16, 17,
                                       18, 19, 20, 21, 22, 24, 25, 26, 27, 29, 30};
constexpr int level_of(int n) {
    if (n < 4) return 0;
    for (int k = 0; k < kFieldLevels; k++)
        if (kLevelN[k] == n) return k + 1;
    return -1;
}

// The planar distances m = a^2+b^2 <= 30, in the order in which a row's masks
// E_m lie in LDS; entry 16 is the part of m = 25 from (5, 0) and (0, 5) alone
// (what (4, 3) adds must not count two rows away: class (4, 3, 2)).
constexpr int kPlanar = 16;
constexpr int kPlanarM[kPlanar] = {0, 1, 2, 4, 5, 8, 9, 10, 13, 16, 17, 18, 20, 25, 26, 29};
constexpr int planar_of(int m) {
    for (int k = 0; k < kPlanar; k++)
        if (kPlanarM[k] == m) return k;
    return -1;
}
// Words per row of masks: 17 used; at a stride of 20 words the 16-byte reads
// of eight consecutive rows fall on distinct LDS banks.
constexpr int kPlanarStride = 20;

// LDS of a tile of 32 x TY x TZ voxels.  Rows of `s` hold the solidity of the
// 64 voxels from 16 before the tile (bit j is x0 - 16 + j), for y and z from
// 6 before the tile to 6 past it.
template <int TY, int TZ>
struct FieldTile {
    static constexpr int kRows = TY * TZ;
    static constexpr int SY = TY + 12, SZ = TZ + 12, DY = TY + 10, DZ = TZ + 10;
    union {
        struct {
            uint2 s[SZ * SY];
            uint2 sy[SZ * DY];
        };
        uint4 e[DZ * TY * (kPlanarStride / 4)];
    };
    union {
        struct {
            uint4 xa[DZ * DY];
            uint2 xb[DZ * DY];
        };
        uint32_t plane[kRows * 6];
    };
};

__device__ __forceinline__ uint32_t funnel(uint32_t hi, uint32_t lo, uint32_t shift) {
    return __builtin_amdgcn_alignbit(hi, lo, shift);
}

__device__ __forceinline__ uint4 or4(uint4 a, uint4 b) {
    return make_uint4(a.x | b.x, a.y | b.y, a.z | b.z, a.w | b.w);
}

// From the solidity rows in L.s (written by the caller, before a barrier) to
// the tile's result in `plane` (LDS; L.plane or elsewhere): for row
// r = z * TY + y, words 6 r to 6 r + 4 are bit planes of each voxel's level
// (0: keep the word, k: FieldWords::word[k]) and word 6 r + 5 the voxels whose
// word is kept (solid, or n < 4).  Every one of the NT threads calls it; it
// ends on a barrier.
template <int TY, int TZ, int NT>
__device__ __forceinline__ void field_tile(FieldTile<TY, TZ>& L, uint32_t* plane, int tid) {
    using T = FieldTile<TY, TZ>;
    static_assert(NT >= T::kRows, "one thread per row of the tile");
    // D: dilate along y, then z, then x; the masks X_a of each row
    for (int i = tid; i < T::SZ * T::DY; i += NT) {
        const int r = (i / T::DY) * T::SY + i % T::DY;
        const uint2 a = L.s[r], b = L.s[r + 1], c = L.s[r + 2];
        L.sy[i] = make_uint2(a.x | b.x | c.x, a.y | b.y | c.y);
    }
    // the tile's own solidity, before its rows are overwritten
    uint32_t solid = 0;
    if (tid < T::kRows) {
        const uint2 v = L.s[(tid / TY + 6) * T::SY + tid % TY + 6];
        solid = funnel(v.y, v.x, 16);
    }
    __syncthreads();
    for (int i = tid; i < T::DZ * T::DY; i += NT) {
        const uint2 a = L.sy[i], b = L.sy[i + T::DY], c = L.sy[i + 2 * T::DY];
        const uint32_t lo = a.x | b.x | c.x, hi = a.y | b.y | c.y;
        const uint32_t dlo = lo | (lo << 1) | funnel(hi, lo, 1);
        const uint32_t dhi = hi | (hi >> 1) | funnel(hi, lo, 31);
        auto at = [&](int k) { return funnel(dhi, dlo, 16 - k) | funnel(dhi, dlo, 16 + k); };
        L.xa[i] = make_uint4(funnel(dhi, dlo, 16), at(1), at(2), at(3));
        L.xb[i] = make_uint2(at(4), at(5));
    }
    __syncthreads();
    for (int i = tid; i < T::DZ * TY; i += NT) {
        const int r = (i / TY) * T::DY + i % TY + kFieldReach;
        const uint4 a0 = L.xa[r];
        const uint2 b0 = L.xb[r];
        const uint4 a1 = or4(L.xa[r - 1], L.xa[r + 1]), a2 = or4(L.xa[r - 2], L.xa[r + 2]),
                    a3 = or4(L.xa[r - 3], L.xa[r + 3]), a4 = or4(L.xa[r - 4], L.xa[r + 4]),
                    a5 = or4(L.xa[r - 5], L.xa[r + 5]);
        const uint2 m1 = L.xb[r - 1], p1 = L.xb[r + 1], m2 = L.xb[r - 2], p2 = L.xb[r + 2];
        const uint32_t b3 = L.xb[r - 3].x | L.xb[r + 3].x;
        const uint32_t e25a = b0.y | a5.x;
        uint4* e = L.e + i * (kPlanarStride / 4);
        e[0] = make_uint4(a0.x, a0.y | a1.x, a1.y, a0.z | a2.x);                                // 0 1 2 4
        e[1] = make_uint4(a1.z | a2.y, a2.z, a0.w | a3.x, a1.w | a3.y);                         // 5 8 9 10
        e[2] = make_uint4(a2.w | a3.z, b0.x | a4.x, m1.x | p1.x | a4.y, a3.w);                  // 13 16 17 18
        e[3] = make_uint4(m2.x | p2.x | a4.z, e25a | b3 | a4.w, m1.y | p1.y | a5.y,             // 20 25 26
                          m2.y | p2.y | a5.z);                                                  // 29
        e[4].x = e25a;
    }
    __syncthreads();
    if (tid < T::kRows) {
        uint32_t t[kFieldLevels + 1] = {};
        // rows at +-c along z; e4 is read only where m = 25 must leave (4, 3) out
        auto add = [&](auto cc, const uint4* e) {
            constexpr int c = decltype(cc)::value;
            uint32_t m[kPlanar];
#pragma unroll
            for (int q = 0; q < 4; q++) {
                if (kPlanarM[4 * q] + c * c > 30) continue;
                const uint4 v = e[q];
                m[4 * q] = v.x;
                m[4 * q + 1] = v.y;
                m[4 * q + 2] = v.z;
                m[4 * q + 3] = v.w;
            }
            if (c == 2) m[planar_of(25)] = e[4].x;
#pragma unroll
            for (int k = 0; k < kPlanar; k++) {
                const int n = kPlanarM[k] + c * c;
                if (n > 30) continue;
                if (n == 29 && (c == 3 || c == 4)) continue;  // (4, 2) at 3 and (3, 2) at 4: class (4, 3, 2)
                t[level_of(n)] |= m[k];
            }
        };
        const uint4* e = L.e + ((tid / TY + kFieldReach) * TY + tid % TY) * (kPlanarStride / 4);
        constexpr int kZ = TY * (kPlanarStride / 4);
        add(std::integral_constant<int, 0>{}, e);
        add(std::integral_constant<int, 1>{}, e - kZ);
        add(std::integral_constant<int, 1>{}, e + kZ);
        add(std::integral_constant<int, 2>{}, e - 2 * kZ);
        add(std::integral_constant<int, 2>{}, e + 2 * kZ);
        add(std::integral_constant<int, 3>{}, e - 3 * kZ);
        add(std::integral_constant<int, 3>{}, e + 3 * kZ);
        add(std::integral_constant<int, 4>{}, e - 4 * kZ);
        add(std::integral_constant<int, 4>{}, e + 4 * kZ);
        add(std::integral_constant<int, 5>{}, e - 5 * kZ);
        add(std::integral_constant<int, 5>{}, e + 5 * kZ);
        // Level of a voxel = the number of levels not reached, a sorted list
        // of flags ~t[0], ~t[1], ... once t is made cumulative: bit j of that
        // count is the parity of the flags at 2^j - 1, 2 * 2^j - 1, ...
#pragma unroll
        for (int k = 1; k <= kFieldLevels; k++) t[k] |= t[k - 1];
        uint32_t p0 = 0, p1 = 0, p2 = 0;
#pragma unroll
        for (int k = 0; k <= kFieldLevels; k++) p0 ^= t[k];
#pragma unroll
        for (int k = 1; k <= kFieldLevels; k += 2) p1 ^= t[k];
#pragma unroll
        for (int k = 3; k <= kFieldLevels; k += 4) p2 ^= t[k];
        static_assert(kFieldLevels == 23, "24 flags: even counts for planes 0-2, three for plane 3, one for plane 4");
        uint32_t* p = plane + tid * 6;
        p[0] = p0;
        p[1] = p1;
        p[2] = p2;
        p[3] = ~(t[7] ^ t[15] ^ t[23]);
        p[4] = ~t[15];
        p[5] = solid | t[0];
    }
    __syncthreads();
}

// Level of the voxel at bit b of the row whose planes are at p.
__device__ __forceinline__ uint32_t level_at(const uint32_t p[5], uint32_t b) {
    uint32_t v = 0;
#pragma unroll
    for (int k = 0; k < 5; k++) v |= __builtin_amdgcn_ubfe(p[k], b, 1) << k;
    return v;
}

// Four voxels of a row, at any word of the grid.
typedef int32_t vox4 __attribute__((ext_vector_type(4), aligned(4)));

}  // namespace dev
}  // namespace vrt
