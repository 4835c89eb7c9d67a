// vrt_edit.hip — depth field and voxel edits on the device.
//
// fixDepthField (src/render.cpp:226-253) gives an empty voxel (word < 0) the
// largest table distance d* over its SOLID neighbours with d* > -6 (strict,
// :240), and then: d* > -2 -> the word is left as it was (:244-249);
// -6 < d* <= -2 -> the bits of d*; no such neighbour -> the bits of -6.0f.
// The result depends only on which neighbours are solid, and a jump word is
// negative (never solid), so every voxel of a region can be fixed in
// parallel, in place, with the same result as the reference's sequential
// loops.  d* is computed on bit masks, 32 voxels at a time (vrt_field.h).
#include <hip/hip_runtime.h>

#include <algorithm>

#include "vrt_field.h"
#include "vrt_internal.h"

namespace vrt {

namespace {

// Solidity bitmap of the grid: row (y, z) is W words, bit x + 16 of the row is
// voxel x (bits of x < 0 and x >= X are 0), so the 64 voxels from 16 before x0
// = 32 k are words k and k + 1 of their row.  A lane reads four voxels (16
// bytes) of each of kBitRows rows, all loads in flight together; eight lanes
// make one word.  Memory bound: 1 GiB in 242 us (4.4 TB/s); one voxel per lane
// with one ballot per row segment, 723 us.
constexpr int kBitRows = 4;
__global__ void __launch_bounds__(256) k_solid_bits(GridDesc g, uint32_t* __restrict__ bits, uint32_t W,
                                                    uint64_t rows) {
    const uint32_t Q = W * 8;  // quads of four voxels per row, a multiple of 8: eight lanes share a row
    const uint64_t base = (uint64_t)blockIdx.x * 256;
    const uint64_t rg0 = base / Q;
    const uint32_t q0 = (uint32_t)(base % Q) + threadIdx.x;
    const uint32_t q = q0 % Q;
    const uint64_t r0 = (rg0 + q0 / Q) * kBitRows;
    const int64_t x = (int64_t)q * 4 - 16;
    uint32_t m[kBitRows] = {};
    if (x >= 0 && x + 3 < (int64_t)g.X) {
        dev::vox4 v[kBitRows];
#pragma unroll
        for (int j = 0; j < kBitRows; j++)
            if (r0 + j < rows) v[j] = *(const dev::vox4*)(g.vox + (r0 + j) * g.X + x);
            else v[j] = -1;
#pragma unroll
        for (int j = 0; j < kBitRows; j++)
            m[j] = (v[j].x >= 0 ? 1u : 0u) | (v[j].y >= 0 ? 2u : 0u) | (v[j].z >= 0 ? 4u : 0u) |
                   (v[j].w >= 0 ? 8u : 0u);
    } else {
        for (int j = 0; j < kBitRows; j++)
            for (int k = 0; k < 4; k++)
                if (r0 + j < rows && x + k >= 0 && x + k < (int64_t)g.X && g.vox[(r0 + j) * g.X + x + k] >= 0)
                    m[j] |= 1u << k;
    }
#pragma unroll
    for (int j = 0; j < kBitRows; j++) {
        uint32_t w = m[j] << (4 * (threadIdx.x & 7));
        w |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)w, 0xB1, 0xf, 0xf, true);   // lane ^ 1
        w |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)w, 0x4E, 0xf, 0xf, true);   // lane ^ 2
        w |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)w, 0x141, 0xf, 0xf, true);  // the other four of eight
        if ((threadIdx.x & 7) == 0 && r0 + j < rows) bits[(r0 + j) * W + (q >> 3)] = w;
    }
}

// Whole-grid build: one workgroup per kTileRun tiles of 32 x 8 x 16 voxels side
// by side in x, whose distances come from the bitmap (field_tile), one tile
// after the other.  Tiles without a solid voxel in reach take -6 and tiles of
// solid voxels keep their words, both without that work.  The words then go to
// the grid and, with the words that are kept, to the padded render copy, so the
// copy needs no pass of its own; only words that are kept are read.
//
// Bound by memory, the writes above all.  1024x256x1024 (1 GiB): 0.68 ms, where
// a table scan per voxel took 7.18 ms and 0.38 ms more to copy the grid; the
// 2.1 GB that it must move take 0.45 ms at the rate of a large copy.  The
// copy's rows start anywhere in a 128-byte line, so a run's two ends write
// parts of lines: runs of one tile (128 bytes) took 0.81 ms.  (Rows padded to
// whole lines gained 5% there and cost 1% of every frame.)  Workgroup b runs on
// XCD b mod 8 and takes the tiles of that eighth of the grid, so neighbours
// share the L2 that holds the bitmap's rows and the lines between two runs:
// writing such runs without that order took twice as long.
constexpr int kTileY = 8, kTileZ = 16, kTileThreads = kTileY * kTileZ, kTileRun = 4;
__global__ void __launch_bounds__(kTileThreads) k_field_tiles(GridDesc g, GridDesc r, FieldWords words,
                                                              const uint32_t* __restrict__ bits, uint32_t W,
                                                              uint32_t runs, uint32_t ny, uint32_t total) {
    using Tile = dev::FieldTile<kTileY, kTileZ>;
    __shared__ Tile L;
    __shared__ uint32_t planes[kTileRun][kTileThreads * 6];
    __shared__ int32_t word[kFieldLevels + 2];
    const uint32_t run = (blockIdx.x % 8) * (gridDim.x / 8) + blockIdx.x / 8;
    if (run >= total) return;
    const int32_t tid = threadIdx.x;
    const uint32_t k0 = (run % runs) * kTileRun;  // the run's first bitmap word
    const int32_t y0 = (int32_t)((run / runs) % ny) * kTileY, z0 = (int32_t)(run / (runs * ny)) * kTileZ;
    const int32_t tiles = (int32_t)min((uint32_t)kTileRun, W - 1 - k0);
    if (tid < kFieldLevels + 2) word[tid] = words.word[tid];
    // bitmap rows of a tile, two words each, kRowSteps rows per thread
    constexpr int kRowSteps = (Tile::SZ * Tile::SY + kTileThreads - 1) / kTileThreads;
    uint2 rows[kRowSteps];
    auto load_rows = [&](int32_t t) {
#pragma unroll
        for (int j = 0; j < kRowSteps; j++) {
            const int32_t i = tid + j * kTileThreads;
            const int32_t gy = y0 - 6 + i % Tile::SY, gz = z0 - 6 + i / Tile::SY;
            rows[j] = make_uint2(0, 0);
            if (i < Tile::SZ * Tile::SY && gy >= 0 && gz >= 0 && (uint32_t)gy < g.Y && (uint32_t)gz < g.Z) {
                const uint32_t* rw = bits + ((uint64_t)gy + (uint64_t)g.Y * (uint64_t)gz) * W + k0 + t;
                rows[j] = make_uint2(rw[0], rw[1]);
            }
        }
    };
    load_rows(0);
    for (int32_t t = 0; t < tiles; t++) {
        bool any = false, full = true;
#pragma unroll
        for (int j = 0; j < kRowSteps; j++) {
            const int32_t i = tid + j * kTileThreads;
            const int32_t y = i % Tile::SY - 6, z = i / Tile::SY - 6;
            if (i >= Tile::SZ * Tile::SY) continue;
            L.s[i] = rows[j];
            any |= (rows[j].x | rows[j].y) != 0u;
            if (y >= 0 && y < kTileY && z >= 0 && z < kTileZ)
                full &= dev::funnel(rows[j].y, rows[j].x, 16) == 0xffffffffu;
        }
        if (t + 1 < tiles) load_rows(t + 1);  // in flight during this tile's work
        any = __syncthreads_or(any) != 0;
        full = any && __syncthreads_and(full) != 0;
        if (any && !full) {
            dev::field_tile<kTileY, kTileZ, kTileThreads>(L, planes[t], tid);
        } else {
            uint32_t* p = planes[t] + tid * 6;
#pragma unroll
            for (int k = 0; k < 5; k++) p[k] = !full && ((kFieldLevels + 1) >> k & 1) ? 0xffffffffu : 0u;
            p[5] = full ? 0xffffffffu : 0u;
            __syncthreads();
        }
    }
    // four voxels per lane, the run's lanes side by side: 512 bytes of a row
    constexpr int kLanes = 8 * kTileRun, kSteps = 8;
    const int32_t lane = tid % kLanes, x = (int32_t)(k0 * 32) + 4 * lane;
    if (lane >= 8 * tiles || (int64_t)x >= (int64_t)g.X) return;
    const uint32_t* plane = planes[lane / 8];
    const uint32_t b = 4 * (lane % 8);
    auto cell = [&](const GridDesc& d, int row) {
        return d.origin + (uint64_t)x + (uint64_t)d.SX * (uint64_t)(y0 + row % kTileY) +
               d.SXY * (uint64_t)(z0 + row / kTileY);
    };
    auto inside = [&](int row) {
        return (uint32_t)(y0 + row % kTileY) < g.Y && (uint32_t)(z0 + row / kTileY) < g.Z;
    };
    for (int row0 = tid / kLanes; row0 < Tile::kRows; row0 += kSteps * (kTileThreads / kLanes)) {
        if ((int64_t)x + 3 < (int64_t)g.X) {
            dev::vox4 v[kSteps];
#pragma unroll
            for (int j = 0; j < kSteps; j++) {
                const int row = row0 + j * (kTileThreads / kLanes);
                if (inside(row) && ((plane[row * 6 + 5] >> b) & 15u)) v[j] = *(const dev::vox4*)(g.vox + cell(g, row));
            }
#pragma unroll
            for (int j = 0; j < kSteps; j++) {
                const int row = row0 + j * (kTileThreads / kLanes);
                if (!inside(row)) continue;
                const uint32_t* p = plane + row * 6;
                const uint32_t keep = (p[5] >> b) & 15u;
                const uint32_t pl[5] = {p[0], p[1], p[2], p[3], p[4]};
                dev::vox4 o;
                o.x = keep & 1u ? v[j].x : word[dev::level_at(pl, b)];
                o.y = keep & 2u ? v[j].y : word[dev::level_at(pl, b + 1)];
                o.z = keep & 4u ? v[j].z : word[dev::level_at(pl, b + 2)];
                o.w = keep & 8u ? v[j].w : word[dev::level_at(pl, b + 3)];
                if (keep != 15u) *(dev::vox4*)(g.vox + cell(g, row)) = o;
                *(dev::vox4*)(r.vox + cell(r, row)) = o;
            }
        } else {
            for (int j = 0; j < kSteps; j++) {
                const int row = row0 + j * (kTileThreads / kLanes);
                if (!inside(row)) continue;
                const uint32_t* p = plane + row * 6;
                const uint32_t pl[5] = {p[0], p[1], p[2], p[3], p[4]};
                for (int k = 0; k < 4 && (int64_t)x + k < (int64_t)g.X; k++) {
                    int32_t* w = g.vox + cell(g, row) + k;
                    int32_t o;
                    if (p[5] >> (b + k) & 1u) o = *w;
                    else *w = o = word[dev::level_at(pl, b + k)];
                    r.vox[cell(r, row) + k] = o;
                }
            }
        }
    }
}

// destroyVoxel and fixDepthField over the box of w x h x d voxels at
// (x0, y0, z0) (inside the grid), in one pass: voxels with
// (x-cx)^2+(y-cy)^2+(z-cz)^2 < cr^2 become -1 (cr <= 0: none), then the empty
// ones within sr^2 of the centre (sr < 0: the whole box) are fixed, and every
// voxel of the box goes to the render copy r (r.vox null: no copy).
//
// One workgroup of NT threads per tile of 32 x 8 x 8 voxels of the box.  A wave
// reads a row of its surroundings with one load (64 voxels; only those within
// reach) and makes the bitmap's row by a ballot, kEditRows rows in flight at
// once; field_tile does the rest.
// Workgroups of one launch may read a voxel that another has already carved
// or fixed: it is not solid before or after (the carve test is applied to
// what is read), and solid voxels outside the carve are never written.
// Latency bound (launch, two or four rounds of loads, five barriers): eight
// removeSpheres of radius 1-8 one after another 35 us (114 us when the device
// was idle before), against 112 and 341 us for three launches each (carve,
// per-voxel table scans over the box, copy of the box).
constexpr int kEditY = 8, kEditZ = 8;
constexpr int kEditRows = 25;
template <int NT>
__global__ void __launch_bounds__(NT) k_edit_box(GridDesc g, GridDesc r, FieldWords words, int32_t x0, int32_t y0,
                                                 int32_t z0, int32_t w, int32_t h, int32_t d, uint32_t nbx,
                                                 uint32_t nby, int32_t cx, int32_t cy, int32_t cz, int32_t sr,
                                                 int32_t cr) {
    using Tile = dev::FieldTile<kEditY, kEditZ>;
    __shared__ Tile L;
    __shared__ int32_t word[kFieldLevels + 2];
    const int32_t tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    if (tid < kFieldLevels + 2) word[tid] = words.word[tid];
    const uint32_t b = blockIdx.x;
    // the tile's corner in the box and the extent of the box in the tile
    const int32_t ox = (int32_t)(b % nbx) * 32, oy = (int32_t)((b / nbx) % nby) * kEditY,
                  oz = (int32_t)(b / (nbx * nby)) * kEditZ;
    const int32_t tw = w - ox < 32 ? w - ox : 32;
    const int32_t bx = x0 + ox, by = y0 + oy, bz = z0 + oz;
    auto dist2 = [&](int32_t x, int32_t y, int32_t z) {
        const int32_t ex = x - cx, ey = y - cy, ez = z - cz;
        return ex * ex + ey * ey + ez * ez;
    };
    auto carved = [&](int32_t x, int32_t y, int32_t z) { return cr > 0 && dist2(x, y, z) < cr * cr; };
    // this thread's voxels: 32 along x, kCells rows apart in steps
    constexpr int kCells = 32 * kEditY * kEditZ / NT;
    const int32_t x = bx + (tid & 31);
    int32_t was[kCells], old[kCells];
    bool mine[kCells], fix = false;
#pragma unroll
    for (int j = 0; j < kCells; j++) {
        const int32_t row = (tid >> 5) + j * (NT / 32);
        const int32_t ly = row % kEditY, lz = row / kEditY;
        mine[j] = ((tid & 31) < tw) & (oy + ly < h) & (oz + lz < d);
        was[j] = mine[j] ? g.vox[(uint64_t)x + g.X * (uint64_t)(by + ly) + g.XY * (uint64_t)(bz + lz)] : 0;
    }
    // rows within 6 voxels of the tile, x from 16 before it
    constexpr int kRows = Tile::SY * Tile::SZ, kWaves = NT / 64;
    const int32_t gx = bx - 16 + lane;
    const bool in_x = lane >= 10 && lane < 22 + tw && gx >= 0 && (uint32_t)gx < g.X;
    for (int i0 = wave; i0 < kRows; i0 += kWaves * kEditRows) {
        int32_t v[kEditRows];
#pragma unroll
        for (int j = 0; j < kEditRows; j++) {
            const int32_t i = i0 + j * kWaves;
            const int32_t gy = by - 6 + i % Tile::SY, gz = bz - 6 + i / Tile::SY;
            v[j] = -1;
            if (i < kRows && gy >= 0 && gz >= 0 && (uint32_t)gy < g.Y && (uint32_t)gz < g.Z && in_x)
                v[j] = g.vox[(uint64_t)gx + g.X * (uint64_t)gy + g.XY * (uint64_t)gz];
        }
#pragma unroll
        for (int j = 0; j < kEditRows; j++) {
            const int32_t i = i0 + j * kWaves;
            const uint64_t m = __ballot(v[j] >= 0 && !carved(gx, by - 6 + i % Tile::SY, bz - 6 + i / Tile::SY));
            if (lane == 0 && i < kRows) L.s[i] = make_uint2((uint32_t)m, (uint32_t)(m >> 32));
        }
    }
#pragma unroll
    for (int j = 0; j < kCells; j++) {
        const int32_t row = (tid >> 5) + j * (NT / 32);
        const int32_t y = by + row % kEditY, z = bz + row / kEditY;
        old[j] = mine[j] && carved(x, y, z) ? -1 : was[j];
        fix |= mine[j] && old[j] < 0 && (sr < 0 || dist2(x, y, z) < sr * sr);
    }
    const bool any = __syncthreads_or(fix) != 0;
    if (any) dev::field_tile<kEditY, kEditZ, NT>(L, L.plane, tid);
#pragma unroll
    for (int j = 0; j < kCells; j++) {
        if (!mine[j]) continue;
        const int32_t row = (tid >> 5) + j * (NT / 32);
        const int32_t y = by + row % kEditY, z = bz + row / kEditY;
        int32_t now = old[j];
        if (any && now < 0 && (sr < 0 || dist2(x, y, z) < sr * sr)) {
            const uint32_t* p = L.plane + row * 6;
            const uint32_t pl[5] = {p[0], p[1], p[2], p[3], p[4]};
            if (!(p[5] >> (tid & 31) & 1u)) now = word[dev::level_at(pl, tid & 31)];
        }
        if (now != was[j]) g.vox[(uint64_t)x + g.X * (uint64_t)y + g.XY * (uint64_t)z] = now;
        if (r.vox) r.vox[r.origin + (uint64_t)x + (uint64_t)r.SX * (uint64_t)y + r.SXY * (uint64_t)z] = now;
    }
}

// One voxel of the grid and of the render copy.
__global__ void k_set_voxel(int32_t* vox, int32_t* copy, int32_t v, int32_t* top, int32_t y) {
    if (threadIdx.x == 0) {
        *vox = v;
        *copy = v;
        if (v >= 0 && top) atomicMax(top, y);
    }
}

// Words [first, first + n) of the box of nx x ny x ... voxels at (x0, y0, z0),
// x fastest, from `src` (pinned host memory, read over the link) into the grid
// and the render copy; `top`: the highest y of a solid voxel among them.
__global__ void __launch_bounds__(256) k_put_box(GridDesc g, GridDesc r, const int32_t* __restrict__ src,
                                                 uint64_t first, uint32_t n, uint32_t nx, uint32_t ny, uint32_t x0,
                                                 uint32_t y0, uint32_t z0, int32_t top) {
    const uint32_t i = blockIdx.x * 256u + threadIdx.x;
    if (i == 0 && top > *g.top) *g.top = top;
    if (i >= n) return;
    const int32_t v = src[i];
    const uint64_t k = first + i, row = k / nx;
    const uint64_t x = x0 + k % nx, y = y0 + row % ny, z = z0 + row / ny;
    g.vox[x + g.X * y + g.XY * z] = v;
    r.vox[r.origin + x + (uint64_t)r.SX * y + r.SXY * z] = v;
}

__global__ void k_set_word(int32_t* p, int32_t v) {
    if (threadIdx.x == 0) *p = v;
}

// Highest y with a solid voxel over rows (y, z) of the box [x0, x0+w) x
// [y0, y0+h) x [z0, z0+d): a wave reads a row's words with its 64 lanes, keeps
// the highest y of its rows with any solid word and raises *top once.
__global__ void __launch_bounds__(256) k_solid_top(GridDesc g, int32_t x0, int32_t w, int32_t y0, int32_t h,
                                                    int32_t z0, int64_t rows, int32_t* top) {
    const int32_t lane = threadIdx.x & 63;
    const int64_t waves = (int64_t)gridDim.x * (blockDim.x >> 6);
    int32_t best = -1;
    for (int64_t r = (int64_t)blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6); r < rows; r += waves) {
        const int32_t y = y0 + (int32_t)(r % h);
        const int32_t z = z0 + (int32_t)(r / h);
        if (y <= best) continue;
        const int32_t* row = g.vox + (uint64_t)g.X * (uint64_t)y + g.XY * (uint64_t)z + (uint64_t)x0;
        bool any = false;
        for (int32_t x = lane; x < w; x += 64) any |= row[x] >= 0;
        if (__builtin_amdgcn_ballot_w64(any) != 0) best = y;
    }
    if (lane == 0 && best >= 0) atomicMax(top, best);
}

// The whole grid in one pass: words from `src` (the grid itself, or a level
// elsewhere on the device) into the render copy and, when they come from
// elsewhere, the grid; *top is raised to the highest y of a solid voxel.  A
// lane moves four voxels of each of kLoadRows rows, all loads in flight
// together; a block raises *top only when it holds something higher than it
// already says (one atomic per wave on that word took 0.33 ms by itself).
// Memory bound: 1 GiB in 0.62 ms (3.2 GB, 5.2 TB/s), against 1.20 ms for three
// passes (copy 0.49, solid top 0.33, render copy 0.38).
constexpr int kLoadRows = 4;
__global__ void __launch_bounds__(256) k_load_grid(GridDesc g, GridDesc r, const int32_t* src, uint64_t rows,
                                                   uint32_t Q, uint64_t blocks) {
    __shared__ int32_t best;
    int32_t high = -1;
    for (uint64_t b = blockIdx.x; b < blocks; b += gridDim.x) {
        // quads of four voxels, Q per row; row (y, z) is y + Y * z
        const uint64_t base = b * 256, rg0 = base / Q;
        const uint32_t q0 = (uint32_t)(base % Q) + threadIdx.x;
        const uint64_t row0 = (rg0 + q0 / Q) * kLoadRows;
        const uint32_t x = q0 % Q * 4;
        const uint64_t zb = rg0 * kLoadRows / g.Y;
        uint32_t y = (uint32_t)(rg0 * kLoadRows - zb * g.Y) + q0 / Q * kLoadRows;
        uint64_t z = zb + y / g.Y;
        y %= g.Y;
        const uint32_t n = x + 4 <= g.X ? 4 : g.X - x;
        dev::vox4 v[kLoadRows];
#pragma unroll
        for (int j = 0; j < kLoadRows; j++) {
            const int32_t* p = src + (row0 + j) * g.X + x;
            v[j] = -1;
            if (row0 + j >= rows) continue;
            if (n == 4) {
                v[j] = *(const dev::vox4*)p;
            } else {
                v[j].x = p[0];
                if (n > 1) v[j].y = p[1];
                if (n > 2) v[j].z = p[2];
            }
        }
#pragma unroll
        for (int j = 0; j < kLoadRows; j++) {
            if (row0 + j < rows) {
                int32_t* c = r.vox + (r.origin + x + (uint64_t)r.SX * y + r.SXY * z);
                int32_t* d = g.vox + (row0 + j) * g.X + x;
                if (n == 4) {
                    *(dev::vox4*)c = v[j];
                    if (src != g.vox) *(dev::vox4*)d = v[j];
                } else {
                    for (uint32_t k = 0; k < n; k++) {
                        const int32_t w = k == 0 ? v[j].x : (k == 1 ? v[j].y : v[j].z);
                        c[k] = w;
                        if (src != g.vox) d[k] = w;
                    }
                }
                if ((v[j].x & v[j].y & v[j].z & v[j].w) >= 0) high = max(high, (int32_t)y);
            }
            if (++y == g.Y) {
                y = 0;
                z++;
            }
        }
    }
    if (threadIdx.x == 0) best = __atomic_load_n(g.top, __ATOMIC_RELAXED);
    __syncthreads();
    const int32_t seen = best;
    __syncthreads();
    if (high > seen) atomicMax(&best, high);
    __syncthreads();
    if (threadIdx.x == 0 && best > seen) atomicMax(g.top, best);
}

// Grid copy, 16 bytes per lane per step (a plain streaming copy of known size).
__global__ void __launch_bounds__(256) k_copy(int4* __restrict__ dst, const int4* __restrict__ src, uint64_t n16,
                                               int32_t* __restrict__ dst_tail, const int32_t* __restrict__ src_tail,
                                               uint32_t tail) {
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    const uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    for (uint64_t i = t; i < n16; i += stride) dst[i] = src[i];
    if (t < tail) dst_tail[t] = src_tail[t];
}

// One wave per x-row segment of the box (four rows per workgroup, the y and z
// loops covering boxes taller or deeper than the launch); each lane moves the
// words lane, lane+64, ... of its row, four loads in flight.
__global__ void __launch_bounds__(256) k_copy_box(GridDesc src, GridDesc dst, int64_t x0, int64_t y0, int64_t z0,
                                                  uint32_t nx, uint32_t ny, uint32_t nz) {
    const uint32_t lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    for (uint32_t z = blockIdx.z; z < nz; z += gridDim.z) {
        for (uint32_t y = blockIdx.y * 4 + w; y < ny; y += gridDim.y * 4) {
            const uint64_t gy = (uint64_t)(y0 + y), gz = (uint64_t)(z0 + z);
            const int32_t* __restrict__ s = src.vox + (src.origin + (uint64_t)x0 + src.SX * gy + src.SXY * gz);
            int32_t* __restrict__ d = dst.vox + (dst.origin + (uint64_t)x0 + dst.SX * gy + dst.SXY * gz);
            uint32_t x = lane;
            for (; x + 192 < nx; x += 256) {
                const int32_t a = s[x], b = s[x + 64], c = s[x + 128], e = s[x + 192];
                d[x] = a;
                d[x + 64] = b;
                d[x + 128] = c;
                d[x + 192] = e;
            }
            for (; x < nx; x += 64) d[x] = s[x];
        }
    }
}

__global__ void __launch_bounds__(256) k_fill(int32_t* p, uint64_t n, int32_t v) {
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) p[i] = v;
}

__global__ void __launch_bounds__(64) k_fill_corner(GridDesc r) {
    const uint32_t i = threadIdx.x, z = blockIdx.x;
    if (i < kGuard * kGuard) r.vox[i % kGuard + (uint64_t)r.SX * (i / kGuard) + r.SXY * z] = kGuardCorner;
}

// Clip [lo, hi) to [0, n).
inline void clip(int64_t& lo, int64_t& hi, int64_t n) {
    if (lo < 0) lo = 0;
    if (hi > n) hi = n;
}

}  // namespace

int launch_edit_box(const GridDesc& g, const GridDesc& render, const FieldWords& words, int64_t x0, int64_t y0,
                    int64_t z0, int64_t x1, int64_t y1, int64_t z1, int32_t cx, int32_t cy, int32_t cz, int32_t sr,
                    int32_t cr, hipStream_t s) {
    clip(x0, x1, g.X);
    clip(y0, y1, g.Y);
    clip(z0, z1, g.Z);
    if (x1 <= x0 || y1 <= y0 || z1 <= z0) return VRT_OK;
    const int64_t w = x1 - x0, h = y1 - y0, d = z1 - z0;
    const int64_t nbx = (w + 31) / 32, nby = (h + kEditY - 1) / kEditY, nbz = (d + kEditZ - 1) / kEditZ;
    // An edit without a render copy is a server's, beside batches that fill the
    // device: a workgroup of 512 threads waits there until some CU has two
    // wave slots free on each SIMD (24 requests with 2 edits: 2801 us, with 256
    // threads 2777).  On a device with room 512 threads are faster (above: 35
    // and 114 us, with 256 threads 51 and 165).
    const int threads = render.vox ? 512 : 256;
    // a launch holds fewer than 2^32 threads: deep boxes go in slabs along z
    const int64_t most = ((int64_t)1 << 32) / threads - 1;
    if (nbx * nby > most) return fail(VRT_ERR_INVALID, "box too large");
    const int64_t slab = most / (nbx * nby);
    for (int64_t k = 0; k < nbz; k += slab) {
        const dim3 blocks((uint32_t)(nbx * nby * std::min(slab, nbz - k)));
        auto* kernel = render.vox ? k_edit_box<512> : k_edit_box<256>;
        hipLaunchKernelGGL(kernel, blocks, dim3(threads), 0, s, g, render, words, (int32_t)x0, (int32_t)y0,
                           (int32_t)(z0 + k * kEditZ), (int32_t)w, (int32_t)h, (int32_t)(d - k * kEditZ),
                           (uint32_t)nbx, (uint32_t)nby, cx, cy, cz, sr, cr);
        VRT_HIP(hipGetLastError());
    }
    return VRT_OK;
}

uint32_t solid_bits_words(const GridDesc& g) { return (g.X + 31u) / 32u + 1u; }

int launch_build_depth_field(const GridDesc& g, const GridDesc& render, const FieldWords& words, uint32_t* bits,
                             hipStream_t s) {
    const uint32_t W = solid_bits_words(g);
    const uint64_t rows = (uint64_t)g.Y * g.Z;
    const uint64_t bit_blocks = ((rows + kBitRows - 1) / kBitRows * (W * 8ull) + 255) / 256;
    const uint64_t runs = (g.X + 32ull * kTileRun - 1) / (32 * kTileRun), ny = (g.Y + kTileY - 1ull) / kTileY, nz = (g.Z + kTileZ - 1ull) / kTileZ;
    const uint64_t total = runs * ny * nz;
    if (bit_blocks > 0x7fffffffull || runs * ny > 0x7ffffff0ull || total > 0x7ffffff0ull)
        return fail(VRT_ERR_INVALID, "grid too large for the build");
    hipLaunchKernelGGL(k_solid_bits, dim3((uint32_t)bit_blocks), dim3(256), 0, s, g, bits, W, rows);
    VRT_HIP(hipGetLastError());
    hipLaunchKernelGGL(k_field_tiles, dim3((uint32_t)((total + 7) / 8 * 8)), dim3(kTileThreads), 0, s, g, render, words,
                       bits, W, (uint32_t)runs, (uint32_t)ny, (uint32_t)total);
    VRT_HIP(hipGetLastError());
    return VRT_OK;
}

int launch_set_voxel(const GridDesc& g, const GridDesc& render, int32_t x, int32_t y, int32_t z, int32_t v,
                     hipStream_t s) {
    if (x < 0 || y < 0 || z < 0 || (uint32_t)x >= g.X || (uint32_t)y >= g.Y || (uint32_t)z >= g.Z)
        return fail(VRT_ERR_INVALID, "voxel out of range");
    auto at = [&](const GridDesc& d) {
        return d.vox + (d.origin + (uint64_t)x + (uint64_t)d.SX * (uint64_t)y + d.SXY * (uint64_t)z);
    };
    hipLaunchKernelGGL(k_set_voxel, dim3(1), dim3(64), 0, s, at(g), at(render), v, g.top, y);
    VRT_HIP(hipGetLastError());
    return VRT_OK;
}

int launch_load_grid(const GridDesc& g, const GridDesc& render, const int32_t* src, hipStream_t s) {
    if (!g.top) return fail(VRT_ERR_INVALID, "grid without a solid-top word");
    if ((uintptr_t)src & 15) return fail(VRT_ERR_INVALID, "copy buffers must be 16-byte aligned");
    const uint64_t rows = (uint64_t)g.Y * g.Z;
    const uint32_t Q = (g.X + 3u) / 4u;
    const uint64_t blocks = ((rows + kLoadRows - 1) / kLoadRows * Q + 255) / 256;
    hipLaunchKernelGGL(k_set_word, dim3(1), dim3(64), 0, s, g.top, -1);
    VRT_HIP(hipGetLastError());
    hipLaunchKernelGGL(k_load_grid, dim3((uint32_t)std::min<uint64_t>(blocks, 1u << 23)), dim3(256), 0, s, g, render,
                       src, rows, Q, blocks);
    VRT_HIP(hipGetLastError());
    return VRT_OK;
}

int launch_put_box(const GridDesc& g, const GridDesc& render, const int32_t* src, int64_t first, int64_t n, int64_t nx,
                   int64_t ny, int64_t x0, int64_t y0, int64_t z0, int32_t top, hipStream_t s) {
    if (n <= 0) return VRT_OK;
    if (n > 0x7fffffff) return fail(VRT_ERR_INVALID, "too many words in one piece");
    hipLaunchKernelGGL(k_put_box, dim3((uint32_t)((n + 255) / 256)), dim3(256), 0, s, g, render, src, (uint64_t)first,
                       (uint32_t)n, (uint32_t)nx, (uint32_t)ny, (uint32_t)x0, (uint32_t)y0, (uint32_t)z0, top);
    VRT_HIP(hipGetLastError());
    return VRT_OK;
}

int launch_solid_top(const GridDesc& g, int64_t x0, int64_t y0, int64_t z0, int64_t x1, int64_t y1, int64_t z1,
                     hipStream_t s) {
    if (!g.top) return fail(VRT_ERR_INVALID, "grid without a solid-top word");
    clip(x0, x1, g.X);
    clip(y0, y1, g.Y);
    clip(z0, z1, g.Z);
    if (x1 <= x0 || y1 <= y0 || z1 <= z0) return VRT_OK;
    const int64_t rows = (y1 - y0) * (z1 - z0);
    int64_t blocks = (rows + 3) / 4;  // 4 waves per block, one row each to start
    if (blocks > 8192) blocks = 8192;
    hipLaunchKernelGGL(k_solid_top, dim3((uint32_t)blocks), dim3(256), 0, s, g, (int32_t)x0, (int32_t)(x1 - x0),
                       (int32_t)y0, (int32_t)(y1 - y0), (int32_t)z0, rows, g.top);
    VRT_HIP(hipGetLastError());
    return VRT_OK;
}

int launch_copy(int32_t* dst, const int32_t* src, uint64_t n, hipStream_t s) {
    if (n == 0) return VRT_OK;
    if (((uintptr_t)dst | (uintptr_t)src) & 15) return fail(VRT_ERR_INVALID, "copy buffers must be 16-byte aligned");
    const uint64_t n16 = n / 4;
    const uint32_t tail = (uint32_t)(n % 4);
    uint64_t blocks = (n16 + 255) / 256;
    if (blocks > 8192) blocks = 8192;
    if (blocks == 0) blocks = 1;
    hipLaunchKernelGGL(k_copy, dim3((uint32_t)blocks), dim3(256), 0, s, (int4*)dst, (const int4*)src, n16,
                       dst + 4 * n16, src + 4 * n16, tail);
    VRT_HIP(hipGetLastError());
    return VRT_OK;
}

int launch_copy_box(const GridDesc& src, const GridDesc& dst, int64_t x0, int64_t y0, int64_t z0, int64_t nx,
                    int64_t ny, int64_t nz, hipStream_t s) {
    if (nx <= 0 || ny <= 0 || nz <= 0) return VRT_OK;
    if (x0 < 0 || y0 < 0 || z0 < 0 || x0 + nx > src.X || y0 + ny > src.Y || z0 + nz > src.Z || src.X != dst.X ||
        src.Y != dst.Y || src.Z != dst.Z)
        return fail(VRT_ERR_INVALID, "copy box outside the grid");
    const uint32_t by = (uint32_t)std::min<int64_t>((ny + 3) / 4, 65535), bz = (uint32_t)std::min<int64_t>(nz, 65535);
    hipLaunchKernelGGL(k_copy_box, dim3(1, by, bz), dim3(256), 0, s, src, dst, x0, y0, z0, (uint32_t)nx,
                       (uint32_t)ny, (uint32_t)nz);
    VRT_HIP(hipGetLastError());
    return VRT_OK;
}

int launch_fill(int32_t* p, uint64_t n, int32_t v, hipStream_t s) {
    if (n == 0) return VRT_OK;
    uint64_t blocks = (n + 255) / 256;
    if (blocks > 65536ull * 16) blocks = 65536ull * 16;
    hipLaunchKernelGGL(k_fill, dim3((uint32_t)blocks), dim3(256), 0, s, p, n, v);
    VRT_HIP(hipGetLastError());
    return VRT_OK;
}

int launch_fill_guard(const GridDesc& render, hipStream_t s) {
    if (int rc = launch_fill(render.vox, render.count, kGuardValue, s)) return rc;
    hipLaunchKernelGGL(k_fill_corner, dim3((uint32_t)(render.Z + 2 * kGuard)), dim3(64), 0, s, render);
    VRT_HIP(hipGetLastError());
    return VRT_OK;
}

}  // namespace vrt
