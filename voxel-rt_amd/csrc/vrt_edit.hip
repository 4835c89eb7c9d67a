// vrt_edit.hip — depth field and voxel edits on the device.
//
// fixDepthField (src/render.cpp:226-253) gives an empty voxel (word < 0) the
// largest table distance d* over its SOLID neighbours with d* > -6 (strict,
// :240), and then: d* > -2 -> the word is left as it was (:244-249);
// -6 < d* <= -2 -> the bits of d*; no such neighbour -> the bits of -6.0f.
// The result depends only on which neighbours are solid, and a jump word is
// negative (never solid), so every voxel of a region can be fixed in
// parallel, in place, with the same result as the reference's sequential
// loops.  Whole-grid builds compute d* on bit masks, 32 voxels at a time
// (vrt_field.h); boxes scan the table in order of decreasing distance, so the
// first solid neighbour found is d*.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "vrt_field.h"
#include "vrt_internal.h"

namespace vrt {

namespace {

constexpr int32_t kMinus6Bits = (int32_t)0xC0C00000;  // bits of -6.0f

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

constexpr int32_t kHalo = 7;
constexpr int32_t kSpan = 8 + 2 * kHalo;  // 22 cells per row of the neighbourhood

// fixDepthField's result for the voxel at (lx, ly, lz) of a brick whose
// 22x22x22 neighbourhood solidity is in `rows` (bit b of row (ry, rz) is
// x = lx - 7 + b).  The table is grouped by (distance, dy, dz): the first
// group with a solid neighbour gives d*, as the first solid entry of the
// sorted table would, and the group's dx mask (bit dx + 7) lines up with the
// row shifted right by lx.  Eight groups per step keep eight LDS reads in
// flight.
__device__ __forceinline__ int32_t scan_groups(const uint32_t* rows, const DepthTableDev& t, int32_t lx, int32_t ly,
                                               int32_t lz, int32_t old) {
    const int32_t my_row = (lz + kHalo) * kSpan + ly + kHalo;
    auto hits = [&](int32_t r) {
        const int32_t dy = ((r >> 16) & 31) - 8, dz = ((r >> 21) & 31) - 8;
        return ((rows[my_row + dz * kSpan + dy] >> lx) & (uint32_t)(r & 0x7fff)) != 0u;
    };
    int32_t found = -1;
    int32_t k = 0;
    for (; k + 8 <= t.n_rows; k += 8) {
        uint32_t m = 0;
#pragma unroll
        for (int j = 0; j < 8; j++) m |= (uint32_t)hits(t.rows[k + j]) << j;
        if (m) {
            found = k + __builtin_ctz(m);
            break;
        }
    }
    if (found < 0)
        for (; k < t.n_rows; k++)
            if (hits(t.rows[k])) {
                found = k;
                break;
            }
    if (found < 0) return kMinus6Bits;
    return found < t.n_rows_near ? old : __float_as_int(t.rows_dist[found]);
}

// The neighbourhood solidity of the brick at (bx0, by0, bz0) read from the
// grid itself: thread r < 484 gathers the 22 voxels of row r (independent
// loads, all in flight) into one word.
__device__ __forceinline__ void fill_rows_from_grid(const GridDesc& g, uint32_t* rows, int32_t bx0, int32_t by0,
                                                    int32_t bz0, int32_t c) {
    if (c >= kSpan * kSpan) return;
    const int32_t gy = by0 - kHalo + c % kSpan, gz = bz0 - kHalo + c / kSpan;
    uint32_t v = 0;
    if (((uint32_t)gy < g.Y) & ((uint32_t)gz < g.Z)) {
        const int32_t* row = g.vox + (uint64_t)g.X * (uint64_t)gy + g.XY * (uint64_t)gz;
#pragma unroll
        for (int32_t b = 0; b < kSpan; b++) {
            const int32_t gx = bx0 - kHalo + b;
            if ((uint32_t)gx < g.X && row[gx] >= 0) v |= 1u << b;
        }
    }
    rows[c] = v;
}

// Whole-grid build: one workgroup per tile of 32 x 8 x 16 voxels, whose
// distances come from the bitmap (field_tile).  Tiles without a solid voxel in
// reach take -6 and tiles of solid voxels keep their words, both without that
// work.  The tile's words go to the grid and, with the words that are kept, to
// the padded render copy, so the copy needs no pass of its own; only words
// that are kept are read.  Workgroup b runs on XCD b mod 8 and takes the tiles
// of that eighth of the grid, so a tile's neighbours share the L2 that holds
// the bitmap's rows and the copy's lines between two tiles.
// 1024x256x1024 (1 GiB): 0.90 ms, against 7.18 ms for a table scan per voxel
// plus 0.09 ms of brick flags and 0.38 ms of copying to the render copy; the
// memory it must move (the copy and the changed words written, the kept ones
// read, 2.1 GB) takes 0.45 ms at the rate of a large copy.
constexpr int kTileY = 8, kTileZ = 16, kTileThreads = kTileY * kTileZ;
__global__ void __launch_bounds__(kTileThreads) k_field_tiles(GridDesc g, GridDesc r, FieldWords words,
                                                              const uint32_t* __restrict__ bits, uint32_t W,
                                                              uint32_t nx, uint32_t ny, uint32_t tiles) {
    using Tile = dev::FieldTile<kTileY, kTileZ>;
    __shared__ Tile L;
    const uint32_t tile = (blockIdx.x % 8) * (gridDim.x / 8) + blockIdx.x / 8;
    if (tile >= tiles) return;
    const int32_t tid = threadIdx.x;
    const uint32_t kx = tile % nx;
    const int32_t x0 = (int32_t)(kx * 32), y0 = (int32_t)((tile / nx) % ny) * kTileY,
                  z0 = (int32_t)(tile / (nx * ny)) * kTileZ;
    bool any = false, full = true;
    for (int32_t i = tid; i < Tile::SZ * Tile::SY; i += kTileThreads) {
        const int32_t y = i % Tile::SY - 6, z = i / Tile::SY - 6;
        const int64_t gy = (int64_t)y0 + y, gz = (int64_t)z0 + z;
        uint2 v = make_uint2(0, 0);
        if (gy >= 0 && gz >= 0 && gy < (int64_t)g.Y && gz < (int64_t)g.Z) {
            const uint32_t* rw = bits + ((uint64_t)gy + (uint64_t)g.Y * (uint64_t)gz) * W + kx;
            v = make_uint2(rw[0], rw[1]);
        }
        L.s[i] = v;
        any |= (v.x | v.y) != 0u;
        if (y >= 0 && y < kTileY && z >= 0 && z < kTileZ) full &= dev::funnel(v.y, v.x, 16) == 0xffffffffu;
    }
    any = __syncthreads_or(any) != 0;
    full = any && __syncthreads_and(full) != 0;
    if (any && !full) {
        dev::field_tile<kTileY, kTileZ, kTileThreads>(L, tid, words);
    } else {
        if (tid < kFieldLevels + 2) L.word[tid] = words.word[tid];
        uint32_t* p = L.plane + tid * 6;
#pragma unroll
        for (int k = 0; k < 5; k++) p[k] = !full && ((kFieldLevels + 1) >> k & 1) ? 0xffffffffu : 0u;
        p[5] = full ? 0xffffffffu : 0u;
        __syncthreads();
    }
    // four voxels per lane and step, eight lanes per row: 128 bytes of a row
    constexpr int kSteps = 8;
    dev::vox4 v[kSteps];
    const int32_t quad = tid & 7, x = x0 + 4 * quad;
    auto row_of = [&](int j) { return j * (kTileThreads / 8) + (tid >> 3); };
    auto cell = [&](const GridDesc& d, int row) {
        return d.origin + (uint64_t)x + (uint64_t)d.SX * (uint64_t)(y0 + row % kTileY) +
               d.SXY * (uint64_t)(z0 + row / kTileY);
    };
    auto inside = [&](int row) {
        return (uint32_t)(y0 + row % kTileY) < g.Y && (uint32_t)(z0 + row / kTileY) < g.Z;
    };
    if ((int64_t)x + 3 < (int64_t)g.X) {
#pragma unroll
        for (int j = 0; j < kSteps; j++) {
            const int row = row_of(j);
            if (inside(row) && ((L.plane[row * 6 + 5] >> (4 * quad)) & 15u))
                v[j] = *(const dev::vox4*)(g.vox + cell(g, row));
        }
#pragma unroll
        for (int j = 0; j < kSteps; j++) {
            const int row = row_of(j);
            if (!inside(row)) continue;
            const uint32_t* p = L.plane + row * 6;
            const uint32_t b = 4 * quad, keep = (p[5] >> b) & 15u;
            const uint32_t pl[5] = {p[0], p[1], p[2], p[3], p[4]};
            dev::vox4 o;
            o.x = keep & 1u ? v[j].x : L.word[dev::level_at(pl, b)];
            o.y = keep & 2u ? v[j].y : L.word[dev::level_at(pl, b + 1)];
            o.z = keep & 4u ? v[j].z : L.word[dev::level_at(pl, b + 2)];
            o.w = keep & 8u ? v[j].w : L.word[dev::level_at(pl, b + 3)];
            if (keep != 15u) *(dev::vox4*)(g.vox + cell(g, row)) = o;
            *(dev::vox4*)(r.vox + cell(r, row)) = o;
        }
    } else {
        for (int j = 0; j < kSteps; j++) {
            const int row = row_of(j);
            if (!inside(row)) continue;
            const uint32_t* p = L.plane + row * 6;
            const uint32_t pl[5] = {p[0], p[1], p[2], p[3], p[4]};
            for (int k = 0; k < 4 && (int64_t)x + k < (int64_t)g.X; k++) {
                const uint32_t b = 4 * quad + k;
                int32_t* w = g.vox + cell(g, row) + k;
                int32_t o;
                if (p[5] >> b & 1u) o = *w;
                else *w = o = L.word[dev::level_at(pl, b)];
                r.vox[cell(r, row) + k] = o;
            }
        }
    }
}

// fixDepthField over the box [x0,x1) x [y0,y1) x [z0,z1) (already clipped);
// with sr >= 0 only voxels with (x-cx)^2+(y-cy)^2+(z-cz)^2 < sr^2.  The box
// is tiled into 8x8x8 bricks from its corner, one workgroup each: the
// brick's neighbourhood solidity is gathered from the grid into LDS and its
// voxels scan the grouped table against it.
__global__ void __launch_bounds__(512) k_fix_depth_box(GridDesc g, DepthTableDev t, int32_t x0, int32_t y0,
                                                        int32_t z0, int32_t w, int32_t h, int32_t d, int32_t nbx,
                                                        int32_t nby, int32_t cx, int32_t cy, int32_t cz, int32_t sr) {
    __shared__ uint32_t rows[kSpan * kSpan];
    const int32_t b = (int32_t)blockIdx.x;
    const int32_t bx0 = x0 + (b % nbx) * 8, by0 = y0 + ((b / nbx) % nby) * 8, bz0 = z0 + (b / (nbx * nby)) * 8;
    const int32_t c = threadIdx.x;
    const int32_t lx = c & 7, ly = (c >> 3) & 7, lz = c >> 6;
    const int32_t x = bx0 + lx, y = by0 + ly, z = bz0 + lz;
    bool mine = (x < x0 + w) & (y < y0 + h) & (z < z0 + d);
    if (sr >= 0) {
        const int32_t ex = x - cx, ey = y - cy, ez = z - cz;
        mine &= ex * ex + ey * ey + ez * ez < sr * sr;
    }
    const uint64_t i = (uint64_t)x + g.X * (uint64_t)y + g.XY * (uint64_t)z;
    const int32_t old = mine ? g.vox[i] : 0;
    if (!__syncthreads_or(mine && old < 0)) return;  // nothing to fix in this brick
    fill_rows_from_grid(g, rows, bx0, by0, bz0, c);
    __syncthreads();
    if (!mine || old >= 0) return;
    const int32_t nv = scan_groups(rows, t, lx, ly, lz, old);
    if (nv != old) g.vox[i] = nv;
}

// destroyVoxel over the clipped box of removeSphere's first loop
// (src/level.cpp:31-42): (x-cx)^2+(y-cy)^2+(z-cz)^2 < r^2.
__global__ void __launch_bounds__(256) k_carve(GridDesc g, int32_t x0, int32_t y0, int32_t z0, int32_t w, int32_t h,
                                                int32_t d, int32_t cx, int32_t cy, int32_t cz, int32_t r) {
    const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= (int64_t)w * h * d) return;
    const int32_t x = x0 + (int32_t)(k % w);
    const int32_t y = y0 + (int32_t)((k / w) % h);
    const int32_t z = z0 + (int32_t)(k / ((int64_t)w * h));
    const int32_t ex = x - cx, ey = y - cy, ez = z - cz;
    if (ex * ex + ey * ey + ez * ez >= r * r) return;
    g.vox[(uint64_t)x + g.X * (uint64_t)y + g.XY * (uint64_t)z] = -1;
}

__global__ void k_set_voxel(int32_t* vox, uint64_t i, int32_t v, int32_t* top, int32_t y) {
    if (threadIdx.x == 0) {
        vox[i] = v;
        if (v >= 0 && top) atomicMax(top, y);
    }
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

// Clip [lo, hi) to [0, n).
inline void clip(int64_t& lo, int64_t& hi, int64_t n) {
    if (lo < 0) lo = 0;
    if (hi > n) hi = n;
}

}  // namespace

int launch_fix_depth_box(const GridDesc& g, const DepthTableDev& t, int32_t x0, int32_t y0, int32_t z0, int32_t x1,
                         int32_t y1, int32_t z1, int32_t scx, int32_t scy, int32_t scz, int32_t sr, hipStream_t s) {
    int64_t ax = x0, bx_ = x1, ay = y0, by_ = y1, az = z0, bz_ = z1;
    clip(ax, bx_, g.X);
    clip(ay, by_, g.Y);
    clip(az, bz_, g.Z);
    if (bx_ <= ax || by_ <= ay || bz_ <= az) return VRT_OK;
    const int64_t w = bx_ - ax, h = by_ - ay, d = bz_ - az;
    const int64_t nbx = (w + 7) / 8, nby = (h + 7) / 8, nbz = (d + 7) / 8;
    const int64_t blocks = nbx * nby * nbz;
    if (blocks > 0x7fffffff) return fail(VRT_ERR_INVALID, "box too large");
    hipLaunchKernelGGL(k_fix_depth_box, dim3((uint32_t)blocks), dim3(512), 0, s, g, t, (int32_t)ax, (int32_t)ay,
                       (int32_t)az, (int32_t)w, (int32_t)h, (int32_t)d, (int32_t)nbx, (int32_t)nby, scx, scy, scz,
                       sr);
    VRT_HIP(hipGetLastError());
    return VRT_OK;
}

uint32_t solid_bits_words(const GridDesc& g) { return (g.X + 31u) / 32u + 1u; }

int launch_build_depth_field(const GridDesc& g, const GridDesc& render, const FieldWords& words, uint32_t* bits,
                             hipStream_t s) {
    const uint32_t W = solid_bits_words(g);
    const uint64_t rows = (uint64_t)g.Y * g.Z;
    const uint64_t bit_blocks = ((rows + kBitRows - 1) / kBitRows * (W * 8ull) + 255) / 256;
    const uint64_t nx = (g.X + 31ull) / 32, ny = (g.Y + kTileY - 1ull) / kTileY, nz = (g.Z + kTileZ - 1ull) / kTileZ;
    const uint64_t tiles = nx * ny * nz;
    if (bit_blocks > 0x7fffffffull || nx * ny > 0x7ffffff0ull || tiles > 0x7ffffff0ull)
        return fail(VRT_ERR_INVALID, "grid too large for the build");
    hipLaunchKernelGGL(k_solid_bits, dim3((uint32_t)bit_blocks), dim3(256), 0, s, g, bits, W, rows);
    VRT_HIP(hipGetLastError());
    hipLaunchKernelGGL(k_field_tiles, dim3((uint32_t)((tiles + 7) / 8 * 8)), dim3(kTileThreads), 0, s, g, render, words,
                       bits, W, (uint32_t)nx, (uint32_t)ny, (uint32_t)tiles);
    VRT_HIP(hipGetLastError());
    return VRT_OK;
}

int launch_carve_sphere(const GridDesc& g, int32_t cx, int32_t cy, int32_t cz, int32_t r, hipStream_t s) {
    if (r <= 0) return VRT_OK;
    int64_t ax = (int64_t)cx - r, bx_ = (int64_t)cx + r, ay = (int64_t)cy - r, by_ = (int64_t)cy + r,
            az = (int64_t)cz - r, bz_ = (int64_t)cz + r;
    clip(ax, bx_, g.X);
    clip(ay, by_, g.Y);
    clip(az, bz_, g.Z);
    if (bx_ <= ax || by_ <= ay || bz_ <= az) return VRT_OK;
    const int64_t w = bx_ - ax, h = by_ - ay, d = bz_ - az;
    const int64_t blocks = (w * h * d + 255) / 256;
    if (blocks > 0x7fffffff) return fail(VRT_ERR_INVALID, "sphere too large");
    hipLaunchKernelGGL(k_carve, dim3((uint32_t)blocks), dim3(256), 0, s, g, (int32_t)ax, (int32_t)ay, (int32_t)az,
                       (int32_t)w, (int32_t)h, (int32_t)d, cx, cy, cz, r);
    VRT_HIP(hipGetLastError());
    return VRT_OK;
}

int launch_set_voxel(const GridDesc& g, int64_t index, int32_t y, int32_t v, hipStream_t s) {
    if (index < 0 || (uint64_t)index >= g.count) return fail(VRT_ERR_INVALID, "voxel index out of range");
    hipLaunchKernelGGL(k_set_voxel, dim3(1), dim3(64), 0, s, g.vox, (uint64_t)index, v, g.top, y);
    VRT_HIP(hipGetLastError());
    return VRT_OK;
}

int launch_solid_top(const GridDesc& g, int64_t x0, int64_t y0, int64_t z0, int64_t x1, int64_t y1, int64_t z1,
                     bool reset, hipStream_t s) {
    if (!g.top) return fail(VRT_ERR_INVALID, "grid without a solid-top word");
    if (reset) {
        hipLaunchKernelGGL(k_set_word, dim3(1), dim3(64), 0, s, g.top, -1);
        VRT_HIP(hipGetLastError());
    }
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

}  // namespace vrt
