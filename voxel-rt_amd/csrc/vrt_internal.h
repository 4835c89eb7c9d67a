// vrt_internal.h — declarations shared by the libvrt sources (host side).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <string>
#include <vector>

#include "../../include/vrt.h"

namespace vrt {

// Sets the thread's last error message and returns `code`.
int fail(int code, const std::string& msg);
int hip_fail(hipError_t e, const char* what);

#define VRT_HIP(call)                                        \
    do {                                                     \
        hipError_t e_ = (call);                              \
        if (e_ != hipSuccess) return vrt::hip_fail(e_, #call); \
    } while (0)

// Render copy of the grid: every side padded with kGuard cells holding
// kGuardValue, the bits of a NaN.  A walk that steps onto one takes it for a
// depth-field jump of NaN cells, which ends the walk at once as a miss, as
// src/fshader.glsl:123-125 ends it on a cell outside the grid: the traversal
// then needs no bounds test per step.  (A NaN jump inside the grid ends the
// walk the same way in the reference, :114-121 then :83.)
constexpr int32_t kGuard = 3;
constexpr int32_t kGuardValue = (int32_t)0xFFC00000u;
// The guard cells with x < 0 and y < 0 hold another NaN, by which a walk knows
// that it left the grid there (cast_ray).
constexpr int32_t kGuardCorner = (int32_t)0xFFC00001u;

// Grid as the kernels see it.  Cell (x, y, z) is vox[origin + x + SX*y +
// SXY*z]; X, Y, Z are the grid's extents.  The library's grid is dense
// (SX = X, SXY = XY, origin 0); the render copy is padded (kGuard cells on
// every side).
struct GridDesc {
    int32_t* vox;
    uint32_t X, Y, Z;
    uint64_t XY;
    uint64_t count;  // words allocated at vox
    uint32_t SX;
    uint64_t SXY;
    uint64_t origin;
    // Device word: an upper bound on the y of every solid voxel (-1 when there
    // is none).  Every entry point that can add solid voxels raises it; edits
    // that only remove leave it high, which stays an upper bound.  Render
    // kernels stop a shadow ray once it is provably above it; null: they walk
    // every shadow ray to the reference's end.
    int32_t* top;
    // The extents as floats, at most 2^22 (render copies): a start below them
    // lies inside the grid and in the range of the walk's arithmetic.
    float FX, FY, FZ;
    // The y and z a walk can index (the grid's and two cells past it on
    // either side) fit signed 24-bit multiplies.
    bool yz24() const { return (uint64_t)Y + 2 < (1ull << 23) && (uint64_t)Z + 2 < (1ull << 23); }
    // Index fits the 32-bit / 24-bit-multiply form (see Idx32).
    bool small() const { return count <= 0xffffffffull && SX < (1u << 23) && SXY < (1ull << 23) && yz24(); }
    // Byte offset fits the 32-bit / 24-bit-multiply form (see IdxB).
    bool bytes32() const {
        return count <= (1ull << 30) && 4ull * SX < (1ull << 23) && 4ull * SXY < (1ull << 23) && yz24();
    }
};

// floor(2^32 / d), at most 2^32 - 1: with it a kernel divides by d on the
// scalar unit.
inline uint32_t tile_rcp(uint32_t d) { return d <= 1 ? 0xffffffffu : (uint32_t)(((uint64_t)1 << 32) / d); }

// One frame as the kernels see it: vrt_frame plus derived per-frame values.
struct FrameDesc {
    vrt_frame f;
    float render_lim;   // (float)render_dist
    // Per light: the largest float t with sqrt_rn(t) <= radius, so that
    // length(v) <= radius  <=>  dot(v, v) <= t  (sqrt_rn is monotone).
    float light_dd_max[VRT_MAX_LOCAL_LIGHTS];
    // Per light: the largest float a >= 0 with RN(a * a) <= light_dd_max.
    // dot(v, v) >= RN(v.x * v.x) (a sum of non-negative terms, each rounding
    // monotone), so |v.x| > a already puts the light out of range.
    float light_axis_max[VRT_MAX_LOCAL_LIGHTS];
    float light_x[VRT_MAX_LOCAL_LIGHTS];  // the lights' x
    // Bit i set when light i is placed: every coordinate >= 0 (unused slots
    // hold -1, src/render.cpp:304-311; NaN compares false).
    uint32_t light_valid;
    float light_rinv[VRT_MAX_LOCAL_LIGHTS];  // RN(1 / radius)
    float inv_w, inv_h;                      // RN(1 / width), RN(1 / height) of the target
    uint32_t tiles_rcp;                      // tile_rcp(tiles across), for the kernels' tile arithmetic
    // Primary rays may stop above every solid voxel too: only when nothing
    // shows their step count (no depth view, no step map in the target).
    int32_t primary_cutoff;
    // k_render_plain deals tile rows from this one on, wrapping to row 0
    // (dispatch order only; see plain_row_rotation).
    int32_t row_rot;
};

// Ray/step counters: kCounterSlots slots of one 128-byte line each
// (u64 rays, DDA steps, pixels); a wave adds into slot (its wave id mod
// kCounterSlots), so waves rarely share a line and the atomics never queue
// on one address.  Stats are the sum over slots.
constexpr int kCounterSlots = 4096;
constexpr int kCounterStride = 16;  // u64 per slot

// Plain draws do not add into the counters at the end of every wave: a
// device-scope atomic there keeps the wave's slot (and with it the start of
// the next workgroup, which needs a slot on every SIMD of the CU) until it
// completes, 3% of a 1080p frame.  Each wave stores its tile's totals into
// the context's partial-count array instead, one u64 per tile (DDA iterations
// in the low 32 bits, rays and pixels in 16 bits each above them), at the
// next free entries; the entries are added into the counters by a fold kernel
// when the array is full and before stats are read.  Under stream capture
// the draw keeps the atomics (a replayed graph would rewrite one set of
// entries).  The packed sums are exact while a tile's iteration total stays
// below 2^32: 64 lanes x 18 rays x lim < 2^32 for lim < kTileSum32Lim.
constexpr int64_t kPartsCap = (int64_t)1 << 22;  // entries (32 MiB)
constexpr float kTileSum32Lim = 3.7e6f;

// Queue of the persistent batch kernel: 8 counters (one per XCD), 128 B apart.
constexpr size_t kQueueBytes = 8 * 128;
// Tiles one multi-view launch may hold (queue counters are 32-bit).
constexpr int64_t kMaxBatchTiles = 0xffffffffll - 65536;

// Per-view work description for the persistent batch kernel.
struct ViewDesc {
    FrameDesc frame;
    vrt_target target;
    int32_t tiles_x;       // tiles across
    int32_t tiles;         // tiles in this view
    int64_t first_tile;    // prefix sum of tiles over earlier views
};

// The words that a depth field can give an empty voxel, nearest first
// (vrt_field.h): entry 0 is unused (the word is left as it was), entries 1 to
// kFieldLevels the bits of the table's distances in (-6, -2], the last -6.0f.
constexpr int kFieldLevels = 23;
struct FieldWords {
    int32_t word[kFieldLevels + 2];
};

// Words of one of the two pieces of a context's upload staging (1 MiB).
constexpr int64_t kStagePiece = (int64_t)1 << 18;

struct Ctx;

// ---- kernels launch wrappers (vrt_render.hip / vrt_edit.hip / vrt_world.hip)
// parts == nullptr: the wave totals go into `counters` by atomics; else into
// parts[tile] (see kPartsCap).
int launch_render_plain(const GridDesc& g, const FrameDesc& f, const vrt_target& t,
                        unsigned long long* counters, unsigned long long* parts, hipStream_t s);
// Adds parts[0, n) into the counter slots.
int launch_fold_parts(const unsigned long long* parts, int64_t n, unsigned long long* counters, hipStream_t s);
int launch_cast_rays(const GridDesc& g, int64_t n, const float* start, const float* dir,
                     const int32_t* dist, int32_t render_dist, int64_t* hit, float* hit_pos,
                     uint8_t* face, uint32_t* steps, hipStream_t s);
// How a launch's waves count (lanes: each lane its iterations) and are grouped
// (far: four a workgroup); for several views, what any of them needs.
struct DrawForm {
    bool lanes = false, far = false;
    DrawForm& operator|=(const DrawForm& o) {
        lanes |= o.lanes;
        far |= o.far;
        return *this;
    }
};
DrawForm draw_form(const GridDesc& g, const FrameDesc& f);
// parts (chunk_tiles 0 only; nullptr: atomics): one entry per 64-pixel pass
// (batch_items), added into the counters by launch_fold_parts afterwards.
int launch_render_batch(const GridDesc& g, const ViewDesc* views_dev, int32_t n_views,
                        int64_t total_tiles, const vrt_batch_config& cfg, DrawForm form, int32_t n_workgroups,
                        unsigned int* queue, unsigned long long* counters, unsigned long long* parts,
                        hipStream_t s);
inline DrawForm draw_form(const GridDesc& g, const std::vector<ViewDesc>& views) {
    DrawForm form;
    for (const ViewDesc& v : views) form |= draw_form(g, v.frame);
    return form;
}
// Entries a hardware-scheduled multi-view launch writes into `parts`, or -1
// when its counts must go by atomics (a view's render_lim too large for the
// 32-bit pass sums, or a persistent configuration).
int64_t batch_items(const std::vector<ViewDesc>& views, int64_t total_tiles, const vrt_batch_config& cfg);
int launch_queue_reset(unsigned int* queue, hipStream_t s);
int selftest_division(uint32_t d_begin, uint32_t d_count, unsigned long long* bad_dev, hipStream_t s);
int selftest_reciprocal(uint64_t first, uint64_t count, unsigned long long* bad_dev, hipStream_t s);
int batch_occupancy(const vrt_batch_config& cfg, int32_t* waves_per_cu);

// destroyVoxel within cr of (cx, cy, cz) (cr <= 0: none), then fixDepthField
// within sr of it (sr < 0: everywhere), over the voxels of the box [x0,x1) x
// [y0,y1) x [z0,z1) (clipped to the grid); the box goes to `render` too unless
// render.vox is null.  cr <= sr where both apply.
int launch_edit_box(const GridDesc& g, const GridDesc& render, const FieldWords& words, int64_t x0, int64_t y0,
                    int64_t z0, int64_t x1, int64_t y1, int64_t z1, int32_t cx, int32_t cy, int32_t cz, int32_t sr,
                    int32_t cr, hipStream_t s);
// Whole-grid depth field: solidity bitmap (Y*Z rows of solid_bits_words(g)
// words), then every tile's words into the grid and into `render`, the
// padded copy of the whole grid.
uint32_t solid_bits_words(const GridDesc& g);
int launch_build_depth_field(const GridDesc& g, const GridDesc& render, const FieldWords& words, uint32_t* bits,
                             hipStream_t s);
// One voxel of the grid and of the render copy; raises *g.top for a solid one.
int launch_set_voxel(const GridDesc& g, const GridDesc& render, int32_t x, int32_t y, int32_t z, int32_t v,
                     hipStream_t s);
// The whole grid from `src` (device; g.vox: the grid itself) into the render
// copy and the grid; sets *g.top to the highest y with a solid voxel.
int launch_load_grid(const GridDesc& g, const GridDesc& render, const int32_t* src, hipStream_t s);
// Words [first, first + n) of the box at (x0, y0, z0), nx x ny voxels per z,
// from pinned host memory into the grid and the render copy; raises *g.top to
// `top`.
int launch_put_box(const GridDesc& g, const GridDesc& render, const int32_t* src, int64_t first, int64_t n, int64_t nx,
                   int64_t ny, int64_t x0, int64_t y0, int64_t z0, int32_t top, hipStream_t s);
// Raises *g.top to the highest y with a solid voxel in the box [x0,x1) x
// [y0,y1) x [z0,z1) (clipped to the grid).
int launch_solid_top(const GridDesc& g, int64_t x0, int64_t y0, int64_t z0, int64_t x1, int64_t y1, int64_t z1,
                     hipStream_t s);
int launch_fill(int32_t* p, uint64_t n, int32_t v, hipStream_t s);
// Every word of a padded copy: kGuardCorner where x < 0 and y < 0, else kGuardValue.
int launch_fill_guard(const GridDesc& render, hipStream_t s);
// dst's cells of the box [x0,x0+nx) x [y0,y0+ny) x [z0,z0+nz) := src's.
int launch_copy_box(const GridDesc& src, const GridDesc& dst, int64_t x0, int64_t y0, int64_t z0, int64_t nx,
                    int64_t ny, int64_t nz, hipStream_t s);
int launch_copy(int32_t* dst, const int32_t* src, uint64_t n, hipStream_t s);
int launch_world_generate(const GridDesc& g, const vrt_world_params& p, const int32_t* cave_list,
                          int32_t n_caves, const int32_t* box_list, int32_t n_boxes,
                          const int32_t* cave_bins, const int32_t* box_bins, int32_t bin_size,
                          int32_t bins_x, int32_t bins_z, hipStream_t s);

// ---- host helpers
double now_seconds();

// World generator pieces shared by the host and device generators.
struct WorldPlan {
    vrt_world_params p;
    std::vector<int32_t> caves;  // cx, cy, cz, r
    std::vector<int32_t> boxes;  // x0, y0, z0, x1, y1, z1 (half-open, clipped)
};
int make_world_plan(const vrt_world_params& p, WorldPlan& plan);

}  // namespace vrt

// Context behind the opaque vrt_ctx handle.
struct vrt_ctx {
    int32_t device = 0;
    hipStream_t own_stream = nullptr;
    hipStream_t stream = nullptr;
    vrt::GridDesc grid{};
    // Padded render copy of `grid` (see kGuard); every entry point that
    // writes the grid refreshes the part it wrote, on the same stream.
    vrt::GridDesc rgrid{};
    vrt_frame frame{};
    bool frame_set = false;
    unsigned long long* counters = nullptr;  // rays, iters, pixels
    unsigned long long* parts = nullptr;     // plain draws' partial counts (kPartsCap entries)
    int64_t parts_used = 0;                  // entries not yet folded into `counters`
    uint64_t draws = 0;
    vrt::FieldWords words{};
    uint32_t* solid_bits = nullptr;  // whole-grid build scratch, allocated by the first build
    // Pinned staging of small partial uploads, two pieces of kStagePiece words,
    // allocated by the first one; no upload leaves work on it when it returns.
    int32_t* stage = nullptr;
    hipEvent_t stage_done[2] = {nullptr, nullptr};
    int32_t num_cus = 0;
    bool tuned = false;
    vrt_batch_config tuned_cfg{8, 8, 0, 0};
    bool shadow_cutoff = true;  // vrt_set_shadow_cutoff
    // Host copy of *grid.top, read back by the entry points that can raise it
    // (they synchronize anyway or are not on a per-frame path).
    int32_t top_host = -1;
};

namespace vrt {
// The grid as the render kernels get it: the padded copy, with `top` only
// with the shadow cutoff on.
inline GridDesc render_grid(const vrt_ctx* c) {
    GridDesc g = c->rgrid;
    g.top = c->shadow_cutoff ? c->grid.top : nullptr;
    return g;
}
// Copies the box [x0,x1) x [y0,y1) x [z0,z1) (clipped to the grid) of the
// grid into the render copy, on the context's stream.
int refresh_render(vrt_ctx* c, int64_t x0, int64_t y0, int64_t z0, int64_t x1, int64_t y1, int64_t z1);
// removeSphere on stream s: carve and depth-field repair of the grid and, unless
// render.vox is null, of the edited box of that padded copy.
int remove_sphere_on(vrt_ctx* c, const GridDesc& render, int32_t cx, int32_t cy, int32_t cz, int32_t radius,
                     hipStream_t s);
// The same refresh, and that of a removeSphere's box, into another copy laid
// out like the render copy.
int refresh_copy_on(vrt_ctx* c, const GridDesc& dst, hipStream_t s, int64_t x0, int64_t y0, int64_t z0, int64_t x1,
                    int64_t y1, int64_t z1);
int remove_sphere_refresh_into(vrt_ctx* c, const GridDesc& dst, int32_t cx, int32_t cy, int32_t cz, int32_t radius,
                               hipStream_t s);
}  // namespace vrt

namespace vrt {
int world_generate_device(const GridDesc& g, const vrt_world_params& p, hipStream_t s);
FrameDesc make_frame_desc(const vrt_frame& f, const vrt_target& target);
int32_t plain_row_rotation(const vrt_frame& f, const vrt_target& t, int32_t top, bool primary_cutoff);
int check_frame(const vrt_frame& f);
// Tile shape in {8x8, 16x4, 32x2, 16x16, 64x1}, chunk_tiles in [0, 4096],
// waves_per_cu in [0, 64]; the batch kernels assume all three.
int check_batch_config(const vrt_batch_config& c);
// One view's descriptor for a multi-view launch, its tiles numbered from
// first_tile; checks the frame and target.
struct ViewDesc;
int make_view_desc(const vrt_view& v, const vrt_batch_config& cfg, int64_t first_tile, ViewDesc& d);
// Persistent workgroups of a multi-view launch, from occupancy; 0 when the
// hardware schedules (chunk_tiles 0), where the launch counts its own.
int persistent_workgroups(vrt_ctx* c, const vrt_batch_config& cfg, int64_t total_tiles, int32_t* out);
int check_target(const vrt_target& t);
}  // namespace vrt
