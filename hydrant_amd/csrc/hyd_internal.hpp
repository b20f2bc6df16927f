// Internal declarations shared by the C ABI implementation and the kernels.
#pragma once

#include <hip/hip_runtime.h>

#include <array>
#include <cmath>
#include <cstdarg>
#include <cstdint>
#include <cstdio>
#include <string>
#include <utility>
#include <vector>

#include "../../include/hydrant_hip.h"
#include "hyd_math.hpp"

namespace hyd {

void set_error(const char *fmt, ...);

#define HYD_CHECK_HIP(expr)                                                          \
  do {                                                                               \
    hipError_t _e = (expr);                                                          \
    if (_e != hipSuccess) {                                                          \
      ::hyd::set_error("%s failed: %s (%s:%d)", #expr, hipGetErrorString(_e), __FILE__, \
                       __LINE__);                                                    \
      return HYD_ERR_HIP;                                                            \
    }                                                                                \
  } while (0)

#define HYD_REQUIRE(cond, code, ...)   \
  do {                                 \
    if (!(cond)) {                     \
      ::hyd::set_error(__VA_ARGS__);   \
      return (code);                   \
    }                                  \
  } while (0)

// Device-resident paging state.  page[i] = {k, b.x, b.y, b.z}.
struct Paging {
  const int32_t *vaddr = nullptr;
  int32_t vdim[3] = {0, 0, 0};
  const float4 *page = nullptr;
  int32_t n_pages = 0;
  int32_t lowest_blkcnt = 0;
};

struct Pool {
  const void *data = nullptr;
  int32_t fmt = -1;
  int32_t pad = 0;       // padded brick edge
  int32_t n_pages = 0;
  bool owned = false;
};

struct Grid {
  const int32_t *data = nullptr;
  int32_t dim[3] = {0, 0, 0};
};

struct GridF {
  const float *data = nullptr;
  int32_t dim[3] = {0, 0, 0};
};

struct Ctx {
  int device = 0;
  hipStream_t stream = nullptr;
  hipStream_t own_stream = nullptr;
  Pool pool;
  Paging paging;
  Grid cheb;
  GridF mean;
  const float *tf = nullptr;
  int32_t tf_n = 0;
  uint64_t pool_gen = 0;          // bumped by every pool upload / bind
  // bumped whenever device memory a captured batch graph reads may move
  // (pool upload / bind, transfer function, volume set)
  uint64_t batch_state_gen = 0;
  // owned device allocations (freed at destroy)
  void *own_pool = nullptr;
  void *own_oriented = nullptr;   // the pool's oriented layouts (batched renderer)
  size_t oriented_cap = 0;
  int oriented_pairs = 0;          // own_oriented holds the y- and z-fastest single-voxel layouts (0),
                                   // the three row-pair layouts (1) or the three quad layouts (2)
  uint64_t oriented_gen = ~0ull;  // pool_gen the oriented layouts were made from
  int32_t *own_vaddr = nullptr;
  float4 *own_page = nullptr;
  size_t vaddr_cap = 0, page_cap = 0;   // bytes of own_vaddr / own_page
  // host copies of the page table and chebyshev grid, combined into one code per
  // brick (see VolumeArgs::codes) while their dims agree
  std::vector<int32_t> host_vaddr, host_cheb;
  int32_t *own_codes = nullptr;
  size_t codes_cap = 0;
  bool codes_valid = false;
  int32_t *own_cheb = nullptr;
  float *own_mean = nullptr;
  float *own_tf = nullptr;
  float page_lo = 0.f, page_hi = 0.f;   // over the page mappings: least b, greatest k + b (NaN: none)
  float page_k_min = 0.f, page_k_max = 0.f;
  bool tf_finite = false;         // every transfer-function entry is finite
  float tf_alpha_min = 0.f, tf_alpha_max = 0.f, tf_rgb_max = 0.f;   // tf_rgb_max: of the magnitudes
  float *srgb8_t = nullptr;       // 256 sRGB byte thresholds (srgb8_thresholds)
  // multi-volume set of the batched renderer
  void *own_vols = nullptr;       // BatchVolDev[n_vols]
  int32_t *own_cells = nullptr;   // concatenated cell codes
  int32_t n_vols = 0;
  int32_t vol_pad = 0;            // padded brick edge shared by every volume
  int32_t vol_max_page = -1;   // largest page a cell of the volume set names (-1: none)
  int32_t n_cus = 0;
  // macrocells of the pool (hyd_macro.hpp): value ranges, and their classes under
  // the transfer function for the frame marches (owned pools only: a bound
  // pool's contents may change without notice).  The classes are made by the first
  // frame that can use them, and pages written since (dirty) join them at the
  // next frame or isosurface.
  float2 *own_mm = nullptr;
  uint8_t *own_mcls = nullptr;
  // {macrocells of class 0, of class >= 3} (launch_macro_classes): of the frame classes, in
  // one of two slots (the other is zero, for the next), then of the batch's
  unsigned long long *own_mcount = nullptr;
  int32_t mcount_slot = 0;
  hipEvent_t macro_ev = nullptr;  // behind the last update of the ranges and frame classes
  bool macro_pending = false;     // ... which may still run
  size_t macro_cap = 0;           // macrocells the arrays hold
  uint64_t mm_gen = ~0ull;        // pool_gen the ranges were made from
  std::vector<std::pair<int32_t, int32_t>> mm_dirty;   // runs {first, number} of pages whose ranges are behind
  bool mcls_valid = false;        // own_mcls belongs to own_mm and the current transfer function
  // classes for the batched renderer: each page under the value scale of its
  // volume (NaN: none, or two that differ), made at the first batched launch
  // after a change of pool, transfer function or volume set
  std::vector<std::pair<int32_t, float>> vol_pages;   // {page, value scale} of every resident cell
  std::vector<std::array<float, 3>> vol_bmax;   // extent of each volume of the set
  float *own_bscale = nullptr;
  uint8_t *own_bcls = nullptr;
  size_t bcls_cap = 0, bscale_cap = 0;
  uint64_t bcls_gen = ~0ull;      // batch_state_gen of own_bcls
  double bcls_empty = 0.0, bcls_deep = 0.0;   // shares of class > 0 and of class >= 3
  // differentiable renderer: device copy of the views
  void *own_diff_views = nullptr;
  int32_t diff_view_cap = 0;
  void *own_diff_scratch = nullptr;   // adjoint scratch (per-sample dL/ds), grown on demand
  size_t diff_scratch_cap = 0;
};

// Flattened kernel arguments for the volume march (passed by value).
// Tile order of a frame launch (one 8x8 tile per workgroup, grid x = tile
// column): row r of the tile grid is rotated by HYD_TILE_ROTATE * r tiles, a
// bijection on each row.  Workgroups are dealt round-robin over the 8 XCDs and
// then over each XCD's 32 CUs, so one CU receives workgroups 256 apart; in a
// 64-tile-wide grid (512 pixels) those are the tiles of one image column,
// every fourth tile row, and the CUs that hold the centre columns, whose rays
// are the longest, set the frame.  The rotation spreads a CU's tiles over 16
// columns.  512^2 frames: plain FP32 0.551 -> 0.528 ms, paged u8 0.351 ->
// 0.317 ms (rotations 3, 5, 9, 11, 23: 0.531-0.557 and 0.316-0.319 ms).
#ifndef HYD_TILE_ROTATE
#define HYD_TILE_ROTATE 7
#endif
__device__ __forceinline__ int rotated_tile_x() {
  return (int)((blockIdx.x + (unsigned)HYD_TILE_ROTATE * blockIdx.y) % gridDim.x);
}

// The pool's macrocells as a march sees them.  Every page has one mapping
// (tap coordinate = x K + B on each axis), so its constants are scalars.
struct MacroGrid {
  const uint8_t *cls;   // classes, page after page (null: none)
  int32_t nm, cells;    // macrocells per page edge and per page
  float K, B;           // voxels per brick unit, tap coordinate of x = 0
  float run_max;        // longest run to skip at once
  // the classes are looked up while *count, of the macrocells that may contribute (one
  // lane a ray) or of those deep in empty space (several), lies in this range
  const unsigned long long *count;
  unsigned long long count_min, count_max;
};

// Samplers of a march (hyd_sampler.hpp): the clamping one for every sample;
// the inner one for groups of samples whose taps are found inside their page;
// or the inner one throughout (every page maps a brick inside its tap centres).
enum { kInnerNever = 0, kInnerTest = 1, kInnerAlways = 2 };

struct VolumeArgs {
  // shader
  f3 bmin, bmax;
  float step;
  int32_t max_steps;
  int32_t mode;
  float rank;
  float density;
  int32_t schedule;
  float ert;
  // view
  float trans[16];
  float ctg;
  f3 ray_o;
  int32_t W, H;
  // tables
  const float *tf;
  int32_t tf_n;
  const int32_t *cheb;
  int32_t cdim[3];
  const int32_t *vaddr;
  int32_t vdim[3];
  // one code per brick when the chebyshev and page-table grids have equal dims
  // (else null): page id >= 0, -1 not resident, <= -2 empty at distance -1 - code
  const int32_t *codes;
  int32_t lowest_blkcnt;
  const float4 *page;
  const void *pool;
  uint64_t pool_elems;    // voxels in the pool (n_pages * pad^3)
  int32_t pad;
  int32_t inner;          // kInner*: which samples take the sampler without wraps and clamps
  float full_rays;        // the launch's work in rays of its longest chord (host: lanes per ray)
  int32_t lanes;          // frames: lanes per ray (frame_lanes)
  int32_t monotone;       // opacities in [0, 1]: a ray's alpha never falls
  MacroGrid macro;        // hyd_macro.hpp
  // outputs
  hyd_volume_pixel *film;
  float4 *rgba;
  unsigned long long *samples;
  // sort-last segments: slots[ord * W*H + ray], nslots[ray]
  float4 *slots;
  int32_t *nslots;
  int32_t max_slots;
  const uint64_t *page_base;   // segment sets: first voxel of each page, in voxels from pool
  const int32_t *page_local;   // segment sets: each page's id in its own batch (Paging mode colours by it)
};

// The work of a frame as a number of rays of its longest chord (hyd_api.cpp).
float full_rays(const float *trans, float ctg, f3 ray_o, int W, int H, f3 bmin, f3 bmax);

// The work (full_rays) up to which a march of a pool of that size runs four
// lanes per ray (measurements: k_volume.hip).
inline float lane_rays(double pool_bytes) { return 75e3f + 36e3f * (float)std::log2(1.0 + pool_bytes / 24e6); }

// Lanes per ray of a frame over a pool of that size: 16, 4 or 1 (k_volume.hip).
int32_t frame_lanes(int W, int H, float full_rays, double pool_bytes);

hipError_t launch_volume(const VolumeArgs &a, int fmt, bool resume, hipStream_t s);
hipError_t launch_segments_clear(float4 *slots, size_t n, hipStream_t s);
hipError_t launch_segments_pass(const VolumeArgs &a, int fmt, hipStream_t s);
// A segment set's batches in one launch: codes, page descriptors, bases and local
// ids run over the pages of every batch, pool is the lowest of their pools,
// span_bytes the distance from it to the end of the highest (which the offsets
// have to reach) and pool_bytes what the pools hold (which the launch reads).
hipError_t launch_segments_set(const VolumeArgs &a, uint64_t span_bytes, uint64_t pool_bytes, int fmt, hipStream_t s);
constexpr int kMaxSegBatches = 16;
hipError_t launch_segments_composite(const float4 *slots, const int32_t *nslots, int max_slots, int P, float4 *rgba,
                                     hipStream_t s);
hipError_t launch_volume_trace(const VolumeArgs &a, int fmt, int x, int y, hyd_trace_rec *out_dev, int max_recs,
                               int *n_dev, hipStream_t s);
hipError_t launch_pixel_pass(const float4 *rgba, int W, int H, uchar3 clear, uint8_t *rgb, hipStream_t s);
hipError_t launch_fetch_pass(const hyd_volume_pixel *film, int W, int H, hyd_fetch_pixel *out, hipStream_t s);
// The z order of a composite, held by the launch's arguments up to kArgZ images
// and in device memory beyond (256 bytes of arguments; a node's ranks fit).
// An allocation, a copy and a free about each composite of eight 1024^2 images made
// it 83 us; without them, and with four images' loads in flight, it takes 77
// (the copy's rate gives 61).
constexpr int kArgZ = 64;
struct ZOrder {
  const int32_t *dev;   // null: v
  int32_t v[kArgZ];
  __host__ __device__ int at(int k) const { return dev ? dev[k] : v[k]; }
};
hipError_t launch_composite(int n, const hyd_fetch_pixel *partials, const ZOrder &z, int W, int H,
                            float4 *rgba, uint8_t *rgb, const float *srgb_t, hipStream_t s);
hipError_t launch_iso_fetch(const hyd_iso_pixel *px, int W, int H, hyd_iso_fetch_pixel *out, hipStream_t s);
hipError_t launch_iso_composite(int n, const hyd_iso_fetch_pixel *partials, const ZOrder &z, int W, int H,
                                uint8_t *rgb, float *depth, hipStream_t s);
// t[0] = -inf, t[k] (k = 1..255) = least float whose saturated sRGB byte is >= k
// (volume.cc:175-181,284-288 evaluated on the host).
void srgb8_thresholds(float t[256]);

struct BlocksArgs {
  f3 bmin, bmax;
  float step;
  int32_t max_steps;
  int32_t mode;
  float density;
  float trans[16];
  float ctg;
  f3 ray_o;
  int32_t W, H;
  const int32_t *cheb;
  const float *mean;
  int32_t dim[3];
  const int32_t *vaddr;   // page table (HYD_BLOCKS_PAGING)
  int32_t vdim[3];
  int32_t lowest;         // pages at or above this id are level-0 pages
  float4 *rgba;
};
hipError_t launch_blocks(const BlocksArgs &a, hipStream_t s);

struct IsoArgs {
  f3 bmin, bmax;
  float step, du;
  int32_t max_steps;
  int32_t mode;
  float to_world[16];
  f3 eye_pos, light_pos, surface_color;
  float isovalue;
  int32_t corrected, bisect_steps;
  float trans[16];
  float ctg;
  f3 ray_o;
  int32_t W, H;
  const int32_t *cheb;
  int32_t cdim[3];
  const int32_t *vaddr;
  int32_t vdim[3];
  const int32_t *codes;   // as VolumeArgs::codes
  const float4 *page;
  const void *pool;
  uint64_t pool_elems;    // voxels in the pool (n_pages * pad^3)
  int32_t pad;
  int32_t inner;          // as VolumeArgs::inner
  // value ranges of the pool's macrocells as stored (null: none) and the factor
  // to their values (hyd_macro.hpp); macro.cls is not used
  const float2 *mm;
  float mm_scale;
  MacroGrid macro;
  hyd_iso_pixel *out;
  unsigned long long *samples;
};
hipError_t launch_iso(const IsoArgs &a, int fmt, hipStream_t s);

int32_t activate(Ctx *c);
// Whether the context's stream is being captured.  A replay may meet another page
// table (hyd_set_page_table rewrites it in place), so a captured march takes
// nothing that the host derived from the table's mappings: its samples are
// tested per group, and no macrocells are passed over.
bool capturing(const Ctx *c);
// After pool pages [first, first + n) were overwritten in place: updates the
// batched renderer's oriented copies of those pages if they are current.
int32_t refresh_oriented_pages(Ctx *c, int32_t first, int32_t n);
// Macrocells of a pool (hyd_macro.cpp).  After an upload: its ranges (on the
// stream; the caller waits).  After a write of pages [first, first + n): noted for
// the next march, or, where the batched renderer's classes are current, brought
// up to date in place (on the stream; the caller waits).
int32_t macro_pool_uploaded(Ctx *c);
int32_t macro_pages_written(Ctx *c, int32_t first, int32_t n);
void macro_free(Ctx *c);
// Points the march at the classes when they apply to it, else leaves it without;
// brings them up to date first, ahead of the march on its stream (not under capture).
int32_t macro_fill(Ctx *c, VolumeArgs &a);
// The batched renderer's classes of the current pool, brought up to date
// (complete on return); null in *cls when the march, of that many lanes a ray,
// should sample throughout.
int32_t macro_batch(Ctx *c, int32_t lanes, const uint8_t **cls);
int32_t macro_fill_iso(Ctx *c, IsoArgs &a);

}  // namespace hyd

// The opaque handle of the C ABI.
struct hyd_ctx : hyd::Ctx {};
