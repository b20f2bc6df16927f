// Host side of the macrocells: when they are made and when a march may use them.
#include <algorithm>
#include <cmath>
#include <vector>

#include "hyd_macro.hpp"

namespace hyd {
namespace {

// When the lookups pay.  One lane a ray: from a share of empty macrocells (class > 0)
// of 0.1 on; frames of volumes 11 to 90% empty run 1.01 to 6 times as fast, batches
// from 12% on.  Several lanes a ray take a whole macrocell in one group, so a
// skip saves little but deep in empty space, and what tells is the share of macrocells
// of class 3 or more (none may contribute within two): frames with lookups, 400^2
// and 150^2 pixels, against without, by that share (of three kinds of data at 11
// to 90% empty):
//   256^3 u8    4 lanes  .06 0.91  .10 0.99  .16 1.04  .25 1.08    16 lanes  .12 0.94  .32 0.93  .42 1.01  .51 1.21
//   256^3 FP32  4 lanes  .06 0.91  .10 0.98  .16 1.05  .25 1.11    16 lanes  .12 1.03  .32 0.97  .42 1.10  .51 1.28
//   448^3 u8    4 lanes  .02 0.96  .05 1.05  .10 1.09  .26 1.23    16 lanes  .12 0.94  .17 0.99  .25 1.03  .52 1.22
//   448^3 FP32  4 lanes  .02 0.97  .05 1.05  .10 1.16  .26 1.55    16 lanes  .05 1.01  .17 1.13  .25 1.18  .52 1.37
// So the lines fall with the pool's size, as samples cost more where the caches do not
// hold them. Pages of fewer than 6 macrocells an edge (32^3 bricks) count as deep more
// than they save, since a page sees only itself: twice the share, and nothing for 16
// lanes, whose group crosses half of such a page. Batches: one lane as frames (24
// views at 256 to 384 pixels: 15% 1.02, 40% 1.21, 60% 1.52; 8 at 128 to 160 break even
// at a third); four lanes, 0.98 to 1.21 in eight batches with .16 to .26 deep. At 0.1
// of empties for all of them a 160^2 frame of the 256^3 FP32 volume, 30% empty, took
// 235 us for 191 without.
constexpr double kWorthEmpty = 0.1, kWorthBatch = 0.12, kWorthBatchDeep = 0.1;
constexpr int kSmallPage = 6;
double worth_deep(int32_t lanes, int nm, double pool_bytes) {
  const double l = std::log2(1.0 + pool_bytes / 24e6);
  const double share = lanes == 4 ? std::max(0.02, 0.17 - 0.033 * l) : std::max(0.05, 0.39 - 0.06 * l);
  return nm < kSmallPage ? 2.0 * share : share;
}

// Macrocells (of 512 voxels) from which an upload takes the ranges behind its copy, where
// they are lost in it (40 of 2400 us for one 256^3 FP32 page); a kernel behind the copy of
// a 32^3 u8 page made its upload 45 us of 28.
constexpr size_t kRangesWithUpload = 8192;

size_t page_cells(const Ctx *c) {
  const size_t nm = (size_t)macro_edge(c->pool.pad);
  return nm * nm * nm;
}

constexpr size_t kCounts = 6;   // two slots of the frame classes, and the batch's
constexpr int kBatchCounts = 4;

bool reserve(Ctx *c, size_t cells) {
  if (c->macro_cap >= cells) return true;
  macro_free(c);
  const size_t counts = kCounts * sizeof(*c->own_mcount);
  if (hipMalloc((void **)&c->own_mm, cells * sizeof(float2)) != hipSuccess ||
      hipMalloc((void **)&c->own_mcls, cells) != hipSuccess ||
      hipMalloc((void **)&c->own_mcount, counts) != hipSuccess ||
      hipMemsetAsync(c->own_mcount, 0, counts, c->stream) != hipSuccess ||
      hipEventCreateWithFlags(&c->macro_ev, hipEventDisableTiming) != hipSuccess) {
    (void)hipGetLastError();   // no memory for them: the marches sample everything
    macro_free(c);
    return false;
  }
  c->mcount_slot = 0;
  c->macro_cap = cells;
  return true;
}

MacroRuns run_of(int32_t first, int32_t n) {
  MacroRuns r{};
  r.n = 1;
  r.total = n;
  r.first[0] = first;
  return r;
}

int32_t ranges(Ctx *c, const MacroRuns &r) {
  HYD_CHECK_HIP(launch_macro_minmax(c->pool.fmt, c->pool.data, c->pool.pad, r, c->own_mm, c->stream));
  return HYD_OK;
}

int32_t classes(Ctx *c, const MacroRuns &r, bool replace) {
  const float scale = c->pool.fmt == HYD_FMT_U8 ? 1.f / 255.f : 1.f;
  if (!replace) c->mcount_slot ^= 1;   // zero: the last full pass or reserve() made it so
  HYD_CHECK_HIP(launch_macro_classes(c->own_mm, c->pool.pad, r, c->tf, c->tf_n, scale, nullptr, c->own_mcls, replace,
                                     c->own_mcount + 2 * c->mcount_slot,
                                     replace ? nullptr : c->own_mcount + 2 * (c->mcount_slot ^ 1), c->stream));
  return HYD_OK;
}

// Complete on return, with the shares of the batch's classes.
int32_t batch_classes(Ctx *c, const MacroRuns &r, bool replace) {
  unsigned long long *counts = c->own_mcount + kBatchCounts, n[2] = {0, 0};
  if (!replace) HYD_CHECK_HIP(hipMemcpyAsync(counts, n, sizeof(n), hipMemcpyHostToDevice, c->stream));
  HYD_CHECK_HIP(launch_macro_classes(c->own_mm, c->pool.pad, r, c->tf, c->tf_n, 1.f, c->own_bscale, c->own_bcls,
                                     replace, counts, nullptr, c->stream));
  HYD_CHECK_HIP(hipMemcpyAsync(n, counts, sizeof(n), hipMemcpyDeviceToHost, c->stream));
  HYD_CHECK_HIP(hipStreamSynchronize(c->stream));
  const double cells = (double)c->pool.n_pages * (double)page_cells(c);
  c->bcls_empty = 1.0 - (double)n[0] / cells;
  c->bcls_deep = (double)n[1] / cells;
  return HYD_OK;
}

// Puts the context's stream behind the last update of the ranges and frame classes,
// which may have been queued on another.
int32_t await(Ctx *c) {
  if (!c->macro_pending) return HYD_OK;
  const hipError_t e = hipEventQuery(c->macro_ev);
  if (e == hipErrorNotReady) {
    (void)hipGetLastError();
    HYD_CHECK_HIP(hipStreamWaitEvent(c->stream, c->macro_ev, 0));
    return HYD_OK;
  }
  HYD_CHECK_HIP(e);
  c->macro_pending = false;
  return HYD_OK;
}

// Brings the ranges, and with_classes the frame classes, up to date on the
// context's stream.
int32_t refresh(Ctx *c, bool with_classes) {
  int32_t st = await(c);
  if (st) return st;
  std::vector<std::pair<int32_t, int32_t>> &d = c->mm_dirty;
  const bool dirty = !d.empty(), make = with_classes && !c->mcls_valid;
  if (!dirty && !make) return HYD_OK;
  const bool update = dirty && c->mcls_valid;
  c->mcls_valid = false;   // until all of it is queued
  if (dirty) {
    std::sort(d.begin(), d.end());
    MacroRuns r{};
    for (const auto &[first, n] : d) {   // each page once: the counts follow its old and new classes
      const int32_t end = first + n, last = r.n > 0 ? r.first[r.n - 1] + (r.total - r.start[r.n - 1]) : -1;
      if (end <= last) continue;
      const int32_t from = std::max(first, last);
      r.first[r.n] = from;
      r.start[r.n++] = r.total;
      r.total += end - from;
    }
    if ((st = ranges(c, r)) || (update && (st = classes(c, r, true)))) return st;
  }
  if (make && (st = classes(c, run_of(0, c->pool.n_pages), false))) return st;
  HYD_CHECK_HIP(hipEventRecord(c->macro_ev, c->stream));
  c->macro_pending = true;
  d.clear();
  c->mcls_valid = update || make;
  return HYD_OK;
}

}  // namespace

void macro_free(Ctx *c) {
  for (void *p : {(void *)c->own_mm, (void *)c->own_mcls, (void *)c->own_mcount, (void *)c->own_bscale,
                  (void *)c->own_bcls})
    if (p) (void)hipFree(p);
  if (c->macro_ev) (void)hipEventDestroy(c->macro_ev);
  c->macro_ev = nullptr;
  c->macro_pending = false;
  c->own_mm = nullptr;
  c->own_mcls = nullptr;
  c->own_mcount = nullptr;
  c->own_bscale = nullptr;
  c->own_bcls = nullptr;
  c->bcls_cap = c->bscale_cap = 0;
  c->bcls_gen = ~0ull;
  c->macro_cap = 0;
  c->mm_gen = ~0ull;
  c->mm_dirty.clear();
  c->mcls_valid = false;
}

int32_t macro_pool_uploaded(Ctx *c) {
  c->mcls_valid = false;
  c->mm_gen = ~0ull;
  c->mm_dirty.clear();
  if (!reserve(c, (size_t)c->pool.n_pages * page_cells(c))) return HYD_OK;
  c->mm_gen = c->pool_gen;
  if ((size_t)c->pool.n_pages * page_cells(c) < kRangesWithUpload) {
    c->mm_dirty.emplace_back(0, c->pool.n_pages);   // taken with the classes
    return HYD_OK;
  }
  int32_t st = ranges(c, run_of(0, c->pool.n_pages));
  if (st) c->mm_gen = ~0ull;
  return st;
}

int32_t macro_pages_written(Ctx *c, int32_t first, int32_t n) {
  if (c->mm_gen != c->pool_gen || n <= 0) return HYD_OK;
  if (c->bcls_gen == c->batch_state_gen) {   // in place: captured graphs read them
    const MacroRuns r = run_of(first, n);
    int32_t st = await(c);
    if (st || (st = ranges(c, r)) || (st = batch_classes(c, r, true))) return st;
    if (!c->mcls_valid) return HYD_OK;   // the frame classes will be made from these ranges
  }
  std::vector<std::pair<int32_t, int32_t>> &d = c->mm_dirty;
  for (auto &[f, k] : d) {
    if (first >= f && first + n <= f + k) return HYD_OK;
    if (first == f + k) {   // pages in their order extend a run
      k += n;
      return HYD_OK;
    }
  }
  d.emplace_back(first, n);
  return d.size() < (size_t)kMacroRuns ? (int32_t)HYD_OK : refresh(c, false);
}

// Classes of every page under the scale of the volumes that name it, for the
// batched march: made once per state of pool, table and volume set.
int32_t macro_batch(Ctx *c, int32_t lanes, const uint8_t **cls) {
  *cls = nullptr;
  // a zero contribution leaves the composite as it is while colours are finite
  if (!c->tf_finite || !(c->tf_rgb_max <= 1e15f) || !(c->tf_alpha_min >= 0.f)) return HYD_OK;
  // without oriented copies the march reads a bound pool as it is at the launch
  if (!c->pool.owned && !c->own_oriented) return HYD_OK;
  const size_t n = (size_t)c->pool.n_pages, cells = n * page_cells(c);
  if (c->bcls_gen != c->batch_state_gen) {
    if (capturing(c)) return HYD_OK;   // made by the next launch outside it
    c->bcls_gen = ~0ull;
    if (cells > 0xffffffffull || !reserve(c, cells)) return HYD_OK;   // 32-bit class offsets
    if (c->bcls_cap < cells || c->bscale_cap < n) {
      for (void *p : {(void *)c->own_bscale, (void *)c->own_bcls})
        if (p) (void)hipFree(p);
      c->own_bscale = nullptr;
      c->own_bcls = nullptr;
      c->bcls_cap = c->bscale_cap = 0;
      if (hipMalloc((void **)&c->own_bscale, n * sizeof(float)) != hipSuccess ||
          hipMalloc((void **)&c->own_bcls, cells) != hipSuccess) {
        (void)hipGetLastError();
        return HYD_OK;
      }
      c->bcls_cap = cells;
      c->bscale_cap = n;
    }
    int32_t st = HYD_OK;
    if (c->mm_gen != c->pool_gen) {   // a bound pool's, with its oriented copies
      if ((st = ranges(c, run_of(0, (int32_t)n)))) return st;
      c->mm_gen = c->pool_gen;
      c->mm_dirty.clear();
      c->mcls_valid = false;
    }
    if ((st = refresh(c, false))) return st;
    std::vector<float> scale(n, 0.f);   // the set's pages lie in the pool (fill_args)
    for (const auto &[pg, sc] : c->vol_pages) scale[pg] = scale[pg] == 0.f || scale[pg] == sc ? sc : NAN;
    for (float &sc : scale) sc = sc == 0.f ? NAN : sc;
    HYD_CHECK_HIP(hipMemcpyAsync(c->own_bscale, scale.data(), n * sizeof(float), hipMemcpyHostToDevice, c->stream));
    if ((st = batch_classes(c, run_of(0, (int32_t)n), false))) return st;
    c->bcls_gen = c->batch_state_gen;
  }
  if (lanes > 1 ? c->bcls_deep >= kWorthBatchDeep : c->bcls_empty >= kWorthBatch) *cls = c->own_bcls;
  return HYD_OK;
}

namespace {
// The grid for marches within [bmin, bmax]; false when it does not apply.
bool grid_of(const Ctx *c, f3 bmin, f3 bmax, MacroGrid &g) {
  if (!c->pool.owned || c->mm_gen != c->pool_gen) return false;
  // every page has the same mapping, one b on each axis, inside the page
  const float k = c->page_k_min, lo = c->page_lo;
  if (!(k > 0.f && c->page_k_max == k && lo >= 0.f && c->page_hi == k + lo && k + lo <= 1.000001f)) return false;
  const size_t cells = page_cells(c);
  if ((uint64_t)c->pool.n_pages * cells > 0xffffffffull) return false;   // 32-bit class offsets
  // n position additions at coordinates up to D voxels round by at most n D
  // 2^-24 voxels, which has to stay below kMacroSlack
  float ext = 0.f;
  for (float v : {bmin.x, bmin.y, bmin.z, bmax.x, bmax.y, bmax.z}) ext = std::max(ext, std::fabs(v));
  const float K = k * float(c->pool.pad);
  const float run = kMacroSlack * 16777216.f / (ext * K);
  if (!(run >= 8.f)) return false;
  g.nm = macro_edge(c->pool.pad);
  g.cells = (int32_t)cells;
  g.K = K;
  g.B = lo * float(c->pool.pad) - 0.5f;
  g.run_max = std::min(std::floor(run), 4096.f);
  return true;
}
}  // namespace

int32_t macro_fill(Ctx *c, VolumeArgs &a) {
  // opacities in [0, 1] and colours whose length is finite keep the composite
  // finite, so that a zero contribution leaves it as it is
  if (!a.monotone || !(c->tf_rgb_max <= 1e15f)) return HYD_OK;
  if (a.mode == HYD_MODE_PARTITION && !(std::fabs(a.rank) <= 1e15f)) return HYD_OK;
  const int nm = macro_edge(c->pool.pad);
  if (a.lanes == 16 && nm < kSmallPage) return HYD_OK;
  if (!grid_of(c, a.bmin, a.bmax, a.macro)) return HYD_OK;
  int32_t st = refresh(c, true);
  if (st) return st;
  const double cells = (double)c->pool.n_pages * (double)page_cells(c);
  const double bytes = (double)a.pool_elems * (c->pool.fmt == HYD_FMT_U8 ? 1 : c->pool.fmt == HYD_FMT_F16 ? 2 : 4);
  a.macro.cls = c->own_mcls;
  a.macro.count = c->own_mcount + 2 * c->mcount_slot + (a.lanes > 1 ? 1 : 0);
  a.macro.count_min = a.lanes > 1 ? (unsigned long long)std::ceil(worth_deep(a.lanes, nm, bytes) * cells) : 0;
  a.macro.count_max = a.lanes > 1 ? ~0ull : (unsigned long long)((1.0 - kWorthEmpty) * cells);
  return HYD_OK;
}

int32_t macro_fill_iso(Ctx *c, IsoArgs &a) {
  if (!grid_of(c, a.bmin, a.bmax, a.macro)) return HYD_OK;
  int32_t st = refresh(c, false);
  if (st) return st;
  a.mm = c->own_mm;
  a.mm_scale = c->pool.fmt == HYD_FMT_U8 ? 1.f / 255.f : 1.f;
  return HYD_OK;
}

}  // namespace hyd
