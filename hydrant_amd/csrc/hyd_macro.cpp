// Host side of the macrocells: when they are made and when a march may use them.
#include <algorithm>
#include <cmath>
#include <vector>

#include "hyd_macro.hpp"

namespace hyd {
namespace {

// Share of empty macrocells from which a frame looks them up: the lookups cost
// about 5% of a march (the 1024^3 fBm volume, 16% empty, breaks even: 186 and 187
// us a paged frame without and with them), and 44% empty saves 27% of it.
constexpr double kMacroWorth = 0.1;

size_t page_cells(const Ctx *c) {
  const size_t nm = (size_t)macro_edge(c->pool.pad);
  return nm * nm * nm;
}

bool reserve(Ctx *c, size_t cells) {
  if (c->macro_cap >= cells) return true;
  macro_free(c);
  if (hipMalloc((void **)&c->own_mm, cells * sizeof(float2)) != hipSuccess ||
      hipMalloc((void **)&c->own_mflags, cells) != hipSuccess ||
      hipMalloc((void **)&c->own_mcls, cells) != hipSuccess ||
      hipMalloc((void **)&c->own_mcount, sizeof(*c->own_mcount)) != hipSuccess) {
    (void)hipGetLastError();   // no memory for them: the marches sample everything
    macro_free(c);
    return false;
  }
  c->macro_cap = cells;
  return true;
}

int32_t batch_classes(Ctx *c, int32_t first, int32_t n) {
  HYD_CHECK_HIP(launch_macro_classes(c->own_mm, c->pool.pad, first, n, c->tf, c->tf_n, 1.f, c->own_bscale,
                                     c->own_bflags, c->own_bcls, c->own_mcount, c->stream));
  return HYD_OK;
}

int32_t classes(Ctx *c, int32_t first, int32_t n) {
  const float scale = c->pool.fmt == HYD_FMT_U8 ? 1.f / 255.f : 1.f;
  HYD_CHECK_HIP(launch_macro_classes(c->own_mm, c->pool.pad, first, n, c->tf, c->tf_n, scale, nullptr,
                                     c->own_mflags, c->own_mcls, c->own_mcount, c->stream));
  return HYD_OK;
}

}  // namespace

void macro_free(Ctx *c) {
  for (void *p : {(void *)c->own_mm, (void *)c->own_mflags, (void *)c->own_mcls, (void *)c->own_mcount})
    if (p) (void)hipFree(p);
  c->own_mm = nullptr;
  c->own_mflags = c->own_mcls = nullptr;
  c->own_mcount = nullptr;
  for (void *p : {(void *)c->own_bscale, (void *)c->own_bflags, (void *)c->own_bcls})
    if (p) (void)hipFree(p);
  c->own_bscale = nullptr;
  c->own_bflags = c->own_bcls = nullptr;
  c->bcls_cap = c->bscale_cap = 0;
  c->bcls_gen = ~0ull;
  c->macro_cap = 0;
  c->mm_gen = ~0ull;
  c->mcls_valid = false;
}

int32_t macro_pool_uploaded(Ctx *c) {
  c->mcls_valid = false;
  c->mm_gen = ~0ull;
  if (!reserve(c, (size_t)c->pool.n_pages * page_cells(c))) return HYD_OK;
  HYD_CHECK_HIP(launch_macro_minmax(c->pool.fmt, c->pool.data, c->pool.pad, 0, c->pool.n_pages, c->own_mm,
                                    c->stream));
  c->mm_gen = c->pool_gen;
  return c->tf ? macro_tf_set(c) : HYD_OK;   // the caller waits for the stream
}

int32_t macro_tf_set(Ctx *c) {
  c->mcls_valid = false;
  if (c->mm_gen != c->pool_gen) return HYD_OK;
  unsigned long long n = 0;
  HYD_CHECK_HIP(hipMemcpyAsync(c->own_mcount, &n, sizeof(n), hipMemcpyHostToDevice, c->stream));
  int32_t st = classes(c, 0, c->pool.n_pages);
  if (st) return st;
  HYD_CHECK_HIP(hipMemcpyAsync(&n, c->own_mcount, sizeof(n), hipMemcpyDeviceToHost, c->stream));
  HYD_CHECK_HIP(hipStreamSynchronize(c->stream));   // complete before a march on another stream reads them
  c->macro_empty = 1.0 - (double)n / ((double)c->pool.n_pages * (double)page_cells(c));
  c->mcls_valid = true;
  return HYD_OK;
}

int32_t macro_pages_written(Ctx *c, int32_t first, int32_t n) {
  if (c->mm_gen != c->pool_gen || n <= 0) return HYD_OK;
  HYD_CHECK_HIP(launch_macro_minmax(c->pool.fmt, c->pool.data, c->pool.pad, first, n, c->own_mm, c->stream));
  if (c->mcls_valid) {
    int32_t st = classes(c, first, n);
    if (st) return st;
  }
  if (c->bcls_gen == c->batch_state_gen) {   // in place: captured graphs read them
    int32_t st = batch_classes(c, first, n);
    if (st) return st;
  }
  HYD_CHECK_HIP(hipStreamSynchronize(c->stream));
  return HYD_OK;
}

// Classes of every page under the scale of the volumes that name it, for the
// batched march: made once per state of pool, table and volume set.
int32_t macro_batch(Ctx *c, const uint8_t **cls) {
  *cls = nullptr;
  // a zero contribution leaves the composite as it is while colours are finite
  if (!c->tf_finite || !(c->tf_rgb_max <= 1e15f) || !(c->tf_alpha_min >= 0.f)) return HYD_OK;
  const size_t n = (size_t)c->pool.n_pages, cells = n * page_cells(c);
  if (c->bcls_gen != c->batch_state_gen) {
    if (capturing(c)) return HYD_OK;   // made by the next launch outside it
    c->bcls_gen = ~0ull;
    if (cells > 0xffffffffull || !reserve(c, cells)) return HYD_OK;   // 32-bit class offsets
    if (c->bcls_cap < cells || c->bscale_cap < n) {
      for (void *p : {(void *)c->own_bscale, (void *)c->own_bflags, (void *)c->own_bcls})
        if (p) (void)hipFree(p);
      c->own_bscale = nullptr;
      c->own_bflags = c->own_bcls = nullptr;
      c->bcls_cap = c->bscale_cap = 0;
      if (hipMalloc((void **)&c->own_bscale, n * sizeof(float)) != hipSuccess ||
          hipMalloc((void **)&c->own_bflags, cells) != hipSuccess ||
          hipMalloc((void **)&c->own_bcls, cells) != hipSuccess) {
        (void)hipGetLastError();
        return HYD_OK;
      }
      c->bcls_cap = cells;
      c->bscale_cap = n;
    }
    if (c->mm_gen != c->pool_gen) {   // a bound pool's, with its oriented copies
      HYD_CHECK_HIP(launch_macro_minmax(c->pool.fmt, c->pool.data, c->pool.pad, 0, (int)n, c->own_mm, c->stream));
      c->mm_gen = c->pool_gen;
      c->mcls_valid = false;
    }
    std::vector<float> scale(n, 0.f);   // the set's pages lie in the pool (fill_args)
    for (const auto &[pg, sc] : c->vol_pages) scale[pg] = scale[pg] == 0.f || scale[pg] == sc ? sc : NAN;
    for (float &sc : scale) sc = sc == 0.f ? NAN : sc;
    unsigned long long count = 0;
    HYD_CHECK_HIP(hipMemcpyAsync(c->own_bscale, scale.data(), n * sizeof(float), hipMemcpyHostToDevice, c->stream));
    HYD_CHECK_HIP(hipMemcpyAsync(c->own_mcount, &count, sizeof(count), hipMemcpyHostToDevice, c->stream));
    int32_t st = batch_classes(c, 0, (int32_t)n);
    if (st) return st;
    HYD_CHECK_HIP(hipMemcpyAsync(&count, c->own_mcount, sizeof(count), hipMemcpyDeviceToHost, c->stream));
    HYD_CHECK_HIP(hipStreamSynchronize(c->stream));
    c->bcls_empty = 1.0 - (double)count / (double)cells;
    c->bcls_gen = c->batch_state_gen;
  }
  if (c->bcls_empty >= kMacroWorth) *cls = c->own_bcls;
  return HYD_OK;
}

namespace {
// The grid for marches within [bmin, bmax]; false when it does not apply.
bool grid_of(const Ctx *c, f3 bmin, f3 bmax, MacroGrid &g) {
  if (!c->pool.owned || c->mm_gen != c->pool_gen || capturing(c)) return false;
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

void macro_fill(const Ctx *c, VolumeArgs &a) {
  if (!c->mcls_valid || c->macro_empty < kMacroWorth || !grid_of(c, a.bmin, a.bmax, a.macro)) return;
  // opacities in [0, 1] and colours whose length is finite keep the composite
  // finite, so that a zero contribution leaves it as it is
  if (!a.monotone || !(c->tf_rgb_max <= 1e15f)) return;
  if (a.mode == HYD_MODE_PARTITION && !(std::fabs(a.rank) <= 1e15f)) return;
  a.macro.cls = c->own_mcls;
}

void macro_fill_iso(const Ctx *c, IsoArgs &a) {
  if (!grid_of(c, a.bmin, a.bmax, a.macro)) return;
  a.mm = c->own_mm;
  a.mm_scale = c->pool.fmt == HYD_FMT_U8 ? 1.f / 255.f : 1.f;
}

}  // namespace hyd
