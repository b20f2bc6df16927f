// Macrocells: which 8^3 blocks of tap cells of a brick cannot contribute.
//
// A march spends its time on sampling (taps, interpolation, transfer function).
// Under a transfer function whose alpha is zero over a block's value range
// those samples composite exactly nothing, so a march that knows the block may
// advance over it with the position updates alone: the same samples, the same
// escalation, the same image bit for bit, without their loads and arithmetic.
//
// 8^3: a run of about ten half-voxel samples per macrocell pays for the lookup,
// and 38% of the 256^3 blob volume lies in empty ones (4^3: 42%, 16^3: 30%).
// 512^2 FP32 frame of it: 471 -> 345 us; ragged 765 x 431 FP16 lattice frame of
// a 500^3 one: 1517 -> 725 us, grouped samples included.
//
// Macrocell (mx, my, mz) of a page holds the tap cells whose lower tap index
// lies in [8m, 8m + 7] on each axis (voxels 8m .. 8m + 8).  Its class is 0 when
// it may contribute, else the Chebyshev radius d >= 1 such that every macrocell
// of the page within distance d - 1 is empty (at most kMacroCap).
#pragma once

#include "hyd_internal.hpp"

namespace hyd {

constexpr int kMacro = 8;      // tap cells per macrocell edge
constexpr int kMacroCap = 4;   // largest class

inline int macro_edge(int pad) { return (pad + kMacro - 1) / kMacro; }

// Position slack in voxels: a run of skipped samples ends this far inside the
// box it crosses, and starts at least kMacroGuard inside its macrocell.  The
// host bounds the run so that the rounding of its position additions stays
// below kMacroSlack.
constexpr float kMacroSlack = 1.f / 64.f;
constexpr float kMacroGuard = 1.f / 1024.f;

// Whether enough macrocells are empty for the lookups to pay: read by the march, since
// the host would have to wait for the count.
__device__ __forceinline__ bool macro_pays(const MacroGrid &g) {
  if (!g.cls) return false;
  const unsigned long long n = *g.count;
  return n >= g.count_min && n <= g.count_max;
}

// How far outside [lo, hi] a value interpolated in it may lie: the rounding of
// three lerps, 2^-19 of the range's magnitude; below the normal floats it no longer
// shrinks with it (half the least denormal rounds to zero).  The ranges are kept widened
// by it, so that a lookup compares and no more.
__device__ __forceinline__ float range_margin(float lo, float hi) {
  return fmaf(fmaxf(fabsf(lo), fabsf(hi)), 1.9073486e-6f, 1e-37f);
}

// Macrocell coordinate (clamped to the page) of a tap coordinate / 8.
__device__ __forceinline__ float macro_floor(float f8, float hi) {
  return __builtin_amdgcn_fmed3f(floorf(f8), 0.f, hi);
}

// Index of x's macrocell among the pool's, the cell clamped to its page (x
// in brick coordinates, x = o - floor(o)).  Float arithmetic good to far below
// kMacroGuard; page * cells stays below 2^32 (the host sees to it).
__device__ __forceinline__ uint32_t macro_index(const MacroGrid &g, int pgid, f3 x) {
  const float inv8 = 1.f / float(kMacro), hi = float(g.nm - 1), k8 = g.K * inv8, b8 = g.B * inv8;
  const float mx = macro_floor(fmaf(x.x, k8, b8), hi), my = macro_floor(fmaf(x.y, k8, b8), hi),
              mz = macro_floor(fmaf(x.z, k8, b8), hi);
  const uint32_t cell = (uint32_t)fmaf(fmaf(mz, float(g.nm), my), float(g.nm), mx);   // nm <= 128: below 2^24
  return (uint32_t)pgid * (uint32_t)g.cells + cell;
}

// Class of the macrocell at x (brick coordinates, x = o - floor(o)) of page
// pgid.  A march issues this load with the tap loads of a group for the
// position that follows the group, so that it never waits for it before
// sampling.
__device__ __forceinline__ int macro_class(const MacroGrid &g, int pgid, f3 x) { return g.cls[macro_index(g, pgid, x)]; }

// Number of samples from x in steps of d * sstep that lie in empty macrocells
// of the page, starting with the one at x, given the class c >= 1 of x's
// macrocell; 0 when x is too near its faces to tell.  invr = 1 / d.
__device__ __forceinline__ int macro_run(const MacroGrid &g, int c, f3 x, f3 invr, float sstep) {
  const float inv8 = 1.f / float(kMacro), hi = float(g.nm - 1), h = 0.5f * float(kMacro);
  const float fx = fmaf(x.x, g.K, g.B), fy = fmaf(x.y, g.K, g.B), fz = fmaf(x.z, g.K, g.B);
  const float gx = fmaf(macro_floor(fx * inv8, hi), float(kMacro), h), gy = fmaf(macro_floor(fy * inv8, hi), float(kMacro), h),
              gz = fmaf(macro_floor(fz * inv8, hi), float(kMacro), h);
  const float off = fmaxf(fmaxf(fabsf(fx - gx), fabsf(fy - gy)), fabsf(fz - gz));
  if (off > h - kMacroGuard) return 0;
  // the empty box, clipped to the brick; the exit face of each axis, kMacroSlack inside
  const float r = float(kMacro) * (float(c) - 0.5f) - kMacroSlack;
  const float bl = g.B + kMacroSlack, bh = g.B + g.K - kMacroSlack;
  const float ex = invr.x > 0.f ? fminf(gx + r, bh) : fmaxf(gx - r, bl);
  const float ey = invr.y > 0.f ? fminf(gy + r, bh) : fmaxf(gy - r, bl);
  const float ez = invr.z > 0.f ? fminf(gz + r, bh) : fmaxf(gz - r, bl);
  const float t = fminf(fminf((ex - fx) * invr.x, (ey - fy) * invr.y), (ez - fz) * invr.z);
  const float n = t * __builtin_amdgcn_rcpf(g.K * sstep);   // steps that stay inside the box
  if (!(n >= 0.f)) return 0;
  return (int)fminf(n + 1.f, g.run_max);
}

// Runs of pages that a launch works on, one after another.
constexpr int kMacroRuns = 64;
struct MacroRuns {
  int32_t n, total;                             // runs, pages in all
  int32_t first[kMacroRuns], start[kMacroRuns];   // each run's first page and the pages before it
};

// mm: {min, max} of every macrocell's voxels as stored (u8 as counts), widened by
// range_margin(); {NaN, NaN} when a voxel is not finite or beyond 1e30.
hipError_t launch_macro_minmax(int fmt, const void *pool, int pad, const MacroRuns &runs, float2 *mm, hipStream_t s);
// Classes under a transfer function (value = stored * scale; page_scale, if not
// null, holds each page's own scale, NaN: never empty).  counts[0] and counts[1]
// gain the macrocells of class 0 and of class 3 or more; replace: and lose those of
// the classes that stood there.  Two counts at zero (if not null) are set to 0.
hipError_t launch_macro_classes(const float2 *mm, int pad, const MacroRuns &runs, const float *tf, int tf_n, float scale,
                                const float *page_scale, uint8_t *cls, bool replace, unsigned long long *counts,
                                unsigned long long *zero, hipStream_t s);

}  // namespace hyd
