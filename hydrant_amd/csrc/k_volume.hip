// Volume ray-march kernels for gfx950.
//
// One, 4 or 16 lanes per pixel; a 64-lane workgroup covers the tile of its rays
// (8x8 pixels at one lane), so a wavefront marches a coherent ray packet.  Ray emit, box clip and the march
// loop are fused (the reference splits them over ray_emit_kernel_impl and a
// device-function-pointer call to VolumeShaderKernel::main,
// src/slave/core/cuda_shading.cu:14-37 and volume_shader.cu:32-81).
//
// Sampling is done in software with the reference CPU backend's exact
// arithmetic (CpuSampler, include/hydrant/bridge/cpu_sampler.hpp:88-166):
// hardware texture filtering would not reproduce it.  The transfer function is
// staged in LDS per workgroup.
#include <hip/hip_fp16.h>

#include <cstdlib>
#include <type_traits>
#include <utility>

#include "hyd_internal.hpp"
#include "hyd_macro.hpp"
#include "hyd_sampler.hpp"

namespace hyd {
namespace {

constexpr int kTile = 8;           // 8x8 pixel packet per wavefront
constexpr int kMaxTf = 256;        // LDS capacity of the TF table (entries)

template <int FMT> struct Voxel;
template <> struct Voxel<HYD_FMT_F32> {
  static __device__ __forceinline__ float at(const void *base, size_t i) {
    return static_cast<const float *>(base)[i];
  }
};
template <> struct Voxel<HYD_FMT_F16> {
  static __device__ __forceinline__ float at(const void *base, size_t i) {
    return __half2float(static_cast<const __half *>(base)[i]);
  }
};
template <> struct Voxel<HYD_FMT_U8> {
  static __device__ __forceinline__ float at(const void *base, size_t i) {
    return u8_norm(static_cast<const uint8_t *>(base)[i]);
  }
};

// Point lookup in an int grid with Clamp addressing (Options::as_array,
// basic_renderer.hpp:147-159; CpuSampler filter_none).
__device__ __forceinline__ int grid_index(f3 p, const int32_t dim[3]) {
  float fx = gclamp(p.x, 0.f, float(dim[0]));
  float fy = gclamp(p.y, 0.f, float(dim[1]));
  float fz = gclamp(p.z, 0.f, float(dim[2]));
  int ix = iclamp((int)floorf(fx), 0, dim[0] - 1);
  int iy = iclamp((int)floorf(fy), 0, dim[1] - 1);
  int iz = iclamp((int)floorf(fz), 0, dim[2] - 1);
  return iz * dim[0] * dim[1] + iy * dim[0] + ix;
}

struct TapIdx { int ix, iy, iz, jx, jy, jz; };

// The last march sample's taps: first and last tap index (which fix all eight)
// and their values.
struct VolTaps {
  size_t id0 = ~(size_t)0, id7 = ~(size_t)0;
  float v[8];
};

// Brick sample: BlockSamplerMapping (k*x + b) then CpuSampler Wrap + Linear +
// normalised coordinates over a pad^3 brick (block_paging.hpp:11-36,
// cpu_sampler.hpp:88-104,142-166), for consecutive march samples of one ray:
// the eight taps are loaded only when they change (at half-voxel steps about
// half the samples share their predecessor's cell); the value does not depend
// on whether they were reloaded.
template <int FMT>
__device__ __forceinline__ float brick_sample_reuse(const void *pool, int pad, int pgid, float4 pg, f3 x,
                                                    TapIdx *taps, VolTaps &c) {
  const float fd = float(pad);
  float u[3] = {x.x * pg.x + pg.y, x.y * pg.x + pg.z, x.z * pg.x + pg.w};
  float a[3];
  int i[3], j[3];
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    float fx = fd * u[k];
    fx = wrap_mod(fx, fd);   // Wrap: glm mod(fx, fd)
    fx = fx - 0.5f;
    float flr = floorf(fx);
    a[k] = fx - flr;
    i[k] = iclamp((int)flr, 0, pad - 1);
    j[k] = iclamp((int)ceilf(fx), 0, pad - 1);
  }
  if (taps) *taps = TapIdx{i[0], i[1], i[2], j[0], j[1], j[2]};
  const size_t base = (size_t)pgid * pad * pad * pad;
  const size_t row_ii = base + ((size_t)i[2] * pad + i[1]) * pad;
  const size_t row_jj = base + ((size_t)j[2] * pad + j[1]) * pad;
  if (row_ii + i[0] != c.id0 || row_jj + j[0] != c.id7) {
    const size_t row_ji = base + ((size_t)i[2] * pad + j[1]) * pad;
    const size_t row_ij = base + ((size_t)j[2] * pad + i[1]) * pad;
    c.v[0] = Voxel<FMT>::at(pool, row_ii + i[0]); c.v[1] = Voxel<FMT>::at(pool, row_ii + j[0]);
    c.v[2] = Voxel<FMT>::at(pool, row_ji + i[0]); c.v[3] = Voxel<FMT>::at(pool, row_ji + j[0]);
    c.v[4] = Voxel<FMT>::at(pool, row_ij + i[0]); c.v[5] = Voxel<FMT>::at(pool, row_ij + j[0]);
    c.v[6] = Voxel<FMT>::at(pool, row_jj + i[0]); c.v[7] = Voxel<FMT>::at(pool, row_jj + j[0]);
    c.id0 = row_ii + i[0];
    c.id7 = row_jj + j[0];
  }
  const float ax = a[0], bx = 1.f - ax;
  float x00 = c.v[0] * bx + c.v[1] * ax;
  float x10 = c.v[2] * bx + c.v[3] * ax;
  float x01 = c.v[4] * bx + c.v[5] * ax;
  float x11 = c.v[6] * bx + c.v[7] * ax;
  const float ay = a[1], by = 1.f - ay;
  float y0 = x00 * by + x10 * ay;
  float y1 = x01 * by + x11 * ay;
  const float az = a[2], bz = 1.f - az;
  return y0 * bz + y1 * az;
}

// The transfer function in LDS, edge entries repeated: entry i + 1 holds tf[i],
// entry 0 tf[0] and entry n + 1 tf[n - 1], so the lookup needs no clamps; entries n + 2
// and n + 3 are zero, where a value outside [0, 1] looks (the Border).
constexpr int kTfLds = kMaxTf + 4;
__device__ __forceinline__ void stage_tf(float4 *ext, const float *tf, int n) {
  for (int i = threadIdx.x; i < n + 4; i += blockDim.x)
    ext[i] = i < n + 2 ? reinterpret_cast<const float4 *>(tf)[iclamp(i - 1, 0, n - 1)] : make_float4(0.f, 0.f, 0.f, 0.f);
}

// Transfer function: Border + Linear + normalised 1-D lookup
// (transfer_fn.hpp:14-28, cpu_sampler.hpp:117-124,142-166).  fx - 0.5 lies in
// [-0.5, n - 0.5], so floor + 1 indexes the staged table.  The upper entry is the next one
// wherever the weight is not zero; at weight zero the reference reads the lower
// entry twice, the same sum as with the next one while the table is finite
// (FINITE), which saves the select.
template <bool FINITE = false>
__device__ __forceinline__ float4 tf_sample(const float4 *ext, int n, float s) {
  const float fd = float(n);
  float fx = fd * s;
  fx = __builtin_amdgcn_fmed3f(fx, 0.f, fd) == fx ? fx : fd + 1.5f;   // outside, or NaN: the zero entries
  fx = fx - 0.5f;
  const float flr = floorf(fx);
  const float a = fx - flr, w = 1.f - a;
  const float4 *e = ext + ((int)flr + 1);
  const float4 p = e[0], q = e[FINITE || a != 0.f ? 1 : 0];
  return make_float4(p.x * w + q.x * a, p.y * w + q.y * a, p.z * w + q.z * a, p.w * w + q.w * a);
}

struct MarchState {
  f3 o, d;
  int nsteps, step_size;
  float4 v;
  f3 theta;
  float phi;
};

// Shade one resolved sample and composite it front to back
// (volume_shader.cu:52-70, plus the density scale on the TF alpha).  theta and
// phi are carried only for a film (the fetch pass exports them); without one
// they are never observed and THETA = false leaves them out.
// shade_sample gives the premultiplied colour of a sample (it does not depend
// on the ray's state), composite_ub adds it behind what the ray holds.
template <bool WEIGHTED = false, bool FINITE = false>
__device__ __forceinline__ float4 shade_sample(const VolumeArgs &a, const float4 *tf, float s, int pgid, float w) {
  float4 ub = tf_sample<FINITE>(tf, a.tf_n, s);
  ub.w = ub.w * a.density;
  if (WEIGHTED) ub.w = ub.w * w;
  if (__builtin_expect(a.mode != HYD_MODE_DEFAULT, 0)) {   // one uniform branch a sample
    if (a.mode == HYD_MODE_PARTITION) {
      float l = length3(f3{ub.x, ub.y, ub.z});
      float r = a.rank, q = 1.f - r;
      ub = make_float4((1.f * q + 0.f * r) * l, (0.f * q + 0.f * r) * l, (0.f * q + 1.f * r) * l, ub.w);
    } else {
      ub = pgid >= a.lowest_blkcnt ? make_float4(0.f, 1.f, 0.f, ub.w) : make_float4(1.f, 0.f, 0.f, ub.w);
    }
  }
  const float aw = ub.w;
  ub.x = ub.x * aw; ub.y = ub.y * aw; ub.z = ub.z * aw;
  return ub;
}

template <bool THETA = true>
__device__ __forceinline__ void composite_ub(float4 ub, MarchState &st) {
  if (THETA) {
    st.theta.x = st.theta.x + ub.x * st.phi;
    st.theta.y = st.theta.y + ub.y * st.phi;
    st.theta.z = st.theta.z + ub.z * st.phi;
    st.phi = st.phi * (1.f - ub.w);
  }
  const float t = 1.f - st.v.w;
  st.v.x = st.v.x + ub.x * t;
  st.v.y = st.v.y + ub.y * t;
  st.v.z = st.v.z + ub.z * t;
  st.v.w = st.v.w + ub.w * t;
}

__device__ __forceinline__ void shade_composite(const VolumeArgs &a, const float4 *tf, float s, int pgid,
                                                MarchState &st) {
  composite_ub(shade_sample(a, tf, s, pgid, 1.f), st);
}

// The chebyshev and page-table entries of the brick the last sample fell in:
// consecutive samples inside one brick read them once (the page entry only
// for a non-empty brick).
// With the combined per-brick code (equal grid dims) this is one load.
struct BrickLookup {
  f3 ip = {-INFINITY, -INFINITY, -INFINITY};
  int cd = 0, gi = 0, pg = -1;
  // true when p is another brick
  __device__ __forceinline__ bool update(const VolumeArgs &a, f3 p) {
    if (p.x == ip.x && p.y == ip.y && p.z == ip.z) return false;
    ip = p;
    if (a.codes) {
      gi = grid_index(p, a.vdim);
      const int code = a.codes[gi];
      cd = code <= -2 ? -1 - code : 0;
      pg = code;
      return true;
    }
    cd = a.cheb[grid_index(p, a.cdim)];
    if (cd == 0) {
      gi = grid_index(p, a.vdim);
      pg = a.vaddr[gi];
    }
    return true;
  }
};

// Cell code of brick ip: page id, -1 not resident, or -1 - chebyshev distance.
__device__ __forceinline__ int cell_code(const VolumeArgs &a, f3 ip) {
  if (a.codes) return a.codes[grid_index(ip, a.vdim)];
  const int cd = a.cheb[grid_index(ip, a.cdim)];
  return cd ? -1 - cd : a.vaddr[grid_index(ip, a.vdim)];
}

// VolumeShaderKernel::main (volume_shader.cu:32-81), reference step schedule.
// The escalation tests compare float alpha with the double literals 0.93 and
// 0.85; for binary32 inputs `x > 0.93` equals `x >= 0.93f` (0.93f rounds up),
// likewise for 0.85.
template <int FMT, bool COUNT, bool TRACE>
__device__ void march_reference(const VolumeArgs &a, const float4 *tf, MarchState &st,
                                unsigned &count, hyd_trace_rec *trace, int max_trace, int &ntrace) {
  const float cdu = 1.f / comp_max(abs3(st.d));
  const f3 d = st.d;
  f3 o = st.o;
  int nsteps = st.nsteps;
  int step_size = st.step_size;
  VolTaps tc;                 // taps of the last sample
  int cpg = -1;               // page of the cached descriptor
  float4 pgd = make_float4(0.f, 0.f, 0.f, 0.f);
  BrickLookup bl;
  while (nsteps > 0) {
    const f3 ip = floor3(o);
    bl.update(a, ip);
    const int cd = bl.cd;
    if (cd) {
      // skip_nblock_steps (volume_shader.cu:5-14) with step * step_size
      const float sstep = a.step * float(step_size);
      float tn, tfar;
      intersect_box(o, d, ip, f3{ip.x + 1.f, ip.y + 1.f, ip.z + 1.f}, tn, tfar);
      const float di = ceilf((tfar + float(cd - 1) * cdu) / sstep);
      o = add(o, muls(muls(d, di), sstep));
      nsteps -= (int)di;
    } else {
      const int gi = bl.gi;
      const int pgid = bl.pg;
      if (pgid == -1) break;
      if (pgid != cpg) {
        pgd = a.page[pgid];
        cpg = pgid;
      }
      TapIdx taps;
      const float s = brick_sample_reuse<FMT>(a.pool, a.pad, pgid, pgd, sub(o, ip), TRACE ? &taps : nullptr,
                                              tc);
      if (TRACE && ntrace < max_trace) {
        const int gx = gi % a.vdim[0], gy = (gi / a.vdim[0]) % a.vdim[1], gz = gi / (a.vdim[0] * a.vdim[1]);
        trace[ntrace++] = hyd_trace_rec{gx, gy, gz, pgid, taps.ix, taps.iy, taps.iz, taps.jx, taps.jy, taps.jz};
      }
      shade_composite(a, tf, s, pgid, st);
      if (COUNT) ++count;
      if (st.v.w >= 0.93f) {
        step_size = 16;
      } else if (st.v.w >= 0.85f) {
        step_size = 4;
      }
    }
    o = add(o, muls(muls(d, a.step), float(step_size)));
    nsteps -= step_size;
  }
  st.o = o;
  st.nsteps = nsteps;
  st.step_size = step_size;
}

// ---------------------------------------------------------------------------
// The reference schedule with the tap loads of up to U consecutive samples in
// flight together.  A ray is one long chain of dependent samples, and a frame
// holds only a few waves per SIMD (one lane per pixel), so issuing one
// sample's loads and waiting for them before the next leaves the memory
// latency exposed on every sample.  Inside one brick the next sample positions
// follow from the current step size alone (o += (d * step) * step_size, the
// same binary32 operations one at a time), so a group of U samples resolves
// its positions, values and colours first (they do not depend on the ray's
// state) and then composites the samples in order.  (Skipping the loads of a
// sample whose cell repeats its predecessor's saved memory work, but its
// branches and register copies cost more instructions than the loads.)
// Escalation changes the step size; a group stops at the sample that escalates
// (the ones after it were placed with the old step and are dropped), so
// positions, taps, values and step budget are those of the one-sample-at-a-time
// march, bit for bit.  Samples are also cut at the brick's boundary and at the
// end of the step budget.
//
// Voxels are addressed by element offsets from the pool base: 32-bit when the
// pool is below 4 GiB (OFF = uint32_t, so the base stays in scalar registers),
// else 64-bit.

// Rays per wave below which a wave of the one-lane-per-ray march (FP32 and
// FP16 frames) hands its remaining rays to the cooperative march (kCoopLanes
// lanes per ray).  Measured when the paged 1024^3 u8 frame at 512^2 still ran
// one lane per ray: 0.587 ms without the handover; 0.543 / 0.519 / 0.550 /
// 0.565 ms with 2 / 4 / 8 / 16 lanes per ray.  The plain FP32 frame is
// unchanged by it: its last waves still hold more rays than the handover
// takes.
#ifndef HYD_COOP_LANES
#define HYD_COOP_LANES 4
#endif
constexpr int kCoopLanes = HYD_COOP_LANES;
constexpr int kCoopRays = 64 / kCoopLanes;

// Advances o over the samples that lie in empty macrocells of brick ip, where
// o's macrocell has class c >= 1: the march's own additions, one per sample,
// and its step budget, without the sampling.  Returns their number (0: the
// sample at o may contribute).
__device__ __forceinline__ int skip_empty(const VolumeArgs &a, int c, f3 ip, f3 invr, f3 inc,
                                          int step_size, f3 &o, int &nsteps) {
  // 1, 4 or 16; a film from elsewhere may hold anything
  if (step_size <= 0 || (step_size & (step_size - 1)) != 0) return 0;
  int n = macro_run(a.macro, c, sub(o, ip), invr, a.step * float(step_size));
  // samples left in the step budget: ceil(nsteps / step_size)
  n = min(n, (int)(((unsigned)nsteps + (unsigned)step_size - 1u) >> (31 - __clz(step_size))));
#pragma unroll 4
  for (int i = 0; i < n; ++i) o = add(o, inc);
  nsteps -= n * step_size;
  return n;
}

// Colours ub[j] of a group's samples x[j] (brick coordinates) where ok[j];
// WEIGHTED: their opacities scaled by w[j].
template <int FMT, class OFF, int N, bool WEIGHTED = false>
__device__ __forceinline__ void group_colours(const VolumeArgs &a, const float4 *tf, bool inner, const f3 (&x)[N],
                                              const bool (&ok)[N], float4 pgd, OFF page_base, int pgid,
                                              float4 (&ub)[N], const float *w = nullptr) {
  float s[N];
  group_values<FMT, OFF, N>(a.pool, a.pad, inner, x, ok, pgd, page_base, s);
  if (a.inner != kInnerNever) {   // the table is finite
#pragma unroll
    for (int j = 0; j < N; ++j) ub[j] = shade_sample<WEIGHTED, true>(a, tf, s[j], pgid, WEIGHTED ? w[j] : 1.f);
  } else {
#pragma unroll
    for (int j = 0; j < N; ++j) ub[j] = shade_sample<WEIGHTED, false>(a, tf, s[j], pgid, WEIGHTED ? w[j] : 1.f);
  }
}

// Alpha at which a sample changes the step (volume_shader.cu:71-76: v.w > 0.93
// gives 16, else v.w > 0.85 gives 4; see march_reference for the literals).  At 16
// with an alpha past 0.93 only a falling alpha does, which opacities in [0, 1] rule
// out; a film may hold a step of 16 at a lower alpha (written under other
// opacities), which the next escalation changes.
__device__ __forceinline__ float escalation_alpha(const VolumeArgs &a, int step_size, float alpha) {
  return step_size == 4 ? 0.93f : step_size == 16 && a.monotone && alpha >= 0.93f ? INFINITY : 0.85f;
}
__device__ __forceinline__ int escalated_step(float alpha, int step_size) {
  return alpha >= 0.93f ? 16 : alpha >= 0.85f ? 4 : step_size;
}

// Composites samples J .. N-1 of a group while they are valid and the alpha is
// below esc; n counts them.
template <int J, int N, bool THETA, class UB>
__device__ __forceinline__ void composite_group(const UB &ub, const bool (&ok)[N], float esc, MarchState &st, int &n) {
  composite_ub<THETA>(ub(std::integral_constant<int, J>{}), st);
  n = J + 1;
  if constexpr (J + 1 < N) {
    if (ok[J + 1] & !(st.v.w >= esc)) composite_group<J + 1, N, THETA>(ub, ok, esc, st, n);
  }
}

template <int FMT, int U, bool COUNT, bool THETA, class OFF>
__device__ void march_reference_grouped(const VolumeArgs &a, const float4 *tf, MarchState &st,
                                        unsigned &count, bool &handed) {
  const float cdu = 1.f / comp_max(abs3(st.d));
  const f3 d = st.d;
  const f3 invr = recip3(d);
  f3 o = st.o;
  int nsteps = st.nsteps;
  int step_size = st.step_size;
  const OFF pad3 = (OFF)a.pad * (OFF)a.pad * (OFF)a.pad;
  int cpg = -1;
  float4 pgd = make_float4(0.f, 0.f, 0.f, 0.f);
  OFF page_base = 0;
  BrickLookup bl;
  int cls = -1;   // class of o's macrocell (-1: not looked up)
  while (nsteps > 0) {
    // few rays left in this wave: the wave's lanes take them over together
    if (__popcll(__ballot(1)) <= kCoopRays) {
      handed = true;
      break;
    }
    const f3 ip = floor3(o);
    if (bl.update(a, ip)) cls = -1;
    if (bl.cd) {
      // skip_nblock_steps (volume_shader.cu:5-14) with step * step_size
      const float sstep = a.step * float(step_size);
      float tn, tfar;
      intersect_box_inv(o, invr, ip, f3{ip.x + 1.f, ip.y + 1.f, ip.z + 1.f}, tn, tfar);
      const float di = ceilf((tfar + float(bl.cd - 1) * cdu) / sstep);
      o = add(o, muls(muls(d, di), sstep));
      nsteps -= (int)di;
      o = add(o, muls(muls(d, a.step), float(step_size)));
      nsteps -= step_size;
      continue;
    }
    const int pgid = bl.pg;
    if (pgid == -1) break;
    if (pgid != cpg) {
      pgd = a.page[pgid];
      page_base = (OFF)pgid * pad3;
      cpg = pgid;
    }
    // positions of the group: the same additions the one-sample march makes
    const f3 inc = muls(muls(d, a.step), float(step_size));
    if (cls > 0) {   // samples in empty macrocells: their position updates alone
      const int k = skip_empty(a, cls, ip, invr, inc, step_size, o, nsteps);
      if (k > 0) {
        if (COUNT) count += (unsigned)k;
        cls = macro_class(a.macro, pgid, sub(o, ip));
        continue;
      }
    }
    f3 q = o, x[U];
    bool ok[U];
    x[0] = sub(o, ip);
    ok[0] = true;
    int left = nsteps;
#pragma unroll
    for (int j = 1; j < U; ++j) {
      q = add(q, inc);
      x[j] = sub(q, ip);
      left -= step_size;
      ok[j] = ok[j - 1] & (left > 0) & in_unit(x[j]);
    }
    bool inner = a.inner == kInnerAlways;
    if (a.inner == kInnerTest) inner = __all(ok[U - 1] & inner_span(x[0], x[U - 1], pgd, a.pad));
    // the class at the position after the group: loaded behind the taps, waited for after the shading
    int cnext = -1;
    float4 ub[U];
    if (a.macro.cls) cnext = macro_class(a.macro, pgid, sub(add(q, inc), ip));
    group_colours<FMT, OFF, U>(a, tf, inner, x, ok, pgd, page_base, pgid, ub);
    int n = 0;
    composite_group<0, U, THETA>([&](auto j) { return ub[decltype(j)::value]; }, ok, escalation_alpha(a, step_size, st.v.w),
                                 st, n);
    if (COUNT) count += (unsigned)n;
    // samples 0 .. n-2 advanced by the group's step, the last by its own
    const int last_ss = escalated_step(st.v.w, step_size);
    cls = n == U && last_ss == step_size ? cnext : -1;
    if (n == U) {
      o = q;
    } else {   // the last sample's position, by the same additions
      for (int j = 1; j < n; ++j) o = add(o, inc);
    }
    o = add(o, muls(muls(d, a.step), float(last_ss)));
    nsteps -= (n - 1) * step_size + last_ss;
    step_size = last_ss;
  }
  st.o = o;
  st.nsteps = nsteps;
  st.step_size = step_size;
}

// Calls f(std::integral_constant<int, j>) for j = 0 .. N-1, so that the body
// sees j as a constant (DPP controls must be).
template <int... I, class F>
__device__ __forceinline__ void static_for_impl(std::integer_sequence<int, I...>, F &&f) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <int N, class F> __device__ __forceinline__ void static_for(F &&f) {
  static_for_impl(std::make_integer_sequence<int, N>{}, f);
}

// Lane J of each group of G lanes, to every lane of the group.  Groups of 4
// are the hardware quads: one DPP quad_perm move (a VALU operation) instead
// of an LDS permute.
template <int G, int J> __device__ __forceinline__ float group_bcast(float v) {
  if constexpr (G == 4)
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), J * 0x55, 0xF, 0xF, false));
  else if constexpr (G == 16)   // row_newbcast
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x150 + J, 0xF, 0xF, false));
  else
    return __shfl(v, J, G);
}

// The reference march of one ray by G lanes that hold identical state
// (lane h of the ray's lane group): per group of G * UL consecutive samples
// of one brick, lane h resolves samples h, h + G, ... (taps, loads issued
// together, interpolation, shading: the colour does not depend on the ray's
// state) and every lane composites the group's colours in order, taken from
// their lanes, stopping where the step escalates.  Positions come from the
// same additions as the one-lane march and each value from the same taps, so
// the ray's samples, values and composite equal march_reference_grouped's bit
// for bit.  A lane's instruction stream per group holds UL samples' sampling
// and shading instead of G * UL, which is what a long ray's time is made of.
template <int FMT, bool COUNT, bool THETA, class OFF, int G, int UL = 1>
__device__ void march_reference_coop(const VolumeArgs &a, const float4 *tf, MarchState &st, int h,
                                     unsigned &count) {
  constexpr int N = G * UL;
  const float cdu = 1.f / comp_max(abs3(st.d));
  const f3 d = st.d;
  const f3 invr = recip3(d);
  f3 o = st.o;
  int nsteps = st.nsteps;
  int step_size = st.step_size;
  const OFF pad3 = (OFF)a.pad * (OFF)a.pad * (OFF)a.pad;
  int cpg = -1;
  float4 pgd = make_float4(0.f, 0.f, 0.f, 0.f);
  OFF page_base = 0;
  BrickLookup bl;
  int cls = -1;   // class of o's macrocell (-1: not looked up)
  while (nsteps > 0) {
    const f3 ip = floor3(o);
    if (bl.update(a, ip)) cls = -1;
    if (bl.cd) {
      // skip_nblock_steps (volume_shader.cu:5-14) with step * step_size
      const float sstep = a.step * float(step_size);
      float tn, tfar;
      intersect_box_inv(o, invr, ip, f3{ip.x + 1.f, ip.y + 1.f, ip.z + 1.f}, tn, tfar);
      const float di = ceilf((tfar + float(bl.cd - 1) * cdu) / sstep);
      o = add(o, muls(muls(d, di), sstep));
      nsteps -= (int)di;
      o = add(o, muls(muls(d, a.step), float(step_size)));
      nsteps -= step_size;
      continue;
    }
    const int pgid = bl.pg;
    if (pgid == -1) break;
    if (pgid != cpg) {
      pgd = a.page[pgid];
      page_base = (OFF)pgid * pad3;
      cpg = pgid;
    }
    const f3 inc = muls(muls(d, a.step), float(step_size));
    if (cls > 0) {   // samples in empty macrocells: their position updates alone
      const int k = skip_empty(a, cls, ip, invr, inc, step_size, o, nsteps);
      if (k > 0) {
        if (COUNT && h == 0) count += (unsigned)k;
        cls = macro_class(a.macro, pgid, sub(o, ip));
        continue;
      }
    }
    f3 p[N];
    bool ok[N];
    p[0] = o;
    ok[0] = true;
    int left = nsteps;
#pragma unroll
    for (int j = 1; j < N; ++j) {
      p[j] = add(p[j - 1], inc);
      left -= step_size;
      ok[j] = ok[j - 1] & (left > 0) & in_unit(sub(p[j], ip));
    }
    // this lane's samples h + G * k
    f3 x[UL];
    bool okh[UL];
#pragma unroll
    for (int k = 0; k < UL; ++k) {
      f3 ph = p[G * k];
      okh[k] = ok[G * k];
#pragma unroll
      for (int q = 1; q < G; ++q) {
        if (h == q) {
          ph = p[G * k + q];
          okh[k] = ok[G * k + q];
        }
      }
      x[k] = sub(ph, ip);
    }
    bool inner = a.inner == kInnerAlways;
    if (a.inner == kInnerTest) inner = __all(ok[N - 1] & inner_span(sub(o, ip), sub(p[N - 1], ip), pgd, a.pad));
    // a lane past the group's end repeats its ray's first sample
    x[0] = pick(okh[0], x[0], sub(o, ip));
    okh[0] = true;
    int cnext = -1;   // the class at the position after the group
    if (a.macro.cls) cnext = macro_class(a.macro, pgid, sub(add(p[N - 1], inc), ip));
    float4 ubh[UL];
    group_colours<FMT, OFF, UL>(a, tf, inner, x, okh, pgd, page_base, pgid, ubh);
    // composite in order, each sample's colour from its lane
    int n = 0;
    composite_group<0, N, THETA>(
        [&](auto jc) {
          constexpr int j = decltype(jc)::value;
          const float4 &uk = ubh[j / G];
          return make_float4(group_bcast<G, j % G>(uk.x), group_bcast<G, j % G>(uk.y), group_bcast<G, j % G>(uk.z),
                             group_bcast<G, j % G>(uk.w));
        },
        ok, escalation_alpha(a, step_size, st.v.w), st, n);
    if (COUNT && h == 0) count += (unsigned)n;
    const int last_ss = escalated_step(st.v.w, step_size);
    cls = n == N && last_ss == step_size ? cnext : -1;
    if (n == N) {
      o = p[N - 1];
    } else {   // the last sample's position, by the same additions
      for (int j = 1; j < n; ++j) o = add(o, inc);
    }
    o = add(o, muls(muls(d, a.step), float(last_ss)));
    nsteps -= (n - 1) * step_size + last_ss;
    step_size = last_ss;
  }
  st.o = o;
  st.nsteps = nsteps;
  st.step_size = step_size;
}

// Sample k of the lattice walk: position o0 + d * ((k + w/2) * step), w = min(1, L - k).
__device__ __forceinline__ f3 lattice_pos(f3 o0, f3 d, float lf, float step, int k, float &w) {
  w = gmin(1.f, lf - float(k));
  const float t = (float(k) + 0.5f * w) * step;
  return add(o0, muls(d, t));
}

// Lattice schedule: sample k covers w = min(1, L - k) steps (L the ray extent
// in steps, k < ceil(L)), sits at the covered segment's midpoint
// o0 + d * ((k + w/2) * step) and its opacity is scaled by w; empty regions are
// skipped to the next lattice point; early
// termination once v.w > ert.  G lanes hold one ray (as in
// march_reference_coop), lane h.  Film: o = o0, nsteps slot = bits of L (float),
// step_size = next lattice index.  Samples go in groups of U of one brick, as
// in the reference march (one at a time the march waited out each sample's
// loads); runs in empty macrocells move k alone.
template <int FMT, int G, int U, bool COUNT, bool THETA, class OFF>
__device__ void march_lattice(const VolumeArgs &a, const float4 *tf, MarchState &st, int h, unsigned &count) {
  constexpr int N = G * U;
  const f3 o0 = st.o, d = st.d;
  const f3 invr = recip3(d);
  const float lf = __int_as_float(st.nsteps);
  int k = st.step_size;
  const int kend = (int)ceilf(lf);
  const float cdu = 1.f / comp_max(abs3(d));
  // v.w > ert as v.w >= the next float; NaN, which no alpha reaches, without termination
  const float stop = a.ert > 0.f ? __uint_as_float(__float_as_uint(a.ert) + 1u) : NAN;
  const OFF pad3 = (OFF)a.pad * (OFF)a.pad * (OFF)a.pad;
  int cpg = -1;               // page of the cached descriptor
  float4 pgd = make_float4(0.f, 0.f, 0.f, 0.f);
  OFF page_base = 0;
  BrickLookup bl;
  int cls = -1;               // class of sample k's macrocell (-1: not looked up)
  while (k < kend) {
    float w0;
    const f3 o = lattice_pos(o0, d, lf, a.step, k, w0);
    const f3 ip = floor3(o);
    if (bl.update(a, ip)) cls = -1;
    if (bl.cd) {
      const float t = (float(k) + 0.5f * w0) * a.step;
      float tn, tfar;
      intersect_box_inv(o, invr, ip, f3{ip.x + 1.f, ip.y + 1.f, ip.z + 1.f}, tn, tfar);
      const float t_exit = t + tfar + float(bl.cd - 1) * cdu;
      const int kn = (int)ceilf(t_exit / a.step - 0.5f);
      k = kn > k + 1 ? kn : k + 1;
      continue;
    }
    const int pgid = bl.pg;
    if (pgid == -1) break;
    if (pgid != cpg) {
      pgd = a.page[pgid];
      page_base = (OFF)pgid * pad3;
      cpg = pgid;
    }
    if (cls > 0) {
      const int n = min(macro_run(a.macro, cls, sub(o, ip), invr, a.step), kend - k);
      if (n > 0) {
        k += n;
        if (COUNT && h == 0) count += (unsigned)n;
        float wk;
        cls = macro_class(a.macro, pgid, sub(lattice_pos(o0, d, lf, a.step, k, wk), ip));
        continue;
      }
    }
    // this lane's samples k + h + G u
    f3 x[U];
    float w[U];
    bool ok[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int kk = k + h + G * u;
      x[u] = sub(lattice_pos(o0, d, lf, a.step, kk, w[u]), ip);
      ok[u] = (kk < kend) & in_unit(x[u]);
      if (u == 0) ok[u] |= h == 0;
    }
    const bool mine = ok[0];
    bool inner = a.inner == kInnerAlways;
    if (a.inner == kInnerTest) inner = __all(ok[U - 1] & inner_span(sub(o, ip), x[U - 1], pgd, a.pad));
    if (G > 1) {   // a lane past the run repeats its ray's first sample
      x[0] = pick(mine, x[0], sub(o, ip));
      ok[0] = true;
    }
    int cnext = -1;           // the class at the sample after the group
    if (a.macro.cls) {
      float wk;
      cnext = macro_class(a.macro, pgid, sub(lattice_pos(o0, d, lf, a.step, k + N, wk), ip));
    }
    float4 ub[U];
    group_colours<FMT, OFF, U, true>(a, tf, inner, x, ok, pgd, page_base, pgid, ub, w);
    bool okn[N];
    static_for<N>([&](auto jc) {
      constexpr int j = decltype(jc)::value;
      const bool mine_j = j / G == 0 ? mine : ok[j / G];
      if constexpr (G > 1) okn[j] = group_bcast<G, j % G>(mine_j ? 1.f : 0.f) != 0.f;
      else okn[j] = mine_j;
    });
    int n = 0;
    composite_group<0, N, THETA>(
        [&](auto jc) {
          constexpr int j = decltype(jc)::value;
          const float4 &uk = ub[j / G];
          if constexpr (G > 1)
            return make_float4(group_bcast<G, j % G>(uk.x), group_bcast<G, j % G>(uk.y), group_bcast<G, j % G>(uk.z),
                               group_bcast<G, j % G>(uk.w));
          else
            return uk;
        },
        okn, stop, st, n);
    if (COUNT && h == 0) count += (unsigned)n;
    cls = n == N ? cnext : -1;
    k += n;
    if (st.v.w >= stop) k = kend;
  }
  st.step_size = k;
}

// ray_emit_shader_impl (shader.hpp:113-137) + VolumeShaderKernel::init.
__device__ __forceinline__ bool emit(const VolumeArgs &a, int x, int y, MarchState &st) {
  st.d = pixel_ray_dir(a.trans, a.ctg, a.ray_o, x, y, a.W, a.H);
  st.o = a.ray_o;
  st.v = make_float4(0.f, 0.f, 0.f, 0.f);
  st.theta = f3{0.f, 0.f, 0.f};
  st.phi = 1.f;
  float tnear, tfar;
  if (intersect_box(st.o, st.d, a.bmin, a.bmax, tnear, tfar)) {
    if (tnear < 0) tnear = 0;
    if (tfar < 0) tfar = 0;
    st.o = add(st.o, muls(st.d, tnear));
    if (a.schedule == HYD_SCHED_LATTICE) {
      st.nsteps = __float_as_int(gmin((tfar - tnear) / a.step, float(a.max_steps)));
      st.step_size = 0;
    } else {
      const int n = (int)((tfar - tnear) / a.step);
      st.nsteps = a.max_steps < n ? a.max_steps : n;
      st.step_size = 1;
    }
    return true;
  }
  st.nsteps = 0;   // also the bits of 0.f for the lattice schedule
  st.step_size = a.schedule == HYD_SCHED_LATTICE ? 0 : 1;
  return false;
}

__device__ __forceinline__ void store_pixel(const VolumeArgs &a, size_t idx, const MarchState &st) {
  if (a.film) {
    float4 *f = reinterpret_cast<float4 *>(a.film + idx);
    f[0] = make_float4(st.o.x, st.o.y, st.o.z, st.d.x);
    f[1] = make_float4(st.d.y, st.d.z, __int_as_float(st.nsteps), __int_as_float(st.step_size));
    f[2] = st.v;
    f[3] = make_float4(st.theta.x, st.theta.y, st.theta.z, st.phi);
  }
  if (a.rgba) a.rgba[idx] = st.v;
}

__device__ __forceinline__ void load_pixel(const VolumeArgs &a, size_t idx, MarchState &st) {
  const float4 *f = reinterpret_cast<const float4 *>(a.film + idx);
  float4 f0 = f[0], f1 = f[1];
  st.o = f3{f0.x, f0.y, f0.z};
  st.d = f3{f0.w, f1.x, f1.y};
  st.nsteps = __float_as_int(f1.z);
  st.step_size = __float_as_int(f1.w);
  st.v = f[2];
  float4 f3v = f[3];
  st.theta = f3{f3v.x, f3v.y, f3v.z};
  st.phi = f3v.w;
}

// Samples whose tap loads a one-lane reference-schedule or lattice group issues
// together, per brick format: 4 keeps the marches within 128 registers (8 for u8: 145;
// 640^2 and 1024^2 frames of a 500^3 volume 713 and 1274 us with 8, 800 and 1181
// with 4).
#ifndef HYD_REF_GROUP_U8
#define HYD_REF_GROUP_U8 4
#endif
#ifndef HYD_REF_GROUP_F16
#define HYD_REF_GROUP_F16 4
#endif
#ifndef HYD_REF_GROUP_F32
#define HYD_REF_GROUP_F32 4
#endif
template <int FMT> constexpr int ref_group() {
  return FMT == HYD_FMT_U8 ? HYD_REF_GROUP_U8 : FMT == HYD_FMT_F16 ? HYD_REF_GROUP_F16 : HYD_REF_GROUP_F32;
}

// Lanes per ray of a frame.  A ray is one dependent chain of groups; a SIMD
// with one wave on it issues that chain no faster than one with four.  Several
// lanes shorten it (each resolves a share of a group's samples; all composite
// them in order), at the price of repeating the positions and the compositing
// on every lane.  So: 16 lanes while the launch stays around six waves per SIMD
// (a group's colours then come by DPP row broadcasts), 4 while the chains of
// the longest rays and not the sum of the work set the time, then one.  The
// work is counted in rays of the longest chord (full_rays), and the line moves
// with the pool's size: chains wait longer for taps the caches do not hold.
// Frames in us, 1 / 4 / 16 lanes (reference schedule unless noted; full_rays
// about 0.42 of the pixels of these square views, all of the 356 x 882 ones):
//                             48 x 40       160^2         200^2        512^2     640^2       800^2
//   256^3 FP32 brick       440/205/142   431/201/171   -/200/210   412/398   476/575     599/842
//   400^3 FP32 fBm bricks  495/213/163   523/280/265   -/320/337   991/852   1206/1103   1399/1434
//   500^3 FP16 bricks      628/343/238   733/356/280   -/373/318   943/716   1118/902    1187/1230
//   400^3 u8 fBm bricks    425/212/162   431/250/237   -/263/317   654/641   745/907     940/1309
//   500^3 FP16, lattice    689/281/177   697/299/221   -/310/318   915/726   1180/957    1360/1358
//   356 x 882: 35^3 FP16 79/128, 64^3 FP16 128/182, 120^3 FP32 226/327; 60^3 u8 at 500^2 101/132
constexpr int kLanes = 4, kManyLanes = 16;
template <int L> constexpr int coop_group() { return L == kManyLanes ? 16 : 8; }   // samples a group
// A wave's tile of rays.
template <int L> constexpr int tile_w() { return L == kManyLanes ? 4 : kTile; }
template <int L> constexpr int tile_h() { return 64 / L / tile_w<L>(); }
constexpr long long kManyLaneRays = 24576;
// A tall frame's workgroups of L lanes a ray fit a launch's y axis (16 lanes always
// do, at kManyLaneRays).
template <int L> bool rows_fit(int H) { return (H + tile_h<L>() - 1) / tile_h<L>() <= 65535; }

// Render modes of volume_kernel: emit into an RGBA image only, emit into a film
// (and optionally RGBA), or resume a film.
enum { kEmitRgba = 0, kEmitFilm = 1, kResume = 2 };

template <int FMT, bool COUNT, int MODE, bool BIG, int LANES>
__global__ __launch_bounds__(64) void volume_kernel(VolumeArgs a) {
  constexpr bool RESUME = MODE == kResume;
  constexpr bool THETA = MODE != kEmitRgba;
  __shared__ float4 s_tf[kTfLds];
  __shared__ unsigned long long s_count;
  stage_tf(s_tf, a.tf, a.tf_n);
  if (COUNT && threadIdx.x == 0) s_count = 0;
  __syncthreads();
  if (!macro_pays(a.macro)) a.macro.cls = nullptr;

  using OFF = std::conditional_t<BIG, uint64_t, uint32_t>;
  const int ray = (int)threadIdx.x / LANES, h = (int)threadIdx.x % LANES;
  const int tx = rotated_tile_x();
  const int x = tx * tile_w<LANES>() + (ray % tile_w<LANES>());
  const int y = blockIdx.y * tile_h<LANES>() + (ray / tile_w<LANES>());
  unsigned count = 0;
  bool handed = false;   // this lane's ray went to the cooperative march
  MarchState st;
  size_t idx = 0;
  if (x < a.W && y < a.H) {
    idx = (size_t)y * a.W + x;
    bool live;
    if (RESUME) {
      load_pixel(a, idx, st);
      live = st.nsteps > 0;
    } else {
      live = emit(a, x, y, st);
    }
    if (live) {
      if constexpr (LANES > 1)
        march_reference_coop<FMT, COUNT, THETA, OFF, LANES, coop_group<LANES>() / LANES>(a, s_tf, st, h, count);
      else
        march_reference_grouped<FMT, ref_group<FMT>(), COUNT, THETA, OFF>(a, s_tf, st, count, handed);
    }
    if (!handed && h == 0) store_pixel(a, idx, st);
  }
  // the rays handed over: kCoopLanes lanes each, with the state copied through LDS
  const unsigned long long hm = __ballot(handed);
  if (hm) {
    __shared__ MarchState s_st[kCoopRays];
    __shared__ size_t s_idx[kCoopRays];
    const int lane = (int)threadIdx.x;
    // at most kCoopRays lanes hand over: they all leave the march together, in
    // the iteration where the wave's marching lanes first number kCoopRays or fewer
    if (handed) {
      const int slot = __popcll(hm & ((1ull << lane) - 1ull));
      if (slot < kCoopRays) {
        s_st[slot] = st;
        s_idx[slot] = idx;
      }
    }
    __syncthreads();
    const int r = lane / kCoopLanes, h = lane % kCoopLanes;
    if (r < __popcll(hm)) {
      MarchState c = s_st[r];
      march_reference_coop<FMT, COUNT, THETA, OFF, kCoopLanes>(a, s_tf, c, h, count);
      if (h == 0) store_pixel(a, s_idx[r], c);
    }
  }
  if (COUNT) {
    if (count) atomicAdd(&s_count, (unsigned long long)count);
    __syncthreads();
    if (threadIdx.x == 0 && s_count) atomicAdd(a.samples, s_count);
  }
}

// Lattice-schedule frame, LANES lanes per ray (a kernel of its own: in
// volume_kernel it cost the reference march 11 registers).
template <int FMT, bool COUNT, int MODE, bool BIG, int LANES>
__global__ __launch_bounds__(64) void lattice_kernel(VolumeArgs a) {
  __shared__ float4 s_tf[kTfLds];
  __shared__ unsigned long long s_count;
  stage_tf(s_tf, a.tf, a.tf_n);
  if (COUNT && threadIdx.x == 0) s_count = 0;
  __syncthreads();
  if (!macro_pays(a.macro)) a.macro.cls = nullptr;
  const int ray = (int)threadIdx.x / LANES, h = (int)threadIdx.x % LANES;
  const int x = rotated_tile_x() * tile_w<LANES>() + (ray % tile_w<LANES>());
  const int y = blockIdx.y * tile_h<LANES>() + (ray / tile_w<LANES>());
  unsigned count = 0;
  if (x < a.W && y < a.H) {
    const size_t idx = (size_t)y * a.W + x;
    MarchState st;
    bool live;
    if (MODE == kResume) {
      load_pixel(a, idx, st);
      live = st.nsteps > 0;
    } else {
      live = emit(a, x, y, st);
    }
    constexpr int U = LANES > 1 ? coop_group<LANES>() / LANES : ref_group<FMT>();
    if (live)
      march_lattice<FMT, LANES, U, COUNT, MODE != kEmitRgba, std::conditional_t<BIG, uint64_t, uint32_t>>(a, s_tf, st,
                                                                                                         h, count);
    if (h == 0) store_pixel(a, idx, st);
  }
  if (COUNT) {
    if (count) atomicAdd(&s_count, (unsigned long long)count);
    __syncthreads();
    if (threadIdx.x == 0 && s_count) atomicAdd(a.samples, s_count);
  }
}

template <int FMT>
__global__ __launch_bounds__(64) void volume_trace_kernel(VolumeArgs a, int x, int y, hyd_trace_rec *out,
                                                          int max_recs, int *n_out) {
  __shared__ float4 s_tf[kTfLds];
  stage_tf(s_tf, a.tf, a.tf_n);
  __syncthreads();
  if (threadIdx.x != 0) return;
  MarchState st;
  unsigned count = 0;
  int nt = 0;
  if (emit(a, x, y, st)) march_reference<FMT, false, true>(a, s_tf, st, count, out, max_recs, nt);
  *n_out = nt;
}

// ---------------------------------------------------------------------------
// Sort-last segments.  The lattice walk of a ray visits cells in order (every
// coordinate of o0 + d*t is monotone in t, so a cell is never revisited); the
// k-th visited cell owns slot k of the ray.  A pass composites, front to back
// from zero, the samples of every visited cell whose brick is resident in the
// current page table into its slot (each sample reads the brick of its own
// floor(p), exactly as the single march does); empty cells write a transparent
// slot; cells not resident now are left for a later pass.  The final fold
// composites the slots in order and stops at the first slot no pass filled
// (the reference stops a ray at its first non-resident brick).
//
// A cell's samples are a run of lattice indices [k, kend_cell) (positions are
// monotone in t, so a cell is entered once); the run's end is estimated from
// the cell's exit distance and then moved until it agrees with floor() of the
// sample positions, evaluated exactly as the walk evaluates them, so every
// pass sees the same cells and samples as the single march.  A cell not
// resident in this pass is passed over in one step; a resident one composites
// its run with the tap loads of up to U samples in flight together (every
// sample loads its taps: skipping a repeated cell's loads cost more in
// branches and register copies, 4.60 against 4.51 ms for the 3-batch set).
#ifndef HYD_SEG_GROUP
#define HYD_SEG_GROUP 4
#endif

__device__ __forceinline__ bool same_cell(f3 p, f3 ip) {
  const f3 q = floor3(p);
  return q.x == ip.x && q.y == ip.y && q.z == ip.z;
}

// The walk's step at lattice index k.  An empty cell writes a transparent
// slot and a cell not resident in this pass leaves its slot; both advance k
// and the slot index and return false.  A resident cell returns true with
// its run [k, kc), its cell ip and its page id, k and ord unchanged.
__device__ __forceinline__ bool seg_walk_cell(const VolumeArgs &a, f3 o0, f3 d, f3 invr, float lf, int kend,
                                              float cdu, size_t P, size_t ray, bool writes, int &k, int &ord, f3 &ip, int &kc,
                                              int &pgid) {
  float w;
  const f3 o = lattice_pos(o0, d, lf, a.step, k, w);
  const float t = (float(k) + 0.5f * w) * a.step;
  ip = floor3(o);
  const int code = cell_code(a, ip);
  const int cd = code <= -2 ? -1 - code : 0;
  float tn, tfar;
  intersect_box_inv(o, invr, ip, f3{ip.x + 1.f, ip.y + 1.f, ip.z + 1.f}, tn, tfar);
  if (cd) {   // empty cell: same skip as the single lattice march
    const float t_exit = t + tfar + float(cd - 1) * cdu;
    const int kn = (int)ceilf(t_exit / a.step - 0.5f);
    k = kn > k + 1 ? kn : k + 1;
    if (writes) a.slots[(size_t)ord * P + ray] = make_float4(0.f, 0.f, 0.f, 0.f);
    ++ord;
    return false;
  }
  // the cell's run [k, kc): estimate from the exit distance, then agree with floor()
  kc = (int)ceilf((t + tfar) / a.step - 0.5f);
  kc = kc > k + 1 ? kc : k + 1;
  kc = kc < kend ? kc : kend;
  float wq;
  while (kc < kend && same_cell(lattice_pos(o0, d, lf, a.step, kc, wq), ip)) ++kc;
  while (kc - 1 > k && !same_cell(lattice_pos(o0, d, lf, a.step, kc - 1, wq), ip)) --kc;
  pgid = code;
  if (pgid < 0) {   // not resident in this pass: the slot is left for another
    ++ord;
    k = kc;
    return false;
  }
  return true;
}

// Samples [kk, min(kk + G U, kc)) of a run in cell ip of page pgid, their tap
// loads in flight together, composited in order into seg.  The G lanes of a
// ray resolve samples kk + h + G u each and composite all of them.
template <int FMT, bool COUNT, int G, int U, typename OFF>
__device__ __forceinline__ void seg_sample_group(const VolumeArgs &a, const float4 *s_tf, f3 o0, f3 d, float lf, f3 ip,
                                                 float4 pgd, OFF page_base, int pgid, int kk, int kc, int h,
                                                 MarchState &seg, unsigned &count) {
  f3 x[U];
  bool ok[U], okn[G * U];
  float w[U];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    // a slot past the run repeats its last sample, so that x[0] .. x[U - 1] spans
    // every sample read
    const int k = kk + h + G * u;
    x[u] = sub(lattice_pos(o0, d, lf, a.step, k < kc ? k : kc - 1, w[u]), ip);
    ok[u] = k < kc || (G > 1 && u == 0);
  }
#pragma unroll
  for (int j = 0; j < G * U; ++j) okn[j] = kk + j < kc;
  bool inner = a.inner == kInnerAlways;
  if (a.inner == kInnerTest) inner = __all(inner_span(x[0], x[U - 1], pgd, a.pad));
  float4 ub[U];
  group_colours<FMT, OFF, U, true>(a, s_tf, inner, x, ok, pgd, page_base, pgid, ub, w);
  int n = 0;
  composite_group<0, G * U, false>(
      [&](auto jc) {
        constexpr int j = decltype(jc)::value;
        const float4 &uk = ub[j / G];
        if constexpr (G > 1)
          return make_float4(group_bcast<G, j % G>(uk.x), group_bcast<G, j % G>(uk.y), group_bcast<G, j % G>(uk.z),
                             group_bcast<G, j % G>(uk.w));
        else
          return uk;
      },
      okn, NAN, seg, n);   // no alpha stops a segment
  if (COUNT && h == 0) count += (unsigned)n;
}

// MULTI: a segment set, whose cells name the pages of every batch: the ray is
// walked once for all batches.  (With one layer of workgroups per batch, each
// walked every ray's cells and found a third of them resident: 4.10 against
// 2.81 ms for three batches of a 1024^3 u8 volume at 512^2.)
// The 64-bit offsets of a set whose pools lie far apart are held to three waves per
// SIMD (one register too many leaves two: 1024^2 FP16 frame of two pools 10 GB apart
// 3.89 ms, 2.98 with three, and 3.12 with 32-bit offsets).
template <int FMT, bool COUNT, bool BIG, bool MULTI, int LANES>
__global__ __launch_bounds__(64, BIG && MULTI && LANES == 1 ? 3 : 1) void segment_kernel(VolumeArgs a) {
  using OFF = std::conditional_t<BIG, uint64_t, uint32_t>;
  constexpr int U = LANES > 1 ? coop_group<LANES>() / LANES : HYD_SEG_GROUP;
  __shared__ float4 s_tf[kTfLds];
  __shared__ unsigned long long s_count;
  stage_tf(s_tf, a.tf, a.tf_n);
  if (COUNT && threadIdx.x == 0) s_count = 0;
  __syncthreads();
  const int r = (int)threadIdx.x / LANES, h = (int)threadIdx.x % LANES;
  const int x = rotated_tile_x() * tile_w<LANES>() + (r % tile_w<LANES>());
  const int y = blockIdx.y * tile_h<LANES>() + (r / tile_w<LANES>());
  unsigned count = 0;
  if (x < a.W && y < a.H) {
    const size_t P = (size_t)a.W * a.H, ray = (size_t)y * a.W + x;
    MarchState st;
    int ord = 0;
    if (emit(a, x, y, st)) {
      const f3 o0 = st.o, d = st.d;
      const float lf = __int_as_float(st.nsteps);
      const int kend = (int)ceilf(lf);
      const float cdu = 1.f / comp_max(abs3(d));
      const f3 invr = recip3(d);
      const OFF pad3 = (OFF)a.pad * (OFF)a.pad * (OFF)a.pad;
      int k = 0, kc = 0, pgid = -1;
      f3 ip{0.f, 0.f, 0.f};
      MarchState seg;
      if constexpr (MULTI || LANES > 1) {
        // the wave walks its rays' cells in lock-step (the lanes in resident
        // cells composite their runs while the others wait): its rays stay in
        // the same bricks, whose lines they share, and it issues the fewest
        // instructions
        while (k < kend && ord < a.max_slots) {
          if (!seg_walk_cell(a, o0, d, invr, lf, kend, cdu, P, ray, h == 0, k, ord, ip, kc, pgid)) continue;
          const float4 pgd = a.page[pgid];
          const OFF page_base = MULTI ? (OFF)a.page_base[pgid] : (OFF)pgid * pad3;
          const int id = MULTI && a.mode == HYD_MODE_PAGING ? a.page_local[pgid] : pgid;
          seg.v = make_float4(0.f, 0.f, 0.f, 0.f);
          for (int kk = k; kk < kc; kk += LANES * U)
            seg_sample_group<FMT, COUNT, LANES, U, OFF>(a, s_tf, o0, d, lf, ip, pgd, page_base, id, kk, kc, h, seg,
                                                        count);
          if (h == 0) a.slots[(size_t)ord * P + ray] = seg.v;
          ++ord;
          k = kc;
        }
      } else {
        // one batch of a large frame: lanes idle in lock-step cost time where
        // most cells are not resident, so each lane composites U samples of
        // its own run per iteration; lanes whose run ended wait until a
        // quarter of the wave's busy lanes (or all of them) need to walk, then
        // walk together to their next resident run (7.47 -> 6.84 ms for three
        // one-batch passes of the 1024^3 frame; 4.21 -> 6.53 ms in a set,
        // whose rays then leave each other's bricks)
        bool in_run = false;
        int kk = 0;
        float4 pgd = make_float4(0.f, 0.f, 0.f, 0.f);
        OFF page_base = 0;
        while (true) {
          const bool want = !in_run && k < kend && ord < a.max_slots;
          const uint64_t m_want = __ballot(want), m_run = __ballot(in_run);
          if ((m_want | m_run) == 0) break;
          const bool walk_now = m_run == 0 || 4 * __popcll(m_want) >= __popcll(m_want | m_run);
          if (want && walk_now) {
            while (k < kend && ord < a.max_slots) {
              if (!seg_walk_cell(a, o0, d, invr, lf, kend, cdu, P, ray, true, k, ord, ip, kc, pgid)) continue;
              pgd = a.page[pgid];
              page_base = (OFF)pgid * pad3;
              seg.v = make_float4(0.f, 0.f, 0.f, 0.f);
              kk = k;
              in_run = true;
              break;
            }
          }
          if (!in_run) continue;
          seg_sample_group<FMT, COUNT, 1, U, OFF>(a, s_tf, o0, d, lf, ip, pgd, page_base, pgid, kk, kc, 0, seg,
                                                  count);
          kk += U;
          if (kk >= kc) {   // the run is complete: its slot, then the next cell
            a.slots[(size_t)ord * P + ray] = seg.v;
            ++ord;
            k = kc;
            in_run = false;
          }
        }
      }
    }
    if (h == 0) a.nslots[ray] = ord;
  }
  if (COUNT) {
    if (count) atomicAdd(&s_count, (unsigned long long)count);
    __syncthreads();
    if (threadIdx.x == 0 && s_count) atomicAdd(a.samples, s_count);
  }
}

__global__ __launch_bounds__(256) void segment_clear_kernel(float4 *slots, size_t n) {
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (i < n) slots[i] = make_float4(0.f, 0.f, 0.f, -1.f);   // alpha -1: not filled yet
}

__global__ __launch_bounds__(256) void segment_fold_kernel(const float4 *slots, const int32_t *nslots,
                                                           int max_slots, int P, float4 *rgba) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= P) return;
  float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
  const int n = min(nslots[i], max_slots);
  for (int ord = 0; ord < n; ++ord) {
    const float4 s = slots[(size_t)ord * P + i];
    if (s.w < 0.f) break;
    const float t = 1.f - v.w;
    v = make_float4(v.x + s.x * t, v.y + s.y * t, v.z + s.z * t, v.w + s.w * t);
  }
  rgba[i] = v;
}

template <int FMT, int MODE, bool BIG, int L>
void launch_lanes(const VolumeArgs &a, hipStream_t s) {
  constexpr int w = tile_w<L>(), h = tile_h<L>();
  const dim3 block(64), grid((a.W + w - 1) / w, (a.H + h - 1) / h);
  if (a.schedule == HYD_SCHED_LATTICE) {
    if (a.samples) hipLaunchKernelGGL((lattice_kernel<FMT, true, MODE, BIG, L>), grid, block, 0, s, a);
    else hipLaunchKernelGGL((lattice_kernel<FMT, false, MODE, BIG, L>), grid, block, 0, s, a);
  } else {
    if (a.samples) hipLaunchKernelGGL((volume_kernel<FMT, true, MODE, BIG, L>), grid, block, 0, s, a);
    else hipLaunchKernelGGL((volume_kernel<FMT, false, MODE, BIG, L>), grid, block, 0, s, a);
  }
}

template <int FMT, int MODE, bool BIG>
void launch_mode(const VolumeArgs &a, hipStream_t s) {
  if (a.lanes == kManyLanes) launch_lanes<FMT, MODE, BIG, kManyLanes>(a, s);
  else if (a.lanes == kLanes) launch_lanes<FMT, MODE, BIG, kLanes>(a, s);
  else launch_lanes<FMT, MODE, BIG, 1>(a, s);
}

template <int FMT, bool BIG>
void launch_fmt_off(const VolumeArgs &a, bool resume, hipStream_t s) {
  if (resume) launch_mode<FMT, kResume, BIG>(a, s);
  else if (a.film) launch_mode<FMT, kEmitFilm, BIG>(a, s);
  else launch_mode<FMT, kEmitRgba, BIG>(a, s);
}

// HYD_VOLUME_OFFSETS64=1 selects the 64-bit offsets for any pool (they render the
// same image; the switch lets a small pool exercise that variant).
bool force_offsets64() {
  static const bool on = [] {
    const char *e = std::getenv("HYD_VOLUME_OFFSETS64");
    return e && e[0] == '1';
  }();
  return on;
}

template <int FMT, bool MULTI, int L>
void launch_segments_lanes(const VolumeArgs &a, bool big, hipStream_t s) {
  constexpr int w = tile_w<L>(), h = tile_h<L>();
  const dim3 grid((a.W + w - 1) / w, (a.H + h - 1) / h), block(64);
  if (a.samples) {
    if (big) hipLaunchKernelGGL((segment_kernel<FMT, true, true, MULTI, L>), grid, block, 0, s, a);
    else hipLaunchKernelGGL((segment_kernel<FMT, true, false, MULTI, L>), grid, block, 0, s, a);
  } else {
    if (big) hipLaunchKernelGGL((segment_kernel<FMT, false, true, MULTI, L>), grid, block, 0, s, a);
    else hipLaunchKernelGGL((segment_kernel<FMT, false, false, MULTI, L>), grid, block, 0, s, a);
  }
}

// Lanes per ray as for frames, from the bytes the launch reads, but 4 lanes up
// to twice the work: in lock-step a run of 4-lane groups wastes less of its
// wave (512^2 frame of a 1024^3 u8 set: 4.21 ms with one lane, 2.81 with four;
// eight drawn sets 1.17 and 2.19 times as fast as one layer of workgroups per batch).
template <int FMT, bool MULTI>
hipError_t launch_segments(const VolumeArgs &a, uint64_t span, uint64_t bytes, hipStream_t s) {
  const bool big = span > (1ull << 32) || force_offsets64();
  if ((long long)a.W * a.H <= kManyLaneRays) launch_segments_lanes<FMT, MULTI, kManyLanes>(a, big, s);
  else if (rows_fit<kLanes>(a.H) && a.full_rays <= 2.f * lane_rays((double)bytes)) launch_segments_lanes<FMT, MULTI, kLanes>(a, big, s);
  else launch_segments_lanes<FMT, MULTI, 1>(a, big, s);
  return hipGetLastError();
}

template <int FMT>
hipError_t launch_fmt(const VolumeArgs &a, bool resume, hipStream_t s) {
  // 32-bit byte offsets while every byte of the pool is below 4 GiB
  const uint64_t bytes = a.pool_elems * (uint64_t)sizeof(typename RawVox<FMT>::T);
  // the x-pair loads need two voxels per row (hyd_upload_pool refuses smaller bricks)
  if (bytes <= (1ull << 32) && !force_offsets64()) launch_fmt_off<FMT, false>(a, resume, s);
  else launch_fmt_off<FMT, true>(a, resume, s);
  return hipGetLastError();
}

}  // namespace

int32_t frame_lanes(int W, int H, float full_rays, double pool_bytes) {
  if ((long long)W * H <= kManyLaneRays) return kManyLanes;
  return rows_fit<kLanes>(H) && full_rays <= lane_rays(pool_bytes) ? kLanes : 1;
}

hipError_t launch_volume(const VolumeArgs &a, int fmt, bool resume, hipStream_t s) {
  switch (fmt) {
    case HYD_FMT_U8: return launch_fmt<HYD_FMT_U8>(a, resume, s);
    case HYD_FMT_F16: return launch_fmt<HYD_FMT_F16>(a, resume, s);
    default: return launch_fmt<HYD_FMT_F32>(a, resume, s);
  }
}

hipError_t launch_segments_clear(float4 *slots, size_t n, hipStream_t s) {
  hipLaunchKernelGGL(segment_clear_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, slots, n);
  return hipGetLastError();
}

hipError_t launch_segments_pass(const VolumeArgs &a, int fmt, hipStream_t s) {
  switch (fmt) {
    case HYD_FMT_U8: return launch_segments<HYD_FMT_U8, false>(a, a.pool_elems, a.pool_elems, s);
    case HYD_FMT_F16: return launch_segments<HYD_FMT_F16, false>(a, a.pool_elems * 2, a.pool_elems * 2, s);
    default: return launch_segments<HYD_FMT_F32, false>(a, a.pool_elems * 4, a.pool_elems * 4, s);
  }
}

hipError_t launch_segments_set(const VolumeArgs &a, uint64_t span_bytes, uint64_t pool_bytes, int fmt, hipStream_t s) {
  switch (fmt) {
    case HYD_FMT_U8: return launch_segments<HYD_FMT_U8, true>(a, span_bytes, pool_bytes, s);
    case HYD_FMT_F16: return launch_segments<HYD_FMT_F16, true>(a, span_bytes, pool_bytes, s);
    default: return launch_segments<HYD_FMT_F32, true>(a, span_bytes, pool_bytes, s);
  }
}

hipError_t launch_segments_composite(const float4 *slots, const int32_t *nslots, int max_slots, int P, float4 *rgba,
                                     hipStream_t s) {
  hipLaunchKernelGGL(segment_fold_kernel, dim3((P + 255) / 256), dim3(256), 0, s, slots, nslots, max_slots, P, rgba);
  return hipGetLastError();
}

hipError_t launch_volume_trace(const VolumeArgs &a, int fmt, int x, int y, hyd_trace_rec *out_dev, int max_recs,
                               int *n_dev, hipStream_t s) {
  switch (fmt) {
    case HYD_FMT_U8:
      hipLaunchKernelGGL(volume_trace_kernel<HYD_FMT_U8>, dim3(1), dim3(64), 0, s, a, x, y, out_dev, max_recs, n_dev);
      break;
    case HYD_FMT_F16:
      hipLaunchKernelGGL(volume_trace_kernel<HYD_FMT_F16>, dim3(1), dim3(64), 0, s, a, x, y, out_dev, max_recs, n_dev);
      break;
    default:
      hipLaunchKernelGGL(volume_trace_kernel<HYD_FMT_F32>, dim3(1), dim3(64), 0, s, a, x, y, out_dev, max_recs, n_dev);
  }
  return hipGetLastError();
}

}  // namespace hyd
