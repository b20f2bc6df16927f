// Blocks.Volume / Blocks.Solid and Isosurface kernels for gfx950.
// One lane per pixel, 8x8 pixel packets per 64-lane workgroup.
#include <hip/hip_fp16.h>

#include "hyd_internal.hpp"
#include "hyd_macro.hpp"
#include "hyd_sampler.hpp"

#include <cstdlib>
#include <type_traits>

namespace hyd {
namespace {

constexpr int kTile = 8;

__device__ __forceinline__ int grid_index(f3 p, const int32_t dim[3]) {
  float fx = gclamp(p.x, 0.f, float(dim[0]));
  float fy = gclamp(p.y, 0.f, float(dim[1]));
  float fz = gclamp(p.z, 0.f, float(dim[2]));
  int ix = iclamp((int)floorf(fx), 0, dim[0] - 1);
  int iy = iclamp((int)floorf(fy), 0, dim[1] - 1);
  int iz = iclamp((int)floorf(fz), 0, dim[2] - 1);
  return iz * dim[0] * dim[1] + iy * dim[0] + ix;
}

// skip_nblock_steps (blocks_shader.cu:5-14, isosurface_shader.cu:5-14).
__device__ __forceinline__ int skip_nblock_steps(f3 &o, f3 d, f3 ip, int nblocks, float cdu, float step) {
  float tn, tfar;
  intersect_box(o, d, ip, f3{ip.x + 1.f, ip.y + 1.f, ip.z + 1.f}, tn, tfar);
  const float di = ceilf((tfar + float(nblocks - 1) * cdu) / step);
  o = add(o, muls(muls(d, di), step));
  return (int)di;
}

// skip_nblock_steps with the ray's reciprocal direction computed once (same result).
__device__ __forceinline__ int skip_nblock_steps_inv(f3 &o, f3 invr, f3 d, f3 ip, int nblocks, float cdu,
                                                     float step) {
  float tn, tfar;
  intersect_box_inv(o, invr, ip, f3{ip.x + 1.f, ip.y + 1.f, ip.z + 1.f}, tn, tfar);
  const float di = ceilf((tfar + float(nblocks - 1) * cdu) / step);
  o = add(o, muls(muls(d, di), step));
  return (int)di;
}

// VisBlocksShaderKernel::main, blocks_shader.cu:16-50; HYD_BLOCKS_PAGING is the
// Paging renderer's residency view, PagingShaderKernel::main (paging_shader.cu:24-61).
__global__ __launch_bounds__(64) void blocks_kernel(BlocksArgs a) {
  const int x = blockIdx.x * kTile + (threadIdx.x % kTile);
  const int y = blockIdx.y * kTile + (threadIdx.x / kTile);
  if (x >= a.W || y >= a.H) return;
  const f3 d = pixel_ray_dir(a.trans, a.ctg, a.ray_o, x, y, a.W, a.H);
  f3 o = a.ray_o;
  float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
  float tnear, tfar;
  if (intersect_box(o, d, a.bmin, a.bmax, tnear, tfar)) {
    if (tnear < 0) tnear = 0;
    if (tfar < 0) tfar = 0;
    o = add(o, muls(d, tnear));
    const int n = (int)((tfar - tnear) / a.step);
    int nsteps = a.max_steps < n ? a.max_steps : n;
    const float cdu = 1.f / comp_max(abs3(d));
    const float opacity_threshold = 0.95f;
    const f3 hi = f3{a.bmax.x - 1.f, a.bmax.y - 1.f, a.bmax.z - 1.f};
    const f3 ext = sub(a.bmax, a.bmin);
    while (nsteps > 0) {
      const f3 ip = floor3(o);
      const int gi = grid_index(ip, a.dim);
      const int cd = a.cheb[gi];
      if (cd) {
        nsteps -= skip_nblock_steps(o, d, ip, cd, cdu, a.step);
      } else if (a.mode == HYD_BLOCKS_PAGING) {
        // PagingShaderKernel::main (paging_shader.cu:34-59): one composite per
        // resident brick, green for a level-0 page, red for a lower-level one
        const int pgid = a.vaddr[grid_index(ip, a.vdim)];
        if (pgid == -1) break;   // page fault
        const float4 col = pgid >= a.lowest ? make_float4(0.f, .5f, 0.f, .5f) : make_float4(.2f, 0.f, 0.f, .2f);
        nsteps -= skip_nblock_steps(o, d, ip, 1, cdu, a.step);
        const float t = 1.f - v.w;
        v = make_float4(v.x + col.x * t, v.y + col.y * t, v.z + col.z * t, v.w + col.w * t);
        if (v.w > opacity_threshold) break;
      } else {
        const f3 c = {gclamp(ip.x, a.bmin.x, hi.x), gclamp(ip.y, a.bmin.y, hi.y), gclamp(ip.z, a.bmin.z, hi.z)};
        const f3 rip = {c.x / ext.x, c.y / ext.y, c.z / ext.z};
        if (a.mode == HYD_BLOCKS_VOLUME) {
          const float mean = a.mean[gi];
          const float4 col = make_float4(rip.x * a.density * mean, rip.y * a.density * mean,
                                         rip.z * a.density * mean, 1.f * a.density * mean);
          const float t = 1.f - v.w;
          v = make_float4(v.x + col.x * t, v.y + col.y * t, v.z + col.z * t, v.w + col.w * t);
          if (v.w > opacity_threshold) break;
        } else {
          v = make_float4(rip.x, rip.y, rip.z, 1.f);
          break;
        }
      }
      o = add(o, muls(d, a.step));
      nsteps -= 1;
    }
  }
  a.rgba[(size_t)y * a.W + x] = v;
}

template <int FMT> __device__ __forceinline__ float vox(const void *pool, size_t i);
template <> __device__ __forceinline__ float vox<HYD_FMT_F32>(const void *pool, size_t i) {
  return static_cast<const float *>(pool)[i];
}
template <> __device__ __forceinline__ float vox<HYD_FMT_F16>(const void *pool, size_t i) {
  return __half2float(static_cast<const __half *>(pool)[i]);
}
template <> __device__ __forceinline__ float vox<HYD_FMT_U8>(const void *pool, size_t i) {
  return u8_norm(static_cast<const uint8_t *>(pool)[i]);
}

// BlockSampler::sample_3d (mapping + CpuSampler Wrap/Linear), as in the volume kernel.
template <int FMT>
__device__ float iso_sample(const IsoArgs &a, int pgid, f3 x) {
  const float4 pg = a.page[pgid];
  const int pad = a.pad;
  const float fd = float(pad);
  float u[3] = {x.x * pg.x + pg.y, x.y * pg.x + pg.z, x.z * pg.x + pg.w};
  float w[3];
  int i[3], j[3];
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    float fx = fd * u[c];
    fx = fx - fd * floorf(fx / fd);
    fx = fx - 0.5f;
    float flr = floorf(fx);
    w[c] = fx - flr;
    i[c] = iclamp((int)flr, 0, pad - 1);
    j[c] = iclamp((int)ceilf(fx), 0, pad - 1);
  }
  const size_t base = (size_t)pgid * pad * pad * pad;
  auto at = [&](int xx, int yy, int zz) { return vox<FMT>(a.pool, base + ((size_t)zz * pad + yy) * pad + xx); };
  const float bx = 1.f - w[0], by = 1.f - w[1], bz = 1.f - w[2];
  float x00 = at(i[0], i[1], i[2]) * bx + at(j[0], i[1], i[2]) * w[0];
  float x10 = at(i[0], j[1], i[2]) * bx + at(j[0], j[1], i[2]) * w[0];
  float x01 = at(i[0], i[1], j[2]) * bx + at(j[0], i[1], j[2]) * w[0];
  float x11 = at(i[0], j[1], j[2]) * bx + at(j[0], j[1], j[2]) * w[0];
  float y0 = x00 * by + x10 * w[1];
  float y1 = x01 * by + x11 * w[1];
  return y0 * bz + y1 * w[2];
}

__device__ __forceinline__ float gsign(float x) { return float((0.f < x) - (x < 0.f)); }

// IsosurfaceShaderKernel::linear_to_srgb: double arithmetic on a float input
// (isosurface_shader.cu:25-32).
__device__ __forceinline__ float iso_srgb(float linear) {
  const double l = linear;
  if (l <= 0.0031308) return (float)(12.92 * l);
  return (float)((1.0 + 0.055) * pow(l, 1.0 / 2.4) - 0.055);
}

// IsosurfaceShaderKernel::main (isosurface_shader.cu:50-125) when
// corrected == 0; bracketing + bisection + oriented central differences when
// corrected == 1.  Two kernels: the march finds each ray's first crossing and
// leaves its state in the output pixel (v = march position and previous value,
// depth = value at the crossing, hit = kIsoPending); the hit kernel then
// refines and shades those pixels.  The march kernel carries none of the
// refinement's registers, so more of its waves fit on a SIMD to cover the
// latency of the tap loads.
constexpr int32_t kIsoPending = -1;

// Side of the isovalue that every sample of a macrocell lies on, from its
// (widened) value range: +1, -1, or 0 when both sides (or a voxel that is not
// finite) are possible.
__device__ __forceinline__ float range_side(float2 r, float scale, float iso) {
  return r.x * scale > iso ? 1.f : r.y * scale < iso ? -1.f : 0.f;
}

// The march of IsosurfaceShaderKernel::main up to the first crossing, with the
// tap loads of up to U consecutive samples in flight together (the step is
// fixed, so the next positions inside a brick follow from the same additions
// the one-step march makes).  The group is evaluated, then scanned in order for
// the first crossing; values, positions, counts and the pending pixel are those
// of the one-step march, but for a skipped sample's value (below).
//
// Macrocells on one side of the isovalue, the previous sample's side, cannot
// hold a crossing: their samples move the position alone, and the previous
// value becomes the range's end nearest the isovalue (only its side is used).
// In the 512^3 sphere field 93% of the macrocells are such, and a ray takes 32
// quarter-voxel samples across one.  The ranges are compared here rather than
// classified ahead for an isovalue: it is an argument of every frame.  The
// range at the position that follows a group is loaded behind the group's taps.
// 1024^2 FP16 frame of that field: 2427 -> 947 us.
template <int FMT, int U, class OFF>
__device__ bool iso_march_grouped(const IsoArgs &a, f3 &o, f3 d, int nsteps, float cdu, hyd_iso_pixel &px,
                                  unsigned &count) {
  const f3 invr = recip3(d);
  const OFF pad3 = (OFF)a.pad * (OFF)a.pad * (OFF)a.pad;
  const f3 inc = muls(d, a.step);
  float prev_value = 0.f;
  bool have_prev = false;
  f3 cip = {-INFINITY, -INFINITY, -INFINITY};
  int ccd = 0, cpg = -1, dpg = -1;
  float4 pgd = make_float4(0.f, 0.f, 0.f, 0.f);
  OFF page_base = 0;
  float2 range = make_float2(NAN, NAN);   // of o's macrocell (NaN: not looked up)
  while (nsteps > 0) {
    const f3 ip = floor3(o);
    if (ip.x != cip.x || ip.y != cip.y || ip.z != cip.z) {
      cip = ip;
      range = make_float2(NAN, NAN);
      if (a.codes) {
        const int code = a.codes[grid_index(ip, a.vdim)];
        ccd = code <= -2 ? -1 - code : 0;
        cpg = code;
      } else {
        ccd = a.cheb[grid_index(ip, a.cdim)];
        if (ccd == 0) cpg = a.vaddr[grid_index(ip, a.vdim)];
      }
    }
    if (ccd) {
      nsteps -= skip_nblock_steps_inv(o, invr, d, ip, ccd, cdu, a.step);
      have_prev = false;
      o = add(o, muls(d, a.step));
      nsteps -= 1;
      continue;
    }
    const int pgid = cpg;
    if (pgid == -1) break;
    if (pgid != dpg) {
      pgd = a.page[pgid];
      page_base = (OFF)pgid * pad3;
      dpg = pgid;
    }
    f3 x[U];
    x[0] = sub(o, ip);
    const float side = range_side(range, a.mm_scale, a.isovalue);
    const bool same = a.corrected && !have_prev ? true : side == gsign(prev_value - a.isovalue);
    if (side != 0.f && same) {
      const int n = min(macro_run(a.macro, 1, x[0], invr, a.step), nsteps);
      if (n > 0) {
#pragma unroll 4
        for (int i = 0; i < n; ++i) o = add(o, inc);
        nsteps -= n;
        count += (unsigned)n;
        if (a.corrected) { prev_value = (side > 0.f ? range.x : range.y) * a.mm_scale; have_prev = true; }
        range = a.mm[macro_index(a.macro, pgid, sub(o, ip))];
        continue;
      }
    }
    bool ok[U];
    f3 q = o;
    ok[0] = true;
#pragma unroll
    for (int j = 1; j < U; ++j) {
      q = add(q, inc);
      x[j] = sub(q, ip);
      ok[j] = ok[j - 1] & (nsteps - j > 0) & in_unit(x[j]);
    }
    bool inner = a.inner == kInnerAlways;
    if (a.inner == kInnerTest) inner = __all(ok[U - 1] & inner_span(x[0], x[U - 1], pgd, a.pad));
    float2 rnext = make_float2(NAN, NAN);
    if (a.mm) rnext = a.mm[macro_index(a.macro, pgid, sub(add(q, inc), ip))];
    float value[U];
    group_values<FMT, OFF, U>(a.pool, a.pad, inner, x, ok, pgd, page_base, value);
    // n: samples before the crossing; cross: the value there
    int n = 0;
    bool live = true;
    float cross = 0.f;
#pragma unroll
    for (int j = 0; j < U; ++j) {
      const float s = gsign(value[j] - a.isovalue);
      const bool differs = s != gsign(prev_value - a.isovalue) && (have_prev || !a.corrected);
      const bool on = ok[j] & live;
      if (on) {
        cross = value[j];
        live = !differs;
      }
      if (on & !differs) {
        ++n;
        if (a.corrected) { prev_value = value[j]; have_prev = true; }
      }
    }
    count += (unsigned)n;
    if (n == U) {
      o = add(q, inc);
    } else {
      for (int j = 0; j < n; ++j) o = add(o, inc);   // the same additions
    }
    if (!live) {
      ++count;
      px.v[0] = o.x; px.v[1] = o.y; px.v[2] = o.z; px.v[3] = prev_value;
      px.depth = cross;
      px.hit = kIsoPending;
      return true;
    }
    nsteps -= n;
    range = rnext;
    if (n < U) range = make_float2(NAN, NAN);
  }
  return false;
}

#ifndef HYD_ISO_GROUP
#define HYD_ISO_GROUP 4
#endif

template <int FMT, bool BIG>
__global__ __launch_bounds__(64) void iso_march_grouped_kernel(IsoArgs a) {
  const int x = rotated_tile_x() * kTile + (threadIdx.x % kTile);
  const int y = blockIdx.y * kTile + (threadIdx.x / kTile);
  if (x >= a.W || y >= a.H) return;
  unsigned count = 0;
  const f3 d = pixel_ray_dir(a.trans, a.ctg, a.ray_o, x, y, a.W, a.H);
  f3 o = a.ray_o;
  hyd_iso_pixel px;
  px.v[0] = px.v[1] = px.v[2] = px.v[3] = 0.f;
  px.depth = INFINITY;
  px.hit = 0;
  float tnear, tfar;
  if (intersect_box(o, d, a.bmin, a.bmax, tnear, tfar)) {
    if (tnear < 0) tnear = 0;
    if (tfar < 0) tfar = 0;
    o = add(o, muls(d, tnear));
    const int n = (int)((tfar - tnear) / a.step);
    const int nsteps = a.max_steps < n ? a.max_steps : n;
    const float cdu = 1.f / comp_max(abs3(d));
    iso_march_grouped<FMT, HYD_ISO_GROUP, std::conditional_t<BIG, uint64_t, uint32_t>>(a, o, d, nsteps, cdu,
                                                                                        px, count);
  }
  a.out[(size_t)y * a.W + x] = px;
  if (a.samples && count) atomicAdd(a.samples, (unsigned long long)count);
}

// Refinement and shading of the pixels the march left pending: the crossing's
// march position o (its brick ip = floor(o) and page from the page table, as
// the march had them), the previous and the crossing value.
template <int FMT>
__global__ __launch_bounds__(64) void iso_hit_kernel(IsoArgs a) {
  const int x = blockIdx.x * kTile + (threadIdx.x % kTile);
  const int y = blockIdx.y * kTile + (threadIdx.x / kTile);
  if (x >= a.W || y >= a.H) return;
  hyd_iso_pixel *out = a.out + (size_t)y * a.W + x;
  const hyd_iso_pixel st = *out;
  if (st.hit != kIsoPending) return;
  const f3 d = pixel_ray_dir(a.trans, a.ctg, a.ray_o, x, y, a.W, a.H);
  const f3 origin = a.ray_o;
  const f3 o = f3{st.v[0], st.v[1], st.v[2]};
  const float prev_value = st.v[3], value = st.depth;
  const f3 ip = floor3(o);
  const int pgid = a.vaddr[grid_index(ip, a.vdim)];
  const f3 p = o;
  const float dt = a.step;
  float4 v = make_float4(a.surface_color.x, a.surface_color.y, a.surface_color.z, 1.f);
  f3 inter_p, nn;
  if (!a.corrected) {
    const float al = (a.isovalue - prev_value) / (value - prev_value);
    const float bl = 1.f - al;
    inter_p = f3{bl * (p.x - dt * d.x) + al * p.x, bl * (p.y - dt * d.y) + al * p.y,
                 bl * (p.z - dt * d.z) + al * p.z};
    const f3 q = sub(inter_p, ip);
    const float h = a.du * 2.f;
    nn = f3{iso_sample<FMT>(a, pgid, f3{q.x - h, q.y - 0.f, q.z - 0.f}) -
                iso_sample<FMT>(a, pgid, f3{q.x + h, q.y + 0.f, q.z + 0.f}),
            iso_sample<FMT>(a, pgid, f3{q.x - 0.f, q.y - h, q.z - 0.f}) -
                iso_sample<FMT>(a, pgid, f3{q.x + 0.f, q.y + h, q.z + 0.f}),
            iso_sample<FMT>(a, pgid, f3{q.x - 0.f, q.y - 0.f, q.z - h}) -
                iso_sample<FMT>(a, pgid, f3{q.x + 0.f, q.y + 0.f, q.z + h})};
  } else {
    f3 plo = p;
    f3 phi = f3{p.x - dt * d.x, p.y - dt * d.y, p.z - dt * d.z};
    const float sprev = gsign(prev_value - a.isovalue);
    for (int it = 0; it < a.bisect_steps; ++it) {
      const f3 mid = {(plo.x + phi.x) * 0.5f, (plo.y + phi.y) * 0.5f, (plo.z + phi.z) * 0.5f};
      const f3 mip = floor3(mid);
      const int mpg = a.vaddr[grid_index(mip, a.vdim)];
      const float mv = mpg == -1 ? value : iso_sample<FMT>(a, mpg, sub(mid, mip));
      if (gsign(mv - a.isovalue) == sprev) phi = mid; else plo = mid;
    }
    inter_p = f3{(plo.x + phi.x) * 0.5f, (plo.y + phi.y) * 0.5f, (plo.z + phi.z) * 0.5f};
    f3 gip = floor3(inter_p);
    int gpg = a.vaddr[grid_index(gip, a.vdim)];
    if (gpg == -1) { gpg = pgid; gip = ip; }
    const f3 q = sub(inter_p, gip);
    const float h = a.du;
    const f3 g = {iso_sample<FMT>(a, gpg, f3{q.x + h, q.y + 0.f, q.z + 0.f}) -
                      iso_sample<FMT>(a, gpg, f3{q.x - h, q.y - 0.f, q.z - 0.f}),
                  iso_sample<FMT>(a, gpg, f3{q.x + 0.f, q.y + h, q.z + 0.f}) -
                      iso_sample<FMT>(a, gpg, f3{q.x - 0.f, q.y - h, q.z - 0.f}),
                  iso_sample<FMT>(a, gpg, f3{q.x + 0.f, q.y + 0.f, q.z + h}) -
                      iso_sample<FMT>(a, gpg, f3{q.x - 0.f, q.y - 0.f, q.z - h})};
    nn = muls(g, sprev);
  }
  float wp4[4], n4[4];
  mat4_vec4(a.to_world, inter_p.x, inter_p.y, inter_p.z, 1.f, wp4);
  mat4_vec4(a.to_world, nn.x, nn.y, nn.z, 0.f, n4);
  const f3 world_p = {wp4[0], wp4[1], wp4[2]};
  const f3 nrm = normalize3(f3{n4[0], n4[1], n4[2]});
  const f3 light_dir = normalize3(sub(a.light_pos, world_p));
  const f3 hv = a.corrected ? normalize3(add(light_dir, normalize3(sub(a.eye_pos, world_p))))
                            : normalize3(sub(light_dir, world_p));
  const float ambient = 0.2f;
  const float diffuse = .6f * gclamp(dot3(light_dir, nrm), 0.f, 1.f);
  const float specular = .2f * powf(gclamp(dot3(hv, nrm), 0.f, 1.f), 100.f);
  const float dist = length3(sub(world_p, a.eye_pos)) / 2.f;
  if (a.mode == HYD_ISO_COLOR) {
    const float sc = ambient + (diffuse + specular) / dist;
    v = make_float4(v.x * sc, v.y * sc, v.z * sc, v.w * sc);
    v = make_float4(iso_srgb(v.x), iso_srgb(v.y), iso_srgb(v.z), v.w);
  } else if (a.mode == HYD_ISO_POSITION) {
    v = make_float4(inter_p.x / a.bmax.x, inter_p.y / a.bmax.y, inter_p.z / a.bmax.z, 1.f);
  } else {
    v = make_float4(nrm.x, nrm.y, nrm.z, 1.f);
  }
  const float depth = a.corrected ? length3(sub(inter_p, origin)) : length3(sub(origin, o));
  hyd_iso_pixel px;
  px.v[0] = v.x; px.v[1] = v.y; px.v[2] = v.z; px.v[3] = v.w;
  px.depth = depth;
  px.hit = 1;
  *out = px;
}

}  // namespace

hipError_t launch_blocks(const BlocksArgs &a, hipStream_t s) {
  dim3 grid((a.W + kTile - 1) / kTile, (a.H + kTile - 1) / kTile);
  hipLaunchKernelGGL(blocks_kernel, grid, dim3(64), 0, s, a);
  return hipGetLastError();
}

namespace {
// HYD_VOLUME_OFFSETS64=1 selects the 64-bit offsets for any pool (same image).
bool iso_force_offsets64() {
  static const bool on = [] {
    const char *e = std::getenv("HYD_VOLUME_OFFSETS64");
    return e && e[0] == '1';
  }();
  return on;
}

template <int FMT>
void launch_iso_fmt(const IsoArgs &a, hipStream_t s) {
  dim3 grid((a.W + kTile - 1) / kTile, (a.H + kTile - 1) / kTile);
  const uint64_t bytes = a.pool_elems * (uint64_t)sizeof(typename RawVox<FMT>::T);
  if (bytes <= (1ull << 32) && !iso_force_offsets64())
    hipLaunchKernelGGL((iso_march_grouped_kernel<FMT, false>), grid, dim3(64), 0, s, a);
  else
    hipLaunchKernelGGL((iso_march_grouped_kernel<FMT, true>), grid, dim3(64), 0, s, a);
  hipLaunchKernelGGL(iso_hit_kernel<FMT>, grid, dim3(64), 0, s, a);
}
}  // namespace

hipError_t launch_iso(const IsoArgs &a, int fmt, hipStream_t s) {
  switch (fmt) {
    case HYD_FMT_U8: launch_iso_fmt<HYD_FMT_U8>(a, s); break;
    case HYD_FMT_F16: launch_iso_fmt<HYD_FMT_F16>(a, s); break;
    default: launch_iso_fmt<HYD_FMT_F32>(a, s);
  }
  return hipGetLastError();
}

}  // namespace hyd
