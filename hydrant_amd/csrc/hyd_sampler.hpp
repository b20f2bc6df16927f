// The reference CPU sampler (BlockSamplerMapping + CpuSampler Wrap/Linear over
// a padded brick, block_paging.hpp:11-36, cpu_sampler.hpp:88-104,142-166)
// split into the steps a march pipelines: tap offsets and weights of a
// sample, the loads of its taps, their conversion to float, and the trilinear
// interpolation.  Shared by the volume and isosurface marches.
#pragma once

#include <hip/hip_fp16.h>

#include <type_traits>

#include "hyd_internal.hpp"

namespace hyd {

// Reference sampler taps of one sample: the element offsets of the four rows
// (y, z) = (i, i), (j, i), (i, j), (j, j) of the padded brick, the x taps and the
// weights (BlockSamplerMapping + CpuSampler Wrap/Linear, block_paging.hpp:11-36,
// cpu_sampler.hpp:88-104,142-166).
template <class OFF> struct RefTap {
  OFF r00, r10, r01, r11;
  int ix, jx;
  float ax, ay, az;
};

// floor(fx) and ceil(fx) are integers, so clamping them to [0, pad - 1] as floats
// (one med3) and converting gives the reference's clamped int taps.  Row
// offsets below 2^24 voxels per page use 24-bit multiplies (pad <= 1024, so
// z * pad + y < 2^20 and a row start < 2^30).
template <class OFF>
__device__ __forceinline__ RefTap<OFF> ref_tap(f3 x, float4 pg, int pad, OFF page_base) {
  const float fd = float(pad);
  const float hi = fd - 1.f;
  const float u[3] = {x.x * pg.x + pg.y, x.y * pg.x + pg.z, x.z * pg.x + pg.w};
  float a[3];
  uint32_t i[3], j[3];
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    float fx = fd * u[k];
    fx = wrap_mod(fx, fd);   // Wrap: glm mod(fx, fd)
    fx = fx - 0.5f;
    const float flr = floorf(fx);
    a[k] = fx - flr;
    i[k] = (uint32_t)__builtin_amdgcn_fmed3f(flr, 0.f, hi);
    j[k] = (uint32_t)__builtin_amdgcn_fmed3f(ceilf(fx), 0.f, hi);
  }
  RefTap<OFF> t;
  const uint32_t p = (uint32_t)pad;
  t.r00 = page_base + (OFF)__umul24(__umul24(i[2], p) + i[1], p);
  t.r10 = page_base + (OFF)__umul24(__umul24(i[2], p) + j[1], p);
  t.r01 = page_base + (OFF)__umul24(__umul24(j[2], p) + i[1], p);
  t.r11 = page_base + (OFF)__umul24(__umul24(j[2], p) + j[1], p);
  t.ix = (int)i[0];
  t.jx = (int)j[0];
  t.ax = a[0];
  t.ay = a[1];
  t.az = a[2];
  return t;
}

// Raw taps as loaded.  Every row is read as an x pair: the two voxels at
// m = min(ix, pad - 2) and m + 1 in one load (8 bytes at 4-byte alignment for
// FP32, 4 bytes at 2-byte alignment for FP16, 2 bytes at any alignment for
// u8), which the vector memory unit serves at the per-lane cost of one of the
// two single loads; the taps are then v(ix) = ix == m ? lo : hi and
// v(jx) = jx == m + 1 ? hi : lo, which also covers the clamped and integral
// cases (ix == jx).  Each load has a register of its own (pairs of rows packed
// into one register would make each load wait for the previous one).  A
// grouped u8 march issues 8 samples x 4 row loads per group; with one load per
// tap it issued 64, and the vector memory unit's per-instruction cost (one
// cache-line lookup per distinct line a wave's lanes touch) set the time of a
// group, not the memory latency.  Values are converted to float once, when a
// sample uses them.
template <int FMT> struct RawVox;
template <> struct RawVox<HYD_FMT_F32> { using T = float; static constexpr int N = 8; };
template <> struct RawVox<HYD_FMT_F16> { using T = uint16_t; static constexpr int N = 4; };
template <> struct RawVox<HYD_FMT_U8> { using T = uint8_t; static constexpr int N = 4; };

template <int FMT> struct RawTaps { uint32_t v[RawVox<FMT>::N]; };

// float(c) / 255.f, correctly rounded, for a count c in 0 .. 255
// (Texture3D<u8> NormalizedFloat): 1/255 split into two floats, whose FMA
// rounds to the quotient for all 256 counts.  Two VALU operations per tap; the
// 256-entry LDS table it replaces cost an address and a dependent, bank-conflicting
// LDS read per tap, eight a sample.
__host__ __device__ __forceinline__ float u8_norm(uint32_t c) {
  const float v = float(c);
  return fmaf(v, 0x1.010102p-8f, v * -0x1.fdfdfep-33f);
}

// Row k's x pair, loaded from p.
template <int FMT> __device__ __forceinline__ void raw_load(const char *p, RawTaps<FMT> &r, int k) {
  if constexpr (FMT == HYD_FMT_F32) {
    __builtin_memcpy(&r.v[2 * k], p, 8);
  } else if constexpr (FMT == HYD_FMT_F16) {
    __builtin_memcpy(&r.v[k], p, 4);
  } else {
    uint16_t pair;
    __builtin_memcpy(&pair, p, 2);
    r.v[k] = pair;
  }
}

// Row k's two voxels as floats.
template <int FMT> __device__ __forceinline__ void raw_pair(const RawTaps<FMT> &r, int k, float &lo, float &hi) {
  if constexpr (FMT == HYD_FMT_F32) {
    lo = __uint_as_float(r.v[2 * k]);
    hi = __uint_as_float(r.v[2 * k + 1]);
  } else if constexpr (FMT == HYD_FMT_F16) {
    lo = __half2float(__ushort_as_half((unsigned short)(r.v[k] & 0xffffu)));
    hi = __half2float(__ushort_as_half((unsigned short)(r.v[k] >> 16)));
  } else {
    lo = u8_norm(r.v[k] & 0xffu);
    hi = u8_norm(r.v[k] >> 8);
  }
}

// Byte offsets are formed in OFF, so with 32-bit offsets a load is the pool's
// scalar base plus one 32-bit register.
template <int FMT, class OFF>
__device__ __forceinline__ void ref_fetch(const void *pool, const RefTap<OFF> &t, int pad, RawTaps<FMT> &r) {
  const char *b = static_cast<const char *>(pool);
  constexpr OFF sz = (OFF)sizeof(typename RawVox<FMT>::T);
  const OFF rows[4] = {t.r00 * sz, t.r10 * sz, t.r01 * sz, t.r11 * sz};
  const OFF xm = (OFF)min(t.ix, pad - 2) * sz;
#pragma unroll
  for (int k = 0; k < 4; ++k) raw_load<FMT>(b + (rows[k] + xm), r, k);
}

// The eight tap values of a fresh sample, x-y-z order.
template <int FMT, class OFF>
__device__ __forceinline__ void ref_values(const RawTaps<FMT> &r, const RefTap<OFF> &t, int pad, float (&v)[8]) {
  const int m = min(t.ix, pad - 2);
  const bool i_lo = t.ix == m, j_hi = t.jx == m + 1;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    float lo, hi;
    raw_pair<FMT>(r, k, lo, hi);
    v[2 * k] = i_lo ? lo : hi;
    v[2 * k + 1] = j_hi ? hi : lo;
  }
}

// The reference's tap coordinate pad * (x * k + b) - 0.5 on one axis, before the Wrap.
__device__ __forceinline__ float tap_coord(float x, float k, float b, float fd) { return fd * (x * k + b) - 0.5f; }

// A sample whose tap coordinates all lie in [0, pad - 1): the Wrap is the
// identity, no tap clamps, and the upper taps follow the lower ones.  Where a
// weight is zero the reference reads the lower tap twice; reading the next
// voxel instead gives the same sum while that voxel is finite (v * 1 + u * 0),
// and a NaN where it is not (group_values then falls back).  So the four rows
// sit at fixed distances from one offset, and nothing is selected: with the
// table lookups below, 165 -> 127 VALU instructions a sample of the 512^2 FP32
// frame (508 -> 471 us; VALU 71% and the texture data unit 71% busy), and
// 239 -> 186 us for the paged 1024^3 u8 frame, whose longest rays' instruction
// streams set its time.
template <class OFF> struct InnerTap {
  OFF off;            // byte offset of tap (i, i, i)
  float ax, ay, az;
};

template <int FMT, class OFF>
__device__ __forceinline__ InnerTap<OFF> inner_tap(f3 x, float4 pg, int pad, OFF page_base) {
  const float fd = float(pad);
  const float fx = tap_coord(x.x, pg.x, pg.y, fd), fy = tap_coord(x.y, pg.x, pg.z, fd),
              fz = tap_coord(x.z, pg.x, pg.w, fd);
  const float flx = floorf(fx), fly = floorf(fy), flz = floorf(fz);
  InnerTap<OFF> t;
  t.ax = fx - flx;
  t.ay = fy - fly;
  t.az = fz - flz;
  // row index z * pad + y formed in float (exact below 2^20), then one 24-bit product
  const uint32_t i = __umul24((uint32_t)fmaf(flz, fd, fly), (uint32_t)pad) + (uint32_t)flx;
  t.off = (page_base + (OFF)i) * (OFF)sizeof(typename RawVox<FMT>::T);
  return t;
}

template <int FMT, class OFF>
__device__ __forceinline__ void inner_fetch(const void *pool, OFF off, int pad, RawTaps<FMT> &r) {
  using T = typename RawVox<FMT>::T;
  const char *b = static_cast<const char *>(pool);
  const int dy = pad * (int)sizeof(T), dz = pad * dy;   // uniform: four scalar bases, one offset register
  raw_load<FMT>(b + off, r, 0);
  raw_load<FMT>(b + dy + off, r, 1);
  raw_load<FMT>(b + dz + off, r, 2);
  raw_load<FMT>(b + (dy + dz) + off, r, 3);
}

template <class TAP> __device__ __forceinline__ float ref_interp(const float (&v)[8], const TAP &t);

// Values of a group of samples x[j] (brick coordinates) of one page, their tap
// loads in flight together; s[j] is defined where ok[j] (ok[0] holds).  `inner`
// (the same for the wave): every ok sample's taps are inside the page as
// InnerTap needs them.  Same values bit for bit either way (but for the sign
// of a zero).
template <int FMT, class OFF, int N>
__device__ __forceinline__ void group_values(const void *pool, int pad, bool inner, const f3 (&x)[N],
                                             const bool (&ok)[N], float4 pg, OFF page_base, float (&s)[N]) {
  if (inner) {
    InnerTap<OFF> t[N];
    RawTaps<FMT> raw[N];
#pragma unroll
    for (int j = 0; j < N; ++j) {
      t[j] = inner_tap<FMT, OFF>(x[j], pg, pad, page_base);
      if (j > 0) t[j].off = ok[j] ? t[j].off : t[0].off;   // no branch: a sample that is not read repeats the first's loads
      inner_fetch<FMT, OFF>(pool, t[j].off, pad, raw[j]);
    }
    bool bad = false;
#pragma unroll
    for (int j = 0; j < N; ++j) {
      float v[8];
#pragma unroll
      for (int k = 0; k < 4; ++k) raw_pair<FMT>(raw[j], k, v[2 * k], v[2 * k + 1]);
      s[j] = ref_interp(v, t[j]);
      if (FMT != HYD_FMT_U8) bad |= !(fabsf(s[j]) <= 3.4028235e38f);   // a voxel that is not finite
    }
    inner = !bad;
  }
  if (!inner) {
    constexpr int V = (N + 1) / 2;   // the clamping taps take more registers: two halves
#pragma unroll
    for (int j0 = 0; j0 < N; j0 += V) {
      RefTap<OFF> t[V];
      RawTaps<FMT> raw[V];
#pragma unroll
      for (int i = 0; i < V && j0 + i < N; ++i) {
        t[i] = ref_tap<OFF>(x[j0 + i], pg, pad, page_base);
        if (ok[j0 + i]) ref_fetch<FMT, OFF>(pool, t[i], pad, raw[i]);
      }
#pragma unroll
      for (int i = 0; i < V && j0 + i < N; ++i) {
        if (ok[j0 + i]) {
          float v[8];
          ref_values<FMT, OFF>(raw[i], t[i], pad, v);
          s[j0 + i] = ref_interp(v, t[i]);
        }
      }
    }
  }
}

// True when every tap coordinate of the samples from x0 to x1 (brick
// coordinates of a ray's samples, so monotone on each axis) lies in [0, pad - 1).
__device__ __forceinline__ bool inner_span(f3 x0, f3 x1, float4 pg, int pad) {
  const float fd = float(pad);
  const float a = tap_coord(x0.x, pg.x, pg.y, fd), b = tap_coord(x1.x, pg.x, pg.y, fd);
  const float c = tap_coord(x0.y, pg.x, pg.z, fd), d = tap_coord(x1.y, pg.x, pg.z, fd);
  const float e = tap_coord(x0.z, pg.x, pg.w, fd), f = tap_coord(x1.z, pg.x, pg.w, fd);
  // NaN fails: min and max drop it, the sum keeps it
  return fminf(fminf(fminf(a, b), fminf(c, d)), fminf(e, f)) >= 0.f &&
         fmaxf(fmaxf(fmaxf(a, b), fmaxf(c, d)), fmaxf(e, f)) < fd - 1.f && (a + b) + (c + d) + (e + f) >= 0.f;
}

// x in [0, 1) on every axis, where x = p - floor-of-the-brick: p is in the
// brick.  (As unsigned bits, negative and NaN values exceed those of [0, 1).)
// Exact for p >= 0; a p within rounding below 0 may test false in brick -1, which
// only ends a group early.
__device__ __forceinline__ bool in_unit(f3 x) {
  return max(max(__float_as_uint(x.x), __float_as_uint(x.y)), __float_as_uint(x.z)) < 0x3f800000u;
}

// x -> y -> z lerps with x * (1 - t) + y * t (cpu_sampler.hpp:126-129).
template <class TAP>
__device__ __forceinline__ float ref_interp(const float (&v)[8], const TAP &t) {
  const float bx = 1.f - t.ax;
  const float x00 = v[0] * bx + v[1] * t.ax;
  const float x10 = v[2] * bx + v[3] * t.ax;
  const float x01 = v[4] * bx + v[5] * t.ax;
  const float x11 = v[6] * bx + v[7] * t.ax;
  const float by = 1.f - t.ay;
  const float y0 = x00 * by + x10 * t.ay;
  const float y1 = x01 * by + x11 * t.ay;
  const float bz = 1.f - t.az;
  return y0 * bz + y1 * t.az;
}


}  // namespace hyd
