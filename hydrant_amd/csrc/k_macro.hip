// Macrocell ranges and classes (hyd_macro.hpp).
#include <hip/hip_fp16.h>

#include <algorithm>

#include "hyd_macro.hpp"

namespace hyd {
namespace {

constexpr int kColumns = 4096;   // column ranges staged in LDS (32 KiB)
constexpr int kMaxTf = 256;

template <int FMT> struct MVox;
template <> struct MVox<HYD_FMT_U8> {
  using T = uint8_t;
  static __device__ __forceinline__ float get(T v) { return float(v); }
};
template <> struct MVox<HYD_FMT_F16> {
  using T = __half;
  static __device__ __forceinline__ float get(T v) { return __half2float(v); }
};
template <> struct MVox<HYD_FMT_F32> {
  using T = float;
  static __device__ __forceinline__ float get(T v) { return v; }
};

// One workgroup per (page, z row of macrocells): each thread takes the range of
// one x column over a macrocell row's 9 x 9 (y, z) voxels, so reads run along
// x; the columns are then reduced by 9 in LDS.  Bound by the voxel reads (1.27
// of the pool, the overlaps from the L2); runs once per pool upload.
template <int FMT>
__global__ __launch_bounds__(256) void macro_minmax_kernel(const void *pool, int pad, int first, float2 *mm) {
  using V = MVox<FMT>;
  __shared__ float2 s_col[kColumns];
  const int nm = (pad + kMacro - 1) / kMacro;
  const size_t page = (size_t)first + blockIdx.x;
  const typename V::T *pg = static_cast<const typename V::T *>(pool) + page * pad * pad * pad;
  float2 *out = mm + page * nm * nm * nm;
  const int mz = blockIdx.y, z0 = mz * kMacro, z1 = min(z0 + kMacro, pad - 1);
  const int rows = kColumns / pad;
  for (int my0 = 0; my0 < nm; my0 += rows) {
    const int nr = min(rows, nm - my0);
    for (int i = threadIdx.x; i < nr * pad; i += 256) {
      const int y0 = (my0 + i / pad) * kMacro, y1 = min(y0 + kMacro, pad - 1), x = i % pad;
      float lo = INFINITY, hi = -INFINITY;
      bool bad = false;
      for (int z = z0; z <= z1; ++z)
        for (int y = y0; y <= y1; ++y) {
          const float v = V::get(pg[((size_t)z * pad + y) * pad + x]);
          bad = bad || !(fabsf(v) <= 1e30f);
          lo = fminf(lo, v);
          hi = fmaxf(hi, v);
        }
      s_col[i] = bad ? make_float2(-INFINITY, INFINITY) : make_float2(lo, hi);
    }
    __syncthreads();
    for (int i = threadIdx.x; i < nr * nm; i += 256) {
      const int r = i / nm, mx = i % nm, x0 = mx * kMacro, x1 = min(x0 + kMacro, pad - 1);
      float lo = INFINITY, hi = -INFINITY;
      for (int x = x0; x <= x1; ++x) {
        lo = fminf(lo, s_col[r * pad + x].x);
        hi = fmaxf(hi, s_col[r * pad + x].y);
      }
      const bool bad = lo == -INFINITY || hi == INFINITY;
      out[((size_t)mz * nm + my0 + r) * nm + mx] = bad ? make_float2(NAN, NAN) : make_float2(lo, hi);
    }
    __syncthreads();
  }
}

// flag = 1 when the macrocell may contribute: some transfer-function entry that
// a value of its range can touch has a non-zero alpha.  The range is widened by
// 2^-19 of its magnitude (the interpolation's rounding) and the entry positions
// by 1e-3.
__global__ __launch_bounds__(256) void macro_flag_kernel(const float2 *mm, int cells, size_t first_cell, size_t n,
                                                         const float *tf, int tf_n, float scale,
                                                         const float *page_scale, uint8_t *flags,
                                                         unsigned long long *n_flagged) {
  __shared__ int s_pre[kMaxTf + 1];   // s_pre[i]: non-zero alphas among entries 0 .. i - 1
  if (threadIdx.x == 0) {
    int c = 0;
    for (int i = 0; i < tf_n; ++i) {
      s_pre[i] = c;
      c += tf[4 * i + 3] != 0.f ? 1 : 0;
    }
    s_pre[tf_n] = c;
  }
  __syncthreads();
  unsigned mine = 0;
  for (size_t j = (size_t)blockIdx.x * 256 + threadIdx.x; j < n; j += (size_t)gridDim.x * 256) {
    const size_t i = first_cell + j;
    const float2 r = mm[i];
    const float sc = page_scale ? page_scale[i / cells] : scale;
    const float m = fmaxf(fabsf(r.x), fabsf(r.y)) * 1.9073486e-6f;
    const float lo = (r.x - m) * sc, hi = (r.y + m) * sc;
    uint8_t f = 1;
    if (hi < 0.f || lo > 1.f) {
      f = 0;   // outside the table: the border's zero
    } else if (lo <= hi) {   // false for NaN ranges and scales
      const float a = float(tf_n) * fmaxf(lo, 0.f) - 0.5f, b = float(tf_n) * fminf(hi, 1.f) - 0.5f;
      const int e0 = iclamp((int)floorf(a - 1e-3f), 0, tf_n - 1), e1 = iclamp((int)ceilf(b + 1e-3f), 0, tf_n - 1);
      f = s_pre[e1 + 1] != s_pre[e0] ? 1 : 0;
    }
    flags[i] = f;
    mine += f;
  }
  for (int o = 32; o > 0; o >>= 1) mine += __shfl_xor(mine, o);
  if ((threadIdx.x & 63) == 0 && mine) atomicAdd(n_flagged, (unsigned long long)mine);
}

// Class of every macrocell: 0 if flagged, else one more than the largest radius
// r < kMacroCap whose rings 1 .. r hold no flag inside the page.
__global__ __launch_bounds__(256) void macro_class_kernel(const uint8_t *flags, int nm, size_t first_cell, size_t n,
                                                          uint8_t *cls) {
  const int cells = nm * nm * nm;
  for (size_t j = (size_t)blockIdx.x * 256 + threadIdx.x; j < n; j += (size_t)gridDim.x * 256) {
    const size_t i = first_cell + j;
    const int c = (int)(i % cells);
    const uint8_t *pg = flags + (i - c);
    int d = 0;
    if (!pg[c]) {
      const int x = c % nm, y = (c / nm) % nm, z = c / (nm * nm);
      d = 1;
      for (int r = 1; r < kMacroCap; ++r) {
        bool any = false;
        for (int dz = -r; dz <= r && !any; ++dz)
          for (int dy = -r; dy <= r && !any; ++dy) {
            const int zz = z + dz, yy = y + dy;
            if (zz < 0 || zz >= nm || yy < 0 || yy >= nm) continue;
            const bool face = dz == -r || dz == r || dy == -r || dy == r;
            for (int dx = -r; dx <= r; dx += face ? 1 : 2 * r) {
              const int xx = x + dx;
              if (xx >= 0 && xx < nm && pg[(zz * nm + yy) * nm + xx]) any = true;
            }
          }
        if (any) break;
        d = r + 1;
      }
    }
    cls[i] = (uint8_t)d;
  }
}

}  // namespace

hipError_t launch_macro_minmax(int fmt, const void *pool, int pad, int first, int n, float2 *mm, hipStream_t s) {
  // a launch holds fewer than 2^32 threads on an axis: 256 a page
  constexpr int kPages = 1 << 22;
  for (; n > 0; first += kPages, n -= kPages) {
    const dim3 grid(std::min(n, kPages), macro_edge(pad));
    switch (fmt) {
      case HYD_FMT_U8:
        hipLaunchKernelGGL(macro_minmax_kernel<HYD_FMT_U8>, grid, dim3(256), 0, s, pool, pad, first, mm);
        break;
      case HYD_FMT_F16:
        hipLaunchKernelGGL(macro_minmax_kernel<HYD_FMT_F16>, grid, dim3(256), 0, s, pool, pad, first, mm);
        break;
      default:
        hipLaunchKernelGGL(macro_minmax_kernel<HYD_FMT_F32>, grid, dim3(256), 0, s, pool, pad, first, mm);
    }
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

hipError_t launch_macro_classes(const float2 *mm, int pad, int first, int n, const float *tf, int tf_n, float scale,
                                const float *page_scale, uint8_t *flags, uint8_t *cls, unsigned long long *n_flagged,
                                hipStream_t s) {
  if (n <= 0) return hipSuccess;
  const int nm = macro_edge(pad), cells = nm * nm * nm;
  const size_t total = (size_t)n * cells, at = (size_t)first * cells;
  const unsigned grid = (unsigned)std::min<size_t>((total + 255) / 256, 8192);
  hipLaunchKernelGGL(macro_flag_kernel, dim3(grid), dim3(256), 0, s, mm, cells, at, total, tf, tf_n, scale,
                     page_scale, flags, n_flagged);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(macro_class_kernel, dim3(grid), dim3(256), 0, s, flags, nm, at, total, cls);
  return hipGetLastError();
}

}  // namespace hyd
