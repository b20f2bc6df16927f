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

// One workgroup per (page, z row of macrocells, `rows` of their y rows): each
// thread takes the ranges of V neighbouring x columns over a macrocell row's 9 x 9
// (y, z) voxels, nine loads of V voxels in flight; the columns are then reduced by
// 9 in LDS.  Bound by the voxel reads (1.27 of the pool, the overlaps from the
// L2); runs once per pool upload, behind the copy.  With single-voxel loads and
// every y row in one workgroup (32 of them for one 256^3 page) an upload of that
// page in FP32 took 3.77 ms and one of 4096 u8 pages of 66^3 44.3 ms; 2.38 and
// 39.5 ms so, and 2.58 and 41.5 before there were ranges.
template <int FMT, int V>
__global__ __launch_bounds__(256) void macro_minmax_kernel(const void *pool, int pad, int first, int rows, float2 *mm) {
  using X = MVox<FMT>;
  __shared__ float2 s_col[kColumns];
  const int nm = (pad + kMacro - 1) / kMacro, nx = (pad + V - 1) / V;
  const size_t page = (size_t)first + blockIdx.x;
  const typename X::T *pg = static_cast<const typename X::T *>(pool) + page * pad * pad * pad;
  float2 *out = mm + page * nm * nm * nm;
  const int mz = blockIdx.y, z0 = mz * kMacro, z1 = min(z0 + kMacro, pad - 1);
  const int my0 = blockIdx.z * rows, nr = min(rows, nm - my0);
  for (int i = threadIdx.x; i < nr * nx; i += 256) {
    const int r = i / nx, x = min((i % nx) * V, pad - V), y0 = (my0 + r) * kMacro;
    float lo[V], hi[V];
    bool bad[V];
#pragma unroll
    for (int v = 0; v < V; ++v) {
      lo[v] = INFINITY;
      hi[v] = -INFINITY;
      bad[v] = false;
    }
    for (int z = z0; z <= z1; ++z) {
      typename X::T t[kMacro + 1][V];
#pragma unroll
      for (int y = 0; y <= kMacro; ++y)   // the last rows of a page repeat
        __builtin_memcpy(t[y], pg + ((size_t)z * pad + min(y0 + y, pad - 1)) * pad + x, sizeof(t[y]));
#pragma unroll
      for (int y = 0; y <= kMacro; ++y)
#pragma unroll
        for (int v = 0; v < V; ++v) {
          const float f = X::get(t[y][v]);
          bad[v] = bad[v] || !(fabsf(f) <= 1e30f);
          lo[v] = fminf(lo[v], f);
          hi[v] = fmaxf(hi[v], f);
        }
    }
#pragma unroll
    for (int v = 0; v < V; ++v)
      s_col[r * pad + x + v] = bad[v] ? make_float2(-INFINITY, INFINITY) : make_float2(lo[v], hi[v]);
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

namespace {
template <int FMT>
hipError_t minmax_pages(const void *pool, int pad, int first, int n, int rows, float2 *mm, hipStream_t s) {
  const int nm = macro_edge(pad);
  const dim3 grid(n, nm, (nm + rows - 1) / rows), block(256);
  if (pad >= 4) hipLaunchKernelGGL((macro_minmax_kernel<FMT, 4>), grid, block, 0, s, pool, pad, first, rows, mm);
  else hipLaunchKernelGGL((macro_minmax_kernel<FMT, 1>), grid, block, 0, s, pool, pad, first, rows, mm);
  return hipGetLastError();
}
}  // namespace

hipError_t launch_macro_minmax(int fmt, const void *pool, int pad, int first, int n, float2 *mm, hipStream_t s) {
  // a launch holds fewer than 2^32 threads on an axis: 256 a page
  constexpr int kPages = 1 << 22;
  // as many y rows a workgroup as its LDS holds, or fewer while that leaves the chip idle
  const int nm = macro_edge(pad), most = std::min(nm, kColumns / pad);
  const int rows = (int64_t)n * nm >= 4096 ? most : std::min(most, std::max(1, 256 / pad));
  for (; n > 0; first += kPages, n -= kPages) {
    const int k = std::min(n, kPages);
    const hipError_t e = fmt == HYD_FMT_U8    ? minmax_pages<HYD_FMT_U8>(pool, pad, first, k, rows, mm, s)
                         : fmt == HYD_FMT_F16 ? minmax_pages<HYD_FMT_F16>(pool, pad, first, k, rows, mm, s)
                                              : minmax_pages<HYD_FMT_F32>(pool, pad, first, k, rows, mm, s);
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
