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

// Page of entry b among the runs' pages.
__device__ __forceinline__ int run_page(const MacroRuns &r, int b) {
  int i = 0;
  while (i + 1 < r.n && b >= r.start[i + 1]) ++i;
  return r.first[i] + (b - r.start[i]);
}

// One workgroup per (page, z row of macrocells, `rows` of their y rows): each
// thread takes the ranges of V neighbouring x columns over a macrocell row's 9 x 9
// (y, z) voxels, nine loads of V voxels in flight; the columns are then reduced by
// 9 in LDS.  Bound by the voxel reads (1.27 of the pool, the overlaps from the
// L2); runs once per pool upload, behind the copy.  With single-voxel loads and
// every y row in one workgroup (32 of them for one 256^3 page) an upload of that
// page in FP32 took 3.77 ms and one of 4096 u8 pages of 66^3 44.3 ms; 2.38 and
// 39.5 ms so, and 2.58 and 41.5 before there were ranges.
template <int FMT, int V>
__global__ __launch_bounds__(256) void macro_minmax_kernel(const void *pool, int pad, MacroRuns runs, int base, int rows,
                                                           float2 *mm) {
  using X = MVox<FMT>;
  __shared__ float2 s_col[kColumns];
  const int nm = (pad + kMacro - 1) / kMacro, nx = (pad + V - 1) / V;
  const size_t page = (size_t)run_page(runs, base + (int)blockIdx.x);
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
    const float m = range_margin(lo, hi);
    out[((size_t)mz * nm + my0 + r) * nm + mx] = bad ? make_float2(NAN, NAN) : make_float2(lo - m, hi + m);
  }
}

// Classes of whole pages (up to 16 macrocells an edge, as many pages as give 256
// rows) or of tiles of 8 macrocells an edge.  A macrocell is flagged when it may
// contribute: some transfer-function entry that a value of its range can touch
// has a non-zero alpha; the entry positions are widened by 1e-3.  The flags of a page
// or of a tile with its neighbours up to kMacroCap - 1 away are one word of bits per
// x row in LDS; widened by one macrocell on every axis, a thread a row, the r-th
// time they hold what lies within r, so the class is the number of widenings
// that leave a macrocell clear, and one more.  Bound by the latency of the ranges'
// loads; 4096 pages of 9^3 macrocells in 30 us, one of 32^3 in 12.  With a byte per
// flag in memory, up to 343 of them read for each class, and the table counted by one
// thread a workgroup, hyd_set_tf took 456 us for the 4096 pages (20 without classes).
constexpr int kTileM = 8, kWholeM = 16, kAhead = 3;   // kAhead: ranges a thread loads together
__global__ __launch_bounds__(256) void macro_class_kernel(const float2 *mm, int nm, MacroRuns runs, int pages, int groups,
                                                          const float *tf, int tf_n, float scale,
                                                          const float *page_scale, uint8_t *cls, bool replace,
                                                          unsigned long long *counts, unsigned long long *zero) {
  __shared__ int s_pre[kMaxTf + 1];   // s_pre[i]: non-zero alphas among entries 0 .. i - 1
  __shared__ int s_wave[4];
  __shared__ int s_page[256];
  __shared__ uint32_t s_bits[kMacroCap][256];
  __shared__ int s_sum[2];
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const bool nz = t < tf_n && tf[4 * t + 3] != 0.f;
  const unsigned long long m = __ballot(nz);
  if (lane == 0) s_wave[wave] = __popcll(m);
  if (t < 2) s_sum[t] = 0;
  __syncthreads();
  int pre = __popcll(m & ((1ull << lane) - 1ull));
  for (int w = 0; w < wave; ++w) pre += s_wave[w];
  if (t < tf_n) s_pre[t] = pre;
  if (t == tf_n - 1) s_pre[tf_n] = pre + (nz ? 1 : 0);
  const bool whole = nm <= kWholeM;
  const int tl = whole ? 1 : (nm + kTileM - 1) / kTileM, tiles = tl * tl * tl, cells = nm * nm * nm;
  int n0 = 0, n3 = 0;   // macrocells of class 0, and of class 3 or more
  for (int g = blockIdx.x; g < groups; g += gridDim.x) {
    const int b0 = whole ? g * pages : g / tiles, np = whole ? min(pages, runs.total - b0) : 1;
    int i0[3], i1[3], e0[3], e[3];   // the macrocells to class, and with their neighbours
    int q = whole ? 0 : g % tiles;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      const int c = q % tl;
      q /= tl;
      i0[k] = c * kTileM;
      i1[k] = whole ? nm : min(i0[k] + kTileM, nm);
      e0[k] = max(i0[k] - (kMacroCap - 1), 0);
      e[k] = min(i1[k] + (kMacroCap - 1), nm) - e0[k];
    }
    const int R = e[1] * e[2], ce = e[0] * R;
    __syncthreads();   // s_pre, and the last group's bits are read
    if (t < np) s_page[t] = run_page(runs, b0 + t);
    s_bits[0][t] = 0;
    __syncthreads();
    for (int first = t; first < np * ce; first += 256 * kAhead) {
      float2 rg[kAhead];
      int at[kAhead], bit[kAhead], page[kAhead];
#pragma unroll
      for (int k = 0; k < kAhead; ++k) {   // past the end: the last one again
        const int i = min(first + 256 * k, np * ce - 1);
        const int pi = i / ce, c = i - pi * ce, row = c / e[0], z = row / e[1];
        bit[k] = c - row * e[0];
        at[k] = pi * R + row;
        page[k] = s_page[pi];
        rg[k] = mm[(size_t)page[k] * cells + ((size_t)(e0[2] + z) * nm + (e0[1] + row - z * e[1])) * nm + (e0[0] + bit[k])];
      }
#pragma unroll
      for (int k = 0; k < kAhead; ++k) {
        const float2 r = rg[k];
        const float sc = page_scale ? page_scale[page[k]] : scale;
        const float lo = r.x * sc, hi = r.y * sc;
        bool f = true;
        if (hi < 0.f || lo > 1.f) {
          f = false;   // outside the table: the border's zero
        } else if (lo <= hi) {   // false for NaN ranges and scales
          const float a = float(tf_n) * fmaxf(lo, 0.f) - 0.5f, b = float(tf_n) * fminf(hi, 1.f) - 0.5f;
          const int j0 = iclamp((int)floorf(a - 1e-3f), 0, tf_n - 1), j1 = iclamp((int)ceilf(b + 1e-3f), 0, tf_n - 1);
          f = s_pre[j1 + 1] != s_pre[j0];
        }
        if (f) atomicOr(&s_bits[0][at[k]], 1u << bit[k]);
      }
    }
    __syncthreads();
    const int row = t % R, ry = row % e[1], rz = row / e[1];   // this thread's row of page t / R
#pragma unroll
    for (int r = 1; r < kMacroCap; ++r) {
      if (t < np * R) {
        uint32_t v = 0;
        for (int dz = -1; dz <= 1; ++dz)
          for (int dy = -1; dy <= 1; ++dy)
            if (ry + dy >= 0 && ry + dy < e[1] && rz + dz >= 0 && rz + dz < e[2]) v |= s_bits[r - 1][t + dz * e[1] + dy];
        s_bits[r][t] = v | v << 1 | v >> 1;
      }
      __syncthreads();
    }
    const int ix = i1[0] - i0[0], iy = i1[1] - i0[1], ci = ix * iy * (i1[2] - i0[2]);
    for (int i = t; i < np * ci; i += 256) {
      const int pi = i / ci, c = i - pi * ci, row = c / ix, x = i0[0] + c - row * ix, z = i0[2] + row / iy,
                y = i0[1] + row % iy;
      const int at = pi * R + (z - e0[2]) * e[1] + (y - e0[1]);
      int d = 0;
#pragma unroll
      for (int r = 0; r < kMacroCap; ++r) d += (s_bits[r][at] >> (x - e0[0]) & 1u) ? 0 : 1;
      uint8_t *out = cls + (size_t)s_page[pi] * cells + ((size_t)z * nm + y) * nm + x;
      if (replace) {
        const int old = *out;
        n0 -= old == 0;
        n3 -= old >= 3;
      }
      *out = (uint8_t)d;
      n0 += d == 0;
      n3 += d >= 3;
    }
  }
  for (int o = 32; o > 0; o >>= 1) {
    n0 += __shfl_xor(n0, o);
    n3 += __shfl_xor(n3, o);
  }
  if (lane == 0) {
    atomicAdd(&s_sum[0], n0);
    atomicAdd(&s_sum[1], n3);
  }
  __syncthreads();
  if (blockIdx.x == 0 && t < 2 && zero) zero[t] = 0;
  if (t < 2 && s_sum[t] != 0) atomicAdd(counts + t, (unsigned long long)(long long)s_sum[t]);
}

template <int FMT>
hipError_t minmax_pages(const void *pool, int pad, const MacroRuns &runs, int base, int n, int rows, float2 *mm,
                        hipStream_t s) {
  const int nm = macro_edge(pad);
  const dim3 grid(n, nm, (nm + rows - 1) / rows), block(256);
  if (pad >= 4) hipLaunchKernelGGL((macro_minmax_kernel<FMT, 4>), grid, block, 0, s, pool, pad, runs, base, rows, mm);
  else hipLaunchKernelGGL((macro_minmax_kernel<FMT, 1>), grid, block, 0, s, pool, pad, runs, base, rows, mm);
  return hipGetLastError();
}

}  // namespace

hipError_t launch_macro_minmax(int fmt, const void *pool, int pad, const MacroRuns &runs, float2 *mm, hipStream_t s) {
  // a launch holds fewer than 2^32 threads on an axis: 256 a page
  constexpr int kPages = 1 << 22;
  // as many y rows a workgroup as its LDS holds, or fewer while that leaves the chip idle
  const int nm = macro_edge(pad), most = std::min(nm, kColumns / pad);
  const int rows = (int64_t)runs.total * nm >= 4096 ? most : std::min(most, std::max(1, 256 / pad));
  for (int base = 0; base < runs.total; base += std::min(kPages, runs.total - base)) {
    const int k = std::min(runs.total - base, kPages);
    const hipError_t e = fmt == HYD_FMT_U8    ? minmax_pages<HYD_FMT_U8>(pool, pad, runs, base, k, rows, mm, s)
                         : fmt == HYD_FMT_F16 ? minmax_pages<HYD_FMT_F16>(pool, pad, runs, base, k, rows, mm, s)
                                              : minmax_pages<HYD_FMT_F32>(pool, pad, runs, base, k, rows, mm, s);
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

hipError_t launch_macro_classes(const float2 *mm, int pad, const MacroRuns &runs, const float *tf, int tf_n, float scale,
                                const float *page_scale, uint8_t *cls, bool replace, unsigned long long *counts,
                                unsigned long long *zero, hipStream_t s) {
  if (runs.total <= 0) return hipSuccess;
  const int nm = macro_edge(pad), tl = (nm + kTileM - 1) / kTileM;
  const int pages = std::max(1, 256 / (nm * nm));   // of one workgroup
  const int groups = nm <= kWholeM ? (runs.total + pages - 1) / pages : runs.total * tl * tl * tl;
  const unsigned grid = (unsigned)std::min(groups, 2048);
  hipLaunchKernelGGL(macro_class_kernel, dim3(grid), dim3(256), 0, s, mm, nm, runs, pages, groups, tf, tf_n, scale,
                     page_scale, cls, replace, counts, zero);
  return hipGetLastError();
}

}  // namespace hyd
