// Batched c2c rows and strided axes of smooth lengths (smooth.h), one pass over memory.
// Bound by HBM with what the barriers leave uncovered: 7680 rows of 640 (79 MB) in 23 us (46 as a 1536-point
// Bluestein chain), 16 x 480 x 640 down the 480 axis in 19 us (54 at 1024 points), 3.4 and 4.1 TB/s.  The strided
// axis at the 16-column runs of 64 bytes that let two workgroups share a CU.
// The inverse exchanges the planes: its re is the forward transform's im, of (im, re).
#include "smooth.h"

namespace tfa {

// Rows per workgroup: as many (a power of two) as let three workgroups share a CU's LDS.
template <int N>
constexpr int smooth_rows() {
  int r = 256;
  while (r * Smooth<N>::N1 > 1024 || 3 * r * Smooth<N>::AREA * 8 > kLdsBytes - 4096) r /= 2;
  return r;
}

// Rows enter and leave as the workgroup's contiguous run of each plane, four floats per lane (n is a
// multiple of 4, so a group of four lies in one row).
template <int N, int XF>
__global__ __launch_bounds__((SmoothGroup<N, XF>::THREADS)) void smooth_rows_kernel(
    const float* in_re, const float* in_im, float* out_re, float* out_im, const float2* __restrict__ tw,
    long long batch, float scale) {
  using G = SmoothGroup<N, XF>;
  using S = Smooth<N>;
  constexpr int N1 = S::N1, N2 = S::N2, AREA = S::AREA, THREADS = G::THREADS;
  float2* const lds = smooth_lds;  // XF * AREA
  const long long r0 = (long long)blockIdx.x * XF;
  const int rows = batch - r0 < XF ? (int)(batch - r0) : XF;
  const size_t base = (size_t)r0 * N;
  const int t = threadIdx.x;
  constexpr int QUADS = XF * N / 4, STEPS = (QUADS + THREADS - 1) / THREADS;
  {
    const int quads = rows * (N / 4);
    Quad re[STEPS], im[STEPS];
    // (past the last row: the last quad again, not stored)
#pragma unroll
    for (int u = 0; u < STEPS; ++u) {
      const int q = t + u * THREADS, qc = q < quads ? q : quads - 1;
      const Quad zero = {0.0f, 0.0f, 0.0f, 0.0f};
      re[u] = in_re ? ld_quad(in_re + base + 4 * qc) : zero;
      im[u] = in_im ? ld_quad(in_im + base + 4 * qc) : zero;
    }
#pragma unroll
    for (int u = 0; u < STEPS; ++u) {
      const int q = t + u * THREADS;
      if (q < QUADS) {
        float2* d = lds + q / (N / 4) * AREA + q % (N / 4) * 4;
        d[0] = make_float2(re[u].x, im[u].x);
        d[1] = make_float2(re[u].y, im[u].y);
        d[2] = make_float2(re[u].z, im[u].z);
        d[3] = make_float2(re[u].w, im[u].w);
      }
    }
  }
  __syncthreads();
  {
    float2 v[G::ROUNDS][N1];
#pragma unroll
    for (int r = 0; r < G::ROUNDS; ++r) {
      const int i = t + r * THREADS, ic = i < XF * N2 ? i : 0;
      const float2* x = lds + ic / N2 * AREA + ic % N2;
#pragma unroll
      for (int e = 0; e < N1; ++e) v[r][e] = x[N2 * e];
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < G::ROUNDS; ++r) {
      const int i = t + r * THREADS;
      if ((r + 1) * THREADS > XF * N2 && i >= XF * N2) break;
      S::first(v[r], tw, i % N2);
      S::store(v[r], lds + i / N2 * AREA, i % N2);
    }
  }
  __syncthreads();
  {
    const bool on = t < XF * N1;
    const int xf = on ? t / N1 : 0, k1 = t % N1;
    float2 v[N2];
    S::second(v, lds + xf * AREA, k1);
    __syncthreads();
    if (on) {
#pragma unroll
      for (int k = 0; k < N2; ++k) lds[xf * AREA + k1 + N1 * k] = v[k];
    }
  }
  __syncthreads();
  for (int q = t; q < rows * (N / 4); q += THREADS) {
    const float2* s = lds + q / (N / 4) * AREA + q % (N / 4) * 4;
    const float2 a = s[0], b = s[1], c = s[2], d = s[3];
    st_quad(out_re + base + 4 * q, {a.x * scale, b.x * scale, c.x * scale, d.x * scale});
    st_quad(out_im + base + 4 * q, {a.y * scale, b.y * scale, c.y * scale, d.y * scale});
  }
}

// Columns of x viewed as (outer, N, stride): CT consecutive columns per workgroup, lanes over the columns, so
// every access to memory is a run of CT floats and the exchange [element][column] meets all banks.
constexpr int kSmoothCols = 16;

// (beyond kSmoothLds the array is the kernel's own, and the workgroup's waves spread evenly over the SIMDs)
template <int N>
struct SmoothCols {
  static constexpr bool DYN = N * kSmoothCols * 8 <= kSmoothLds;
  static constexpr int ROUND = DYN ? 64 : 256;
  static constexpr int THREADS = (kSmoothCols * Smooth<N>::N2 + ROUND - 1) / ROUND * ROUND;
};

template <int N>
__global__ __launch_bounds__((SmoothCols<N>::THREADS)) void smooth_strided_kernel(
    const float* in_re, const float* in_im, float* out_re, float* out_im, const float2* __restrict__ tw,
    long long stride, long long col_tiles, float scale) {
  using S = Smooth<N>;
  constexpr int CT = kSmoothCols, N1 = S::N1, N2 = S::N2;
  __shared__ float2 own[SmoothCols<N>::DYN ? 1 : N * CT];
  float2* const lds = SmoothCols<N>::DYN ? smooth_lds : own;
  const long long tile = xcd_tile_remap(blockIdx.x, gridDim.x);
  const long long o = tile / col_tiles;
  const long long c0 = (tile - o * col_tiles) * CT;
  const int c = threadIdx.x % CT, j = threadIdx.x / CT;
  const bool in_cols = c0 + c < stride;
  const size_t base = (size_t)o * N * stride + (size_t)(in_cols ? c0 + c : stride - 1);  // (past the end: repeated)
  if (j < N2) {
    float2 v[N1];
#pragma unroll
    for (int e = 0; e < N1; ++e) {
      const size_t i = base + (size_t)(j + N2 * e) * stride;
      v[e] = make_float2(in_re ? in_re[i] : 0.0f, in_im ? in_im[i] : 0.0f);
    }
    S::first(v, tw, j);
#pragma unroll
    for (int k = 0; k < N1; ++k) lds[(k * N2 + j) * CT + c] = v[k];
  }
  __syncthreads();
  if (j < N1) {
    float2 v[N2];
#pragma unroll
    for (int e = 0; e < N2; ++e) v[e] = lds[(j * N2 + e) * CT + c];
    Dft<N2, -1>::run(v);
    if (in_cols) {
#pragma unroll
      for (int k = 0; k < N2; ++k) {
        const size_t i = base + (size_t)(j + N1 * k) * stride;
        out_re[i] = v[k].x * scale;
        out_im[i] = v[k].y * scale;
      }
    }
  }
}

template <int N, int XF>
static hipError_t launch_rows(const SmoothArgs& a) {
  const long long blocks = (a.outer + XF - 1) / XF;
  if (blocks > 0x7fffffffLL) return hipErrorInvalidValue;
  constexpr unsigned LDS = XF * Smooth<N>::AREA * 8;
  static_assert(LDS <= kSmoothLds, "rows exceed LDS");
  hipLaunchKernelGGL((smooth_rows_kernel<N, XF>), dim3((unsigned)blocks), dim3(SmoothGroup<N, XF>::THREADS), LDS,
                     a.stream, a.inverse ? a.in_im : a.in_re, a.inverse ? a.in_re : a.in_im,
                     a.inverse ? a.out_im : a.out_re, a.inverse ? a.out_re : a.out_im, a.tw, a.outer, a.scale);
  return hipGetLastError();
}

hipError_t launch_smooth_rows(int n, const SmoothArgs& a) {
  hipError_t err = hipErrorInvalidValue;
  smooth_dispatch(n, [&](auto nn) {
    constexpr int N = decltype(nn)::value, XF = smooth_rows<N>();
    // a quarter of the rows per workgroup while that leaves CUs without one
    err = a.outer > (long long)XF * kNumCUs ? launch_rows<N, XF>(a) : launch_rows<N, XF / 4>(a);
  });
  return err;
}

hipError_t launch_smooth_strided(int n, const SmoothArgs& a) {
  hipError_t err = hipErrorInvalidValue;
  smooth_dispatch(n, [&](auto nn) {
    constexpr int N = decltype(nn)::value;
    const long long col_tiles = (a.stride + kSmoothCols - 1) / kSmoothCols, blocks = a.outer * col_tiles;
    if (blocks > 0x7fffffffLL) return;
    hipLaunchKernelGGL((smooth_strided_kernel<N>), dim3((unsigned)blocks),
                       dim3(SmoothCols<N>::THREADS), SmoothCols<N>::DYN ? N * kSmoothCols * 8 : 0, a.stream,
                       a.inverse ? a.in_im : a.in_re, a.inverse ? a.in_re : a.in_im,
                       a.inverse ? a.out_im : a.out_re, a.inverse ? a.out_re : a.out_im, a.tw, a.stride, col_tiles,
                       a.scale);
    err = hipGetLastError();
  });
  return err;
}

}  // namespace tfa
