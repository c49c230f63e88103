// Fused STFT of n_fft points, n_fft a smooth length (smooth.h): framing, reflect padding, window, transform
// and the (bins, frames) transpose in one pass over memory.
//
// A real frame of N samples is one complex transform of H = N / 2 points z_j = x_2j + i x_2j+1; bin k is
// (Z_k + conj Z_{H-k}) / 2 - i W_N^k (Z_k - conj Z_{H-k}) / 2.  (Two frames in one transform would save nothing
// here and let a non-finite sample reach a frame that does not hold it.)
//
// Bound by the latencies between its four barriers, at two or three workgroups per CU, and by the bin rows' partial
// lines: 64 x 160000 at n_fft 400, hop 160 (144 MB) in 51 us, against 148 for one 768-point Bluestein chain
// per frame.  Samples read from memory frame by frame instead of as the tile's span, with the window and the
// twiddles read again in each round, kept the L1 busy (28.0 M accesses for 1.35 M memory instructions): 75 us.
#include "smooth.h"

namespace tfa {

// Frames per workgroup: their bins leave in runs of that many floats (20 and 26, which would let another
// workgroup share the CU, took 12 to 20 % longer than 16).  Calls of few frames take a quarter, so that four times the
// workgroups share the work of a tile: 1 x 16000 at n_fft 400, hop 400, 14.7 -> 8.7 us.
// 64 x 160000 samples, hop 2n/5: n_fft 100 30.1 us with 64 frames and 31.3 with 32, 120 34.9 and 31.3, 140 38.3 and 31.9, 168 34.9 and
// 32.4; with 32 and with 16, 448 39.8 and 34.0, 480 38.9 and 34.8, 500 56.2 and 44.8.  (So 32 from 108 and 16 from 420 on are faster on
// large calls, by 3 to 25 %; calls of 1 to 32 signals are up to 19 % slower with them, and the lines stand between.)
template <int N>
constexpr int smooth_stft_frames() {
  return N <= 128 ? 64 : N <= 448 ? 32 : 16;
}
// (n_fft 400: three workgroups per CU instead of two, 59 -> 51 us)
template <int N, int FR>
using StftSmooth = Smooth<N / 2, smooth_pad<N / 2, FR>(0)>;

template <int N, int FR>
__global__ __launch_bounds__((SmoothGroup<N / 2, FR>::THREADS)) void stft_smooth_kernel(
    const float* __restrict__ sig, const float* __restrict__ win, float* __restrict__ out_re,
    float* __restrict__ out_im, const float2* __restrict__ tw, const float2* __restrict__ twn, int length, int hop,
    int pad, int n_frames, int n_bins, int tiles_per_signal, float scale, bool frames_major) {
  constexpr int H = N / 2;
  using G = SmoothGroup<H, FR>;
  using S = StftSmooth<N, FR>;
  constexpr int N1 = S::N1, N2 = S::N2, AREA = S::AREA, THREADS = G::THREADS;
  float2* const lds = smooth_lds;  // FR * AREA
  const unsigned tile = xcd_tile_remap32(blockIdx.x, gridDim.x);
  const unsigned b = tile / (unsigned)tiles_per_signal;
  const int f0 = (int)(tile - b * (unsigned)tiles_per_signal) * FR;
  const int t = threadIdx.x;
  const float* x = sig + (size_t)b * length;
  const int nfr = n_frames - f0 < FR ? n_frames - f0 : FR;
  // block-uniform: no padding anywhere in the tile's span (64-bit: a long hop)
  const long long s0 = (long long)f0 * hop - pad, span = (long long)(nfr - 1) * hop + N;
  const bool interior = s0 >= 0 && s0 + span <= length;
  const auto reflected = [&](long long idx) {
    // without repeating the edge sample (torch.nn.functional.pad mode="reflect")
    idx = idx < 0 ? -idx : idx;
    idx = idx >= length ? 2LL * (length - 1) - idx : idx;
    return (int)(idx < 0 ? 0 : (idx >= length ? length - 1 : idx));
  };

  // the tile's samples, as one run of the signal where the frames' areas hold it (frames overlap: each
  // sample is read once); frames past the last one repeat it, and are not stored
  float2 v[G::ROUNDS][N1];
  constexpr int SPAN = 2 * FR * AREA;
  if (span <= SPAN) {
    float* const y = reinterpret_cast<float*>(lds);
    const int len = (int)span;
    if (interior) {
      // four loads of four samples in flight per thread (the last one ends with the span)
      for (int i0 = 4 * t; i0 < len; i0 += 16 * THREADS) {
        Quad q[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const int i = i0 + 4 * u * THREADS;
          q[u] = ld_quad(x + s0 + (i < len - 4 ? i : len - 4));
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const int i = i0 + 4 * u * THREADS;
          if (i < len) st_quad(y + (i < len - 4 ? i : len - 4), q[u]);
        }
      }
    } else {
      for (int i0 = t; i0 < len; i0 += 8 * THREADS) {
        float q[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
          const int i = i0 + u * THREADS;
          q[u] = x[reflected(s0 + (i < len ? i : len - 1))];
        }
#pragma unroll
        for (int u = 0; u < 8; ++u)
          if (i0 + u * THREADS < len) y[i0 + u * THREADS] = q[u];
      }
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < G::ROUNDS; ++r) {
      const int i = t + r * THREADS, fl = i / N2 < nfr ? i / N2 : nfr - 1;
      const float* p = y + fl * hop + 2 * (i % N2);
#pragma unroll
      for (int e = 0; e < N1; ++e) v[r][e] = make_float2(p[2 * N2 * e], p[2 * N2 * e + 1]);
    }
    __syncthreads();
  } else {
#pragma unroll
    for (int r = 0; r < G::ROUNDS; ++r) {
      const int i = t + r * THREADS, fl = i / N2 < nfr ? i / N2 : nfr - 1;
      const long long p = s0 + (long long)fl * hop + 2 * (i % N2);
#pragma unroll
      for (int e = 0; e < N1; ++e) v[r][e] = make_float2(x[reflected(p + 2 * N2 * e)], x[reflected(p + 2 * N2 * e + 1)]);
    }
  }
  // window and exchange twiddles, once per thread where all its rounds have the same j2
  constexpr bool SAME = THREADS % N2 == 0;
  float2 w[N1], q[N1];
#pragma unroll
  for (int r = 0; r < G::ROUNDS; ++r) {
    const int i = t + r * THREADS;
    if ((r + 1) * THREADS > FR * N2 && i >= FR * N2) break;
    const int j2 = SAME ? t % N2 : i % N2;
    if (r == 0 || !SAME) {
#pragma unroll
      for (int e = 0; e < N1; ++e) {
        w[e] = ld_pair(win + 2 * (j2 + N2 * e));
        q[e] = tw[e * N2 + j2];
      }
    }
#pragma unroll
    for (int e = 0; e < N1; ++e) v[r][e] = make_float2(v[r][e].x * w[e].x, v[r][e].y * w[e].y);
    Dft<N1, -1>::run(v[r]);
#pragma unroll
    for (int e = 1; e < N1; ++e) v[r][e] = cmul(v[r][e], q[e]);
    S::store(v[r], lds + i / N2 * AREA, j2);
  }
  __syncthreads();
  {
    const bool on = t < FR * N1;
    const int fl = on ? t / N1 : 0, k1 = t % N1;
    float2 v[N2];
    S::second(v, lds + fl * AREA, k1);
    __syncthreads();
    if (on) {
#pragma unroll
      for (int k = 0; k < N2; ++k) lds[fl * AREA + k1 + N1 * k] = v[k];
    }
  }
  __syncthreads();

  const float hs = 0.5f * scale;
  // bins k and H - k: (s + W^k d) / 2 and conj(s - W^k d) / 2
  const auto two_bins = [&](const float2* Z, int k, float2 w, float2& lo, float2& hi) {
    const float2 a = Z[k], c = Z[k > 0 ? H - k : 0];
    const float2 s = make_float2((a.x + c.x) * hs, (a.y - c.y) * hs);
    const float2 d = cmul(make_float2((a.y + c.y) * hs, (c.x - a.x) * hs), w);
    lo = cadd(s, d);
    hi = make_float2(s.x - d.x, d.y - s.y);
  };
  if (frames_major) {
    // (batch, n_frames, n_bins): the tile is one contiguous run per plane
    const size_t ob = ((size_t)b * n_frames + f0) * n_bins;
    float* cre = out_re + ob;
    float* cim = out_im + ob;
    const float rb = 1.0f / (float)n_bins;
    // lanes start early by the run's misalignment to a 128-byte line, so that full-wave stores cover
    // whole lines (non-temporal stores of partial lines each reach HBM)
    const int sh = (int)((reinterpret_cast<uintptr_t>(cre) >> 2) & 31);
    for (int i = t - sh; i < nfr * n_bins; i += THREADS) {
      if (i < 0) continue;
      int k;
      const int fl = divmod_small(i, n_bins, rb, k);
      const int m = k <= H ? k : N - k;  // two-sided: X_k = conj X_{N-k}
      const int q = m <= H / 2 ? m : H - m;
      float2 lo, hi;
      two_bins(lds + fl * AREA, q, twn[q], lo, hi);
      const float2 y = q == m ? lo : hi;
      st_stream(cre + i, y.x);
      st_stream(cim + i, k <= H ? y.y : -y.y);
    }
    return;
  }
  constexpr int KS = THREADS / FR, KN = H / 2 + 1;  // bin pairs per step, of KN
  const int fr = t % FR;
  if (f0 + fr >= n_frames || t >= KS * FR) return;
  const float2* Z = lds + fr * AREA;
  // 32-bit offsets from the signal's (uniform) base: the host keeps n_bins * n_frames within 2^30
  const size_t ob = (size_t)b * n_bins * n_frames + f0;
  float* ore = out_re + ob;
  float* oim = out_im + ob;
  const bool two_sided = n_bins == N;
  const auto put = [&](int k, float2 y) {
    const unsigned off = (unsigned)(fr + k * n_frames);
    ore[off] = y.x;
    oim[off] = y.y;
    if (two_sided && k > 0 && k < H) {
      const unsigned off2 = (unsigned)(fr + (N - k) * n_frames);
      ore[off2] = y.x;
      oim[off2] = -y.y;
    }
  };
  constexpr int U = 4;
  for (int k0 = t / FR; k0 < KN; k0 += U * KS) {
    float2 w[U];
#pragma unroll
    for (int u = 0; u < U; ++u) w[u] = twn[k0 + u * KS < KN ? k0 + u * KS : 0];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int k = k0 + u * KS;
      if (k >= KN) break;
      float2 lo, hi;
      two_bins(Z, k, w[u], lo, hi);
      put(k, lo);
      if (2 * k != H) put(H - k, hi);
    }
  }
}

template <int N, int FR>
static hipError_t launch_stft_tiles(const StftArgs& a) {
  constexpr unsigned LDS = FR * StftSmooth<N, FR>::AREA * 8;
  static_assert(LDS <= kSmoothLds, "frame tile exceeds LDS");
  const int tiles = (a.n_frames + FR - 1) / FR;
  const long long blocks = a.batch * (long long)tiles;
  if (blocks > 0x7fffffffLL || a.n_bins > N) return hipErrorInvalidValue;
  hipLaunchKernelGGL((stft_smooth_kernel<N, FR>), dim3((unsigned)blocks), dim3(SmoothGroup<N / 2, FR>::THREADS), LDS,
                     a.stream, a.signal, a.window, a.out_re, a.out_im, a.tw, a.twn, a.length, a.hop, a.pad,
                     a.n_frames, a.n_bins, tiles, a.scale, a.frames_major);
  return hipGetLastError();
}

hipError_t launch_stft_smooth(int n_fft, const StftArgs& a) {
  hipError_t e = hipErrorInvalidValue;
  smooth_dispatch(n_fft, [&](auto n) {
    constexpr int N = decltype(n)::value, FR = smooth_stft_frames<N>();
    e = a.batch * (long long)((a.n_frames + FR - 1) / FR) >= kNumCUs ? launch_stft_tiles<N, FR>(a)
                                                                    : launch_stft_tiles<N, FR / 4>(a);
  });
  return e;
}

}  // namespace tfa
