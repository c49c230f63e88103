// Fused inverse STFT of onesided spectra at smooth n_fft (smooth.h), and the gradient of the forward STFT with
// respect to its padded signal, which has the same form.
//
// A workgroup owns the output samples of FR - halo frames and also transforms the halo = floor((N - 1) / hop)
// frames before them.  Frame by frame: Z_k = (X_k + conj X_{H-k}) + i W_N^-k (X_k - conj X_{H-k}), k < H = N / 2 (the
// imaginary parts of X_0 and X_H do not reach a real frame), the inverse transform of H points, whose
// values are the frame's samples in pairs; then every owned sample sums its frames from LDS.
//
// Bound by the latencies between its barriers, as the forward kernel: 64 x 201 x 1001 bins at n_fft 400, hop 160,
// in 59 us, against 306 for one 1024-point Bluestein chain per frame.  With the bins staged four loads at a
// time and a division per sample 121 us; every load issued before the first store, and a thread keeping one phase of
// the hop with its window values, 88; two workgroups per CU (smooth_lds) 61, three 59.
#include "smooth.h"

namespace tfa {

// Frames per workgroup: above the longest halo that the plan accepts (32 frames up to n_fft 128, else 16), which asks for 64 up
// to 128; 20 is what LDS holds at n_fft 640.  64 signals, 160000 samples, hop 2n/5: n_fft 140 44.6 us with 64 frames and 37.9 with 32,
// 168 40.2 and 38.5; with 32 and with 20, 420 51.8 and 53.0, 432 63.8 and 48.4, 448 50.0 and 46.5.
template <int N>
constexpr int smooth_istft_frames() {
  return N <= 128 ? 64 : N <= 448 ? 32 : 20;
}
template <int N>
using IstftSmooth = Smooth<N / 2, smooth_pad<N / 2, smooth_istft_frames<N>()>(4 * N)>;

template <int N>
__global__ __launch_bounds__((SmoothGroup<N / 2, smooth_istft_frames<N>()>::THREADS)) void istft_smooth_kernel(
    const float* __restrict__ sre, const float* __restrict__ sim, const float* __restrict__ win,
    float* __restrict__ out, const float2* __restrict__ tw, const float2* __restrict__ twn, int n_frames, int hop,
    int halo, int owned, int tiles_per_signal, int expected_len, int start, int write_len, int out_pitch, float scale,
    bool adjoint, bool frames_major) {
  constexpr int H = N / 2, K = H + 1, FR = smooth_istft_frames<N>();
  using G = SmoothGroup<H, FR>;
  using S = IstftSmooth<N>;
  constexpr int N1 = S::N1, N2 = S::N2, AREA = S::AREA, THREADS = G::THREADS;
  float2* const lds = smooth_lds;  // FR * AREA
  float* const wl = reinterpret_cast<float*>(lds + FR * AREA);  // the window, N floats
  const unsigned tile = xcd_tile_remap32(blockIdx.x, gridDim.x);
  const unsigned b = tile / (unsigned)tiles_per_signal;
  const int t0 = (int)(tile - b * (unsigned)tiles_per_signal) * owned;  // first owned frame
  const int ta = t0 - halo > 0 ? t0 - halo : 0;                         // first frame of the tile
  const int nf = (t0 + owned < n_frames ? t0 + owned : n_frames) - ta;  // frames in the tile (<= FR)
  const int t = threadIdx.x;

  for (int i = t; i < N; i += THREADS) wl[i] = win[i];
  // 1. the frames' bins (frames past nf: repeated, not read later), the edge bins without imaginary part;
  //    the adjoint of the onesided transform counts them twice against the others
  const float edge = adjoint ? 2.0f : 1.0f;
  const auto put = [&](int f, int k, float re, float im) {
    const bool e = k == 0 || k == H;
    lds[f * AREA + k] = make_float2(e ? re * edge : re, e ? 0.0f : im);
  };
  if (frames_major) {
    const float* bre = sre + ((size_t)b * n_frames + ta) * K;
    const float* bim = sim + ((size_t)b * n_frames + ta) * K;
    const float rk = 1.0f / (float)K;
    for (int i0 = t; i0 < K * nf; i0 += 4 * THREADS) {
      float sr[4], si[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int i = i0 + u * THREADS, ic = i < K * nf ? i : K * nf - 1;
        sr[u] = bre[ic];
        si[u] = bim[ic];
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int i = i0 + u * THREADS;
        if (i < K * nf) {
          int k;
          const int f = divmod_small(i, K, rk, k);
          put(f, k, sr[u], si[u]);
        }
      }
    }
  } else {
    // every load is issued before the first is stored
    constexpr int KS = THREADS / FR, STEPS = (K + KS - 1) / KS;
    const int f = t % FR, k0 = t / FR, fc = f < nf ? f : nf - 1;
    const size_t sbase = (size_t)b * K * n_frames + ta + fc;
    float sr[STEPS], si[STEPS];
#pragma unroll
    for (int u = 0; u < STEPS; ++u) {
      const int kc = k0 + u * KS < K ? k0 + u * KS : K - 1;
      sr[u] = sre[sbase + (size_t)kc * n_frames];
      si[u] = sim[sbase + (size_t)kc * n_frames];
    }
#pragma unroll
    for (int u = 0; u < STEPS; ++u)
      if (k0 < KS && k0 + u * KS < K) put(f, k0 + u * KS, sr[u], si[u]);
  }
  __syncthreads();
  // 2. the inverse transforms (re and im exchanged around the forward one)
  {
    float2 v[G::ROUNDS][N1];
#pragma unroll
    for (int r = 0; r < G::ROUNDS; ++r) {
      const int i = t + r * THREADS, ic = i < FR * N2 ? i : 0;
      const float2* X = lds + ic / N2 * AREA;
#pragma unroll
      for (int e = 0; e < N1; ++e) {
        const int k = ic % N2 + N2 * e;
        const float2 a = X[k], c = X[H - k], w = twn[k];
        const float2 s = make_float2(a.x + c.x, a.y - c.y), d = make_float2(a.x - c.x, a.y + c.y);
        // i W^-k d = (d.x w.y' ...) with W^-k = conj w
        const float2 q = make_float2(d.x * w.x + d.y * w.y, d.y * w.x - d.x * w.y);
        v[r][e] = make_float2(s.y + q.x, s.x - q.y);
      }
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < G::ROUNDS; ++r) {
      const int i = t + r * THREADS;
      if ((r + 1) * THREADS > FR * N2 && i >= FR * N2) break;
      S::first(v[r], tw, i % N2);
      S::store(v[r], lds + i / N2 * AREA, i % N2);
    }
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
      for (int k = 0; k < N2; ++k) lds[fl * AREA + k1 + N1 * k] = make_float2(v[k].y * scale, v[k].x * scale);
    }
  }
  __syncthreads();
  // 3. owned samples [t0 * hop, (t0 + owned) * hop), the last tile up to the end of the signal; each sums
  //    its covering frames t, t - 1, ... (offsets s - t * hop < N)
  const float* y = reinterpret_cast<const float*>(lds);
  const long long s_end = (long long)(t0 + owned) * hop;
  const int s_hi = (t0 + owned >= n_frames || s_end > expected_len) ? expected_len : (int)s_end;
  float* dst = out + (size_t)b * out_pitch;
  const int t_end = ta + nf - 1;
  const auto sample = [&](int fr, int j) {  // sample fr * hop + j, frames from fr down to ta
    float acc = 0.0f, raw = 0.0f, env = 0.0f;
    for (; fr >= ta && j < N; --fr, j += hop) {
      const float v = y[(fr - ta) * (2 * AREA) + j], w = wl[j];
      acc += v * w;
      raw += v;
      env += w * w;
    }
    return adjoint ? acc : env > 1e-8f ? acc / env : raw;
  };
  constexpr int TAPS = 4;
  if (halo < TAPS && hop <= THREADS) {
    // a thread keeps one phase j = s mod hop, its window values and the reciprocal of their envelope,
    // for every G-th frame; samples that fewer frames cover take the general form
    const int G = THREADS / hop, g = t / hop, j = t - g * hop;
    if (g < G) {
      float w[TAPS], env = 0.0f;
#pragma unroll
      for (int m = 0; m < TAPS; ++m) {
        w[m] = j + m * hop < N ? wl[j + m * hop] : 0.0f;
        env += w[m] * w[m];
      }
      const bool plain = j < N && (adjoint || env > 1e-8f);
      const float inv = adjoint ? 1.0f : 1.0f / env;
      int off[TAPS];  // tap m's sample relative to the frame's first (a tap past the window reads sample j)
#pragma unroll
      for (int m = 0; m < TAPS; ++m) off[m] = j + m * hop < N ? j + m * hop - m * 2 * AREA : j < N ? j : 0;
      for (int fr = t0 + g; (long long)fr * hop < s_hi; fr += G) {
        const int s = fr * hop + j, o = s - start;
        if (s >= s_hi || o < 0 || o >= write_len) continue;
        if (plain && fr >= halo && fr <= t_end) {
          const float* f = y + (fr - ta) * (2 * AREA);
          float acc = 0.0f;
#pragma unroll
          for (int m = 0; m < TAPS; ++m) acc += f[off[m]] * w[m];
          dst[o] = acc * inv;
        } else {
          const int last = fr < t_end ? fr : t_end;
          dst[o] = sample(last, s - last * hop);
        }
      }
    }
  } else {
    for (int s = t0 * hop + t; s < s_hi; s += THREADS) {
      const int o = s - start;
      if (o < 0 || o >= write_len) continue;
      int fr = (int)((unsigned)s / (unsigned)hop);
      if (fr > t_end) fr = t_end;
      dst[o] = sample(fr, s - fr * hop);
    }
  }
  // samples past the end of the signal up to the requested length are zero
  if (t0 + owned >= n_frames)
    for (int o = write_len + t; o < out_pitch; o += THREADS) dst[o] = 0.0f;
}

hipError_t launch_istft_smooth(int n_fft, const IstftArgs& a) {
  hipError_t e = hipErrorInvalidValue;
  smooth_dispatch(n_fft, [&](auto n) {
    constexpr int N = decltype(n)::value, FR = smooth_istft_frames<N>();
    constexpr unsigned LDS = (FR * IstftSmooth<N>::AREA + N / 2) * 8;
    static_assert(LDS <= kSmoothLds, "frame tile exceeds LDS");
    const int owned = FR - a.halo;
    if (a.halo < 0 || a.hop < 1 || owned < 1) return;
    const int tiles = (a.n_frames + owned - 1) / owned;
    const long long blocks = a.batch * (long long)tiles;
    if (blocks > 0x7fffffffLL) return;
    hipLaunchKernelGGL((istft_smooth_kernel<N>), dim3((unsigned)blocks), dim3(SmoothGroup<N / 2, FR>::THREADS), LDS,
                       a.stream, a.spec_re, a.spec_im, a.window, a.out, a.tw, a.twn, a.n_frames, a.hop, a.halo, owned,
                       tiles, (int)a.expected_len, (int)a.start, (int)a.write_len, (int)a.out_pitch, a.scale,
                       a.adjoint, a.frames_major);
    e = hipGetLastError();
  });
  return e;
}

}  // namespace tfa
