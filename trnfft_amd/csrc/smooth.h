// Transforms whose length is a multiple of 4 with no prime factor above 7 (36 to 640 points): N = N1 * N2 in
// two in-register DFTs with one LDS exchange between them, instead of the two padded transforms of a
// Bluestein chain.
//
// The reference runs Bluestein's chain at these lengths with chirp angles pi k^2 / n rounded to fp32, which
// is what its results differ by from the exact transform: about 1.15e-7 n, growing with n.  The direct
// transform has no such error (1e-7, and is held to 1e-6 log2 n of float64), so it differs from the reference's result by
// the reference's own.  In parts of the parity bound 1e-5 log2 n that is, on random rows, 0.48 at n = 400, 0.67 at 500, 0.75
// at 640, 0.73 to 0.83 from 648 to 720 and past it from 875 on; a tone meets the chirp's worst angles: at most 1.0
// below 256, up to 2.4 at 600 and 640 (2.0 where it is Hann-windowed).  Longer lengths are further off, and the kernels were
// measured and tested up to the 640 points of a camera's row: from there on, and at lengths with other factors, rows follow
// the reference's chain.
#pragma once
#include <initializer_list>
#include <type_traits>

#include "kernels.h"

namespace tfa {

constexpr int kSmoothMin = 36, kSmoothMax = 640;

__host__ __device__ constexpr bool smooth7(int n) {
  for (int p : {2, 3, 5, 7})
    while (n % p == 0) n /= p;
  return n == 1;
}
// N1 <= N2, the most balanced split of n into two register radices (at most 32); 0 if there is none
__host__ __device__ constexpr int smooth_n1(int n) {
  for (int d = 32; d > 1; --d)
    if (n % d == 0 && d * d <= n && n / d <= 32 && smooth7(d) && smooth7(n / d)) return d;
  return 0;
}
__host__ __device__ constexpr bool smooth_len(long long n) {
  return n >= kSmoothMin && n <= kSmoothMax && n % 4 == 0 && (n & (n - 1)) != 0 && smooth7((int)n) &&
         smooth_n1((int)n) != 0 && smooth_n1((int)n / 2) != 0;
}

// x^ = DFT of odd prime length: pairs (a_j, a_{R-j}) as sums and differences
template <int R, int DIR>
struct DftOddPrime {
  __device__ __forceinline__ static void run(float2* a) {
    constexpr int H = R / 2;
    float2 s[H], d[H];
    float2 x0 = a[0];
#pragma unroll
    for (int j = 0; j < H; ++j) {
      s[j] = cadd(a[j + 1], a[R - 1 - j]);
      d[j] = csub(a[j + 1], a[R - 1 - j]);
      x0 = cadd(x0, s[j]);
    }
    out<1>(a, s, d);
    a[0] = x0;
  }
  template <int K>
  __device__ __forceinline__ static void out(float2* a, const float2* s, const float2* d) {
    if constexpr (K <= R / 2) {
      float2 c = a[0], q = make_float2(0.0f, 0.0f);
      term<K, 1>(c, q, s, d);
      const float2 iq = mul_diri<DIR>(q);
      out<K + 1>(a, s, d);
      a[K] = cadd(c, iq);
      a[R - K] = csub(c, iq);
    }
  }
  template <int K, int J>
  __device__ __forceinline__ static void term(float2& c, float2& q, const float2* s, const float2* d) {
    if constexpr (J <= R / 2) {
      constexpr float cs = (float)cos2pi(J * K, R), sn = (float)sin2pi(J * K, R);
      c = make_float2(c.x + cs * s[J - 1].x, c.y + cs * s[J - 1].y);
      q = J == 1 ? cscale(d[0], sn) : make_float2(q.x + sn * d[J - 1].x, q.y + sn * d[J - 1].y);
      term<K, J + 1>(c, q, s, d);
    }
  }
};
template <int DIR> struct Dft<5, DIR> : DftOddPrime<5, DIR> {};
template <int DIR> struct Dft<7, DIR> : DftOddPrime<7, DIR> {};
template <int DIR> struct Dft<9, DIR> : DftSplit<3, 3, DIR> {};
template <int DIR> struct Dft<10, DIR> : DftSplit<2, 5, DIR> {};
template <int DIR> struct Dft<14, DIR> : DftSplit<2, 7, DIR> {};
template <int DIR> struct Dft<15, DIR> : DftSplit<3, 5, DIR> {};
template <int DIR> struct Dft<18, DIR> : DftSplit<2, 9, DIR> {};
template <int DIR> struct Dft<20, DIR> : DftSplit<4, 5, DIR> {};
template <int DIR> struct Dft<21, DIR> : DftSplit<3, 7, DIR> {};
template <int DIR> struct Dft<25, DIR> : DftSplit<5, 5, DIR> {};
template <int DIR> struct Dft<27, DIR> : DftSplit<3, 9, DIR> {};
template <int DIR> struct Dft<28, DIR> : DftSplit<4, 7, DIR> {};
template <int DIR> struct Dft<30, DIR> : DftSplit<5, 6, DIR> {};

// Forward transform of N points, one LDS area of AREA float2 per transform.  Item j2 < N2 of the first pass
// holds x[j2 + N2 j1] (j1 < N1), item k1 < N1 of the second holds X[k1 + N1 k2] (k2 < N2).  The exchange
// has an odd pitch, and so has the area, so that both passes and lanes over several transforms at
// one index meet distinct banks.  (PAD false: a pitch of N2, where that lets another workgroup share the CU; 100-point
// rows are 14 % slower without the padding.)  (The inverse is the forward transform with re and im exchanged in both
// its input and its output.)
template <int N, bool PAD = true>
struct Smooth {
  static constexpr int N1 = smooth_n1(N), N2 = N / N1, PITCH = PAD ? N2 | 1 : N2;
  static constexpr int AREA = (N1 * PITCH > N + 1 ? N1 * PITCH : N + 1) | 1;

  // tw: W_N^(k1 j2) at k1 * N2 + j2
  __device__ __forceinline__ static void first(float2 (&v)[N1], const float2* __restrict__ tw, int j2) {
    Dft<N1, -1>::run(v);
#pragma unroll
    for (int k = 1; k < N1; ++k) v[k] = cmul(v[k], tw[k * N2 + j2]);
  }
  __device__ __forceinline__ static void store(const float2 (&v)[N1], float2* area, int j2) {
#pragma unroll
    for (int k = 0; k < N1; ++k) area[k * PITCH + j2] = v[k];
  }
  __device__ __forceinline__ static void second(float2 (&v)[N2], const float2* area, int k1) {
#pragma unroll
    for (int j = 0; j < N2; ++j) v[j] = area[k1 * PITCH + j];
    Dft<N2, -1>::run(v);
  }
};

// Workgroup of XF transforms of N points: the second pass takes its XF * N1 items in one round, the first
// its XF * N2 in one (N2 < 1.5 N1: a third of the lanes at most idle in the second) or in N2 / N1 rounds.
template <int N, int XF>
struct SmoothGroup {
  using S = Smooth<N>;
  static constexpr int WIDE = 2 * S::N2 < 3 * S::N1 ? S::N2 : S::N1;
  static constexpr int THREADS = (XF * WIDE + 63) / 64 * 64;
  static constexpr int ROUNDS = (XF * S::N2 + THREADS - 1) / THREADS;
};

constexpr int kSmoothLds3 = 53760;  // LDS that lets three workgroups share a CU (160 KB in units of 1280 bytes)
// Padded, unless XF areas of N points, and `more` bytes, let three workgroups share the CU only without padding.  That takes
// 64 x 160000 samples, STFT and inverse, from 43.4 to 37.2 us and 52.9 to 44.2 at n_fft 392, from 42.5 to 40.2 and 56.9 to 54.8 at
// 400.  A pitch that is a multiple of 8 keeps the padding, as its lanes would share banks: at 384 (N2 = 16) the inverse
// takes 45.2 us padded, 53.9 without.
template <int N, int XF>
constexpr bool smooth_pad(int more) {
  return !(XF * Smooth<N, true>::AREA * 8 + more > kSmoothLds3 && XF * Smooth<N, false>::AREA * 8 + more <= kSmoothLds3 &&
           Smooth<N>::N2 % 8 != 0);
}

// The kernels' LDS.  Its size is given at the launch: where the compiler knows that LDS leaves room for few
// waves it rounds the register count up to just that many per SIMD, and a workgroup of 5 waves, which
// puts two of them on the first SIMD each time, then found no room beside another one (the inverse STFT
// at n_fft 400 ran one workgroup per CU instead of two, 88 us against 61).
extern __shared__ float2 smooth_lds[];
constexpr int kSmoothLds = 65536;  // what a launch may ask for as it is

// f(integral_constant<N>) for the smooth length n; false if n is none
template <int N = kSmoothMin, class F>
bool smooth_dispatch(int n, F&& f) {
  if constexpr (N > kSmoothMax) {
    return false;
  } else {
    if constexpr (smooth_len(N)) {
      if (n == N) {
        f(std::integral_constant<int, N>{});
        return true;
      }
    }
    return smooth_dispatch<N + 4>(n, f);
  }
}

}  // namespace tfa
