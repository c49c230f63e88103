// Complex GEMM on the bf16 matrix cores at fp32 precision (v_mfma_f32_32x32x16_bf16), split re/im planes.
//
//   C = alpha * (op(A) @ op(B)) + bias,  op(X) = X, X^T, conj(X)^T or conj(X)
//   C_re = A_re B_re - A_im B_im,  C_im = A_re B_im + A_im B_re   (on the op'ed operands)
//
// Every fp32 operand is the exact sum of three bf16 pieces of 8 significant bits each, every one rounded to
// nearest (x1 = bf16(x), x2 = bf16(x - x1), x3 = x - x1 - x2; Henry, Tang and Heinecke, "Leveraging the bfloat16
// Artificial Intelligence Datatype For Higher-Precision Computations", ARITH 2019), so a product a b is the sum
// of nine bf16 products, each exact in fp32.  Six of them (a1 b1, a1 b2, a2 b1, a2 b2, a1 b3, a3 b1) run on the
// matrix cores into fp32 accumulators.  x2 is at most 2^-8 and x3 2^-16 of the power of two below |x|, so the other
// three are at most 2^-23 of a b together, 5.7e-9 in the mean square and of either sign.  (Pieces cut by truncation lost up
// to 4.7e-7, always towards zero.)
// Against 64 bits (random normal operands, relative 2-norm) that is closer than fp32 products were: 1.1e-7
// against 8.1e-7 at K = 1024, 5.4e-8 against 1.46e-7 at K = 33, and without their drift where the operands have one
// sign: 6.0e-8 against 5.9e-7 at K = 1024.  Where a sum is one product (a diagonal matrix times another) the
// instruction's own rounding shows: 3.2e-8, at most 1.4e-7, against 2.6e-8 and 6e-8.
// The matrix rate is what pays for it: 8192 x
// 1024 x 1024 takes 313 to 328 us back to back (512 with v_mfma_f32_32x32x2f32 at 85 % of its peak), 412 GF of bf16
// products at 1.26 to 1.32 PF; the matrix cores are busy 67 to 68 % of the cycles, at 1.66 to 1.83 GHz by card
// (rocprofv3; spread thinner, 52 % busy, it clocked 1.95 GHz and took 390 us against 348), probably the power limit.
//
// One kernel computes all four real products: each k-step loads the fragments of the three pieces of
// A_re/A_im and B_re/B_im once from LDS for 24 MFMAs per 32 x 32 tile of the two accumulator sets (the
// NKI kernel's "stationary reuse" idea, trnfft/nki/dispatch.py:121-200 and :267-345, in CDNA4 form).
// Workgroup tile 128 x 128 (per plane), 8 waves of 64 x 32, 16 k per stage, two stages in LDS (one
// barrier per stage): while one stage is multiplied the next is split and stored, and the one after
// it is on its way from memory in registers.  The splitting, and the fp32 additions of the stage before, are
// pinned behind the MFMA pairs that hide them (splitting before or after the MFMAs by wave: 1109 to 1190 us
// for the linear layer's three products, 1030 pinned).
#include <algorithm>
#include <utility>

#include "kernels.h"

namespace tfa {

typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

constexpr int GBM = 128, GBN = 128, GBK = 16;
constexpr int kThreads = 512;
typedef floatx16 Acc[2];  // a wave's 64 x 32 sums of one plane

// A stage of one operand is 128 rows x 16 k x 2 planes: a thread holds eight k (half) of one row of one plane.
//   k contiguous in memory (plain A, transposed B): lanes 2r and 2r + 1 hold the halves of row r,
//   so a row's 64 bytes are one run;
//   rows contiguous (transposed A, plain B): lanes run over the rows, a wave's load instruction
//   covers 64 consecutive floats of one k.
template <bool KMAJOR>
struct Slot {
  int plane, row, half;
  __device__ __forceinline__ Slot(int t, int w) {  // w: the wave (uniform)
    plane = w >> 2;
    row = KMAJOR ? (t & 255) >> 1 : t & 127;
    half = KMAJOR ? t & 1 : (w >> 1) & 1;
  }
};

// One operand's tile: 128 rows from row0, k below K.  Rows past the last one repeat it: what they add
// to is not stored.
template <bool KMAJOR>
struct Operand {
  const float* P;  // this thread's plane, at its row (k contiguous) or the tile's first row
  long long ld;
  int K, col;  // rows contiguous: this thread's row in the tile
  Slot<KMAJOR> q;

  __device__ __forceinline__ Operand(const float* re, const float* im, long long ld_, int rows, int K_, int row0,
                                     int t, int w)
      : ld(ld_), K(K_), q(t, w) {
    const int left = rows - 1 - row0;
    col = q.row < left ? q.row : left;
    P = (q.plane ? im : re) + (KMAJOR ? (size_t)(row0 + col) * ld : (size_t)row0);
  }
  // a whole stage: k0 + GBK <= K
  __device__ __forceinline__ void load(int k0, float (&x)[8]) const {
    const int kq = k0 + q.half * 8;
    if constexpr (KMAJOR) {
      const Quad a = ld_quad(P + kq), b = ld_quad(P + kq + 4);
      x[0] = a.x; x[1] = a.y; x[2] = a.z; x[3] = a.w;
      x[4] = b.x; x[5] = b.y; x[6] = b.z; x[7] = b.w;
    } else {
      const float* p = P + (size_t)kq * ld;
#pragma unroll
      for (int c = 0; c < 8; ++c) x[c] = (p + c * ld)[col];
    }
  }
  // the last, partial stage: k at or past K reads as zero
  __device__ __forceinline__ void load_tail(int k0, float (&x)[8]) const {
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      const int k = k0 + q.half * 8 + c, kc = k < K ? k : K - 1;
      x[c] = KMAJOR ? P[kc] : P[(size_t)kc * ld + col];
    }
#pragma unroll
    for (int c = 0; c < 8; ++c)
      if (k0 + q.half * 8 + c >= K) x[c] = 0.0f;
  }
};

// LDS of the pieces: per operand and plane three blocks, each two halves of the stage's 16 k, a half
// 128 rows of 8 k (16 bytes).  An MFMA fragment (lane l: row l % 32, half l / 32) is then one ds_read_b128
// over two contiguous runs; the 64 bytes between the halves keep the k-contiguous stores (lanes alternate
// between the halves) off each other's banks.
constexpr int kHalf = GBM * 16 + 64;  // bytes
constexpr int kPiece = 2 * kHalf;
constexpr int kPlane = 3 * kPiece;
constexpr int kOperand = 2 * kPlane;
constexpr int kStage = 2 * kOperand;
static_assert(GBM == GBN, "both operands are staged alike");

// Eight k of one row, split into their three pieces in four steps of two k.
struct Split {
  unsigned p[3][4];
  template <int C>
  __device__ __forceinline__ void step(const float (&x)[8]) {
    floatx2 r = {x[2 * C], x[2 * C + 1]};
#pragma unroll
    for (int q = 0; q < 3; ++q) {
      // both rounded to nearest, in one register
      const unsigned u = __builtin_bit_cast(unsigned, __builtin_convertvector(r, bf16x2));
      p[q][C] = u;
      r[0] -= __uint_as_float(u << 16);
      r[1] -= __uint_as_float(u & 0xffff0000u);
    }
  }
  __device__ __forceinline__ void store(char* dst) const {
#pragma unroll
    for (int q = 0; q < 3; ++q)
      *reinterpret_cast<uint4*>(dst + q * kPiece) = make_uint4(p[q][0], p[q][1], p[q][2], p[q][3]);
  }
};

// bf16 ends at 2^-133, so operands below 2^-110 lose bits as pieces (operands of 1e-36 lost 5e-5 of the result); the
// matrix instructions keep denormals.  The loss is at most 2^-133 max(|a|, |b|) for each of the 2 K real products of a
// sum, or some 2^-149 each where the products are below 2^-118, so it shows only in sums that are near that.
// Each thread keeps the least nonzero and the largest magnitude of either operand that it splits.  Where one is below
// kSmall (without one, products are at least 2^-96) the workgroup compares them: if an operand is below kExact
// or a product may be below kSumFloor, and a sum (0 counts) is below K max(2^-108 |a|, 2^-108 |b|, 2^-118), it
// takes fp32 products; what the others lost is below 2^-24 of the sum.
constexpr float kSmall = 0x1p-48f, kExact = 0x1p-110f;
constexpr float kSumLimit = 0x1p-108f, kSumFloor = 0x1p-118f;
struct Range {
  unsigned lo = ~0u;  // least of 2 bits(|x|) - 1 (zero wraps to the largest)
  float hi = 0.0f;
  template <int C>
  __device__ __forceinline__ void pair(const float (&x)[8]) {
    const unsigned u = 2 * __float_as_uint(x[2 * C]) - 1, v = 2 * __float_as_uint(x[2 * C + 1]) - 1;
    lo = min(min(lo, u), v);
    hi = fmaxf(fmaxf(hi, fabsf(x[2 * C])), fabsf(x[2 * C + 1]));
  }
  __device__ __forceinline__ bool small() const { return lo < 2 * __float_as_uint(kSmall) - 1; }
  // over the workgroup's waves, through 2 * kThreads / 64 words of LDS
  __device__ __forceinline__ void reduce(unsigned* lds, int w) {
#pragma unroll
    for (int d = 32; d > 0; d /= 2) {
      lo = min(lo, (unsigned)__shfl_xor((int)lo, d));
      hi = fmaxf(hi, __shfl_xor(hi, d));
    }
    if ((threadIdx.x & 63) == 0) {
      lds[2 * w] = lo;
      lds[2 * w + 1] = __float_as_uint(hi);
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kThreads / 64; ++i) {
      lo = min(lo, lds[2 * i]);
      hi = fmaxf(hi, __uint_as_float(lds[2 * i + 1]));
    }
  }
  // the least nonzero magnitude (infinity where there is none)
  __device__ __forceinline__ float least() const { return lo == ~0u ? INFINITY : __uint_as_float((lo + 1) / 2); }
};

__device__ __forceinline__ int outside(float x, float limit) {
  const float m = fabsf(x);
  return m < INFINITY && m >= limit ? 0 : 1;
}

// a b + c d over one stage's 16 k, from zero and smallest products first: each instruction rounds its
// sum, and only the last two products meet a sum of full size here.  (Chained through the whole of K
// instead, those roundings add up: operands of one sign 2.4e-6 from 64 bits at K = 1024, against
// 5.9e-7 for fp32 products and 6e-8 for these sums added in fp32.)
// Step S of 12 is one MFMA of each of two chains: im += A_re B_im + A_im B_re, re += A_re B_re - A_im B_im.
template <int S>
__device__ __forceinline__ void product_step(const bf16x8 (&a)[2][3], const bf16x8 (&b)[2][3], const bf16x8 (&nb)[3],
                                             floatx16& im, floatx16& re) {
  constexpr int P[6] = {2, 0, 1, 1, 0, 0}, Q[6] = {0, 2, 1, 0, 1, 0};
  constexpr int p = S < 5 ? S : S < 10 ? S - 5 : 5;  // pieces
  if constexpr (S == 0) im = re = floatx16{};
  if constexpr (S < 5 || S == 10) {
    im = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[0][P[p]], b[1][Q[p]], im, 0, 0, 0);
    re = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[0][P[p]], b[0][Q[p]], re, 0, 0, 0);
  } else {
    im = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[1][P[p]], b[0][Q[p]], im, 0, 0, 0);
    re = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[1][P[p]], nb[Q[p]], re, 0, 0, 0);
  }
}

__device__ __forceinline__ void load_frags(const char* S, bf16x8 (&f)[2][3]) {
#pragma unroll
  for (int p = 0; p < 6; ++p)
    f[p / 3][p % 3] = *reinterpret_cast<const bf16x8*>(S + (p / 3) * kPlane + (p % 3) * kPiece);
}

__device__ __forceinline__ bf16x8 negated(bf16x8 v) {
  uint4 u = __builtin_bit_cast(uint4, v);
  u.x ^= 0x80008000u; u.y ^= 0x80008000u; u.z ^= 0x80008000u; u.w ^= 0x80008000u;
  return __builtin_bit_cast(bf16x8, u);
}

template <int... I, class F>
__device__ __forceinline__ void unroll_impl(std::integer_sequence<int, I...>, F&& f) {
  (f(std::integral_constant<int, I>{}), ...);
}
// f(0), ..., f(N - 1) with constant arguments
template <int N, class F>
__device__ __forceinline__ void unroll(F&& f) {
  unroll_impl(std::make_integer_sequence<int, N>{}, f);
}

__device__ __forceinline__ void clear(Acc& acc) {
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[i][r] = 0.0f;
}

// The tile's sums with fp32 products (v_mfma_f32_32x32x2f32), k from k_begin to K: the pieces of an
// infinity are not its sum and those of the smallest numbers may be flushed, so a workgroup whose sums show either
// (or an overflow) takes this path over, and its results are those of fp32 arithmetic.
// Two stages in LDS, the next one on its way in registers.  8192 x 1024 x 1024 where every workgroup takes it: 840 us, of which
// 520 here (with fp32 products alone 512; 868 with one stage in LDS).
constexpr int GLD = GBM + 2;  // LDS row pitch in floats (pad 2: transposed stores hit distinct banks)
typedef float F32Stage[2][GBK][GLD];  // [plane][k][row]
static_assert(2 * kStage >= 4 * (int)sizeof(F32Stage), "staged in the same LDS");

// S: A's and B's stage, and with more than 16 k a second pair
template <bool CONJ_B, class OpA, class OpB>
__device__ __forceinline__ void tile_f32(F32Stage* S, int k_begin, const OpA& A, const OpB& B, int w, Acc& acc_re,
                                         Acc& acc_im) {
  const int lane = threadIdx.x & 63, wm = w >> 2, wn = w & 3, li = lane & 31, lk = lane >> 5;
  float xa[8], xb[8];
  const auto load = [&](int k0) {
    if (k0 + GBK <= A.K) {
      A.load(k0, xa);
      B.load(k0, xb);
    } else {
      A.load_tail(k0, xa);
      B.load_tail(k0, xb);
    }
  };
  const auto store = [&](F32Stage* T) {
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      T[0][A.q.plane][A.q.half * 8 + c][A.q.row] = xa[c];
      T[1][B.q.plane][B.q.half * 8 + c][B.q.row] = xb[c];
    }
  };
  if (k_begin >= A.K) return;
  load(k_begin);
  store(S);
  __syncthreads();
  int par = 0;
  for (int k0 = k_begin; k0 < A.K; k0 += GBK, par ^= 2) {
    const bool more = k0 + GBK < A.K;
    if (more) load(k0 + GBK);
    const F32Stage &As = S[par], &Bs = S[par + 1];
#pragma unroll
    for (int kk = 0; kk < GBK; kk += 2) {
      const float br = Bs[0][kk + lk][wn * 32 + li], b1 = Bs[1][kk + lk][wn * 32 + li];
      const float bi = CONJ_B ? -b1 : b1;
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const float ar = As[0][kk + lk][wm * 64 + i * 32 + li], ai = As[1][kk + lk][wm * 64 + i * 32 + li];
        acc_re[i] = __builtin_amdgcn_mfma_f32_32x32x2f32(ar, br, acc_re[i], 0, 0, 0);
        acc_re[i] = __builtin_amdgcn_mfma_f32_32x32x2f32(-ai, bi, acc_re[i], 0, 0, 0);
        acc_im[i] = __builtin_amdgcn_mfma_f32_32x32x2f32(ar, bi, acc_im[i], 0, 0, 0);
        acc_im[i] = __builtin_amdgcn_mfma_f32_32x32x2f32(ai, br, acc_im[i], 0, 0, 0);
      }
    }
    if (more) {
      store(S + (par ^ 2));
      __syncthreads();
    }
  }
}

// The tile's sums with split products, k from k_begin to K, and the ranges of the operands that this thread split.
template <bool CONJ_B, class OpA, class OpB>
__device__ __forceinline__ void tile_split(char* smem, int k_begin, const OpA& A, const OpB& B, int w, Acc& acc_re,
                                           Acc& acc_im, Range& range_a, Range& range_b) {
  const int lane = threadIdx.x & 63, wm = w >> 2, wn = w & 3;
  const int foff = (lane >> 5) * kHalf + (lane & 31) * 16;
  const int a_off = foff + wm * 64 * 16, b_off = kOperand + foff + wn * 32 * 16;
  const int a_dst = A.q.plane * kPlane + A.q.half * kHalf + A.q.row * 16;
  const int b_dst = kOperand + B.q.plane * kPlane + B.q.half * kHalf + B.q.row * 16;
  float xa[8], xb[8];
  const auto stage = [&](char* S) {
    Split sa, sb;
    unroll<4>([&](auto c) {
      sa.step<c>(xa);
      sb.step<c>(xb);
      range_a.pair<c>(xa);
      range_b.pair<c>(xb);
    });
    sa.store(S + a_dst);
    sb.store(S + b_dst);
  };
  // conj(B) swaps B_im and -B_im
  const auto load_b = [&](const char* S, bf16x8 (&b)[2][3], bf16x8 (&nb)[3]) {
    load_frags(S + b_off, b);
#pragma unroll
    for (int q = 0; q < 3; ++q) {
      nb[q] = negated(b[1][q]);
      if constexpr (CONJ_B) {
        const bf16x8 t = b[1][q];
        b[1][q] = nb[q];
        nb[q] = t;
      }
    }
  };
  const int k_whole = k_begin + (A.K - k_begin) / GBK * GBK;  // end of the whole stages
  int par = 0;
  if (k_whole > k_begin) {
    const int k_last = k_whole - GBK;
    const auto next = [&](int k) { return k < k_last ? k : k_last; };  // (past the end: repeated, unused)
    A.load(k_begin, xa);
    B.load(k_begin, xb);
    stage(smem);
    A.load(next(k_begin + GBK), xa);
    B.load(next(k_begin + GBK), xb);
    __syncthreads();
    // Each MFMA pair is followed by the VALU work that fits in its shadow (about 12 instructions of 4
    // cycles in 64), pinned there by the scheduling barriers: the previous stage's sums of the second
    // row half and the range of the next stage, then its splitting and the sums of the first row half.  (The range
    // beside those sums instead: linear layer 976 us against 970, 963 without it.)
    floatx16 im0, re0, im1 = {}, re1 = {};
    for (int k0 = k_begin; k0 < k_whole; k0 += GBK, par ^= kStage) {
      char* const cur = smem + par;
      char* const nxt = smem + (par ^ kStage);
      bf16x8 a[2][3], b[2][3], nb[3];
      load_b(cur, b, nb);
      load_frags(cur + a_off, a);
      unroll<12>([&](auto s) {
        product_step<s>(a, b, nb, im0, re0);
        if constexpr (s < 8) {
#pragma unroll
          for (int r = 2 * s; r < 2 * s + 2; ++r) {
            acc_im[1][r] += im1[r];
            acc_re[1][r] += re1[r];
          }
        } else {
          range_a.pair<s - 8>(xa);
          range_b.pair<s - 8>(xb);
        }
        __builtin_amdgcn_sched_barrier(0);
      });
      load_frags(cur + a_off + 32 * 16, a);
      Split sa, sb;
      unroll<12>([&](auto s) {
        product_step<s>(a, b, nb, im1, re1);
        if constexpr (s < 4) sa.step<s>(xa);
        else if constexpr (s < 8) sb.step<s - 4>(xb);
        if constexpr (s == 4) sa.store(nxt + a_dst);
        if constexpr (s == 8) sb.store(nxt + b_dst);
        if constexpr (s >= 8) {
#pragma unroll
          for (int r = 4 * (s - 8); r < 4 * (s - 7); ++r) {
            acc_im[0][r] += im0[r];
            acc_re[0][r] += re0[r];
          }
        }
        __builtin_amdgcn_sched_barrier(0);
      });
      A.load(next(k0 + 2 * GBK), xa);
      B.load(next(k0 + 2 * GBK), xb);
      __syncthreads();
    }
    acc_im[1] += im1;
    acc_re[1] += re1;
  }
  if (k_whole < A.K) {  // the partial stage
    char* const S = smem + par;
    A.load_tail(k_whole, xa);
    B.load_tail(k_whole, xb);
    stage(S);
    __syncthreads();
    bf16x8 a[2][3], b[2][3], nb[3];
    load_b(S, b, nb);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      floatx16 im, re;
      load_frags(S + a_off + i * 32 * 16, a);
      unroll<12>([&](auto s) { product_step<s>(a, b, nb, im, re); });
      acc_im[i] += im;
      acc_re[i] += re;
    }
  }
}

// Operands: A_T = op(A) is a transpose (A stored k x m), B_T = op(B) is one (B stored n x k).  Conjugation:
// conj(A) op(B) = conj(A conj(op(B))), so CONJ_B is that of exactly one operand, and im_sign is -1 where
// A is conjugated.  SPLIT: products of bf16 pieces; otherwise fp32 products throughout, for at most 16 k.
template <bool A_T, bool B_T, bool CONJ_B, bool SPLIT>
__global__ __launch_bounds__(kThreads, SPLIT ? 2 : 4) void cgemm_kernel(
    int M, int N, int K, const float* __restrict__ A_re, const float* __restrict__ A_im, long long lda,
    const float* __restrict__ B_re, const float* __restrict__ B_im, long long ldb, float im_sign,
    const float* __restrict__ bias_re, const float* __restrict__ bias_im, float* __restrict__ C_re,
    float* __restrict__ C_im, long long ldc, float alpha, long long sa, long long sb, long long sc, int k_chunk,
    long long sz) {
  __shared__ __attribute__((aligned(16))) char smem[SPLIT ? 2 * kStage : 2 * sizeof(F32Stage)];
  // batched products: blockIdx.y selects the matrix triple (batch strides in floats; a stride of 0
  // broadcasts one operand over the batch)
  {
    const size_t bz = blockIdx.y;
    A_re += bz * sa;
    A_im += bz * sa;
    B_re += bz * sb;
    B_im += bz * sb;
    C_re += bz * sc + blockIdx.z * sz;
    C_im += bz * sc + blockIdx.z * sz;
  }
  // split products: blockIdx.z sums the k_chunk columns of op(A) from k_begin into its own partial
  const int k_begin = (int)blockIdx.z * k_chunk;
  K = K - k_begin < k_chunk ? K : k_begin + k_chunk;
  const int t = threadIdx.x;
  const int w = __builtin_amdgcn_readfirstlane(t >> 6);
  const int wm = w >> 2, wn = w & 3;
  // XCD-aware: neighbouring row tiles (which share B) run on one XCD
  const long long tiles_n = (N + GBN - 1) / GBN;
  const long long tile = xcd_tile_remap(blockIdx.x, gridDim.x);
  const int row0 = (int)(tile / tiles_n) * GBM;
  const int col0 = (int)(tile % tiles_n) * GBN;

  Acc acc_re, acc_im;
  clear(acc_re);
  clear(acc_im);
  const Operand<!A_T> A(A_re, A_im, lda, M, K, row0, t, w);
  const Operand<B_T> B(B_re, B_im, ldb, N, K, col0, t, w);
  if constexpr (SPLIT) {
    Range range_a, range_b;
    tile_split<CONJ_B>(smem, k_begin, A, B, w, acc_re, acc_im, range_a, range_b);
    // sums below the limit (0 where nothing is lost) or not finite need fp32 products
    float limit = 0.0f;
    if (__syncthreads_or(range_a.small() || range_b.small())) {
      unsigned* const lds = reinterpret_cast<unsigned*>(smem);
      range_a.reduce(lds, w);
      range_b.reduce(lds + 2 * kThreads / 64, w);
      const float a = range_a.least(), b = range_b.least();
      if (fminf(a, b) < kExact || a * b < kSumFloor)
        limit = (float)(K - k_begin) * fmaxf(kSumLimit * fmaxf(range_a.hi, range_b.hi), kSumFloor);
    }
    int odd = 0;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int r = 0; r < 16; ++r) odd |= outside(acc_re[i][r], limit) | outside(acc_im[i][r], limit);
    if (__syncthreads_or(odd)) {
      clear(acc_re);
      clear(acc_im);
      tile_f32<CONJ_B>(reinterpret_cast<F32Stage*>(smem), k_begin, A, B, w, acc_re, acc_im);
    }
  } else {
    tile_f32<CONJ_B>(reinterpret_cast<F32Stage*>(smem), k_begin, A, B, w, acc_re, acc_im);
  }
  const int li = t & 31, lk = (t >> 5) & 1;

  // D layout of both MFMAs: lane l, register r -> row 8*(r/4) + 4*(l/32) + r%4, col l%32
  const int col = col0 + wn * 32 + li;
  if (col >= N) return;
  const float b_re = bias_re ? bias_re[col] : 0.0f;
  const float b_im = bias_im ? bias_im[col] : 0.0f;
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int row = row0 + wm * 64 + i * 32 + 8 * (r >> 2) + 4 * lk + (r & 3);
      if (row < M) {
        C_re[(size_t)row * ldc + col] = acc_re[i][r] * alpha + b_re;
        C_im[(size_t)row * ldc + col] = acc_im[i][r] * (alpha * im_sign) + b_im;
      }
    }
}

// C = alpha * (sum of the partials over z, in order) + bias; V consecutive columns per thread.
// Memory-bound: 8 partials of 1024 x 1024 (67 MB, written just before, so partly in the
// Infinity Cache) in 12 us.
template <int V>
__global__ __launch_bounds__(256) void cgemm_reduce_kernel(const float* __restrict__ ws, int splits, int M, int N,
                                                           const float* __restrict__ bias_re,
                                                           const float* __restrict__ bias_im,
                                                           float* __restrict__ C_re, float* __restrict__ C_im,
                                                           long long ldc, long long sc, float alpha, long long plane) {
  typedef float vec __attribute__((ext_vector_type(V)));
  const long long per = (long long)M * N;
  const long long i = ((long long)blockIdx.x * 256 + threadIdx.x) * V;
  if (i >= per) return;
  const size_t bz = blockIdx.y;
  const float* p = ws + bz * per + i;
  const long long sz = per * gridDim.y;
  vec re = *reinterpret_cast<const vec*>(p), im = *reinterpret_cast<const vec*>(p + plane);
  for (int z = 1; z < splits; ++z) {
    re += *reinterpret_cast<const vec*>(p + z * sz);
    im += *reinterpret_cast<const vec*>(p + plane + z * sz);
  }
  const int row = (int)(i / N), col = (int)(i - (long long)row * N);
  re *= alpha;
  im *= alpha;
  if (bias_re) {
#pragma unroll
    for (int v = 0; v < V; ++v) {
      re[v] += bias_re[col + v];
      im[v] += bias_im[col + v];
    }
  }
  const size_t o = bz * sc + (size_t)row * ldc + col;
  *reinterpret_cast<vec*>(C_re + o) = re;
  *reinterpret_cast<vec*>(C_im + o) = im;
}

constexpr long long kMaxGridY = 65535;

// Number of K ranges a product is summed in (1: no split).  A workgroup computes one 128 x 128 tile, one
// per CU at a time, so the product takes ceil(tiles * ranges / 256) rounds of (K / ranges) / 16 stages of
// about 2 us; a split adds the launch that reduces the partials (4 us and their traffic at 4 TB/s).  The
// number with the least sum of these is taken, each range at least kMinSplitK columns.  Weight gradients
// are such products: (1024 x 8192) x (8192 x 1024) is 64 tiles, 883 us unsplit, 331 us in
// 4 ranges; 220 x 2019 x 334 227 -> 33 us (26 ranges), 1000 x 256 x 1000 40 -> 30 (4); 1500 x 2048 x 1800, 180
// tiles, 256 -> 263.
// The shorter sums also round less (4.4e-7 -> 2.6e-7 at K = 8192).
constexpr int kMinSplitK = 64;
int cgemm_splits(long long batch, long long m, long long n, long long k, int* k_chunk) {
  const long long tiles = ((m + GBM - 1) / GBM) * ((n + GBN - 1) / GBN) * batch;
  *k_chunk = (int)k;
  if (tiles < 1 || tiles >= kNumCUs || batch > kMaxGridY) return 1;
  int best = 1;
  double best_us = (double)((k + GBK - 1) / GBK) * 2.0;
  for (long long s = 2; s <= k / kMinSplitK && s <= 64; ++s) {
    const long long chunk = ((k + s - 1) / s + GBK - 1) / GBK * GBK, parts = (k + chunk - 1) / chunk;
    const double us = (double)((tiles * parts + kNumCUs - 1) / kNumCUs) * (chunk / GBK) * 2.0 + 4.0 +
                      (double)(parts + 1) * batch * m * n * 8.0 / 4e6;
    if (us < best_us) {
      best_us = us;
      best = (int)parts;
      *k_chunk = (int)chunk;
    }
  }
  return best;
}

size_t cgemm_workspace_bytes(long long batch, long long m, long long n, long long k) {
  int kc;
  const int s = cgemm_splits(batch, m, n, k, &kc);
  return s > 1 ? (size_t)s * batch * m * n * 2 * sizeof(float) : 0;
}

template <bool A_T, bool B_T, bool CONJ_B>
static void launch_cgemm_t(const GemmArgs& a, long long tiles) {
  const float im_sign = (a.a_op == 2 || a.a_op == 3) ? -1.0f : 1.0f;
  int k_chunk = (int)a.k;
  const int splits = a.workspace ? cgemm_splits(a.batch, a.m, a.n, a.k, &k_chunk) : 1;
  if (splits > 1) {
    const long long per = a.m * a.n, sz = per * a.batch, plane = sz * splits;
    float* ws = a.workspace;
    hipLaunchKernelGGL((cgemm_kernel<A_T, B_T, CONJ_B, true>), dim3((unsigned)tiles, (unsigned)a.batch, splits),
                       dim3(kThreads), 0, a.stream, (int)a.m, (int)a.n, (int)a.k, a.a_re, a.a_im, a.lda, a.b_re, a.b_im, a.ldb,
                       im_sign, nullptr, nullptr, ws, ws + plane, a.n, 1.0f, a.sa, a.sb, per, k_chunk, sz);
    // four columns per thread where every row of C starts 16-byte aligned
    const bool v4 = a.n % 4 == 0 && a.ldc % 4 == 0 && a.sc % 4 == 0 &&
                    (reinterpret_cast<size_t>(a.c_re) | reinterpret_cast<size_t>(a.c_im) |
                     reinterpret_cast<size_t>(ws)) % 16 == 0;
    auto go = [&](auto kern, int v) {
      const unsigned blocks = (unsigned)((per / v + 255) / 256);
      hipLaunchKernelGGL(kern, dim3(blocks, (unsigned)a.batch), dim3(256), 0, a.stream, ws, splits, (int)a.m, (int)a.n,
                         a.bias_re, a.bias_im, a.c_re, a.c_im, a.ldc, a.sc, a.alpha, plane);
    };
    if (v4) go(cgemm_reduce_kernel<4>, 4);
    else go(cgemm_reduce_kernel<1>, 1);
    return;
  }
  // At most one stage of k: fp32 products leave room for two workgroups per CU, and no MFMA hides the splitting
  // (4096 products of 16 x 16 x 16 80 us against 108, 8192 x 16 x 1024 20.7 against 24.3; two stages of split products,
  // 1000 of 32 x 32 x 32, 39 against 42 for fp32 ones).
  const auto kern = a.k <= GBK ? cgemm_kernel<A_T, B_T, CONJ_B, false> : cgemm_kernel<A_T, B_T, CONJ_B, true>;
  for (long long b0 = 0; b0 < a.batch; b0 += kMaxGridY) {
    const unsigned nb = (unsigned)std::min(kMaxGridY, a.batch - b0);
    hipLaunchKernelGGL(kern, dim3((unsigned)tiles, nb), dim3(kThreads), 0, a.stream, (int)a.m, (int)a.n, (int)a.k, a.a_re + b0 * a.sa, a.a_im + b0 * a.sa, a.lda, a.b_re + b0 * a.sb,
                       a.b_im + b0 * a.sb, a.ldb, im_sign, a.bias_re, a.bias_im, a.c_re + b0 * a.sc,
                       a.c_im + b0 * a.sc, a.ldc, a.alpha, a.sa, a.sb, a.sc, k_chunk, 0LL);
  }
}

hipError_t launch_cgemm(const GemmArgs& a) {
  const long long tiles = ((a.m + GBM - 1) / GBM) * ((a.n + GBN - 1) / GBN);
  const bool at = a.a_op == 1 || a.a_op == 2, bt = a.b_op == 1 || a.b_op == 2;
  const bool conj_b = (a.a_op == 2 || a.a_op == 3) != (a.b_op == 2 || a.b_op == 3);
  using Launch = void (*)(const GemmArgs&, long long);
  static constexpr Launch table[2][2][2] = {
      {{launch_cgemm_t<false, false, false>, launch_cgemm_t<false, false, true>},
       {launch_cgemm_t<false, true, false>, launch_cgemm_t<false, true, true>}},
      {{launch_cgemm_t<true, false, false>, launch_cgemm_t<true, false, true>},
       {launch_cgemm_t<true, true, false>, launch_cgemm_t<true, true, true>}}};
  table[at][bt][conj_b](a, tiles);
  return hipGetLastError();
}

// Column sums of two row-major (rows, cols) planes (a bias gradient).  A workgroup sums 64 columns over one
// chunk of rows, four row lanes of eight loads in flight each, into its partial; with more than one chunk a
// second launch adds the partials in order.  Bound by HBM: 8192 x 1024 (67 MB) in 17 us with
// the second launch, against 52 for two torch sums.
constexpr int kSumCols = 64, kSumLanes = 4, kSumUnroll = 8;

__global__ __launch_bounds__(kSumCols * kSumLanes) void column_sums_kernel(const float* __restrict__ re,
                                                                           const float* __restrict__ im,
                                                                           float* __restrict__ out_re,
                                                                           float* __restrict__ out_im, int rows,
                                                                           int cols, int chunk) {
  __shared__ float part[kSumLanes][kSumCols];
  const int c = threadIdx.x % kSumCols, lane = threadIdx.x / kSumCols;
  const int col = blockIdx.x * kSumCols + c, cc = col < cols ? col : cols - 1;
  const long long r0 = (long long)blockIdx.y * chunk;
  const long long r1 = r0 + chunk < rows ? r0 + chunk : rows;
  const float* p = (blockIdx.z ? im : re) + cc;
  float s[kSumUnroll] = {};
  for (long long r = r0 + lane; r < r1; r += kSumLanes * kSumUnroll) {
    float v[kSumUnroll];
#pragma unroll
    for (int u = 0; u < kSumUnroll; ++u) {
      const long long q = r + u * kSumLanes;
      v[u] = p[(size_t)(q < r1 ? q : r1 - 1) * cols];
    }
#pragma unroll
    for (int u = 0; u < kSumUnroll; ++u)
      if (r + u * kSumLanes < r1) s[u] += v[u];
  }
#pragma unroll
  for (int h = kSumUnroll / 2; h > 0; h /= 2)
#pragma unroll
    for (int u = 0; u < h; ++u) s[u] += s[u + h];
  part[lane][c] = s[0];
  __syncthreads();
  if (lane == 0 && col < cols) {
    float* o = (blockIdx.z ? out_im : out_re) + (size_t)blockIdx.y * cols;
    o[col] = (part[0][c] + part[1][c]) + (part[2][c] + part[3][c]);
  }
}

// rows per chunk: about 2048 workgroups in all, at least 32 rows each
static long long column_sum_chunk(long long rows, long long cols) {
  const long long tiles = 2 * ((cols + kSumCols - 1) / kSumCols);
  const long long chunks = std::max(1LL, std::min({rows / 32, 2048 / tiles, 65535LL}));
  return (rows + chunks - 1) / chunks;
}

size_t column_sums_workspace_bytes(long long rows, long long cols) {
  if (rows < 1) return 0;
  const long long chunk = column_sum_chunk(rows, cols), chunks = (rows + chunk - 1) / chunk;
  return chunks > 1 ? (size_t)chunks * cols * 2 * sizeof(float) : 0;
}

hipError_t launch_column_sums(const float* re, const float* im, float* out_re, float* out_im, long long rows,
                              long long cols, float* ws, hipStream_t stream) {
  const long long chunk = ws ? column_sum_chunk(rows, cols) : rows, chunks = (rows + chunk - 1) / chunk;
  const unsigned tiles = (unsigned)((cols + kSumCols - 1) / kSumCols);
  const dim3 block(kSumCols * kSumLanes);
  float* p_re = chunks > 1 ? ws : out_re;
  float* p_im = chunks > 1 ? ws + chunks * cols : out_im;
  hipLaunchKernelGGL(column_sums_kernel, dim3(tiles, (unsigned)chunks, 2), block, 0, stream, re, im, p_re, p_im,
                     (int)rows, (int)cols, (int)chunk);
  if (chunks > 1)
    hipLaunchKernelGGL(column_sums_kernel, dim3(tiles, 1, 2), block, 0, stream, p_re, p_im, out_re, out_im, (int)chunks,
                       (int)cols, (int)chunks);
  return hipGetLastError();
}

}  // namespace tfa
