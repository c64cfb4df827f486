// fft_reg.hpp -- register-resident FFTs of the lengths of PHZ_REG_LENGTHS (48 to
// 256, even, with factors 2, 3 and 5) and, for the SO(3) grid, up to 320 for
// gfx950: each line is split as L = R1 * R2 (four-step Cooley-Tukey,
// n = n2 + R2 n1, k = k1 + R1 k2):
//   X[k1 + R1 k2] = sum_n2 W_R2^(n2 k2) W_L^(n2 k1) sum_n1 x[n2 + R2 n1] W_R1^(n1 k1)
// R2 threads per line each load R1 elements straight from HBM, transform
// them in registers, apply the W_L twiddles, exchange once through LDS and
// finish with the R1 transforms of length R2 spread over the line's threads
// (thread n2 takes k1 = n2 + R2 j), storing straight to HBM.  One LDS round
// trip per line instead of one per radix stage.
#pragma once

#include <type_traits>

#include "common.hpp"

namespace phz {

// cos(2 pi m / 16), m = 0..15
constexpr float kC16[16] = {
    1.0f, 0.92387953251128674f, 0.70710678118654752f, 0.38268343236508977f,
    0.0f, -0.38268343236508977f, -0.70710678118654752f, -0.92387953251128674f,
    -1.0f, -0.92387953251128674f, -0.70710678118654752f, -0.38268343236508977f,
    0.0f, 0.38268343236508977f, 0.70710678118654752f, 0.92387953251128674f};

constexpr int bitrev(int x, int bits) {
  int r = 0;
  for (int i = 0; i < bits; ++i) r |= ((x >> i) & 1) << (bits - 1 - i);
  return r;
}
constexpr int ilog2(int x) { return x <= 1 ? 0 : 1 + ilog2(x / 2); }

// exp(DIR * 2 pi i j / len) for len | 16, as a compile-time constant
template <int DIR>
__host__ __device__ __forceinline__ float2 w16(int j, int len) {
  const int m = (j * (16 / len)) & 15;
  const int ms = (m + 12) & 15;  // sin(2 pi m / 16) = cos(2 pi (m - 4) / 16)
  return make_float2(kC16[m], DIR * kC16[ms]);
}

// cos and sin of 2 pi m / len at compile time: the angle is folded into
// [0, pi / 4] by the octant symmetries in whole numbers, then summed by its
// Taylor series in double (terms below 1e-17 there after 10)
constexpr double taylor_cos(double x) {
  double s = 0.0, t = 1.0;
  for (int k = 0; k < 10; ++k) {
    s += t;
    t *= -x * x / ((2 * k + 1) * (2 * k + 2));
  }
  return s;
}
constexpr double taylor_sin(double x) {
  double s = 0.0, t = x;
  for (int k = 0; k < 10; ++k) {
    s += t;
    t *= -x * x / ((2 * k + 2) * (2 * k + 3));
  }
  return s;
}
constexpr double cos_turn(int m, int len) {
  m %= len;
  if (2 * m > len) m = len - m;                       // cos(-x) = cos x
  if (4 * m > len) return -cos_turn(len - 2 * m, 2 * len);  // cos(pi - x) = -cos x
  const double x = 6.283185307179586476925 * m / len;
  return 8 * m > len ? taylor_sin(1.570796326794896619231 - x) : taylor_cos(x);
}
constexpr double sin_turn(int m, int len) {  // sin x = cos(x - pi / 2)
  return cos_turn(4 * m + 3 * len, 4 * len);
}

// The twiddles exp(2 pi i n2 k1 / R) of one split R = P * Q, as a table the
// unrolled transform folds into constants
template <int P, int Q>
struct SplitTable {
  float c[P * Q], s[P * Q];
};
template <int P, int Q>
constexpr SplitTable<P, Q> split_table() {
  SplitTable<P, Q> t{};
  for (int n2 = 0; n2 < Q; ++n2)
    for (int k1 = 0; k1 < P; ++k1) {
      t.c[n2 * P + k1] = (float)cos_turn(n2 * k1, P * Q);
      t.s[n2 * P + k1] = (float)sin_turn(n2 * k1, P * Q);
    }
  return t;
}

// the factor P of a composite R = P * Q: the largest of 5, 4, 3, 2 that
// leaves a transform of its own
constexpr int split_factor(int R) {
  return R % 8 == 0 && R > 8 ? 8 : (R % 5 == 0 ? 5 : (R % 4 == 0 ? 4 : (R % 3 == 0 ? 3 : 2)));
}

constexpr int gcd_of(int a, int b) { return b ? gcd_of(b, a % b) : a; }
// x with a x = 1 mod m
constexpr int inverse_mod(int a, int m) {
  for (int x = 1; x < m; ++x)
    if (a * x % m == 1) return x;
  return 1;
}

// In-register DFT of length R: v[k] <- sum_n v[n] exp(DIR 2 pi i nk / R),
// natural order in and out.  2, 4, 8, 16: radix-2 decimation in frequency,
// then the bit-reversal permutation; 3 and 5: the real / imaginary symmetric
// forms; other products of 2, 3 and 5: split P * Q, for coprime factors by
// the prime-factor index maps n = Q n1 + P n2, k = k1 mod P and k2 mod Q
// (mod R, no twiddles: less work and less rounding), else with twiddles.
// Everything but the data is resolved at compile time.
template <int R, int DIR>
__host__ __device__ __forceinline__ void dft_reg(float2 (&v)[R]) {
  if constexpr (R == 1) {
  } else if constexpr (R == 3) {
    constexpr float s = DIR * 0.86602540378443865f;
    const float2 t1 = cadd(v[1], v[2]), t2 = csub(v[1], v[2]);
    const float2 m1 = make_float2(v[0].x - 0.5f * t1.x, v[0].y - 0.5f * t1.y);
    const float2 m2 = make_float2(-s * t2.y, s * t2.x);  // i s t2
    v[0] = cadd(v[0], t1);
    v[1] = cadd(m1, m2);
    v[2] = csub(m1, m2);
  } else if constexpr (R == 5) {
    constexpr float c1 = 0.30901699437494742f, c2 = -0.80901699437494742f;
    constexpr float s1 = DIR * 0.95105651629515357f, s2 = DIR * 0.58778525229247313f;
    const float2 a = v[0];
    const float2 t1 = cadd(v[1], v[4]), t2 = cadd(v[2], v[3]);
    const float2 t3 = csub(v[1], v[4]), t4 = csub(v[2], v[3]);
    v[0] = cadd(a, cadd(t1, t2));
    const float2 b1 = make_float2(a.x + c1 * t1.x + c2 * t2.x, a.y + c1 * t1.y + c2 * t2.y);
    const float2 b2 = make_float2(a.x + c2 * t1.x + c1 * t2.x, a.y + c2 * t1.y + c1 * t2.y);
    const float2 e1 = make_float2(-(s1 * t3.y + s2 * t4.y), s1 * t3.x + s2 * t4.x);
    const float2 e2 = make_float2(-(s2 * t3.y - s1 * t4.y), s2 * t3.x - s1 * t4.x);
    v[1] = cadd(b1, e1);
    v[4] = csub(b1, e1);
    v[2] = cadd(b2, e2);
    v[3] = csub(b2, e2);
  } else if constexpr (R == 2 || R == 4 || R == 8 || R == 16) {
#pragma unroll
    for (int len = R; len >= 2; len >>= 1) {
#pragma unroll
      for (int b = 0; b < R; b += len) {
#pragma unroll
        for (int j = 0; j < len / 2; ++j) {
          const float2 u = v[b + j], w = v[b + j + len / 2];
          v[b + j] = cadd(u, w);
          const float2 d = csub(u, w);
          if (j == 0) {
            v[b + j + len / 2] = d;
          } else if (4 * j == len) {  // times exp(DIR i pi / 2) = DIR i
            v[b + j + len / 2] = DIR < 0 ? make_float2(d.y, -d.x) : make_float2(-d.y, d.x);
          } else {
            v[b + j + len / 2] = cmul(d, w16<DIR>(j, len));
          }
        }
      }
    }
    float2 t[R];
#pragma unroll
    for (int k = 0; k < R; ++k) t[k] = v[bitrev(k, ilog2(R))];
#pragma unroll
    for (int k = 0; k < R; ++k) v[k] = t[k];
  } else {
    constexpr int P = split_factor(R), Q = R / P;
    static_assert(P < R && P * Q == R, "factors 2, 3 and 5");
    constexpr bool kCoprime = gcd_of(P, Q) == 1;
    constexpr SplitTable<P, Q> W = split_table<P, Q>();
    // k = k1 mod P and k2 mod Q
    constexpr int kp = Q * inverse_mod(Q % P, P), kq = P * inverse_mod(P % Q, Q);
    float2 y[Q][P];
#pragma unroll
    for (int n2 = 0; n2 < Q; ++n2) {
#pragma unroll
      for (int n1 = 0; n1 < P; ++n1)
        y[n2][n1] = v[kCoprime ? (Q * n1 + P * n2) % R : n2 + Q * n1];
      dft_reg<P, DIR>(y[n2]);
#pragma unroll
      for (int k1 = 1; k1 < P; ++k1)
        if (n2 > 0 && !kCoprime)
          y[n2][k1] = cmul(y[n2][k1], make_float2(W.c[n2 * P + k1], DIR * W.s[n2 * P + k1]));
    }
#pragma unroll
    for (int k1 = 0; k1 < P; ++k1) {
      float2 u[Q];
#pragma unroll
      for (int n2 = 0; n2 < Q; ++n2) u[n2] = y[n2][k1];
      dft_reg<Q, DIR>(u);
#pragma unroll
      for (int k2 = 0; k2 < Q; ++k2)
        v[kCoprime ? (kp * k1 + kq * k2) % R : k1 + P * k2] = u[k2];
    }
  }
}

// The lengths of the engine and their splits; other lengths take the LDS
// passes.  R1 elements per thread and R2 threads per line; a workgroup of LINES
// lines is whole waves.  R1 a multiple of R2, or R1 <= R2 near it: the second
// transforms then take whole rounds or a single one (a partly filled second
// round, as 12 x 10 for 120, made the fused cross spectrum twice as slow as one
// of 10 x 12).  LINES = 32 lines make a strided pass read 256-byte runs; 16
// where 32 lines would need many more threads or span more than two z planes,
// 64 for whole waves at odd R2.
// In groups, one per file that builds them for the translation stage.
#define PHZ_REG_LENGTHS_A(X) \
  X(48, 12, 4) X(60, 5, 12) X(64, 8, 8) X(72, 12, 6) X(80, 8, 10) X(90, 9, 10)
#define PHZ_REG_LENGTHS_B(X) \
  X(96, 8, 12) X(100, 10, 10) X(108, 9, 12) X(120, 10, 12) X(128, 16, 8)
#define PHZ_REG_LENGTHS_C(X) X(144, 9, 16) X(150, 10, 15) X(160, 10, 16) X(180, 10, 18)
#define PHZ_REG_LENGTHS_D(X) X(192, 12, 16) X(200, 20, 10) X(216, 12, 18)
#define PHZ_REG_LENGTHS_E(X) X(240, 15, 16) X(256, 16, 16)
#define PHZ_REG_LENGTHS(X)                                                          \
  PHZ_REG_LENGTHS_A(X) PHZ_REG_LENGTHS_B(X) PHZ_REG_LENGTHS_C(X) PHZ_REG_LENGTHS_D(X) \
  PHZ_REG_LENGTHS_E(X)
// the SO(3) grid's sides 2 B reach 320
#define PHZ_REG_LENGTHS_SO3(X) \
  PHZ_REG_LENGTHS(X) X(250, 25, 10) X(288, 16, 18) X(300, 15, 20) X(320, 16, 20)

template <int L>
struct RegFactors;
#define PHZ_REG_FACTORS(LEN, A, B)         \
  template <>                              \
  struct RegFactors<LEN> {                 \
    static_assert(A * B == LEN, "a split of the length"); \
    static constexpr int R1 = A, R2 = B;   \
  };
PHZ_REG_LENGTHS_SO3(PHZ_REG_FACTORS)
#undef PHZ_REG_FACTORS

template <int L>
struct RegSplit {
  static constexpr int R1 = RegFactors<L>::R1, R2 = RegFactors<L>::R2;
  // rounds of the second transforms; kEven: every round is full, and a
  // thread's outputs are the inputs it needs for another transform
  static constexpr int C = (R1 + R2 - 1) / R2;
  static constexpr bool kEven = R1 % R2 == 0;
  // entry j R2 + k2 of for_outputs is frequency n2 + kStep order(i): the
  // entries of a thread in ascending frequency are its order 0, 1, ...
  static constexpr bool kOrdered = kEven || C == 1;
  static constexpr int kStep = kEven ? R2 : R1;
  static constexpr int order(int i) { return kEven ? i / R2 + C * (i % R2) : i; }
  // Exchange pitch of the kernels whose lanes run over n2 first (rows), and the
  // line stride it needs.  A pitch of a multiple of four 8-byte entries meets
  // its own banks again within the lanes of a line, so those get an odd one:
  // c2r over 4 grids of 256^3 123 -> 75 us (14 conflict cycles per access
  // before), r2c of 8 grids of 192^3 72 -> 54, of 16 of 64^3 17.4 -> 16.6; 18
  // gains 6% (c2r at 216); 6 and 10 already spread and lose by the longer
  // lines (r2c at 72 21 -> 22.5, c2r at 200 100 -> 144).
  static constexpr int kRowPitch = R2 % 4 == 0 || R2 > 16 ? R2 | 1 : R2;
  static constexpr int kRowStride = (R1 * kRowPitch > L ? R1 * kRowPitch : L) | 1;
  static constexpr int LINES = R2 % 2 ? 64 : (R2 == 16 || R2 == 20 || L < 64) ? 16 : 32;
  static constexpr int TPB = LINES * R2;
  static_assert(TPB % 64 == 0, "whole waves");
};

// The twiddles of a workgroup's transforms in LDS, entry [k1][n2] = W_L^(n2
// k1): a thread's are at one address plus constants, the same for all lanes
// of an n2 (a broadcast).  Kept in registers they were R1 global loads per
// thread beside its R1 data loads, and 2 R1 registers across every transform;
// as scalar loads they cost a move and a select per component (the forward x
// pass 125 -> 116 us for 16 pairs at L = 128, the cross spectrum 268 -> 253 us
// for 8 at 192 and 353 -> 330 us for 4 at 256).
template <int L>
struct LdsTwiddles {
  const float2* row;  // the table at this thread's n2
  __device__ __forceinline__ float2 operator()(int k1) const {
    return row[k1 * RegSplit<L>::R2];
  }
};
// tw: exp(-2 pi i e / L); table: L entries of LDS.  The caller has a barrier
// between this and the first transform.
template <int L>
__device__ __forceinline__ LdsTwiddles<L> stage_twiddles(float2* table, int n2,
                                                         const float2* __restrict__ tw) {
  constexpr int R2 = RegSplit<L>::R2;
  for (int i = threadIdx.x; i < L; i += blockDim.x) table[i] = tw[(i % R2) * (i / R2)];
  return LdsTwiddles<L>{table + n2};
}

// The four-step transform of one line held by R2 threads of a workgroup, in
// registers.  On entry thread n2 holds v[n1] = x[n2 + R2 n1]; lbuf is the
// line's LDS scratch, entry i at lbuf[i * stride] (L entries; stride 1 unless
// a line exchanges through its own storage in a larger array).  PITCH > R2
// spreads the second transforms' reads over the banks where the lanes of a
// wave are the threads of few lines (kRowPitch; R1 PITCH entries then).  On return
// out[j * R2 + k2] = X[k1 + R1 k2], k1 = n2 + R2 j, for k1 < R1 (the entries
// of a thread past the last k1 are not set).  A line that is not active
// touches no LDS.  Contains one __syncthreads, so every thread of the
// workgroup must call it.
template <int DIR, int L, int PITCH = RegSplit<L>::R2, class TW>
__device__ __forceinline__ void fft_four_step_reg(
    float2 (&v)[RegSplit<L>::R1], int n2, float2* lbuf, const TW& tw,
    float2 (&out)[RegSplit<L>::C * RegSplit<L>::R2], int stride = 1, bool active = true) {
  constexpr int R1 = RegSplit<L>::R1, R2 = RegSplit<L>::R2, C = RegSplit<L>::C;
  dft_reg<R1, DIR>(v);
#pragma unroll
  for (int k1 = 1; k1 < R1; ++k1) {
    float2 w = tw(k1);
    if (DIR > 0) w.y = -w.y;
    v[k1] = cmul(v[k1], w);
  }
  if (active) {
#pragma unroll
    for (int k1 = 0; k1 < R1; ++k1) lbuf[(k1 * PITCH + n2) * stride] = v[k1];
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < C; ++j) {
    const int k1 = n2 + R2 * j;
    if (active && (RegSplit<L>::kEven || k1 < R1)) {
      float2 u[R2];
#pragma unroll
      for (int m = 0; m < R2; ++m) u[m] = lbuf[(k1 * PITCH + m) * stride];
      dft_reg<R2, DIR>(u);
#pragma unroll
      for (int k2 = 0; k2 < R2; ++k2) out[j * R2 + k2] = u[k2];
    }
  }
}

// calls f(i, k) for every entry i of a thread's fft_four_step_reg output,
// k its frequency
template <int L, class F>
__device__ __forceinline__ void for_outputs(int n2, F f) {
  constexpr int R1 = RegSplit<L>::R1, R2 = RegSplit<L>::R2, C = RegSplit<L>::C;
#pragma unroll
  for (int j = 0; j < C; ++j)
    if (RegSplit<L>::kEven || n2 + R2 * j < R1) {
#pragma unroll
      for (int k2 = 0; k2 < R2; ++k2) f(j * R2 + k2, (n2 + R2 * j) + R1 * k2);
    }
}

// the same in ascending order of the frequency, with the entry's place e in
// that order; place_frequency gives the frequency of a place
template <int L, class F>
__device__ __forceinline__ void for_outputs_ascending(int n2, F f) {
  constexpr int R1 = RegSplit<L>::R1, R2 = RegSplit<L>::R2, C = RegSplit<L>::C;
#pragma unroll
  for (int k2 = 0; k2 < R2; ++k2)
#pragma unroll
    for (int j = 0; j < C; ++j)
      if (RegSplit<L>::kEven || n2 + R2 * j < R1)
        f(j * R2 + k2, (n2 + R2 * j) + R1 * k2, k2 * C + j);
}
template <int L>
__device__ __forceinline__ int place_frequency(int n2, int e) {
  constexpr int C = RegSplit<L>::C;
  return n2 + RegSplit<L>::R2 * (e % C) + RegSplit<L>::R1 * (e / C);
}

// The same transform with store(k, X[k]) called for each output.
template <int DIR, int L, class Store, class TW>
__device__ __forceinline__ void fft_four_step(float2 (&v)[RegSplit<L>::R1], int n2, float2* lbuf,
                                              const TW& tw, Store store, bool active = true) {
  float2 out[RegSplit<L>::C * RegSplit<L>::R2];
  fft_four_step_reg<DIR, L>(v, n2, lbuf, tw, out, 1, active);
  if (active) for_outputs<L>(n2, [&](int i, int k) { store(k, out[i]); });
}

// The transform of a line whose thread n2 holds the entries of
// for_outputs<L> (entry i of v at index k of the line), without another
// exchange to reach the layout fft_four_step starts from: the split with the
// factors in the other order, k = k1 + R1 k2,
//   x[m1 + R2 m2] = sum_k1 W_R1^(k1 m2) W_L^(k1 m1) sum_k2 v[k1 + R1 k2] W_R2^(k2 m1),
// so the thread's own R2 entries of each k1 are transformed first.  table:
// the twiddles of stage_twiddles.  lbuf as above (L entries).  store(m, x[m]).
template <int DIR, int L, class Store>
__device__ __forceinline__ void fft_from_outputs(
    float2 (&v)[RegSplit<L>::C * RegSplit<L>::R2], int n2, float2* lbuf, const float2* table,
    Store store) {
  constexpr int R1 = RegSplit<L>::R1, R2 = RegSplit<L>::R2, C = RegSplit<L>::C;
#pragma unroll
  for (int j = 0; j < C; ++j) {
    const int k1 = n2 + R2 * j;
    if (RegSplit<L>::kEven || k1 < R1) {
      float2 u[R2];
#pragma unroll
      for (int k2 = 0; k2 < R2; ++k2) u[k2] = v[j * R2 + k2];
      dft_reg<R2, DIR>(u);
#pragma unroll
      for (int m1 = 0; m1 < R2; ++m1) {
        float2 w = table[k1 * R2 + m1];  // W_L^(k1 m1)
        if (DIR > 0) w.y = -w.y;
        lbuf[m1 * R1 + k1] = m1 ? cmul(u[m1], w) : u[m1];
      }
    }
  }
  __syncthreads();
  float2 y[R1];
#pragma unroll
  for (int k1 = 0; k1 < R1; ++k1) y[k1] = lbuf[n2 * R1 + k1];
  dft_reg<R1, DIR>(y);
#pragma unroll
  for (int m2 = 0; m2 < R1; ++m2) store(n2 + R2 * m2, y[m2]);
}

// Lines of length L of complex data: line q of batch z starts at data +
// z*batch_stride + (q / inner) * L * inner + q % inner and has stride
// `inner`.  LINES lines per workgroup, R2 threads per line (the line index
// runs fastest across threads, so strided lines load coalesced).
// tw: exp(-2 pi i e / L), e < L (conjugated for DIR = +1).
template <int DIR, int L>
__global__ void __launch_bounds__(RegSplit<L>::TPB) k_fft_lines(
    float2* __restrict__ data, int64_t batch_stride, int nlines, int inner,
    const float2* __restrict__ tw) {
  constexpr int R1 = RegSplit<L>::R1, R2 = RegSplit<L>::R2, kLines = RegSplit<L>::LINES;
  constexpr int S = L + 1;  // LDS stride per line (odd: spreads banks)
  __shared__ float2 buf[kLines * S];
  __shared__ float2 table[L];
  const int c = threadIdx.x % kLines, n2 = threadIdx.x / kLines;
  const int q = blockIdx.x * kLines + c;
  const bool live = q < nlines;
  const LdsTwiddles<L> w = stage_twiddles<L>(table, n2, tw);
  float2* base = data + blockIdx.y * batch_stride;
  if (live) base += (int64_t)(q / inner) * L * inner + (q % inner);
  float2 v[R1];
#pragma unroll
  for (int n1 = 0; n1 < R1; ++n1)
    v[n1] = live ? base[(int64_t)(n2 + R2 * n1) * inner] : make_float2(0.f, 0.f);
  __syncthreads();
  fft_four_step<DIR, L>(v, n2, buf + c * S, w, [&](int k, float2 x) {
    if (live) base[(int64_t)k * inner] = x;
  });
}

}  // namespace phz
