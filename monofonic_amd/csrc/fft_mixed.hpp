// fft_mixed.hpp -- mixed-radix transforms of any 7-smooth length with the
// stage schedule in kernel arguments.
//
// A line lives in ONE LDS buffer and every stage works in place: a butterfly
// reads its R slots, transforms them in registers and writes the same slots
// back, so one barrier separates two stages and the buffer is not doubled as
// a Stockham ping-pong would need.  Two orders of the same stages are used:
//
//   decimation in frequency (DIF): natural slots in, digit-reversed slots
//     out; stage s transforms the slots base + q I_s (I_s the product of the
//     later radices) and multiplies output k by W^(k i P_s) (i the butterfly's
//     offset inside its group, P_s the product of the earlier radices)
//   decimation in time (DIT): the transpose, digit-reversed slots in, natural
//     slots out; stages in reverse order, the twiddles before the butterfly
//
// The first DIF stage takes its inputs from global memory straight into the
// butterfly's registers and the last one hands its outputs over in registers,
// so a line of three stages crosses LDS twice.  A DIF stage sequence followed
// by a DIT one needs no permutation: that is how the projection (turn) passes
// and the fused real-space products run.
//
// The radix of a stage is a uniform value, so the switch over the butterflies
// is one scalar branch per stage.
//
// Against the Stockham kernels with direct odd-prime DFTs that ran these lengths
// before (fft_generic.hpp), per launch:
//   columns, y pass of 576 lines, 576 x 193 columns, FP32   528 -> 234 us (3.6 TB/s)
//   columns, y pass of 300 lines, 300 x 101 columns, FP64   164 ->  71 us (3.4 TB/s)
//   rows, r2c of 40500 rows of 300, FP64                     305 ->  48 us (4.0 TB/s)
//   rows, c2r of the same                                    294 ->  51 us (3.8 TB/s)
//   rows, product of 57600 rows of 240, FP32                 685 ->  55 us
// The column passes and the plain rows are bound by memory (runs of 64 to 128
// bytes), the products by the latency of their stages.
#pragma once
#include "fft_passes.hpp"

namespace mfx {

// ---------------------------------------------------------------- butterflies
// The butterfly that meets the raw values of a line decides how far the line's mean
// enters its longest waves: a sum of raw values is rounded at the mean's size, and
// where such sums are subtracted again the rounding stays in the output.  Radices 2,
// 4, 8 and 12 form the outputs k = +-1 from differences of values, and so do 6 and 10
// with their radix 2 first; an odd radix does it only from differences with one of
// its values (mix_first_bf: the first butterfly of a forward transform).  A line of
// mean 1 with 1 % fluctuations, 240 points in single precision, rms error of k = 1 in
// units of 2^-24 of the fluctuations: 1.3 with 8 first, 1.5 with 10 first in that form,
// 43 with a 10 whose 5-point parts take raw values.
template <int R, bool INV, typename T>
struct MixBF : BF<R, INV, T> {};

// odd prime P from the sums and differences of the pairs (a_j, a_(P-j)):
// X_k = a_0 + sum_j cos(2 pi j k / P) s_j -+ i sum_j sin(2 pi j k / P) d_j.
// The cosines of an output sum to -1/2 (c_1 + .. + c_H), so that sum c_j s_j =
// -s_H / 2 + sum c_j (s_j - s_H): with rounded constants a constant line cancels
// exactly.  FIRST: s_j from differences with a_0, X_k = sum_j c_j s_j -+ .. and
// X_0 = P a_0 + sum_j s_j; for values without a mean it rounds more (the sources of a
// 160^3 FP32 grid err by 3.2e-7 with it in every stage, 2.6e-7 without).
template <int P, bool INV, typename T, bool FIRST>
struct MixPrime {
  static __device__ __forceinline__ void run(cx<T>* a, const T* cs, const T* sn) {
    constexpr int H = (P - 1) / 2, N = FIRST ? H : H - 1;
    cx<T> s[H], d[H], o[P], base = mk(T(0), T(0));
#pragma unroll
    for (int j = 0; j < H; ++j) {
      s[j] = FIRST ? (a[j + 1] - a[0]) + (a[P - 1 - j] - a[0]) : a[j + 1] + a[P - 1 - j];
      d[j] = a[j + 1] - a[P - 1 - j];
    }
    if constexpr (FIRST) {
      cx<T> sum = s[0];
#pragma unroll
      for (int j = 1; j < H; ++j) sum = sum + s[j];
      o[0] = mk(fma(T(P), a[0].x, sum.x), fma(T(P), a[0].y, sum.y));
    } else {
      o[0] = a[0];
#pragma unroll
      for (int j = 0; j < H; ++j) o[0] = o[0] + s[j];
      base = a[0] - s[H - 1] * T(0.5);
#pragma unroll
      for (int j = 0; j < H - 1; ++j) s[j] = s[j] - s[H - 1];
    }
#pragma unroll
    for (int k = 1; k <= H; ++k) {
      cx<T> re = base, im = mk(T(0), T(0));
#pragma unroll
      for (int j = 1; j <= H; ++j) {
        const int r = (j * k) % P;  // cos is even, sin odd in r <-> P - r
        const T c = cs[r <= H ? r - 1 : P - r - 1], q = r <= H ? sn[r - 1] : -sn[P - r - 1];
        if (j <= N) re = re + s[j - 1] * c;
        im = im + d[j - 1] * q;
      }
      const cx<T> m = mul_mi<INV>(im);
      o[k] = re + m;
      o[P - k] = re - m;
    }
#pragma unroll
    for (int k = 0; k < P; ++k) a[k] = o[k];
  }
};

template <bool INV, typename T, bool FIRST>
__device__ __forceinline__ void mix3(cx<T>* a) {
  const T cs[1] = {T(-0.5)}, sn[1] = {T(0.866025403784438646763723170752936183)};
  MixPrime<3, INV, T, FIRST>::run(a, cs, sn);
}
template <bool INV, typename T, bool FIRST>
__device__ __forceinline__ void mix5(cx<T>* a) {
  const T cs[2] = {T(0.309016994374947424102293417182819), T(-0.809016994374947424102293417182819)};
  const T sn[2] = {T(0.951056516295153572116439333379382), T(0.587785252292473129168705954639073)};
  MixPrime<5, INV, T, FIRST>::run(a, cs, sn);
}
template <bool INV, typename T, bool FIRST>
__device__ __forceinline__ void mix7(cx<T>* a) {
  const T cs[3] = {T(0.623489801858733530525004884004240), T(-0.222520933956314404288902564496794),
                   T(-0.900968867902419126236102319507445)};
  const T sn[3] = {T(0.781831482468029808708444526674058), T(0.974927912181823607018131682993932),
                   T(0.433883739117558120475768332848359)};
  MixPrime<7, INV, T, FIRST>::run(a, cs, sn);
}

template <bool INV, typename T>
struct MixBF<5, INV, T> {
  static __device__ __forceinline__ void run(cx<T>* a) { mix5<INV, T, false>(a); }
};
template <bool INV, typename T>
struct MixBF<7, INV, T> {
  static __device__ __forceinline__ void run(cx<T>* a) { mix7<INV, T, false>(a); }
};

// 2 P for an odd P without inner twiddles: inputs 2 n1 + P n2, output k = k1 mod P =
// k2 mod 2.  TWO: the radix 2 first
template <int P, bool INV, typename T, bool TWO>
__device__ __forceinline__ void mix_twice(cx<T>* a) {
  cx<T> t[2][P];
#pragma unroll
  for (int n1 = 0; n1 < P; ++n1) {
    t[0][n1] = a[(2 * n1) % (2 * P)];
    t[1][n1] = a[(2 * n1 + P) % (2 * P)];
  }
  auto two = [&] {
#pragma unroll
    for (int n1 = 0; n1 < P; ++n1) {
      const cx<T> u = t[0][n1], v = t[1][n1];
      t[0][n1] = u + v;
      t[1][n1] = u - v;
    }
  };
  auto odd = [&] {
    MixBF<P, INV, T>::run(t[0]);
    MixBF<P, INV, T>::run(t[1]);
  };
  if constexpr (TWO) {
    two();
    odd();
  } else {
    odd();
    two();
  }
#pragma unroll
  for (int k2 = 0; k2 < 2; ++k2) {
#pragma unroll
    for (int k1 = 0; k1 < P; ++k1) a[k1 % 2 == k2 ? k1 : k1 + P] = t[k2][k1];
  }
}
template <bool INV, typename T>
struct MixBF<6, INV, T> {
  static __device__ __forceinline__ void run(cx<T>* a) { mix_twice<3, INV, T, false>(a); }
};
template <bool INV, typename T>
struct MixBF<10, INV, T> {
  static __device__ __forceinline__ void run(cx<T>* a) { mix_twice<5, INV, T, false>(a); }
};

// radix 9 as 3 x 3 with the inner twiddles W9^(n2 k1)
template <bool INV, typename T, bool FIRST>
__device__ __forceinline__ void mix9(cx<T>* a) {
  const cx<T> w1 = mk(T(0.766044443118978035202392650555417), T(-0.642787609686539326322643409907263)),
              w2 = mk(T(0.173648177666930348851716626769315), T(-0.984807753012208059366743024589523)),
              w4 = mk(T(-0.939692620785908384054109277324731), T(-0.342020143325668733044099614682260));
  auto three = [](cx<T>* v) {
    if constexpr (FIRST)
      mix3<INV, T, true>(v);
    else
      BF<3, INV, T>::run(v);
  };
  cx<T> t[3][3];
#pragma unroll
  for (int n2 = 0; n2 < 3; ++n2) {
#pragma unroll
    for (int n1 = 0; n1 < 3; ++n1) t[n2][n1] = a[3 * n1 + n2];
    three(t[n2]);
  }
  t[1][1] = twmul<INV>(t[1][1], w1);
  t[1][2] = twmul<INV>(t[1][2], w2);
  t[2][1] = twmul<INV>(t[2][1], w2);
  t[2][2] = twmul<INV>(t[2][2], w4);
#pragma unroll
  for (int k1 = 0; k1 < 3; ++k1) {
    cx<T> u[3] = {t[0][k1], t[1][k1], t[2][k1]};
    three(u);
#pragma unroll
    for (int k2 = 0; k2 < 3; ++k2) a[k1 + 3 * k2] = u[k2];
  }
}
template <bool INV, typename T>
struct MixBF<9, INV, T> {
  static __device__ __forceinline__ void run(cx<T>* a) { mix9<INV, T, false>(a); }
};

// the butterfly of a line's raw values: the first of a forward transform
template <int R, bool INV, typename T>
__device__ __forceinline__ void mix_first_bf(cx<T>* a) {
  if constexpr (INV)
    MixBF<R, INV, T>::run(a);
  else if constexpr (R == 3)
    mix3<INV, T, true>(a);
  else if constexpr (R == 5)
    mix5<INV, T, true>(a);
  else if constexpr (R == 7)
    mix7<INV, T, true>(a);
  else if constexpr (R == 9)
    mix9<INV, T, true>(a);
  else if constexpr (R == 6 || R == 10)
    mix_twice<R / 2, INV, T, true>(a);
  else
    MixBF<R, INV, T>::run(a);
}

// ---------------------------------------------------------------- schedule
#define MFX_MIX_RADICES(X) X(2) X(3) X(4) X(5) X(6) X(7) X(8) X(9) X(10) X(12)

// FP64 lines take no radix 12: with its 48 registers of data the row kernels
// and the operator pass spill (up to 228 bytes a lane)
template <typename T>
constexpr int MIX_RMAX = sizeof(T) == 4 ? 12 : 10;
// the fused row kernels, which hold up to twelve operands beside a butterfly
constexpr int MIX_ZMAX = 8;

// frequency of output q = 0 of the last-stage DIF butterfly b (slots b R ..);
// output q is at + q L / R
__device__ __forceinline__ int mix_freq(const MixPlan& p, int b) {
  int k = 0;
  for (int s = 0; s + 2 < p.nr; ++s) {
    const int d = p.J[s](b);
    k += d * p.P[s];
    b -= d * p.J[s].d;
  }
  return p.nr > 1 ? k + b * p.P[p.nr - 2] : 0;
}

// slot of frequency k in the digit-reversed order
__device__ __forceinline__ int mix_slot(const MixPlan& p, int k) {
  int s = 0, r = k;
  for (int q = 0; q + 1 < p.nr; ++q) {
    const int up = p.R[q](r);
    s += (r - up * p.R[q].d) * p.I[q].d;
    r = up;
  }
  return s + r;
}

// one in-place stage over a line of L slots in LDS (slot stride ls): butterflies
// t, t + nthr, ...; DIF multiplies by the twiddles after the butterfly, DIT
// before.  The stage's entries of the plan come by value: read inside the
// radix switch they are so many uses of the kernel argument that the compiler
// gives it a copy in scratch.
template <typename T, bool INV, bool DIT, int R>
__device__ __forceinline__ void mix_run(cx<T>* x, int ls, int L, MixDiv Id, int P, int t, int nthr, lcx<T>* tw) {
  const int I = Id.d, nb = L / R, step = I * ls;
  for (int b = t; b < nb; b += nthr) {
    const int o = Id(b), i = b - o * I;
    cx<T>* y = x + (o * (R * I) + i) * ls;
    cx<T> a[R];
#pragma unroll
    for (int q = 0; q < R; ++q) a[q] = y[q * step];
    if (DIT) {
#pragma unroll
      for (int q = 1; q < R; ++q) a[q] = twmul<INV>(a[q], ld(tw, q * i * P));
    }
    MixBF<R, INV, T>::run(a);
    if (!DIT && I > 1) {  // the last stage has none
#pragma unroll
      for (int q = 1; q < R; ++q) a[q] = twmul<INV>(a[q], ld(tw, q * i * P));
    }
#pragma unroll
    for (int q = 0; q < R; ++q) y[q * step] = a[q];
  }
}

// stages [s0, s1) in DIF order or, with DIT, s1-1 down to s0; a barrier ends
// every stage
template <typename T, bool INV, bool DIT, int RMAX = MIX_RMAX<T>>
__device__ __forceinline__ void mix_stages(cx<T>* x, int ls, const MixPlan& p, int s0, int s1, int t, int nthr,
                                           lcx<T>* tw) {
  const int L = p.L;
  for (int n = s0; n < s1; ++n) {
    const int s = DIT ? s0 + s1 - 1 - n : n;
    const MixDiv I = p.I[s];
    const int P = p.P[s];
    switch (p.R[s].d) {
#define MFX_CASE(R)                                                                   \
  case R:                                                                             \
    if constexpr (R <= RMAX) mix_run<T, INV, DIT, R>(x, ls, L, I, P, t, nthr, tw);    \
    break;
      MFX_MIX_RADICES(MFX_CASE)
#undef MFX_CASE
    }
    __syncthreads();
  }
}

// the first DIF stage, its inputs from load(n) (natural index n); `copy` runs
// once, after the first butterfly's loads are in flight, and brings the
// twiddle table into LDS (it ends with a barrier)
template <typename T, bool INV, int R, class Load, class Copy>
__device__ __forceinline__ void mix_first_run(cx<T>* x, int ls, const MixPlan& p, int t, int nthr, lcx<T>* tw,
                                              Load&& load, Copy&& copy) {
  const int I = p.I[0].d, step = I * ls;
  cx<T> a[R];
  const int b0 = t < I ? t : 0;
#pragma unroll
  for (int q = 0; q < R; ++q) a[q] = load(b0 + q * I);
  copy();
  for (int b = t; b < I; b += nthr) {
    if (b != t) {
#pragma unroll
      for (int q = 0; q < R; ++q) a[q] = load(b + q * I);
    }
    mix_first_bf<R, INV, T>(a);
#pragma unroll
    for (int q = 1; q < R; ++q) a[q] = twmul<INV>(a[q], ld(tw, q * b));
    cx<T>* y = x + b * ls;
#pragma unroll
    for (int q = 0; q < R; ++q) y[q * step] = a[q];
  }
}

template <typename T, bool INV, class Load, class Copy>
__device__ __forceinline__ void mix_first(cx<T>* x, int ls, const MixPlan& p, int t, int nthr, lcx<T>* tw, Load&& load,
                                          Copy&& copy) {
  switch (p.R[0].d) {
#define MFX_CASE(R)                                                \
  case R:                                                                                     \
    if constexpr (R <= MIX_RMAX<T>) mix_first_run<T, INV, R>(x, ls, p, t, nthr, tw, load, copy); \
    break;
    MFX_MIX_RADICES(MFX_CASE)
#undef MFX_CASE
  }
  __syncthreads();
}

// the last DIF stage: done(a, k, K) gets output q at frequency k + q K
template <typename T, bool INV, int R, class Done>
__device__ __forceinline__ void mix_last_run(const cx<T>* x, int ls, const MixPlan& p, int t, int nthr, Done&& done) {
  const int nb = p.L / R;
  for (int b = t; b < nb; b += nthr) {
    const cx<T>* y = x + b * R * ls;
    cx<T> a[R];
#pragma unroll
    for (int q = 0; q < R; ++q) a[q] = y[q * ls];
    MixBF<R, INV, T>::run(a);
    done(a, mix_freq(p, b), nb, std::integral_constant<int, R>{});
  }
}

template <typename T, bool INV, class Done>
__device__ __forceinline__ void mix_last(const cx<T>* x, int ls, const MixPlan& p, int t, int nthr, Done&& done) {
  switch (p.R[p.nr - 1].d) {
#define MFX_CASE(R)                                      \
  case R:                                                                           \
    if constexpr (R <= MIX_RMAX<T>) mix_last_run<T, INV, R>(x, ls, p, t, nthr, done); \
    break;
    MFX_MIX_RADICES(MFX_CASE)
#undef MFX_CASE
  }
}

// ---------------------------------------------------------------- column pass
// A workgroup transforms a tile of C = 2^lc adjacent columns of one line set,
// slot s of column c at x[s C + c]; nthr threads per column.
template <typename T>
__device__ __forceinline__ void mix_copy_table(cx<T>* lt, const cx<T>* __restrict__ tw, int L) {
  for (int i = threadIdx.x; i < L; i += blockDim.x) lt[i] = tw[i];
  __syncthreads();
}

template <typename T, bool INV, class Src, class Dst>
__global__ void __launch_bounds__(1024)
    k_mix_col(Src src, Dst dst, const cx<T>* __restrict__ tw, int ncols, MixPlan p, int lc, int nthr) {
  extern __shared__ __align__(16) unsigned char col_lds_raw[];
  cx<T>* const x = reinterpret_cast<cx<T>*>(col_lds_raw);
  cx<T>* const lt = x + (p.L << lc);
  const int C = 1 << lc;
  const int c = threadIdx.x & (C - 1), t = threadIdx.x >> lc;
  int tile, b;
  xcd_tile(tile, b);
  const int col = tile * C + c;
  const bool act = col < ncols;
  const int colc = act ? col : ncols - 1;
  lcx<T>* const ltw = lds_table(lt);
  mix_first<T, INV>(
      x + c, C, p, t, nthr, ltw, [&](int n) { return src.load(b, colc, n); },
      [&] { mix_copy_table(lt, tw, p.L); });
  mix_stages<T, INV, false>(x + c, C, p, 1, p.nr - 1, t, nthr, ltw);
  mix_last<T, INV>(x + c, C, p, t, nthr, [&](cx<T>* a, int k, int K, auto r) {
    constexpr int R = decltype(r)::value;
    cx<T> old[R];
#pragma unroll
    for (int q = 0; q < R; ++q) old[q] = dst.load_old(b, colc, k + q * K);
    if (act) {
      if constexpr (Streams<Dst>::value) {
        if (dst.nt) {
#pragma unroll
          for (int q = 0; q < R; ++q) dst.template store<true>(b, col, k + q * K, a[q], old[q]);
          return;
        }
      }
#pragma unroll
      for (int q = 0; q < R; ++q) dst.store(b, col, k + q * K, a[q], old[q]);
    }
  });
}

// projection of a padded line onto the modes of the n-grid (k_col_turn):
// the last DIF butterfly of the forward transform, the projection and the
// first DIT butterfly of the inverse one share their registers
template <typename T, int R>
__device__ __forceinline__ void mix_turn_run(cx<T>* x, int ls, const MixPlan& p, int t, int nthr, int n, bool nyqc,
                                             T fscale, T iscale) {
  const int nb = p.L / R, nh = n >> 1;
  for (int b = t; b < nb; b += nthr) {
    cx<T>* y = x + b * R * ls;
    cx<T> a[R];
#pragma unroll
    for (int q = 0; q < R; ++q) a[q] = y[q * ls];
    MixBF<R, false, T>::run(a);
    const int k0 = mix_freq(p, b);
#pragma unroll
    for (int q = 0; q < R; ++q) {
      const int k = k0 + q * nb;
      const bool zero = ((k > nh) & (k <= n)) | (k == nh) | nyqc;
      const cx<T> o = a[q] * fscale;  // the n-grid value
      a[q] = or_zero(!zero, o * iscale);
    }
    MixBF<R, true, T>::run(a);
#pragma unroll
    for (int q = 0; q < R; ++q) y[q * ls] = a[q];
  }
}

// the last DIT stage (s = 0) with its outputs to done(a, n, K): natural index
// n + q K
template <typename T, bool INV, int R, class Done>
__device__ __forceinline__ void mix_end_run(const cx<T>* x, int ls, const MixPlan& p, int t, int nthr, lcx<T>* tw,
                                            Done&& done) {
  const int I = p.I[0].d, step = I * ls;
  for (int b = t; b < I; b += nthr) {
    const cx<T>* y = x + b * ls;
    cx<T> a[R];
#pragma unroll
    for (int q = 0; q < R; ++q) a[q] = y[q * step];
#pragma unroll
    for (int q = 1; q < R; ++q) a[q] = twmul<INV>(a[q], ld(tw, q * b));
    MixBF<R, INV, T>::run(a);
    done(a, b, I, std::integral_constant<int, R>{});
  }
}

template <typename T, class TurnA>
__global__ void __launch_bounds__(1024)
    k_mix_turn(TurnA a, const cx<T>* __restrict__ tw, int ncols, MixPlan p, int lc, int nthr) {
  extern __shared__ __align__(16) unsigned char col_lds_raw[];
  cx<T>* const x = reinterpret_cast<cx<T>*>(col_lds_raw);
  cx<T>* const lt = x + (p.L << lc);
  const int C = 1 << lc;
  const int c = threadIdx.x & (C - 1), t = threadIdx.x >> lc;
  int tile, b;
  xcd_tile(tile, b);
  const int col = tile * C + c;
  const bool act = col < ncols;
  const int colc = act ? col : ncols - 1;
  lcx<T>* const ltw = lds_table(lt);
  const cx<T>* const src = a.from(b) + colc;
  mix_first<T, false>(
      x + c, C, p, t, nthr, ltw, [&](int n) { return src[(long long)n * a.sp]; },
      [&] { mix_copy_table(lt, tw, p.L); });
  mix_stages<T, false, false>(x + c, C, p, 1, p.nr - 1, t, nthr, ltw);
  switch (p.R[p.nr - 1].d) {
#define MFX_CASE(R)                                                                              \
  case R:                                                                                   \
    if constexpr (R <= MIX_RMAX<T>)                                                         \
      mix_turn_run<T, R>(x + c, C, p, t, nthr, a.n, colc == a.n / 2, a.fscale, a.iscale);   \
    break;
    MFX_MIX_RADICES(MFX_CASE)
#undef MFX_CASE
  }
  __syncthreads();
  mix_stages<T, true, true>(x + c, C, p, 1, p.nr - 1, t, nthr, ltw);
  cx<T>* const out = a.to(b) + col;
  auto done = [&](cx<T>* v, int k, int K, auto r) {
    constexpr int R = decltype(r)::value;
    if (act) {
      if (a.nt) {
#pragma unroll
        for (int q = 0; q < R; ++q) put<true>(out + (long long)(k + q * K) * a.osp, v[q]);
      } else {
#pragma unroll
        for (int q = 0; q < R; ++q) out[(long long)(k + q * K) * a.osp] = v[q];
      }
    }
  };
  switch (p.R[0].d) {
#define MFX_CASE(R)                                                     \
  case R:                                                                                    \
    if constexpr (R <= MIX_RMAX<T>) mix_end_run<T, true, R>(x + c, C, p, t, nthr, ltw, done); \
    break;
    MFX_MIX_RADICES(MFX_CASE)
#undef MFX_CASE
  }
}

// ---------------------------------------------------------------- rows (z axis)
// Two real rows A and B are one complex line A + i B of the full length M: its
// transform needs no half-length split step, no second twiddle table and no
// even M / 2, and a workgroup holds `pairs` such lines.  The half spectra
// combine as Z[k] = A[k] + i B[k], Z[M - k] = conj(A[k]) + i conj(B[k]).  The price is
// precision of the smaller row: both are rounded at the size of the larger one (rows
// of a pair are neighbours of a field), and taking them apart rounds once more.
struct MixRowArgs {
  MixPlan p;
  MixDiv nthr;  // threads per pair
  int pairs;
  long long nrows;
};

// A thread's place: pair, its rows, and t, its index among the pair's threads
// (at least M for the threads beyond the last pair, which then own nothing).
// A pair past the end reads the workgroup's first row and stores nothing.
template <typename T>
struct MixRow {
  int t, nthr;
  cx<T>* x;
  lcx<T>* tw;
  cx<T>* lt;
  long long first, ra, rb;  // the workgroup's first row, the pair's rows
  bool actA, actB;
  __device__ __forceinline__ MixRow(const MixRowArgs& a, cx<T>* lds) {
    nthr = a.nthr.d;
    int pr = a.nthr((int)threadIdx.x);
    t = (int)threadIdx.x - pr * nthr;
    if (pr >= a.pairs) {
      pr = 0;
      t = a.p.L;
    }
    first = 2LL * a.pairs * blockIdx.x;
    ra = first + 2 * pr;
    rb = ra + 1;
    actA = ra < a.nrows;
    actB = rb < a.nrows;
    if (!actA) ra = first;
    if (!actB) rb = ra;
    x = lds + pr * a.p.L;
    lt = lds + a.pairs * a.p.L;
    tw = lds_table(lt);
  }
};

// Entry k of the two half spectra (scaled by f) goes to the line's places k and
// M - k; the imaginary parts of the zero and the Nyquist entry do not enter.
template <typename T>
__device__ __forceinline__ void mix_put(cx<T>* x, int M, int k, cx<T> a, cx<T> b, T f) {
  a = a * f;
  b = b * f;
  if (k == 0 || 2 * k == M) {
    x[k] = mk(a.x, b.x);
  } else {
    x[k] = mk(a.x - b.y, a.y + b.x);
    x[M - k] = mk(a.x + b.y, b.x - a.y);
  }
}

template <typename T>
struct MixOne {
  __device__ __forceinline__ T operator()(int) const { return T(1); }
};

// entry k < hout of both rows' half spectra from the transform F of A + i B,
// slot(k) its place
template <typename T, class Slot>
__device__ __forceinline__ void mix_unpack(const MixRow<T>& r, int t, int M, int hout, T scale, cx<T>* da, cx<T>* db,
                                           Slot&& slot) {
  for (int k = t; k < hout; k += r.nthr) {
    const cx<T> f = r.x[slot(k)], g = conj(r.x[slot(k ? M - k : 0)]);
    const cx<T> e = (f + g) * T(0.5), d = (f - g) * T(0.5);
    if (r.actA) da[k] = e * scale;
    if (r.actB) db[k] = mk(d.y, -d.x) * scale;
  }
}

template <typename T>
__global__ void __launch_bounds__(512)
    k_mix_r2c(const T* src, long long spitch, cx<T>* dst, long long dpitch, int hout, T scale, MixRowArgs a,
              const cx<T>* __restrict__ tw) {
  extern __shared__ __align__(16) unsigned char col_lds_raw[];
  const MixRow<T> r(a, reinterpret_cast<cx<T>*>(col_lds_raw));
  const MixPlan& p = a.p;
  const T *sa = src + r.ra * spitch, *sb = src + r.rb * spitch;
  mix_first<T, false>(
      r.x, 1, p, r.t, r.nthr, r.tw, [&](int n) { return mk(sa[n], sb[n]); },
      [&] { mix_copy_table(r.lt, tw, p.L); });
  mix_stages<T, false, false>(r.x, 1, p, 1, p.nr, r.t, r.nthr, r.tw);
  mix_unpack(r, r.t, p.L, hout, scale, dst + r.ra * dpitch, dst + r.rb * dpitch, [&](int k) { return mix_slot(p, k); });
}

template <typename T, int R, class Done>
__device__ __forceinline__ void mix_last_rows(const MixRow<T>& r, const MixPlan& p, Done&& done) {
  const int nb = p.L / R;
  for (int k = r.t; k < nb; k += r.nthr) {
    const cx<T>* y = r.x + mix_slot(p, k);
    cx<T> v[R];
#pragma unroll
    for (int q = 0; q < R; ++q) v[q] = y[q];
    MixBF<R, true, T>::run(v);
#pragma unroll
    for (int q = 0; q < R; ++q) done(v[q], k + q * nb);
  }
}

// c2r up to its last stage, whose outputs (points k + q K of both rows, lanes
// along k) go to done
template <typename T, class Done>
__device__ __forceinline__ void mix_c2r_rows(const MixRow<T>& r, const MixPlan& p, const cx<T>* A, const cx<T>* B,
                                             int hin, const cx<T>* __restrict__ tw, Done&& done) {
  // all hin = M/2 + 1 entries are stored
  for (int k = r.t; k < hin; k += r.nthr) mix_put(r.x, p.L, k, A[k], B[k], T(1));
  mix_copy_table(r.lt, tw, p.L);
  mix_stages<T, true, false>(r.x, 1, p, 0, p.nr - 1, r.t, r.nthr, r.tw);
  switch (p.R[p.nr - 1].d) {
#define MFX_CASE(R)                                                                      \
  case R:                                                                                \
    if constexpr (R <= MIX_RMAX<T>) mix_last_rows<T, R>(r, p, done);                     \
    break;
    MFX_MIX_RADICES(MFX_CASE)
#undef MFX_CASE
  }
}

template <typename T>
__global__ void __launch_bounds__(512)
    k_mix_c2r(const cx<T>* src, long long spitch, int hin, T* dst, long long dpitch, T scale, MixRowArgs a,
              const cx<T>* __restrict__ tw) {
  extern __shared__ __align__(16) unsigned char col_lds_raw[];
  const MixRow<T> r(a, reinterpret_cast<cx<T>*>(col_lds_raw));
  const int M = a.p.L;
  T *da = dst + r.ra * dpitch, *db = dst + r.rb * dpitch;
  mix_c2r_rows<T>(r, a.p, src + r.ra * spitch, src + r.rb * spitch, hin, tw, [&](cx<T> v, int k) {
    if (r.actA) da[k] = v.x * scale;
    if (r.actB) db[k] = v.y * scale;
  });
  // the two padding reals of an in-place row
  if (dpitch >= M + 2)
    for (int q = r.t; q < 2; q += r.nthr) {
      if (r.actA) da[M + q] = T(0);
      if (r.actB) db[M + q] = T(0);
    }
}

// c2r writing FP64 particles (see k_row_c2r_part); n is even, so both rows of a
// pair belong to one component
template <typename T>
__global__ void __launch_bounds__(512)
    k_mix_c2r_part(const cx<T>* src, long long spitch, int hin, PartOut po, T scale, double lunit, double qoff,
                   MixRowArgs a, const cx<T>* __restrict__ tw) {
  extern __shared__ __align__(16) unsigned char col_lds_raw[];
  const MixRow<T> r(a, reinterpret_cast<cx<T>*>(col_lds_raw));
  const int n = a.p.L;
  const int w = (int)(r.ra / ((long long)n * n)), code = po.code(w), idim = code & 3, kind = code >> 2;
  auto qrow = [&](long long row) {
    return (double)(idim == 0 ? (int)(row / n) - w * n : (int)(row % n)) / (double)n * lunit + qoff;
  };
  const double qa = qrow(r.ra), qb = qrow(r.rb);
  double* const o = po.array(w) - (long long)w * n * n * n;
  double *oa = o + r.ra * n, *ob = o + r.rb * n;
  mix_c2r_rows<T>(r, a.p, src + r.ra * spitch, src + r.rb * spitch, hin, tw, [&](cx<T> v, int k) {
    double fa = (double)(v.x * scale), fb = (double)(v.y * scale);
    if (kind == 0) {
      const double q = (double)k / (double)n * lunit + qoff;
      fa = (idim == 2 ? q : qa) + fa;
      fb = (idim == 2 ? q : qb) + fb;
    }
    if (r.actA) oa[k] = fa;
    if (r.actB) ob[k] = fb;
  });
}

// ---------------------------------------------------------------- fused rows
// The real-space products: every thread owns one butterfly of the fixed last
// radix S = MIX_S (threads per pair = M / S), so after a c2r it holds S points
// of both rows in registers, at the same places for every operand; products
// are formed there, and a product's r2c starts with the same butterfly in DIT
// order, from the registers.
template <typename T>
struct MixZ {
  static constexpr int S = MIX_S<T>;
  const MixRow<T>& r;
  const MixPlan& p;
  // The thread index passes through an empty asm statement for every
  // transform: the kernels loop over their transforms, and without it the
  // slot and wave-number arithmetic of every radix is hoisted out of the loop
  // and held in registers (256 VGPRs and scratch).
  __device__ __forceinline__ int thread() const {
    int t = r.t;
    asm volatile("" : "+v"(t));
    return t;
  }
  // An operand has n/2 + 1 = M/3 + 1 entries, which is NK - 1 for each thread
  // and the Nyquist one: they are fetched into registers one transform ahead.
  static constexpr int NK = S / 3 + 1;
  struct Raw {
    cx<T> a[NK], b[NK];
  };
  // y: the operand's array (uniform)
  __device__ __forceinline__ void fetch(Raw& w, const cx<T>* y, long long pitch) const {
    const cx<T>* base = y + r.first * pitch;  // uniform; the lanes add 32-bit offsets
    const unsigned oa = (unsigned)((int)(r.ra - r.first) * (int)pitch), ob = (unsigned)((int)(r.rb - r.first) * (int)pitch);
    const int t = r.t < r.nthr ? r.t : 0;
#pragma unroll
    for (int q = 0; q < NK; ++q) {
      const unsigned k = (unsigned)(q + 1 < NK ? t + q * r.nthr : (NK - 1) * r.nthr);
      w.a[q] = base[oa + k];
      w.b[q] = base[ob + k];
    }
  }
  // the pair's S points per thread of the fetched operand times mul(k); the
  // line is free (a barrier has passed)
  template <class Mul>
  __device__ __forceinline__ void c2r(cx<T> (&v)[S], const Raw& w, Mul&& mul) const {
    const int t = thread(), M = p.L;
    if (t < r.nthr) {
#pragma unroll
      for (int q = 0; q + 1 < NK; ++q) mix_put(r.x, M, t + q * r.nthr, w.a[q], w.b[q], mul(t + q * r.nthr));
      if (t == 0) mix_put(r.x, M, (NK - 1) * r.nthr, w.a[NK - 1], w.b[NK - 1], mul((NK - 1) * r.nthr));
      // the entries above the Nyquist one are zero: places n/2 + 1 .. n - 1
#pragma unroll
      for (int q = 0; q + 1 < NK; ++q) {
        const int k = (NK - 1) * r.nthr + 1 + t + q * r.nthr;
        if (k < 2 * (NK - 1) * r.nthr) r.x[k] = mk(T(0), T(0));
      }
    }
    __syncthreads();
    mix_stages<T, true, false, MIX_ZMAX>(r.x, 1, p, 0, p.nr - 1, t, r.nthr, r.tw);
    const int b = t < r.nthr ? t : 0;
#pragma unroll
    for (int q = 0; q < S; ++q) v[q] = r.x[b * S + q];
    MixBF<S, true, T>::run(v);
    __syncthreads();
  }
  // r2c of the points w into the first hout entries of both rows
  __device__ __forceinline__ void r2c(const cx<T> (&w)[S], cx<T>* da, cx<T>* db, int hout) const {
    cx<T> v[S];
#pragma unroll
    for (int q = 0; q < S; ++q) v[q] = w[q];
    // FP32 products come without their mean (launch_row_mean); the engine's rows have
    // none, or one of the size of their fluctuations
    if constexpr (S % 2 == 1)
      mix_first_bf<S, false, T>(v);
    else
      MixBF<S, false, T>::run(v);
    const int t = thread();
    if (t < r.nthr) {
#pragma unroll
      for (int q = 0; q < S; ++q) r.x[t * S + q] = v[q];
    }
    __syncthreads();
    mix_stages<T, false, true, MIX_ZMAX>(r.x, 1, p, 0, p.nr - 1, t, r.nthr, r.tw);
    mix_unpack(r, t, p.L, hout, T(1), da, db, [](int k) { return k; });
    __syncthreads();
  }
};

template <typename T>
__device__ __forceinline__ cx<T> mix_pmul(cx<T> a, cx<T> b) {
  return mk(a.x * b.x, a.y * b.y);
}

// The mean of a product of the m x m rows of two half spectra, from MIX_MEAN_ROWS of
// them on a lattice: a row's mean is Re(a_0) Re(b_0) + 2 sum Re(a_k conj(b_k)).  One
// workgroup, two rows a wave, whose loads are all in flight together.
constexpr int MIX_MEAN_ROWS = 32;
template <typename T>
__global__ void __launch_bounds__(1024)
    k_mix_mean(const cx<T>* a, const cx<T>* b, long long spitch, int hin, int m, T* mean) {
  __shared__ T part[16];
  constexpr int N = MIX_MEAN_ROWS, U = 4;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const cx<T>*u[N / 16], *v[N / 16];
#pragma unroll
  for (int q = 0; q < N / 16; ++q) {
    const int s = wave + 16 * q;
    const long long row = ((long long)(s * m / N) * m + (19 * s) % N * m / N) * spitch;
    u[q] = a + row;
    v[q] = b + row;
  }
  T sum = 0;
  for (int k0 = lane; k0 < hin; k0 += 64 * U) {
    cx<T> x[N / 16][U], y[N / 16][U];
#pragma unroll
    for (int q = 0; q < N / 16; ++q)
#pragma unroll
      for (int e = 0; e < U; ++e) {
        const int k = k0 + 64 * e < hin ? k0 + 64 * e : hin - 1;
        x[q][e] = u[q][k];
        y[q][e] = v[q][k];
      }
#pragma unroll
    for (int q = 0; q < N / 16; ++q)
#pragma unroll
      for (int e = 0; e < U; ++e) {
        const int k = k0 + 64 * e;
        const T re = x[q][e].x * y[q][e].x, im = x[q][e].y * y[q][e].y;
        sum += pick(k == 0, re, pick(k < hin, T(2) * (re + im), T(0)));
      }
  }
  sum = sum * (T(1) / T(N));
#pragma unroll
  for (int d = 32; d > 0; d >>= 1) sum += __shfl_down(sum, d);
  if (lane == 0) part[wave] = sum;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < 16; ++w) sum += part[w];
    *mean = sum;
  }
}

// P3: c2r of two half spectra, pointwise product less *mean (if not null), r2c
template <typename T>
__global__ void __launch_bounds__(512)
    k_mix_prod(const cx<T>* a, const cx<T>* b, long long spitch, cx<T>* dst, long long dpitch, int hout,
               const T* mean, MixRowArgs ra, const cx<T>* __restrict__ tw) {
  extern __shared__ __align__(16) unsigned char col_lds_raw[];
  const MixRow<T> r(ra, reinterpret_cast<cx<T>*>(col_lds_raw));
  const MixZ<T> z{r, ra.p};
  cx<T> u[MixZ<T>::S], v[MixZ<T>::S];
  typename MixZ<T>::Raw wa, wb;
  z.fetch(wa, a, spitch);
  z.fetch(wb, b, spitch);
  mix_copy_table(r.lt, tw, ra.p.L);
  z.c2r(u, wa, MixOne<T>{});
  z.c2r(v, wb, MixOne<T>{});
#pragma unroll
  for (int q = 0; q < MixZ<T>::S; ++q) u[q] = mix_pmul(u[q], v[q]);
  if (mean) {
    const T c = *mean;
#pragma unroll
    for (int q = 0; q < MixZ<T>::S; ++q) u[q] = u[q] - mk(c, c);
  }
  z.r2c(u, dst + r.ra * dpitch, dst + r.rb * dpitch, hout);
}

}  // namespace mfx
