// fft_passes.hpp -- pass-level building blocks shared by the FFT, Orszag and
// LPT-engine translation units: launch configuration, line sources/sinks
// (plain, zero-padded with Fourier multiplier, truncating, output operator),
// the column kernel over tiles of adjacent columns and the z-row kernels
// (r2c, c2r, fused c2r-product-r2c).
#pragma once
#include "mfx_internal.hpp"
#include "ops.hpp"
#include "row_fft.hpp"

#include <cmath>
#include <cstdint>
#include <string>
#include <type_traits>

namespace mfx {

// ------------------------------------------------------------------ config
constexpr int CU_LDS = 160 * 1024;  // LDS of a compute unit

// Tile widths of a column pass of length L (plan variant V): C, the widest
// tile (at most 16 columns) whose exchange area fits 64 KiB of LDS, and CW =
// 2C where C < 16 and a tile of 2C columns still fits one workgroup (1024
// threads; exchanged in two parts, TwLds), else 0.  Wider tiles read longer runs
// of each line (2C complex values).
template <typename T, int L, int V = 0>
struct ColCfg {
  static constexpr int TPS = PlanInfo<L, V>::TPS;
  static constexpr int lim_lds = 65536 / (L * (int)sizeof(cx<T>));
  static constexpr int lim_thr = 1024 / TPS;
  static constexpr int lim = (lim_lds < lim_thr ? lim_lds : lim_thr) < 16 ? (lim_lds < lim_thr ? lim_lds : lim_thr) : 16;
  static constexpr int C = lim >= 16 ? 16 : lim >= 8 ? 8 : lim >= 4 ? 4 : lim >= 2 ? 2 : 1;
  static constexpr int CW =
      (C < 16 && 2 * C * TPS <= 1024 && TwLds<T, L, 2 * C, V>::bytes <= (size_t)160 * 1024) ? 2 * C : 0;
};


// ------------------------------------------------------------------ sources / sinks
template <typename T>
__device__ __forceinline__ T kval(int i, int n, T kfac, int nyq) {
  // grid_fft.hh:282-296 (get_k) and 376-385 (gradient, zero at n/2)
  if (nyq && i == (n >> 1)) return T(0);
  return (T(i) - T(i > (n >> 1)) * T(n)) * kfac;
}

template <typename T>
struct MultDev {
  int nterms;
  T cre[2], cim[2];
  int pw[2][3];
  int nyq[2];
  __device__ __forceinline__ cx<T> eval(int i, int j, int k, int n, T kfac) const {
    T sr = 0, si = 0;
    const int idx[3] = {i, j, k};
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      if (t >= nterms) break;
      T f = 1;
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        T kd = kval<T>(idx[d], n, kfac, nyq[t]);
        for (int p = 0; p < pw[t][d]; ++p) f *= kd;
      }
      sr += cre[t] * f;
      si += cim[t] * f;
    }
    return mk(sr, si);
  }
};

template <typename T>
MultDev<T> to_dev(const MultSpec& m) {
  MultDev<T> d;
  d.nterms = m.nterms;
  for (int t = 0; t < 2; ++t) {
    d.cre[t] = T(m.coef_re[t]);
    d.cim[t] = T(m.coef_im[t]);
    d.nyq[t] = m.nyq[t];
    for (int q = 0; q < 3; ++q) d.pw[t][q] = m.pow[t][q];
  }
  return d;
}

// Position t + c of a line: in the tuned column kernels c = W e is the constant of
// a thread's element e (W threads a line of L positions), so that a line's
// address is formed once for each thread and an element adds a uniform stride,
// and what depends on the range c .. c + W - 1 is decided when the kernel is
// compiled.  From a plain position (the run-time kernels) W = 0.
struct Pos {
  int t, c, W, L;
  __device__ __forceinline__ Pos(int p) : t(p), c(0), W(0), L(0) {}
  __device__ __forceinline__ Pos(int t_, int c_, int W_, int L_) : t(t_), c(c_), W(W_), L(L_) {}
  __device__ __forceinline__ operator int() const { return t + c; }
};

// Streaming (non-temporal) stores of a column pass: only where every line of a
// tile of C columns is whole 128-byte cache lines (run C*sizeof(cx), base and
// strides all multiples of 128 bytes, as in the padded work grids); a partial
// line stored past the L2 costs a read and write of the whole line.  Plain passes
// of 257 columns (FP32; GB/s without -> with): 768 lines, pitch 272, 16 columns:
// out of place 4627 -> 5232 (y), 4154 -> 4669 (x), in place 4111 -> 4731, 3834 ->
// 4343; 8 columns (64-byte runs) 4313 -> 4088; 512 lines, pitch 257: 4982 -> 2616.
// FP64, 384 lines, 8 columns in place (y) 5201 -> 6678.
inline bool streams(const void* p, int C, long long sb, long long sp, size_t size) {
  return (C * size) % 128 == 0 && ((unsigned long long)sb * size) % 128 == 0 &&
         ((unsigned long long)sp * size) % 128 == 0 && (reinterpret_cast<uintptr_t>(p) & 127) == 0;
}

template <bool NT, typename T>
__device__ __forceinline__ void put(cx<T>* p, cx<T> v) {
  if constexpr (NT) {
    typedef T pair __attribute__((ext_vector_type(2)));
    __builtin_nontemporal_store(pair{v.x, v.y}, reinterpret_cast<pair*>(p));
  } else {
    *p = v;
  }
}

// Whether a destination has a streaming form: a flag nt, set by stream(C) at the
// launch, and store<true>.
template <class D, class = void>
struct Streams {
  static constexpr bool value = false;
};
template <class D>
struct Streams<D, std::void_t<decltype(&D::stream)>> {
  static constexpr bool value = true;
};
template <class D>
void set_stream(D& d, int C) {
  if constexpr (Streams<D>::value) d.stream(C);
}

// element t + c of a line: column col of line set base (uniform), line stride sp
template <typename C>
__device__ __forceinline__ C* line_at(C* base, long long sp, int col, int t, int c) {
  return base + ((long long)t * sp + col) + (long long)c * sp;
}

// Position of a line padded from n to 3n/2: kept positions hold index t + c of the
// n-grid, whose signed wave index is t + k0 (n/2 positive); the others are zero.
// drop(): no position of the element's range is kept.
struct Kept {
  bool keep, nyq;
  int t, c, k0;
  static __device__ __forceinline__ bool drop(const Pos& p) {
    return p.W && p.c > p.L / 3 && p.c + p.W - 1 <= 2 * (p.L / 3);
  }
  __device__ __forceinline__ Kept(const Pos& p, int n) {
    const int m = p.W ? 2 * (p.L / 3) : n, nh = m >> 1;
    if (p.W && p.c + p.W - 1 < nh) {
      keep = true;
      nyq = false;
      t = p.t;
      c = k0 = p.c;
    } else if (p.W && p.c == nh && p.c + p.W - 1 <= m) {
      // the Nyquist position and padding: every lane addresses the former
      keep = nyq = p.t == 0;
      t = 0;
      c = k0 = nh;
    } else if (p.W && p.c >= m) {
      keep = p.c > m || p.t != 0;
      nyq = false;
      t = p.t;
      c = p.c - nh;
      k0 = p.c - (m + nh);
    } else {
      const int q = p.t + p.c;
      const bool pad = (q > nh) & (q <= m);
      keep = !pad;
      t = pad ? 0 : (q <= nh ? q : q - nh);
      c = 0;
      nyq = t == nh;
      k0 = t > nh ? -m : 0;
    }
  }
};

// v or zero by selects on values: a conditional expression of complex type is
// compiled to a branch around the load of v, and the loads of a thread are then
// waited for one by one (the y stage at 576 lines, FP32: 3.7 instead of 2.8 ms)
template <typename T>
__device__ __forceinline__ T pick(bool c, T a, T b) {
  return c ? a : b;
}
template <typename T>
__device__ __forceinline__ cx<T> or_zero(bool keep, cx<T> v) {
  return mk(pick(keep, v.x, T(0)), pick(keep, v.y, T(0)));
}

template <typename T>
struct SrcPlain {
  const cx<T>* p;
  long long sb, sp;
  __device__ __forceinline__ cx<T> load(int b, int col, Pos pos) const {
    return *line_at(p + (long long)b * sb, sp, col, pos.t, pos.c);
  }
};

// lines of several equal arrays in one launch: batch b is line set b % nb of
// array b / nb, the arrays sq apart
template <typename T>
struct SrcSplit {
  const cx<T>* p;
  long long sb, sp, sq;
  int nb;
  __device__ __forceinline__ cx<T> load(int b, int col, Pos pos) const {
    const int q = b / nb;
    return *line_at(p + (long long)q * sq + (long long)(b - q * nb) * sb, sp, col, pos.t, pos.c);
  }
};

template <typename T>
struct DstPlain {
  cx<T>* p;
  long long sb, sp;
  T scale;
  int nt = 0;
  void stream(int C) { nt = streams(p, C, sb, sp, sizeof(cx<T>)); }
  __device__ __forceinline__ cx<T> load_old(int, int, int) const { return mk(T(0), T(0)); }
  template <bool NT = false>
  __device__ __forceinline__ void store(int b, int col, Pos pos, cx<T> v, cx<T>) const {
    put<NT>(line_at(p + (long long)b * sb, sp, col, pos.t, pos.c), v * scale);
  }
};

// line of an n-grid zero-padded to M = 3n/2: position pos <- source index
// pos (pos <= n/2) or pos - n/2 (pos > n); convolution.hh:569-592
template <typename T, bool MULT>
struct SrcPad {
  const cx<T>* p;
  long long sb, sp;
  int n;
  T scale;
  T kfac;
  MultDev<T> m;  // used when MULT: line axis = x (i), b = y (j), col = kz
  // The load is unconditional (index clamped into the line) and the padding
  // is applied by a select, so all loads of a thread can be in flight at once.
  __device__ __forceinline__ cx<T> load(int b, int col, Pos pos) const {
    if (Kept::drop(pos)) return mk(T(0), T(0));
    const Kept k(pos, n);
    cx<T> v = *line_at(p + (long long)b * sb, sp, col, k.t, k.c);
    if (MULT) v = cmul(v, m.eval(k.t + k.c, b, col, n, kfac));
    return or_zero(k.keep, v * scale);
  }
};

// zero-padded line times g(i)^pw with g the Nyquist-zeroed gradient wave
// number of the source index i (one Hessian factor per transformed axis)
template <typename T>
struct SrcPadPow {
  const cx<T>* p;
  long long sb, sp;
  int n, pw;
  T scale, kfac;
  __device__ __forceinline__ cx<T> load(int b, int col, Pos pos) const {
    if (Kept::drop(pos)) return mk(T(0), T(0));
    const Kept k(pos, n);
    const cx<T> x = *line_at(p + (long long)b * sb, sp, col, k.t, k.c);
    const T g = pick(k.nyq, T(0), T(k.t + k.k0) * kfac);
    const T f1 = pick(pw == 0, scale, scale * g);
    const T f = pick(pw == 2, f1 * g, f1);
    return or_zero(k.keep, x * f);
  }
};

// The y stage of a field's Hessian rows in one launch: batch b is output b % 6
// of x-plane b / 6.  Outputs 0..2 are the powers 0, 1, 2 of g_y of X_0, 3 and 4
// the powers 0, 1 of X_1, 5 is X_2.  The outputs of a plane that share their
// source follow one another on an XCD, a plane (1.1 MB at n = 512, FP32) apart.
// One launch instead of six: 96^3 FP64 75 -> 47 us for a field, 256^3 FP64 0.82 ->
// 0.67 ms, 512^3 FP32 2.80 -> 2.75 ms (2.00 with streaming stores).
template <typename T>
struct SrcHessY {
  const cx<T>* x[3];
  long long sb, sp;
  int n;
  T kfac;
  __device__ __forceinline__ cx<T> load(int b, int col, Pos pos) const {
    const int plane = b / 6, o = b - 6 * plane;
    const cx<T>* p = o < 3 ? x[0] : (o < 5 ? x[1] : x[2]);
    const int pw = o < 3 ? o : (o == 4 ? 1 : 0);
    return SrcPadPow<T>{p, sb, sp, n, pw, T(1), kfac}.load(plane, col, pos);
  }
};
template <typename T>
struct DstHessY {
  cx<T>* y[6];
  long long sb, sp;
  int nt = 0;
  void stream(int C) {
    nt = 1;
    for (cx<T>* q : y) nt &= streams(q, C, sb, sp, sizeof(cx<T>));
  }
  __device__ __forceinline__ cx<T> load_old(int, int, int) const { return mk(T(0), T(0)); }
  template <bool NT = false>
  __device__ __forceinline__ void store(int b, int col, Pos pos, cx<T> v, cx<T>) const {
    const int plane = b / 6, o = b - 6 * plane;
    cx<T>* p = o < 2 ? (o == 0 ? y[0] : y[1]) : (o < 4 ? (o == 2 ? y[2] : y[3]) : (o == 4 ? y[4] : y[5]));
    put<NT>(line_at(p + (long long)plane * sb, sp, col, pos.t, pos.c), v);
  }
};

// keep the n retained outputs of an M-line (convolution.hh:629-634)
template <typename T>
struct DstTrunc {
  cx<T>* p;
  long long sb, sp;
  int n;
  int nt = 0;
  void stream(int C) { nt = streams(p, C, sb, sp, sizeof(cx<T>)); }
  __device__ __forceinline__ cx<T> load_old(int, int, int) const { return mk(T(0), T(0)); }
  template <bool NT = false>
  __device__ __forceinline__ void store(int b, int col, Pos pos, cx<T> v, cx<T>) const {
    if (Kept::drop(pos)) return;
    const Kept k(pos, n);
    if (k.keep) put<NT>(line_at(p + (long long)b * sb, sp, col, k.t, k.c), v);
  }
};

// final x pass: truncation, Nyquist zeroing (convolution.hh:637-643), scale
// and the output operator on the flat k-space array (operators.hh:25-35)
template <typename T>
struct DstTruncOp {
  cx<T>* out[4];     // batch b is line set b % nb of output array b / nb
  int nb;
  long long sb, sp;  // line set (j) stride, pos (i) stride (complex units)
  int n;
  int op;
  T opfac, scale;
  int invlap;  // fold apply_InverseLaplacian (grid_fft.hh:440-449)
  T kfac;
  __device__ __forceinline__ cx<T>* array(int q) const {
    return q < 2 ? (q == 0 ? out[0] : out[1]) : (q == 2 ? out[2] : out[3]);
  }
  // previous output value for the accumulating operators, loaded for every
  // element of the thread before any store (clamped index, no branch)
  __device__ __forceinline__ cx<T> load_old(int b, int col, Pos pos) const {
    if (op == OP_ASSIGN || Kept::drop(pos)) return mk(T(0), T(0));
    const Kept k(pos, n);
    const int q = b / nb;
    return *line_at(array(q) + (long long)(b - q * nb) * sb, sp, col, k.t, k.c);
  }
  // The value is formed without a branch and only its store is predicated: what
  // does not depend on the element is then computed once for each thread.
  __device__ __forceinline__ void store(int b, int col, Pos pos, cx<T> v, cx<T> prev) const {
    if (Kept::drop(pos)) return;
    const Kept k(pos, n);
    const int nh = n >> 1, q = b / nb, j = b - q * nb;
    const bool nyq = k.nyq | (j == nh) | (col == nh);
    const T w = op == OP_SUB ? T(-1) : (op == OP_MULADD ? opfac : T(1));
    const cx<T> val = or_zero(!nyq, v * scale);
    cx<T> o = prev + val * w;  // prev is zero for the assignment
    if (invlap) {
      const T ky = kval<T>(j, n, kfac, 0), kz = kval<T>(col, n, kfac, 0), kx = T(k.t + k.k0) * kfac;
      const T k2 = kx * kx + ky * ky + kz * kz;
      const bool dc = (k.t + k.c == 0) & (j == 0) & (col == 0);
      o = or_zero(!dc, mk(-o.x / k2, -o.y / k2));
    }
    if (k.keep) *line_at(array(q) + (long long)j * sb, sp, col, k.t, k.c) = o;
  }
};

// DstTruncOp of one array for a product transformed without (nearly all of) its
// mean: *mean times the number of points goes back to the k = 0 mode
template <typename T>
struct DstTruncOpMean : DstTruncOp<T> {
  const T* mean;
  T count;
  __device__ __forceinline__ void store(int b, int col, Pos pos, cx<T> v, cx<T> prev) const {
    const bool dc = ((int)pos == 0) & (b == 0) & (col == 0);
    DstTruncOp<T>::store(b, col, pos, mk(v.x + pick(dc, *mean * count, T(0)), v.y), prev);
  }
};

// The last (x) pass of the noise's forward transform writing phi(1) instead
// of the k-space noise (ic_generator.cc:341-346,450-457): each transformed
// value is scaled as the plain pass would store it (rounded to T) and turned
// into phi(1) by the same per-mode function the phi(1) kernel uses, so the
// result is bit-identical to transform-then-phi(1).  Lines along x (pos = i),
// column j H + kz.
template <typename T>
struct DstPhi1 {
  cx<T>* phi;
  long long sp;
  int n, H;
  T scale;
  double kfac;
  const double* amp;
  NoiseNorm nn;
  __device__ __forceinline__ cx<T> load_old(int, int, int) const { return mk(T(0), T(0)); }
  __device__ __forceinline__ void store(int, int col, Pos pos, cx<T> v, cx<T>) const {
    const int j = col / H;
    *line_at(phi, sp, col, pos.t, pos.c) = phi1_value(v * scale, pos, j, col - j * H, n, kfac, amp, nn);
  }
};

// ------------------------------------------------------------------ column kernel
// Workgroups are dealt round-robin to the 8 XCDs, each with its own L2.  The
// linear workgroup id is remapped so that every XCD processes one contiguous
// range of (batch, tile) work items: neighbouring column tiles, which share
// 128-byte lines, then run on the same XCD close in time.  gridDim.x is the
// number of tiles, gridDim.y the batch.
__device__ __forceinline__ void xcd_tile(int& tile, int& b) {
  constexpr int NX = 8;
  const int ntiles = gridDim.x;
  const long long total = (long long)gridDim.x * gridDim.y;
  const long long id = (long long)blockIdx.y * gridDim.x + blockIdx.x;
  const long long per = total / NX, rem = total % NX;
  const long long x = id % NX, local = id / NX;
  const long long w = (x < rem) ? x * (per + 1) + local : rem * (per + 1) + (x - rem) * per + local;
  tile = __builtin_amdgcn_readfirstlane((int)(w % ntiles));
  b = __builtin_amdgcn_readfirstlane((int)(w / ntiles));
}

// waves per SIMD that a column kernel is compiled for: two workgroups of 1024
// threads where their LDS allows it (the wide FP32 tiles, at most 64 VGPRs), else
// what one workgroup needs.  The accumulating output operator takes 70 VGPRs and
// would spill.
template <typename T, int L, int C, int V, bool TWO = true>
constexpr int col_waves() {
  constexpr int threads = C * PlanInfo<L, V>::TPS;
  return TWO && threads == 1024 && sizeof(T) == 4 && 2 * TwLds<T, L, C, V>::bytes <= (size_t)CU_LDS ? 8 : (threads + 255) / 256;
}

// a thread's elements of one line to a destination
template <int TPS, int L, bool NT, typename T, int EPT, class Dst>
__device__ __forceinline__ void store_elements(const Dst& dst, int b, int col, int t, const cx<T> (&v)[EPT],
                                               const cx<T> (&old)[EPT]) {
#pragma unroll
  for (int e = 0; e < EPT; ++e)
    if constexpr (NT)
      dst.template store<true>(b, col, Pos(t, TPS * e, TPS, L), v[e], old[e]);
    else
      dst.store(b, col, Pos(t, TPS * e, TPS, L), v[e], old[e]);
}
template <int TPS, int L, typename T, int EPT, class Dst>
__device__ __forceinline__ void store_line(const Dst& dst, int b, int col, int t, const cx<T> (&v)[EPT],
                                           const cx<T> (&old)[EPT]) {
  if constexpr (Streams<Dst>::value) {
    if (dst.nt) {
      store_elements<TPS, L, true>(dst, b, col, t, v, old);
      return;
    }
  }
  store_elements<TPS, L, false>(dst, b, col, t, v, old);
}

// C adjacent columns per workgroup (the tile width chosen by the autotuner)
template <typename T, int L, bool INV, class Src, class Dst, int C, int V = 0>
__global__ void __launch_bounds__((C * PlanInfo<L, V>::TPS), (col_waves<T, L, C, V, Streams<Dst>::value>()))
    k_col(Src src, Dst dst, const cx<T>* __restrict__ tw, int ncols) {
  constexpr int EPT = PlanInfo<L, V>::EPT, TPS = PlanInfo<L, V>::TPS;
  extern __shared__ __align__(16) unsigned char col_lds_raw[];  // TwLds<T, L, C, V>::bytes
  const int c = threadIdx.x % C, t = threadIdx.x / C;
  int tile, b;
  xcd_tile(tile, b);
  const int col = tile * C + c;
  const bool act = col < ncols;
  // lanes past the last column load column ncols-1 and store nothing
  const int colc = act ? col : ncols - 1;
  cx<T> v[EPT];
#pragma unroll
  for (int e = 0; e < EPT; ++e) v[e] = src.load(b, colc, Pos(t, TPS * e, TPS, L));
  const ColTw<T, L, C, V> ft(tw, col_lds_raw);  // after the loads: their latency overlaps the table copy
  ft.template exec<INV>(v, c, t);
  int ts = t;  // the stores' addresses are formed here, not before the transform
  asm volatile("" : "+v"(ts));
  cx<T> old[EPT];
#pragma unroll
  for (int e = 0; e < EPT; ++e) old[e] = dst.load_old(b, colc, Pos(ts, TPS * e, TPS, L));
  if (act) store_line<TPS, L>(dst, b, col, ts, v, old);
}

// Persistent, software-pipelined variant of k_col: gridDim.x workgroups (a
// multiple of 8, as many as are resident at once) each walk a strided subset
// of the work items (batch, tile), and the loads of a workgroup's next item
// are issued before the transform and stores of its current one, so that a
// workgroup keeps a tile's worth of loads in flight while it computes.  Work
// items are split into 8 contiguous ranges, one per XCD (workgroups are dealt
// to the XCDs round-robin), and the workgroups of an XCD interleave within its
// range, so that the tiles in flight on one XCD are neighbours in memory.
__device__ __forceinline__ bool pipe_range(long long nitems, long long& w, long long& hi, int& step) {
  constexpr int NX = 8;
  const int xcd = blockIdx.x % NX, slot = blockIdx.x / NX;
  step = gridDim.x / NX;
  const long long per = nitems / NX, rem = nitems % NX;
  const long long lo = xcd < rem ? xcd * (per + 1) : rem * (per + 1) + (xcd - rem) * per;
  hi = lo + per + (xcd < rem ? 1 : 0);
  w = lo + slot;
  return w < hi;
}

template <typename T, int L, bool INV, class Src, class Dst, int C, int V = 0>
__global__ void __launch_bounds__((C * PlanInfo<L, V>::TPS))
    k_col_pipe(Src src, Dst dst, const cx<T>* __restrict__ tw, int ncols, int ntiles, long long nitems) {
  constexpr int EPT = PlanInfo<L, V>::EPT, TPS = PlanInfo<L, V>::TPS;
  extern __shared__ __align__(16) unsigned char col_lds_raw[];  // TwLds<T, L, C, V>::bytes
  const int c = threadIdx.x % C, t = threadIdx.x / C;
  long long w, hi;
  int step;
  if (!pipe_range(nitems, w, hi, step)) return;
  cx<T> nx[EPT];
  auto fetch = [&](long long item, int tq, cx<T>(&v)[EPT]) {
    const int b = __builtin_amdgcn_readfirstlane((int)(item / ntiles)),
              col = __builtin_amdgcn_readfirstlane((int)(item % ntiles)) * C + c;
    const int colc = col < ncols ? col : ncols - 1;
#pragma unroll
    for (int e = 0; e < EPT; ++e) v[e] = src.load(b, colc, Pos(tq, TPS * e, TPS, L));
  };
  fetch(w, t, nx);
  const ColTw<T, L, C, V> ft(tw, col_lds_raw);
  for (; w < hi; w += step) {
    // per-element positions recomputed each item (an empty asm statement
    // hides that they do not change), not held in registers across the loop
    int tq = t;
    asm volatile("" : "+v"(tq));
    cx<T> v[EPT];
#pragma unroll
    for (int e = 0; e < EPT; ++e) v[e] = nx[e];
    if (w + step < hi) fetch(w + step, tq, nx);
    // every stage exchange of the previous item ended with a barrier after
    // its last LDS read, so the first exchange of this one may write
    ft.template exec<INV>(v, c, t);
    const int b = __builtin_amdgcn_readfirstlane((int)(w / ntiles)),
              col = __builtin_amdgcn_readfirstlane((int)(w % ntiles)) * C + c;
    const int colc = col < ncols ? col : ncols - 1;
    cx<T> old[EPT];
#pragma unroll
    for (int e = 0; e < EPT; ++e) old[e] = dst.load_old(b, colc, Pos(tq, TPS * e, TPS, L));
    if (col < ncols) store_line<TPS, L>(dst, b, col, tq, v, old);
  }
}

// Several outputs of one launch over the same tiles.  A spec M provides the
// output count `no` and, for output o, load(o, b, col, pos) and
// store(o, b, col, pos, v); o is uniform, so a spec picks kernel-argument
// fields by selects without indexing into private memory.  The kernel reads
// each output's source values again instead of holding them in registers,
// which would cost occupancy; a re-read follows the first read of the same
// workgroup by one transform and is served by the L2 or the MALL, so HBM sees
// a shared source once.
//
// MultiPow: up to three outputs of one source (the x and y stages of the
// Hessian rows): output o transforms the zero-padded source line times the
// power pw[o] of its wavenumber factor (SrcPadPow) into out[o] (DstPlain
// strides).
template <typename T>
struct MultiPow {
  SrcPadPow<T> src;
  DstPlain<T> dst;
  cx<T>* out[3];
  int pw[3];
  int no;
  int nt = 0;
  void stream(int C) {
    nt = 1;
    for (int o = 0; o < no; ++o) nt &= streams(out[o], C, dst.sb, dst.sp, sizeof(cx<T>));
  }
  __device__ __forceinline__ cx<T> load(int o, int b, int col, Pos pos) const {
    SrcPadPow<T> s = src;
    s.pw = o == 0 ? pw[0] : (o == 1 ? pw[1] : pw[2]);
    return s.load(b, col, pos);
  }
  template <bool NT = false>
  __device__ __forceinline__ void store(int o, int b, int col, Pos pos, cx<T> v) const {
    DstPlain<T> d = dst;
    d.p = o == 0 ? out[0] : (o == 1 ? out[1] : out[2]);
    d.template store<NT>(b, col, pos, v, v);
  }
};

template <typename T, int L, bool INV, int C, int V, class M>
__global__ void __launch_bounds__((C * PlanInfo<L, V>::TPS), (col_waves<T, L, C, V>()))
    k_col_multi(M a, const cx<T>* __restrict__ tw, int ncols) {
  constexpr int EPT = PlanInfo<L, V>::EPT, TPS = PlanInfo<L, V>::TPS;
  extern __shared__ __align__(16) unsigned char col_lds_raw[];  // TwLds<T, L, C, V>::bytes
  const int c = threadIdx.x % C, t = threadIdx.x / C;
  int tile, b;
  xcd_tile(tile, b);
  const int col = tile * C + c;
  const bool act = col < ncols;
  const int colc = act ? col : ncols - 1;
  const ColTw<T, L, C, V> ft(tw, col_lds_raw);
#pragma unroll 1
  for (int o = 0; o < a.no; ++o) {
    // the line position and column pass through an empty asm statement per
    // output, so that the element addresses and wavenumber factors are
    // recomputed for each output instead of being held in registers across
    // the loop (about 60 VGPRs, which would halve the resident workgroups)
    int tq = t, cq = colc, colq = col;
    asm volatile("" : "+v"(tq), "+v"(cq), "+v"(colq));
    cx<T> v[EPT];
#pragma unroll
    for (int e = 0; e < EPT; ++e) v[e] = a.load(o, b, cq, Pos(tq, TPS * e, TPS, L));
    // the previous output's last exchange ended with a barrier after its
    // last LDS read, so this transform's first exchange may write
    ft.template exec<INV>(v, c, tq);
    asm volatile("" : "+v"(tq), "+v"(colq));
    if (act) {
      if (a.nt) {
#pragma unroll
        for (int e = 0; e < EPT; ++e) a.template store<true>(o, b, colq, Pos(tq, TPS * e, TPS, L), v[e]);
      } else {
#pragma unroll
        for (int e = 0; e < EPT; ++e) a.store(o, b, colq, Pos(tq, TPS * e, TPS, L), v[e]);
      }
    }
  }
}

// one output of a multi-output spec as a plain source / destination (the
// generic-length path runs one pass per output)
template <typename T, class M>
struct MultiSrc {
  M m;
  int o;
  __device__ __forceinline__ cx<T> load(int b, int col, Pos pos) const { return m.load(o, b, col, pos); }
};
template <typename T, class M>
struct MultiDst {
  M m;
  int o;
  __device__ __forceinline__ cx<T> load_old(int, int, int) const { return mk(T(0), T(0)); }
  __device__ __forceinline__ void store(int b, int col, Pos pos, cx<T> v, cx<T>) const { m.store(o, b, col, pos, v); }
};

// Projection of a padded line onto the modes of the n-grid: forward
// transform, truncation to the n kept modes with the Nyquist mode and the
// Nyquist column (kz = n/2) zeroed and the scale fscale (the truncating pass
// of the Orszag chain, unpad), then padding with the scale iscale and the
// inverse transform (pad_insert).  The truncated and padded positions
// coincide (position pos <-> index pos or pos - n/2), so the line stays in
// registers and the truncated field never exists.  The output may be the
// source line itself: every line is read before it is written, by the
// workgroup that owns it.
template <typename T>
struct TurnArgs {
  const cx<T>* src;
  long long sb, sp;  // source strides (batch, line position)
  int n;
  T fscale, iscale;
  cx<T>* out;
  long long osb, osp;
  int nb;            // line sets of one array; further arrays sq apart
  long long sq, osq;
  int nt = 0;
  void stream(int C) {
    nt = streams(out, C, osb, osp, sizeof(cx<T>)) && ((unsigned long long)osq * sizeof(cx<T>)) % 128 == 0;
  }
  __device__ __forceinline__ const cx<T>* from(int b) const {
    const int q = b / nb;
    return src + (long long)q * sq + (long long)(b - q * nb) * sb;
  }
  __device__ __forceinline__ cx<T>* to(int b) const {
    const int q = b / nb;
    return out + (long long)q * osq + (long long)(b - q * nb) * osb;
  }
};

// whether position t + c (c .. c + W - 1 the element's range) of a padded line of
// L = 3n/2 positions is dropped or the Nyquist one: n/2 .. n
__device__ __forceinline__ bool turn_zero(int t, int c, int W, int L) {
  const int nh = L / 3, n = 2 * (L / 3);
  if (c + W - 1 < nh || c > n) return false;
  if (c >= nh && c + W - 1 <= n) return true;
  return (t + c >= nh) & (t + c <= n);
}

template <typename T, int L, int C, int V = 0>
__global__ void __launch_bounds__((C * PlanInfo<L, V>::TPS), (col_waves<T, L, C, V>()))
    k_col_turn(TurnArgs<T> a, const cx<T>* __restrict__ tw, int ncols) {
  constexpr int EPT = PlanInfo<L, V>::EPT, TPS = PlanInfo<L, V>::TPS;
  extern __shared__ __align__(16) unsigned char col_lds_raw[];  // TwLds<T, L, C, V>::bytes
  const int c = threadIdx.x % C, t = threadIdx.x / C;
  int tile, b;
  xcd_tile(tile, b);
  const int col = tile * C + c;
  const bool act = col < ncols;
  const int colc = act ? col : ncols - 1;
  const int nh = a.n >> 1;
  const cx<T>* const from = a.from(b);
  cx<T> x[EPT];
#pragma unroll
  for (int e = 0; e < EPT; ++e) x[e] = *line_at(from, a.sp, colc, t, TPS * e);
  const ColTw<T, L, C, V> ft(tw, col_lds_raw);
  ft.template exec<false>(x, c, t);
  const bool nyqc = colc == nh;
#pragma unroll
  for (int e = 0; e < EPT; ++e) {
    // dropped positions and the Nyquist mode (index n/2 is position n/2 = L/3)
    const bool zero = turn_zero(t, TPS * e, TPS, L) | nyqc;
    const cx<T> o = x[e] * a.fscale;  // the n-grid value
    x[e] = or_zero(!zero, o * a.iscale);
  }
  __syncthreads();  // the forward transform's exchange reads are done
  int ti = t;  // LDS and line addresses formed again, not held in registers since the forward transform
  asm volatile("" : "+v"(ti));
  ft.template exec<true>(x, c, ti);
  if (act) {
    cx<T>* const to = a.to(b);
    if (a.nt) {
#pragma unroll
      for (int e = 0; e < EPT; ++e) put<true>(line_at(to, a.osp, col, ti, TPS * e), x[e]);
    } else {
#pragma unroll
      for (int e = 0; e < EPT; ++e) *line_at(to, a.osp, col, ti, TPS * e) = x[e];
    }
  }
}

// persistent, software-pipelined k_col_turn (see k_col_pipe)
template <typename T, int L, int C, int V = 0>
__global__ void __launch_bounds__((C * PlanInfo<L, V>::TPS))
    k_col_turn_pipe(TurnArgs<T> a, const cx<T>* __restrict__ tw, int ncols, int ntiles, long long nitems) {
  constexpr int EPT = PlanInfo<L, V>::EPT, TPS = PlanInfo<L, V>::TPS;
  extern __shared__ __align__(16) unsigned char col_lds_raw[];  // TwLds<T, L, C, V>::bytes
  const int c = threadIdx.x % C, t = threadIdx.x / C;
  const int nh = a.n >> 1;
  long long w, hi;
  int step;
  if (!pipe_range(nitems, w, hi, step)) return;
  cx<T> nx[EPT];
  auto fetch = [&](long long item, int tq, cx<T>(&v)[EPT]) {
    const int b = __builtin_amdgcn_readfirstlane((int)(item / ntiles)),
              col = __builtin_amdgcn_readfirstlane((int)(item % ntiles)) * C + c;
    const int colc = col < ncols ? col : ncols - 1;
    const cx<T>* const from = a.from(b);
#pragma unroll
    for (int e = 0; e < EPT; ++e) v[e] = *line_at(from, a.sp, colc, tq, TPS * e);
  };
  fetch(w, t, nx);
  const ColTw<T, L, C, V> ft(tw, col_lds_raw);
  for (; w < hi; w += step) {
    int tq = t;  // recomputed per item (see k_col_pipe)
    asm volatile("" : "+v"(tq));
    cx<T> x[EPT];
#pragma unroll
    for (int e = 0; e < EPT; ++e) x[e] = nx[e];
    if (w + step < hi) fetch(w + step, tq, nx);
    const int b = __builtin_amdgcn_readfirstlane((int)(w / ntiles)),
              col = __builtin_amdgcn_readfirstlane((int)(w % ntiles)) * C + c;
    const int colc = col < ncols ? col : ncols - 1;
    ft.template exec<false>(x, c, t);
    const bool nyqc = colc == nh;
#pragma unroll
    for (int e = 0; e < EPT; ++e) {
      const bool zero = turn_zero(tq, TPS * e, TPS, L) | nyqc;
      const cx<T> o = x[e] * a.fscale;
      x[e] = or_zero(!zero, o * a.iscale);
    }
    __syncthreads();  // the forward transform's exchange reads are done
    ft.template exec<true>(x, c, t);
    if (col < ncols) {
      cx<T>* const to = a.to(b);
      if (a.nt) {
#pragma unroll
        for (int e = 0; e < EPT; ++e) put<true>(line_at(to, a.osp, col, tq, TPS * e), x[e]);
      } else {
#pragma unroll
        for (int e = 0; e < EPT; ++e) *line_at(to, a.osp, col, tq, TPS * e) = x[e];
      }
    }
  }
}

#define MFX_COL_LENGTHS(X) \
  X(16) X(24) X(32) X(48) X(64) X(72) X(96) X(128) X(144) X(192) X(256) X(288) X(384) X(512) X(768) X(1024) X(1536)
#define MFX_ROW_LENGTHS(X) \
  X(8) X(12) X(16) X(24) X(32) X(36) X(48) X(64) X(72) X(96) X(128) X(144) X(192) X(256) X(288) X(384) X(512) X(768)

// Workgroups of a persistent kernel: as many as are resident at once on the
// device (occupancy x compute units), a multiple of the 8 XCDs, at most the
// number of work items rounded up to 8.
template <class K>
unsigned pipe_grid(Ctx& c, K kernel, int block, long long nitems, size_t dyn = 0) {
  int& per_cu = c.occupancy[(const void*)kernel];  // one query per kernel
  if (per_cu == 0) {
    int n = 0;
    MFX_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, kernel, block, dyn));
    per_cu = n > 0 ? n : 1;
  }
  long long g = (long long)per_cu * c.num_cus();
  const long long cap = (nitems + 7) / 8 * 8;
  if (g > cap) g = cap;
  return (unsigned)((g + 7) / 8 * 8);
}

// A column kernel's LDS (TwLds) is dynamic; beyond the default 64 KiB per
// workgroup the kernel must be allowed more, once per kernel.
template <class K>
void col_lds_prep(Ctx& c, K kernel, size_t dyn) {
  if (dyn <= 65536) return;
  MFX_REQUIRE(dyn <= (size_t)CU_LDS, "column tile too large for one compute unit's LDS");
  int& done = c.lds_attr[(const void*)kernel];
  if (done < (int)dyn) {
    MFX_HIP(hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)dyn));
    done = (int)dyn;
  }
}

template <typename T, int L, int C, bool INV, bool PIPE, int V, class Src, class Dst>
void launch_col_LC(Ctx& c, Src s, Dst d, int ncols, int nbatch, const char* name, double bytes) {
  const dim3 block(C * PlanInfo<L, V>::TPS);
  const int ntiles = (ncols + C - 1) / C;
  set_stream(d, C);
  LaunchScope ls(c, name, bytes);
  constexpr size_t dyn = TwLds<T, L, C, V>::bytes;
  if constexpr (PIPE) {
    const long long nitems = (long long)ntiles * nbatch;
    auto k = k_col_pipe<T, L, INV, Src, Dst, C, V>;
    col_lds_prep(c, k, dyn);
    hipLaunchKernelGGL(k, dim3(pipe_grid(c, k, (int)block.x, nitems, dyn)), block, dyn, c.stream, s, d,
                       c.twiddles<T>(L), ncols, ntiles, nitems);
  } else {
    auto k = k_col<T, L, INV, Src, Dst, C, V>;
    col_lds_prep(c, k, dyn);
    hipLaunchKernelGGL(k, dim3(ntiles, nbatch), block, dyn, c.stream, s, d, c.twiddles<T>(L), ncols);
  }
  check_launch(name);
}

// Column-pass variants: tile width (the widest tile whose exchange area fits
// 64 KiB of LDS, ColCfg, or half of it), plain or persistent-pipelined
// kernel, and radix plan (variant 1 where the length has one); the context's
// tuning table (col_tile) picks one.
template <typename T, int L, bool INV, int V, class Src, class Dst>
void launch_col_LV(Ctx& c, int v, Src s, Dst d, int ncols, int nbatch, const char* name, double bytes) {
  constexpr int CM = ColCfg<T, L, V>::C, CW = ColCfg<T, L, V>::CW;
  const bool pipe = (v & COL_PIPELINED) != 0;
  if constexpr (CW > 0) {
    if ((v & COL_WIDTH) == CW) {
      if (pipe)
        launch_col_LC<T, L, CW, INV, true, V>(c, s, d, ncols, nbatch, name, bytes);
      else
        launch_col_LC<T, L, CW, INV, false, V>(c, s, d, ncols, nbatch, name, bytes);
      return;
    }
  }
  if constexpr (CM >= 2) {
    if ((v & COL_WIDTH) == CM / 2) {
      if (pipe)
        launch_col_LC<T, L, CM / 2, INV, true, V>(c, s, d, ncols, nbatch, name, bytes);
      else
        launch_col_LC<T, L, CM / 2, INV, false, V>(c, s, d, ncols, nbatch, name, bytes);
      return;
    }
  }
  if (pipe)
    launch_col_LC<T, L, CM, INV, true, V>(c, s, d, ncols, nbatch, name, bytes);
  else
    launch_col_LC<T, L, CM, INV, false, V>(c, s, d, ncols, nbatch, name, bytes);
}

// Destinations whose store path needs many registers per element: with the
// second radix plan's 24 elements per thread the final x pass (DstTruncOp)
// compiles to 172 VGPRs (2 waves per SIMD) instead of 88 and measured slower
// (2.33 vs 2.11 ms for the five 768-line x passes of 3LPT at 512^3), so such
// passes keep plan 0; their tile width and kernel form are tuned on their own
// (COL_TRUNC_OP).
template <class D>
struct HeavyDst {
  static constexpr bool value = false;
};
template <typename T>
struct HeavyDst<DstTruncOp<T>> {
  static constexpr bool value = true;
};

// Passes over padded lines: out of place, on the work grids' pitch, where tiles stream
// their stores.  The in-place passes of a plain grid of the same length have other
// best variants (inverse y pass of 192 lines, FP32: 14.0 us with its own choice, 16.9
// with that of the Hessian rows; x passes of 384, FP64: 153 and 157 us, 160 and 180 with
// the choice for a row of columns at a time).
template <class S>
struct PaddedPass {
  static constexpr bool value = false;
};
template <typename T, bool MULT>
struct PaddedPass<SrcPad<T, MULT>> {
  static constexpr bool value = true;
};
template <typename T>
struct PaddedPass<DstTrunc<T>> {
  static constexpr bool value = true;
};
template <class S>
struct HessPass {
  static constexpr bool value = false;
};
template <typename T>
struct HessPass<SrcHessY<T>> {
  static constexpr bool value = true;
};

// the kind a pass is tuned as
template <bool INV, class Src, class Dst>
constexpr int col_kind() {
  if (HeavyDst<Dst>::value) return COL_TRUNC_OP;
  if (HessPass<Src>::value) return COL_HESS_Y;
  return (PaddedPass<Src>::value || PaddedPass<Dst>::value ? COL_PAD : 0) + (INV ? 1 : 0);
}

template <typename T, int L, bool INV, class Src, class Dst>
void launch_col_L(Ctx& c, Src s, Dst d, int ncols, int nbatch, const char* name, double bytes) {
  const int v = c.col_tile(L, (int)sizeof(T), col_kind<INV, Src, Dst>(), ColCfg<T, L>::C, stride_class(s.sp, (int)sizeof(cx<T>)));
  if constexpr (PlanAlt<L>::value && !HeavyDst<Dst>::value) {
    if (v & COL_PLAN_ALT) {
      launch_col_LV<T, L, INV, 1>(c, v, s, d, ncols, nbatch, name, bytes);
      return;
    }
  }
  launch_col_LV<T, L, INV, 0>(c, v, s, d, ncols, nbatch, name, bytes);
}

// widest tile for length L, precision T
template <typename T>
int col_tile_max(int L) {
  switch (L) {
#define MFX_CASE(LL) \
  case LL:           \
    return ColCfg<T, LL>::C;
    MFX_COL_LENGTHS(MFX_CASE)
#undef MFX_CASE
    default:
      throw Error(1, "unsupported transform length " + std::to_string(L));
  }
}

// the wide tile width of length L, plan variant alt (0 if none)
template <typename T>
int col_tile_wide(int L, int alt) {
  switch (L) {
#define MFX_CASE(LL)                                                         \
  case LL:                                                                   \
    if constexpr (PlanAlt<LL>::value) {                                      \
      if (alt) return ColCfg<T, LL, PlanAlt<LL>::value ? 1 : 0>::CW;         \
    }                                                                        \
    return ColCfg<T, LL>::CW;
    MFX_COL_LENGTHS(MFX_CASE)
#undef MFX_CASE
    default:
      return 0;
  }
}

// whether length L has a second radix plan
inline bool col_plan_alt(int L) {
  switch (L) {
#define MFX_CASE(LL) \
  case LL:           \
    return PlanAlt<LL>::value;
    MFX_COL_LENGTHS(MFX_CASE)
#undef MFX_CASE
    default:
      return false;
  }
}

// The particle arrays of up to six components of an n^3 grid, n^2 rows each, in
// one launch: component w = row / n^2 goes to out[w]; code(w) & 3 is its axis,
// code(w) >> 2 its kind (0 positions, 1 velocities).
struct PartOut {
  double* out[6];
  unsigned codes;  // four bits for each component
  __device__ __forceinline__ double* array(int w) const {
    return w < 2 ? (w == 0 ? out[0] : out[1]) : (w < 4 ? (w == 2 ? out[2] : out[3]) : (w == 4 ? out[4] : out[5]));
  }
  __device__ __forceinline__ int code(int w) const { return (int)(codes >> (4 * w)) & 15; }
};

// ------------------------------------------------------------------ lengths without tuned kernels
// (mixed_kernels.hip: run-time schedules)
template <typename T, bool INV, class Src, class Dst>
void launch_col_any(Ctx& c, int L, Src s, Dst d, int ncols, int nbatch, const char* name, double bytes);
template <typename T>
void launch_turn_any(Ctx& c, int L, const TurnArgs<T>& a, int ncols, int nbatch, const char* name, double bytes);
template <typename T>
void launch_row_r2c_any(Ctx& c, int K, const T* src, long long spitch, cx<T>* dst, long long dpitch, int hout,
                        long long nrows, T scale, const char* name, double bytes);
template <typename T>
void launch_row_c2r_any(Ctx& c, int K, const cx<T>* src, long long spitch, int hin, T* dst, long long dpitch,
                        long long nrows, T scale, const char* name, double bytes);
template <typename T>
void launch_row_c2r_part_any(Ctx& c, int K, const cx<T>* src, long long spitch, int hin, const PartOut& po,
                             long long nrows, T scale, double lunit, double qoff, const char* name, double bytes);
template <typename T>
void launch_row_prod_any(Ctx& c, int K, const cx<T>* a, const cx<T>* b, long long spitch, int hin, cx<T>* dst,
                         long long dpitch, int hout, long long nrows, const T* mean, const char* name, double bytes);
// the mean of such a product into *mean, where launch_row_prod is to take it off
// (false: it is not)
template <typename T>
bool launch_row_mean(Ctx& c, int K, const cx<T>* a, const cx<T>* b, long long spitch, int hin, long long nrows,
                     T* mean, const char* name);

template <typename T, bool INV, class Src, class Dst>
void launch_col(Ctx& c, int L, Src s, Dst d, int ncols, int nbatch, const char* name, double bytes) {
  switch (L) {
#define MFX_CASE(LL)                                                    \
  case LL:                                                              \
    launch_col_L<T, LL, INV, Src, Dst>(c, s, d, ncols, nbatch, name, bytes); \
    return;
    MFX_COL_LENGTHS(MFX_CASE)
#undef MFX_CASE
    default:
      launch_col_any<T, INV>(c, L, s, d, ncols, nbatch, name, bytes);
  }
}

// The padded lengths M = 3n/2 of the Orszag and LPT passes (n = 16 ... 1024)
// and the corresponding z-row lengths K = M/2: the fused engine instantiates
// its passes for these only.
#define MFX_PAD_LENGTHS(X) X(24) X(48) X(72) X(96) X(144) X(192) X(288) X(384) X(768) X(1536)
#define MFX_PAD_K_LENGTHS(X) X(12) X(24) X(36) X(48) X(72) X(96) X(144) X(192) X(384) X(768)

template <typename T, bool INV, class Src, class Dst>
void launch_col_pad(Ctx& c, int L, Src s, Dst d, int ncols, int nbatch, const char* name, double bytes) {
  switch (L) {
#define MFX_CASE(LL)                                                    \
  case LL:                                                              \
    launch_col_L<T, LL, INV, Src, Dst>(c, s, d, ncols, nbatch, name, bytes); \
    return;
    MFX_PAD_LENGTHS(MFX_CASE)
#undef MFX_CASE
    default:
      launch_col_any<T, INV>(c, L, s, d, ncols, nbatch, name, bytes);
  }
}

// the y stage of the Hessian rows of `planes` x-planes (lpt_engine.hip)
template <typename T>
void launch_hess_y(Ctx& c, int m, const SrcHessY<T>& s, const DstHessY<T>& d, int ncols, int planes, const char* name,
                   double bytes);

template <typename T, int L, int C, bool PIPE, int V>
void launch_turn_LC(Ctx& c, TurnArgs<T> a, int ncols, int nbatch, const char* name, double bytes) {
  set_stream(a, C);
  const dim3 block(C * PlanInfo<L, V>::TPS);
  const int ntiles = (ncols + C - 1) / C;
  LaunchScope ls(c, name, bytes);
  constexpr size_t dyn = TwLds<T, L, C, V>::bytes;
  if constexpr (PIPE) {
    const long long nitems = (long long)ntiles * nbatch;
    auto k = k_col_turn_pipe<T, L, C, V>;
    col_lds_prep(c, k, dyn);
    hipLaunchKernelGGL(k, dim3(pipe_grid(c, k, (int)block.x, nitems, dyn)), block, dyn, c.stream, a,
                       c.twiddles<T>(L), ncols, ntiles, nitems);
  } else {
    auto k = k_col_turn<T, L, C, V>;
    col_lds_prep(c, k, dyn);
    hipLaunchKernelGGL(k, dim3(ntiles, nbatch), block, dyn, c.stream, a, c.twiddles<T>(L), ncols);
  }
  check_launch(name);
}

template <typename T, int L, int V>
void launch_turn_LV(Ctx& c, int v, const TurnArgs<T>& a, int ncols, int nbatch, const char* name, double bytes) {
  constexpr int CM = ColCfg<T, L, V>::C, CW = ColCfg<T, L, V>::CW;
  const bool pipe = (v & COL_PIPELINED) != 0;
  if constexpr (CW > 0) {
    if ((v & COL_WIDTH) == CW) {
      if (pipe)
        launch_turn_LC<T, L, CW, true, V>(c, a, ncols, nbatch, name, bytes);
      else
        launch_turn_LC<T, L, CW, false, V>(c, a, ncols, nbatch, name, bytes);
      return;
    }
  }
  if constexpr (CM >= 2) {
    if ((v & COL_WIDTH) == CM / 2) {
      if (pipe)
        launch_turn_LC<T, L, CM / 2, true, V>(c, a, ncols, nbatch, name, bytes);
      else
        launch_turn_LC<T, L, CM / 2, false, V>(c, a, ncols, nbatch, name, bytes);
      return;
    }
  }
  if (pipe)
    launch_turn_LC<T, L, CM, true, V>(c, a, ncols, nbatch, name, bytes);
  else
    launch_turn_LC<T, L, CM, false, V>(c, a, ncols, nbatch, name, bytes);
}

// at the variant tuned for the turn passes of (L, T) (key COL_TURN)
template <typename T, int L>
void launch_turn_L(Ctx& c, const TurnArgs<T>& a, int ncols, int nbatch, const char* name, double bytes) {
  const int v = c.col_tile(L, (int)sizeof(T), COL_TURN, ColCfg<T, L>::C, stride_class(a.sp, (int)sizeof(cx<T>)));
  if constexpr (PlanAlt<L>::value) {
    if (v & COL_PLAN_ALT) {
      launch_turn_LV<T, L, 1>(c, v, a, ncols, nbatch, name, bytes);
      return;
    }
  }
  launch_turn_LV<T, L, 0>(c, v, a, ncols, nbatch, name, bytes);
}

template <typename T>
void launch_turn(Ctx& c, int L, const TurnArgs<T>& a, int ncols, int nbatch, const char* name, double bytes) {
  switch (L) {
#define MFX_CASE(LL)                                           \
  case LL:                                                     \
    launch_turn_L<T, LL>(c, a, ncols, nbatch, name, bytes);     \
    return;
    MFX_PAD_LENGTHS(MFX_CASE)
#undef MFX_CASE
    default:
      launch_turn_any<T>(c, L, a, ncols, nbatch, name, bytes);
  }
}

template <typename T, int L, int C, bool INV, int V, class M>
void launch_multi_LC(Ctx& c, M a, int ncols, int nbatch, const char* name, double bytes) {
  set_stream(a, C);
  const dim3 block(C * PlanInfo<L, V>::TPS);
  const int ntiles = (ncols + C - 1) / C;
  LaunchScope ls(c, name, bytes);
  constexpr size_t dyn = TwLds<T, L, C, V>::bytes;
  auto k = k_col_multi<T, L, INV, C, V, M>;
  col_lds_prep(c, k, dyn);
  hipLaunchKernelGGL(k, dim3(ntiles, nbatch), block, dyn, c.stream, a, c.twiddles<T>(L), ncols);
  check_launch(name);
}

template <typename T, int L, bool INV, int V, class M>
void launch_multi_LV(Ctx& c, int v, const M& a, int ncols, int nbatch, const char* name, double bytes) {
  constexpr int CM = ColCfg<T, L, V>::C, CW = ColCfg<T, L, V>::CW;
  if constexpr (CW > 0) {
    if ((v & COL_WIDTH) == CW) {
      launch_multi_LC<T, L, CW, INV, V>(c, a, ncols, nbatch, name, bytes);
      return;
    }
  }
  if constexpr (CM >= 2) {
    if ((v & COL_WIDTH) == CM / 2) {
      launch_multi_LC<T, L, CM / 2, INV, V>(c, a, ncols, nbatch, name, bytes);
      return;
    }
  }
  launch_multi_LC<T, L, CM, INV, V>(c, a, ncols, nbatch, name, bytes);
}

// at the tile width tuned for (L, T, INV) and the stride class of line
// stride sp; the multi-output kernel has no pipelined form and always runs
// plan 0 (with the second plan the three-output Hessian pass compiled to 179
// instead of 95 VGPRs, two waves per SIMD instead of five; plan 0 now takes 80)
template <typename T, int L, bool INV, class M>
void launch_multi_L(Ctx& c, const M& a, long long sp, int ncols, int nbatch, const char* name, double bytes) {
  const int v = c.col_tile(L, (int)sizeof(T), COL_PAD + (INV ? 1 : 0), ColCfg<T, L>::C, stride_class(sp, (int)sizeof(cx<T>)));
  launch_multi_LV<T, L, INV, 0>(c, v, a, ncols, nbatch, name, bytes);
}

// a.no outputs of one launch; sp is the line stride of the source (for the
// tuning class); bytes: the algorithmic bytes of the launch.  Lengths
// without tuned kernels run one generic pass per output.
template <typename T, bool INV, class M>
void launch_multi(Ctx& c, int L, const M& a, long long sp, int ncols, int nbatch, const char* name, double bytes) {
  switch (L) {
#define MFX_CASE(LL)                                                \
  case LL:                                                          \
    launch_multi_L<T, LL, INV>(c, a, sp, ncols, nbatch, name, bytes); \
    return;
    MFX_COL_LENGTHS(MFX_CASE)
#undef MFX_CASE
    default:
      for (int o = 0; o < a.no; ++o)
        launch_col_any<T, INV>(c, L, MultiSrc<T, M>{a, o}, MultiDst<T, M>{a, o}, ncols, nbatch, name, bytes / a.no);
  }
}

// MultiPow outputs of one source; bytes: the source read once plus a.no outputs
template <typename T, bool INV>
void launch_col_multi(Ctx& c, int L, const MultiPow<T>& a, int ncols, int nbatch, const char* name, double bsrc,
                      double bdst) {
  MFX_REQUIRE(a.no >= 1 && a.no <= 3, "multi-output pass: 1 to 3 outputs");
  launch_multi<T, INV>(c, L, a, a.src.sp, ncols, nbatch, name, bsrc + a.no * bdst);
}

// ------------------------------------------------------------------ row kernels (z axis)
// One workgroup = one wavefront holding RowLanes<K>::RPW rows (two wavefronts
// holding one row for K >= 768); the row
// transforms are the LDS-resident ones of row_fft.hpp.
template <typename T, int K>
struct RowBlk {
  static constexpr int P = RowLanes<K>::P, RPW = RowLanes<K>::RPW, LB = RowLanes<K>::LB;
  static constexpr int THREADS = RowLanes<K>::THREADS;
  static constexpr int LDS = RPW * 2 * LB;  // complex elements of LDS per workgroup
};

// The twiddle tables (K entries each) are copied to LDS once per workgroup:
// the transforms then read them with LDS loads, which leaves the vector
// memory counter to the row data alone, so that a row fetched ahead of its
// use is not waited for by every twiddle access.
#define MFX_ROW_PROLOGUE(T, K)                                                      \
  constexpr int P_ = RowBlk<T, K>::P, LB_ = RowBlk<T, K>::LB;                       \
  __shared__ cx<T> lds_[RowBlk<T, K>::LDS];                                         \
  __shared__ cx<T> tw_[2 * (K)];                                                    \
  for (int i_ = threadIdx.x; i_ < (K); i_ += RowBlk<T, K>::THREADS) {             \
    tw_[i_] = twK[i_];                                                              \
    tw_[(K) + i_] = twM[i_];                                                        \
  }                                                                                 \
  __syncthreads();                                                                  \
  const int lane = threadIdx.x % P_, r_ = threadIdx.x / P_;                         \
  MFX_ROW_LOOP_BEGIN(T, K)

// A row workgroup loops over rows base + r_, base = blockIdx.x*RPW, advancing
// by gridDim.x*RPW (the same trip count for every lane): the twiddle tables
// are copied to LDS once per workgroup, not once per row.  Every transform
// begins with a barrier, so one row's buffers are free when the next row's
// transform writes them.  The row context takes an opaque zero (lz_) so that
// its per-lane twiddles and indices are loaded and computed per row rather
// than held in registers across the loop.
#define MFX_ROW_LOOP_BEGIN(T, K)                                                                    \
  for (long long base_ = (long long)blockIdx.x * RowBlk<T, K>::RPW; base_ < nrows;                   \
       base_ += (long long)gridDim.x * RowBlk<T, K>::RPW) {                                          \
    const long long row = base_ + r_;                                                               \
    const bool act = row < nrows;                                                                   \
    const long long rowc = act ? row : 0;                                                           \
    int lz_ = 0;                                                                                    \
    asm volatile("" : "+v"(lz_));                                                                   \
    RowCtx<T, K> rc{lds_ + r_ * 2 * LB_ + lz_, lds_ + r_ * 2 * LB_ + LB_ + lz_, lane + lz_, tw_ + lz_, \
                    tw_ + (K) + lz_};
#define MFX_ROW_LOOP_END }

// One row (per row slot r_) per workgroup, for the fused z kernels: holding
// their many operand rows leaves no registers for a row loop.
#define MFX_ROW_PROLOGUE1(T, K)                                                     \
  constexpr int P_ = RowBlk<T, K>::P, LB_ = RowBlk<T, K>::LB;                       \
  __shared__ cx<T> lds_[RowBlk<T, K>::LDS];                                         \
  __shared__ cx<T> tw_[2 * (K)];                                                    \
  for (int i_ = threadIdx.x; i_ < (K); i_ += RowBlk<T, K>::THREADS) {             \
    tw_[i_] = twK[i_];                                                              \
    tw_[(K) + i_] = twM[i_];                                                        \
  }                                                                                 \
  __syncthreads();                                                                  \
  const int lane = threadIdx.x % P_, r_ = threadIdx.x / P_;                         \
  const long long row = (long long)blockIdx.x * RowBlk<T, K>::RPW + r_;             \
  const bool act = row < nrows;                                                     \
  const long long rowc = act ? row : 0;                                             \
  RowCtx<T, K> rc{lds_ + r_ * 2 * LB_, lds_ + r_ * 2 * LB_ + LB_, lane, tw_, tw_ + (K)};

template <typename T, int K>
__global__ void __launch_bounds__(RowLanes<K>::THREADS)
    k_row_r2c(const T* __restrict__ src, long long spitch, cx<T>* dst, long long dpitch, int hout,
              long long nrows, T scale, const cx<T>* __restrict__ twK, const cx<T>* __restrict__ twM) {
  MFX_ROW_PROLOGUE(T, K)
  constexpr int E = RowCtx<T, K>::E;
  const __amdgpu_buffer_rsrc_t r = row_rsrc_u<RowLanes<K>::RPW == 1>(src + rowc * spitch, K * sizeof(cx<T>));
  cx<T> v[E];
#pragma unroll
  for (int e = 0; e < E; ++e) v[e] = buf_load<T>(r, (unsigned)(lane + P_ * e) * sizeof(cx<T>));
  rc.r2c_store(v, dst + rowc * dpitch, hout, act, scale);
  MFX_ROW_LOOP_END
}

template <typename T, int K>
__global__ void __launch_bounds__(RowLanes<K>::THREADS)
    k_row_c2r(const cx<T>* src, long long spitch, int hin, T* dst, long long dpitch, long long nrows, T scale,
              const cx<T>* __restrict__ twK, const cx<T>* __restrict__ twM) {
  MFX_ROW_PROLOGUE(T, K)
  constexpr int E = RowCtx<T, K>::E;
  cx<T> v[E];
  rc.c2r(v, src + rowc * spitch, hin);
  // K packed pairs, and the two padding reals of an in-place row set to zero;
  // an inactive row stores nothing (zero-length resource)
  const unsigned nst = act ? (unsigned)(dpitch >= 2 * K + 2 ? K + 1 : K) : 0u;
  const __amdgpu_buffer_rsrc_t r = row_rsrc_u<RowLanes<K>::RPW == 1>(dst + rowc * dpitch, nst * sizeof(cx<T>));
#pragma unroll
  for (int e = 0; e <= E; ++e) {
    const int n = lane + P_ * e;
    if (n <= K) buf_store<T>(n < K ? v[e < E ? e : E - 1] * scale : mk(T(0), T(0)), r, (unsigned)n * sizeof(cx<T>));
  }
  MFX_ROW_LOOP_END
}

// c2r of the z rows of an n^3 grid straight into the FP64 particle arrays
// (particle_generator.hh:525-541 positions, 622-632 velocities): each real
// value is scaled and rounded to T as the in-place c2r stores it, converted
// to double and, for positions (kind 0), added to the lattice coordinate
// q_d = i_d/n * lunit.  Row r = i*n + j holds particles r*n .. r*n + n-1.
template <typename T, int K>
__global__ void __launch_bounds__(RowLanes<K>::THREADS)
    k_row_c2r_part(const cx<T>* src, long long spitch, int hin, PartOut po, long long nrows, T scale, double lunit,
                   double qoff, const cx<T>* __restrict__ twK, const cx<T>* __restrict__ twM) {
  MFX_ROW_PROLOGUE(T, K)
  constexpr int E = RowCtx<T, K>::E, n = 2 * K;
  cx<T> v[E];
  rc.c2r(v, src + rowc * spitch, hin);
  const int rw = (int)(rowc / n);  // component w, x index i
  const int w = rw / n, i = rw - w * n, j = (int)(rowc - (long long)rw * n);
  const int code = po.code(w), idim = code & 3, kind = code >> 2;
  const double qrow = (double)(idim == 0 ? i : j) / (double)n * lunit + qoff;
  const __amdgpu_buffer_rsrc_t r = row_rsrc_u<RowLanes<K>::RPW == 1>(po.array(w) + ((long long)i * n + j) * n,
                                                                     act ? (unsigned)(n * sizeof(double)) : 0u);
#pragma unroll
  for (int e = 0; e < E; ++e) {
    const int m = lane + P_ * e;
    if (m < K) {
      double f0 = (double)(v[e].x * scale), f1 = (double)(v[e].y * scale);
      if (kind == 0) {
        if (idim == 2) {
          f0 = (double)(2 * m) / (double)n * lunit + qoff + f0;
          f1 = (double)(2 * m + 1) / (double)n * lunit + qoff + f1;
        } else {
          f0 = qrow + f0;
          f1 = qrow + f1;
        }
      }
      buf_store<double>(mk(f0, f1), r, (unsigned)m * sizeof(cx<double>));
    }
  }
  MFX_ROW_LOOP_END
}

// P3: c2r of two truncated half spectra, pointwise product, r2c, truncation
template <typename T, int K>
__global__ void __launch_bounds__(RowLanes<K>::THREADS)
    k_row_prod(const cx<T>* a, const cx<T>* b, long long spitch, int hin, cx<T>* dst, long long dpitch,
               int hout, long long nrows, const cx<T>* __restrict__ twK, const cx<T>* __restrict__ twM) {
  MFX_ROW_PROLOGUE(T, K)
  constexpr int E = RowCtx<T, K>::E;
  cx<T> va[E], vb[E];
  rc.c2r(va, a + rowc * spitch, hin);
  rc.c2r(vb, b + rowc * spitch, hin);
  // packed real product: z[n] = x[2n] + i x[2n+1]
#pragma unroll
  for (int e = 0; e < E; ++e) va[e] = mk(va[e].x * vb[e].x, va[e].y * vb[e].y);
  rc.r2c_store(va, dst + rowc * dpitch, hout, act, T(1));
  MFX_ROW_LOOP_END
}

template <typename T, int K>
dim3 row_grid(long long nrows) {
  // enough workgroups for several residency rounds on 256 CUs; each loops
  // over nrows / (16384 RPW) rows
  const long long need = (nrows + RowBlk<T, K>::RPW - 1) / RowBlk<T, K>::RPW;
  return dim3((unsigned)(need < 16384 ? need : 16384));
}

// one workgroup per RPW rows (MFX_ROW_PROLOGUE1 kernels)
template <typename T, int K>
dim3 row_grid1(long long nrows) {
  return dim3((unsigned)((nrows + RowBlk<T, K>::RPW - 1) / RowBlk<T, K>::RPW));
}

template <typename T, int K>
void launch_row_r2c_K(Ctx& c, const T* src, long long spitch, cx<T>* dst, long long dpitch, int hout,
                      long long nrows, T scale, const char* name, double bytes) {
  const dim3 grid = row_grid<T, K>(nrows);
  LaunchScope ls(c, name, bytes);
  hipLaunchKernelGGL((k_row_r2c<T, K>), grid, dim3(RowBlk<T, K>::THREADS), 0, c.stream, src, spitch, dst, dpitch, hout, nrows, scale,
                     c.twiddles<T>(K), c.twiddles<T>(2 * K));
  check_launch(name);
}

template <typename T, int K>
void launch_row_c2r_K(Ctx& c, const cx<T>* src, long long spitch, int hin, T* dst, long long dpitch,
                      long long nrows, T scale, const char* name, double bytes) {
  const dim3 grid = row_grid<T, K>(nrows);
  LaunchScope ls(c, name, bytes);
  hipLaunchKernelGGL((k_row_c2r<T, K>), grid, dim3(RowBlk<T, K>::THREADS), 0, c.stream, src, spitch, hin, dst, dpitch, nrows, scale,
                     c.twiddles<T>(K), c.twiddles<T>(2 * K));
  check_launch(name);
}

template <typename T, int K>
void launch_row_prod_K(Ctx& c, const cx<T>* a, const cx<T>* b, long long spitch, int hin, cx<T>* dst,
                       long long dpitch, int hout, long long nrows, const char* name, double bytes) {
  const dim3 grid = row_grid<T, K>(nrows);
  LaunchScope ls(c, name, bytes);
  hipLaunchKernelGGL((k_row_prod<T, K>), grid, dim3(RowBlk<T, K>::THREADS), 0, c.stream, a, b, spitch, hin, dst, dpitch, hout, nrows,
                     c.twiddles<T>(K), c.twiddles<T>(2 * K));
  check_launch(name);
}

// rows of a length without tuned kernels go to the run-time schedules (GEN)
#define MFX_ROW_SWITCH(K, CALL, GEN) \
  switch (K) {                       \
    MFX_ROW_LENGTHS(CALL)            \
    default:                         \
      GEN;                           \
  }

template <typename T>
void launch_row_r2c(Ctx& c, int K, const T* src, long long spitch, cx<T>* dst, long long dpitch, int hout,
                    long long nrows, T scale, const char* name, double bytes) {
#define MFX_CASE(KK)                                                                              \
  case KK:                                                                                        \
    launch_row_r2c_K<T, KK>(c, src, spitch, dst, dpitch, hout, nrows, scale, name, bytes);       \
    return;
  MFX_ROW_SWITCH(K, MFX_CASE, launch_row_r2c_any<T>(c, K, src, spitch, dst, dpitch, hout, nrows, scale, name, bytes))
#undef MFX_CASE
}

template <typename T>
void launch_row_c2r(Ctx& c, int K, const cx<T>* src, long long spitch, int hin, T* dst, long long dpitch,
                    long long nrows, T scale, const char* name, double bytes) {
#define MFX_CASE(KK)                                                                              \
  case KK:                                                                                        \
    launch_row_c2r_K<T, KK>(c, src, spitch, hin, dst, dpitch, nrows, scale, name, bytes);        \
    return;
  MFX_ROW_SWITCH(K, MFX_CASE, launch_row_c2r_any<T>(c, K, src, spitch, hin, dst, dpitch, nrows, scale, name, bytes))
#undef MFX_CASE
}

template <typename T, int K>
void launch_row_c2r_part_K(Ctx& c, const cx<T>* src, long long spitch, int hin, const PartOut& po, long long nrows,
                           T scale, double lunit, double qoff, const char* name, double bytes) {
  const dim3 grid = row_grid<T, K>(nrows);
  LaunchScope ls(c, name, bytes);
  hipLaunchKernelGGL((k_row_c2r_part<T, K>), grid, dim3(RowBlk<T, K>::THREADS), 0, c.stream, src, spitch, hin, po,
                     nrows, scale, lunit, qoff, c.twiddles<T>(K), c.twiddles<T>(2 * K));
  check_launch(name);
}

template <typename T>
void launch_row_c2r_part(Ctx& c, int K, const cx<T>* src, long long spitch, int hin, const PartOut& po,
                         long long nrows, T scale, double lunit, double qoff, const char* name, double bytes) {
#define MFX_CASE(KK)                                                                                  \
  case KK:                                                                                            \
    launch_row_c2r_part_K<T, KK>(c, src, spitch, hin, po, nrows, scale, lunit, qoff, name, bytes);    \
    return;
  MFX_ROW_SWITCH(K, MFX_CASE,
                 launch_row_c2r_part_any<T>(c, K, src, spitch, hin, po, nrows, scale, lunit, qoff, name, bytes))
#undef MFX_CASE
}

// mean: what launch_row_mean gave, or null
template <typename T>
void launch_row_prod(Ctx& c, int K, const cx<T>* a, const cx<T>* b, long long spitch, int hin, cx<T>* dst,
                     long long dpitch, int hout, long long nrows, const T* mean, const char* name, double bytes) {
#define MFX_CASE(KK)                                                                                \
  case KK:                                                                                          \
    launch_row_prod_K<T, KK>(c, a, b, spitch, hin, dst, dpitch, hout, nrows, name, bytes);        \
    return;
  MFX_ROW_SWITCH(K, MFX_CASE, 
                 launch_row_prod_any<T>(c, K, a, b, spitch, hin, dst, dpitch, hout, nrows, mean, name, bytes))
#undef MFX_CASE
}


}  // namespace mfx
