// mixed_kernels.hip -- transforms of lengths without tuned kernels: the choice
// of schedule and launch shape (mix_cfg) and the launches of the mixed-radix
// kernels (fft_mixed.hpp), or of the direct-DFT kernels (fft_generic.hpp) for
// lengths with a prime factor above 7.  The line between them is what the
// butterflies cover; where both can run the mixed-radix kernels are 2 to 12 times
// as fast (fft_mixed.hpp).
#include "fft_mixed.hpp"
#include "fft_generic.hpp"

#include <algorithm>

namespace mfx {

namespace {

// vector instructions of a radix-R butterfly and its twiddles, and its LDS
// traffic in the same units: the weights by which schedules are compared
double mix_cost(int R) {
  const double bf = R == 2 ? 4 : R == 3 ? 16 : R == 4 ? 16 : R == 5 ? 40 : R == 6 ? 44 : R == 7 ? 84 : R == 8 ? 64
                    : R == 9 ? 120 : R == 10 ? 100 : 136;
  return bf + 4.0 * (R - 1) + 6.0 * R;
}

// all ways to write m as a product of radices (not increasing), the cheapest
// kept; `last` (0: none) is a further fixed radix
struct Search {
  int L = 0, nthr = 0;  // nthr > 0: the butterflies are taken in rounds by that many threads
  int best_n = 0, best[MIX_STAGES];
  double best_cost = 1e300;
  int cur[MIX_STAGES];
  void go(int m, int maxr, int n, double cost) {
    if (m == 1) {
      if (cost < best_cost) {
        best_cost = cost;
        best_n = n;
        for (int i = 0; i < n; ++i) best[i] = cur[i];
      }
      return;
    }
    if (n == MIX_STAGES - 1) return;
    static const int radix[] = {12, 10, 9, 8, 7, 6, 5, 4, 3, 2};
    for (int R : radix)
      if (R <= maxr && m % R == 0) {
        cur[n] = R;
        // per line element, and a barrier for each stage
        const double c = nthr ? mix_cost(R) * ((L / R + nthr - 1) / nthr) * nthr / L + 60.0 * nthr / L
                              : mix_cost(R) / R + 3.0;
        go(m / R, R, n + 1, cost + c);
      }
  }
};

bool mix_plan(int L, int rmax, int fixed_last, MixPlan& p) {
  if (L < 4 || (fixed_last && (L % fixed_last || L == fixed_last))) return false;
  Search s;
  s.L = L;
  s.nthr = fixed_last ? L / fixed_last : 0;
  s.go(fixed_last ? L / fixed_last : L, rmax, 0, 0.0);
  if (!s.best_n) return false;
  int r[MIX_STAGES], n = s.best_n;
  for (int i = 0; i < n; ++i) r[i] = s.best[i];
  if (fixed_last) {
    r[n++] = fixed_last;
  } else {
    if (n == 1) {  // a single butterfly: the first and last stages differ, so split it
      int f = 2;
      while (f < r[0] && r[0] % f) ++f;
      if (f == r[0]) return false;
      r[1] = f;
      r[0] /= f;
      n = 2;
    }
    // an odd radix last: its butterflies read runs of slots that start in
    // different LDS banks
    for (int i = 0; i < n; ++i)
      if (r[i] % 2) {
        const int t = r[i];
        for (int q = i; q + 1 < n; ++q) r[q] = r[q + 1];
        r[n - 1] = t;
        break;
      }
    // an even radix first where there is one: it keeps a line's mean out of its
    // longest waves without the more costly odd form (mix_first_bf)
    if (r[0] % 2)
      for (int i = 1; i < n; ++i)
        if (r[i] % 2 == 0) {
          for (int q = i; q > 0; --q) std::swap(r[q], r[q - 1]);
          break;
        }
  }
  p = MixPlan{};
  p.L = L;
  p.nr = n;
  int P = 1;
  for (int i = 0; i < n; ++i) {
    p.R[i] = mix_div(r[i]);
    p.P[i] = P;
    P *= r[i];
    p.I[i] = mix_div(L / P);
    p.J[i] = mix_div(i + 1 < n ? L / P / r[n - 1] : 1);
  }
  return true;
}

// share of the butterfly slots that do work when `nthr` threads take the
// stages' butterflies in rounds
double mix_fill(const MixPlan& p, int nthr) {
  double work = 0, slots = 0;
  for (int i = 0; i < p.nr; ++i) {
    const int R = p.R[i].d, nb = p.L / R, rounds = (nb + nthr - 1) / nthr;
    work += mix_cost(R) * nb;
    slots += mix_cost(R) * rounds * nthr;
  }
  return work / slots;
}

template <typename T>
MixCfg make_cfg(int L, int kind) {
  MixCfg c;
  const int cs = (int)sizeof(cx<T>);
  if (!mix_plan(L, kind == MIX_Z ? MIX_ZMAX : MIX_RMAX<T>, kind == MIX_Z ? MIX_S<T> : 0, c.p)) return c;
  c.lc = 0;
  c.pairs = 1;
  if (kind == MIX_COL) {
    // the widest tile, up to 128-byte runs, that leaves room for three
    // workgroups on a compute unit; at least four columns where two fit
    const int wide = 128 / cs;
    auto bytes = [&](int lc) { return ((1LL << lc) + 1) * L * cs; };
    while ((2 << c.lc) <= wide && bytes(c.lc + 1) <= CU_LDS / 3) ++c.lc;
    while (c.lc < 2 && bytes(c.lc + 1) <= CU_LDS / 2) ++c.lc;
    if (bytes(c.lc) > CU_LDS) return c;
    const int C = 1 << c.lc, unit = C >= 64 ? 1 : 64 / C;
    double best = -1;
    for (int n = unit; n * C <= 1024; n += unit) {
      // idle slots cost little beside too few waves to hide the loads
      const double f = mix_fill(c.p, n) * (n * C >= 256 ? 1.0 : n * C / 256.0);
      if (f > best * 1.02 || (f >= best * 0.98 && n * C <= 512)) {
        best = f > best ? f : best;
        c.nthr = n;
      }
    }
    c.block = c.nthr * C;
    c.lds = (size_t)bytes(c.lc);
  } else {
    auto shape = [&](int nthr, int& pairs, int& block) {
      pairs = 256 / nthr;
      if (pairs < 1) pairs = 1;
      while (pairs > 1 && (pairs + 1LL) * L * cs > CU_LDS / 4) --pairs;
      block = (pairs * nthr + 63) / 64 * 64;
      return (double)pairs * nthr / block;
    };
    if (kind == MIX_Z) {
      c.nthr = L / MIX_S<T>;
      shape(c.nthr, c.pairs, c.block);
    } else {
      double best = -1;
      int most = 0;
      for (int i = 0; i < c.p.nr; ++i) most = std::max(most, L / c.p.R[i].d);
      for (int n = std::max(1, most / 4); n <= most && n <= 512; ++n) {
        int pairs, block;
        const double f = shape(n, pairs, block) * mix_fill(c.p, n);
        if (f >= best) {
          best = f;
          c.nthr = n;
          c.pairs = pairs;
          c.block = block;
        }
      }
      if (best < 0) return c;
    }
    c.lds = (size_t)(c.pairs + 1) * L * cs;
    if (c.block > 512 || c.lds > (size_t)CU_LDS) return c;
  }
  c.nthrd = mix_div(c.nthr);
  c.ok = true;
  return c;
}

}  // namespace

template <typename T>
const MixCfg& mix_cfg(Ctx& c, int L, int kind) {
  const auto key = std::make_tuple(L, (int)sizeof(T), kind);
  auto it = c.mix.find(key);
  if (it == c.mix.end()) it = c.mix.emplace(key, make_cfg<T>(L, kind)).first;
  return it->second;
}
template const MixCfg& mix_cfg<float>(Ctx&, int, int);
template const MixCfg& mix_cfg<double>(Ctx&, int, int);

// ------------------------------------------------------------------ columns
// The passes that only the fused engine runs, at lengths with a schedule (its own
// condition); the others take the direct-DFT kernel where there is none.
template <class Src>
struct EnginePass {
  static constexpr bool value = false;
};
template <typename T>
struct EnginePass<SrcHessY<T>> {
  static constexpr bool value = true;
};
template <typename T>
struct EnginePass<SrcSplit<T>> {
  static constexpr bool value = true;
};
template <typename T>
struct EnginePass<MultiSrc<T, MultiPow<T>>> {
  static constexpr bool value = true;
};

template <typename T, bool INV, class Src, class Dst>
void launch_col_any(Ctx& c, int L, Src s, Dst d, int ncols, int nbatch, const char* name, double bytes) {
  const MixCfg& m = mix_cfg<T>(c, L, MIX_COL);
  if (m.ok) {
    auto k = k_mix_col<T, INV, Src, Dst>;
    col_lds_prep(c, k, m.lds);
    set_stream(d, 1 << m.lc);
    LaunchScope ls(c, name, bytes);
    hipLaunchKernelGGL(k, dim3((ncols + (1 << m.lc) - 1) >> m.lc, nbatch), dim3(m.block), m.lds, c.stream, s, d,
                       c.twiddles<T>(L), ncols, m.p, m.lc, m.nthr);
    check_launch(name);
    return;
  }
  if constexpr (EnginePass<Src>::value) {
    throw Error(1, "unsupported transform length " + std::to_string(L));
  } else {
    const GenPlan plan = gen_plan(L);
    const int C = gen_col_tile<T>(L);
    const size_t lds = 2 * (size_t)L * C * sizeof(cx<T>);
    auto k = k_col_gen<T, INV, Src, Dst>;
    col_lds_prep(c, k, lds);
    LaunchScope ls(c, name, bytes);
    hipLaunchKernelGGL(k, dim3((ncols + C - 1) / C, nbatch), dim3(GEN_THREADS), lds, c.stream, s, d, c.twiddles<T>(L),
                       ncols, plan, C);
    check_launch(name);
  }
}

// only reached for lengths with a schedule: the fused engine runs no others
template <typename T>
void launch_turn_any(Ctx& c, int L, const TurnArgs<T>& a, int ncols, int nbatch, const char* name, double bytes) {
  const MixCfg& m = mix_cfg<T>(c, L, MIX_COL);
  MFX_REQUIRE(m.ok, "unsupported transform length " + std::to_string(L));
  auto k = k_mix_turn<T, TurnArgs<T>>;
  col_lds_prep(c, k, m.lds);
  LaunchScope ls(c, name, bytes);
  TurnArgs<T> ta = a;
  set_stream(ta, 1 << m.lc);
  hipLaunchKernelGGL(k, dim3((ncols + (1 << m.lc) - 1) >> m.lc, nbatch), dim3(m.block), m.lds, c.stream, ta,
                     c.twiddles<T>(L), ncols, m.p, m.lc, m.nthr);
  check_launch(name);
}

// the line sources and destinations in use
template <typename T>
using PadMult = SrcPad<T, true>;
template <typename T>
using PadOnly = SrcPad<T, false>;
template <typename T>
using PowSrc = MultiSrc<T, MultiPow<T>>;
template <typename T>
using PowDst = MultiDst<T, MultiPow<T>>;
#define MFX_COL_ANY(INV, S, D)                                                                               \
  template void launch_col_any<float, INV>(Ctx&, int, S<float>, D<float>, int, int, const char*, double); \
  template void launch_col_any<double, INV>(Ctx&, int, S<double>, D<double>, int, int, const char*, double);
MFX_COL_ANY(false, SrcPlain, DstPlain)
MFX_COL_ANY(false, SrcPlain, DstPhi1)
MFX_COL_ANY(false, SrcPlain, DstTrunc)
MFX_COL_ANY(false, SrcPlain, DstTruncOp)
MFX_COL_ANY(false, SrcPlain, DstTruncOpMean)
MFX_COL_ANY(true, SrcPlain, DstPlain)
MFX_COL_ANY(true, PadMult, DstPlain)
MFX_COL_ANY(true, PadOnly, DstPlain)
MFX_COL_ANY(true, SrcHessY, DstHessY)
MFX_COL_ANY(false, SrcSplit, DstTruncOp)
MFX_COL_ANY(true, PowSrc, PowDst)
#undef MFX_COL_ANY
template void launch_turn_any<float>(Ctx&, int, const TurnArgs<float>&, int, int, const char*, double);
template void launch_turn_any<double>(Ctx&, int, const TurnArgs<double>&, int, int, const char*, double);

// ------------------------------------------------------------------ rows
static MixRowArgs row_args(const MixCfg& m, long long nrows) { return MixRowArgs{m.p, m.nthrd, m.pairs, nrows}; }

static dim3 row_blocks(const MixCfg& m, long long nrows) {
  const long long nb = (nrows + 2LL * m.pairs - 1) / (2LL * m.pairs);
  MFX_REQUIRE(nb < (1LL << 31), "too many rows for one launch");
  return dim3((unsigned)nb);
}

// one launch of a row-pair kernel (lengths with a schedule) ...
#define MFX_MIX_ROW(KERNEL, M, ...)                                                                               \
  do {                                                                                                            \
    auto k_ = KERNEL<T>;                                                                                          \
    const dim3 nb_ = row_blocks(M, nrows);                                                                        \
    col_lds_prep(c, k_, (M).lds);                                                                                 \
    LaunchScope ls_(c, name, bytes);                                                                              \
    hipLaunchKernelGGL(k_, nb_, dim3((M).block), (M).lds, c.stream, __VA_ARGS__, row_args(M, nrows),              \
                       c.twiddles<T>(2 * K));                                                                     \
    check_launch(name);                                                                                           \
  } while (0)

// ... or of a direct-DFT one, one row per workgroup
#define MFX_GEN_ROW(KERNEL, NBUF, ...)                                                                            \
  do {                                                                                                            \
    const GenPlan plan_ = gen_plan(K);                                                                            \
    const size_t lds_ = gen_row_lds<T>(K, NBUF);                                                                  \
    auto k_ = KERNEL<T>;                                                                                          \
    col_lds_prep(c, k_, lds_);                                                                                    \
    MFX_REQUIRE(nrows < (1LL << 31), "too many rows for one launch");                                             \
    LaunchScope ls_(c, name, bytes);                                                                              \
    hipLaunchKernelGGL(k_, dim3((unsigned)nrows), dim3(GEN_THREADS), lds_, c.stream, __VA_ARGS__, plan_,          \
                       c.twiddles<T>(K), c.twiddles<T>(2 * K));                                                   \
    check_launch(name);                                                                                           \
  } while (0)

template <typename T>
void launch_row_r2c_any(Ctx& c, int K, const T* src, long long spitch, cx<T>* dst, long long dpitch, int hout,
                        long long nrows, T scale, const char* name, double bytes) {
  const MixCfg& m = mix_cfg<T>(c, 2 * K, MIX_ROW);
  if (m.ok)
    MFX_MIX_ROW(k_mix_r2c, m, src, spitch, dst, dpitch, hout, scale);
  else
    MFX_GEN_ROW(k_row_r2c_gen, 2, src, spitch, dst, dpitch, hout, scale);
}

template <typename T>
void launch_row_c2r_any(Ctx& c, int K, const cx<T>* src, long long spitch, int hin, T* dst, long long dpitch,
                        long long nrows, T scale, const char* name, double bytes) {
  const MixCfg& m = mix_cfg<T>(c, 2 * K, MIX_ROW);
  MFX_REQUIRE(!m.ok || hin == K + 1, "the row kernel reads whole half spectra");
  if (m.ok)
    MFX_MIX_ROW(k_mix_c2r, m, src, spitch, hin, dst, dpitch, scale);
  else
    MFX_GEN_ROW(k_row_c2r_gen, 2, src, spitch, hin, dst, dpitch, scale);
}

template <typename T>
void launch_row_c2r_part_any(Ctx& c, int K, const cx<T>* src, long long spitch, int hin, const PartOut& po,
                             long long nrows, T scale, double lunit, double qoff, const char* name, double bytes) {
  const MixCfg& m = mix_cfg<T>(c, 2 * K, MIX_ROW);
  MFX_REQUIRE(!m.ok || hin == K + 1, "the row kernel reads whole half spectra");
  if (m.ok)
    MFX_MIX_ROW(k_mix_c2r_part, m, src, spitch, hin, po, scale, lunit, qoff);
  else
    MFX_GEN_ROW(k_row_c2r_part_gen, 2, src, spitch, hin, po, scale, lunit, qoff);
}

// whether rows of 2 K run the pair kernel of products: the half spectra of an n-grid
// padded to 2 K = 3n/2
static bool mix_prod_rows(const MixCfg& m, int K, int hin) { return m.ok && hin == 2 * K / 3 + 1; }

// A product's mean is as large as the product itself, and the y pass rounds its sums
// over a plane at that size before they meet along x: 0.8 units of 2^-24 of the mean a
// plane, which decided the error of the product's longest waves.  With the mean (to
// the few per cent that MIX_MEAN_ROWS rows give) taken off before the transform and
// added to the k = 0 mode after it, the rounding is that of the rest.  The 2LPT source
// of a 160^3 FP32 grid by separate convolutions, median and maximum error over 20
// seeds: 3.1e-7 and 3.5e-7, with the mean 7.8e-7 and 1.5e-6; of 240^3 3.4e-7 and 4.3e-7,
// with it 1.4e-6 and 2.0e-6.  The launch takes 5 us a product (160^3: 180 us).  FP64
// results err by 1e-15 either way.
template <typename T>
bool launch_row_mean(Ctx& c, int K, const cx<T>* a, const cx<T>* b, long long spitch, int hin, long long nrows,
                     T* mean, const char* name) {
  if constexpr (sizeof(T) == 8) return false;
  switch (K) {
#define MFX_CASE(KK) case KK:
    MFX_ROW_LENGTHS(MFX_CASE)
#undef MFX_CASE
    return false;
  }
  if (!mix_prod_rows(mix_cfg<T>(c, 2 * K, MIX_Z), K, hin)) return false;
  MFX_REQUIRE(nrows == 4LL * K * K, "the rows are not those of a cube");
  LaunchScope ls(c, name, 0);
  hipLaunchKernelGGL(k_mix_mean<T>, dim3(1), dim3(1024), 0, c.stream, a, b, spitch, hin, 2 * K, mean);
  check_launch(name);
  return true;
}
template bool launch_row_mean<float>(Ctx&, int, const cx<float>*, const cx<float>*, long long, int, long long, float*,
                                     const char*);
template bool launch_row_mean<double>(Ctx&, int, const cx<double>*, const cx<double>*, long long, int, long long,
                                      double*, const char*);

template <typename T>
void launch_row_prod_any(Ctx& c, int K, const cx<T>* a, const cx<T>* b, long long spitch, int hin, cx<T>* dst,
                         long long dpitch, int hout, long long nrows, const T* mean, const char* name, double bytes) {
  const MixCfg& m = mix_cfg<T>(c, 2 * K, MIX_Z);
  if (mix_prod_rows(m, K, hin))
    MFX_MIX_ROW(k_mix_prod, m, a, b, spitch, dst, dpitch, hout, mean);
  else
    MFX_GEN_ROW(k_row_prod_gen, 4, a, b, spitch, hin, dst, dpitch, hout);
}

#define MFX_ROW_ANY(T)                                                                                             \
  template void launch_row_r2c_any<T>(Ctx&, int, const T*, long long, cx<T>*, long long, int, long long, T,        \
                                      const char*, double);                                                        \
  template void launch_row_c2r_any<T>(Ctx&, int, const cx<T>*, long long, int, T*, long long, long long, T,        \
                                      const char*, double);                                                        \
  template void launch_row_c2r_part_any<T>(Ctx&, int, const cx<T>*, long long, int, const PartOut&, long long, T,  \
                                           double, double, const char*, double);                                   \
  template void launch_row_prod_any<T>(Ctx&, int, const cx<T>*, const cx<T>*, long long, int, cx<T>*, long long,   \
                                       int, long long, const T*, const char*, double);
MFX_ROW_ANY(float)
MFX_ROW_ANY(double)
#undef MFX_ROW_ANY

}  // namespace mfx
