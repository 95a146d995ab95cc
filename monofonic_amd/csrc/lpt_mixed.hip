// lpt_mixed.hip -- the z stages of the fused LPT engine for padded lengths
// without tuned kernels (any n divisible by 4 whose factors are at most 7):
// the stages A and C of lpt_engine.hip on pairs of rows (MixZ).
//
// Each stage is ONE loop over its transforms, so that a transform's code (with
// the switch over its radices) exists once in a kernel; what is done with the
// points is a uniform switch on the loop index, and every operand stays in
// registers.
//
// Before, these sizes ran the convolve sequence: 33 two-operand products of 3LPT,
// each with its own padded transforms.  3LPT sources of a 384^3 FP32 grid
// (padded 576^3): 130 ms by the sequence on the generic kernels, 20.5 ms here, of
// which stage A takes 4.0 ms (3 waves per SIMD) and stage C 8.4 ms (2 waves per
// SIMD); a whole 200^3 FP64 3LPT realisation 108 ms and 7.0 ms.  Both stages are
// bound by the latency of a transform's stages (two to four barriers each) at
// that occupancy, not by memory (1.7 TB/s in stage C).
#include "fft_mixed.hpp"
#include "lpt_common.hpp"

namespace mfx {

// Hessian component order xx, yy, zz, xy, xz, yz (cs): its Y array by selects,
// which keep the kernel argument out of private memory
template <typename T>
__device__ __forceinline__ const cx<T>* mix_hess_row(const FieldY<T>& f, int o) {
  const cx<T>* y = f.y[hess_idx(0, 0)];
  y = o == 1 ? f.y[hess_idx(1, 1)] : y;
  y = o == 2 ? f.y[hess_idx(2, 2)] : y;
  y = o == 3 ? f.y[hess_idx(0, 1)] : y;
  y = o == 4 ? f.y[hess_idx(0, 2)] : y;
  y = o == 5 ? f.y[hess_idx(1, 2)] : y;
  return y;
}
// a or b by value: a conditional on array elements themselves selects their
// addresses and puts the arrays into scratch
template <typename T>
__device__ __forceinline__ cx<T> mix_pick(bool c, cx<T> a, cx<T> b) {
  return mk(c ? a.x : b.x, c ? a.y : b.y);
}
__device__ __forceinline__ int mix_hess_pz(int o) { return o == 2 ? 2 : (o >= 4 ? 1 : 0); }

// stage A (k_lpt_zA): S2 and, for 3LPT, I1..I4 and the stored real rows.  The
// stored rows are only read by stage C, so they keep the threads' order: point
// q of thread t of a pair at q nthr + t.
template <typename T, bool THREE>
__global__ void __launch_bounds__(512)
    k_mix_zA(FieldY<T> f, cx<T>* S2, cx<T>* I1, cx<T>* I2, cx<T>* I3, cx<T>* I4, cx<T>* R, long long rstride,
             long long pitch, int hin, int n, T kfac, MixRowArgs ra, const cx<T>* __restrict__ tw) {
  extern __shared__ __align__(16) unsigned char col_lds_raw[];
  constexpr int S = MixZ<T>::S;
  const MixRow<T> r(ra, reinterpret_cast<cx<T>*>(col_lds_raw));
  const MixZ<T> z{r, ra.p};
  const long long oa = r.ra * pitch, ob = r.rb * pitch;
  // m: phi_xx, then phi_xx + phi_yy, then phi_xy; d: phi_xx phi_yy
  cx<T> m[S], d[S], s2[S], v[S];
  typename MixZ<T>::Raw w;
  z.fetch(w, mix_hess_row(f, 0), pitch);
  mix_copy_table(r.lt, tw, ra.p.L);
#pragma unroll
  for (int q = 0; q < S; ++q) m[q] = d[q] = s2[q] = mk(T(0), T(0));
#pragma unroll 1
  for (int o = 0; o < 6; ++o) {
    z.c2r(v, w, KzMul<T>{n, mix_hess_pz(o), kfac, T(-1)});
    if (o < 5) z.fetch(w, mix_hess_row(f, o + 1), pitch);
    if (THREE && r.actA && r.t < r.nthr) {
      cx<T>* dst = R + o * rstride + (r.ra >> 1) * ra.p.L + r.t;
#pragma unroll
      for (int q = 0; q < S; ++q) dst[q * r.nthr] = v[q];
    }
    if (o == 1) {
#pragma unroll
      for (int q = 0; q < S; ++q) d[q] = mix_pmul(m[q], v[q]);
    }
    if (o == 2) {
#pragma unroll
      for (int q = 0; q < S; ++q) s2[q] = d[q] + mix_pmul(m[q], v[q]);
    }
    if (o > 2) {
#pragma unroll
      for (int q = 0; q < S; ++q) s2[q] = s2[q] - mix_pmul(v[q], v[q]);
    }
    if (o == 0 || o == 3) {
#pragma unroll
      for (int q = 0; q < S; ++q) m[q] = v[q];
    } else if (o == 1) {
#pragma unroll
      for (int q = 0; q < S; ++q) m[q] = m[q] + v[q];
    }
    // products that are complete now: I1 after xy, I2 and I4 after xz, I3 and
    // S2 after yz
    const int ne = o < 3 ? 0 : (THREE ? (o == 3 ? 1 : 2) : (o == 5 ? 1 : 0));
#pragma unroll 1
    for (int e = 0; e < ne; ++e) {
      const bool last = o == 5 && (e == 1 || !THREE);
      cx<T>* out = last ? S2 : o == 3 ? I1 : o == 4 ? (e == 0 ? I2 : I4) : I3;
      cx<T> u[S];
#pragma unroll
      for (int q = 0; q < S; ++q) {
        const cx<T> sq = mix_pmul(v[q], v[q]);
        const cx<T> p = mix_pick(o == 3, d[q] - sq, mix_pmul(m[q], v[q]));
        u[q] = mix_pick(last, s2[q], mix_pick(o == 3 || (o == 4 && e == 0), p, sq));
      }
      z.r2c(u, out + oa, out + ob, hin);
    }
  }
}

// stage C over the stored rows (k_lpt_zC): steps 0..5 transform phi2's Hessian
// rows, steps 6..11 take phi's stored rows one by one with, for xx, yy, zz and
// yz, the intermediate paired with them
template <typename T>
__global__ void __launch_bounds__(512)
    k_mix_zC(FieldY<T> f2, const cx<T>* R, long long rstride, cx<T>* I1, cx<T>* I2, cx<T>* I3, cx<T>* I4,
             long long pitch, int hin, int n, T kfac, MixRowArgs ra, const cx<T>* __restrict__ tw) {
  extern __shared__ __align__(16) unsigned char col_lds_raw[];
  constexpr int S = MixZ<T>::S;
  const MixRow<T> r(ra, reinterpret_cast<cx<T>*>(col_lds_raw));
  const MixZ<T> z{r, ra.p};
  typename MixZ<T>::Raw w;
  z.fetch(w, mix_hess_row(f2, 0), pitch);
  mix_copy_table(r.lt, tw, ra.p.L);
  const long long oa = r.ra * pitch, ob = r.rb * pitch;
  const cx<T>* const stored = R + (r.ra >> 1) * ra.p.L + (r.t < r.nthr ? r.t : 0);
  const T c57 = T(5.0 / 7.0), c107 = T(10.0 / 7.0);
  cx<T> h[6][S], p3[S], ax[S], ay[S], az[S], v[S];
#pragma unroll
  for (int q = 0; q < S; ++q) {
#pragma unroll
    for (int c = 0; c < 6; ++c) h[c][q] = mk(T(0), T(0));
    p3[q] = ax[q] = ay[q] = az[q] = mk(T(0), T(0));
  }
#pragma unroll 1
  for (int step = 0; step < 12; ++step) {
    const int o = step - 6;
    const bool hess = step < 6;
    if (hess || o < 3 || o == 5) {
      z.c2r(v, w, KzMul<T>{n, hess ? mix_hess_pz(step) : 0, kfac, hess ? T(-1) : T(1)});
      // the next operand: phi2's rows, then I3, I4, I1, I2
      if (o < 5) z.fetch(w, step < 5 ? mix_hess_row(f2, step + 1) : o < 0 ? I3 : o == 0 ? I4 : o == 1 ? I1 : I2, pitch);
    }
    if (hess) {
#define MFX_KEEP(c)                                   \
  if (step == c) {                                    \
    _Pragma("unroll") for (int q = 0; q < S; ++q) h[c][q] = v[q]; \
  }
      MFX_KEEP(0) MFX_KEEP(1) MFX_KEEP(2) MFX_KEEP(3) MFX_KEEP(4) MFX_KEEP(5)
#undef MFX_KEEP
      continue;
    }
    cx<T> a[S];
#pragma unroll
    for (int q = 0; q < S; ++q) a[q] = stored[o * rstride + q * r.nthr];
    if (o == 0) {
#pragma unroll
      for (int q = 0; q < S; ++q) {
        p3[q] = mix_pmul(a[q], h[1][q] + h[2][q]) * (-c57) - mix_pmul(a[q], v[q]);
        ay[q] = mix_pmul(h[4][q], a[q]);
        az[q] = mk(T(0), T(0)) - mix_pmul(h[3][q], a[q]);
      }
    } else if (o == 1) {
#pragma unroll
      for (int q = 0; q < S; ++q) {
        p3[q] = p3[q] - mix_pmul(a[q], h[0][q] + h[2][q]) * c57 - mix_pmul(a[q], v[q]);
        ax[q] = ax[q] - mix_pmul(h[5][q], a[q]);
        az[q] = az[q] + mix_pmul(h[3][q], a[q]);
      }
    } else if (o == 2) {
#pragma unroll
      for (int q = 0; q < S; ++q) {
        p3[q] = p3[q] - mix_pmul(a[q], h[0][q] + h[1][q]) * c57 + mix_pmul(a[q], v[q]);
        ax[q] = ax[q] + mix_pmul(h[5][q], a[q]);
        ay[q] = ay[q] - mix_pmul(h[4][q], a[q]);
      }
    } else if (o == 3) {
#pragma unroll
      for (int q = 0; q < S; ++q) {
        p3[q] = p3[q] + mix_pmul(a[q], h[3][q]) * c107;
        ax[q] = ax[q] - mix_pmul(h[4][q], a[q]);
        ay[q] = ay[q] + mix_pmul(h[5][q], a[q]);
        az[q] = az[q] + mix_pmul(a[q], h[0][q] - h[1][q]);
      }
    } else if (o == 4) {
#pragma unroll
      for (int q = 0; q < S; ++q) {
        p3[q] = p3[q] + mix_pmul(a[q], h[4][q]) * c107;
        ax[q] = ax[q] + mix_pmul(h[3][q], a[q]);
        ay[q] = ay[q] + mix_pmul(a[q], h[2][q] - h[0][q]);
        az[q] = az[q] - mix_pmul(h[5][q], a[q]);
      }
    } else {
#pragma unroll
      for (int q = 0; q < S; ++q) {
        p3[q] = p3[q] + mix_pmul(a[q], h[5][q]) * c107 + mix_pmul(a[q], v[q]) * T(2);
        ax[q] = ax[q] + mix_pmul(a[q], h[1][q] - h[2][q]);
        ay[q] = ay[q] - mix_pmul(h[3][q], a[q]);
        az[q] = az[q] + mix_pmul(h[4][q], a[q]);
      }
    }
  }
  // phi3 -> I1, A3x -> I2, A3y -> I3, A3z -> I4: every row has been read
#pragma unroll 1
  for (int e = 0; e < 4; ++e) {
    cx<T>* out = e == 0 ? I1 : e == 1 ? I2 : e == 2 ? I3 : I4;
    cx<T> u[S];
#pragma unroll
    for (int q = 0; q < S; ++q) u[q] = mix_pick(e < 2, mix_pick(e == 0, p3[q], ax[q]), mix_pick(e == 2, ay[q], az[q]));
    z.r2c(u, out + oa, out + ob, hin);
  }
}

static dim3 z_blocks(const MixCfg& m, long long nrows) {
  return dim3((unsigned)((nrows + 2LL * m.pairs - 1) / (2LL * m.pairs)));
}

template <typename T>
void launch_zA_mix(Ctx& c, const FieldY<T>& f, cx<T>* S2, cx<T>* const* I, bool three, cx<T>* R, long long rstride,
                   long long pitch, int hin, int n, T kfac, long long nrows, double bytes) {
  const int L = 3 * n / 2;
  const MixCfg& m = mix_cfg<T>(c, L, MIX_Z);
  MFX_REQUIRE(m.ok, "unsupported padded length " + std::to_string(L));
  MFX_REQUIRE(!three || R, "the mixed-radix 3LPT stages run the stored path");
  const MixRowArgs ra{m.p, m.nthrd, m.pairs, nrows};
  auto k = three ? k_mix_zA<T, true> : k_mix_zA<T, false>;
  col_lds_prep(c, k, m.lds);
  LaunchScope ls(c, "lpt_zA", bytes);
  hipLaunchKernelGGL(k, z_blocks(m, nrows), dim3(m.block), m.lds, c.stream, f, S2, three ? I[0] : S2,
                     three ? I[1] : S2, three ? I[2] : S2, three ? I[3] : S2, R, rstride, pitch, hin, n, kfac, ra,
                     c.twiddles<T>(L));
  check_launch("lpt_zA");
}

template <typename T>
void launch_zC_mix(Ctx& c, const FieldY<T>& f2, const cx<T>* R, long long rstride, cx<T>* const* I, long long pitch,
                   int hin, int n, T kfac, long long nrows, double bytes) {
  const int L = 3 * n / 2;
  const MixCfg& m = mix_cfg<T>(c, L, MIX_Z);
  MFX_REQUIRE(m.ok, "unsupported padded length " + std::to_string(L));
  const MixRowArgs ra{m.p, m.nthrd, m.pairs, nrows};
  auto k = k_mix_zC<T>;
  col_lds_prep(c, k, m.lds);
  LaunchScope ls(c, "lpt_zC", bytes);
  hipLaunchKernelGGL(k, z_blocks(m, nrows), dim3(m.block), m.lds, c.stream, f2, R, rstride, I[0], I[1], I[2], I[3],
                     pitch, hin, n, kfac, ra, c.twiddles<T>(L));
  check_launch("lpt_zC");
}

#define MFX_Z_MIX(T)                                                                                               \
  template void launch_zA_mix<T>(Ctx&, const FieldY<T>&, cx<T>*, cx<T>* const*, bool, cx<T>*, long long, long long, \
                                 int, int, T, long long, double);                                                  \
  template void launch_zC_mix<T>(Ctx&, const FieldY<T>&, const cx<T>*, long long, cx<T>* const*, long long, int,   \
                                 int, T, long long, double);
MFX_Z_MIX(float)
MFX_Z_MIX(double)
#undef MFX_Z_MIX

}  // namespace mfx
