// lpt_common.hpp -- what the z stages of the fused LPT engine share: the Hessian
// rows of a field and their kz factors (lpt_engine.hip: the lengths with tuned
// kernels; lpt_mixed.hip: the mixed-radix ones).
#pragma once
#include "fft_passes.hpp"
#include "ops.hpp"

namespace mfx {

// Y arrays of one field: 0 -> Y0, 1 -> Yx, 2 -> Yy, 3 -> Yxx, 4 -> Yxy, 5 -> Yyy
template <typename T>
struct FieldY {
  const cx<T>* y[6];
};

// Hessian component (a,b) -> Y array and kz power
constexpr int hess_idx(int a, int b) {
  return (a > b) ? hess_idx(b, a)
                 : (a == 0 && b == 0) ? 3
                 : (a == 1 && b == 1) ? 5
                 : (a == 2 && b == 2) ? 0
                 : (a == 0 && b == 1) ? 4
                 : (a == 0 && b == 2) ? 1
                                      : 2;
}
constexpr int hess_pz(int a, int b) { return (a == 2) + (b == 2); }

template <typename T>
struct KzMul {
  int n, pz;
  T kfac, sgn;
  __device__ __forceinline__ T operator()(int k) const {
    T g = kval<T>(k, n, kfac, 1);
    return pz == 0 ? sgn : (pz == 1 ? sgn * g : sgn * g * g);
  }
};

namespace cs {
// stored component order xx, yy, zz, xy, xz, yz
constexpr int ca[6] = {0, 1, 2, 0, 0, 1};
constexpr int cb[6] = {0, 1, 2, 1, 2, 2};
}  // namespace cs

// z stages of padded lengths without tuned kernels (lpt_mixed.hip)
template <typename T>
void launch_zA_mix(Ctx& c, const FieldY<T>& f, cx<T>* S2, cx<T>* const* I, bool three, cx<T>* R, long long rstride,
                   long long pitch, int hin, int n, T kfac, long long nrows, double bytes);
template <typename T>
void launch_zC_mix(Ctx& c, const FieldY<T>& f2, const cx<T>* R, long long rstride, cx<T>* const* I, long long pitch,
                   int hin, int n, T kfac, long long nrows, double bytes);

}  // namespace mfx
