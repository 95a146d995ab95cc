// mix_plan.hpp -- run-time schedules of the mixed-radix transforms
// (fft_mixed.hpp): the stage radices of a length and the launch shape chosen
// for it.
#pragma once
#include <hip/hip_runtime.h>

#include <cstddef>

namespace mfx {

constexpr int MIX_STAGES = 8;

// x / d for x d < 2^32 as the high word of x * mg (mg = ceil(2^32 / d)); d = 1
// has no 32-bit mg and is told apart by mg = 0
struct MixDiv {
  int d;
  unsigned mg;
  __device__ __forceinline__ int operator()(int x) const { return mg ? (int)__umulhi((unsigned)x, mg) : x; }
};
inline MixDiv mix_div(int d) {
  return MixDiv{d, d > 1 ? (unsigned)(((1ull << 32) + (unsigned)d - 1) / (unsigned)d) : 0u};
}

struct MixPlan {
  int L, nr;
  MixDiv R[MIX_STAGES];  // radices in DIF order
  int P[MIX_STAGES];     // product of the earlier radices
  MixDiv I[MIX_STAGES];  // product of the later radices (the slot stride of a butterfly)
  MixDiv J[MIX_STAGES];  // I without the last radix: the digits of a last-stage butterfly
};

// what a plan is made for: column tiles, row pairs, and the fused row kernels
// whose last radix is fixed (MIX_S) and whose threads own one butterfly of it
enum { MIX_COL = 0, MIX_ROW = 1, MIX_Z = 2 };
template <typename T>
constexpr int MIX_S = sizeof(T) == 4 ? 6 : 3;

struct MixCfg {
  bool ok = false;  // false: the length has no schedule (a prime factor above 7, or a single stage)
  MixPlan p;
  int lc;        // columns: log2 of the tile width
  int nthr;      // threads per column or per row pair
  MixDiv nthrd;  // the same as a divisor
  int pairs;     // rows: pairs per workgroup
  int block;     // threads per workgroup
  size_t lds;    // dynamic LDS bytes
};

struct Ctx;
// the schedule and launch shape for a length, made once per context
template <typename T>
const MixCfg& mix_cfg(Ctx& c, int L, int kind);

}  // namespace mfx
