// The planned passes at the grid lengths without tuned variants: every even
// length 2^a 3^b 5^c 7^d from 8 to 512 that matvec.hip does not plan itself.
// Compiled several times (DDA_PLAN_PART = 0 .. 7: the precision and a quarter
// of the lengths each), so that the parts build in parallel.
//
// A length runs as two stages of nearly equal radices wherever both are at
// most 28, so that a transform passes through LDS once (the run-time planned
// kernels: once per radix and twice more to load and store). The FP64 Z pass, which
// holds three components in registers, takes three smaller radices above 256
// points (two of 18 .. 28 would leave one wave per SIMD).
#include "passes.hpp"
#include "plan_list.hpp"

#ifndef DDA_PLAN_PART
#define DDA_PLAN_PART 0
#endif

namespace dda {

namespace {

#if DDA_PLAN_PART < 4
typedef float Real;
constexpr int kPrec = 32;
#else
typedef double Real;
constexpr int kPrec = 64;
#endif

template <int N, typename PL, typename PZ>
const AxisOps* ops_of() {
  static const AxisOps ops = {launch_gen_col<Real, N, PL>,
                              launch_pass3_plan<Real, N, PZ, gen_cols<Real, N, PZ::TPC>(16)>,
                              launch_x_plan<Real, N, PL>, PZ::TPC};
  return &ops;
}

}  // namespace

const AxisOps* DDA_CAT(axis_ops_part, DDA_PLAN_PART)(int n, int prec) {
  if (prec != kPrec) return nullptr;
  switch (n) {
#define X(N, L, Z)                                                                                                 \
  case N:                                                                                                          \
    return ops_of<N, GenPlan<N, DDA_ARGS L>, std::conditional_t<kPrec == 64, GenPlan<N, DDA_ARGS Z>, GenPlan<N, DDA_ARGS L>>>();
#if DDA_PLAN_PART % 4 == 0
    DDA_GEN_SIZES_0(X)
#elif DDA_PLAN_PART % 4 == 1
    DDA_GEN_SIZES_1(X)
#elif DDA_PLAN_PART % 4 == 2
    DDA_GEN_SIZES_2(X)
#else
    DDA_GEN_SIZES_3(X)
#endif
#undef X
    default:
      return nullptr;
  }
}

}  // namespace dda
