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

#ifndef DDA_PLAN_PART
#define DDA_PLAN_PART 0
#endif

// N, the plan of the X and Y passes (and the Z pass), the FP64 Z pass's plan
#define DDA_GEN_SIZES_0(X)                                                                              \
  X(8, (4, 2), (4, 2)) X(10, (2, 5), (2, 5)) X(12, (4, 3), (4, 3)) X(14, (2, 7), (2, 7))                 \
  X(16, (4, 4), (4, 4)) X(18, (6, 3), (6, 3)) X(20, (4, 5), (4, 5)) X(24, (6, 4), (6, 4))                \
  X(28, (4, 7), (4, 7)) X(30, (6, 5), (6, 5)) X(36, (6, 6), (6, 6)) X(40, (8, 5), (8, 5))                \
  X(42, (6, 7), (6, 7)) X(50, (10, 5), (10, 5)) X(54, (6, 9), (6, 9)) X(56, (8, 7), (8, 7))              \
  X(60, (10, 6), (10, 6)) X(70, (10, 7), (10, 7))
#define DDA_GEN_SIZES_1(X)                                                                              \
  X(72, (8, 9), (8, 9)) X(80, (10, 8), (10, 8)) X(84, (12, 7), (12, 7)) X(90, (10, 9), (10, 9))          \
  X(98, (14, 7), (14, 7)) X(100, (10, 10), (10, 10)) X(108, (12, 9), (12, 9)) X(112, (14, 8), (14, 8))   \
  X(120, (12, 10), (12, 10)) X(126, (14, 9), (14, 9)) X(140, (14, 10), (14, 10))                         \
  X(144, (12, 12), (12, 12)) X(150, (10, 15), (10, 15)) X(160, (16, 10), (16, 10))
#define DDA_GEN_SIZES_2(X)                                                                              \
  X(162, (18, 9), (18, 9)) X(168, (14, 12), (14, 12)) X(180, (12, 15), (12, 15)) X(196, (14, 14), (14, 14)) \
  X(200, (20, 10), (20, 10)) X(210, (14, 15), (14, 15)) X(216, (18, 12), (18, 12))                       \
  X(224, (16, 14), (16, 14)) X(240, (16, 15), (16, 15)) X(250, (10, 25), (10, 5, 5))                     \
  X(252, (18, 14), (18, 14)) X(270, (18, 15), (6, 5, 9)) X(280, (20, 14), (8, 5, 7))
#define DDA_GEN_SIZES_3(X)                                                                              \
  X(288, (18, 16), (6, 6, 8)) X(294, (14, 21), (6, 7, 7)) X(300, (20, 15), (6, 5, 10))                   \
  X(320, (20, 16), (8, 5, 8)) X(324, (18, 18), (6, 6, 9)) X(336, (16, 21), (6, 7, 8))                    \
  X(350, (14, 25), (10, 5, 7)) X(360, (20, 18), (8, 5, 9)) X(378, (18, 21), (6, 7, 9))                   \
  X(384, (24, 16), (6, 8, 8)) X(392, (28, 14), (8, 7, 7)) X(400, (20, 20), (8, 5, 10))                   \
  X(420, (20, 21), (6, 7, 10)) X(432, (24, 18), (6, 8, 9)) X(448, (28, 16), (8, 7, 8))                   \
  X(450, (18, 25), (10, 5, 9)) X(480, (24, 20), (6, 8, 10)) X(486, (18, 27), (6, 9, 9))                  \
  X(490, (10, 7, 7), (10, 7, 7)) X(500, (20, 25), (10, 5, 10)) X(504, (24, 21), (8, 7, 9))

#define DDA_CAT2(a, b) a##b
#define DDA_CAT(a, b) DDA_CAT2(a, b)
#define DDA_ARGS(...) __VA_ARGS__

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
                              launch_x_plan<Real, N, PL>};
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
