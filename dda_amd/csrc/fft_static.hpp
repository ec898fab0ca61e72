// Compile-time planned Stockham FFT for the column passes.
//
// A transform of length N = R0 * R1 * ... over a tile of T adjacent columns.
// Every thread owns PPT points of one column in every stage (PPT divisible by
// each radix), so a stage is PPT / R butterflies per thread: butterfly
// j_i = t + i * TPC, TPC = N / PPT threads per column (general plans, below, let
// the threads a stage has no butterfly for sit it out). The first stage takes its
// inputs x[j + m N / R0] from registers the caller filled (straight from HBM),
// the last stage leaves X[j + m N / R_last] in registers, and only the stages
// in between pass through LDS. Running the inverse with the radices reversed
// makes its first stage consume exactly the points the forward transform left
// in a thread's registers, so FFT -> pointwise product -> inverse FFT needs no
// exchange in the middle. Twiddles W_{Ns R}^{m k} come from the host's table
// of N roots of unity; the constants of the in-register DFTs are evaluated at
// compile time.
#pragma once

#include "common.hpp"

namespace dda {

// ------------------------------------------------------------------------------------
// The roots of unity of the in-register DFTs, at compile time: cos and sin(2 pi t / n)
// by exact octant reduction of t / n and Taylor series on [0, pi / 4], in sums of
// two doubles (the error-free sum and product of Knuth and Dekker), so that each is
// the closest double. (In plain double half of them came out a unit or two in the
// last place off, cos(2 pi / 3) among them, which made the FP64 products at
// lengths of the factors 3 and 4 up to 1.4 times as far from the exact ones.)
// ------------------------------------------------------------------------------------
struct TwoDoubles {
  double hi, lo;
};
constexpr TwoDoubles two_sum(double a, double b) {
  const double s = a + b, t = s - a;
  return {s, (a - (s - t)) + (b - t)};
}
constexpr TwoDoubles two_prod(double a, double b) {
  const double k = 134217729.0;  // 2^27 + 1
  const double p = a * b, ca = k * a, cb = k * b;
  const double ah = ca - (ca - a), al = a - ah, bh = cb - (cb - b), bl = b - bh;
  return {p, ((ah * bh - p) + ah * bl + al * bh) + al * bl};
}
constexpr TwoDoubles add2(TwoDoubles a, TwoDoubles b) {
  const TwoDoubles s = two_sum(a.hi, b.hi);
  return two_sum(s.hi, s.lo + a.lo + b.lo);
}
constexpr TwoDoubles mul2(TwoDoubles a, TwoDoubles b) {
  const TwoDoubles p = two_prod(a.hi, b.hi);
  return two_sum(p.hi, p.lo + a.hi * b.lo + a.lo * b.hi);
}
constexpr TwoDoubles div2(TwoDoubles a, double d) {
  const double q = a.hi / d;
  const TwoDoubles p = two_prod(q, d);
  return two_sum(q, ((a.hi - p.hi) - p.lo + a.lo) / d);
}
// cos x (first = 0) or sin x (first = 1): x^m / m!, m = first, first + 2, ..
constexpr double taylor(TwoDoubles x, int first) {
  TwoDoubles term = first ? x : TwoDoubles{1, 0}, sum = term;
  const TwoDoubles x2 = mul2(x, x);
  for (int m = first + 2; m < 30; m += 2) {
    term = div2(mul2(term, x2), -(double)(m * (m - 1)));
    sum = add2(sum, term);
  }
  return sum.hi;
}
// cos(2 pi t / n) (which = 0) or sin(2 pi t / n) (which = 1)
constexpr double cexpr_trig(long long t, long long n, int which) {
  long long M = 8 * n;
  long long v = 8 * (((t % n) + n) % n);  // angle 2 pi v / M, v in [0, M)
  double sgn_s = 1, sgn_c = 1;
  if (2 * v > M) {  // theta > pi: sin(-), cos(+) with theta -> 2 pi - theta
    v = M - v;
    sgn_s = -1;
  }
  if (4 * v > M) {  // theta > pi/2: theta -> pi - theta, cos(-)
    v = M / 2 - v;
    sgn_c = -sgn_c;
  }
  bool swap = false;
  if (8 * v > M) {  // theta > pi/4: use pi/2 - theta
    v = M / 4 - v;
    swap = true;
  }
  const TwoDoubles pi = {3.141592653589793116, 1.2246467991473531772e-16};
  const TwoDoubles x = div2(mul2(pi, {(double)(2 * v), 0}), (double)M);
  const double s = taylor(x, swap ? 0 : 1), c = taylor(x, swap ? 1 : 0);
  return which ? sgn_s * s : sgn_c * c;
}
template <int N> struct RootsOfUnity {
  double cos[N] = {}, sin[N] = {};
  constexpr RootsOfUnity() {
    for (int t = 0; t < N; t++) {
      cos[t] = cexpr_trig(t, N, 0);
      sin[t] = cexpr_trig(t, N, 1);
    }
  }
};
template <int N> constexpr RootsOfUnity<N> kRoots{};
static_assert(kRoots<3>.cos[1] == -0.5 && kRoots<12>.sin[1] == 0.5 && kRoots<3>.sin[1] == 0.86602540378443864676 &&
                  kRoots<8>.cos[1] == 0.70710678118654752440 && kRoots<7>.cos[1] == 0.62348980185873353053 &&
                  kRoots<9>.sin[2] == 0.98480775301220805937 && kRoots<16>.cos[3] == 0.38268343236508977173 &&
                  kRoots<27>.sin[13] == 0.11609291412523022967 && kRoots<25>.cos[12] == -0.99211470131447783105,
              "roots of unity to the last place");

// ------------------------------------------------------------------------------------
// In-register DFT of length R (forward exp(-2 pi i jk/R) unless INV).
// Composite lengths R = P * Q by one Cooley-Tukey split with constant twiddles:
// X[k1 + P k2] = sum_q W_Q^{q k2} W_R^{q k1} sum_p a[q + Q p] W_P^{p k1}.
// ------------------------------------------------------------------------------------
template <int R> struct SmallFactor {
  static constexpr int value = (R % 4 == 0 && R > 4)   ? 4
                               : (R % 2 == 0 && R > 2) ? 2
                               : (R % 3 == 0 && R > 3) ? 3
                               : (R % 5 == 0 && R > 5) ? 5
                                                       : R;
};

template <int R, bool INV, typename C> struct RDft;

// a * W_R^k (W_R = exp(-2 pi i / R), conjugated when INV). k and R are
// constants once the calling loops are unrolled, so the branches fold away and
// multiples of a quarter turn become swaps and sign changes.
template <int R, bool INV, typename C>
__device__ __forceinline__ C cmul_w(C a, int k) {
  typedef decltype(C().x) F;
  k = k % R;
  if (k == 0) return a;
  if (2 * k == R) return cmake<C>(-a.x, -a.y);
  if (4 * k == R) return INV ? cmul_pi(a) : cmul_mi(a);
  if (4 * k == 3 * R) return INV ? cmul_mi(a) : cmul_pi(a);
  const F c = (F)kRoots<R>.cos[k];
  const F s = (F)kRoots<R>.sin[k];
  return cmul(a, cmake<C>(c, INV ? s : -s));
}

template <bool INV, typename C> struct RDft<1, INV, C> {
  static __device__ inline void run(C*) {}
};
template <bool INV, typename C> struct RDft<2, INV, C> {
  static __device__ inline void run(C* a) {
    const C t = a[0];
    a[0] = cadd(t, a[1]);
    a[1] = csub(t, a[1]);
  }
};
template <bool INV, typename C> struct RDft<4, INV, C> {
  static __device__ inline void run(C* a) {
    const C t0 = cadd(a[0], a[2]), t1 = csub(a[0], a[2]);
    const C t2 = cadd(a[1], a[3]), d = csub(a[1], a[3]);
    const C t3 = INV ? cmul_pi(d) : cmul_mi(d);
    a[0] = cadd(t0, t2);
    a[2] = csub(t0, t2);
    a[1] = cadd(t1, t3);
    a[3] = csub(t1, t3);
  }
};

// Odd primes by symmetric pairs.
template <int R, bool INV, typename C> struct RDftOdd {
  static __device__ inline void run(C* a) {
    typedef decltype(C().x) F;
    constexpr int H = (R - 1) / 2;
    C s[H + 1], d[H + 1];
#pragma unroll
    for (int m = 1; m <= H; m++) {
      s[m] = cadd(a[m], a[R - m]);
      d[m] = csub(a[m], a[R - m]);
    }
    C x0 = a[0];
#pragma unroll
    for (int m = 1; m <= H; m++) x0 = cadd(x0, s[m]);
#pragma unroll
    for (int k = 1; k <= H; k++) {
      C cs = a[0];
      C sn = czero<C>();
#pragma unroll
      for (int m = 1; m <= H; m++) {
        const F cv = (F)kRoots<R>.cos[m * k % R];
        const F sv = (F)kRoots<R>.sin[m * k % R];
        cs.x += cv * s[m].x;
        cs.y += cv * s[m].y;
        sn.x += sv * d[m].x;
        sn.y += sv * d[m].y;
      }
      const C isn = cmul_pi(sn);
      if (INV) {
        a[k] = cadd(cs, isn);
        a[R - k] = csub(cs, isn);
      } else {
        a[k] = csub(cs, isn);
        a[R - k] = cadd(cs, isn);
      }
    }
    a[0] = x0;
  }
};
template <bool INV, typename C> struct RDft<3, INV, C> : RDftOdd<3, INV, C> {};
template <bool INV, typename C> struct RDft<5, INV, C> : RDftOdd<5, INV, C> {};
template <bool INV, typename C> struct RDft<7, INV, C> : RDftOdd<7, INV, C> {};

template <int R, bool INV, typename C> struct RDft {
  static_assert(SmallFactor<R>::value < R, "unsupported in-register DFT length");
  static __device__ inline void run(C* a) {
    constexpr int P = SmallFactor<R>::value;
    constexpr int Q = R / P;
    C b[R];
#pragma unroll
    for (int q = 0; q < Q; q++) {
      C t[P];
#pragma unroll
      for (int p = 0; p < P; p++) t[p] = a[q + Q * p];
      RDft<P, INV, C>::run(t);
#pragma unroll
      for (int k1 = 0; k1 < P; k1++) b[q + Q * k1] = cmul_w<R, INV>(t[k1], q * k1);
    }
#pragma unroll
    for (int k1 = 0; k1 < P; k1++) {
      C t[Q];
#pragma unroll
      for (int q = 0; q < Q; q++) t[q] = b[q + Q * k1];
      RDft<Q, INV, C>::run(t);
#pragma unroll
      for (int k2 = 0; k2 < Q; k2++) a[k1 + P * k2] = t[k2];
    }
  }
};

// DFT of length R (even) whose inputs a[R/2 .. R-1] are zero; those slots are
// not read. X[2j] = DFT_{R/2}(a)[j], X[2j+1] = DFT_{R/2}(a[m] W_R^m)[j].
template <int R, bool INV, typename C> struct RDftHalfIn {
  static_assert(R % 2 == 0, "half-input DFT needs an even length");
  static __device__ inline void run(C* a) {
    constexpr int H = R / 2;
    C e[H], o[H];
#pragma unroll
    for (int m = 0; m < H; m++) {
      e[m] = a[m];
      o[m] = cmul_w<R, INV>(a[m], m);
    }
    RDft<H, INV, C>::run(e);
    RDft<H, INV, C>::run(o);
#pragma unroll
    for (int j = 0; j < H; j++) {
      a[2 * j] = e[j];
      a[2 * j + 1] = o[j];
    }
  }
};

// How a stage gets its butterfly's twiddles W^m, m = 1 .. R - 1 (W^m = tw[m s],
// tw the table of N roots of unity, each correct to half a unit in the last place):
//   TW_CHAIN  one load, then repeated multiplication: W^m carries m times its
//             rounding. The plans with radices up to 16 of the powers of two, the
//             long lengths: where every load shows.
//   TW_SPLIT  powers 1, 2, 3 and the multiples of 4 loaded, the others one product
//             of two of those
//   TW_HELD   powers formed once by the caller for all its transforms
// General plans take TW_SPLIT: their radices go up to 28, whose chained powers
// made the FP64 product at 80^3 2.1e-16 and the FP32 one at 96 x 70 x 120 9.9e-8
// from the exact one, against 1.6e-16 and 8.1e-8 with run-time planned radices up
// to 8; with TW_SPLIT it is 1.5e-16 and 6.5e-8, over 150 grids of all general
// lengths 0.93 (FP64) and 0.82 (FP32) of the run-time planned kernels' error.
// Loading every power (FP64) gave no smaller error and took 22% longer at
// 180 x 144 x 120. TW_SPLIT in the plans of the powers of two halves the FP32
// error at 512^3 but makes their products 2 to 9% slower.
enum TwiddleMode { TW_CHAIN = 0, TW_SPLIT = 1, TW_HELD = 2 };

template <int R, typename C> struct TwiddleRow {
  C lo[4], hi[(R + 3) / 4];
  __device__ __forceinline__ TwiddleRow(const C* __restrict__ tw, int s) {
#pragma unroll
    for (int m = 1; m < 4 && m < R; m++) lo[m] = tw[m * s];
#pragma unroll
    for (int m = 4; m < R; m += 4) hi[m / 4] = tw[m * s];
  }
  // W^m, r = m mod 4
  __device__ __forceinline__ C power(int r, int m) const {
    if (m < 4) return lo[m];
    return r ? cmul(hi[m / 4], lo[r]) : hi[m / 4];
  }
};

// ------------------------------------------------------------------------------------
// Plans
// ------------------------------------------------------------------------------------
template <int... Rs> struct RadixList {};

// StaticPlan<N, WIDE>: PPT, TPC, the radix order (Fwd) and that of the single inverse
// transforms (Bwd). WIDE plans (used
// for complex float) hold 16 points per thread and need one LDS exchange fewer;
// narrow plans (complex double) hold 8 to keep three components in registers.
template <int N, bool WIDE> struct StaticPlan { static constexpr bool exists = false; };
#define DDA_PLAN(N, W, P, ...)                            \
  template <> struct StaticPlan<N, W> {                   \
    static constexpr bool exists = true, general = false; \
    static constexpr int PPT = P;                         \
    static constexpr int TPC = N / P;                     \
    typedef RadixList<__VA_ARGS__> Fwd;                   \
    typedef Fwd Bwd;                                      \
    template <typename R> static constexpr int twiddles = TW_CHAIN; \
  };
DDA_PLAN(32, false, 8, 8, 4)
DDA_PLAN(32, true, 16, 16, 2)
DDA_PLAN(48, false, 12, 12, 4)
DDA_PLAN(48, true, 12, 12, 4)
DDA_PLAN(64, false, 8, 8, 8)
DDA_PLAN(64, true, 8, 8, 8)
DDA_PLAN(96, false, 12, 6, 4, 4)
DDA_PLAN(96, true, 12, 6, 4, 4)
DDA_PLAN(128, false, 8, 8, 4, 4)
DDA_PLAN(128, true, 16, 16, 8)
DDA_PLAN(192, false, 12, 12, 4, 4)
DDA_PLAN(192, true, 12, 12, 4, 4)
DDA_PLAN(256, false, 8, 8, 8, 4)
DDA_PLAN(256, true, 16, 16, 16)
DDA_PLAN(512, false, 8, 8, 8, 8)
DDA_PLAN(512, true, 16, 16, 16, 2)
DDA_PLAN(1024, false, 8, 8, 8, 4, 4)
DDA_PLAN(1024, true, 16, 16, 16, 4)
#undef DDA_PLAN

// A plan given by its points per thread and radix order directly (the Z
// pass's long-column variants: 1024 = 32 x 32 holds 32 points per thread and
// needs a single LDS exchange per transform).
template <int N, int P, typename L, int TW = TW_CHAIN> struct PlanOf {
  static constexpr bool exists = true, general = false;
  static constexpr int PPT = P;
  static constexpr int TPC = N / P;
  typedef L Fwd;
  typedef L Bwd;
  template <typename R> static constexpr int twiddles = TW;
};

template <typename L> struct Reverse;
template <> struct Reverse<RadixList<>> { typedef RadixList<> type; };
template <int R, int... Rs> struct Reverse<RadixList<R, Rs...>> {
  template <typename A, int X> struct Append;
  template <int... As, int X> struct Append<RadixList<As...>, X> { typedef RadixList<As..., X> type; };
  typedef typename Append<typename Reverse<RadixList<Rs...>>::type, R>::type type;
};

// Butterflies of radix R that a thread of a column with TPC threads owns:
// j_i = t + i * TPC, i < per; the last may lie beyond the stage's N / R.
template <int N, int TPC, int R> struct Butterflies {
  static constexpr int count = N / R;
  static constexpr int per = (count + TPC - 1) / TPC;
  static constexpr bool exact = per * TPC == count;
};

// A plan of radices R0, Rs... (R0 even) whose threads hold one butterfly of each
// stage where they have one: TPC = N / (smallest radix) threads per column, so
// that lengths such as 80 = 10 * 8 or 294 = 6 * 7 * 7 run as two or three stages
// of nearly equal radices; in a stage of radix R, threads t >= N / R idle.
template <int N, int R0, int... Rs> struct GenPlan {
  static constexpr int cmin(int a) { return a; }
  template <typename... A> static constexpr int cmin(int a, int b, A... r) { return cmin(a < b ? a : b, r...); }
  static constexpr int cmax(int a) { return a; }
  template <typename... A> static constexpr int cmax(int a, int b, A... r) { return cmax(a > b ? a : b, r...); }
  static constexpr int cprod(int a) { return a; }
  template <typename... A> static constexpr int cprod(int a, int b, A... r) { return cprod(a * b, r...); }
  static constexpr bool exists = true, general = true;
  static constexpr int PPT = cmax(R0, Rs...);
  static constexpr int TPC = N / cmin(R0, Rs...);
  typedef RadixList<R0, Rs...> Fwd;
  typedef typename Reverse<Fwd>::type Bwd;  // ends on R0: the cropped half is never formed
  template <typename R> static constexpr int twiddles = TW_SPLIT;
  static_assert(R0 % 2 == 0 && cprod(R0, Rs...) == N, "radices");
};

// Stage helpers. v[i * R + m] is input m of butterfly j_i = t + i * TPC, its
// twiddle W_{NS R}^{k m} (TwiddleRow). HALF (first stage only): inputs m >= R/2 are zero
// and not read.
// TW_HELD: tw holds the R - 1 twiddle powers of the thread's one butterfly of
// the twiddled stage. Idle butterflies are computed on whatever v holds and
// never stored.
template <int N, int TPC, int R, int NS, bool INV, bool HALF, typename C, int TW>
__device__ inline void stage_compute(C* v, int t, const C* __restrict__ tw) {
#pragma unroll
  for (int i = 0; i < Butterflies<N, TPC, R>::per; i++) {
    C* a = v + i * R;
    const int j = t + i * TPC;
    const int k = j % NS;  // NS is a compile-time constant
    constexpr int step = N / (NS * R);
    if constexpr (NS > 1 && TW == TW_HELD) {
#pragma unroll
      for (int m = 1; m < R; m++) a[m] = INV ? cmulc(a[m], tw[m - 1]) : cmul(a[m], tw[m - 1]);
    } else if constexpr (NS > 1 && TW == TW_SPLIT) {
      TwiddleRow<R, C> w(tw, k * step);
#pragma unroll
      for (int r = 0; r < 4 && r < R; r++)
#pragma unroll
        for (int m = r ? r : 4; m < R; m += 4) {
          const C wm = w.power(r, m);
          a[m] = INV ? cmulc(a[m], wm) : cmul(a[m], wm);
        }
    } else if constexpr (NS > 1) {
      const C w1 = tw[k * step];
      C w = w1;
#pragma unroll
      for (int m = 1; m < R; m++) {
        a[m] = INV ? cmulc(a[m], w) : cmul(a[m], w);
        if (m + 1 < R) w = cmul(w, w1);
      }
    }
    if constexpr (HALF && NS == 1)
      RDftHalfIn<R, INV, C>::run(a);
    else
      RDft<R, INV, C>::run(a);
  }
}

// Forms v[0 .. K) here: the compiler does not defer it to a later use.
template <int K, typename C> __device__ __forceinline__ void keep_here(C* v) {
#pragma unroll
  for (int m = 0; m < K; m++) asm volatile("" : "+v"(v[m].x), "+v"(v[m].y));
}

// Writes the stage outputs to the tile at their Stockham positions.
template <int N, int TPC, int R, int NS, typename C>
__device__ inline void stage_store(C* v, int t, C* tile, int lp, int l) {
  typedef Butterflies<N, TPC, R> B;
#pragma unroll
  for (int i = 0; i < B::per; i++) {
    const int j = t + i * TPC;
    if constexpr (!B::exact) {
      // (formed before the branch: the compiler would move into it all that
      // leads to them)
      keep_here<R>(v + i * R);
      if (j >= B::count) continue;
    }
    const int q = j / NS, k = j % NS;
    const int base = q * NS * R + k;
#pragma unroll
    for (int m = 0; m < R; m++) tile[(base + m * NS) * lp + l] = v[i * R + m];
  }
}

// Reads the inputs of a stage of radix R from the tile (an idle butterfly reads
// butterfly 0's: no branch, which would keep v out of registers).
template <int N, int TPC, int R, typename C>
__device__ inline void stage_load(C* v, int t, const C* tile, int lp, int l) {
  typedef Butterflies<N, TPC, R> B;
#pragma unroll
  for (int i = 0; i < B::per; i++) {
    int j = t + i * TPC;
    if (!B::exact) j = j < B::count ? j : 0;
#pragma unroll
    for (int m = 0; m < R; m++) v[i * R + m] = tile[(j + m * (N / R)) * lp + l];
  }
}

// Runs all stages of RadixList from registers to registers with LDS exchanges
// in between. On entry v holds the first stage's inputs, on exit the last
// stage's outputs (both in the layout described above). Ends with a barrier if
// any exchange happened, so the caller may reuse the tile. HALF: the upper half
// of every first-stage butterfly's inputs is zero (a zero-padded transform of
// at most N/2 points) and is neither read nor computed with.
// TW: the twiddles' TwiddleMode; TW_HELD for two-stage plans with one butterfly
// per thread per stage (TwoStage), tw the thread's second-stage powers.
template <int N, int TPC, bool INV, int NS, typename C, typename L, bool HALF = false, int TW = TW_CHAIN>
struct RunStages;

template <int N, int TPC, bool INV, int NS, typename C, int R, bool HALF, int TW>
struct RunStages<N, TPC, INV, NS, C, RadixList<R>, HALF, TW> {
  static __device__ inline void run(C* v, int t, C* tile, int lp, int l, const C* tw) {
    stage_compute<N, TPC, R, NS, INV, HALF, C, TW>(v, t, tw);
  }
};

template <int N, int TPC, bool INV, int NS, typename C, int R, int R2, int... Rs, bool HALF, int TW>
struct RunStages<N, TPC, INV, NS, C, RadixList<R, R2, Rs...>, HALF, TW> {
  static __device__ inline void run(C* v, int t, C* tile, int lp, int l, const C* tw) {
    stage_compute<N, TPC, R, NS, INV, HALF, C, TW>(v, t, tw);
    stage_store<N, TPC, R, NS>(v, t, tile, lp, l);
    __syncthreads();
    stage_load<N, TPC, R2>(v, t, tile, lp, l);
    __syncthreads();
    RunStages<N, TPC, INV, NS * R, C, RadixList<R2, Rs...>, false, TW>::run(v, t, tile, lp, l, tw);
  }
};

// Plans of two stages with one butterfly of each per thread: the thread's
// second-stage twiddles are W_N^(t m), m = 1 .. R1 - 1, in the forward transform
// and, conjugated, W_N^(t m), m = 1 .. R0 - 1, in the inverse, whose radices run
// the other way round.
template <int N, int TPC, typename L> struct TwoStage { static constexpr bool value = false; };
template <int N, int TPC, int R0, int R1> struct TwoStage<N, TPC, RadixList<R0, R1>> {
  static constexpr bool value = R0 * R1 == N && TPC == (R0 > R1 ? R0 : R1);
};
// W_N^(t m), m = 1 .. K (t < N), formed as MODE says
template <int K, int MODE, typename C>
__device__ inline void twiddle_powers(C* wp, int t, const C* __restrict__ tw) {
  if constexpr (MODE == TW_CHAIN) {
    const C w1 = tw[t];
    C w = w1;
#pragma unroll
    for (int m = 0; m < K; m++) {
      wp[m] = w;
      if (m + 1 < K) w = cmul(w, w1);
    }
  } else {
    TwiddleRow<K + 1, C> w(tw, t);
#pragma unroll
    for (int m = 1; m <= K; m++) wp[m - 1] = w.power(m % 4, m);
  }
}

template <typename L> struct FirstRadix;
template <int R, int... Rs> struct FirstRadix<RadixList<R, Rs...>> { static constexpr int value = R; };

// Registers v[0 .. first_count) that the first stage of plan L uses, and the
// point index held in v[e] (e = i * R0 + m). With idle butterflies a thread's
// point may not be its own: first_ok says whether it is.
template <int N, int TPC, typename L>
__device__ __forceinline__ constexpr int first_count() {
  return Butterflies<N, TPC, FirstRadix<L>::value>::per * FirstRadix<L>::value;
}
template <int N, int TPC, typename L>
__device__ inline int first_point(int t, int e) {
  constexpr int R0 = FirstRadix<L>::value;
  return t + (e / R0) * TPC + (e % R0) * (N / R0);
}
template <int N, int TPC, typename L>
__device__ __forceinline__ bool first_ok(int t, int e) {
  typedef Butterflies<N, TPC, FirstRadix<L>::value> B;
  return B::exact || t + (e / FirstRadix<L>::value) * TPC < B::count;
}

// Whether v[e] of that layout lies in the upper half of the transform (point
// >= N/2) for every thread: m = e mod R0 >= R0 / 2 with R0 even. A transform of
// at most N/2 points neither reads (first stage) nor writes (last stage) them.
template <typename L>
__device__ __forceinline__ constexpr bool upper_half(int e) {
  return FirstRadix<L>::value % 2 == 0 && (e % FirstRadix<L>::value) >= FirstRadix<L>::value / 2;
}

}  // namespace dda
