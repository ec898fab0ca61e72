// The FFT'd interaction tensor, octant by octant: each component of the Green's
// function is even or odd in each axis (DDA/DMatrixCpu.cpp:49-63), and so is its
// transform, so every pass reads the non-negative offsets alone, reflects them
// as it loads its lines, and stores the non-negative frequencies alone.
//
//   X  the function at the offsets |i| < cx of the lines j < cy, k < cz (one
//      sincos for the six components), reflected and transformed
//   Y  in place; Z from the k < cz planes to the octant, times -1/N
//      (DDA/DMatrixCpu.cpp:200), in the operator's precision
//
// All in double precision and for the six components at once. Compiled in four
// parts (DDA_PLAN_PART), each with the lengths of one part of plan_list.hpp, the
// first also with those that have tuned matvec variants.
//
// The transforms of one component on the whole grid, which this replaces, moved
// eight times the points in five launches each: at 192 x 144 x 120 (FP64) the
// thirty launches took 900 us, these three 82 (25, 30 and 27).
#include "passes.hpp"
#include "plan_list.hpp"

#ifndef DDA_PLAN_PART
#define DDA_PLAN_PART 0
#endif

namespace dda {

namespace {

// The Green's function at offset (i, j, k) >= 0, not all zero, in units of the
// grid spacing (DDA/DMatrixCpu.cpp:124-131,169-193):
// exp(i kr) / r^3 * [(3 - kr^2 - 3 i kr) q_mu q_nu + delta (kr^2 - 1 + i kr)]
// for (mu, nu) = xx, xy, xz, yy, yz, zz.
__device__ inline void green_at(int i, int j, int k, double kd, double2 g[6]) {
  const double r[3] = {(double)i, (double)j, (double)k};
  const double rr = sqrt(r[0] * r[0] + r[1] * r[1] + r[2] * r[2]);
  const double kr = kd * rr;
  const double kr2 = kr * kr;
  double sn, cs;
  sincos(kr, &sn, &cs);
  const double inv3 = 1.0 / (rr * rr * rr);
  const double q[3] = {r[0] / rr, r[1] / rr, r[2] / rr};
  int c = 0;
#pragma unroll
  for (int mu = 0; mu < 3; mu++)
#pragma unroll
    for (int nu = mu; nu < 3; nu++, c++) {
      const double qmn = q[mu] * q[nu];
      double br = (3.0 - kr2) * qmn, bi = -3.0 * kr * qmn;
      if (mu == nu) {
        br += kr2 - 1.0;
        bi += kr;
      }
      g[c].x = (cs * br - sn * bi) * inv3;
      g[c].y = (cs * bi + sn * br) * inv3;
    }
}

// Input p of a line of length N that holds the offsets q < clip (clip <= N / 2)
// and is even or odd about 0: element at(q), its sign changed, or zero.
template <int N, typename F>
__device__ __forceinline__ double2 reflected(int p, int clip, bool odd, F&& at) {
  const int q = p <= N / 2 ? p : N - p;
  if (q >= clip) return czero<double2>();
  double2 v = at(q);
  if (odd && p > N / 2) v = make_double2(-v.x, -v.y);
  return v;
}

// Rows (of six components each) per work-group of the X pass: about 256 threads.
template <typename PL> constexpr int green_rows() {
  return 256 / (6 * PL::TPC) > 0 ? 256 / (6 * PL::TPC) : 1;
}

// X pass: rows r0 .. r0 + RN - 1 of the cy * cz ones; thread (l, t) runs line
// l = 6 * (row in the group) + component. w: [6][cstride], row (j, k) at
// k * zstride + j * (N / 2 + 1). Bound by its butterflies and LDS trips; the
// function's values take a tenth of it.
template <int N, typename PL>
__global__ __launch_bounds__(6 * green_rows<PL>() * PL::TPC) void k_green_rows(double2* __restrict__ w, int cx, int cy,
                                                                              int nrows, double kd, long long cstride,
                                                                              long long zstride,
                                                                              const double2* __restrict__ tw) {
  constexpr int TPC = PL::TPC, RN = green_rows<PL>(), L = 6 * RN, lp = L + 1;
  typedef typename PL::Fwd F;
  typedef typename Reverse<F>::type Out;
  constexpr int NF = first_count<N, TPC, F>(), NO = first_count<N, TPC, Out>();
  extern __shared__ char smem[];
  double2* tile = reinterpret_cast<double2*>(smem);
  const int r0 = blockIdx.x * RN;
  for (int q = threadIdx.x; q < RN * cx; q += L * TPC) {
    const int rr = q / cx, i = q - rr * cx, row = r0 + rr;
    const int k = row / cy, j = row - k * cy;
    double2 g[6];
    if (row < nrows && (i | j | k) != 0) {
      green_at(i, j, k, kd, g);
    } else {
#pragma unroll
      for (int c = 0; c < 6; c++) g[c] = czero<double2>();
    }
#pragma unroll
    for (int c = 0; c < 6; c++) tile[i * lp + rr * 6 + c] = g[c];
  }
  __syncthreads();
  const int t = threadIdx.x % TPC, l = threadIdx.x / TPC;
  const int rr = l / 6, c = l - rr * 6, row = r0 + rr;
  const bool odd = c == 1 || c == 2;
  double2 v[PL::PPT];
#pragma unroll
  for (int e = 0; e < NF; e++)
    v[e] = first_ok<N, TPC, F>(t, e)
               ? reflected<N>(first_point<N, TPC, F>(t, e), cx, odd, [&](int q) { return tile[q * lp + l]; })
               : czero<double2>();
  __syncthreads();
  RunStages<N, TPC, false, 1, double2, F, false, PL::template twiddles<double>>::run(v, t, tile, lp, l, tw);
  if (row >= nrows) return;
  const int k = row / cy, j = row - k * cy;
  double2* dst = w + c * cstride + k * zstride + (long long)j * (N / 2 + 1);
#pragma unroll
  for (int e = 0; e < NO; e++) {
    const int p = first_point<N, TPC, Out>(t, e);
    if (first_ok<N, TPC, Out>(t, e) && p <= N / 2) dst[p] = v[e];
  }
}

// Y and Z passes: T adjacent columns of batch b of component c (blockIdx.y =
// c * nb + b), in place or not (a work-group stores after it has read all that
// it reads: every plan has an LDS exchange in between). RO: the output's type.
template <int N, int T, typename PL, typename RO>
__global__ __launch_bounds__(T * PL::TPC) void k_tensor_cols(const double2* in, typename CxT<RO>::T* out,
                                                             TensorCols tc, const double2* __restrict__ tw) {
  constexpr int TPC = PL::TPC, lp = (T & 1) ? T : T + 1;
  typedef typename PL::Fwd F;
  typedef typename Reverse<F>::type Out;
  constexpr int NF = first_count<N, TPC, F>(), NO = first_count<N, TPC, Out>();
  extern __shared__ char smem[];
  double2* tile = reinterpret_cast<double2*>(smem);
  const int l = threadIdx.x % T, t = threadIdx.x / T;
  const int col = blockIdx.x * T + l;
  const int c = blockIdx.y / tc.nb, b = blockIdx.y - c * tc.nb;
  const bool colok = col < tc.ncols;
  const bool odd = (tc.odd >> c) & 1;
  const double2* src = in + c * tc.cstride_in + b * tc.bstride + col;
  typename CxT<RO>::T* dst = out + c * tc.cstride_out + b * tc.bstride + col;
  double2 v[PL::PPT];
#pragma unroll
  for (int e = 0; e < NF; e++)
    v[e] = colok && first_ok<N, TPC, F>(t, e)
               ? reflected<N>(first_point<N, TPC, F>(t, e), tc.clip, odd, [&](int q) { return src[q * tc.pstride]; })
               : czero<double2>();
  RunStages<N, TPC, false, 1, double2, F, false, PL::template twiddles<double>>::run(v, t, tile, lp, l, tw);
#pragma unroll
  for (int e = 0; e < NO; e++) {
    const int p = first_point<N, TPC, Out>(t, e);
    if (colok && first_ok<N, TPC, Out>(t, e) && p <= N / 2)
      dst[p * tc.pstride] = cmake<typename CxT<RO>::T>(v[e].x * tc.scale, v[e].y * tc.scale);
  }
}

template <int N, typename PL>
dda_status launch_green_rows(void* w, int cx, int cy, int cz, double kd, long long cstride, long long zstride,
                             const void* tw, hipStream_t st) {
  constexpr int RN = green_rows<PL>();
  const size_t lds = (size_t)N * (6 * RN + 1) * sizeof(double2);
  auto k = k_green_rows<N, PL>;
  DDA_TRY(set_lds(k, lds));
  hipLaunchKernelGGL(k, dim3((cy * cz + RN - 1) / RN), dim3(6 * RN * PL::TPC), lds, st, (double2*)w, cx, cy, cy * cz, kd,
                     cstride, zstride, (const double2*)tw);
  DDA_TRY_HIP(hipGetLastError());
  return DDA_OK;
}

template <int N, typename PL>
dda_status launch_tensor_cols(const void* in, void* out, int out_prec, const TensorCols& tc, const void* tw,
                              hipStream_t st) {
  constexpr int T = gen_cols<double, N, PL::TPC>(16);
  constexpr int lp = (T & 1) ? T : T + 1;
  const size_t lds = (size_t)N * lp * sizeof(double2);
  const dim3 grid((tc.ncols + T - 1) / T, 6 * tc.nb), block(T * PL::TPC);
  if (out_prec == 64) {
    auto k = k_tensor_cols<N, T, PL, double>;
    DDA_TRY(set_lds(k, lds));
    hipLaunchKernelGGL(k, grid, block, lds, st, (const double2*)in, (double2*)out, tc, (const double2*)tw);
  } else {
    auto k = k_tensor_cols<N, T, PL, float>;
    DDA_TRY(set_lds(k, lds));
    hipLaunchKernelGGL(k, grid, block, lds, st, (const double2*)in, (float2*)out, tc, (const double2*)tw);
  }
  DDA_TRY_HIP(hipGetLastError());
  return DDA_OK;
}

template <int N, typename PL>
const TensorOps* tensor_ops_of() {
  static const TensorOps ops = {launch_green_rows<N, PL>, launch_tensor_cols<N, PL>};
  return &ops;
}

}  // namespace

const TensorOps* DDA_CAT(tensor_ops_part, DDA_PLAN_PART)(int n) {
  switch (n) {
#define X(N, L, Z) \
  case N:          \
    return tensor_ops_of<N, GenPlan<N, DDA_ARGS L>>();
    DDA_CAT(DDA_GEN_SIZES_, DDA_PLAN_PART)(X)
#undef X
#if DDA_PLAN_PART == 0
#define X(N) \
  case N:    \
    return tensor_ops_of<N, StaticPlan<N, false>>();
    DDA_STATIC_SIZES(X)
#undef X
#endif
    default:
      return nullptr;
  }
}

}  // namespace dda
