// The compile-time planned passes of the matvec: kernels and their launchers.
// matvec.hip instantiates them for the lengths with tuned variants, plans.hip
// for the other lengths.
#pragma once

#include <type_traits>

#include "fft_static.hpp"
#include "internal.hpp"

namespace dda {

__device__ inline bool stopped(const RhsFlags& f, int rhs) { return f.done != nullptr && f.done[rhs * f.stride] != 0; }

// A cell without a dipole in the cell map.
constexpr uint32_t kNoDipole = 0xffffffffu;

// The buffers of right-hand sides r0 .. r0 + nrhs - 1 of an operator: what one
// sequence of the five passes works on (the whole block, or one half of it
// when the halves run on two streams).
struct MvView {
  void* a1;
  void* a2;
  const void* ccs;
  MvDims d;  // member table shifted to r0
};

// Strided column FFT over T adjacent columns. Column `col` of batch b, point p
// lives at base[b * bstride + p * pstride + col]; inputs beyond in_len are zero,
// only the first out_len points are stored. With yr (the matvec's Y passes, batch
// b of plane b mod nz), a forward transform reads and an inverse one stores the
// plane's occupied range [yr.x, yr.y) alone: the rows outside it are zero before
// and no dipole's after. A particle that fills 79% of its rows (any ellipsoid)
// saves a fifth of A1's traffic: two FP32 right-hand sides at 256^3 606 -> 579
// us, 128 at 128 x 96 x 64 1,657 -> 1,580.
struct ColParams {
  int ncols;
  int in_len, out_len;
  long long pstride_in, pstride_out;
  long long bstride_in, bstride_out;
  const int2* yr = nullptr;
  FastDiv nz = {1, 0, 0};
};

// ------------------------------------------------------------------------------------
// Compile-time planned variants of the column passes (fft_static.hpp). Thread
// (l, t) = (tid mod T, tid / T) owns column c0 + l and the plan's points t + ...
// ------------------------------------------------------------------------------------

// Buffer resources (V#) for the Z pass: raw (stride 0) buffers whose range
// check turns loads beyond `bytes` into zeros and drops such stores, so that
// the zero padding and the cropping need neither branches nor 64-bit address
// arithmetic per access (the offset is a 32-bit byte offset from a uniform
// base). Word 3 selects 32-bit data format, as gfx9-family buffers require.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t zrsrc(const void* p, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), (short)0, (int)bytes, 0x00020000);
}
__device__ __forceinline__ float2 zload(__amdgpu_buffer_rsrc_t r, uint32_t off, float2*) {
  return __builtin_bit_cast(float2, __builtin_amdgcn_raw_buffer_load_b64(r, off, 0, 0));
}
__device__ __forceinline__ double2 zload(__amdgpu_buffer_rsrc_t r, uint32_t off, double2*) {
  return __builtin_bit_cast(double2, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0));
}
typedef int zi2 __attribute__((ext_vector_type(2)));
typedef int zi4 __attribute__((ext_vector_type(4)));
constexpr int kStoreNT = 2;  // buffer cache policy: nt
// The Z pass's stores and those of the X-forward and Y-inverse passes are
// non-temporal (nt): their outputs are read by the next pass only after this
// kernel's end, and streaming them leaves little dirty data in the L2s to be
// written back when the kernel ends (the gap before the next kernel).
// Measured in a solve at 256^3: 591 -> 560 us per 2-RHS matvec; the Y-forward
// pass keeps ordinary stores (non-temporal ones made it 5% slower).
__device__ __forceinline__ void zstore(__amdgpu_buffer_rsrc_t r, uint32_t off, float2 v) {
  __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(zi2, v), r, off, 0, kStoreNT);
}
__device__ __forceinline__ void zstore(__amdgpu_buffer_rsrc_t r, uint32_t off, double2 v) {
  __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(zi4, v), r, off, 0, kStoreNT);
}
template <bool NT> __device__ __forceinline__ void cstore(float2* p, float2 v) {
  if constexpr (NT) {
    typedef float f2 __attribute__((ext_vector_type(2)));
    __builtin_nontemporal_store(__builtin_bit_cast(f2, v), reinterpret_cast<f2*>(p));
  } else {
    *p = v;
  }
}
template <bool NT> __device__ __forceinline__ void cstore(double2* p, double2 v) {
  if constexpr (NT) {
    typedef double d2 __attribute__((ext_vector_type(2)));
    __builtin_nontemporal_store(__builtin_bit_cast(d2, v), reinterpret_cast<d2*>(p));
  } else {
    *p = v;
  }
}

// Waves per SIMD the Z pass is compiled for, a register budget: FP32
// 16-point plans at 3 (168 VGPRs: the tensor loads of several points stay in
// flight), other FP32 plans at 4, FP64 left to the compiler. At 1024 points
// the 16-point plan runs 1024-thread work-groups, which fit a CU only at 4
// waves per SIMD (128 VGPRs, a few spilled).
// 32-point plans (FP32) hold 192 VGPRs of data: 2 waves per SIMD (256), as
// general plans above 20 points are.
// 64 columns of 8-point threads are 512-thread work-groups: 6 waves per SIMD (80
// VGPRs, without held twiddle powers) fit three of them to a CU, 5 only two (128
// right-hand sides at 128 x 96 x 64: 739 us with two, 695 with three).
template <typename R, int N, int PPT, int T> struct P3Waves {
  static constexpr bool many = sizeof(R) == 4 && PPT <= 8 && T == 64;
  static constexpr int value = sizeof(R) == 4 ? (PPT > 20 ? 2 : PPT > 12 && N < 1024 ? 3 : many ? 6 : 4) : 1;
};

// Pass 3 with a static plan of length N = Gz (see k_pass3 for the mapping).
// Thread (l, t) holds, of every component, the points z = t + K_e of the plan's
// first stage (K_e a compile-time constant per register e), so one lane offset
// t * Gy * Gx + l addresses all of them from per-(component, e) uniform bases;
// each such buffer's range ends at z = Bz (points at and beyond it read as zero
// and are not stored) and spans at most TPC planes, which have to stay below 4 GiB
// (z_offsets_fit). The tensor is read through one buffer per component with a lane
// offset per point.
// PL is the plan (StaticPlan<N, W>, a PlanOf variant or a GenPlan, whose idle
// threads the ranges and, for the tensor, first_ok leave out).
template <typename R, int N, int T, typename PL>
__global__ __launch_bounds__(T * PL::TPC)
__attribute__((amdgpu_waves_per_eu(P3Waves<R, N, PL::PPT, T>::value))) void k_pass3s(typename CxT<R>::T* a2,
                                                                              const typename CxT<R>::T* __restrict__ dhat,
                                                MvDims d, const typename CxT<R>::T* __restrict__ tw, int nwork,
                                                int nper, int nrhs, RhsFlags fl) {
  typedef typename CxT<R>::T C;
  typedef PL P;
  constexpr int PPT = P::PPT;
  constexpr int TPC = P::TPC;
  typedef typename P::Fwd F;
  typedef typename Reverse<F>::type Inv;
  const int ntx = (d.Gx + T - 1) / T;
  const int ftn = (ntx + 1) / 2;
  const int hx = d.Gx / 2, hy = d.Gy / 2, hz = N / 2;
  const int w = (blockIdx.x & 7) * nper + (blockIdx.x >> 3);
  if (w >= nwork) return;
  const int sub = w & 3, q = w >> 2;
  const int rhs = q % nrhs, grp = q / nrhs;
  if (stopped(fl, rhs)) return;
  a2 += (long long)rhs * 3 * d.Bz * d.p2;
  if (d.dhat_tab) dhat = (const typename CxT<R>::T*)d.dhat_tab[d.member[rhs]];
  const int ft = grp % ftn, fyp = grp / ftn;
  int ky = fyp, tile_x = ft;
  if (sub & 2) {
    if (fyp == 0 || fyp == hy) return;
    ky = d.Gy - fyp;
  }
  if (sub & 1) {
    tile_x = ntx - 1 - ft;
    if (tile_x == ft) return;
  }
  extern __shared__ char smem[];
  C* tile = reinterpret_cast<C*>(smem);
  constexpr int lp = (T & 1) ? T : T + 1;
  const int l = threadIdx.x % T, t = threadIdx.x / T;
  const int kx = tile_x * T + l;
  const bool colok = kx < d.Gx;
  const long long cstride = (long long)d.Bz * d.p2;
  const uint32_t zstride = (uint32_t)d.p2;
  C* base = a2 + (long long)ky * d.rs + (long long)tile_x * T;
  // lanes of columns beyond Gx address past every range
  const uint32_t voff = colok ? ((uint32_t)t * zstride + l) * (uint32_t)sizeof(C) : 0xfffffff0u;
  auto range = [&](const C* b, int c, int e) {
    const int z0 = first_point<N, TPC, F>(0, e);
    // the planes of register e: one per thread that has the butterfly, up to Bz
    constexpr int R0 = FirstRadix<F>::value;
    const int own = N / R0 - e / R0 * TPC < TPC ? N / R0 - e / R0 * TPC : TPC;
    const int nz = d.Bz - z0 < own ? d.Bz - z0 : own;
    return zrsrc(b + c * cstride + (long long)z0 * zstride, nz > 0 ? (uint32_t)nz * zstride * sizeof(C) : 0u);
  };
  constexpr int NF = first_count<N, TPC, F>(), NI = first_count<N, TPC, Inv>();
  C reg[3][PPT];
#pragma unroll
  for (int c = 0; c < 3; c++)
#pragma unroll
    for (int e = 0; e < NF; e++)
      reg[c][e] = upper_half<F>(e) ? czero<C>() : zload(range(base, c, e), voff, (C*)nullptr);
  // Bz <= N/2 (the grid holds at least twice the box): the forward transforms
  // skip the zero upper half and the inverse ones never form it; two-stage
  // plans form the second-stage twiddle powers once for all six transforms
  // (FP64 and 32-point plans: no registers to spare)
  constexpr bool PRE = TwoStage<N, TPC, F>::value && sizeof(R) == 4 && PPT <= 16 && !P3Waves<R, N, PPT, T>::many;
  C wp[PRE ? PPT - 1 : 1];
  if constexpr (PRE) twiddle_powers<PPT - 1, P::template twiddles<R>>(wp, t, tw);
  const C* twp = PRE ? wp : tw;
  constexpr int TW = PRE ? (int)TW_HELD : P::template twiddles<R>;
#pragma unroll
  for (int c = 0; c < 3; c++) {
    RunStages<N, TPC, false, 1, C, F, true, TW>::run(reg[c], t, tile, lp, l, twp);
    // (General plans: one component's last stage at a time, and below one point
    // of the product at a time. Left to itself the compiler keeps the three
    // components' inputs and all points' tensor values until the stores of the
    // next stage, and spills: 448 bytes a lane at 72 = 8 * 9 points, FP32.)
    if constexpr (P::general) keep_here<NI>(reg[c]);
  }
  const uint32_t plane = (uint32_t)(hy + 1) * (hx + 1);
  const uint32_t oct = plane * (uint32_t)(hz + 1);
  const int fy = ky <= hy ? ky : d.Gy - ky;
  const R sy = ky <= hy ? (R)1 : (R)-1;
  const int fx = kx <= hx ? kx : d.Gx - kx;
  const R sx = kx <= hx ? (R)1 : (R)-1;
  const uint32_t fyx = colok ? (uint32_t)fy * (hx + 1) + fx : 0u;
  const R sxy = sx * sy;
  // (issuing point e + 1's tensor loads before point e is formed was measured
  // slower: 275 -> 310 us per 2-RHS FP32 launch at 256^3, 300 -> 347 us FP64; in
  // general plans the loads of 2 or 4 points together: 57 -> 62 us, the product
  // of a two-material FP64 particle at 80 x 80 x 72)
#pragma unroll
  for (int e = 0; e < NI; e++) {
    if constexpr (P::general) __builtin_amdgcn_sched_barrier(0);
    const int kz = first_point<N, TPC, Inv>(t, e);
    const int fz = kz <= hz ? kz : N - kz;
    const R sz = kz <= hz ? (R)1 : (R)-1;
    uint32_t o = ((uint32_t)fz * plane + fyx) * (uint32_t)sizeof(C);
    // a butterfly that the thread does not have reads beyond the range: zeros
    if constexpr (P::general) o = max(o, first_ok<N, TPC, Inv>(t, e) ? 0u : 0xfffffff0u);
    C dc[6];
#pragma unroll
    for (int c = 0; c < 6; c++) dc[c] = zload(zrsrc(dhat + (size_t)c * oct, oct * sizeof(C)), o, (C*)nullptr);
    const C d0 = dc[0], d1 = cscale(dc[1], sxy), d2 = cscale(dc[2], sx * sz), d3 = dc[3], d4 = cscale(dc[4], sy * sz),
            d5 = dc[5];
    const C x0 = reg[0][e], x1 = reg[1][e], x2 = reg[2][e];
    reg[0][e] = cdot3(d0, x0, d1, x1, d2, x2);
    reg[1][e] = cdot3(d1, x0, d3, x1, d4, x2);
    reg[2][e] = cdot3(d2, x0, d4, x1, d5, x2);
    if constexpr (P::general) {
#pragma unroll
      for (int c = 0; c < 3; c++) keep_here<1>(&reg[c][e]);
    }
  }
  // the store resources are formed anew (an opaque copy of the base keeps the
  // compiler from holding the load ones in scalar registers across the
  // transforms)
  C* sbase = base;
  asm volatile("" : "+s"(sbase));
#pragma unroll
  for (int c = 0; c < 3; c++) {
    RunStages<N, TPC, true, 1, C, Inv, false, TW>::run(reg[c], t, tile, lp, l, twp);
#pragma unroll
    for (int e = 0; e < NF; e++)
      if (!upper_half<F>(e)) zstore(range(sbase, c, e), voff, reg[c][e]);
  }
}

// Pass 1 with a static plan of length N = Gx. A work-group takes LN consecutive
// lines g = c * n_list + slot over the rows of row_list (those in the planes'
// occupied ranges, which pass 2 reads; null: every row); thread (l, t),
// t = tid mod TPC along the line, reads its first-stage points straight from the
// vector through the cell map (only x < Bx <= N/2 can hold dipoles) and stores
// its outputs, TPC consecutive points per line, coalesced.
// (With the row's dipoles scattered into a zeroed LDS tile first, two barriers
// and two LDS trips more: 70 us at 256^3, FP64 and two FP32 right-hand sides,
// against 57; 282 against 250 at 512^3. What is left is writing A1.)
template <typename R, int N, typename PL, int BS = 256>
__global__ __launch_bounds__(BS) void k_pass1s(const typename CxT<R>::T* __restrict__ x,
                                                typename CxT<R>::T* __restrict__ a1,
                                                const uint32_t* __restrict__ row_list, int n_list,
                                                const uint32_t* __restrict__ cell, const uint8_t* __restrict__ mat,
                                                const typename CxT<R>::T* __restrict__ ccs, MvDims d,
                                                const typename CxT<R>::T* __restrict__ tw, int conj, RhsFlags fl) {
  typedef typename CxT<R>::T C;
  typedef PL P;
  constexpr int PPT = P::PPT;
  constexpr int TPC = P::TPC;
  constexpr int LN = BS / TPC;
  // (threads beyond LN * TPC, where TPC does not divide BS, work on a line of
  // the tile that is never filled from or stored to the vectors)
  constexpr int LP = (BS + TPC - 1) / TPC;
  constexpr int lp = (LP & 1) ? LP : LP + 1;
  constexpr int NF = first_count<N, TPC, typename P::Fwd>(), NO = first_count<N, TPC, typename Reverse<typename P::Fwd>::type>();
  typedef typename P::Fwd F;
  typedef typename Reverse<F>::type Out;
  const int rhs = blockIdx.y;
  if (stopped(fl, rhs)) return;
  x += (long long)rhs * 3 * d.S;
  a1 += (long long)rhs * 3 * d.nrows * d.rs;
  ccs += rhs * 3 * d.nmat;
  if (d.member) mat += (size_t)d.member[rhs] * d.nv;
  extern __shared__ char smem[];
  C* tile = reinterpret_cast<C*>(smem);
  const int t = threadIdx.x % TPC, l = threadIdx.x / TPC;
  const int nlines = 3 * n_list;
  const int g = l < LN ? (int)blockIdx.x * LN + l : nlines;
  const bool ok = g < nlines;
  const int c = ok ? g / n_list : 0, slot = ok ? g - c * n_list : 0;
  const int row = row_list ? (int)row_list[slot] : slot;
  const uint32_t* cells = cell + (size_t)row * d.Bx;
  x += (size_t)c * d.S;
  uint32_t at[NF];
#pragma unroll
  for (int e = 0; e < NF; e++) {
    const int p = first_point<N, TPC, F>(t, e);
    at[e] = !upper_half<F>(e) && ok && p < d.Bx && first_ok<N, TPC, F>(t, e) ? cells[p] : kNoDipole;
  }
  C v[PPT];
#pragma unroll
  for (int e = 0; e < NF; e++) {
    v[e] = czero<C>();
    if (!upper_half<F>(e) && at[e] != kNoDipole) {
      const C xv = x[at[e]];
      v[e] = cmul(ccs[3 * (d.nmat > 1 ? mat[at[e]] : 0) + c], conj ? cconj(xv) : xv);
    }
  }
  RunStages<N, TPC, false, 1, C, F, true, P::template twiddles<R>>::run(v, t, tile, lp, l, tw);
  if (ok) {
    C* dst = a1 + ((size_t)c * d.nrows + row) * d.rs;
#pragma unroll
    for (int e = 0; e < NO; e++)
      if (first_ok<N, TPC, Out>(t, e)) cstore<true>(dst + first_point<N, TPC, Out>(t, e), v[e]);
  }
}

// The sums a pass 5 work-group forms over the entries it writes, in double,
// with x and y as stored: x.y (DOT_U: q0, q1), |y|^2 (DOT_NORM: q0) or |y|^2
// and x.conj(y) (DOT_OM: q0, q1, q2). Block sums of them, in a fixed order,
// are stored as a solver's partial sums:
// quantity q of work-group b of the launch's right-hand side r at
// dot[(r * 4 + q) * gridDim.x + b]. Every thread of the block calls it.
template <int BS>
__device__ inline void dot_partials(double* dot, int op, double q0, double q1, double q2) {
  __shared__ double red[3][BS / 64];
  for (int off = 32; off > 0; off >>= 1) {
    q0 += __shfl_xor(q0, off, 64);
    q1 += __shfl_xor(q1, off, 64);
    q2 += __shfl_xor(q2, off, 64);
  }
  const int w = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) {
    red[0][w] = q0;
    red[1][w] = q1;
    red[2][w] = q2;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    const int nq = op == DOT_U ? 2 : op == DOT_NORM ? 1 : 3;
    double* p = dot + (long long)blockIdx.y * 4 * gridDim.x + blockIdx.x;
    for (int q = 0; q < nq; q++) {
      double t = 0;
      for (int i = 0; i < BS / 64; i++) t += red[q][i];
      p[(long long)q * gridDim.x] = t;
    }
  }
}

// Pass 5 with a static plan: lines g = c * n_list + slot over the non-empty
// rows; inverse transform from A1 (loads coalesced), the kept half (x < Bx) goes
// from the registers of the last stage to the dipoles that the cell map names.
// (Through an LDS tile and the rows' dipole lists: 66 us at 256^3 (two FP32
// right-hand sides) against 58, 231 against 218 at 512^3, 168 against 159 for 128
// right-hand sides at 128 x 96 x 64; with the cells loaded after A1, whose loads
// the entries of x then wait for, 68, 235 and 177.)
// dot_op != DOT_NONE: also the partial sums of x and y (dot_partials) into dot.
template <typename R, int N, typename PL, int BS = 256>
__global__ __launch_bounds__(BS) void k_pass5s(const typename CxT<R>::T* __restrict__ a1,
                                                const typename CxT<R>::T* __restrict__ x,
                                                typename CxT<R>::T* __restrict__ y,
                                                const uint32_t* __restrict__ row_list, int n_list,
                                                const uint32_t* __restrict__ cell, const uint8_t* __restrict__ mat,
                                                const typename CxT<R>::T* __restrict__ ccs, MvDims d,
                                                const typename CxT<R>::T* __restrict__ tw, int conj, RhsFlags fl,
                                                double* __restrict__ dot, int dot_op) {
  typedef typename CxT<R>::T C;
  typedef PL P;
  constexpr int PPT = P::PPT;
  constexpr int TPC = P::TPC;
  constexpr int LN = BS / TPC;
  constexpr int LP = (BS + TPC - 1) / TPC;  // as in k_pass1s
  constexpr int lp = (LP & 1) ? LP : LP + 1;
  typedef typename P::Bwd F;
  typedef typename Reverse<F>::type Out;
  constexpr int NF = first_count<N, TPC, F>(), NO = first_count<N, TPC, Out>();
  const int rhs = blockIdx.y;
  if (stopped(fl, rhs)) return;
  a1 += (long long)rhs * 3 * d.nrows * d.rs;
  x += (long long)rhs * 3 * d.S;
  y += (long long)rhs * 3 * d.S;
  ccs += rhs * 3 * d.nmat;
  if (d.member) mat += (size_t)d.member[rhs] * d.nv;
  extern __shared__ char smem[];
  C* tile = reinterpret_cast<C*>(smem);
  const int t = threadIdx.x % TPC, l = threadIdx.x / TPC;
  const int g = blockIdx.x * LN + l;
  const bool ok = l < LN && g < 3 * n_list;
  const int c = ok ? g / n_list : 0;
  const int row = ok ? (int)row_list[g - c * n_list] : 0;
  const C* src = a1 + ((size_t)c * d.nrows + row) * d.rs;
  // the dipoles of this thread's outputs come first (their x entries wait for
  // them alone, and are there when the transform ends)
  const uint32_t* cells = cell + (size_t)row * d.Bx;
  x += (size_t)c * d.S;
  uint32_t at[NO];
#pragma unroll
  for (int e = 0; e < NO; e++) {
    const int p = first_point<N, TPC, Out>(t, e);
    at[e] = !upper_half<Out>(e) && ok && p < d.Bx && first_ok<N, TPC, Out>(t, e) ? cells[p] : kNoDipole;
  }
  C v[PPT];
#pragma unroll
  for (int e = 0; e < NF; e++)
    v[e] = ok && first_ok<N, TPC, F>(t, e) ? src[first_point<N, TPC, F>(t, e)] : czero<C>();
  __builtin_amdgcn_sched_barrier(0);
  C ga[NO];
#pragma unroll
  for (int e = 0; e < NO; e++) ga[e] = !upper_half<Out>(e) && at[e] != kNoDipole ? x[at[e]] : czero<C>();
  RunStages<N, TPC, true, 1, C, F, false, P::template twiddles<R>>::run(v, t, tile, lp, l, tw);
  double q0 = 0, q1 = 0, q2 = 0;
#pragma unroll
  for (int e = 0; e < NO; e++) {
    if (!upper_half<Out>(e) && at[e] != kNoDipole) {
      C a = ga[e];
      if (conj) a = cconj(a);
      C r = cadd(cmul(ccs[3 * (d.nmat > 1 ? mat[at[e]] : 0) + c], v[e]), a);
      if (conj) r = cconj(r);
      y[(size_t)c * d.S + at[e]] = r;
      if (dot_op != DOT_NONE) {
        const double xr = ga[e].x, xi = ga[e].y, yr = r.x, yi = r.y;
        const bool du = dot_op == DOT_U;
        q0 += du ? xr * yr - xi * yi : yr * yr + yi * yi;
        q1 += du ? xr * yi + xi * yr : xr * yr + xi * yi;
        q2 += xi * yr - xr * yi;
      }
    }
  }
  if (dot_op != DOT_NONE) dot_partials<BS>(dot, dot_op, q0, q1, q2);
  if (blockIdx.x == 0) {
    const int pad = d.S - d.nv;
    for (int q = threadIdx.x; q < 3 * pad; q += blockDim.x) {
      const int cc = q / pad;
      y[(size_t)cc * d.S + d.nv + (q - cc * pad)] = czero<C>();
    }
  }
}

// Column FFT with a static plan (pass 2 / pass 4 and the tensor generation).
// HIN: in_len <= N/2, the zero upper half of the input is skipped; HOUT:
// out_len <= N/2, the upper half of the output is never formed.
template <typename R, int N, int T, typename PL, bool INV, bool HIN, bool HOUT>
__global__ __launch_bounds__(T * PL::TPC) void k_colfft_s(const typename CxT<R>::T* in,
                                                                                typename CxT<R>::T* out, ColParams cp,
                                                  const typename CxT<R>::T* __restrict__ tw, RhsFlags fl) {
  typedef typename CxT<R>::T C;
  typedef PL P;
  constexpr int PPT = P::PPT;
  constexpr int TPC = P::TPC;
  typedef std::conditional_t<INV, typename P::Bwd, typename P::Fwd> F;
  typedef typename Reverse<F>::type Out;
  constexpr int NF = first_count<N, TPC, F>(), NO = first_count<N, TPC, Out>();
  if (stopped(fl, blockIdx.y / fl.per)) return;
  extern __shared__ char smem[];
  C* tile = reinterpret_cast<C*>(smem);
  constexpr int lp = (T & 1) ? T : T + 1;
  const int l = threadIdx.x % T, t = threadIdx.x / T;
  const int col = blockIdx.x * T + l;
  const bool colok = col < cp.ncols;
  const C* src = in + (long long)blockIdx.y * cp.bstride_in + col;
  C* dst = out + (long long)blockIdx.y * cp.bstride_out + col;
  int in0 = 0, in1 = cp.in_len, out0 = 0, out1 = cp.out_len;
  if (cp.yr) {
    const int2 r = cp.yr[cp.nz.mod(blockIdx.y)];
    (INV ? out0 : in0) = r.x;
    (INV ? out1 : in1) = r.y;
  }
  C v[PPT];
#pragma unroll
  for (int e = 0; e < NF; e++) {
    const int p = first_point<N, TPC, F>(t, e);
    v[e] = (!(HIN && upper_half<F>(e)) && first_ok<N, TPC, F>(t, e) && colok && p >= in0 && p < in1)
               ? src[p * cp.pstride_in] : czero<C>();
  }
  RunStages<N, TPC, INV, 1, C, F, HIN, P::template twiddles<R>>::run(v, t, tile, lp, l, tw);
#pragma unroll
  for (int e = 0; e < NO; e++) {
    const int p = first_point<N, TPC, Out>(t, e);
    if (!(HOUT && upper_half<Out>(e)) && first_ok<N, TPC, Out>(t, e) && colok && p >= out0 && p < out1)
      cstore<INV>(dst + p * cp.pstride_out, v[e]);
  }
}

namespace {

template <typename K>
dda_status set_lds(K kernel, size_t bytes) {
  if (bytes > 64 * 1024) DDA_TRY_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                                         hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes));
  return DDA_OK;
}

// Columns per work-group for a static plan: 128-byte row segments, at most 256
// threads.
// Long columns (512, 1024 points) keep 128-byte segments with larger
// work-groups: up to 1024 threads for a single-component transform, 512 for
// the Z pass, whose threads hold three components. PREF (if nonzero) asks for
// that many columns instead.
template <typename R, int N, bool W, int MAXT = 256, int PREF = 0>
constexpr int static_cols() {
  constexpr int pref = PREF ? PREF : sizeof(R) == 8 ? 8 : 16;
  constexpr int tpc = N / StaticPlan<N, W>::PPT;
  constexpr int cap = N >= 512 ? MAXT : 256;
  // at least one full wavefront per work-group
  constexpr int t = pref * tpc < 64 ? 64 / tpc : pref;
  return t * tpc <= cap ? t : cap / tpc;
}

// Plan width of a static kernel: 1 = wide (16 points per thread where the plan
// has them), 0 = narrow, -1 = the precision's default (wide for complex float).
template <typename R>
inline bool plan_wide(int w) {
  return w < 0 ? sizeof(R) == 4 : w != 0;
}

// The other tile the tuner tries for the FP32 Y passes: twice the default
// columns per work-group where that stays within 1024 threads, else half
// (keeping at least one wavefront).
template <int T, int TPC>
constexpr int other_cols() {
  return 2 * T * TPC <= 1024 ? 2 * T : (T / 2) * TPC >= 64 ? T / 2 : T;
}
// and the third: four times the default columns where that stays within 1024
// threads and the LDS (FP32 tiles of N x (4T + 1) points), else the second
template <int T, int TPC, int N>
constexpr int third_cols() {
  return 4 * T * TPC <= 1024 && (size_t)N * (4 * T + 1) * 8 <= 160 * 1024 ? 4 * T : other_cols<T, TPC>();
}

// ALT: 0 the default tile, 1 other_cols, 2 third_cols
template <typename R, int N, bool W, bool INV, int ALT = 0>
dda_status launch_col_static_w(const void* in, void* out, const ColParams& cp, const void* tw, int nbatch,
                               hipStream_t st, RhsFlags done) {
  typedef typename CxT<R>::T C;
  constexpr int T0 = static_cols<R, N, W, 1024>();
  typedef StaticPlan<N, W> PL;
  constexpr int TPC0 = PL::TPC;
  constexpr int T = ALT == 0 ? T0 : ALT == 1 ? other_cols<T0, TPC0>() : third_cols<T0, TPC0, N>();
  constexpr int threads = T * PL::TPC;
  constexpr int lp = (T & 1) ? T : T + 1;
  const size_t lds = (size_t)N * lp * sizeof(C);
  // the matvec's forward pass reads at most N/2 points and its inverse pass
  // keeps at most N/2; the tensor generation transforms full lengths
  const bool hin = !INV && 2 * cp.in_len <= N, hout = INV && 2 * cp.out_len <= N;
  void (*k)(const C*, C*, ColParams, const C*, RhsFlags);
  if constexpr (ALT != 0) {
    // the other tiles are matvec variants: full-length transforms keep the default
    if (!hin && !hout) return launch_col_static_w<R, N, W, INV, 0>(in, out, cp, tw, nbatch, st, done);
    k = INV ? k_colfft_s<R, N, T, PL, INV, false, INV> : k_colfft_s<R, N, T, PL, INV, !INV, false>;
  } else {
    k = hin ? k_colfft_s<R, N, T, PL, INV, !INV, false>
            : hout ? k_colfft_s<R, N, T, PL, INV, false, INV> : k_colfft_s<R, N, T, PL, INV, false, false>;
  }
  DDA_TRY(set_lds(k, lds));
  hipLaunchKernelGGL(k, dim3((cp.ncols + T - 1) / T, nbatch), dim3(threads), lds, st, (const C*)in, (C*)out, cp,
                     (const C*)tw, done);
  DDA_TRY_HIP(hipGetLastError());
  return DDA_OK;
}

// The FP32 variant of an untuned Y pass over ncols columns of nbatch batches.
// Tiles of 64 columns (512-byte row segments) where they divide the rows and
// leave 24 work-groups per CU: there the pass streams through HBM, and a 96-point
// launch for 128 right-hand sides takes 318 us forward and 298 inverse against
// 357 and 323 (whole products 1.5 to 3.4% less at 64 to 96 points); with fewer
// work-groups 16 columns are as fast or faster, at 192 and 256 points always (by
// up to 7%). At 512 points the narrow plan, which has three stages like the wide
// one and half its registers: 442 and 418 us against 476 and 435 at 512^3.
inline int default_col_variant(int n, int ncols, int nbatch) {
  if (n == 512) return 0;
  if (n > 128 || ncols % 64 || (long long)(ncols / 64) * nbatch < 6144) return 1;
  return n >= 48 ? 5 : 3;
}

// wide: -1 the precision's default plan, 0 narrow, 1 wide; FP32 also 2 and 3,
// narrow and wide with the second tile (other_cols), and 4 and 5 with the
// third (third_cols).
template <typename R, int N, bool INV>
dda_status launch_col_static(const void* in, void* out, const ColParams& cp, const void* tw, int nbatch, hipStream_t st,
                             RhsFlags done, int wide) {
  if constexpr (sizeof(R) == 4) {
    if (wide < 0) wide = default_col_variant(N, cp.ncols, nbatch);
    if (wide >= 4)
      return (wide & 1) ? launch_col_static_w<R, N, true, INV, 2>(in, out, cp, tw, nbatch, st, done)
                        : launch_col_static_w<R, N, false, INV, 2>(in, out, cp, tw, nbatch, st, done);
    if (wide >= 2)
      return (wide & 1) ? launch_col_static_w<R, N, true, INV, 1>(in, out, cp, tw, nbatch, st, done)
                        : launch_col_static_w<R, N, false, INV, 1>(in, out, cp, tw, nbatch, st, done);
  }
  return plan_wide<R>(wide >= 2 ? (wide & 1) : wide) ? launch_col_static_w<R, N, true, INV>(in, out, cp, tw, nbatch, st, done)
                                                    : launch_col_static_w<R, N, false, INV>(in, out, cp, tw, nbatch, st, done);
}

// Whether the passes of nrhs right-hand sides leave out the rows outside the
// planes' occupied ranges: where A1 is larger than half of the L2s. In a small
// one the saved lines cost nothing and the ranges' loads come before the data's:
// the product of the sphere 40 across (6 MB) 37.6 us with them, 37.0 without;
// 256^3 (200 MB) 598 and 622.
inline bool use_ranges(const dda_op_s* op, int nrhs) {
  const MvDims& d = op->dims;
  return op->yrange && (size_t)nrhs * 3 * d.nrows * d.rs * (op->prec / 4) > (16u << 20);
}

inline MvView view_of(const dda_op_s* op, int r0) {
  const MvDims& d = op->dims;
  const size_t csz = op->prec == 64 ? sizeof(double2) : sizeof(float2);
  MvView v;
  v.a1 = (char*)op->a1 + (size_t)r0 * 3 * d.Bz * d.By * d.rs * csz;
  v.a2 = (char*)op->a2 + (size_t)r0 * 3 * d.Bz * d.p2 * csz;
  v.ccs = (const char*)op->ccs + (size_t)r0 * 3 * d.nmat * csz;
  v.d = d;
  if (d.member) v.d.member = d.member + r0;
  return v;
}

template <typename R, int N, typename PL, int T>
dda_status launch_pass3_plan(dda_op_s* op, const MvView& v, hipStream_t st, RhsFlags done, int nrhs) {
  typedef typename CxT<R>::T C;
  constexpr int threads = T * PL::TPC;
  constexpr int lp = (T & 1) ? T : T + 1;
  const MvDims& d = v.d;
  const size_t lds = (size_t)N * lp * sizeof(C);
  const int ntx = (d.Gx + T - 1) / T;
  const int nwork = (d.Gy / 2 + 1) * ((ntx + 1) / 2) * 4 * nrhs;
  const int nper = (nwork + 7) / 8;
  auto k = k_pass3s<R, N, T, PL>;
  DDA_TRY(set_lds(k, lds));
  hipLaunchKernelGGL(k, dim3(8 * nper), dim3(threads), lds, st, (C*)v.a2, (const C*)op->dhat, d,
                     (const C*)op->tw[2], nwork, nper, nrhs, done);
  DDA_TRY_HIP(hipGetLastError());
  return DDA_OK;
}

// The other tile of the FP32 Z pass: 64 columns where the default is 32 (at most
// 64 points), 32 where it is 16 and 32 fit the work-group size the kernel's
// register budget allows (MAXTH threads), else half the default.
template <int T, int TPC, int MAXTH>
constexpr int other_cols_z() {
  return T == 32 ? 64 : 32 * TPC <= MAXTH ? 32 : (T / 2) * TPC >= 64 ? T / 2 : T;
}
// Whether an untuned FP32 Z pass of at most 64 points takes the 64-column tile:
// where tiles pair with their x mirrors (the tensor is read once for both) and
// there are 24 work-groups per CU. 128 right-hand sides at 128 x 96 x 64: 695
// against 756 us, at 128 x 96 x 48 536 against 567, x 32 378 against 381; 32 at
// x 64 2.7% less for the whole product, 8 3% more; 64 x 64 x 64, where one tile
// is its own mirror, 188 against 121 us.
inline bool wide_z_tile(const MvDims& d, int nrhs) {
  return d.Gx % 128 == 0 && (long long)(d.Gx / 64) * d.Gy * nrhs >= 6144;
}

template <typename R, int N, bool W, bool ALT = false>
dda_status launch_pass3_static_w(dda_op_s* op, const MvView& v, hipStream_t st, RhsFlags done, int nrhs) {
  // FP32 1024-point columns: 16 columns (128-byte segments) in a 1024-thread
  // work-group at 128 VGPRs, the CU's whole register file (17.5 ms at 1024^3,
  // against 22.7 ms for two 512-thread work-groups of 8 columns)
  // short FP32 columns (at most 64 points): 32 columns (256-byte segments)
  // per work-group; measured on a 128-RHS block at a 64-point Z grid: 935 ->
  // 781 us per launch
  constexpr int T0 = static_cols<R, N, W, (N == 1024 && sizeof(R) == 4 && W) ? 1024 : 512,
                                 (sizeof(R) == 4 && N <= 64) ? 32 : 0>();
  constexpr int TPC = N / StaticPlan<N, W>::PPT;
  constexpr int T = ALT ? other_cols_z<T0, TPC, 256 * P3Waves<R, N, StaticPlan<N, W>::PPT, T0>::value>() : T0;
  return launch_pass3_plan<R, N, StaticPlan<N, W>, T>(op, v, st, done, nrhs);
}

// Z-pass variants (Tune::p3_wide): -1 the precision's default, 0 narrow,
// 1 wide; at 512 and 1024 points also 2 and 3, plans of 32 points per thread
// (32 x 16 and 32 x 32: one LDS exchange per transform, 2 waves per SIMD, FP32)
// over 16 columns (128-byte segments; at 1024 points 512 threads, one work-group
// per CU by LDS, at 512 points 256 threads, two work-groups) or 8 columns.
// FP32 only: in FP64 the 32-point plan's data alone needs 384 VGPRs. The FP32
// default is 2 there: at 1024^3 (sphere 512 across) 14.8 ms against 17.8 ms
// (wide), 19.2 ms (variant 3) and 33.0 ms (narrow); at 512^3 1,608 us against
// 1,842, 2,385 and 2,051 (the wide plan's 512 threads of 168 VGPRs leave one
// work-group per CU, and a third stage of radix 2 costs it an LDS exchange more).
// At 512 points with TW_SPLIT, the products' error is 1.5e-7 where the wide
// plan's chained powers made it 2.0e-7.
// (Two further forms were measured and dropped. The wide plan without held
// twiddle powers at 4 waves per SIMD, 128 VGPRs: 308.8 against 293.2 us per
// 2-RHS FP32 launch at 256^3, and it spills at 32, 128 and 512 points. A
// persistent kernel, resident work-groups looping over the tiles and loading
// each component of the next tile into the registers its store frees:
// 303.5 against 289.3 us (2-RHS FP32, 256^3), 315.0 against 291.4 us (FP64),
// 15.1 against 14.6 ms (FP32, 1024^3); its loop costs 13% more VALU at 1024
// points than the hidden loads save.)
template <int N> struct Plan32;
template <> struct Plan32<1024> : PlanOf<1024, 32, RadixList<32, 32>> {};
template <> struct Plan32<512> : PlanOf<512, 32, RadixList<32, 16>, TW_SPLIT> {};
// FP32 below 1024 points: 2 and 3 are the narrow and wide plans with the
// other tile (other_cols_z).
inline int p3_variants(int n, int prec) { return prec == 32 ? 4 : 2; }
// The variant of an untuned Z pass.
inline int default_p3_variant(const MvDims& d, int prec, int nrhs) {
  if (prec == 64) return 0;
  return d.Gz >= 512 ? 2 : d.Gz <= 64 && wide_z_tile(d, nrhs) ? 3 : 1;
}

template <typename R, int N>
dda_status launch_pass3_static(dda_op_s* op, const MvView& v, hipStream_t st, RhsFlags done, int nrhs,
                               const dda_op_s::Tune& tn) {
  const int var = tn.p3_wide < 0 ? default_p3_variant(v.d, 8 * (int)sizeof(R), nrhs) : tn.p3_wide;
  if constexpr (N >= 512 && sizeof(R) == 4) {
    if (var == 2) return launch_pass3_plan<R, N, Plan32<N>, 16>(op, v, st, done, nrhs);
    if (var == 3) return launch_pass3_plan<R, N, Plan32<N>, 8>(op, v, st, done, nrhs);
  } else if constexpr (sizeof(R) == 4) {
    if (var >= 2)
      return (var & 1) ? launch_pass3_static_w<R, N, true, true>(op, v, st, done, nrhs)
                       : launch_pass3_static_w<R, N, false, true>(op, v, st, done, nrhs);
  }
  return (var & 1) ? launch_pass3_static_w<R, N, true>(op, v, st, done, nrhs)
                   : launch_pass3_static_w<R, N, false>(op, v, st, done, nrhs);
}

template <typename R, int N, typename PL, int BS = 256>
dda_status launch_x_plan(dda_op_s* op, const MvView& v, bool inverse, const void* x, void* y, int conj,
                             hipStream_t st, RhsFlags done, int nrhs, const PassDotReq& dr) {
  typedef typename CxT<R>::T C;
  constexpr int LN = BS / PL::TPC;
  constexpr int LP = (BS + PL::TPC - 1) / PL::TPC;
  constexpr int lp = (LP & 1) ? LP : LP + 1;
  const MvDims& d = v.d;
  const size_t lds = (size_t)N * lp * sizeof(C);
  if (!inverse) {
    auto k = k_pass1s<R, N, PL, BS>;
    DDA_TRY(set_lds(k, lds));
    const bool part = use_ranges(op, nrhs);
    const int n = part ? op->n_active : d.nrows;
    hipLaunchKernelGGL(k, dim3((3 * n + LN - 1) / LN, nrhs), dim3(BS), lds, st, (const C*)x, (C*)v.a1,
                       part ? op->active_list : nullptr, n, op->cell, op->mat_dev, (const C*)v.ccs, d, (const C*)op->tw[0], conj, done);
  } else {
    auto k = k_pass5s<R, N, PL, BS>;
    DDA_TRY(set_lds(k, lds));
    const int nl = 3 * op->n_nonempty;
    const int nbx = nl > 0 ? (nl + LN - 1) / LN : 1;
    op->p5_blocks = nbx;
    double* dot = dr.op != DOT_NONE ? dr.part + (size_t)dr.r0 * 4 * nbx : nullptr;
    hipLaunchKernelGGL(k, dim3(nbx, nrhs), dim3(BS), lds, st, (const C*)v.a1, (const C*)x, (C*)y, op->row_list,
                       op->n_nonempty, op->cell, op->mat_dev, (const C*)v.ccs, d, (const C*)op->tw[0], conj, done, dot,
                       dr.op);
  }
  DDA_TRY_HIP(hipGetLastError());
  return DDA_OK;
}

template <typename R, int N>
dda_status launch_x_static(dda_op_s* op, const MvView& v, bool inverse, const void* x, void* y, int conj,
                           hipStream_t st, RhsFlags done, int nrhs, const dda_op_s::Tune& tn,
                           const PassDotReq& dr = PassDotReq()) {
  // default narrow for both precisions: half the LDS per wave, twice the waves
  // per CU (measured 52 -> 39 us at 256^3 FP32); FP32 also 2 and 3, narrow
  // and wide over 512-thread work-groups (twice the lines each)
  const int var = tn.x_wide[inverse];
  if constexpr (sizeof(R) == 4) {
    if (var >= 2)
      return (var & 1) ? launch_x_plan<R, N, StaticPlan<N, true>, 512>(op, v, inverse, x, y, conj, st, done, nrhs, dr)
                       : launch_x_plan<R, N, StaticPlan<N, false>, 512>(op, v, inverse, x, y, conj, st, done, nrhs, dr);
  }
  return var >= 0 && (var & 1) ? launch_x_plan<R, N, StaticPlan<N, true>>(op, v, inverse, x, y, conj, st, done, nrhs, dr)
                               : launch_x_plan<R, N, StaticPlan<N, false>>(op, v, inverse, x, y, conj, st, done, nrhs, dr);
}

// ------------------------------------------------------------------------------------
// General lengths: one plan (GenPlan) per length, no tuned variants.
// ------------------------------------------------------------------------------------

// Columns per work-group for a plan of TPC threads per column: at least
// 128-byte row segments, and of 1, 2 or 4 times that (up to `most` columns) the
// first count that gives two wavefronts or more, nine tenths of their lanes in
// use, else the one that wastes the fewest lanes, within 512 threads and 80 KB
// of LDS; fewer columns where even the 128 bytes would take more than 768
// threads. The Z pass takes at most 16: with 32 columns the FP64 product at 80^3
// (240 work-groups in the Z pass, less than one per CU) took 47.8 us, with 16
// 38.3 us, with 8 39.1 us; larger grids showed no difference.
template <typename R, int N, int TPC>
constexpr int gen_cols(int most) {
  int base = sizeof(R) == 8 ? 8 : 16;
  while (base > 4 && base * TPC > 768) base /= 2;
  int best = base;
  double best_use = 0;
  for (int t = base; t <= most; t *= 2) {
    const int threads = t * TPC;
    if (t > base && (threads > 512 || (size_t)N * (t + 1) * 2 * sizeof(R) > 80 * 1024)) break;
    const double use = (double)threads / ((threads + 63) / 64 * 64);
    if (threads >= 128 && use >= 0.9) return t;
    const double score = threads < 64 ? use / 2 : use;
    if (score > best_use) {
      best = t;
      best_use = score;
    }
  }
  return best;
}

// The matvec's Y passes only: in_len (forward) or out_len (inverse) <= N / 2.
template <typename R, int N, typename PL>
dda_status launch_gen_col(bool inv, const void* in, void* out, const ColParams& cp, const void* tw, int nbatch,
                          hipStream_t st, RhsFlags done) {
  typedef typename CxT<R>::T C;
  constexpr int T = gen_cols<R, N, PL::TPC>(sizeof(R) == 8 ? 32 : 64);
  constexpr int lp = (T & 1) ? T : T + 1;
  const size_t lds = (size_t)N * lp * sizeof(C);
  auto k = inv ? k_colfft_s<R, N, T, PL, true, false, true> : k_colfft_s<R, N, T, PL, false, true, false>;
  DDA_TRY(set_lds(k, lds));
  hipLaunchKernelGGL(k, dim3((cp.ncols + T - 1) / T, nbatch), dim3(T * PL::TPC), lds, st, (const C*)in, (C*)out, cp,
                     (const C*)tw, done);
  DDA_TRY_HIP(hipGetLastError());
  return DDA_OK;
}

}  // namespace

// The launchers of one grid length in one precision (plans.hip).
struct AxisOps {
  dda_status (*col)(bool inv, const void* in, void* out, const ColParams& cp, const void* tw, int nbatch,
                    hipStream_t st, RhsFlags done);
  dda_status (*z)(dda_op_s* op, const MvView& v, hipStream_t st, RhsFlags done, int nrhs);
  dda_status (*x)(dda_op_s* op, const MvView& v, bool inverse, const void* x, void* y, int conj, hipStream_t st,
                  RhsFlags done, int nrhs, const PassDotReq& dr);
  int z_threads;  // threads per column of the Z pass
};

// The column passes of the interaction tensor's generation: nb batches of ncols
// columns of each of the six components; offsets below clip are read, bit c of
// odd is set for components that are odd in the axis.
struct TensorCols {
  int ncols, clip, nb;
  unsigned odd;
  long long pstride, bstride, cstride_in, cstride_out;
  double scale;
};

// The launchers of those passes at one grid length (tensor.hip).
struct TensorOps {
  dda_status (*rows)(void* w, int cx, int cy, int cz, double kd, long long cstride, long long zstride, const void* tw,
                     hipStream_t st);
  dda_status (*cols)(const void* in, void* out, int out_prec, const TensorCols& tc, const void* tw, hipStream_t st);
};

}  // namespace dda
