// The steps either side of the solve, on the device: the incident plane wave
// per right-hand side (DDA/Beam.cpp:110-118), LDR/CM polarisabilities
// (DDA/PolarizabilityDescription.cpp:65-110), Cext and Cabs
// (DDA/Beam.cpp:58-68, DDA/AbsCross.cpp:27-48), scattered far fields
// (DDA/CpuFieldCalculator.cpp:48-98) and Jones matrices on an angle grid
// (DDA/FarFieldCalc.cpp:119-174, EMSim/JonesCalculus.cpp:74-86). The reference
// evaluates the far field one direction per launch with a host read-back
// (DDA/GpuFieldCalculator.cpp:64-72); here all directions and right-hand sides
// go through one two-stage reduction, many directions as a matrix product.
#include <cmath>
#include <complex>
#include <cstring>
#include <mutex>
#include <vector>

#include "internal.hpp"

// The fixed device scratch of dda_cross_sections_noalloc: one copy of this
// array per GPU the library runs on, held until the process ends. Host code
// never passes the array's name to a kernel or a copy (on the host it is a
// stand-in, not a device address); it uses the per-device address that
// noalloc_scratch_setup takes with hipGetSymbolAddress.
static __device__ __align__(256) double scratch[DDA_NOALLOC_SCRATCH_DOUBLES];

namespace dda {
namespace {

constexpr int kObsThreads = 256;
constexpr double kPi = 3.14159265358979323846264338327950288;

// Grid point (0,0,0) sits at -(box - 1) / 2 grid units (DipoleGeometry::moveToCenter).
struct Frame {
  double ox, oy, oz, d;
};

// einc[r][c][i] = exp(i k r_i . prop_r) pol_r[c] for i < nv, 0 up to S.
__global__ void k_incident(double2* einc, const uint32_t* __restrict__ pos, const double* __restrict__ dirs, int nv,
                           int S, double k, Frame f) {
  const int r = blockIdx.y;
  const double* pr = dirs + 6 * r;  // prop[3], pol[3]
  double2* e = einc + (long long)r * 3 * S;
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < S; i += gridDim.x * blockDim.x) {
    double2 ph = make_double2(0, 0);
    if (i < nv) {
      const double x = f.ox + pos[3 * i] * f.d, y = f.oy + pos[3 * i + 1] * f.d, z = f.oz + pos[3 * i + 2] * f.d;
      double s, c;
      sincos(k * (x * pr[0] + y * pr[1] + z * pr[2]), &s, &c);
      ph = make_double2(c, s);
    }
    for (int c = 0; c < 3; c++) e[(long long)c * S + i] = make_double2(ph.x * pr[3 + c], ph.y * pr[3 + c]);
  }
}

__device__ inline double block_sum(double v) {
  __shared__ double sh[kObsThreads / 64];
  for (int o = 32; o > 0; o >>= 1) v += __shfl_down(v, o, 64);
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = v;
  __syncthreads();
  double t = 0;
  if (threadIdx.x == 0)
    for (int w = 0; w < kObsThreads / 64; w++) t += sh[w];
  __syncthreads();
  return t;
}

// Per-RHS partials of sum Im(p . conj(E)) and sum multDr |p|^2, where
// multDr = -Im(1/alpha) - 2/3 k^3 comes from mdr [nrhs][nmat][3] or, when mdr
// is null, from alpha itself (ccd [nrhs][nmat][3] complex, nullable: then the
// second sum is 0).
__global__ __launch_bounds__(kObsThreads) void k_cross(const double2* __restrict__ pol,
                                                       const double2* __restrict__ einc,
                                                       const uint8_t* __restrict__ mat,
                                                       const double* __restrict__ mdr,
                                                       const double2* __restrict__ ccd, double k3, int nv, int S,
                                                       int nmat, double* part, const int* member) {
  // the last right-hand sides first: what was written last (the fields, the
  // solutions) may still be in the memory-side cache (128 fields of 51,472
  // dipoles straight after k_incident: the two calls 257 -> 245 us)
  const int r = gridDim.y - 1 - blockIdx.y;
  if (member) mat += (size_t)member[r] * nv;
  const double2* p = pol + (long long)r * 3 * S;
  const double2* e = einc + (long long)r * 3 * S;
  const double* md = mdr ? mdr + (long long)r * 3 * nmat : nullptr;
  const double2* ca = ccd ? ccd + (long long)r * 3 * nmat : nullptr;
  double se = 0, sa = 0;
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < nv; i += gridDim.x * blockDim.x) {
    const int m = mat[i];
    for (int c = 0; c < 3; c++) {
      const double2 pv = p[(long long)c * S + i], ev = e[(long long)c * S + i];
      se += pv.y * ev.x - pv.x * ev.y;
      double w = 0;
      if (md) {
        w = md[3 * m + c];
      } else if (ca) {
        const double2 a = ca[3 * m + c];
        w = a.y / (a.x * a.x + a.y * a.y) - k3;  // -Im(1/a) - 2/3 k^3
      }
      sa += w * (pv.x * pv.x + pv.y * pv.y);
    }
  }
  const double te = block_sum(se), ta = block_sum(sa);
  if (threadIdx.x == 0) {
    part[((long long)r * gridDim.x + blockIdx.x) * 2] = te;
    part[((long long)r * gridDim.x + blockIdx.x) * 2 + 1] = ta;
  }
}

// Second stage of k_cross, one thread per right-hand side, blocks summed in
// order: out[r] = scale * sum_b part[r][b][0], out[nrhs + r] = scale * sum_b part[r][b][1].
__global__ void k_cross_final(const double* __restrict__ part, int nb, int nrhs, double scale, double* out) {
  const int r = blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= nrhs) return;
  double se = 0, sa = 0;
  for (int b = 0; b < nb; b++) {
    se += part[((long long)r * nb + b) * 2];
    sa += part[((long long)r * nb + b) * 2 + 1];
  }
  out[r] = scale * se;
  out[nrhs + r] = scale * sa;
}

// Far-field sums S_q = sum_j p_{rhs_q, j} exp(-i kd n_q . pos_j), first stage:
// block (chunk, query tile) -> partials[chunk][q][6].
constexpr int kQT = 4;
__global__ __launch_bounds__(kObsThreads) void k_far_partial(const double2* __restrict__ pol,
                                                             const uint32_t* __restrict__ pos,
                                                             const double* __restrict__ q, int nq, int nv, int S,
                                                             double kd, int chunk, double* part) {
  const int q0 = blockIdx.y * kQT;
  const int j0 = blockIdx.x * chunk, j1 = min(nv, j0 + chunk);
  double acc[kQT][6];
  double n[kQT][3];
  int rhs[kQT];
#pragma unroll
  for (int t = 0; t < kQT; t++) {
    const int qq = min(q0 + t, nq - 1);
    rhs[t] = (int)q[4 * qq];
    for (int a = 0; a < 3; a++) n[t][a] = -kd * q[4 * qq + 1 + a];
    for (int a = 0; a < 6; a++) acc[t][a] = 0;
  }
  for (int j = j0 + threadIdx.x; j < j1; j += blockDim.x) {
    const double x = pos[3 * j], y = pos[3 * j + 1], z = pos[3 * j + 2];
#pragma unroll
    for (int t = 0; t < kQT; t++) {
      double s, c;
      sincos(n[t][0] * x + n[t][1] * y + n[t][2] * z, &s, &c);
      const double2* p = pol + (long long)rhs[t] * 3 * S + j;
#pragma unroll
      for (int a = 0; a < 3; a++) {
        const double2 v = p[(long long)a * S];
        acc[t][2 * a] += v.x * c - v.y * s;
        acc[t][2 * a + 1] += v.x * s + v.y * c;
      }
    }
  }
#pragma unroll
  for (int t = 0; t < kQT; t++)
#pragma unroll
    for (int a = 0; a < 6; a++) {
      const double v = block_sum(acc[t][a]);
      if (threadIdx.x == 0 && q0 + t < nq) part[((long long)blockIdx.x * nq + q0 + t) * 6 + a] = v;
    }
}

// Second stage, one thread per query, chunks summed in order; then
// E = i k^2 exp(-i k origin . n) (S - n (n . S)).
__global__ void k_far_final(const double* __restrict__ part, const double* __restrict__ q, int nq, int nchunk,
                            double k, Frame f, double* out) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= nq) return;
  double s[6] = {0, 0, 0, 0, 0, 0};
  for (int b = 0; b < nchunk; b++)
    for (int a = 0; a < 6; a++) s[a] += part[((long long)b * nq + i) * 6 + a];
  const double n0 = q[4 * i + 1], n1 = q[4 * i + 2], n2 = q[4 * i + 3];
  const double nsr = n0 * s[0] + n1 * s[2] + n2 * s[4], nsi = n0 * s[1] + n1 * s[3] + n2 * s[5];
  double ps, pc;
  sincos(-k * (f.ox * n0 + f.oy * n1 + f.oz * n2), &ps, &pc);
  // f = i k^2 (pc + i ps) = k^2 (-ps + i pc)
  const double fr = -k * k * ps, fi = k * k * pc;
  const double nn[3] = {n0, n1, n2};
  for (int a = 0; a < 3; a++) {
    const double vr = s[2 * a] - nn[a] * nsr, vi = s[2 * a + 1] - nn[a] * nsi;
    out[6 * i + 2 * a] = fr * vr - fi * vi;
    out[6 * i + 2 * a + 1] = fr * vi + fi * vr;
  }
}

// ------------------------------------------------------------------------------------
// Many directions, on the matrix cores.
//
// On the grid exp(-i kd n . r) = ex[x] ey[y] ez[z], so a direction needs
// Bx / 2 + By + Bz sincos and not one per dipole (k_far_tables), and a row's
// sum over x is multiplied by ey ez once. With coordinates from the box's
// centre, the dipoles p+ at x and p- at -x of a row make
//   p+ e^-iu + p- e^iu = (p+ + p-) cos u - i (p+ - p-) sin u,
// half the multiplications. What is left is a real product
// [values of a row's positions] x [cos, sin of the positions for 64 directions],
// in 16 x 16 x 4 FP64 matrix instructions: 16 rows for the real and imaginary
// parts of up to six values (of them 12 are used), two positions, 16 directions.
//
// The sphere 40 across (33,552 dipoles, 5,551 directions, both solutions) takes
// 148 us; its instructions alone take 80 at the 74 TFLOP/s that a large product
// reaches. What is left is the rows' ey ez (a fifth of the FP64 work) and the
// last round of work-groups. The same sums on the vector units, whole rows of
// dipoles from scalar loads and 24 multiply-adds per dipole, took 264 us, a
// sincos per dipole and direction (k_far_partial) 1,480.
// ------------------------------------------------------------------------------------

constexpr int kFarWaves = 8;

// The angle grid of dda_jones: sin and cos of theta and phi, and the frame.
struct FarGrid {
  const double* trig;  // [ntheta][sin, cos], [nphi][sin, cos]
  int ntheta, nphi, symmetric;
  double prop[3], pol1[3], pol2[3];
};
// Where a slot's direction comes from: dirs ([slot][3]) or, where that is
// null, the angle grid (slot = angle, or 2 * angle + evaluation where symmetric).
struct FarDirs {
  const double* dirs;
  FarGrid g;
  int count;  // slots in use
};

// Direction n, perpendicular pe and parallel pa of evaluation f at angle i.
__device__ inline void jones_frame(const FarGrid& g, int i, int f, double n[3], double pe[3], double pa[3]) {
  const double* th = g.trig + 2 * (i / g.nphi);
  const double* ph = g.trig + 2 * (g.ntheta + i % g.nphi);
  const double st = th[0], ct = th[1], sp = ph[0], cp = ph[1];
  const bool rot = f == 1 && g.symmetric;
#pragma unroll
  for (int a = 0; a < 3; a++) {
    const double X = rot ? g.pol1[a] : g.pol2[a], Y = rot ? -g.pol2[a] : g.pol1[a];
    n[a] = ct * g.prop[a] + st * (cp * X + sp * Y);
    pe[a] = sp * X - cp * Y;
    pa[a] = -st * g.prop[a] + ct * (cp * X + sp * Y);
  }
}
// Component a of a slot's direction in dirs (64-bit: 2^30 slots are accepted).
__host__ __device__ constexpr size_t dir_index(int slot, int a) { return 3 * (size_t)slot + a; }
static_assert(dir_index((1 << 30) - 1, 2) == 3221225471u, "direction index");

__device__ inline void far_direction(const FarDirs& f, int slot, double n[3]) {
  if (f.dirs) {
    for (int a = 0; a < 3; a++) n[a] = f.dirs[dir_index(slot, a)];
  } else {
    double pe[3], pa[3];
    if (f.g.symmetric)
      jones_frame(f.g, slot >> 1, slot & 1, n, pe, pa);
    else
      jones_frame(f.g, slot, 0, n, pe, pa);
  }
}

// Part of a row: positions u0, u0 + 1, .. of its folded half (u = 0 at the
// centre), two a step; its records and those of the next segment are back to back.
struct FarSeg {
  int u0, steps, y, z;
};

// Tables of slots slot0 .. slot0 + nslots - 1. cs: cos and sin of kd n_x u, u < nu,
// as the matrix instructions read them, [slot / 64][u][slot / 16 % 4][cos, sin][16];
// yz[entry][slot]: exp(-i kd n_y y), then those of z.
__global__ __launch_bounds__(64) void k_far_tables(FarDirs f, int slot0, int nslots, int nu, double u_first, int By,
                                                   int Bz, double kd, double* cs, double2* yz) {
  const int s = blockIdx.x * 64 + threadIdx.x;
  double n[3] = {0, 0, 0};
  if (slot0 + s < f.count) far_direction(f, slot0 + s, n);
  const int ne = nu + By + Bz;
  for (int e = blockIdx.y; e < ne; e += gridDim.y) {
    double si, co;
    if (e < nu) {
      sincos(kd * n[0] * (e + u_first), &si, &co);
      double* c = cs + (((long long)blockIdx.x * nu + e) * 4 + (threadIdx.x >> 4)) * 32 + (threadIdx.x & 15);
      c[0] = co;
      c[16] = si;
    } else {
      const int i = e - nu;
      const double r = i < By ? i - 0.5 * (By - 1) : i - By - 0.5 * (Bz - 1);
      sincos(-kd * (i < By ? n[1] : n[2]) * r, &si, &co);
      yz[(long long)i * nslots + s] = make_double2(co, si);
    }
  }
}

// Records of the positions (pair: the dipoles at +u and -u, -1 for none):
// rec[position][cos, sin][16], the factors of cos u and sin u in the matrix
// instruction's 16 rows. Lane l holds rows l / 16 + 4 v, v = 0 .. 3, of the
// result: real and imaginary part of value l / 16 (v = 0, 1), of value
// 4 + l / 16 (v = 2, 3). Right-hand sides NR * blockIdx.y on.
template <int NR>
__global__ __launch_bounds__(256) void k_far_pack(const double2* __restrict__ pol, const int2* __restrict__ pair,
                                                  int npos, int S, double* __restrict__ rec) {
  pol += (long long)blockIdx.y * 3 * NR * S;
  rec += (long long)blockIdx.y * npos * 32;
  for (long long k = blockIdx.x * 256ll + threadIdx.x; k < 16ll * npos; k += gridDim.x * 256ll) {
    const int q = (int)(k >> 4), i = (int)(k & 15);
    const int n = (i & 3) + (i >= 8 ? 4 : 0);
    double c = 0, s = 0;
    if (n < 3 * NR) {
      const int2 d = pair[q];
      const double2 a = d.x >= 0 ? pol[(long long)n * S + d.x] : make_double2(0, 0);
      const double2 b = d.y >= 0 ? pol[(long long)n * S + d.y] : make_double2(0, 0);
      c = (i & 4) ? a.y + b.y : a.x + b.x;
      s = (i & 4) ? b.x - a.x : a.y - b.y;
    }
    rec[(long long)q * 32 + i] = c;
    rec[(long long)q * 32 + 16 + i] = s;
  }
}

typedef double far4 __attribute__((ext_vector_type(4)));

// Sums of 64 directions over the segments of one chunk of waves:
// part[(chunk * 6 NR + value) * nslots + slot]. Wave w of chunk b takes segments
// wave_seg[w] .. wave_seg[w + 1], w = 8 b + wave; their records are a stream,
// read three steps ahead. Four tiles of 16 directions share each record; their
// cos and sin come from LDS (LDSX) or, for boxes too long for it, from L2.
// Records: those of positions pos0 .. pos0 + npos - 1 (where the launch's chunks
// lie) of right-hand side rhs[tile] - r0, or (rhs null) of the only one.
template <int NR, bool LDSX>
__global__ __launch_bounds__(64 * kFarWaves) void k_far_rows(const double* __restrict__ rec, int pos0, int npos,
                                                             const FarSeg* __restrict__ segs,
                                                             const int2* __restrict__ wave_seg,
                                                             const double* __restrict__ cs,
                                                             const double2* __restrict__ yz, int nu, int By, int nslots,
                                                             const int* __restrict__ rhs, int r0,
                                                             double* __restrict__ part) {
  extern __shared__ __align__(16) char smem[];
  const int lane = threadIdx.x & 63, g = lane >> 4, j = lane & 15;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const double* ct = cs + (long long)blockIdx.x * nu * 128;
  if (LDSX) {
    double2* t = reinterpret_cast<double2*>(smem);
    for (int i = threadIdx.x; i < nu * 64; i += 64 * kFarWaves) t[i] = reinterpret_cast<const double2*>(ct)[i];
    __syncthreads();
    ct = reinterpret_cast<const double*>(smem);
  }
  // instruction operand k = g: position g / 2 of the step, cos or sin
  ct += (g >> 1) * 128 + (g & 1) * 16 + j;
  if (rhs) rec += (long long)(rhs[blockIdx.x] - r0) * npos * 32;
  const int2 ws = wave_seg[blockIdx.y * kFarWaves + wave], we = wave_seg[blockIdx.y * kFarWaves + wave + 1];
  const double* r = rec + (long long)(ws.y - pos0) * 32 + lane;
  double acc_r[4][NR], acc_i[4][NR];
#pragma unroll
  for (int t = 0; t < 4; t++)
#pragma unroll
    for (int h = 0; h < NR; h++) acc_r[t][h] = acc_i[t][h] = 0;
  double a0 = r[0], a1 = r[64], a2 = r[128];
  for (int q = ws.x; q < we.x; q++) {
    const FarSeg sg = segs[q];
    const double* b = ct + sg.u0 * 128;
    far4 T[4];
#pragma unroll
    for (int t = 0; t < 4; t++) T[t] = (far4)(0.0);
    for (int s = 0; s < sg.steps; s++, b += 256) {
      const double a = a0;
      a0 = a1;
      a1 = a2;
      r += 64;
      a2 = r[128];
#pragma unroll
      for (int t = 0; t < 4; t++) T[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(a, b[t * 32], T[t], 0, 0, 0);
    }
    const double2* py = yz + (long long)sg.y * nslots + blockIdx.x * 64 + j;
    const double2* pz = yz + (long long)(By + sg.z) * nslots + blockIdx.x * 64 + j;
#pragma unroll
    for (int t = 0; t < 4; t++) {
      const double2 w = cmul(py[t * 16], pz[t * 16]);
#pragma unroll
      for (int h = 0; h < NR; h++) {
        acc_r[t][h] = ffma(T[t][2 * h], w.x, ffma(-T[t][2 * h + 1], w.y, acc_r[t][h]));
        acc_i[t][h] = ffma(T[t][2 * h], w.y, ffma(T[t][2 * h + 1], w.x, acc_i[t][h]));
      }
    }
  }
  // the waves' sums, in their order
  constexpr int NV = 6 * NR;
  double* red = reinterpret_cast<double*>(smem);
  __syncthreads();
#pragma unroll
  for (int h = 0; h < NR; h++)
    if (4 * h + g < 3 * NR)
#pragma unroll
      for (int t = 0; t < 4; t++) {
        double* d = red + (wave * NV + 2 * (4 * h + g)) * 64 + t * 16 + j;
        d[0] = acc_r[t][h];
        d[64] = acc_i[t][h];
      }
  __syncthreads();
  for (int v = wave; v < NV; v += kFarWaves) {
    double t = 0;
    for (int w = 0; w < kFarWaves; w++) t += red[(w * NV + v) * 64 + lane];
    part[((long long)blockIdx.y * NV + v) * nslots + blockIdx.x * 64 + lane] = t;
  }
}

// Last stage, 64 slots per work-group of 64 * 6 NR threads: the chunks' sums in
// their order, then E = i k^2 (S - n (n . S)) of each slot: to out[6 * query]
// (query: the slots' places, -1 for none), or on the angle grid the Jones
// matrices of the two evaluations of each angle, out[8 * angle].
template <int NR>
__global__ __launch_bounds__(384 * NR) void k_far_last(const double* __restrict__ part, FarDirs f, int slot0,
                                                       int nslots, int nchunk, double k, const int* __restrict__ query,
                                                       double* __restrict__ out) {
  constexpr int NV = 6 * NR;
  __shared__ double sh[NV][64];
  const int lane = threadIdx.x & 63, v = threadIdx.x >> 6;
  const int s = blockIdx.x * 64 + lane;
  double t = 0;
  for (int b = 0; b < nchunk; b++) t += part[((long long)b * NV + v) * nslots + s];
  sh[v][lane] = t;
  __syncthreads();
  const int slot = slot0 + s;
  if (v != 0 || slot >= f.count) return;
  // field of right-hand side r of lane l in direction n
  auto field = [&](int r, int l, const double n[3], double e[6]) {
    double nr = 0, ni = 0;
    for (int a = 0; a < 3; a++) {
      nr += n[a] * sh[6 * r + 2 * a][l];
      ni += n[a] * sh[6 * r + 2 * a + 1][l];
    }
    for (int a = 0; a < 3; a++) {
      e[2 * a] = -k * k * (sh[6 * r + 2 * a + 1][l] - n[a] * ni);
      e[2 * a + 1] = k * k * (sh[6 * r + 2 * a][l] - n[a] * nr);
    }
  };
  double n[3], e[6];
  if (f.dirs) {
    if (query[slot] < 0) return;
    far_direction(f, slot, n);
    field(0, lane, n, e);
    for (int a = 0; a < 6; a++) out[6ll * query[slot] + a] = e[a];
    return;
  }
  if (f.g.symmetric && (lane & 1)) return;
  const int i = f.g.symmetric ? slot >> 1 : slot;
  double2 perp[2], par[2];
  for (int q = 0; q < 2; q++) {
    double pe[3], pa[3];
    jones_frame(f.g, i, q, n, pe, pa);
    field(NR == 2 ? q : 0, NR == 2 ? lane : lane + q, n, e);
    perp[q] = par[q] = make_double2(0, 0);
    for (int a = 0; a < 3; a++) {
      perp[q].x += e[2 * a] * pe[a];
      perp[q].y += e[2 * a + 1] * pe[a];
      par[q].x += e[2 * a] * pa[a];
      par[q].y += e[2 * a + 1] * pa[a];
    }
  }
  const double sp = f.g.trig[2 * (f.g.ntheta + i % f.g.nphi)], cp = f.g.trig[2 * (f.g.ntheta + i % f.g.nphi) + 1];
  const double2 J[4] = {cadd(cscale(par[1], cp), cscale(par[0], sp)), csub(cscale(par[1], sp), cscale(par[0], cp)),
                        cadd(cscale(perp[1], cp), cscale(perp[0], sp)),
                        csub(cscale(perp[1], sp), cscale(perp[0], cp))};
  for (int j = 0; j < 4; j++) {
    out[8ll * i + 2 * j] = J[j].x;
    out[8ll * i + 2 * j + 1] = J[j].y;
  }
}

Frame frame_of(const dda_op_s* op) {
  const MvDims& d = op->dims;
  Frame f;
  f.d = op->grid_unit;
  f.ox = -(d.Bx - 1) / 2.0 * f.d;
  f.oy = -(d.By - 1) / 2.0 * f.d;
  f.oz = -(d.Bz - 1) / 2.0 * f.d;
  return f;
}

// Device copy of the dipole positions, made on first use.
dda_status positions_on_device(dda_op_s* op) {
  if (op->pos_dev) return DDA_OK;
  const size_t b = op->pos.size() * sizeof(uint32_t);
  DDA_TRY_HIP(dev_malloc(&op->pos_dev, b));
  op->device_bytes += b;
  DDA_TRY_HIP(hipMemcpyAsync(op->pos_dev, op->pos.data(), b, hipMemcpyHostToDevice, op->ctx->stream));
  DDA_TRY_HIP(hipStreamSynchronize(op->ctx->stream));
  return DDA_OK;
}

// Device scratch of at least `bytes`, kept by the operator between calls (a
// hipMalloc of some megabytes takes 300 us: the context's spare buffers serve a
// new operator's first call).
dda_status obs_scratch(dda_op_s* op, size_t bytes, void** out) {
  if (op->obs_held.got < bytes) {
    if (op->obs_scratch) {
      DDA_TRY_HIP(hipStreamSynchronize(op->ctx->stream));
      ctx_free(op->ctx, op->obs_scratch, op->obs_held);
      op->device_bytes -= op->obs_held.got;
      op->obs_scratch = nullptr;
      op->obs_held = Held();
    }
    Held h;
    DDA_TRY_HIP(ctx_alloc(op->ctx, &op->obs_scratch, bytes, &h));
    op->obs_held = h;
    op->device_bytes += h.got;
  }
  *out = op->obs_scratch;
  return DDA_OK;
}

// ------------------------------------------------------------------------------------
// The operator's positions as k_far_rows takes them, made on first use: the
// folded halves of the occupied rows, each from its innermost to its outermost
// dipole, in segments of at most 32 steps, dealt to the waves in equal numbers of
// steps. Formed on the device from the cell map (or the run-time planned X passes'
// row lists), one wave per row, and four launches and one wait in all: on the host
// (a copy of the positions and two passes over them) the first call on an
// operator of 33,552 dipoles took 470 us more than later ones, of 8.8 million
// 61 ms, which is more than many calls take altogether.
// ------------------------------------------------------------------------------------

// Positions of which the records of one right-hand side take 256 MB.
constexpr int kFarGroup = 1 << 20;

// Chunks for npos positions: 64 steps a wave, at most 64 work-groups' worth of
// waves in each group of positions.
__host__ __device__ inline int far_groups(int npos) { return (npos + kFarGroup - 1) / kFarGroup; }
__host__ __device__ inline int far_chunks(int npos) {
  const int per = 128 * kFarWaves, n = (npos + per - 1) / per, g = far_groups(npos);
  return g > 1 ? 64 * g : n < 64 ? n : 64;
}

// What the plan's kernels share. rows: [nocc] inner and outer fold of each
// occupied row; first: [nocc + 1] its first position and segment; info: positions
// (-1: too many holes), segments, and whether two dipoles share a position.
struct FarMake {
  const uint32_t *row_list, *cell, *row_start, *row_dip, *row_meta;
  int nocc, Bx, By;
  long long most;  // positions
  int2 *rows, *first, *pair, *wave_seg;
  FarSeg* segs;
  int* info;
};

// x of the dipoles at +u (side 0) and -u of a row's centre; fold is the way back.
__device__ inline int far_x(int Bx, int u, int side) { return side ? (Bx - 1) / 2 - u : Bx / 2 + u; }
__device__ inline int far_fold(int Bx, int x) { return abs(2 * x - (Bx - 1)) / 2; }

__global__ __launch_bounds__(256) void k_far_extent(FarMake m) {
  const int i = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (i == 0 && lane < 3) m.info[lane] = 0;
  if (i >= m.nocc) return;
  const uint32_t row = m.row_list[i];
  int lo = m.Bx, hi = -1;
  if (m.cell) {
    const uint32_t* c = m.cell + (size_t)row * m.Bx;
    for (int x = lane; x < m.Bx; x += 64)
      if ((int)c[x] >= 0) {
        const int u = far_fold(m.Bx, x);
        lo = min(lo, u);
        hi = max(hi, u);
      }
  } else {
    for (uint32_t k = m.row_start[row] + lane; k < m.row_start[row + 1]; k += 64) {
      const int u = far_fold(m.Bx, m.row_meta[k] & 0xffff);
      lo = min(lo, u);
      hi = max(hi, u);
    }
  }
  for (int o = 32; o > 0; o >>= 1) {
    lo = min(lo, __shfl_xor(lo, o, 64));
    hi = max(hi, __shfl_xor(hi, o, 64));
  }
  if (lane == 0) m.rows[i] = make_int2(lo, hi);
}

// One work-group: the rows' first positions (an even number each) and segments.
__global__ __launch_bounds__(1024) void k_far_scan(FarMake m) {
  __shared__ long long wp[16];
  __shared__ int ws[16];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  long long pos0 = 0;
  int seg0 = 0;
  for (int i0 = 0; i0 < m.nocc; i0 += 1024) {
    const int i = i0 + threadIdx.x;
    int n = 0;
    if (i < m.nocc) n = m.rows[i].y - m.rows[i].x + 1;
    const int np = (n + 1) & ~1, ns = (n + 63) / 64;
    long long p = np;
    int s = ns;
    for (int o = 1; o < 64; o <<= 1) {
      const long long pp = __shfl_up(p, o, 64);
      const int ss = __shfl_up(s, o, 64);
      if (lane >= o) {
        p += pp;
        s += ss;
      }
    }
    if (lane == 63) {
      wp[wave] = p;
      ws[wave] = s;
    }
    __syncthreads();
    long long pb = pos0;
    int sb = seg0;
    for (int w = 0; w < 16; w++) {
      if (w < wave) {
        pb += wp[w];
        sb += ws[w];
      }
      pos0 += wp[w];
      seg0 += ws[w];
    }
    if (i < m.nocc) m.first[i] = make_int2((int)(pb + p - np), sb + s - ns);
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    m.first[m.nocc] = make_int2((int)pos0, seg0);
    m.info[0] = pos0 > m.most ? -1 : (int)pos0;
    m.info[1] = seg0;
  }
}

// Segments and pairs of each row; the last work-group: where each wave starts,
// the first segment that ends at or after its share of the steps.
__global__ __launch_bounds__(256) void k_far_fill(FarMake m) {
  const int npos = m.info[0];
  if (npos < 0) return;
  if (blockIdx.x == gridDim.x - 1) {
    const long long steps = npos / 2;
    const int nw = far_chunks(npos) * kFarWaves;
    for (int w = threadIdx.x; w <= nw; w += 256) {
      const long long t = steps * w / nw;
      // the row i in which step t lies: it starts before t (row 0: t = 0)
      int a = 0, b = m.nocc;
      while (b - a > 1) {
        const int c = (a + b) / 2;
        (m.first[c].x / 2 < t ? a : b) = c;
      }
      const int2 f = m.first[a], e = m.first[a + 1];
      const int j = (int)((t - f.x / 2 + 31) / 32);
      m.wave_seg[w] = make_int2(f.y + j, min(f.x + 64 * j, e.x));
    }
    return;
  }
  const int i = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (i >= m.nocc) return;
  const uint32_t row = m.row_list[i];
  const int lo = m.rows[i].x, hi = m.rows[i].y;
  const int2 f = m.first[i], e = m.first[i + 1];
  for (int q = f.y + lane; q < e.y; q += 64) {
    const int u = lo + 64 * (q - f.y);
    m.segs[q] = {u, min(32, (hi - u + 2) / 2), (int)(row % m.By), (int)(row / m.By)};
  }
  if (m.cell) {
    const uint32_t* c = m.cell + (size_t)row * m.Bx;
    for (int p = lane; p < e.x - f.x; p += 64) {
      const int u = lo + p, xa = far_x(m.Bx, u, 0), xb = far_x(m.Bx, u, 1);
      m.pair[f.x + p] = make_int2(u <= hi && xa < m.Bx ? (int)c[xa] : -1, u <= hi && xb >= 0 && xb != xa ? (int)c[xb] : -1);
    }
    return;
  }
  for (int p = lane; p < e.x - f.x; p += 64) m.pair[f.x + p] = make_int2(-1, -1);
  __threadfence();  // before the row's own dipoles, which other lanes of the wave write
  for (uint32_t k = m.row_start[row] + lane; k < m.row_start[row + 1]; k += 64) {
    const int x = m.row_meta[k] & 0xffff, u = far_fold(m.Bx, x);
    int2* q = &m.pair[f.x + u - lo];
    if (atomicExch(x == far_x(m.Bx, u, 0) ? &q->x : &q->y, (int)m.row_dip[k]) >= 0) m.info[2] = 1;
  }
}

// far.npos stays 0 where the rows are mostly holes (four positions and more per
// dipole), two dipoles share a position or the memory cannot be had: those go by
// k_far_partial.
dda_status far_segments(dda_op_s* op) {
  dda_op_s::Far& far = op->far;
  if (far.made) return DDA_OK;
  const MvDims& d = op->dims;
  hipStream_t st = op->ctx->stream;
  const int nocc = op->n_nonempty, half = (d.Bx + 1) / 2;
  FarMake m;
  m.row_list = op->row_list;
  m.cell = op->cell;
  m.row_start = op->row_start;
  m.row_dip = op->row_dip;
  m.row_meta = op->row_meta;
  m.nocc = nocc;
  m.Bx = d.Bx;
  m.By = d.By;
  m.most = std::min<long long>(4ll * d.nv + 64, 1 << 26);
  const size_t npos = std::min<long long>(m.most, (long long)nocc * (half + 1));
  const size_t bytes[6] = {npos * sizeof(int2),
                           (size_t)nocc * ((half + 63) / 64) * sizeof(FarSeg),
                           (far_chunks((int)npos) * kFarWaves + 1ull) * sizeof(int2),
                           nocc * sizeof(int2), (nocc + 1ull) * sizeof(int2), 3 * sizeof(int)};
  size_t off[7] = {0};
  for (int i = 0; i < 6; i++) off[i + 1] = off[i] + (bytes[i] + 127) / 128 * 128;
  const hipError_t e = ctx_alloc(op->ctx, &op->far_dev, off[6], &op->far_held);
  if (e == hipErrorOutOfMemory) return DDA_OK;
  DDA_TRY_HIP(e);
  op->device_bytes += op->far_held.got;
  char* dev = (char*)op->far_dev;
  m.pair = (int2*)dev;
  m.segs = (FarSeg*)(dev + off[1]);
  m.wave_seg = (int2*)(dev + off[2]);
  m.rows = (int2*)(dev + off[3]);
  m.first = (int2*)(dev + off[4]);
  m.info = (int*)(dev + off[5]);
  const int nb = (nocc + 3) / 4;
  hipLaunchKernelGGL(k_far_extent, dim3(nb), dim3(256), 0, st, m);
  hipLaunchKernelGGL(k_far_scan, dim3(1), dim3(1024), 0, st, m);
  hipLaunchKernelGGL(k_far_fill, dim3(nb + 1), dim3(256), 0, st, m);
  int info[3] = {-1, 0, 0};
  hipError_t le = hipGetLastError();
  if (le == hipSuccess) le = hipMemcpyAsync(info, m.info, sizeof info, hipMemcpyDeviceToHost, st);
  const hipError_t se = hipStreamSynchronize(st);
  if (le == hipSuccess) le = se;
  if (le == hipSuccess && info[0] > 0 && !info[2] && far_groups(info[0]) > 1) {
    far.start.resize(far_chunks(info[0]) * kFarWaves + 1);
    le = hipMemcpyAsync(far.start.data(), m.wave_seg, far.start.size() * sizeof(int2), hipMemcpyDeviceToHost, st);
    if (le == hipSuccess) le = hipStreamSynchronize(st);
  }
  if (le != hipSuccess || info[0] <= 0 || info[2]) {
    ctx_free(op->ctx, op->far_dev, op->far_held);
    op->device_bytes -= op->far_held.got;
    op->far_dev = nullptr;
    far.made = le == hipSuccess;
    DDA_TRY_HIP(le);
    return DDA_OK;
  }
  far.made = true;
  far.segs = m.segs;
  far.wave_seg = m.wave_seg;
  far.nchunk = far_chunks(info[0]);
  far.npos = info[0];
  return DDA_OK;
}

// Work space of far_batches: the batches' tables, partial sums and records,
// each batch's tables and sums and its records below 256 MB. The records of more
// than kFarGroup positions are made and used group by group.
struct FarPlan {
  int nu;         // positions of the folded x axis, one more for the step's second
  int per_batch;  // slots per batch, a multiple of 64
  int groups;     // of positions
  int recs;       // right-hand sides (NR = 2: pairs) per batch
  size_t cs, yz, parts, bytes;
};
// First position of a group's records, and the end of the last's.
int group_start(const dda_op_s::Far& far, int groups, int g) {
  return groups == 1 ? g * far.npos : far.start[(size_t)g * (far.nchunk / groups) * kFarWaves].y;
}
FarPlan far_plan(const dda_op_s* op, int slots, int nr, int nrec) {
  const MvDims& d = op->dims;
  const size_t most = 256ull << 20;
  FarPlan p;
  p.nu = (d.Bx + 1) / 2 + 1;
  const size_t cs = 16ull * p.nu, yz = 16ull * (d.By + d.Bz), part = 48ull * nr * op->far.nchunk;
  p.groups = far_groups(op->far.npos);
  int npos = 0;
  for (int g = 0; g < p.groups; g++)
    npos = std::max(npos, group_start(op->far, p.groups, g + 1) - group_start(op->far, p.groups, g));
  const size_t rec = 256ull * npos;
  p.per_batch = (int)std::min<size_t>(std::max<size_t>(1, most / (64 * (cs + yz + part))), (slots + 63) / 64) * 64;
  p.recs = p.groups > 1 ? 1 : (int)std::min<size_t>(std::max<size_t>(1, most / rec), std::min(nrec, 65535));
  p.cs = cs * p.per_batch;
  p.yz = yz * p.per_batch;
  p.parts = part * p.per_batch;
  p.bytes = p.cs + p.yz + p.parts + rec * p.recs + 3 * 512;  // read ahead
  return p;
}

// The sums and last stages of the slots of f, in batches. rhs: the right-hand
// side of each 64 slots, ascending, on the host and on the device (null: all of
// record 0); query (device, one per slot) as k_far_last takes it; out_dev on the
// device.
template <int NR>
dda_status far_batches(dda_op_s* op, const double2* pol, const FarDirs& f, const FarPlan& p, const int* rhs_host,
                       const int* rhs, const int* query, double* out_dev, void* work) {
  const MvDims& d = op->dims;
  const dda_op_s::Far& far = op->far;
  hipStream_t st = op->ctx->stream;
  double* cs = (double*)work;
  double2* yz = (double2*)((char*)work + p.cs);
  double* part = (double*)((char*)yz + p.yz);
  double* rec = (double*)((char*)part + p.parts);
  const size_t red = sizeof(double) * kFarWaves * 6 * NR * 64, xt = 1024ull * p.nu;
  const bool ldsx = xt <= 150 * 1024;
  const size_t lds = ldsx ? std::max(red, xt) : red;
  auto k = ldsx ? k_far_rows<NR, true> : k_far_rows<NR, false>;
  if (lds > 64 * 1024)
    DDA_TRY_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(k), hipFuncAttributeMaxDynamicSharedMemorySize,
                                    (int)lds));
  const int tiles = (f.count + 63) / 64;
  int have0 = 0, have1 = 0;  // right-hand sides whose records are there
  for (int t0 = 0, t1; t0 < tiles; t0 = t1) {
    const int r0 = rhs_host ? rhs_host[t0] : 0;
    for (t1 = t0; t1 < tiles && (t1 - t0) * 64 < p.per_batch && (rhs_host ? rhs_host[t1] : 0) < r0 + p.recs;) t1++;
    const int r1 = (rhs_host ? rhs_host[t1 - 1] : 0) + 1;
    const int s0 = t0 * 64, ns = (t1 - t0) * 64;
    hipLaunchKernelGGL(k_far_tables, dim3(t1 - t0, std::min(p.nu + d.By + d.Bz, 64)), dim3(64), 0, st, f, s0, ns, p.nu,
                       d.Bx & 1 ? 0.0 : 0.5, d.By, d.Bz, op->wave_num * op->grid_unit, cs, yz);
    const int chunks = far.nchunk / p.groups;
    for (int gr = 0; gr < p.groups; gr++) {
      const int pos0 = group_start(far, p.groups, gr), np = group_start(far, p.groups, gr + 1) - pos0;
      if (p.groups > 1 || r0 < have0 || r1 > have1) {
        have0 = r0;
        have1 = r1;
        hipLaunchKernelGGL(k_far_pack<NR>, dim3(std::min(1024, (16 * np + 255) / 256), r1 - r0), dim3(256), 0, st,
                           pol + (size_t)r0 * 3 * NR * d.S, (const int2*)op->far_dev + pos0, np, d.S, rec);
      }
      hipLaunchKernelGGL(k, dim3(t1 - t0, chunks), dim3(64 * kFarWaves), lds, st, rec, pos0, np,
                         (const FarSeg*)far.segs, (const int2*)far.wave_seg + (size_t)gr * chunks * kFarWaves, cs, yz,
                         p.nu, d.By, ns, rhs ? rhs + t0 : nullptr, have0,
                         part + (size_t)gr * chunks * 6 * NR * ns);
    }
    hipLaunchKernelGGL(k_far_last<NR>, dim3(t1 - t0), dim3(384 * NR), 0, st, part, f, s0, ns, far.nchunk, op->wave_num,
                       query, out_dev);
    DDA_TRY_HIP(hipGetLastError());
  }
  return DDA_OK;
}

// Whether nq field evaluations of `used` right-hand sides go by k_far_rows. Its
// launches and tables cost what some hundred evaluations by k_far_partial do, the
// records of a right-hand side and 64 directions what 38 do in large particles.
// The two, on an operator that has made the segments and on a new one (whose first
// call of k_far_partial is that much longer too), in us:
//   33,552 dipoles, 256 evaluations        83 and 121   against  90 and  97
//   217,160 dipoles, 48                   116 and 160   against 116 and 121
//   1,099,136 dipoles, 16, 48 and 64      311, 310 and 312   against 198, 339 and 407
//   8,783,848 dipoles, 32, 48 and 256     2,783, 2,789 and 2,598   against 2,411, 3,160
//                                         and 11,907; new, 256: 3,015 against 12,876
// so the line lies at 8 million dipole phases and 48 evaluations of each
// right-hand side. An angle grid's directions and Jones matrices are formed on the
// device too, which pays from 1,000 evaluations on at any size (11,102 of 280
// dipoles: 72 against 426 us). k_far_partial's grid has no room for more than
// kFarDirect.
constexpr int kFarDirect = 4 * 65535;
bool many_directions(const dda_op_s* op, bool angle_grid, long long nq, int used) {
  return nq > kFarDirect || (angle_grid && nq >= 1000) ||
         ((double)nq * op->dims.nv >= 8e6 && nq >= 48ll * used);
}

// Scratch for k_far_rows and what is beside it: DDA_NOT_SUPPORTED where it cannot
// be had, and k_far_partial, which needs less, has to do.
dda_status far_scratch(dda_op_s* op, size_t bytes, void** out) {
  const dda_status rc = obs_scratch(op, bytes, out);
  return rc == DDA_OUT_OF_MEMORY ? DDA_NOT_SUPPORTED : rc;
}

// dda_far_field of many directions; DDA_NOT_SUPPORTED where k_far_partial takes them.
dda_status far_field_many(dda_op_s* op, const double2* pol, int nrhs, const int* rhs, const double* dirs, int nq,
                          double* out) {
  // slots by right-hand side, each's filled up to 64
  std::vector<int> fill(nrhs + 1, 0);
  for (int i = 0; i < nq; i++) fill[(rhs ? rhs[i] : 0) + 1]++;
  long long slots = 0;
  int used = 0;
  for (int r = 0; r < nrhs; r++) {
    const int n = fill[r + 1];
    fill[r] = (int)slots;
    slots += (n + 63) / 64 * 64;
    used += n > 0;
  }
  if (!many_directions(op, false, nq, used) || slots >= (1ll << 30)) return DDA_NOT_SUPPORTED;
  DDA_TRY(far_segments(op));
  if (op->far.npos == 0) return DDA_NOT_SUPPORTED;
  const FarPlan plan = far_plan(op, (int)slots, 1, nrhs);
  const size_t dbytes = 3ull * slots * sizeof(double), ibytes = (slots + slots / 64 + 3) / 4 * 16;
  void* buf = nullptr;
  DDA_TRY(far_scratch(op, plan.bytes + dbytes + ibytes + 6ull * nq * sizeof(double), &buf));
  std::vector<double> hd(3 * slots, 0.0);
  std::vector<int> hi(slots + slots / 64, -1);
  for (int i = 0; i < nq; i++) {
    const int r = rhs ? rhs[i] : 0, s = fill[r]++;
    for (int a = 0; a < 3; a++) hd[dir_index(s, a)] = dirs[dir_index(i, a)];
    hi[s] = i;
    hi[slots + s / 64] = r;
  }
  for (long long t = 0; t < slots / 64; t++) hi[slots + t] = std::max(0, hi[slots + t]);
  double* dd = (double*)((char*)buf + plan.bytes);
  int* id = (int*)((char*)dd + dbytes);
  double* od = (double*)((char*)id + ibytes);
  hipStream_t st = op->ctx->stream;
  DDA_TRY_HIP(hipMemcpyAsync(dd, hd.data(), dbytes, hipMemcpyHostToDevice, st));
  DDA_TRY_HIP(hipMemcpyAsync(id, hi.data(), hi.size() * sizeof(int), hipMemcpyHostToDevice, st));
  FarDirs f;
  std::memset(&f, 0, sizeof f);
  f.dirs = dd;
  f.count = (int)slots;
  DDA_TRY(far_batches<1>(op, pol, f, plan, hi.data() + slots, id + slots, id, od, buf));
  DDA_TRY_HIP(hipMemcpyAsync(out, od, 6ull * nq * sizeof(double), hipMemcpyDeviceToHost, st));
  DDA_TRY_HIP(hipStreamSynchronize(st));
  return DDA_OK;
}

// dda_jones of many angles; DDA_NOT_SUPPORTED where dda_far_field takes them.
dda_status jones_many(dda_op_s* op, const double2* pol, int symmetric, const double prop[3], const double pol1[3],
                      const double pol2[3], uint32_t ntheta, double theta0, double dtheta, uint32_t nphi, double phi0,
                      double dphi, double* out) {
  const size_t count = (size_t)ntheta * nphi, slots = symmetric ? 2 * count : count;
  if (!many_directions(op, true, 2 * (long long)count, 1) || slots >= (1ll << 30)) return DDA_NOT_SUPPORTED;
  DDA_TRY(far_segments(op));
  if (op->far.npos == 0) return DDA_NOT_SUPPORTED;
  const FarPlan plan = far_plan(op, (int)slots, symmetric ? 1 : 2, 1);
  const size_t tbytes = 2 * ((size_t)ntheta + nphi) * sizeof(double);
  void* buf = nullptr;
  DDA_TRY(far_scratch(op, plan.bytes + tbytes + 8 * count * sizeof(double), &buf));
  std::vector<double> trig(2 * ((size_t)ntheta + nphi));
  for (size_t i = 0; i < (size_t)ntheta + nphi; i++) {
    const double a = i < ntheta ? theta0 + (double)i * dtheta : phi0 + (double)(i - ntheta) * dphi;
    trig[2 * i] = std::sin(a);
    trig[2 * i + 1] = std::cos(a);
  }
  double* td = (double*)((char*)buf + plan.bytes);
  double* od = (double*)((char*)td + tbytes);
  hipStream_t st = op->ctx->stream;
  DDA_TRY_HIP(hipMemcpyAsync(td, trig.data(), tbytes, hipMemcpyHostToDevice, st));
  FarDirs f;
  std::memset(&f, 0, sizeof f);
  f.g.trig = td;
  f.g.ntheta = (int)ntheta;
  f.g.nphi = (int)nphi;
  f.g.symmetric = symmetric;
  for (int a = 0; a < 3; a++) {
    f.g.prop[a] = prop[a];
    f.g.pol1[a] = pol1[a];
    f.g.pol2[a] = pol2[a];
  }
  f.count = (int)slots;
  DDA_TRY(symmetric ? far_batches<1>(op, pol, f, plan, nullptr, nullptr, nullptr, od, buf)
                    : far_batches<2>(op, pol, f, plan, nullptr, nullptr, nullptr, od, buf));
  DDA_TRY_HIP(hipMemcpyAsync(out, od, 8 * count * sizeof(double), hipMemcpyDeviceToHost, st));
  DDA_TRY_HIP(hipStreamSynchronize(st));
  return DDA_OK;
}

}  // namespace

// Device addresses of `scratch`, one per device, taken once per device with
// that device current (dda_ctx_create calls this after hipSetDevice).
static std::mutex g_noalloc_mu;
static double* g_noalloc_ptr[kMaxNoAllocDevices] = {};

dda_status noalloc_scratch_setup(int device) {
  if (device < 0 || device >= kMaxNoAllocDevices) {
    set_error("noalloc scratch: device index out of range");
    return DDA_INVALID_ARG;
  }
  std::lock_guard<std::mutex> lk(g_noalloc_mu);
  if (g_noalloc_ptr[device]) return DDA_OK;
  void* p = nullptr;
  const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
  if (e != hipSuccess || !p) {
    set_error(std::string("hipGetSymbolAddress(scratch) failed: ") + hipGetErrorString(e));
    return DDA_HIP_ERROR;
  }
  g_noalloc_ptr[device] = static_cast<double*>(p);
  return DDA_OK;
}

static double* noalloc_scratch(int device) {
  if (device < 0 || device >= kMaxNoAllocDevices) return nullptr;
  std::lock_guard<std::mutex> lk(g_noalloc_mu);
  return g_noalloc_ptr[device];
}

}  // namespace dda

using namespace dda;

// Alpha and sqrt(alpha) of material i, axis c, for the refractive index
// m[(i * mstride + c * cstride)] (complex): CM or LDR (with S from prop and
// pol, or the polarisation average).
static dda_status couple_constants_impl(const char* fn, int kind, uint32_t nmat, const double* m, int mstride,
                                        int cstride, double grid_unit, double kd, const double prop[3],
                                        const double pol[3], double* cc, double* cc_sqrt) {
  if (!m || !prop || !pol || !cc || nmat == 0 || kind < 0 || kind > 2 || !(grid_unit > 0) || !(kd > 0)) {
    set_error(std::string(fn) + ": null argument, nmat 0, unknown kind, or grid_unit / kd <= 0");
    return DDA_INVALID_ARG;
  }
  typedef std::complex<double> Cd;
  const double b1 = 1.8915316, b2 = -0.1648469, b3 = 1.7700004;  // FPConst.hpp:48-50 (doi:10.1086/172396)
  const double vol = grid_unit * grid_unit * grid_unit;
  double S = 0;
  if (kind == DDA_POL_LDR)
    for (int a = 0; a < 3; a++) S += prop[a] * prop[a] * pol[a] * pol[a];
  else if (kind == DDA_POL_LDR_AVGPOL) {
    double p4 = 0;
    for (int a = 0; a < 3; a++) p4 += prop[a] * prop[a] * prop[a] * prop[a];
    S = 0.5 * (1 - p4);
  }
  for (uint32_t i = 0; i < nmat; i++)
    for (int c = 0; c < 3; c++) {
      const double* mi = m + 2 * ((size_t)i * mstride + (size_t)c * cstride);
      const Cd mm(mi[0], mi[1]), m2 = mm * mm;
      const Cd cm = 3 * vol / (4 * kPi) * (m2 - 1.0) / (m2 + 2.0);
      Cd a = cm;
      if (kind != DDA_POL_CM) {
        const Cd t1 = (b1 + (b2 + b3 * S) * m2) * kd * kd + Cd(0, 2.0 / 3.0 * kd * kd * kd);
        a = cm / (1.0 - (cm / vol) * t1);
      }
      cc[2 * (3 * i + c)] = a.real();
      cc[2 * (3 * i + c) + 1] = a.imag();
      if (cc_sqrt) {
        const Cd sq = std::sqrt(a);
        cc_sqrt[2 * (3 * i + c)] = sq.real();
        cc_sqrt[2 * (3 * i + c) + 1] = sq.imag();
      }
    }
  return DDA_OK;
}

extern "C" dda_status dda_couple_constants(int kind, uint32_t nmat, const double* m, double grid_unit, double kd,
                                           const double prop[3], const double pol[3], double* cc, double* cc_sqrt) {
  return couple_constants_impl("dda_couple_constants", kind, nmat, m, 1, 0, grid_unit, kd, prop, pol, cc,
                               cc_sqrt);
}

extern "C" dda_status dda_couple_constants_diag(int kind, uint32_t nmat, const double* m, double grid_unit,
                                                double kd, const double prop[3], const double pol[3], double* cc,
                                                double* cc_sqrt) {
  return couple_constants_impl("dda_couple_constants_diag", kind, nmat, m, 3, 1, grid_unit, kd, prop, pol, cc,
                               cc_sqrt);
}

// Observables scale by the operator's wave number: a pack qualifies only when
// its members share one.
static dda_status one_wave_number(const dda_op_s* op, const char* fn) {
  for (double w : op->pack.wave_num)
    if (w != op->wave_num) {
      set_error(std::string(fn) + ": a pack of members with different wave numbers");
      return DDA_NOT_SUPPORTED;
    }
  return DDA_OK;
}

extern "C" dda_status dda_incident_plane(dda_op_t op, int nrhs, const double* prop, const double* pol,
                                         void* einc_dev) {
  if (!op || nrhs < 1 || !prop || !pol || !einc_dev) {
    set_error("dda_incident_plane: null argument or nrhs < 1");
    return DDA_INVALID_ARG;
  }
  if (op->pack.nmember > 1) {
    set_error("dda_incident_plane: a pack (the field of member m is its own operator's, scattered by the pack map)");
    return DDA_NOT_SUPPORTED;
  }
  DDA_TRY(bind_device(op->ctx));
  DDA_TRY(positions_on_device(op));
  void* buf = nullptr;
  DDA_TRY(obs_scratch(op, 6ull * nrhs * sizeof(double), &buf));
  std::vector<double> h(6ull * nrhs);
  for (int r = 0; r < nrhs; r++)
    for (int a = 0; a < 3; a++) {
      h[6 * r + a] = prop[3 * r + a];
      h[6 * r + 3 + a] = pol[3 * r + a];
    }
  hipStream_t st = op->ctx->stream;
  DDA_TRY_HIP(hipMemcpyAsync(buf, h.data(), h.size() * sizeof(double), hipMemcpyHostToDevice, st));
  const MvDims& d = op->dims;
  hipLaunchKernelGGL(k_incident, dim3(std::min(1024, (d.S + 255) / 256), nrhs), dim3(256), 0, st, (double2*)einc_dev,
                     (const uint32_t*)op->pos_dev, (const double*)buf, d.nv, d.S, op->wave_num, frame_of(op));
  DDA_TRY_HIP(hipGetLastError());
  DDA_TRY_HIP(hipStreamSynchronize(st));
  return DDA_OK;
}

extern "C" dda_status dda_cross_sections(dda_op_t op, const void* pol_dev, const void* einc_dev, int nrhs,
                                         const double* cc, double* cext, double* cabs) {
  if (!op || !pol_dev || nrhs < 1 || (cext && !einc_dev) || (cabs && !cc)) {
    set_error("dda_cross_sections: null argument or nrhs < 1");
    return DDA_INVALID_ARG;
  }
  DDA_TRY(one_wave_number(op, "dda_cross_sections"));
  DDA_TRY(bind_device(op->ctx));
  const MvDims& d = op->dims;
  const int nb = std::max(1, std::min(256, (d.nv + 4095) / 4096));
  const double k = op->wave_num;
  std::vector<double> mdr(3ull * op->nmat * nrhs, 0.0);
  if (cc)
    for (size_t i = 0; i < mdr.size(); i++) {
      const std::complex<double> a(cc[2 * i], cc[2 * i + 1]);
      mdr[i] = -(1.0 / a).imag() - 2.0 / 3.0 * k * k * k;
    }
  void* buf = nullptr;
  const size_t pbytes = 2ull * nb * nrhs * sizeof(double);
  DDA_TRY(obs_scratch(op, pbytes + mdr.size() * sizeof(double), &buf));
  double* part = (double*)buf;
  double* mdr_dev = part + 2ull * nb * nrhs;
  hipStream_t st = op->ctx->stream;
  DDA_TRY_HIP(hipMemcpyAsync(mdr_dev, mdr.data(), mdr.size() * sizeof(double), hipMemcpyHostToDevice, st));
  hipLaunchKernelGGL(k_cross, dim3(nb, nrhs), dim3(kObsThreads), 0, st, (const double2*)pol_dev,
                     (const double2*)(einc_dev ? einc_dev : pol_dev), (const uint8_t*)op->mat_dev, mdr_dev,
                     (const double2*)nullptr, 0.0, d.nv, d.S, (int)op->nmat, part, d.member);
  DDA_TRY_HIP(hipGetLastError());
  std::vector<double> h(2ull * nb * nrhs);
  DDA_TRY_HIP(hipMemcpyAsync(h.data(), part, h.size() * sizeof(double), hipMemcpyDeviceToHost, st));
  DDA_TRY_HIP(hipStreamSynchronize(st));
  for (int r = 0; r < nrhs; r++) {
    double se = 0, sa = 0;
    for (int b = 0; b < nb; b++) {
      se += h[(r * (size_t)nb + b) * 2];
      sa += h[(r * (size_t)nb + b) * 2 + 1];
    }
    if (cext) cext[r] = 4 * kPi * k * se;
    if (cabs) cabs[r] = 4 * kPi * k * sa;
  }
  return DDA_OK;
}

// dda_cross_sections without allocating: alpha, the partial sums and the
// finished sums go through the device's fixed `scratch` array (its address
// from noalloc_scratch_setup), the per-right-hand-side sums are finished on the
// device and copied straight into cext / cabs. No hipMalloc, hipFree or host
// heap allocation happens here. Every k_cross block writes its own partials,
// so nothing needs clearing between calls. Calls that overlap on one GPU share
// the array and race.
extern "C" dda_status dda_cross_sections_noalloc(dda_op_t op, const void* pol_dev, const void* einc_dev, int nrhs,
                                                 const double* cc, double* cext, double* cabs) {
  if (!op || !pol_dev || nrhs < 1 || (cext && !einc_dev) || (cabs && !cc)) {
    set_error("dda_cross_sections_noalloc: null argument or nrhs < 1");
    return DDA_INVALID_ARG;
  }
  DDA_TRY(one_wave_number(op, "dda_cross_sections_noalloc"));
  const MvDims& d = op->dims;
  const int nb = std::max(1, std::min(256, (d.nv + 4095) / 4096));
  const size_t ncc = cc ? 6ull * op->nmat * nrhs : 0;  // alpha, [nrhs][nmat][3] complex
  const size_t npart = 2ull * nb * nrhs, nout = 2ull * nrhs;
  if (ncc + npart + nout > (size_t)DDA_NOALLOC_SCRATCH_DOUBLES) {
    set_error("dda_cross_sections_noalloc: needs " + std::to_string(ncc + npart + nout) +
              " doubles of scratch (6 nmat nrhs + 2 nrhs (blocks + 1)), above the fixed " +
              std::to_string(DDA_NOALLOC_SCRATCH_DOUBLES));
    return DDA_INVALID_ARG;
  }
  DDA_TRY(bind_device(op->ctx));
  double* base = noalloc_scratch(op->ctx->device);
  if (!base) {
    set_error("dda_cross_sections_noalloc: the device scratch of this context's device was not set up");
    return DDA_HIP_ERROR;
  }
  double* ccd = base;
  double* part = base + ncc;
  double* fin = part + npart;
  const double k = op->wave_num;
  hipStream_t st = op->ctx->stream;
  if (cc) DDA_TRY_HIP(hipMemcpyAsync(ccd, cc, ncc * sizeof(double), hipMemcpyHostToDevice, st));
  hipLaunchKernelGGL(k_cross, dim3(nb, nrhs), dim3(kObsThreads), 0, st, (const double2*)pol_dev,
                     (const double2*)(einc_dev ? einc_dev : pol_dev), (const uint8_t*)op->mat_dev,
                     (const double*)nullptr, cc ? (const double2*)ccd : (const double2*)nullptr,
                     2.0 / 3.0 * k * k * k, d.nv, d.S, (int)op->nmat, part, d.member);
  hipLaunchKernelGGL(k_cross_final, dim3((nrhs + 255) / 256), dim3(256), 0, st, part, nb, nrhs, 4 * kPi * k, fin);
  DDA_TRY_HIP(hipGetLastError());
  if (cext) DDA_TRY_HIP(hipMemcpyAsync(cext, fin, nrhs * sizeof(double), hipMemcpyDeviceToHost, st));
  if (cabs) DDA_TRY_HIP(hipMemcpyAsync(cabs, fin + nrhs, nrhs * sizeof(double), hipMemcpyDeviceToHost, st));
  DDA_TRY_HIP(hipStreamSynchronize(st));
  return DDA_OK;
}

extern "C" dda_status dda_far_field(dda_op_t op, const void* pol_dev, int nrhs, const int* rhs, const double* dirs,
                                    int nq, double* out) {
  if (!op || !pol_dev || nrhs < 1 || !dirs || nq < 1 || !out) {
    set_error("dda_far_field: null argument, nrhs < 1 or no directions");
    return DDA_INVALID_ARG;
  }
  DDA_TRY(one_wave_number(op, "dda_far_field"));
  DDA_TRY(bind_device(op->ctx));
  for (int i = 0; i < nq; i++)
    if (rhs && (rhs[i] < 0 || rhs[i] >= nrhs)) {
      set_error("dda_far_field: right-hand side index out of range");
      return DDA_INVALID_ARG;
    }
  if (many_directions(op, false, nq, 1)) {
    const dda_status rc = far_field_many(op, (const double2*)pol_dev, nrhs, rhs, dirs, nq, out);
    if (rc != DDA_NOT_SUPPORTED) return rc;
  }
  DDA_TRY(positions_on_device(op));
  const MvDims& d = op->dims;
  const int chunk = 4096;
  const int nchunk = (d.nv + chunk - 1) / chunk;
  const size_t qbytes = 4ull * nq * sizeof(double), pbytes = 6ull * nchunk * nq * sizeof(double);
  const size_t obytes = 6ull * nq * sizeof(double);
  void* buf = nullptr;
  DDA_TRY(obs_scratch(op, qbytes + pbytes + obytes, &buf));
  double* qd = (double*)buf;
  double* part = qd + 4ull * nq;
  double* od = part + 6ull * nchunk * nq;
  std::vector<double> hq(4ull * nq);
  for (int i = 0; i < nq; i++) {
    hq[4ull * i] = rhs ? rhs[i] : 0;
    for (int a = 0; a < 3; a++) hq[4ull * i + 1 + a] = dirs[dir_index(i, a)];
  }
  hipStream_t st = op->ctx->stream;
  DDA_TRY_HIP(hipMemcpyAsync(qd, hq.data(), qbytes, hipMemcpyHostToDevice, st));
  hipLaunchKernelGGL(k_far_partial, dim3(nchunk, (nq + kQT - 1) / kQT), dim3(kObsThreads), 0, st,
                     (const double2*)pol_dev, (const uint32_t*)op->pos_dev, qd, nq, d.nv, d.S,
                     op->wave_num * op->grid_unit, chunk, part);
  hipLaunchKernelGGL(k_far_final, dim3((nq + 255) / 256), dim3(256), 0, st, part, qd, nq, nchunk, op->wave_num,
                     frame_of(op), od);
  DDA_TRY_HIP(hipGetLastError());
  DDA_TRY_HIP(hipMemcpyAsync(out, od, obytes, hipMemcpyDeviceToHost, st));
  DDA_TRY_HIP(hipStreamSynchronize(st));
  return DDA_OK;
}

extern "C" dda_status dda_jones(dda_op_t op, const void* pol_dev, int symmetric, const double prop[3],
                                const double pol1[3], const double pol2[3], uint32_t ntheta, double theta0,
                                double dtheta, uint32_t nphi, double phi0, double dphi, double* out) {
  if (!op || !pol_dev || !prop || !pol1 || !pol2 || !out || ntheta == 0 || nphi == 0) {
    set_error("dda_jones: null argument or empty angle grid");
    return DDA_INVALID_ARG;
  }
  DDA_TRY(one_wave_number(op, "dda_jones"));
  const size_t count = (size_t)ntheta * nphi;
  DDA_TRY(bind_device(op->ctx));
  {
    const dda_status rc = jones_many(op, (const double2*)pol_dev, symmetric, prop, pol1, pol2, ntheta, theta0, dtheta,
                                     nphi, phi0, dphi, out);
    if (rc != DDA_NOT_SUPPORTED) return rc;
  }
  // two field evaluations per angle: (p1; X = pol2, Y = pol1) and
  // (p2; X = pol2, Y = pol1) or, for a symmetric target, (p1; X = pol1, Y = -pol2)
  std::vector<double> dirs(6 * count), pe(12 * count), pa(12 * count);
  std::vector<int> rhs(2 * count);
  for (size_t i = 0; i < count; i++) {
    const double th = theta0 + (double)(i / nphi) * dtheta, ph = phi0 + (double)(i % nphi) * dphi;
    const double st = std::sin(th), ct = std::cos(th), sp = std::sin(ph), cp = std::cos(ph);
    for (int f = 0; f < 2; f++) {
      double X[3], Y[3];
      const bool rot = f == 1 && symmetric;
      for (int a = 0; a < 3; a++) {
        X[a] = rot ? pol1[a] : pol2[a];
        Y[a] = rot ? -pol2[a] : pol1[a];
      }
      const size_t qi = 2 * i + f;
      rhs[qi] = f == 1 && !symmetric ? 1 : 0;
      for (int a = 0; a < 3; a++) {
        dirs[3 * qi + a] = ct * prop[a] + st * (cp * X[a] + sp * Y[a]);
        pe[3 * qi + a] = sp * X[a] - cp * Y[a];
        pa[3 * qi + a] = -st * prop[a] + ct * (cp * X[a] + sp * Y[a]);
      }
    }
  }
  std::vector<double> e(12 * count);
  DDA_TRY(dda_far_field(op, pol_dev, symmetric ? 1 : 2, rhs.data(), dirs.data(), (int)(2 * count), e.data()));
  typedef std::complex<double> Cd;
  for (size_t i = 0; i < count; i++) {
    Cd perp[2], par[2];
    for (int f = 0; f < 2; f++) {
      const size_t qi = 2 * i + f;
      perp[f] = par[f] = 0;
      for (int a = 0; a < 3; a++) {
        const Cd v(e[6 * qi + 2 * a], e[6 * qi + 2 * a + 1]);
        perp[f] += v * pe[3 * qi + a];
        par[f] += v * pa[3 * qi + a];
      }
    }
    const double ph = phi0 + (double)(i % nphi) * dphi, sp = std::sin(ph), cp = std::cos(ph);
    const Cd J[4] = {cp * par[1] + sp * par[0], sp * par[1] - cp * par[0], cp * perp[1] + sp * perp[0],
                     sp * perp[1] - cp * perp[0]};
    for (int j = 0; j < 4; j++) {
      out[8 * i + 2 * j] = J[j].real();
      out[8 * i + 2 * j + 1] = J[j].imag();
    }
  }
  return DDA_OK;
}
