// Direct stream-function solver (iterate=0): PS/momentum.f90:172-653.
//
// build_SF_matrix assembles the banded operator of the whole grid (one row per
// node, Database 1 or 2 ordering, LDAB = 2 kl + ku + 1), scales its rows by
// DGBEQU's factors and factors it with partial pivoting (DGBTF2's column
// order, so the factors match the unblocked LAPACK routine bit for bit);
// solve_SF_equation forms the buoyancy vector, runs DGBTRS and scatters the
// solution into psi with its ghost images (Stream_grid).
//
// Device layout: AB column-major, A(p,q) at AB[(q-1)*LDAB + kl+ku+p-q]; the
// factorization walks the columns in panels, a wavefront per column; the solve
// is one workgroup whose band window lives in an LDS ring.
#include "pt_internal.hpp"

#include <algorithm>
#include <cstring>
#include <type_traits>

namespace pt {

// ---------------------------------------------------------------------------
// assembly
// ---------------------------------------------------------------------------
struct SfArgs {
  double D1[7], D2[7], D3[7], D4[7];                        // offsets -3..3
  double Drs[7][7], Drss[7][7], Drrs[7][7], Drrss[7][7];    // [k+3][i+3] = D?(i,k)
  double dr, ds, dr2, ds2, dr3, ds3, dr4, ds4, drds, drds2, dr2ds, dr2ds2;
  int nx, nz, Vbc, Database, kl, ku, n, pitch;              // pitch of the vis array (nx+7)
};

// pf / indices (PS/momentum.f90:221-253)
__device__ __forceinline__ int sf_pf(const SfArgs& a, int ip, int kp) {
  return a.Database == 1 ? (a.nx + 1) * kp + ip + 1 : (a.nz + 1) * ip + kp + 1;
}
__device__ __forceinline__ void sf_indices(const SfArgs& a, int p, int& ip, int& kp) {
  if (a.Database == 1) {
    const int N = a.nx + 1;
    ip = p - N * ((p - 1) / N) - 1; kp = (p - 1) / N;
  } else {
    const int N = a.nz + 1;
    kp = p - N * ((p - 1) / N) - 1; ip = (p - 1) / N;
  }
}

struct VisTerms {
  double vis, visx, visz, visxx, viszz, visxz;
};

// Matrix_element (PS/momentum.f90:507-606) for the stencil point (i,k) of row
// (ip,kp), with the uniform-grid metrics xr = zs = 1 and their derivatives 0
// kept in the expressions so that signs and roundings follow the reference;
// `m` is the band entry, updated in place
__device__ __forceinline__ void sf_element(const SfArgs& a, int i, int k, int ip, int kp, int rsym, int ssym,
                                           const VisTerms& v, double& m) {
  const double xr = 1.0, xrr = 0.0, xrrr = 0.0, xrrrr = 0.0, zs = 1.0, zss = 0.0, zsss = 0.0, zssss = 0.0;
  double Ss = 0.0, Sss = 0.0, Ssss = 0.0, Sssss = 0.0, Sr = 0.0, Srr = 0.0, Srrr = 0.0, Srrrr = 0.0;
  if (i == 0) {
    Ss = a.D1[k + 3] / a.ds; Sss = a.D2[k + 3] / a.ds2; Ssss = a.D3[k + 3] / a.ds3; Sssss = a.D4[k + 3] / a.ds4;
  }
  if (ssym == 1 && a.Vbc == 0) { Ss = -Ss; Sss = -Sss; Ssss = -Ssss; Sssss = -Sssss; }
  if (k == 0) {
    Sr = a.D1[i + 3] / a.dr; Srr = a.D2[i + 3] / a.dr2; Srrr = a.D3[i + 3] / a.dr3; Srrrr = a.D4[i + 3] / a.dr4;
  }
  if (rsym == 1) { Sr = -Sr; Srr = -Srr; Srrr = -Srrr; Srrrr = -Srrrr; }
  const double Sx = Sr / xr;
  const double Sxx = (Srr - Sx * xrr) / (xr * xr);
  const double Sxxx = (Srrr - 3.0 * Sxx * xr * xrr - Sx * xrrr) / (xr * xr * xr);
  const double Sxxxx =
      (Srrrr - 6.0 * Sxxx * xrr * (xr * xr) - (3.0 * (xrr * xrr) + 4.0 * xr * xrrr) * Sxx - Sx * xrrrr) /
      ((xr * xr) * (xr * xr));
  const double Sz = Ss / zs;
  const double Szz = (Sss - Sz * zss) / (zs * zs);
  const double Szzz = (Ssss - 3.0 * Szz * zs * zss - Sz * zsss) / (zs * zs * zs);
  const double Szzzz =
      (Sssss - 6.0 * Szzz * zss * (zs * zs) - (3.0 * (zss * zss) + 4.0 * zs * zsss) * Szz - Sz * zssss) /
      ((zs * zs) * (zs * zs));
  double Srs = a.Drs[k + 3][i + 3] / a.drds, Srss = a.Drss[k + 3][i + 3] / a.drds2;
  double Srrs = a.Drrs[k + 3][i + 3] / a.dr2ds, Srrss = a.Drrss[k + 3][i + 3] / a.dr2ds2;
  const bool flip = (a.Vbc == 0) ? ((rsym == 1) != (ssym == 1)) : (rsym == 1);
  if (flip) { Srs = -Srs; Srss = -Srss; Srrs = -Srrs; Srrss = -Srrss; }
  const double Sxz = Srs / xr / zs;
  const double Sxxz = (Srrs - Sxz * zs * xrr) / zs / (xr * xr);
  const double Sxzz = (Srss - Sxz * xr * zss) / xr / (zs * zs);
  const double Sxxzz = (Srrss - Sxzz * xrr * (zs * zs) - Sxxz * zss * (xr * xr) - Sxz * xrr * zss) / ((xr * zs) * (xr * zs));
  const bool wall_x = (ip == 0 || ip == a.nx), wall_z = (kp == 0 || kp == a.nz);
  if (wall_x) {
    m = m + Sxx;
  } else if (wall_z) {
    if (a.Vbc == 0) m = m + Szz;
  } else {
    const double term1 = (v.visxx - v.viszz) * (Sxx - Szz);
    const double term2 = v.vis * (Sxxxx + Szzzz);
    const double term3 = 2.0 * v.vis * Sxxzz;
    const double term4 = 4.0 * v.visxz * Sxz;
    const double term5 = 2.0 * v.visx * (Sxxx + Sxzz);
    const double term6 = 2.0 * v.visz * (Szzz + Sxxz);
    m = m + term1 + term2 + term3 + term4 + term5 + term6;
  }
}

// one stencil point folded into the domain (PS/momentum.f90:383-474)
__device__ __forceinline__ void sf_point(const SfArgs& a, int i, int k, int ip, int kp, int p, const VisTerms& v,
                                         double* ab) {
  int rsym = 0, ssym = 0, iq = ip + i, kq = kp + k;
  if (iq < 0) { iq = -iq; rsym = 1; }
  else if (iq > a.nx) { iq = a.nx - (iq - a.nx); rsym = 1; }
  if (kq < 0) { kq = -kq; ssym = 1; }
  else if (kq > a.nz) { kq = a.nz - (kq - a.nz); ssym = 1; }
  const int q = sf_pf(a, iq, kq);
  const int ld = 2 * a.kl + a.ku + 1, kk1 = a.kl + a.ku + 1;
  double& m = ab[(long)(q - 1) * ld + (kk1 + p - q - 1)];
  sf_element(a, i, k, ip, kp, rsym, ssym, v, m);
}

// the rows of build_SF_matrix (PS/momentum.f90:362-478) into a zeroed AB; one
// thread per row, which owns every entry (p, q) of its row
__global__ void k_sf_assemble(SfArgs a, const double* vis, double* ab) {
  const int p = 1 + blockIdx.x * blockDim.x + threadIdx.x;
  if (p > a.n) return;
  int ip, kp;
  sf_indices(a, p, ip, kp);
  const int ld = 2 * a.kl + a.ku + 1, kk1 = a.kl + a.ku + 1;
  const bool corner = (ip == 0 || ip == a.nx) && (kp == 0 || kp == a.nz);
  if (corner || (a.Vbc == 1 && (kp == 0 || kp == a.nz))) {
    ab[(long)(p - 1) * ld + (kk1 - 1)] = 1.0;
    return;
  }
  VisTerms v = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
  if (ip > 0 && ip < a.nx && kp > 0 && kp < a.nz) {
    // second-order viscosity derivatives, D1_so = (-1/2, 0, 1/2), D2_so =
    // (1, -2, 1), Drs_so = D1_so x D1_so (PS/momentum.f90:369-381)
    const double d1[3] = {-0.5, 0.0, 0.5}, d2[3] = {1.0, -2.0, 1.0};
    const int P = a.pitch;
    auto V = [&](int i, int k) { return vis[(long)(k + H3) * P + (i + H3)]; };
    double visr = 0.0, visrr = 0.0, viss = 0.0, visss = 0.0, visrs = 0.0;
    for (int j = -1; j <= 1; j++) visr = visr + d1[j + 1] * V(ip + j, kp);
    for (int j = -1; j <= 1; j++) visrr = visrr + d2[j + 1] * V(ip + j, kp);
    for (int j = -1; j <= 1; j++) viss = viss + d1[j + 1] * V(ip, kp + j);
    for (int j = -1; j <= 1; j++) visss = visss + d2[j + 1] * V(ip, kp + j);
    for (int b = -1; b <= 1; b++)
      for (int q = -1; q <= 1; q++) visrs = visrs + (d1[q + 1] * d1[b + 1]) * V(ip + q, kp + b);
    visr = visr / a.dr; visrr = visrr / a.dr2; viss = viss / a.ds; visss = visss / a.ds2; visrs = visrs / a.drds;
    v.vis = V(ip, kp);
    v.visx = visr / 1.0;
    v.visz = viss / 1.0;
    v.visxx = (visrr - v.visx * 0.0) / 1.0;
    v.viszz = (visss - v.visz * 0.0) / 1.0;
    v.visxz = visrs / 1.0 / 1.0;
  }
  for (int i = -3; i <= 3; i += 6) sf_point(a, i, 0, ip, kp, p, v, ab);
  for (int k = -3; k <= 3; k += 6) sf_point(a, 0, k, ip, kp, p, v, ab);
  for (int i = -2; i <= 2; i++)
    for (int k = -2; k <= 2; k++) sf_point(a, i, k, ip, kp, p, v, ab);
}

// ---------------------------------------------------------------------------
// DGBTF2 (band LU with partial pivoting, LAPACK's unblocked column order) in
// panels of LU_NB columns, each column held by a wavefront in registers.
//   k_lu_panel: one workgroup factors columns p0 .. p0+LU_NB-1, a wavefront
//     per column.  At step s the columns behind it apply the step (interchange,
//     rank-1 update); the wavefront of column s+1 then finds its pivot (DPP
//     maxima), scales the multipliers and leaves them in LDS.  One barrier per
//     step.  It records ju after every step (the last column DGBTF2's step
//     touches; -1 for a zero pivot, which DGBTF2 skips).
//   k_lu_trailing: a wavefront per column beyond the panel replays the panel's
//     steps on it in order -- the interchange, then x = x + L(t,j) (-A(j,c)) --
//     while the column is within the step's ju.
// Every element sees the operations of DGBTF2 in the same order, so the
// factors are DGBTF2's bit for bit.  AB's fill rows start zero (memset) and
// are first written by the step that DGBTF2 zeroes them at, so that zeroing
// is not repeated.
// Bound by the chain of steps: apply to the next column, pivot search, scaling,
// barrier, one compute unit at work.  100x100 (n = 10201, kl = 303), device
// time of the build: 38.6 ms with a thread per row, the panel in LDS and three barriers per
// column (panel of 32: 100 us; trailing columns in LDS 25 us); 14.5 ms now
// (panel of 16: 14.2 us, trailing 8.0 us).  With rows per thread and the panel
// in registers every column's pivot row passes through LDS, in any form of it
// 1.6 us a step: 22 ms.  Panels of 32 (two columns per wavefront) 18.6 ms, of
// 24 19.6, of 8 19.4 (these three with more registers than now).
// ---------------------------------------------------------------------------
constexpr int LU_NB = 16;                         // panel columns: the wavefronts of a workgroup
constexpr int LU_MAX_KL = 1023;                   // at most 17 rows per lane
constexpr int LU_LDS_LIMIT = 160 * 1024 - 1024;   // dynamic LDS per workgroup (gfx950: 160 KB)
constexpr int LU_TRAIL_WAVES = 8;                 // columns per trailing workgroup

// the value of v in lane `lane` (uniform), as a uniform double
__device__ __forceinline__ double readlane_f64(double v, int lane) {
  const long long x = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_readlane((int)(x & 0xffffffffLL), lane);
  const int hi = __builtin_amdgcn_readlane((int)(x >> 32), lane);
  return __longlong_as_double(((long long)hi << 32) | (long long)(unsigned int)lo);
}

// one DPP step of a maximum of unsigned words over lanes (0 where the step has
// no source lane): a single instruction, where doubles would need two moves
// and two maxima
template <int CTRL, int ROWS>
__device__ __forceinline__ unsigned max_dpp(unsigned v) {
  return max(v, (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, ROWS, 0xf, false));
}
// maxima of each row of 16 lanes, in its lane 15 (row_shr 1, 2, 4, 8)
__device__ __forceinline__ unsigned row_max_dpp(unsigned v) {
  return max_dpp<0x118, 0xf>(max_dpp<0x114, 0xf>(max_dpp<0x112, 0xf>(max_dpp<0x111, 0xf>(v))));
}
// maximum over the wavefront, as a uniform value (row_bcast 15, 31)
__device__ __forceinline__ unsigned wave_max_dpp(unsigned v) {
  return __builtin_amdgcn_readlane(max_dpp<0x143, 0xc>(max_dpp<0x142, 0xa>(row_max_dpp(v))), 63);
}

// A wavefront holds a column of the panel's rows in registers: row 64 q + lane
// in x[q].

// rows s and l of the column change places; returns the new row s.  (No branch
// on the register of row l: where the paths meet, the column would be copied.)
template <int Q>
__device__ __forceinline__ double lu_swap(double (&x)[Q], int s, int l, int lane) {
  const double top = readlane_f64(x[0], s);
  double t = x[0];
#pragma unroll
  for (int q = 0; q < Q; q++) {
    const bool here = 64 * q + lane == l;
    t = here ? x[q] : t;
    x[q] = here ? top : x[q];
  }
  const double low = readlane_f64(t, l & 63);
  x[0] = lane == s ? low : x[0];
  return low;
}

// step s of the panel: the interchange, then x = x + L (-x(s)) on rows s+1 .. last
template <int Q>
__device__ __forceinline__ void lu_apply(double (&x)[Q], const double (&L)[Q], int s, int l, int last, int lane) {
  if (l != s) lu_swap(x, s, l, lane);
  const double temp = -1.0 * readlane_f64(x[0], s);
#pragma unroll
  for (int q = 0; q < Q; q++) {
    const double y = x[q] + L[q] * temp;
    const int r = 64 * q + lane;
    x[q] = (q > 0 || r > s) && r <= last ? y : x[q];
  }
}

struct LuStep { int l, ju, taken, inf; };   // the step's pivot row, and ju and inf after it

// step s's own column: pivot search, interchange, multipliers
template <int Q>
__device__ __forceinline__ LuStep lu_pivot(double (&x)[Q], double* Ls, int s, int col, int last, int ku, int n, int ju,
                                           int inf, int lane) {
  // the first of the rows with the largest entry that is a number
  double v = -1.0;
  int row = 0;
#pragma unroll
  for (int q = 0; q < Q; q++) {
    const double y = fabs(x[q]);
    const int r = 64 * q + lane;
    if ((q > 0 || r >= s) && r <= last && y > v) { v = y; row = r; }
  }
  // over the lanes, magnitudes compare as integers: the high words decide but
  // for ties (DPP maxima of single words, no LDS)
  const unsigned long long key = (unsigned long long)__double_as_longlong(v);
  const unsigned kh = v >= 0.0 ? (unsigned)(key >> 32) + 1u : 0u, hm = wave_max_dpp(kh);
  unsigned long long at = __ballot(kh == hm);
  int l = __builtin_amdgcn_readlane(row, __ffsll((long long)at) - 1);
  if (at & (at - 1)) {
    const unsigned kw = kh == hm ? (unsigned)key : 0u, wm = wave_max_dpp(kw);
    l = ~(int)wave_max_dpp(kh == hm && kw == wm ? ~(unsigned)row : 0u);
  }
  if (hm == 0u) l = s;   // no candidate is a number
  const double piv = l != s ? lu_swap(x, s, l, lane) : readlane_f64(x[0], s);
  LuStep st{l, ju, piv != 0.0, inf};
  if (st.taken) {
    st.ju = max(ju, min(col + ku + (l - s), n));
    const double rcp = 1.0 / piv;
#pragma unroll
    for (int q = 0; q < Q; q++) {
      const double y = rcp * x[q];
      const int r = 64 * q + lane;
      x[q] = (q > 0 || r > s) && r <= last ? y : x[q];
      Ls[r] = x[q];
    }
  } else if (inf == 0) {
    st.inf = col;
  }
  return st;
}

template <int Q>   // rows per lane
__global__ void __launch_bounds__(LU_NB * 64) k_lu_panel(double* ab, int32_t* ipiv, int32_t* ju_rec, int32_t* state,
                                                         int n, int kl, int ku, int p0) {
  __shared__ double Ls[2][64 * Q];   // the step's multipliers
  __shared__ LuStep step[2];
  const int lane = threadIdx.x & 63, c = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const long ld = 2 * kl + ku + 1;
  const int kv = ku + kl, np = min(LU_NB, n - p0 + 1);
  // the wavefront's column: rows p0 .. p0+kl+LU_NB-1 that are stored
  const int lo = c - kv, hi = min(n - p0, c + kl);
  double x[Q];
#pragma unroll
  for (int q = 0; q < Q; q++) {
    const int r = 64 * q + lane;
    x[q] = c < np && r >= lo && r <= hi ? ab[(long)(p0 + c - 1) * ld + (kv + r - c)] : 0.0;
  }
  auto pivot = [&](int ju, int inf) {
    const int col = p0 + c;
    const LuStep st = lu_pivot(x, Ls[c & 1], c, col, c + min(kl, n - col), ku, n, ju, inf, lane);
    if (lane == 0) {
      step[c & 1] = st;
      ipiv[col - 1] = p0 + st.l;
      ju_rec[col - 1] = st.taken ? st.ju : -1;
    }
  };
  // ju and the first zero pivot carried between panels
  if (c == 0) pivot(p0 == 1 ? 1 : state[0], p0 == 1 ? 0 : state[1]);
  for (int s = 0; s < np; s++) {
    __syncthreads();
    const LuStep st = step[s & 1];
    const int l = __builtin_amdgcn_readfirstlane(st.l), ju = __builtin_amdgcn_readfirstlane(st.ju);
    const int taken = __builtin_amdgcn_readfirstlane(st.taken), inf = __builtin_amdgcn_readfirstlane(st.inf);
    if (s + 1 == np) {
      if (threadIdx.x == 0) { state[0] = ju; state[1] = inf; }
      break;
    }
    if (c <= s || c >= np) continue;
    double L[Q];
#pragma unroll
    for (int q = 0; q < Q; q++) L[q] = Ls[s & 1][64 * q + lane];
    if (taken && p0 + c <= ju) lu_apply(x, L, s, l, s + min(kl, n - (p0 + s)), lane);
    if (c == s + 1) pivot(ju, inf);
  }
  // (the loads' addresses are not kept through the loop: they would take as
  // many registers as the column)
  int row0 = lane;
  asm volatile("" : "+v"(row0));
#pragma unroll
  for (int q = 0; q < Q; q++) {
    const int r = 64 * q + row0;
    if (c < np && r >= lo && r <= hi) ab[(long)(p0 + c - 1) * ld + (kv + r - c)] = x[q];
  }
}

template <int Q>   // rows per lane
__global__ void __launch_bounds__(LU_TRAIL_WAVES * 64) k_lu_trailing(double* ab, const int32_t* ipiv,
                                                                     const int32_t* ju_rec, int n, int kl, int ku,
                                                                     int p0) {
  extern __shared__ double Ls[];   // Ls[s*W + r] = L(p0+r, p0+s)
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const long ld = 2 * kl + ku + 1;
  const int kv = ku + kl, W = kl + LU_NB, pe = min(p0 + LU_NB - 1, n), np = pe - p0 + 1;
  const int c = pe + 1 + blockIdx.x * LU_TRAIL_WAVES + wave;
  const bool live = c <= min(n, pe + kv);
  // this wavefront's column: rows p0 .. p0+W-1 that are stored
  const int lo = c - kv - p0, hi = min(n, c + kl) - p0;
  double x[Q];
#pragma unroll
  for (int q = 0; q < Q; q++) {
    const int r = 64 * q + lane;
    x[q] = live && r < W && r >= lo && r <= hi ? ab[(long)(c - 1) * ld + (kv + p0 + r - c)] : 0.0;
  }
  // the panel's multipliers (entries that are none are read from a stored
  // place and not used), and each step's ju and interchange in lane s
  const int js = p0 + min(lane, np - 1);
  const int juv = ju_rec[js - 1], lv = ipiv[js - 1] - p0;
  static_assert(LU_NB == 2 * LU_TRAIL_WAVES, "two of the panel's columns per wavefront");
  double v[2][Q];
#pragma unroll
  for (int u = 0; u < 2; u++) {
    const int sc = min(wave + u * LU_TRAIL_WAVES, np - 1);
#pragma unroll
    for (int q = 0; q < Q; q++)
      v[u][q] = ab[(long)(p0 + sc - 1) * ld + (kv + min(max(64 * q + lane - sc, 0), kl))];
  }
#pragma unroll
  for (int u = 0; u < 2; u++) {
    const int sc = wave + u * LU_TRAIL_WAVES;
#pragma unroll
    for (int q = 0; q < Q; q++)
      if (sc < np && 64 * q + lane < W) Ls[sc * W + 64 * q + lane] = v[u][q];
  }
  __syncthreads();
  if (!live) return;
  double L[Q];
  auto fetch = [&](int sc) {
#pragma unroll
    for (int q = 0; q < Q; q++) L[q] = Ls[sc * W + min(64 * q + lane, W - 1)];
  };
  fetch(0);
  for (int sc = 0; sc < np; sc++) {
    double Lc[Q];
#pragma unroll
    for (int q = 0; q < Q; q++) Lc[q] = L[q];
    fetch(min(sc + 1, np - 1));   // the next step's multipliers
    const int j = p0 + sc, jut = __builtin_amdgcn_readlane(juv, sc);
    if (jut < 0 || c > jut) continue;
    const int l = __builtin_amdgcn_readlane(lv, sc), last = sc + min(kl, n - j);
    lu_apply(x, Lc, sc, l, last, lane);
  }
#pragma unroll
  for (int q = 0; q < Q; q++) {
    const int r = 64 * q + lane;
    if (r < W && r >= lo && r <= hi) ab[(long)(c - 1) * ld + (kv + p0 + r - c)] = x[q];
  }
}

// ---------------------------------------------------------------------------
// DGBTRS('N', one right-hand side), blocked.  The forward and the backward
// substitution each run as one workgroup; b's band window lives in an LDS
// ring (slot = (position-1) mod RING) refilled from global memory in chunks,
// and finished positions are written back in place.  The column steps are
// taken NBH (one wavefront) at a time:
//   head: wavefront 0 runs the block's steps on the block's NBH rows, one row
//     per lane and the block's triangle of L (or U) in registers, with the
//     step's value broadcast by v_readlane: no barrier per step;
//   tail: the other wavefronts then apply the block's steps to the kl (or
//     kl+ku) rows below (above) the head, E rows per thread, in step order.
// Either loads a block's band entries into registers while the other is at
// work: the head its next triangle, the tail its next D column steps.
// Each element sees the same operations in the same order as DGBTRS's
// column-by-column loops, so the results are identical.  Forward blocks
// end early where a pivot row would leave the head (the block's first step
// may pivot anywhere: its swap is made in the ring while every row is
// current); the pivots of this operator are rare and adjacent.
//   forward (L with the interchanges): b(j) <-> b(ipiv(j)), then
//     b(j+1 .. j+kl) += L(., j) (-b(j));
//   backward (DTBSV, upper, bandwidth kl+ku): x(j) = b(j)/U(j,j) unless b(j)
//     is zero, then b(j-1 .. j-kl-ku) -= x(j) U(., j).
// Bound by the chain of a block (head 1.7 us forward, 3.5 us backward with its
// quotients; then the tail) and by what one compute unit draws from memory,
// 40 GB/s (31 and 56 MB a solve, by counters).  At 100x100 (160 blocks, bands 303 and 606) forward and
// backward took 1.73 and 3.56 ms with the loads between the barriers, masked
// steps and divisions, and take 0.78 and 1.39 ms.  (Reloading each register
// right after its step would use the tail's time too, but the compiler gives
// such a loop twice the registers.)
// ---------------------------------------------------------------------------
constexpr int SOLVE_MAX_TAIL = 640;   // tail threads: 11 wavefronts leave 168 registers each
constexpr int RING = 4096;
constexpr int CHUNK = 512;
constexpr int NBH = 64;   // head rows per block: one wavefront

__device__ __forceinline__ int ring_slot(int pos) { return (pos - 1) & (RING - 1); }

// The columns of AB from j0 on, in step order: entry r of a column lies at
// p[r - j0].  Moves on to the next column with every step and stays at the
// last one that is used.
struct BandCursor {
  const double* p;
  int left, step;   // columns to go; the distance of one
  __device__ __forceinline__ void next() {
    p += left > 0 ? step : 0;
    left--;
  }
};

// the band entries of the next D steps, for the rows off[e] from the block's first
template <int E, int D>
__device__ __forceinline__ void band_load(double (&lt)[E][D], BandCursor& next, const int (&off)[E]) {
#pragma unroll
  for (int q = 0; q < D; q++) {
#pragma unroll
    for (int e = 0; e < E; e++) lt[e][q] = next.p[off[e]];
    next.next();
  }
}

// the tail's steps of one block, the first D of which have their band entries
// in lt.  valid(e, sc): the step is taken and the row is within its band (ALL:
// they all are).
template <bool ALL, bool BACK, int E, int D, class Valid>
__device__ __forceinline__ void band_tail(double (&v)[E], double (&lt)[E][D], const double* T, BandCursor& next,
                                          const int (&off)[E], Valid valid) {
#pragma unroll
  for (int k0 = 0; k0 < NBH; k0 += D) {
#pragma unroll
    for (int q = 0; q < D; q++) {
      const int sc = BACK ? NBH - 1 - (k0 + q) : k0 + q;
      const double ts = T[sc];
#pragma unroll
      for (int e = 0; e < E; e++) {
        const double y = BACK ? v[e] - ts * lt[e][q] : v[e] + lt[e][q] * ts;
        v[e] = ALL || valid(e, sc) ? y : v[e];
      }
    }
    if (k0 + D < NBH) band_load(lt, next, off);
  }
}

// forward: L y = P b, in place on b.  (ab has NBH entries of padding: lanes
// beyond a column's band read past it and drop what they read.)
template <int E, int D>
__global__ void __launch_bounds__(SOLVE_MAX_TAIL + 64) k_band_forward(const double* __restrict__ ab,
                                                                      const int32_t* __restrict__ ipiv, double* b,
                                                                      int n, int kl, int ku) {
  __shared__ double R[RING];
  __shared__ double T[NBH];   // -b(j) of the block's steps
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const long ld = 2 * kl + ku + 1;
  if (kl == 0 || n < 2) return;
  int hi = min(n, NBH + kl + CHUNK);
  for (int pos = 1 + tid; pos <= hi; pos += blockDim.x) R[ring_slot(pos)] = b[pos - 1];
  __syncthreads();
  // L(r, j) = AB(kl+ku+1+r-j, j), 1-based; columns past n-1 are not used
  auto columns = [&](int j0) {
    const int j = min(j0, n - 1);
    return BandCursor{ab + ((long)(j - 1) * ld + (kl + ku + j0 - j)), n - 1 - j, (int)ld - 1};
  };
  auto pivots = [&](int j0) { return ipiv[min(j0 + lane, n - 1) - 1]; };
  // the block from j0: steps j0 .. j0+nb-1, the pivots of all but the first inside the head
  auto steps = [&](int j0, int pl) {
    const bool out = lane >= 1 && j0 + lane <= n - 1 && pl > j0 + NBH - 1;
    const unsigned long long m = __ballot(out);
    return min(min(m ? __ffsll((long long)m) - 1 : NBH, NBH), n - j0);
  };
  int pl = pivots(1);
  if (wave == 0) {
    double lc[1][NBH];
    const int off[1] = {lane};
    BandCursor next = columns(1);
    band_load(lc, next, off);
    for (int j0 = 1; j0 <= n - 1;) {
      const int nb = steps(j0, pl), jn = j0 + nb, pn = pivots(jn);
      int me = lane;   // not known outside the loop, or 64 comparisons of it would be kept
      asm volatile("" : "+v"(me));
      const int l0 = __builtin_amdgcn_readfirstlane(pl);
      if (l0 != j0 && lane == 0) {
        const double t0 = R[ring_slot(j0)];
        R[ring_slot(j0)] = R[ring_slot(l0)];
        R[ring_slot(l0)] = t0;
      }
      double v = (j0 + lane <= n) ? R[ring_slot(j0 + lane)] : 0.0, tv = 0.0;
      const bool swaps = __ballot(lane >= 1 && lane < nb && pl != j0 + lane) != 0;
      if (nb == NBH && !swaps && kl >= NBH) {
        // each step is one lane read and one multiply-add; what it leaves in
        // the lanes of finished rows is not used
#pragma unroll
        for (int sc = 0; sc < NBH; sc++) {
          const double temp = -1.0 * readlane_f64(v, sc);
          tv = me == sc ? temp : tv;
          v = v + lc[0][sc] * temp;
        }
        v = -1.0 * tv;
      } else {
#pragma unroll
        for (int sc = 0; sc < NBH; sc++) {
          if (sc < nb) {
            const int j = j0 + sc;
            if (sc > 0) {
              const int l = __builtin_amdgcn_readlane(pl, sc);
              if (l != j) {
                const double a = readlane_f64(v, sc), c = readlane_f64(v, l - j0);
                if (me == sc) v = c;
                if (me == l - j0) v = a;
              }
            }
            const double temp = -1.0 * readlane_f64(v, sc);
            tv = me == sc ? temp : tv;
            const double y = v + lc[0][sc] * temp;
            v = me > sc && j0 + me <= min(n, j + kl) ? y : v;
          }
        }
      }
      T[lane] = tv;
      if (lane < nb) b[j0 + lane - 1] = v;                    // y(j0 .. j0+nb-1): final
      else if (j0 + lane <= n) R[ring_slot(j0 + lane)] = v;   // head rows of the next block
      __syncthreads();
      next = columns(jn);   // while the tail works on this block
      band_load(lc, next, off);
      __syncthreads();
      j0 = jn;
      pl = pn;
    }
    if (lane == 0) b[n - 1] = R[ring_slot(n)];
  } else {
    const int nt = blockDim.x - 64;
    int row[E], off[E];   // rows below the head, and within the band of every step
    bool full = true;
    double lt[E][D], v[E];
#pragma unroll
    for (int e = 0; e < E; e++) {
      row[e] = tid - 64 + e * nt;
      off[e] = NBH + min(row[e], kl - 1);
      full = full && NBH + 64 * (wave - 1) + 63 + e * nt <= kl;
    }
    for (int j0 = 1; j0 <= n - 1;) {
      const int nb = steps(j0, pl), jn = j0 + nb;
      pl = pivots(jn);
      BandCursor next = columns(j0);   // while the head works on this block
      band_load(lt, next, off);
      // the rows of the next block; the slots reused belong to rows below j0
      if (const int want = min(n, jn + NBH - 1 + kl); hi < want) {
        const int top = min(n, want + CHUNK);
        for (int pos = hi + 1 + tid - 64; pos <= top; pos += nt) R[ring_slot(pos)] = b[pos - 1];
        hi = top;
      }
      __syncthreads();
#pragma unroll
      for (int e = 0; e < E; e++) v[e] = R[ring_slot(min(j0 + NBH + row[e], n))];
      int room[E];   // steps before the row enters the band
#pragma unroll
      for (int e = 0; e < E; e++) {
        room[e] = NBH + row[e] - kl;
        asm volatile("" : "+v"(room[e]));
      }
      auto valid = [&](int e, int sc) { return sc < nb && room[e] <= sc; };
      if (full && nb == NBH) band_tail<true, false>(v, lt, T, next, off, valid);
      else band_tail<false, false>(v, lt, T, next, off, valid);
#pragma unroll
      for (int e = 0; e < E; e++) {
        const int r = j0 + NBH + row[e];
        if (row[e] < kl && r <= min(n, jn - 1 + kl)) R[ring_slot(r)] = v[e];
      }
      __syncthreads();
      j0 = jn;
    }
  }
}

// backward: U x = y (DTBSV, upper, non-unit, bandwidth kl+ku), in place on b
template <int E, int D>
__global__ void __launch_bounds__(SOLVE_MAX_TAIL + 64) k_band_backward(const double* __restrict__ ab, double* b,
                                                                       int n, int kl, int ku) {
  __shared__ double R[RING];
  __shared__ double X[NBH];              // x(j) of the block's steps
  __shared__ unsigned long long taken;   // the steps taken (b(j) != 0)
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const long ld = 2 * kl + ku + 1;
  const int kk = kl + ku;   // U(i, j) = AB(kk+1+i-j, j)
  int lo = max(1, n - NBH - kk - CHUNK + 1);
  for (int pos = lo + tid; pos <= n; pos += blockDim.x) R[ring_slot(pos)] = b[pos - 1];
  __syncthreads();
  // from column j0+NBH-1 down (there is one: n >= NBH)
  auto columns = [&](int j0) {
    return BandCursor{ab + ((long)(j0 + NBH - 2) * ld + (kk + 1 - NBH)), NBH - 1, 1 - (int)ld};
  };
  if (wave == 0) {
    auto diag = [&](int j0) { return ab[(long)(j0 + lane - 1) * ld + kk]; };
    int j1 = n, j0 = n - NBH + 1;
    BandCursor next = columns(j0);
    double uc[1][NBH], dg = diag(j0);   // uc[0][k]: step k, column j0 + NBH-1 - k
    const int off[1] = {lane};
    band_load(uc, next, off);
    while (j1 >= 1) {
      const int nb = j1 - j0 + 1, jn = max(1, j0 - NBH);
      int me = lane;
      asm volatile("" : "+v"(me));
      double v = (lane < nb) ? R[ring_slot(j0 + lane)] : 0.0, xv = 0.0;
      unsigned long long tk = 0;
      // Quotients from the reciprocals of the diagonal, correctly rounded by
      // two corrections (Markstein) while no exponent is extreme: a chain of 5
      // operations instead of about 14
      const double rd = 1.0 / dg, u = dg;
      const bool mild = fabs(u) > 0x1p-400 && fabs(u) < 0x1p400;
      if (nb == NBH && kk >= NBH && __ballot(!mild) == 0) {
        double vb = 0.0;
#pragma unroll
        for (int k = 0; k < NBH; k++) {
          const int sc = NBH - 1 - k;
          const double bj = readlane_f64(v, sc), us = readlane_f64(u, sc);
          const double rs = readlane_f64(rd, sc), q0 = bj * rs, q1 = __fma_rn(__fma_rn(-q0, us, bj), rs, q0);
          double x = __fma_rn(__fma_rn(-q1, us, bj), rs, q1);
          const unsigned long long bits = (unsigned long long)__double_as_longlong(bj);
          const bool take = (bits << 1) != 0;
          if ((unsigned)((bits >> 52) & 0x7ff) - 523u > 1000u && take) x = bj / us;
          vb = me == sc ? v : vb;
          xv = me == sc ? x : xv;
          if (take) tk |= 1ull << sc;
          const double y = v - x * uc[0][k];
          v = take ? y : v;
        }
        v = (tk >> lane) & 1 ? xv : vb;
      } else {
        // the band may not reach every head row
#pragma unroll
        for (int k = 0; k < NBH; k++) {
          const int sc = NBH - 1 - k;
          const double bj = readlane_f64(v, sc);
          if (sc < nb && bj != 0.0) {
            const double x = bj / readlane_f64(u, sc);
            if (me == sc) v = xv = x;
            const double y = v - x * uc[0][k];
            v = me < sc && sc - me <= kk ? y : v;
            tk |= 1ull << sc;
          }
        }
      }
      X[lane] = xv;
      if (lane == 0) taken = tk;
      if (lane < nb) b[j0 + lane - 1] = v;   // x(j0 .. j1): final
      __syncthreads();
      dg = diag(jn);   // while the tail works on this block
      next = columns(jn);
      band_load(uc, next, off);
      __syncthreads();
      j1 = j0 - 1;
      j0 = jn;
    }
  } else {
    const int nt = blockDim.x - 64;
    int row[E], off[E];   // rows above the head: j0-1-row, and within the band of every step
    bool full = true;
    double lt[E][D], v[E];
    int j1 = n, j0 = n - NBH + 1;
#pragma unroll
    for (int e = 0; e < E; e++) {
      row[e] = tid - 64 + e * nt;
      off[e] = -1 - min(row[e], kk - 1);
      full = full && 64 * (wave - 1) + 63 + e * nt <= kk - NBH;
    }
    while (j1 >= 1) {
      const int jn = max(1, j0 - NBH);
      BandCursor next = columns(j0);   // while the head works on this block
      band_load(lt, next, off);
      // the rows of the next block; the slots reused belong to rows above j1
      if (const int want = max(1, jn - kk); lo > want) {
        const int bot = max(1, want - CHUNK);
        for (int pos = bot + tid - 64; pos < lo; pos += nt) R[ring_slot(pos)] = b[pos - 1];
        lo = bot;
      }
      __syncthreads();
      const unsigned long long tk = taken;
      const bool every = __builtin_amdgcn_readfirstlane((int)(tk & (tk >> 32))) == -1;
#pragma unroll
      for (int e = 0; e < E; e++) v[e] = R[ring_slot(max(j0 - 1 - row[e], 1))];
      int room[E];   // steps from which on the row is in the band
#pragma unroll
      for (int e = 0; e < E; e++) {
        room[e] = kk - 1 - row[e];
        asm volatile("" : "+v"(room[e]));
      }
      auto valid = [&](int e, int sc) { return ((tk >> sc) & 1) && sc <= room[e]; };
      if (full && every) band_tail<true, true>(v, lt, X, next, off, valid);
      else band_tail<false, true>(v, lt, X, next, off, valid);
#pragma unroll
      for (int e = 0; e < E; e++)
        if (row[e] < kk && j0 - 1 - row[e] >= 1) R[ring_slot(j0 - 1 - row[e])] = v[e];
      __syncthreads();
      j1 = j0 - 1;
      j0 = jn;
    }
  }
}

// ---------------------------------------------------------------------------
// buoyancy (PS/momentum.f90:255-285): Bvec(p) = (RaT Tx - RaC Cx) RowB(p) at
// interior nodes, 0 elsewhere
// ---------------------------------------------------------------------------
__global__ void k_sf_buoyancy(SfArgs a, const double* Tb, const double* Cb, const double* row, double RaT, double RaC,
                              double* B) {
  const int p = 1 + blockIdx.x * blockDim.x + threadIdx.x;
  if (p > a.n) return;
  int ip, kp;
  sf_indices(a, p, ip, kp);
  double v = 0.0;
  if (ip > 0 && ip < a.nx && kp > 0 && kp < a.nz) {
    const int p3 = a.nx + 7, p5 = a.nx + 11;
    double tr = 0.0, cr = 0.0;
    for (int j = -2; j <= 2; j++) tr = tr + a.D1[j + 3] * Tb[(long)(kp + H3) * p3 + (ip + j + H3)];
    for (int j = -2; j <= 2; j++) cr = cr + a.D1[j + 3] * Cb[(long)(kp + H5) * p5 + (ip + j + H5)];
    const double Tx = (tr / a.dr) / 1.0, Cx = (cr / a.dr) / 1.0;
    const double rc = 0.0 + RaC * Cx;
    v = (RaT * Tx - rc) * row[p - 1];
  }
  B[p - 1] = v;
}

// Stream_grid (PS/momentum.f90:287-319): psi = Bvec at the nodes; ghosts are
// exact (anti)symmetric images, written here in closed form per node
__global__ void k_sf_scatter(SfArgs a, const double* B, double* SF) {
  const int i = -H3 + (int)(blockIdx.x * blockDim.x + threadIdx.x);
  const int k = -H3 + (int)(blockIdx.y * blockDim.y + threadIdx.y);
  if (i > a.nx + H3 || k > a.nz + H3) return;
  int iq = i, kq = k;
  double sgn = 1.0;
  if (iq < 0) { iq = -iq; sgn = -sgn; }
  else if (iq > a.nx) { iq = 2 * a.nx - iq; sgn = -sgn; }
  if (kq < 0) { kq = -kq; if (a.Vbc == 0) sgn = -sgn; }
  else if (kq > a.nz) { kq = 2 * a.nz - kq; if (a.Vbc == 0) sgn = -sgn; }
  const double v = B[sf_pf(a, iq, kq) - 1];
  SF[(long)(k + H3) * (a.nx + 7) + (i + H3)] = sgn < 0.0 ? -v : v;
}

__global__ void k_fill_f64(double* v, long n, double x) {
  const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t < n) v[t] = x;
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
static SfArgs sf_args(const Context& c) {
  SfArgs a;
  const Tables& t = c.T;
  std::memcpy(a.D1, t.D1, sizeof a.D1); std::memcpy(a.D2, t.D2, sizeof a.D2);
  std::memcpy(a.D3, t.D3, sizeof a.D3); std::memcpy(a.D4, t.D4, sizeof a.D4);
  std::memcpy(a.Drs, t.Drs, sizeof a.Drs); std::memcpy(a.Drss, t.Drss, sizeof a.Drss);
  std::memcpy(a.Drrs, t.Drrs, sizeof a.Drrs); std::memcpy(a.Drrss, t.Drrss, sizeof a.Drrss);
  a.dr = t.dr; a.ds = t.ds; a.dr2 = t.dr2; a.ds2 = t.ds2; a.dr3 = t.dr3; a.ds3 = t.ds3; a.dr4 = t.dr4; a.ds4 = t.ds4;
  a.drds = t.drdsg[1]; a.drds2 = t.drds2g[1]; a.dr2ds = t.dr2dsg[1]; a.dr2ds2 = t.dr2ds2g[1];
  a.nx = t.nx; a.nz = t.nz; a.Vbc = c.P.Vbc; a.Database = c.P.Database;
  a.kl = t.dkl; a.ku = t.dku; a.n = t.dn; a.pitch = t.nx + 7;
  return a;
}

int direct_alloc(Context& c) {
  const Tables& t = c.T;
  if (t.dkl + t.dku + NBH + CHUNK >= RING) {   // the solves' LDS window
    set_error("direct solver: band width " + std::to_string(t.dkl + t.dku) + " exceeds " +
              std::to_string(RING - NBH - CHUNK - 1));
    return PT_ERR_UNSUPPORTED;
  }
  if (t.dn < NBH) {   // the backward solve's blocks are whole ones
    set_error("direct solver: fewer than " + std::to_string(NBH) + " unknowns");
    return PT_ERR_UNSUPPORTED;
  }
  const size_t ld = (size_t)(2 * t.dkl + t.dku + 1);
  if (hipMalloc((void**)&c.dAB, sizeof(double) * (ld * (size_t)t.dn + NBH)) != hipSuccess ||
      hipMalloc((void**)&c.dRow, sizeof(double) * (size_t)t.dn) != hipSuccess ||
      hipMalloc((void**)&c.dB, sizeof(double) * (size_t)t.dn) != hipSuccess ||
      hipMalloc((void**)&c.dipiv, sizeof(int32_t) * (size_t)t.dn) != hipSuccess ||
      hipMalloc((void**)&c.dju, sizeof(int32_t) * (size_t)t.dn) != hipSuccess ||
      hipMalloc((void**)&c.d_lustate, sizeof(int32_t) * 2) != hipSuccess) {
    set_error("direct solver: out of device memory for the band matrix");
    return PT_ERR_HIP;
  }
  return PT_OK;
}

int direct_free(Context& c) {
  void* ps[] = {c.dAB, c.dRow, c.dB, c.dipiv, c.dju, c.d_lustate};
  for (void* p : ps)
    if (p) (void)hipFree(p);
  c.dAB = nullptr; c.dRow = nullptr; c.dB = nullptr; c.dipiv = nullptr; c.dju = nullptr; c.d_lustate = nullptr;
  return PT_OK;
}

// build_SF_matrix with tstep >= 0 (PS/momentum.f90:321-488): vis = visf at the
// nodes (isoviscous: 1), assembly, DGBEQU row scaling, band LU
int build_sf_matrix(Context& c) {
  const Tables& t = c.T;
  if (c.P.iterate != 0) {
    set_error("build_SF_matrix needs a context created with iterate=0");
    return PT_ERR_INVALID;
  }
  const SfArgs a = sf_args(c);
  Level& L1 = c.L[1];
  hipLaunchKernelGGL(k_fill_f64, dim3((unsigned)((L1.nelem + 255) / 256)), dim3(256), 0, c.stream, L1.v.vis,
                     (long)L1.nelem, 1.0);
  const size_t ld = (size_t)(2 * t.dkl + t.dku + 1);
  PT_HIP(hipMemsetAsync(c.dAB, 0, sizeof(double) * ld * (size_t)t.dn, c.stream));
  hipLaunchKernelGGL(k_sf_assemble, dim3((t.dn + 127) / 128), dim3(128), 0, c.stream, a, L1.v.vis, c.dAB);
  PT_TRY(launch_equilibrate(c, c.dAB, c.dRow, t.dn, t.dkl, t.dku));
  if (t.dkl > LU_MAX_KL) {
    set_error("direct solver: lower band width above " + std::to_string(LU_MAX_KL));
    return PT_ERR_UNSUPPORTED;
  }
  const int rows = t.dkl + LU_NB, kv = t.dkl + t.dku;
  auto factor = [&](auto qc) -> int {
    constexpr int Q = decltype(qc)::value;
    static OncePerDevice lds;
    PT_TRY(allow_lds(c, lds, k_lu_trailing<Q>, LU_LDS_LIMIT));
    for (int p0 = 1; p0 <= t.dn; p0 += LU_NB) {
      hipLaunchKernelGGL(k_lu_panel<Q>, dim3(1), dim3(LU_NB * 64), 0, c.stream, c.dAB, c.dipiv, c.dju, c.d_lustate,
                         t.dn, t.dkl, t.dku, p0);
      const int pe = std::min(p0 + LU_NB - 1, t.dn), ncols = std::min(t.dn, pe + kv) - pe;
      if (ncols <= 0) continue;
      hipLaunchKernelGGL(k_lu_trailing<Q>, dim3((ncols + LU_TRAIL_WAVES - 1) / LU_TRAIL_WAVES),
                         dim3(LU_TRAIL_WAVES * 64), sizeof(double) * LU_NB * rows, c.stream, c.dAB, c.dipiv, c.dju,
                         t.dn, t.dkl, t.dku, p0);
    }
    return PT_OK;
  };
  // rows per lane: the band's height in registers, as little padded as these sizes allow
  if (rows <= 128) PT_TRY(factor(std::integral_constant<int, 2>{}));
  else if (rows <= 192) PT_TRY(factor(std::integral_constant<int, 3>{}));
  else if (rows <= 256) PT_TRY(factor(std::integral_constant<int, 4>{}));
  else if (rows <= 320) PT_TRY(factor(std::integral_constant<int, 5>{}));
  else if (rows <= 384) PT_TRY(factor(std::integral_constant<int, 6>{}));
  else if (rows <= 512) PT_TRY(factor(std::integral_constant<int, 8>{}));
  else if (rows <= 640) PT_TRY(factor(std::integral_constant<int, 10>{}));
  else if (rows <= 832) PT_TRY(factor(std::integral_constant<int, 13>{}));
  else PT_TRY(factor(std::integral_constant<int, 17>{}));
  int32_t info = 0;
  PT_HIP(hipMemcpyAsync(&info, c.d_lustate + 1, sizeof(int32_t), hipMemcpyDeviceToHost, c.stream));
  PT_HIP(hipStreamSynchronize(c.stream));
  if (info != 0) {
    set_error("direct solver band LU: zero pivot at column " + std::to_string(info));
    return PT_ERR_SINGULAR_COARSE;
  }
  c.direct_built = true;
  return PT_OK;
}

// solve_SF_equation (PS/momentum.f90:621-653)
int solve_sf_equation(Context& c) {
  const Tables& t = c.T;
  if (!c.direct_built) {
    set_error("solve_SF_equation before build_SF_matrix");
    return PT_ERR_INVALID;
  }
  const SfArgs a = sf_args(c);
  hipLaunchKernelGGL(k_sf_buoyancy, dim3((t.dn + 255) / 256), dim3(256), 0, c.stream, a, c.Tbuoy, c.Cbuoy, c.dRow,
                     c.P.RaT, c.P.RaC, c.dB);
  // one workgroup per triangular solve: the head's wavefront, and tail
  // wavefronts with E rows per thread that load D steps at a time, as the
  // band's height needs and the registers allow.  (E, D) = (2, 32) against
  // (2, 16) with up to 15 tail wavefronts, 20x210 (bands 633 and 1266): 1.46
  // and 1.65 ms; (4, 8) against (4, 16), which spills, 20x250 (753 and 1506):
  // 3.2 and 6.4 ms; 4.6 ms before.
  auto run = [&](int band, auto launch) {
    if (band <= SOLVE_MAX_TAIL) launch(std::integral_constant<int, 1>{}, std::integral_constant<int, 64>{}, band);
    else if (band <= 2 * SOLVE_MAX_TAIL)
      launch(std::integral_constant<int, 2>{}, std::integral_constant<int, 32>{}, band);
    else launch(std::integral_constant<int, 4>{}, std::integral_constant<int, 8>{}, band);
  };
  auto threads = [](int band, int e) { return 64 + (((band + e - 1) / e + 63) & ~63); };
  if (t.dkl + t.dku > 4 * SOLVE_MAX_TAIL) {
    set_error("direct solver: band too wide for the solve kernels");
    return PT_ERR_UNSUPPORTED;
  }
  run(t.dkl, [&](auto e, auto d, int band) {
    constexpr int E = decltype(e)::value, D = decltype(d)::value;
    hipLaunchKernelGGL((k_band_forward<E, D>), dim3(1), dim3(threads(band, E)), 0, c.stream, c.dAB, c.dipiv, c.dB,
                       t.dn, t.dkl, t.dku);
  });
  run(t.dkl + t.dku, [&](auto e, auto d, int band) {
    constexpr int E = decltype(e)::value, D = decltype(d)::value;
    hipLaunchKernelGGL((k_band_backward<E, D>), dim3(1), dim3(threads(band, E)), 0, c.stream, c.dAB, c.dB, t.dn,
                       t.dkl, t.dku);
  });
  dim3 b16(64, 4), g((t.nx + 7 + 63) / 64, (t.nz + 7 + 3) / 4);
  hipLaunchKernelGGL(k_sf_scatter, g, b16, 0, c.stream, a, c.dB, c.SF);
  c.solves++;
  return PT_OK;
}

// update_velocities' iterate=0 branch (PS/momentum.f90:175-179) with the time
// loop's build at tstep=0 (PS/main.f90:247-251): the matrix is built on the
// first solve and, for ivis >= 1, on every solve
int solve_direct(Context& c) {
  if (!c.direct_built || c.P.ivis >= 1) PT_TRY(build_sf_matrix(c));
  return solve_sf_equation(c);
}

}  // namespace pt
