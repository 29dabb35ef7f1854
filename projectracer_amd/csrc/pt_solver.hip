// pt_solver.hip -- stream-function multigrid on gfx950.
//
// Kernels (one HIP kernel per reference loop nest or fused group):
//   k_sweep<R>      several RKC1 stages per launch on LDS tiles: stream_derivatives
//                   + stream_space + stage update + enforceBCs_stream (ghost
//                   write-through), and the residual after the last one
//                                     (PS/iterative_solver.f90:973-1018, 890-911,
//                                      1561-1597, 1616-1664)
//   k_residual<R>   stream_derivatives + compute_residual with per-block |r| sums
//                                      (PS/iterative_solver.f90:415-448)
//   k_restrict      full weighting     (PS/iterative_solver.f90:1107-1145)
//   k_prolong       bilinear prolongation + BCs (PS/iterative_solver.f90:343-396)
//   k_rhs1          compute_RHS level 1 (PS/iterative_solver.f90:1075-1101)
//   k_visf / k_vis_* viscosity hierarchy (PS/rheology.f90:2-23, PS/smoother.f90:454-580,
//                   PS/iterative_solver.f90:472-690, 1147-1211)
//   k_coarse_*      banded coarse operator, DGBEQU row scaling, DGBTF2 LU on one
//                   wavefront, and the solve (DGBTRS) as a dense interior operator
//                   built once per factorization (PS/iterative_solver.f90:1701-1887),
//                   applied by k_coarse_apply (FP64) or k_coarse_apply_wg (mixed)
//   k_velocities    compute_velocities + velocityBCs (PS/momentum.f90:655-710,
//                   PS/composition.f90:1295-1325)
// FP64 kernels are compiled without FMA contraction so each point is
// evaluated in the reference's operation order.
#include <cmath>
#include <cstring>
#include <algorithm>
#include <type_traits>
#include <vector>
#include "pt_internal.hpp"
#include "pt_quotient.hpp"

namespace pt {

#define IDX(i, k, pitch) ((long)((k) + 3) * (pitch) + ((i) + 3))

// ---------------------------------------------------------------------------
// stencil evaluation of stream_space on an LDS tile
// ---------------------------------------------------------------------------
template <typename R>
struct StageArgs {
  const R* Sx;      // the field the operator is applied to
  const R *vis, *vxm, *vxz, *vx, *vz, *rhs, *dts;
  int n, m, pitch;
  R sz;             // ghost sign in z (free-slip -1, rigid +1)
  R dr2, dr3, dr4, ds2, ds3, ds4, drds, dr2ds, drds2, dr2ds2;
  R rdr2, rdr3, rdr4, rds2, rds3, rds4, rdrds, rdr2ds, rdrds2, rdr2ds2;
  R D1[5], D2[5], D3[7], D4[7];
  R Drs[5][5], Drss[5][5], Drrs[5][5], Drrss[5][5];
};

// Accumulation in the reference's order: separate multiply and add for the
// FP64 path (bit-faithful); fused multiply-add for the FP32 smoother.
__device__ __forceinline__ double acc_(double s, double c, double v) { return s + c * v; }
__device__ __forceinline__ float acc_(float s, float c, float v) { return __fmaf_rn(c, v, s); }
// derivative scaling: FP64 divides by the grid power as the reference does;
// FP32 multiplies by the precomputed reciprocal
__device__ __forceinline__ double scale_(double s, double d, double rd) { (void)rd; return s / d; }
__device__ __forceinline__ float scale_(float s, float d, float rd) { (void)d; return s * rd; }

constexpr int TX = 64, TZ = 8, PZ = 1;
constexpr size_t SMALL_LDS_BYTES = 160 * 1024;
constexpr size_t SWEEP_LDS_BYTES = SMALL_LDS_BYTES - 4096;   // two iterates, beside k_sweep's static arrays
constexpr int TW = TX + 6, TH = TZ * PZ + 6;
constexpr int TILE_PER = (TH * TW + TX * TZ - 1) / (TX * TZ);   // tile elements per thread

// pointwise operands of stream_space at one point (read once per launch)
template <typename R>
struct PointCoef {
  R rhs, vis, vxm, vxz, vx, vz;
};

template <typename R, bool IV0>
__device__ __forceinline__ PointCoef<R> load_pc(const StageArgs<R>& a, long g) {
  PointCoef<R> c;
  c.rhs = a.rhs[g];
  c.vis = a.vis[g];
  if constexpr (!IV0) {
    c.vxm = a.vxm[g]; c.vxz = a.vxz[g]; c.vx = a.vx[g]; c.vz = a.vz[g];
  } else {
    c.vxm = c.vxz = c.vx = c.vz = (R)0;
  }
  return c;
}

// stream_derivatives (uniform grid) + stream_space at one point, reference
// summation order per derivative, zero stencil weights skipped.  `at(b, q)`
// reads psi(i+q, k+b).  With IV0 (isoviscous, eta_x = eta_z = eta_xz =
// eta_xx-eta_zz = 0) only the three derivatives stream_space uses are formed;
// each is accumulated exactly as in the general case.
template <typename R, bool IV0, typename At>
__device__ __forceinline__ R stream_space_pt(At at, const StageArgs<R>& a, const PointCoef<R>& pc) {
  R sxx = 0, szz = 0, sxxx = 0, szzz = 0, sxxxx = 0, szzzz = 0;
  if constexpr (!IV0) {
#pragma unroll
    for (int q = -2; q <= 2; q++) sxx = acc_(sxx, a.D2[q + 2], at(0, q));
#pragma unroll
    for (int q = -3; q <= 3; q++) if (q != 0) sxxx = acc_(sxxx, a.D3[q + 3], at(0, q));
  }
#pragma unroll
  for (int q = -3; q <= 3; q++) sxxxx = acc_(sxxxx, a.D4[q + 3], at(0, q));
  if constexpr (!IV0) {
#pragma unroll
    for (int q = -2; q <= 2; q++) szz = acc_(szz, a.D2[q + 2], at(q, 0));
#pragma unroll
    for (int q = -3; q <= 3; q++) if (q != 0) szzz = acc_(szzz, a.D3[q + 3], at(q, 0));
  }
#pragma unroll
  for (int q = -3; q <= 3; q++) szzzz = acc_(szzzz, a.D4[q + 3], at(q, 0));
  R sxz = 0, sxxz = 0, sxzz = 0, sxxzz = 0;
#pragma unroll
  for (int b = -2; b <= 2; b++)
#pragma unroll
    for (int q = -2; q <= 2; q++) {
      R v = at(b, q);
      if constexpr (!IV0) {
        if (b != 0 && q != 0) sxz = acc_(sxz, a.Drs[b + 2][q + 2], v);
        if (b != 0) sxxz = acc_(sxxz, a.Drrs[b + 2][q + 2], v);
        if (q != 0) sxzz = acc_(sxzz, a.Drss[b + 2][q + 2], v);
      }
      sxxzz = acc_(sxxzz, a.Drrss[b + 2][q + 2], v);
    }
  R SFxxxx = scale_(sxxxx, a.dr4, a.rdr4), SFzzzz = scale_(szzzz, a.ds4, a.rds4);
  R SFxxzz = scale_(sxxzz, a.dr2ds2, a.rdr2ds2);
  R sv;
  if constexpr (IV0) {
    R t2 = pc.vis * (SFxxxx + SFzzzz + (R)2 * SFxxzz);
    sv = t2 - pc.rhs;
  } else {
    R SFxx = scale_(sxx, a.dr2, a.rdr2), SFxxx = scale_(sxxx, a.dr3, a.rdr3);
    R SFzz = scale_(szz, a.ds2, a.rds2), SFzzz = scale_(szzz, a.ds3, a.rds3);
    R SFxz = scale_(sxz, a.drds, a.rdrds), SFxxz = scale_(sxxz, a.dr2ds, a.rdr2ds);
    R SFxzz = scale_(sxzz, a.drds2, a.rdrds2);
    R t1 = pc.vxm * (SFxx - SFzz);
    R t2 = pc.vis * (SFxxxx + SFzzzz + (R)2 * SFxxzz);
    R t4 = ((R)4 * pc.vxz) * SFxz;
    R t5 = ((R)2 * pc.vx) * (SFxxx + SFxzz);
    R t6 = ((R)2 * pc.vz) * (SFzzz + SFxxz);
    sv = t1 + t2 + t4 + t5 + t6 - pc.rhs;
  }
  return -sv;
}

template <typename R>
struct TileRegs {
  R v[TILE_PER];
  bool in[TILE_PER];
};
// the thread's tile elements, loaded in two phases so that every global
// load of the launch (tile and pointwise operands) is in flight at once:
// tile_issue loads from addresses clamped to the stored range (so the loads
// are unconditional), tile_commit writes LDS, zero outside the level
template <typename R>
__device__ __forceinline__ TileRegs<R> tile_issue(const R* S, int i0, int k0, int n, int m, int pitch) {
  TileRegs<R> r;
  const int tid = threadIdx.y * TX + threadIdx.x;
#pragma unroll
  for (int u = 0; u < TILE_PER; u++) {
    const int idx = min(tid + u * TX * TZ, TH * TW - 1);
    const int rr = idx / TW, cc = idx - rr * TW;
    const int gi = i0 - 3 + cc, gk = k0 - 3 + rr;
    r.in[u] = gi <= n + 3 && gk <= m + 3;
    r.v[u] = S[IDX(min(gi, n + 3), min(gk, m + 3), pitch)];
  }
  return r;
}
template <typename R>
__device__ __forceinline__ void tile_commit(R (*t)[TW], const TileRegs<R>& r) {
  const int tid = threadIdx.y * TX + threadIdx.x;
#pragma unroll
  for (int u = 0; u < TILE_PER; u++) {
    const int idx = tid + u * TX * TZ;
    if (idx < TH * TW) {
      const int rr = idx / TW, cc = idx - rr * TW;
      t[rr][cc] = r.in[u] ? r.v[u] : (R)0;
    }
  }
}

// store Y(i,k) and its ghost images (enforceBCs_stream: antisymmetric side
// walls, sz-symmetric top/bottom, psi = 0 on the walls which are never written)
template <typename R>
__device__ __forceinline__ void store_with_ghosts(R* Y, int i, int k, int n, int m, int pitch, R y, R sz) {
  Y[IDX(i, k, pitch)] = y;
  bool lo_i = i <= 3, hi_i = i >= n - 3, lo_k = k <= 3, hi_k = k >= m - 3;
  if (lo_i) Y[IDX(-i, k, pitch)] = -y;
  if (hi_i) Y[IDX(2 * n - i, k, pitch)] = -y;
  if (lo_k) {
    Y[IDX(i, -k, pitch)] = sz * y;
    if (lo_i) Y[IDX(-i, -k, pitch)] = -(sz * y);
    if (hi_i) Y[IDX(2 * n - i, -k, pitch)] = -(sz * y);
  }
  if (hi_k) {
    Y[IDX(i, 2 * m - k, pitch)] = sz * y;
    if (lo_i) Y[IDX(-i, 2 * m - k, pitch)] = -(sz * y);
    if (hi_i) Y[IDX(2 * n - i, 2 * m - k, pitch)] = -(sz * y);
  }
}

// residual(i,k) = stream_space(i,k,S); block partial sums of |residual|
template <typename R, bool IV0>
__global__ void __launch_bounds__(TX* TZ) k_residual(StageArgs<R> a, R* res, double* partial) {
  __shared__ R tile[TH][TW];
  __shared__ double red[TX * TZ];
  const int i0 = 1 + blockIdx.x * TX, k0 = 1 + blockIdx.y * TZ * PZ;
  const TileRegs<R> tr = tile_issue<R>(a.Sx, i0, k0, a.n, a.m, a.pitch);
  PointCoef<R> pc[PZ];
  const int i = i0 + threadIdx.x;
#pragma unroll
  for (int pz = 0; pz < PZ; pz++) {
    int k = k0 + threadIdx.y + pz * TZ;
    if (i > a.n - 1 || k > a.m - 1) continue;
    pc[pz] = load_pc<R, IV0>(a, IDX(i, k, a.pitch));
  }
  tile_commit<R>(tile, tr);
  __syncthreads();
  double acc = 0.0;
#pragma unroll
  for (int pz = 0; pz < PZ; pz++) {
    int k = k0 + threadIdx.y + pz * TZ;
    if (i > a.n - 1 || k > a.m - 1) continue;
    int ti = threadIdx.x + 3, tk = threadIdx.y + pz * TZ + 3;
    R F = stream_space_pt<R, IV0>([&](int b, int q) { return tile[tk + b][ti + q]; }, a, pc[pz]);
    res[IDX(i, k, a.pitch)] = F;
    acc = acc + fabs((double)F);
  }
  int tid = threadIdx.y * TX + threadIdx.x;
  red[tid] = acc;
  __syncthreads();
  for (int s = TX * TZ / 2; s > 0; s >>= 1) {
    if (tid < s) red[tid] = red[tid] + red[tid + s];
    __syncthreads();
  }
  if (tid == 0) partial[blockIdx.y * gridDim.x + blockIdx.x] = red[0];
}

// one RK1 smoothing iteration (RKC1=0, PS/iterative_solver.f90:1468-1485,
// :1503-1513) from F = stream_space(S0): psi = S0 + (c dt) F with the local
// step c = 2/(-lb-la+(lb-la) temp), la = -1, lb = -2 r^2/(1+r^2) from the
// point's eigenvalue ratio r (-2 where r is not below 1e99), c = 1 on the
// way up the cycle; then the ghost images (enforceBCs_stream).  Each thread
// reads and writes only its own interior point, so the update is in place.
__global__ void k_rk1_update(double* psi, const double* F, const double* dts, const double* ratio, int n, int m,
                             int pitch, double temp, int dir, double sz) {
  const int i = 1 + blockIdx.x * blockDim.x + threadIdx.x, k = 1 + blockIdx.y * blockDim.y + threadIdx.y;
  if (i > n - 1 || k > m - 1) return;
  const long g = IDX(i, k, pitch);
  double cc = 1.0;
  if (dir == 0) {
    const double la = -1.0, lb_user = -2.0, r = ratio[g];
    double lb = lb_user;
    if (r < 1.0e99) lb = lb_user * (r * r) / (1.0 + r * r);
    cc = 2.0 / (-lb - la + (lb - la) * temp);
  }
  const double y = psi[g] + (cc * dts[g]) * F[g];
  store_with_ghosts<double>(psi, i, k, n, m, pitch, y, sz);
}

// the RKC1 stage count and coefficients of a level's sweeps: the reference's
// nstageS everywhere, or s_coarse stages on the mixed path's levels >= 2
struct LevelRkc {
  int s;
  const double *mewt, *mew, *vv, *cc;
  double stability;
};
static LevelRkc level_rkc(const Context& c, int l, bool fp32) {
  const Tables& t = c.T;
  if (fp32 && l >= 2 && t.s_coarse >= 2) return {t.s_coarse, t.mewt_c, t.mew_c, t.vv_c, t.cc_c, t.RKC1_stability_c};
  return {c.P.nstageS, t.mewt, t.mew, t.vv, t.cc, t.RKC1_stability};
}
constexpr int SMALL_THREADS = 1024;

// ---------------------------------------------------------------------------
// RKC1 sweeps, several stages per launch.  A workgroup owns a core tile of a
// level and computes `ns` consecutive stages on it: the current iterate S1 is
// in LDS (two buffers, one barrier per stage) on the core widened by 3 points
// per evaluation, every point's S0, S2, dt_stream, RHS and viscosity
// coefficients stay in the registers of the thread that owns it, and stage t
// is evaluated on the core widened by 3 points per evaluation still to come,
// so tiles do not exchange anything within a launch (overlap points are
// computed by both neighbours).  A tile that covers the whole level takes the
// whole sweep in one launch.  Each thread owns RB vertically adjacent points
// of one column and reads their common neighbourhood once.  Per point the
// operations and their order are those of one stage per launch
// (stream_space_pt, or the factorised form below), so the results do not
// depend on the tiling.
// Bound by the issue of vector instructions, the overlap's among them, and by
// what a launch costs around them (window, barriers, start and end).  1024x256,
// general operator, FP32, by counters: level 1 (256 tiles, 3 stages) 13.6 us with
// 57% of the issue slots taken, LDS active 18%, 27 MB from and to HBM (its
// operands once: 12.5); levels 2 to 5 8.5, 6.5, 6.2 and 8.2 us with 37, 28, 24
// and 40% on the compute units they use.  FP64 isoviscous, level 1: 13.6 us, 42%.
// ---------------------------------------------------------------------------
constexpr int SWEEP_MAX_STAGES = 64;

// the distinct stencil weights: D1 and D3 are odd, D2 and D4 even, and the
// mixed ones are their products, so the signs are known at compile time and
// the 31 magnitudes stay in scalar registers
template <typename R>
struct SweepWeights {
  R d2[3], d3[3], d4[4];       // d3: offsets -1, -2, -3
  R rs[3], rrs[6], rss[6], rrss[6];
};

template <typename R>
struct SweepArgs {
  const R* S0;      // sweep start (pointwise; stencil source of stage 1)
  const R* Gcur;    // stage j0-1 (S0 when j0 = 1)
  const R* Gprev;   // stage j0-2 (an allocated level buffer also when j0 = 1)
  R* Ocur;          // the last stage on the core, with ghost images
  R* Oprev;         // the stage before it; null on the sweep's last launch
  R* res;           // RHS - L psi of the last stage on the core; null: not wanted
  const R *vis, *vxm, *vxz, *vx, *vz, *rhs, *dts;
  int n, m, pitch;
  int j0, ns;       // first stage (1-based) and number of stages
  int cw, ch, nbx;  // core size, tiles per row
  int w1, nrb, tcol;  // columns of the first stage's region, its blocks of RB rows, threads per block row
  R sz;
  R dr2, dr3, dr4, ds2, ds3, ds4, drds, dr2ds, drds2, dr2ds2;
  R rdr2, rdr3, rdr4, rds2, rds3, rds4, rdrds, rdr2ds, rdrds2, rdr2ds2;
  SweepWeights<R> w;
  R c0[SWEEP_MAX_STAGES], c1[SWEEP_MAX_STAGES], c2[SWEEP_MAX_STAGES], cf[SWEEP_MAX_STAGES];
};

template <bool PW2>
__device__ __forceinline__ float quot(float s, float d, float rd) { (void)d; return s * rd; }

// Sums of the derivatives at one point, updated row by row: row(b, e, x) adds
// the row b points above the point (e: its five values around the column;
// x: on the point's own row the values 3 columns away).  Called with b = -3
// .. 3 in order, every sum is accumulated in stream_space_pt's order.
// EV 0: general operator; 1: isoviscous; 2: isoviscous with psi_xxzz as
// D2_z(D2_x psi) (FP32 levels >= 2)
template <typename R, int EV>
struct PointSums {
  R sxx, szz, sxxx, szzz, sxxxx, szzzz, sxz, sxxz, sxzz, sxxzz;
  __device__ __forceinline__ void clear() {
    sxx = szz = sxxx = szzz = sxxxx = szzzz = sxz = sxxz = sxzz = sxxzz = (R)0;
  }
  template <int B>
  __device__ __forceinline__ void row(const SweepWeights<R>& w, const R* e, R xl, R xr, R d2x) {
    constexpr int ab = B < 0 ? -B : B;
    if constexpr (B == 0) {
      const R at[7] = {xl, e[0], e[1], e[2], e[3], e[4], xr};
      if constexpr (EV == 0) {
#pragma unroll
        for (int q = -2; q <= 2; q++) sxx = acc_(sxx, w.d2[abs(q)], at[q + 3]);
#pragma unroll
        for (int q = -3; q <= 3; q++) if (q != 0) sxxx = acc_(sxxx, q < 0 ? w.d3[-q - 1] : -w.d3[q - 1], at[q + 3]);
      }
      if constexpr (EV == 2) sxxxx = w.d4[3] * xl;
      else sxxxx = acc_(sxxxx, w.d4[3], xl);
#pragma unroll
      for (int q = -2; q <= 3; q++) sxxxx = acc_(sxxxx, w.d4[abs(q)], at[q + 3]);
    }
    if constexpr (EV == 0) {
      if constexpr (ab <= 2) szz = acc_(szz, w.d2[ab], e[2]);
      if constexpr (B != 0) szzz = acc_(szzz, B < 0 ? w.d3[ab - 1] : -w.d3[ab - 1], e[2]);
    }
    szzzz = acc_(szzzz, w.d4[ab], e[2]);
    if constexpr (ab <= 2 && EV == 2) sxxzz = acc_(sxxzz, w.d2[ab], d2x);
    if constexpr (ab <= 2 && EV != 2) {
#pragma unroll
      for (int q = -2; q <= 2; q++) {
        const R v = e[q + 2];
        const int aq = abs(q);
        if constexpr (EV == 0) {
          // D1 is odd: negative where exactly one offset is
          if (B != 0 && q != 0) sxz = acc_(sxz, (B < 0) != (q < 0) ? -w.rs[ab + aq - 2] : w.rs[ab + aq - 2], v);
          if (B != 0) sxxz = acc_(sxxz, B < 0 ? w.rrs[(ab - 1) * 3 + aq] : -w.rrs[(ab - 1) * 3 + aq], v);
          if (q != 0) sxzz = acc_(sxzz, q < 0 ? w.rss[(aq - 1) * 3 + ab] : -w.rss[(aq - 1) * 3 + ab], v);
        }
        const int lo = ab < aq ? ab : aq, hi = ab < aq ? aq : ab;
        sxxzz = acc_(sxxzz, w.rrss[lo == 0 ? hi : lo == 1 ? 2 + hi : 5], v);
      }
    }
  }
  // RHS - L psi from the sums (stream_space)
  template <bool PW2>
  __device__ __forceinline__ R value(const SweepArgs<R>& a, const PointCoef<R>& pc) const {
    if constexpr (EV == 2) {
      const R lap2 = sxxxx * a.rdr4 + szzzz * a.rds4 + (R)2 * (sxxzz * a.rdr2ds2);
      return pc.rhs - pc.vis * lap2;
    } else {
      const R SFxxxx = quot<PW2>(sxxxx, a.dr4, a.rdr4), SFzzzz = quot<PW2>(szzzz, a.ds4, a.rds4);
      const R SFxxzz = quot<PW2>(sxxzz, a.dr2ds2, a.rdr2ds2);
      const R t2 = pc.vis * (SFxxxx + SFzzzz + (R)2 * SFxxzz);
      if constexpr (EV == 1) return -(t2 - pc.rhs);
      const R SFxx = quot<PW2>(sxx, a.dr2, a.rdr2), SFxxx = quot<PW2>(sxxx, a.dr3, a.rdr3);
      const R SFzz = quot<PW2>(szz, a.ds2, a.rds2), SFzzz = quot<PW2>(szzz, a.ds3, a.rds3);
      const R SFxz = quot<PW2>(sxz, a.drds, a.rdrds), SFxxz = quot<PW2>(sxxz, a.dr2ds, a.rdr2ds);
      const R SFxzz = quot<PW2>(sxzz, a.drds2, a.rdrds2);
      const R t1 = pc.vxm * (SFxx - SFzz);
      const R t4 = ((R)4 * pc.vxz) * SFxz;
      const R t5 = ((R)2 * pc.vx) * (SFxxx + SFxzz);
      const R t6 = ((R)2 * pc.vz) * (SFzzz + SFxxz);
      return -(t1 + t2 + t4 + t5 + t6 - pc.rhs);
    }
  }
};

// rows ROW .. RB+2 around a thread's RB points (S: the first point's place in
// LDS), each read once and added to every point it belongs to; s1 receives
// the points' own values, and a point's F = RHS - L psi is formed as soon as
// its last row is in, so that few sums and rows are live at a time
template <typename R, int EV, int RB, bool PW2, int ROW>
__device__ __forceinline__ void sweep_rows(const R* S, int W, const SweepArgs<R>& a, const PointCoef<R>* pc,
                                           PointSums<R, EV>* ps, R* s1, R* F) {
  if constexpr (ROW <= RB + 2) {
    constexpr bool five = ROW >= -2 && ROW <= RB + 1, own = ROW >= 0 && ROW < RB;
    R e[5], xl = 0, xr = 0, d2x = 0;
    const R* q = S + ROW * W;
    e[2] = q[0];
    if constexpr (five) { e[0] = q[-2]; e[1] = q[-1]; e[3] = q[1]; e[4] = q[2]; }
    if constexpr (own) { xl = q[-3]; xr = q[3]; s1[ROW] = e[2]; }
    if constexpr (EV == 2 && five) {
#pragma unroll
      for (int c = 0; c < 5; c++) d2x = acc_(d2x, a.w.d2[abs(c - 2)], e[c]);
    }
    auto add = [&](auto rc) {
      constexpr int r = decltype(rc)::value, B = ROW - r;
      if constexpr (r < RB && B >= -3 && B <= 3) {
        if constexpr (B == -3) ps[r].clear();
        ps[r].template row<B>(a.w, e, xl, xr, d2x);
        if constexpr (B == 3) F[r] = ps[r].template value<PW2>(a, pc[r]);
      }
    };
    add(std::integral_constant<int, 0>{});
    add(std::integral_constant<int, 1>{});
    add(std::integral_constant<int, 2>{});
    add(std::integral_constant<int, 3>{});
    sweep_rows<R, EV, RB, PW2, ROW + 1>(S, W, a, pc, ps, s1, F);
  }
}

template <typename R, int EV, int RB, int NT, bool PW2>
__global__ void __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(NT / 256, NT / 256))) k_sweep(SweepArgs<R> a) {
  static_assert(RB <= 4, "sweep_rows handles up to 4 points per thread");
  extern __shared__ unsigned char smem_raw[];
  const int n = a.n, m = a.m, p = a.pitch, ns = a.ns;
  const int nev = ns + (a.res ? 1 : 0);   // evaluations of the operator
  const int bx = blockIdx.x % a.nbx, bz = blockIdx.x / a.nbx;
  const int cx0 = 1 + bx * a.cw, cx1 = min(cx0 + a.cw, n);   // core [cx0, cx1) x [cz0, cz1)
  const int cz0 = 1 + bz * a.ch, cz1 = min(cz0 + a.ch, m);
  // LDS window: the first evaluation's region and 3 points around it (4
  // where it starts at a wall), rows padded to whole blocks of RB
  const int x1 = max(1, cx0 - 3 * (nev - 1)), z1 = max(1, cz0 - 3 * (nev - 1));
  const int ilo = max(-3, cx0 - 3 * nev), klo = max(-3, cz0 - 3 * nev);
  const int W = a.w1 + 8, rows = a.nrb * RB + 8, ne = W * rows;
  R* const buf = reinterpret_cast<R*>(smem_raw);
  const int tid = threadIdx.x, nthr = blockDim.x;
  __shared__ R coef[4][SWEEP_MAX_STAGES];
  if (tid < SWEEP_MAX_STAGES) {   // at least one wavefront
    const int j = min(a.j0 + tid, SWEEP_MAX_STAGES - 1);
    coef[0][tid] = a.c0[j]; coef[1][tid] = a.c1[j]; coef[2][tid] = a.c2[j]; coef[3][tid] = a.cf[j];
  }
  // the window: each batch's loads are issued before its LDS writes
  constexpr int FB = 4;
  for (int e0 = tid; e0 < ne; e0 += FB * nthr) {
    R v[FB];
#pragma unroll
    for (int u = 0; u < FB; u++) {
      const int e = min(e0 + u * nthr, ne - 1);
      const int rr = e / W, cc = e - rr * W;
      v[u] = a.Gcur[IDX(min(ilo + cc, n + 3), min(klo + rr, m + 3), p)];
    }
#pragma unroll
    for (int u = 0; u < FB; u++) {
      const int e = e0 + u * nthr;
      if (e < ne) {
        buf[e] = v[u];
        buf[ne + e] = (R)0;   // the walls' psi = 0 and the ghosts of the other buffer
      }
    }
  }
  // this thread's column and row block; its points' operands, from clamped
  // (valid) points
  const int rb = tid / a.tcol, ic = x1 + (tid - rb * a.tcol);
  const int k0 = z1 + rb * RB;
  const bool col = rb < a.nrb && tid - rb * a.tcol < a.w1 && ic <= n - 1;
  R s0v[RB], pv[RB], yv[RB], dtv[RB];
  PointCoef<R> pc[RB];
#pragma unroll
  for (int r = 0; r < RB; r++) {
    const long g = IDX(min(ic, n - 1), min(k0 + r, m - 1), p);
    s0v[r] = a.S0[g];
    pv[r] = a.Gprev[g];
    dtv[r] = a.dts[g];
    pc[r].rhs = a.rhs[g];
    pc[r].vis = a.vis[g];
    if constexpr (EV == 0) {
      pc[r].vxm = a.vxm[g]; pc[r].vxz = a.vxz[g]; pc[r].vx = a.vx[g]; pc[r].vz = a.vz[g];
    }
    yv[r] = (R)0;
  }
  __syncthreads();
  int at0 = 0;   // LDS offset of the current iterate
  const int own = (k0 - klo) * W + (ic - ilo);
  // LDS offsets of the points' ghost images (antisymmetric side walls,
  // sz-symmetric top and bottom), 0 where there is none.  On levels of at
  // least 7 cells a point has at most one image per direction; smaller ones
  // take the general form
  const bool tiny = n < 7 || m < 7;
  int gx = 0, gz[RB];
  if (ic <= 3 && -ic >= ilo) gx = -2 * ic;
  else if (ic >= n - 3 && 2 * n - ic < ilo + W) gx = 2 * (n - ic);
#pragma unroll
  for (int r = 0; r < RB; r++) {
    const int k = k0 + r;
    gz[r] = 0;
    if (k <= 3 && -k >= klo) gz[r] = -2 * k * W;
    else if (k >= m - 3 && 2 * m - k < klo + rows) gz[r] = 2 * (m - k) * W;
  }
  for (int t = 0; t < nev; t++) {
    const int h = 3 * (nev - 1 - t);
    if (col && ic >= cx0 - h && ic < cx1 + h && k0 < cz1 + h && k0 + RB > cz0 - h) {
      // the stage's coefficients: from LDS with the window, or (FP64 general
      // operator, short of vector registers) scalar
      R cc0, cc1, cc2, cf;
      if constexpr (sizeof(R) == 8 && EV == 0) {
        const int j = a.j0 + t;
        cc0 = a.c0[j]; cc1 = a.c1[j]; cc2 = a.c2[j]; cf = a.cf[j];
      } else {
        cc0 = coef[0][t]; cc1 = coef[1][t]; cc2 = coef[2][t]; cf = coef[3][t];
      }
      R F[RB], s1[RB];
      PointSums<R, EV> ps[RB];
      sweep_rows<R, EV, RB, PW2, -3>(buf + at0 + own, W, a, pc, ps, s1, F);
      if (t == ns) {
#pragma unroll
        for (int r = 0; r < RB; r++) s0v[r] = F[r];   // the residual
      } else {
        R* const out = buf + (ne - at0) + own;
#pragma unroll
        for (int r = 0; r < RB; r++) {
          R y;
          if (a.j0 + t == 1) y = s0v[r] + (cf * dtv[r]) * F[r];
          else y = ((cc0 * s0v[r] + cc1 * s1[r]) + cc2 * pv[r]) + ((cf * dtv[r]) * F[r]);
          pv[r] = s1[r];
          yv[r] = y;
          if (t < nev - 1 && k0 + r <= m - 1) out[r * W] = y;
        }
        if (t < nev - 1) {
#pragma unroll
          for (int r = 0; r < RB; r++) {
            if (k0 + r > m - 1) continue;
            const R y = yv[r], z = a.sz * y;
            const int at = r * W;
            if (tiny) {
              int i = ic, k = k0 + r;
              asm volatile("" : "+v"(i), "+v"(k));   // not kept in registers between stages
              const int ol = at - 2 * i, orr = at + 2 * (n - i), ob = -2 * k * W, ot = 2 * (m - k) * W;
              const bool gl = i <= 3 && -i >= ilo, gr = i >= n - 3 && 2 * n - i < ilo + W;
              if (gl) out[ol] = -y;
              if (gr) out[orr] = -y;
              if (k <= 3 && -k >= klo) {
                out[at + ob] = z;
                if (gl) out[ol + ob] = -z;
                if (gr) out[orr + ob] = -z;
              }
              if (k >= m - 3 && 2 * m - k < klo + rows) {
                out[at + ot] = z;
                if (gl) out[ol + ot] = -z;
                if (gr) out[orr + ot] = -z;
              }
              continue;
            }
            if (gx) out[at + gx] = -y;
            if (gz[r]) {
              out[at + gz[r]] = z;
              if (gx) out[at + gz[r] + gx] = -z;
            }
          }
        }
      }
    }
    if (t + 1 < nev) __syncthreads();
    at0 = ne - at0;
  }
  if (!col || ic < cx0 || ic >= cx1) return;
#pragma unroll
  for (int r = 0; r < RB; r++) {
    const int k = k0 + r;
    if (k < cz0 || k >= cz1) continue;
    store_with_ghosts<R>(a.Ocur, ic, k, n, m, p, yv[r], a.sz);
    if (a.Oprev) store_with_ghosts<R>(a.Oprev, ic, k, n, m, p, pv[r], a.sz);
    if (a.res) a.res[IDX(ic, k, p)] = s0v[r];
  }
}

// ---------------------------------------------------------------------------
// coarsest grid as a dense operator: G(:,q) = A^-1 (RowB(q) e_q) from the band
// LU factors (DGBTRS's forward and backward sweeps on a unit vector),
// interior unknowns only.  One wavefront per column q, the work vector in
// LDS: each sweep step's band updates are independent across rows and
// spread over the lanes; every element sees the same operations in the same
// order as the sequential sweep.
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(64) k_coarse_inverse(const double* ab, const int32_t* ipiv, const double* RowB,
                                                       double* G, int n, int kl, int ku, int nxc, int nzc) {
  extern __shared__ double Y[];   // n entries
  const int nci = (nxc - 1) * (nzc - 1);
  const int t = blockIdx.x, lane = threadIdx.x;
  const int ld = 2 * kl + ku + 1, kd = ku + kl + 1, N = nzc + 1;
  const int iq = 1 + t % (nxc - 1), kq = 1 + t / (nxc - 1);
  const int q = N * iq + kq + 1;   // 1-based unknown index
#define AB(r, c) ab[(long)((c) - 1) * ld + ((r) - 1)]
  for (int pp = lane; pp < n; pp += 64) Y[pp] = 0.0;
  __syncthreads();
  if (lane == 0) Y[q - 1] = RowB[q - 1];
  __syncthreads();
  for (int j = 1; j <= n - 1; j++) {
    const int lm = min(kl, n - j);
    const int l = ipiv[j - 1];
    if (l != j && lane == 0) {
      double tmp = Y[l - 1];
      Y[l - 1] = Y[j - 1];
      Y[j - 1] = tmp;
    }
    __syncthreads();
    const double temp = -1.0 * Y[j - 1];
    for (int u = 1 + lane; u <= lm; u += 64) Y[j + u - 1] = Y[j + u - 1] + AB(kd + u, j) * temp;
    __syncthreads();
  }
  const int kk = kl + ku, kp1 = kk + 1;
  for (int j = n; j >= 1; j--) {
    const double bj = Y[j - 1];
    if (bj != 0.0) {
      const int l = kp1 - j;
      const double x = bj / AB(kp1, j);
      const int lo = max(1, j - kk);
      __syncthreads();   // every lane has read Y(j) before it is replaced
      if (lane == 0) Y[j - 1] = x;
      for (int i = j - 1 - lane; i >= lo; i -= 64) Y[i - 1] = Y[i - 1] - x * AB(l + i, j);
    }
    __syncthreads();
  }
  for (int pi = lane; pi < nci; pi += 64) {
    const int ip = 1 + pi % (nxc - 1), kp = 1 + pi / (nxc - 1);
    G[(long)t * nci + pi] = Y[N * ip + kp];
  }
#undef AB
}

// coarse correction: err(p) = sum_q G(p,q) rhs(q), fixed order in q
template <typename RI, typename RO>
__global__ void k_coarse_apply(const double* G, const RI* rhs, RO* err, int nxc, int nzc, int pitch, RO sz) {
  extern __shared__ double rv[];
  const int nci = (nxc - 1) * (nzc - 1);
  for (int q = threadIdx.x; q < nci; q += blockDim.x) {
    int iq = 1 + q % (nxc - 1), kq = 1 + q / (nxc - 1);
    rv[q] = (double)rhs[IDX(iq, kq, pitch)];
  }
  __syncthreads();
  int pi = blockIdx.x * blockDim.x + threadIdx.x;
  if (pi >= nci) return;
  double acc = 0.0;
  for (int q = 0; q < nci; q++) acc = acc + G[(long)q * nci + pi] * rv[q];
  int ip = 1 + pi % (nxc - 1), kp = 1 + pi / (nxc - 1);
  store_with_ghosts<RO>(err, ip, kp, nxc, nzc, pitch, (RO)acc, sz);
}

// ---------------------------------------------------------------------------
// reductions: fixed-shape block partials then one block in fixed order
// ---------------------------------------------------------------------------
__global__ void k_reduce2d(const double* d, int n, int m, int pitch, int off, int op, double* partial) {
  __shared__ double red[256];
  int tid = threadIdx.x;
  const bool sum = op == RED_SUM_ABS || op == RED_SUM_SQ;
  double acc = sum ? 0.0 : (op == RED_MAX ? -INFINITY : INFINITY);
  long total = (long)n * m;
  for (long idx = (long)blockIdx.x * 256 + tid; idx < total; idx += (long)gridDim.x * 256) {
    int i = (int)(idx % n), k = (int)(idx / n);
    double v = d[(long)(k + off) * pitch + (i + off)];
    if (op == RED_SUM_ABS) acc = acc + fabs(v);
    else if (op == RED_SUM_SQ) acc = acc + v * v;
    else if (op == RED_MAX) acc = fmax(acc, v);
    else acc = fmin(acc, v);
  }
  red[tid] = acc;
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if (tid < s) {
      double x = red[tid], y = red[tid + s];
      red[tid] = sum ? x + y : (op == RED_MAX ? fmax(x, y) : fmin(x, y));
    }
    __syncthreads();
  }
  if (tid == 0) partial[blockIdx.x] = red[0];
}
__global__ void k_reduce_final(const double* partial, int nb, int op, double* out) {
  __shared__ double red[256];
  int tid = threadIdx.x;
  const bool sum = op == RED_SUM_ABS || op == RED_SUM_SQ;
  double acc = sum ? 0.0 : (op == RED_MAX ? -INFINITY : INFINITY);
  for (int j = tid; j < nb; j += 256) {
    double v = partial[j];
    acc = sum ? acc + v : (op == RED_MAX ? fmax(acc, v) : fmin(acc, v));
  }
  red[tid] = acc;
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if (tid < s) {
      double x = red[tid], y = red[tid + s];
      red[tid] = sum ? x + y : (op == RED_MAX ? fmax(x, y) : fmin(x, y));
    }
    __syncthreads();
  }
  if (tid == 0) *out = red[0];
}
int reduce_to_host(Context& c, const double* d, int n, int m, int pitch, int off, RedOp op, double* out) {
  long total = (long)n * m;
  int nb = (int)std::min<long>(1024, (total + 255) / 256);
  if (nb < 1) nb = 1;
  hipLaunchKernelGGL(k_reduce2d, dim3(nb), dim3(256), 0, c.stream, d, n, m, pitch, off, (int)op, c.red);
  hipLaunchKernelGGL(k_reduce_final, dim3(1), dim3(256), 0, c.stream, c.red, nb, (int)op, c.red_out);
  PT_HIP(hipMemcpyAsync(c.h_red, c.red_out, sizeof(double), hipMemcpyDeviceToHost, c.stream));
  PT_HIP(hipStreamSynchronize(c.stream));
  *out = c.h_red[0];
  return PT_OK;
}

// ---------------------------------------------------------------------------
// grid transfer
// ---------------------------------------------------------------------------
// restrict / restrict_coefficients: out(i,k) (coarse interior) from in (fine)
template <typename RI>
__device__ __forceinline__ double restrict_val(const RI* in, int fpitch, int i, int k) {
  int ii = 2 * i, kk = 2 * k;
  double corners = ((double)in[IDX(ii - 1, kk - 1, fpitch)] + (double)in[IDX(ii - 1, kk + 1, fpitch)] +
                    (double)in[IDX(ii + 1, kk + 1, fpitch)] + (double)in[IDX(ii + 1, kk - 1, fpitch)]) / 16.0;
  double sides = ((double)in[IDX(ii - 1, kk, fpitch)] + (double)in[IDX(ii, kk - 1, fpitch)] +
                  (double)in[IDX(ii + 1, kk, fpitch)] + (double)in[IDX(ii, kk + 1, fpitch)]) / 8.0;
  double centre = (double)in[IDX(ii, kk, fpitch)] / 4.0;
  return corners + sides + centre;
}
template <typename RI, typename RO>
__device__ __forceinline__ void restrict_pt(const RI* in, int fpitch, RO* out, int cpitch, int i, int k) {
  out[IDX(i, k, cpitch)] = (RO)restrict_val<RI>(in, fpitch, i, k);
}
template <typename RI, typename RO>
__global__ void k_restrict(const RI* in, int fpitch, RO* out, int cn, int cm, int cpitch) {
  int i = 1 + blockIdx.x * blockDim.x + threadIdx.x, k = 1 + blockIdx.y * blockDim.y + threadIdx.y;
  if (i > cn - 1 || k > cm - 1) return;
  restrict_pt<RI, RO>(in, fpitch, out, cpitch, i, k);
}

// prolong: fine += bilinear(coarse), then the fine ghosts (four parity classes
// of PS/iterative_solver.f90:364-394 evaluated per fine point)
template <typename RC, typename RF>
__device__ __forceinline__ RF prolong_val(const RC* ec, int cpitch, const RF* ef, int fpitch, int i, int k) {
  RF add;
  bool ie = (i % 2) == 0, ke = (k % 2) == 0;
  if (ie && ke) add = (RF)ec[IDX(i / 2, k / 2, cpitch)];
  else if (ie && !ke) add = ((RF)ec[IDX(i / 2, (k - 1) / 2, cpitch)] + (RF)ec[IDX(i / 2, (k + 1) / 2, cpitch)]) / (RF)2;
  else if (!ie && ke) add = ((RF)ec[IDX((i - 1) / 2, k / 2, cpitch)] + (RF)ec[IDX((i + 1) / 2, k / 2, cpitch)]) / (RF)2;
  else
    add = ((RF)ec[IDX((i - 1) / 2, (k - 1) / 2, cpitch)] + (RF)ec[IDX((i + 1) / 2, (k - 1) / 2, cpitch)] +
           (RF)ec[IDX((i + 1) / 2, (k + 1) / 2, cpitch)] + (RF)ec[IDX((i - 1) / 2, (k + 1) / 2, cpitch)]) / (RF)4;
  return ef[IDX(i, k, fpitch)] + add;
}
template <typename RC, typename RF>
__device__ __forceinline__ void prolong_pt(const RC* ec, int cpitch, RF* ef, int fn, int fm, int fpitch, RF sz, int i,
                                           int k) {
  store_with_ghosts<RF>(ef, i, k, fn, fm, fpitch, prolong_val<RC, RF>(ec, cpitch, ef, fpitch, i, k), sz);
}
template <typename RC, typename RF>
__global__ void k_prolong(const RC* ec, int cpitch, RF* ef, int fn, int fm, int fpitch, RF sz) {
  int i = 1 + blockIdx.x * blockDim.x + threadIdx.x, k = 1 + blockIdx.y * blockDim.y + threadIdx.y;
  if (i > fn - 1 || k > fm - 1) return;
  prolong_pt<RC, RF>(ec, cpitch, ef, fn, fm, fpitch, sz, i, k);
}

// coarse correction err = G rhs by one workgroup (mixed path): the column
// range is split in CA_SEG fixed segments, each summed in order by its own
// thread group (loads issued 8 at a time), and the segment sums are added in
// segment order.  LDS: (1 + CA_SEG) * nci doubles.
constexpr int CA_SEG = 4, CA_ROWS = SMALL_THREADS / CA_SEG;
__device__ __forceinline__ void coarse_apply_wg(const double* G, const float* rhs, float* err, int nxc, int nzc,
                                                int pitch, float sz, double* sm) {
  const int nci = (nxc - 1) * (nzc - 1);
  double* rv = sm;
  double* part = sm + nci;
  for (int q = threadIdx.x; q < nci; q += SMALL_THREADS) {
    int iq = 1 + q % (nxc - 1), kq = 1 + q / (nxc - 1);
    rv[q] = (double)rhs[IDX(iq, kq, pitch)];
  }
  __syncthreads();
  const int seg = threadIdx.x / CA_ROWS, qs = (nci + CA_SEG - 1) / CA_SEG;
  const int q0 = seg * qs, q1 = min(nci, q0 + qs);
  for (int pi = threadIdx.x % CA_ROWS; pi < nci; pi += CA_ROWS) {
    double acc = 0.0;
    int q = q0;
    for (; q + 8 <= q1; q += 8) {
      double g[8];
#pragma unroll
      for (int u = 0; u < 8; u++) g[u] = G[(long)(q + u) * nci + pi];
#pragma unroll
      for (int u = 0; u < 8; u++) acc = acc + g[u] * rv[q + u];
    }
    for (; q < q1; q++) acc = acc + G[(long)q * nci + pi] * rv[q];
    part[seg * nci + pi] = acc;
  }
  __syncthreads();
  for (int pi = threadIdx.x; pi < nci; pi += SMALL_THREADS) {
    double acc = part[pi];
    for (int sgi = 1; sgi < CA_SEG; sgi++) acc = acc + part[sgi * nci + pi];
    int ip = 1 + pi % (nxc - 1), kp = 1 + pi / (nxc - 1);
    store_with_ghosts<float>(err, ip, kp, nxc, nzc, pitch, (float)acc, sz);
  }
}
__global__ void __launch_bounds__(SMALL_THREADS) k_coarse_apply_wg(const double* G, const float* rhs, float* err,
                                                                   int nxc, int nzc, int pitch, float sz) {
  extern __shared__ double ca_sm[];
  coarse_apply_wg(G, rhs, err, nxc, nzc, pitch, sz, ca_sm);
}

// enforceBCs_stream (PS/iterative_solver.f90:1616-1664) on a whole level-1
// field: walls (with their ghost extensions) zero, ghosts from the interior
__global__ void k_stream_bcs(double* S, int n, int m, int p, double sz) {
  const int i = -3 + (int)(blockIdx.x * blockDim.x + threadIdx.x), k = -3 + (int)(blockIdx.y * blockDim.y + threadIdx.y);
  if (i > n + 3 || k > m + 3) return;
  if (i == 0 || i == n || k == 0 || k == m) {
    S[IDX(i, k, p)] = 0.0;
    return;
  }
  if (i >= 1 && i <= n - 1 && k >= 1 && k <= m - 1) store_with_ghosts<double>(S, i, k, n, m, p, S[IDX(i, k, p)], sz);
}

// compute_RHS(1): RaT*d(Tbuoy)/dx - RaC*d(Cbuoy)/dx (5-point D1)
__global__ void k_rhs1(const double* Tb, const double* Cb, double* rhs, int nx, int nz, int p3, int p5, double dr,
                       double RaT, double RaC, double d0, double d1, double d2, double d3, double d4) {
  int i = 1 + blockIdx.x * blockDim.x + threadIdx.x, k = 1 + blockIdx.y * blockDim.y + threadIdx.y;
  if (i > nx - 1 || k > nz - 1) return;
  const double D[5] = {d0, d1, d2, d3, d4};
  double r = 0.0;
  if (RaT != 0.0) {
    double s = 0.0;
    for (int q = -2; q <= 2; q++) s = s + D[q + 2] * Tb[IDX(i + q, k, p3)];
    double Tr = s / dr;
    double Tx = Tr / 1.0;
    r = RaT * Tx;
  }
  double s = 0.0;
  for (int q = -2; q <= 2; q++) s = s + D[q + 2] * Cb[(long)(k + 5) * p5 + (i + q + 5)];
  double Cr = s / dr;
  double Cx = Cr / 1.0;
  r = r - RaC * Cx;
  rhs[IDX(i, k, p3)] = r;
}

// compute_velocities: w = -D1_x psi / dr, u = D1_z psi / ds on (0:nx,0:nz)
__global__ void k_velocities(const double* SF, double* u, double* w, int nx, int nz, int p, double dr, double ds,
                             double d0, double d1, double d2, double d3, double d4) {
  int i = blockIdx.x * blockDim.x + threadIdx.x, k = blockIdx.y * blockDim.y + threadIdx.y;
  if (i > nx || k > nz) return;
  const double D[5] = {d0, d1, d2, d3, d4};
  double sx = 0.0, sz = 0.0;
  for (int q = -2; q <= 2; q++) sx = sx + D[q + 2] * SF[IDX(i + q, k, p)];
  for (int q = -2; q <= 2; q++) sz = sz + D[q + 2] * SF[IDX(i, k + q, p)];
  w[IDX(i, k, p)] = -(sx / dr);
  u[IDX(i, k, p)] = sz / ds;
}

// velocityBCs (PS/composition.f90:1295-1325) as a gather over the ghost frame:
// every ghost takes its value from the interior image with the reference's sign
__global__ void k_velocity_bcs(double* u, double* w, int nx, int nz, int p, int Vbc) {
  int i = -3 + (int)(blockIdx.x * blockDim.x + threadIdx.x), k = -3 + (int)(blockIdx.y * blockDim.y + threadIdx.y);
  if (i > nx + 3 || k > nz + 3) return;
  bool gi = i < 0 || i > nx, gk = k < 0 || k > nz;
  int mi = i < 0 ? -i : (i > nx ? 2 * nx - i : i);
  int mk = k < 0 ? -k : (k > nz ? 2 * nz - k : k);
  // w: symmetric in x, antisymmetric in z; w=0 on k=0,nz (all columns)
  double wv, uv;
  if (!gi && !gk) {
    wv = w[IDX(i, k, p)]; uv = u[IDX(i, k, p)];
  } else {
    double wm = w[IDX(mi, mk, p)], um = u[IDX(mi, mk, p)];
    wv = gk ? -wm : wm;
    double su = (Vbc == 0) ? 1.0 : -1.0;
    uv = gi ? -um : um;
    if (gk) uv = su * uv;
  }
  if (k == 0 || k == nz) wv = 0.0;
  if (i == 0 || i == nx) uv = 0.0;
  if (Vbc == 1 && (k == 0 || k == nz)) uv = 0.0;
  if (gi || gk || k == 0 || k == nz || i == 0 || i == nx) {
    w[IDX(i, k, p)] = wv;
    u[IDX(i, k, p)] = uv;
  }
}

// ---------------------------------------------------------------------------
// viscosity hierarchy
// ---------------------------------------------------------------------------
__global__ void k_visf(const double* Tvis, const double* Cvis, double* vs, int nx, int nz, int p3, int p5, int ivis,
                       double lvT, double lvC, double lvP, double ds, int RaTnz) {
  int i = blockIdx.x * blockDim.x + threadIdx.x, k = blockIdx.y * blockDim.y + threadIdx.y;
  if (i > nx || k > nz) return;
  double zg = ds * (double)k;
  if (k == nz) zg = 1.0;
  double v = 1.0;
  if (ivis == 1) v = exp(-(Tvis[IDX(i, k, p3)] * lvT) + (1.0 - zg) * lvP);
  else if (ivis == 2) {
    double dp = 0.0 + Cvis[(long)(k + 5) * p5 + (i + 5)] * lvC;
    if (RaTnz) v = exp(-(Tvis[IDX(i, k, p3)] * lvT) - dp + (1.0 - zg) * lvP);
    else v = exp(-dp + (1.0 - zg) * lvP);
  }
  vs[IDX(i, k, p3)] = v;
}

// viscosityBCs (PS/iterative_solver.f90:666-690): side ghosts on rows
// -3..m+3 then top/bottom ghosts on columns 0..n.  The side pass reads the
// ghost rows before the top/bottom pass rewrites them, as the reference.
__global__ void k_vis_bcs_side(double* v, int n, int m, int p) {
  int t = blockIdx.x * blockDim.x + threadIdx.x;   // over rows -3..m+3, 3 ghosts each side
  int rows = m + 7;
  if (t >= rows * 3) return;
  int k = -3 + t / 3, i = 1 + t % 3;
  v[IDX(-i, k, p)] = v[IDX(i, k, p)];
  v[IDX(n + i, k, p)] = v[IDX(n - i, k, p)];
}
__global__ void k_vis_bcs_tb(double* v, int n, int m, int p) {
  int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= (n + 1) * 3) return;
  int i = t / 3, k = 1 + t % 3;
  v[IDX(i, -k, p)] = v[IDX(i, k, p)];
  v[IDX(i, m + k, p)] = v[IDX(i, m - k, p)];
}

// v(i,k) = x with its images (n, m >= 3): side images, top and bottom images,
// and the corners' side images of the ghost rows, which hold ghost(k') from
// before
template <class Ghost>
__device__ __forceinline__ void vis_store(double* v, int i, int k, int n, int m, int p, double x, Ghost ghost) {
  const bool left = i >= 1 && i <= 3, right = i <= n - 1 && i >= n - 3;
  auto image = [&](int kg) {
    const double old = ghost(kg);
    v[IDX(i, kg, p)] = x;
    if (left) v[IDX(-i, kg, p)] = old;
    if (right) v[IDX(2 * n - i, kg, p)] = old;
  };
  v[IDX(i, k, p)] = x;
  if (left) v[IDX(-i, k, p)] = x;
  if (right) v[IDX(2 * n - i, k, p)] = x;
  if (k >= 1 && k <= 3) image(-k);
  if (k <= m - 1 && k >= m - 3) image(2 * m - k);
}

// viscosityBCs_initialize (PS/iterative_solver.f90:636-664)
__global__ void k_vis_bcs_init_boundary(double* v, const double* f, int n, int m, int p, int fn, int fm, int fp) {
  int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t <= m - 2) {   // k = 1..m-1
    int k = t + 1;
    v[IDX(0, k, p)] = f[IDX(0, 2 * k, fp)];
    v[IDX(n, k, p)] = f[IDX(fn, 2 * k, fp)];
  }
  if (t <= n) {
    int i = t;
    v[IDX(i, 0, p)] = f[IDX(2 * i, 0, fp)];
    v[IDX(i, m, p)] = f[IDX(2 * i, fm, fp)];
  }
}
__global__ void k_vis_bcs_init_side(double* v, int n, int m, int p) {
  int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= (m + 1) * 3) return;
  int k = t / 3, i = 1 + t % 3;
  v[IDX(-i, k, p)] = v[IDX(i, k, p)];
  v[IDX(n + i, k, p)] = v[IDX(n - i, k, p)];
}
__global__ void k_vis_bcs_init_tb(double* v, int n, int m, int p) {
  int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= (n + 7) * 3) return;
  int i = -3 + t / 3, k = 1 + t % 3;
  v[IDX(i, -k, p)] = v[IDX(i, k, p)];
  v[IDX(i, m + k, p)] = v[IDX(i, m - k, p)];
}

// viscosity_gradients, uniform grid (PS/iterative_solver.f90:488-520)
__global__ void k_vis_grad(VisSet s, int n, int m, int p, int full, int ivis0, double dr, double ds, double dr2,
                           double ds2, double drds, double dtv) {
  int i = blockIdx.x * blockDim.x + threadIdx.x, k = blockIdx.y * blockDim.y + threadIdx.y;
  if (i > n || k > m) return;
  long g = IDX(i, k, p);
  if (ivis0) {
    s.vx[g] = 0; s.vz[g] = 0; s.vxx[g] = 0; s.vzz[g] = 0; s.vxz[g] = 0; s.vxxpzz[g] = 0; s.vxxmzz[g] = 0;
    return;
  }
  const double* v = s.vis;
  if (full) {
    // Drs_so(:,-1)=(.25,0,-.25), (:,0)=0, (:,1)=(-.25,0,.25); sum in column-major order
    double sxz = 0.0;
    sxz = sxz + 0.25 * v[IDX(i - 1, k - 1, p)];
    sxz = sxz + 0.0 * v[IDX(i, k - 1, p)];
    sxz = sxz + (-0.25) * v[IDX(i + 1, k - 1, p)];
    sxz = sxz + 0.0 * v[IDX(i - 1, k, p)];
    sxz = sxz + 0.0 * v[IDX(i, k, p)];
    sxz = sxz + 0.0 * v[IDX(i + 1, k, p)];
    sxz = sxz + (-0.25) * v[IDX(i - 1, k + 1, p)];
    sxz = sxz + 0.0 * v[IDX(i, k + 1, p)];
    sxz = sxz + 0.25 * v[IDX(i + 1, k + 1, p)];
    s.vxz[g] = sxz / drds;
    double sx = 0.0;
    sx = sx + (-0.5) * v[IDX(i - 1, k, p)];
    sx = sx + 0.0 * v[IDX(i, k, p)];
    sx = sx + 0.5 * v[IDX(i + 1, k, p)];
    s.vx[g] = sx / dr;
  }
  double sxx = 0.0;
  sxx = sxx + 1.0 * v[IDX(i - 1, k, p)];
  sxx = sxx + (-2.0) * v[IDX(i, k, p)];
  sxx = sxx + 1.0 * v[IDX(i + 1, k, p)];
  double vxx = sxx / dr2;
  s.vxx[g] = vxx;
  if (full) {
    double sz = 0.0;
    sz = sz + (-0.5) * v[IDX(i, k - 1, p)];
    sz = sz + 0.0 * v[IDX(i, k, p)];
    sz = sz + 0.5 * v[IDX(i, k + 1, p)];
    s.vz[g] = sz / ds;
  }
  double szz = 0.0;
  szz = szz + 1.0 * v[IDX(i, k - 1, p)];
  szz = szz + (-2.0) * v[IDX(i, k, p)];
  szz = szz + 1.0 * v[IDX(i, k + 1, p)];
  double vzz = szz / ds2;
  s.vzz[g] = vzz;
  double xp = vxx + vzz;
  s.vxxpzz[g] = xp;
  if (full) s.vxxmzz[g] = vxx - vzz;
  s.vsmooth[g] = dtv * xp;
}

// test_eigenvalues, RKC1 branch (PS/iterative_solver.f90:1187-1208) + block min of ratio
__global__ void k_test_eig(VisSet s, double* ratio, double* dts, int n, int m, int p, double SR1, double SR2,
                           double SR4, double SR5, double SR6, double SI1, double SI2, double SI4, double SI5,
                           double SI6, double ae, double be, double ctemp, double* partial) {
  __shared__ double red[256];
  int tid = threadIdx.y * blockDim.x + threadIdx.x;
  int i = 1 + blockIdx.x * blockDim.x + threadIdx.x, k = 1 + blockIdx.y * blockDim.y + threadIdx.y;
  double rmin = INFINITY;
  if (i <= n - 1 && k <= m - 1) {
    long g = IDX(i, k, p);
    double vis = s.vis[g];
    double eI = fabs(s.vxxpzz[g] * SI1) + vis * SI2 + fabs(s.vxz[g] * SI4) + fabs(s.vx[g] * SI5) + fabs(s.vz[g] * SI6);
    double eR = s.vxxmzz[g] * SR1 + vis * SR2 + s.vxz[g] * SR4 + s.vx[g] * SR5 + s.vz[g] * SR6;
    double r = fabs(eR / eI);
    ratio[g] = r;
    double qa = eR / ae, qb = eI / be;
    dts[g] = ctemp * eR / (qa * qa + qb * qb);
    rmin = r;
  }
  red[tid] = rmin;
  __syncthreads();
  for (int st = 128; st > 0; st >>= 1) {
    if (tid < st) red[tid] = fmin(red[tid], red[tid + st]);
    __syncthreads();
  }
  if (tid == 0) partial[blockIdx.y * gridDim.x + blockIdx.x] = red[0];
}

// one update from the gradients' vsmooth, and viscosityBCs.  A thread writes
// its node's images too; those in the corners (side images of the ghost rows)
// take the ghost rows as they were before, as the side pass does.
__global__ void k_vis_update(double* v, const double* sm, int n, int m, int p, double c) {
  int i = blockIdx.x * blockDim.x + threadIdx.x, k = blockIdx.y * blockDim.y + threadIdx.y;
  if (i > n || k > m) return;
  long g = IDX(i, k, p);
  vis_store(v, i, k, n, m, p, v[g] + c * sm[g], [&](int kg) { return v[IDX(i, kg, p)]; });
}

// Several updates per launch, for the iterations between which nothing is
// asked of the gradients: v = v + cc dtv (vxx + vzz), each with viscosityBCs.
// A workgroup holds its tile and as many rows and columns around it as there
// are updates in LDS, in two copies; what its edge lacks spoils one more row
// per update and stops short of the tile.  Neighbours across the domain's edge
// are the mirrored ones.  Bound by launches: an update took four (gradients,
// update, two of ghosts), 3.8 + 2.5 + 2.3 + 2.4 us on average over the levels
// of 1024x256, and 3 to 6 of them in one launch take 9.0.
constexpr int VIS_ITS = 6;             // updates per launch at most
constexpr int VIS_TZ = 16;             // tile rows; a tile is 64 - 2 its columns wide
constexpr int VIS_ROWS = VIS_TZ + 2 * VIS_ITS;
struct VisSmooth {
  const double* in;
  double* out;
  double cc[VIS_ITS];
  double dr2, ds2, rdr2, rds2, dtv;
  int n, m, p, its, ghosts;   // ghosts: the last launch, which leaves them
};

template <bool PW2>
__global__ void __launch_bounds__(256) k_vis_smooth(VisSmooth a) {
  __shared__ double V[2][VIS_ROWS][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int H = a.its, n = a.n, m = a.m, p = a.p;
  const int x0 = blockIdx.x * (64 - 2 * H) - H, z0 = blockIdx.y * VIS_TZ - H;   // the tile's corner with its surroundings
  const int rows = VIS_TZ + 2 * H, i = x0 + lane;
  const int il = max(i == 0 ? lane + 1 : lane - 1, 0), ir = min(i == n ? lane - 1 : lane + 1, 63);
  for (int r = wave; r < rows; r += 4)
    V[0][r][lane] = a.in[IDX(min(max(i, 0), n), min(max(z0 + r, 0), m), p)];
  __syncthreads();
  for (int it = 0; it < H; it++) {
    const double(*A)[64] = V[it & 1];
    double(*B)[64] = V[(it + 1) & 1];
    for (int r = wave; r < rows; r += 4) {
      const int k = z0 + r, rd = max(k == 0 ? r + 1 : r - 1, 0), ru = min(k == m ? r - 1 : r + 1, rows - 1);
      const double v = A[r][lane];
      double sxx = 0.0, szz = 0.0;
      sxx = sxx + A[r][il];
      sxx = sxx + (-2.0) * v;
      sxx = sxx + A[r][ir];
      szz = szz + A[rd][lane];
      szz = szz + (-2.0) * v;
      szz = szz + A[ru][lane];
      const double xp = quot<PW2>(sxx, a.dr2, a.rdr2) + quot<PW2>(szz, a.ds2, a.rds2);
      B[r][lane] = v + a.cc[it] * (a.dtv * xp);
    }
    __syncthreads();
  }
  if (lane < H || lane >= 64 - H || i > n) return;
  for (int r = H + wave; r < H + VIS_TZ; r += 4) {
    const int k = z0 + r;
    if (k > m) break;
    if (a.ghosts)
      vis_store(a.out, i, k, n, m, p, V[H & 1][r][lane], [&](int) { return V[(H + 1) & 1][r][lane]; });
    else
      a.out[IDX(i, k, p)] = V[H & 1][r][lane];
  }
}

// ---------------------------------------------------------------------------
// coarsest grid: banded operator, row equilibration, LU, solve
// ---------------------------------------------------------------------------
struct CoarseArgs {
  const double *vis, *vxm, *vxz, *vx, *vz;
  int nxc, nzc, p, kl, ku, ngc, ivis0, Vbc;
  double SM1[7][7], SM2[7][7], SM4[7][7], SM5[7][7], SM6[7][7];
};

__device__ double stream_space_matrix(const CoarseArgs& a, int ip, int kp, int iq, int kq, int sval) {
  int di = iq - ip, dk = kq - kp;
  long g = IDX(ip, kp, a.p);
  double v;
  if (a.ivis0) v = a.vis[g] * a.SM2[dk + 3][di + 3];
  else
    v = a.vxm[g] * a.SM1[dk + 3][di + 3] + a.vis[g] * a.SM2[dk + 3][di + 3] + a.vxz[g] * a.SM4[dk + 3][di + 3] +
        a.vx[g] * a.SM5[dk + 3][di + 3] + a.vz[g] * a.SM6[dk + 3][di + 3];
  if (sval == -1) v = -v;
  return v;
}

// one thread per matrix row p (Compute_Matrix_coarse, analysis=0)
__global__ void k_coarse_assemble(CoarseArgs a, double* Mc, double* RowB) {
  int p = 1 + blockIdx.x * blockDim.x + threadIdx.x;
  if (p > a.ngc) return;
  const int limit[7] = {0, 2, 2, 3, 2, 2, 0};
  int ld = 2 * a.kl + a.ku + 1, kk1 = a.kl + a.ku + 1, N = a.nzc + 1;
  int kp = p - N * ((p - 1) / N) - 1, ip = (p - 1) / N;
  auto M = [&](int r, int q) -> double& { return Mc[(long)(q - 1) * ld + (r - 1)]; };
  if (ip > 0 && ip < a.nxc && kp > 0 && kp < a.nzc) {
    for (int j = -3; j <= 3; j++) {
      int iq = j + ip;
      if (iq >= 0 && iq <= a.nxc)
        for (int kq = kp - limit[j + 3]; kq <= kp + limit[j + 3]; kq++)
          if (kq >= 0 && kq <= a.nzc) {
            int q = N * iq + kq + 1;
            M(kk1 + p - q, q) = stream_space_matrix(a, ip, kp, iq, kq, 1);
          }
    }
    for (int j = -3; j <= 3; j++) {
      int iq = j + ip;
      for (int kq = kp - limit[j + 3]; kq <= kp + limit[j + 3]; kq++)
        if (iq < 0 || iq > a.nxc || kq < 0 || kq > a.nzc) {
          int iiq, kkq, xv, zv;
          if (iq < 0) { iiq = -iq; xv = -1; }
          else if (iq > a.nxc) { iiq = 2 * a.nxc - iq; xv = -1; }
          else { iiq = iq; xv = 1; }
          if (kq < 0) { kkq = -kq; zv = a.Vbc == 0 ? -1 : 1; }
          else if (kq > a.nzc) { kkq = 2 * a.nzc - kq; zv = a.Vbc == 0 ? -1 : 1; }
          else { kkq = kq; zv = 1; }
          int q = N * iiq + kkq + 1;
          M(kk1 + p - q, q) = M(kk1 + p - q, q) + stream_space_matrix(a, ip, kp, iq, kq, xv * zv);
        }
    }
  } else {
    M(kk1, p) = 1.0;   // impermeable boundary rows
  }
}

// DGBEQU row scale factors and row scaling; one thread per row
__global__ void k_coarse_equilibrate(double* Mc, double* RowB, int n, int kl, int ku) {
  int p = 1 + blockIdx.x * blockDim.x + threadIdx.x;
  if (p > n) return;
  int ld = 2 * kl + ku + 1, kk1 = kl + ku + 1;
  double r = 0.0;
  int qlo = std::max(1, p - kl), qhi = std::min(n, p + ku);
  for (int q = qlo; q <= qhi; q++) {
    double a = fabs(Mc[(long)(q - 1) * ld + (kk1 + p - q - 1)]);
    if (a > r) r = a;
  }
  const double smlnum = 2.2250738585072014e-308, bignum = 1.0 / smlnum;
  r = fmin(fmax(r, smlnum), bignum);
  double rb = 1.0 / r;
  RowB[p - 1] = rb;
  for (int q = qlo; q <= qhi; q++) {
    double& m = Mc[(long)(q - 1) * ld + (kk1 + p - q - 1)];
    m = rb * m;
  }
}

// DGBTF2 (LAPACK unblocked band LU with partial pivoting) on one wavefront
__global__ void __launch_bounds__(64) k_band_lu(double* ab, int32_t* ipiv, int n, int kl, int ku, int32_t* info) {
  const int ld = 2 * kl + ku + 1, kv = ku + kl;
  const int lane = threadIdx.x;
#define AB(r, q) ab[(long)((q) - 1) * ld + ((r) - 1)]
  for (int j = ku + 2 + lane; j <= std::min(kv, n); j += 64)
    for (int i = kv - j + 2; i <= kl; i++) AB(i, j) = 0.0;
  __syncthreads();
  int ju = 1, inf = 0;
  for (int j = 1; j <= n; j++) {
    if (j + kv <= n)
      for (int i = 1 + lane; i <= kl; i += 64) AB(i, j + kv) = 0.0;
    int km = std::min(kl, n - j);
    // IDAMAX over AB(kv+1 .. kv+1+km, j): first index of the maximum |.|
    double best = -1.0; int bi = 0x7fffffff;
    for (int t = lane; t <= km; t += 64) {
      double a = fabs(AB(kv + 1 + t, j));
      if (a > best) { best = a; bi = t; }
    }
    for (int off = 32; off > 0; off >>= 1) {
      double ob = __shfl_down(best, off);
      int oi = __shfl_down(bi, off);
      if (ob > best || (ob == best && oi < bi)) { best = ob; bi = oi; }
    }
    int jp = __shfl(bi, 0) + 1;
    __syncthreads();
    if (lane == 0) ipiv[j - 1] = jp + j - 1;
    double piv = AB(kv + jp, j);
    if (piv != 0.0) {
      ju = std::max(ju, std::min(j + ku + jp - 1, n));
      if (jp != 1)
        for (int t = lane; t <= ju - j; t += 64) {
          double* pa = &ab[(long)(j - 1 + t) * ld + (kv + jp - 1 - t)];
          double* pb = &ab[(long)(j - 1 + t) * ld + (kv - t)];
          double tmp = *pa; *pa = *pb; *pb = tmp;
        }
      __syncthreads();
      if (km > 0) {
        double rcp = 1.0 / AB(kv + 1, j);
        for (int t = 1 + lane; t <= km; t += 64) AB(kv + 1 + t, j) = rcp * AB(kv + 1 + t, j);
        __syncthreads();
        // DGER: columns are independent (the pivot-row element y(jj) is not
        // updated), so the (jj, t) pairs are spread over the wavefront
        const int total = (ju - j) * km;
        for (int idx = lane; idx < total; idx += 64) {
          int jj = 1 + idx / km, t = 1 + idx % km;
          double yv = ab[(long)(j - 1 + jj) * ld + (kv - jj)];
          double temp = -1.0 * yv;
          double& x = ab[(long)(j - 1 + jj) * ld + (kv - jj + t)];
          x = x + AB(kv + 1 + t, j) * temp;
        }
      }
    } else if (inf == 0) {
      inf = j;
    }
    __syncthreads();
  }
  if (lane == 0) *info = inf;
#undef AB
}

// ---------------------------------------------------------------------------
// host orchestration
// ---------------------------------------------------------------------------
static dim3 grid2(int ni, int nk, dim3 b) { return dim3((ni + b.x - 1) / b.x, (nk + b.y - 1) / b.y); }

template <typename R>
static StageArgs<R> stage_base(Context& c, int l, bool fp32) {
  StageArgs<R> a;
  std::memset(&a, 0, sizeof a);
  Level& L = c.L[l];
  const LevelGeom& g = L.g;
  a.n = g.n; a.m = g.m; a.pitch = g.pitch;
  a.sz = (R)(c.P.Vbc == 0 ? -1.0 : 1.0);
  a.dr2 = (R)g.dr2; a.dr3 = (R)g.dr3; a.dr4 = (R)g.dr4; a.ds2 = (R)g.ds2; a.ds3 = (R)g.ds3; a.ds4 = (R)g.ds4;
  a.drds = (R)g.drds; a.dr2ds = (R)g.dr2ds; a.drds2 = (R)g.drds2; a.dr2ds2 = (R)g.dr2ds2;
  a.rdr2 = (R)(1.0 / g.dr2); a.rdr3 = (R)(1.0 / g.dr3); a.rdr4 = (R)(1.0 / g.dr4);
  a.rds2 = (R)(1.0 / g.ds2); a.rds3 = (R)(1.0 / g.ds3); a.rds4 = (R)(1.0 / g.ds4);
  a.rdrds = (R)(1.0 / g.drds); a.rdr2ds = (R)(1.0 / g.dr2ds); a.rdrds2 = (R)(1.0 / g.drds2);
  a.rdr2ds2 = (R)(1.0 / g.dr2ds2);
  for (int q = 0; q < 5; q++) { a.D1[q] = (R)c.st.D1[q]; a.D2[q] = (R)c.st.D2[q]; }
  for (int q = 0; q < 7; q++) { a.D3[q] = (R)c.st.D3[q]; a.D4[q] = (R)c.st.D4[q]; }
  for (int b = 0; b < 5; b++)
    for (int q = 0; q < 5; q++) {
      a.Drs[b][q] = (R)c.st.Drs[b][q]; a.Drss[b][q] = (R)c.st.Drss[b][q];
      a.Drrs[b][q] = (R)c.st.Drrs[b][q]; a.Drrss[b][q] = (R)c.st.Drrss[b][q];
    }
  if (!fp32) {
    a.vis = (const R*)L.v.vis; a.vxm = (const R*)L.v.vxxmzz; a.vxz = (const R*)L.v.vxz;
    a.vx = (const R*)L.v.vx; a.vz = (const R*)L.v.vz; a.rhs = (const R*)L.rhs; a.dts = (const R*)L.dts;
  } else {
    a.vis = (const R*)L.fvis; a.vxm = (const R*)L.fvxm; a.vxz = (const R*)L.fvxz;
    a.vx = (const R*)L.fvx; a.vz = (const R*)L.fvz; a.rhs = (const R*)L.frhs; a.dts = (const R*)L.fdts;
  }
  return a;
}

template <typename R>
static void launch_residual(Context& c, dim3 grd, dim3 blk, const StageArgs<R>& a, R* res, double* partial) {
  if (c.P.ivis == 0) hipLaunchKernelGGL((k_residual<R, true>), grd, blk, 0, c.stream, a, res, partial);
  else hipLaunchKernelGGL((k_residual<R, false>), grd, blk, 0, c.stream, a, res, partial);
}

// ---------------------------------------------------------------------------
// sweeps: tiling, launches
// ---------------------------------------------------------------------------
template <typename R, int EV, int RB>
constexpr int sweep_threads() {
  return sizeof(R) == 8 && EV == 0 && RB == 4 ? 512 : 1024;
}
static int sweep_threads_of(bool f32, int ev, int rb) { return !f32 && ev == 0 && rb == 4 ? 512 : 1024; }

// the launch shape of `nev` evaluations on cw x ch cores
struct SweepShape {
  int w1, nrb, tcol, threads, nbx, nblk;
  size_t lds;
};
static SweepShape sweep_shape(int n, int m, int cw, int ch, int rb, int nev, size_t elem) {
  SweepShape s;
  s.w1 = std::min(cw + 6 * (nev - 1), n - 1);
  const int h1 = std::min(ch + 6 * (nev - 1), m - 1);
  s.nrb = (h1 + rb - 1) / rb;
  s.tcol = s.w1;
  s.threads = (s.tcol * s.nrb + 63) & ~63;
  s.nbx = (n - 1 + cw - 1) / cw;
  s.nblk = s.nbx * ((m - 1 + ch - 1) / ch);
  s.lds = 2 * elem * (size_t)(s.w1 + 8) * (s.nrb * rb + 8);
  return s;
}

// the operator's form on a level: general (0), isoviscous (1), or isoviscous
// with the factorised psi_xxzz (2), on some of the FP32 levels >= 2.  k_sweep
// takes either on any level, and both are right to FP32 rounding.  The limits
// below are those of the kernels that these levels had before k_sweep; they are
// kept for one reason: the form decides the rounding of the FP32 corrections,
// so with other limits a mixed solve of the same input would end at another psi
// within its stop test's tolerance.
static int sweep_form(const Context& c, int l, bool f32) {
  if (c.P.ivis != 0) return 0;
  if (!f32 || l < 2) return 1;
  const LevelGeom& g = c.L[l].g;
  const int npts = (g.n - 1) * (g.m - 1);
  if (npts > 4096) return g.m - 1 <= 64 ? 2 : 1;
  if (3 * sizeof(float) * c.L[l].nelem > SMALL_LDS_BYTES) return 1;
  const int b4 = (g.n - 1) * ((g.m + 2) / 4);
  return (b4 <= SMALL_THREADS && 2 * b4 >= SMALL_THREADS) || npts <= SMALL_THREADS ? 2 : 1;
}

// Modelled time (us) of one launch of `nev` evaluations; the constants per
// operator form are a fit to timed sweeps of levels from 7x7 to 1023x255 points:
//   2.9            launch to launch
//   fill, row      window loads per thread and per window row
//   stage          an evaluation's latency (LDS round trip, barrier)
//   wave           VALU time of a SIMD's wavefronts, per point of a thread
//   lds            LDS time of a CU's wavefronts (29, 36, 50 reads for 1, 2, 4 points)
struct SweepCost {
  double fill, row, stage, wave, lds;
};
static double sweep_launch_us(const SweepCost& k, int n, int m, int cw, int ch, int rb, int nev,
                              const SweepShape& s) {
  constexpr int CUS = 256;
  const int per = (s.nblk + CUS - 1) / CUS, rows = s.nrb * rb + 8;   // tiles per CU
  double us = 2.9 + per * (k.fill * (s.w1 + 8) * rows / s.threads * ((s.threads + 255) / 256) + k.row * rows);
  for (int h = 0; h < nev; h++) {
    const int hh = std::min(ch + 6 * h, m - 1), ww = std::min(cw + 6 * h, n - 1);
    const int nb = std::min(s.nrb, (hh + rb - 1) / rb + (h < nev - 1 && rb > 1 ? 1 : 0));
    const int lanes = (ww < s.w1 && s.w1 >= 96 ? ww + 64 : s.w1) * nb;   // active row blocks, in whole wavefronts
    const int waves = std::max(1, (lanes + 63) / 64) * per;
    us += k.stage + k.wave * ((waves + 3) / 4) * rb + k.lds * waves * (rb == 1 ? 29 : rb == 2 ? 36 : 50) / 64;
  }
  return us;
}

// The tiling of a level's sweeps of s stages: the one with the least modelled
// time.  Small tiles use more CUs and large ones recompute less overlap; more
// stages per launch save launches and widen the overlap.  1024x256, 35
// stages: 32x32 cores, 3 stages per launch, 2 points per thread (FP32 general
// operator 150 us a sweep against 35 launches of one stage at 8.5 us; FP64
// isoviscous 144 us against 35 x 6.0); 256x64: 16x4, 3, 1 (FP32 general, 15
// stages: 30 us against 15 x 5.5); 32x32 FP64: one workgroup, all stages, 2
// points per thread (49 us; one point per thread and a row of LDS reads per
// point: 58).  Whole solves with the stages per launch bounded at 1, 2, 3, 4, 5,
// 6 and 8 (tile and rows as the model then takes them) and as the plan is, ms:
//   1024x256 law, mixed    16.6  13.1  11.8  11.7  11.6  11.6  11.6   11.7
//   1024x256 iso, mixed     9.1   6.7   5.7   5.7   5.5   5.5   5.7    5.5
//   1024x256 iso, FP64     50.4  31.8  26.1  25.0  24.1  24.1  24.2   23.1
//   256x64 law, FP64       47.8  29.1  24.2  22.0  21.1  20.3  20.0   18.0
//   64x64 law, FP64        42.4  27.1  22.2  19.7  18.6  17.8  17.3   14.7
static SweepPlan sweep_plan(const Context& c, int l, bool f32, int s) {
  const LevelGeom& g = c.L[l].g;
  const int n = g.n, m = g.m, ev = sweep_form(c, l, f32);
  const SweepCost cost = f32 ? (ev == 0   ? SweepCost{0.10, 0.01, 0.75, 0.21, 0.038}
                                : ev == 1 ? SweepCost{0.18, 0.02, 0.31, 0.081, 0.008}
                                          : SweepCost{0.15, 0.01, 0.46, 0.057, 0.006})
                             : (ev == 0 ? SweepCost{0.034, 0.03, 0.60, 0.453, 0.015}
                                        : SweepCost{0.21, 0.03, 0.59, 0.345, 0.013});
  const size_t elem = f32 ? 4 : 8;
  const int cws[] = {8, 12, 16, 24, 32, 48, 64, 96, 128, 192, 256, n - 1};
  const int chs[] = {4, 8, 12, 16, 24, 32, 48, 64, m - 1};
  // levels >= 2 may form the residual in the last launch
  const int extra = l >= 2 ? 1 : 0;
  SweepPlan best = {std::min(8, n - 1), std::min(4, m - 1), 1, 1};
  double best_us = INFINITY;
  for (int rb = 1; rb <= 4; rb *= 2)
    for (int cw : cws)
      for (int ch : chs) {
        if (cw > n - 1 || ch > m - 1) continue;
        for (int ns = 1; ns <= s; ns++) {
          const int nseg = (s + ns - 1) / ns, base = s / nseg, rem = s % nseg;
          if (c.sweep_stages > 0 && ns > c.sweep_stages) break;
          if (base + (rem ? 1 : 0) != ns) continue;   // a larger ns with as many launches
          const SweepShape widest = sweep_shape(n, m, cw, ch, rb, ns + extra, elem);
          if (widest.threads > sweep_threads_of(f32, ev, rb) || widest.lds > SWEEP_LDS_BYTES) break;
          // not the tilings whose tiles mostly recompute each other's points, nor
          // those of several points per thread in few wavefronts: the model was
          // not fitted to such and calls some of them fast that are not
          double evals = 0.0;
          for (int h = 0; h < ns; h++) evals += (double)std::min(cw + 6 * h, n - 1) * std::min(ch + 6 * h, m - 1);
          if (widest.nblk > 1 && evals * widest.nblk > (nseg == 1 ? 2.0 : 5.0) * ns * (n - 1) * (m - 1)) continue;
          if (rb > 1 && widest.threads < 512) continue;
          double us = rem * sweep_launch_us(cost, n, m, cw, ch, rb, ns, sweep_shape(n, m, cw, ch, rb, ns, elem));
          if (nseg > rem + 1)
            us += (nseg - rem - 1) *
                  sweep_launch_us(cost, n, m, cw, ch, rb, base, sweep_shape(n, m, cw, ch, rb, base, elem));
          const int last = base + (f32 ? 0 : extra);
          us += sweep_launch_us(cost, n, m, cw, ch, rb, last, sweep_shape(n, m, cw, ch, rb, last, elem));
          if (us < best_us) {
            best_us = us;
            best = {cw, ch, ns, rb};
          }
        }
      }
  return best;
}

template <typename R>
static SweepArgs<R> sweep_args(Context& c, int l, bool f32, const LevelRkc& rk, double cpar) {
  SweepArgs<R> a;
  std::memset(&a, 0, sizeof a);
  const StageArgs<R> b = stage_base<R>(c, l, f32);
  a.vis = b.vis; a.vxm = b.vxm; a.vxz = b.vxz; a.vx = b.vx; a.vz = b.vz; a.rhs = b.rhs; a.dts = b.dts;
  a.n = b.n; a.m = b.m; a.pitch = b.pitch; a.sz = b.sz;
  a.dr2 = b.dr2; a.dr3 = b.dr3; a.dr4 = b.dr4; a.ds2 = b.ds2; a.ds3 = b.ds3; a.ds4 = b.ds4;
  a.drds = b.drds; a.dr2ds = b.dr2ds; a.drds2 = b.drds2; a.dr2ds2 = b.dr2ds2;
  a.rdr2 = b.rdr2; a.rdr3 = b.rdr3; a.rdr4 = b.rdr4; a.rds2 = b.rds2; a.rds3 = b.rds3; a.rds4 = b.rds4;
  a.rdrds = b.rdrds; a.rdr2ds = b.rdr2ds; a.rdrds2 = b.rdrds2; a.rdr2ds2 = b.rdr2ds2;
  for (int q = 0; q < 3; q++) { a.w.d2[q] = b.D2[2 + q]; a.w.d3[q] = b.D3[2 - q]; }
  for (int q = 0; q < 4; q++) a.w.d4[q] = b.D4[3 + q];
  a.w.rs[0] = b.Drs[3][3]; a.w.rs[1] = b.Drs[3][4]; a.w.rs[2] = b.Drs[4][4];
  for (int u = 0; u < 2; u++)
    for (int q = 0; q < 3; q++) {
      a.w.rrs[u * 3 + q] = b.Drrs[1 - u][2 + q];
      a.w.rss[u * 3 + q] = b.Drss[2 + q][1 - u];
    }
  for (int q = 0; q < 3; q++) a.w.rrss[q] = b.Drrss[2][2 + q];
  a.w.rrss[3] = b.Drrss[3][3]; a.w.rrss[4] = b.Drrss[3][4]; a.w.rrss[5] = b.Drrss[4][4];
  for (int j = 0; j < SWEEP_MAX_STAGES; j++) {
    a.c0[j] = (R)rk.cc[j]; a.c1[j] = (R)rk.mew[j]; a.c2[j] = (R)rk.vv[j]; a.cf[j] = (R)(rk.mewt[j] * cpar);
  }
  return a;
}

template <typename R, int EV, int RB, bool PW2>
static int launch_sweep_t(Context& c, const SweepShape& s, const SweepArgs<R>& a) {
  constexpr int NT = sweep_threads<R, EV, RB>();
  static OncePerDevice lds;
  PT_TRY(allow_lds(c, lds, k_sweep<R, EV, RB, NT, PW2>, SWEEP_LDS_BYTES));
  hipLaunchKernelGGL((k_sweep<R, EV, RB, NT, PW2>), dim3(s.nblk), dim3(s.threads), s.lds, c.stream, a);
  return PT_OK;
}
template <typename R, int EV, bool PW2>
static int launch_sweep_rb(Context& c, int rb, const SweepShape& s, const SweepArgs<R>& a) {
  switch (rb) {
    case 1: return launch_sweep_t<R, EV, 1, PW2>(c, s, a);
    case 2: return launch_sweep_t<R, EV, 2, PW2>(c, s, a);
    default: return launch_sweep_t<R, EV, 4, PW2>(c, s, a);
  }
}
static int launch_sweep(Context& c, int l, int ev, int rb, const SweepShape& s, const SweepArgs<float>& a) {
  (void)l;
  if (ev == 0) return launch_sweep_rb<float, 0, true>(c, rb, s, a);
  return ev == 1 ? launch_sweep_rb<float, 1, true>(c, rb, s, a) : launch_sweep_rb<float, 2, true>(c, rb, s, a);
}
static int launch_sweep(Context& c, int l, int ev, int rb, const SweepShape& s, const SweepArgs<double>& a) {
  const LevelGeom& g = c.L[l].g;
  // all of the level's grid powers are products of dr and ds
  const bool pw2 = pow2(g.dr) && pow2(g.ds) && pow2(g.dr4) && pow2(g.ds4) && pow2(g.dr2ds2);
  if (ev == 0) return pw2 ? launch_sweep_rb<double, 0, true>(c, rb, s, a) : launch_sweep_rb<double, 0, false>(c, rb, s, a);
  return pw2 ? launch_sweep_rb<double, 1, true>(c, rb, s, a) : launch_sweep_rb<double, 1, false>(c, rb, s, a);
}

// one RKC1 sweep of level l (PS/iterative_solver.f90:1418-1614), the residual
// of its result into `res` when wanted.  The error buffer holds S0 throughout;
// launches read one pair of work buffers and write the other, and the last
// one's output replaces the error buffer by a pointer swap.  One tile that
// covers the level reads and writes the error buffer alone.
template <typename R>
static int sweep_level(Context& c, int l, bool f32, const LevelRkc& rk, double cpar, R* res) {
  Level& L = c.L[l];
  const LevelGeom& g = L.g;
  R** f[5];
  if constexpr (sizeof(R) == 4) {
    R** q[5] = {&L.ferr, &L.fB, &L.fC, &L.fD, &L.fE};
    std::copy(q, q + 5, f);
  } else {
    R** q[5] = {&L.err, &L.bufB, &L.bufC, &L.bufD, &L.bufE};
    std::copy(q, q + 5, f);
  }
  const SweepPlan& p = L.plan[f32];
  const int ev = sweep_form(c, l, f32), s = rk.s;
  const int nseg = (s + p.ns - 1) / p.ns, base = s / nseg, rem = s % nseg;
  const int tk = l == 1 ? PT_K_RKC_STAGE_L1 : PT_K_RKC_STAGE_COARSE;
  SweepArgs<R> a = sweep_args<R>(c, l, f32, rk, cpar);
  a.cw = p.cw; a.ch = p.ch; a.S0 = *f[0];
  int rd = 1, wr = 3, j0 = 1;
  for (int seg = 0; seg < nseg; seg++) {
    const int len = base + (seg < rem ? 1 : 0);
    const bool end = seg == nseg - 1;
    a.j0 = j0; a.ns = len; a.res = end ? res : nullptr;
    const SweepShape sh = sweep_shape(g.n, g.m, p.cw, p.ch, p.rb, len + (a.res ? 1 : 0), sizeof(R));
    if (sh.threads > sweep_threads_of(f32, ev, p.rb) || sh.lds > SWEEP_LDS_BYTES) {
      set_error("sweep tile too large");
      return PT_ERR_INVALID;
    }
    const bool alone = sh.nblk == 1 && nseg == 1;
    a.Gcur = j0 == 1 ? *f[0] : *f[rd];
    a.Gprev = j0 == 1 ? *f[0] : *f[rd + 1];
    a.Ocur = alone ? *f[0] : *f[wr];
    a.Oprev = end ? nullptr : *f[wr + 1];
    a.nbx = sh.nbx; a.w1 = sh.w1; a.nrb = sh.nrb; a.tcol = sh.tcol;
    if (c.timing) timer_begin(c, tk, (int64_t)len * (g.n - 1) * (g.m - 1));
    PT_TRY(launch_sweep(c, l, ev, p.rb, sh, a));
    if (c.timing) timer_end(c, tk);
    if (alone) return PT_OK;
    std::swap(rd, wr);
    j0 += len;
  }
  std::swap(*f[0], *f[rd]);
  return PT_OK;
}

static int launch_coarse_apply_wg(Context& c, const float* rhs, float* err, int n, int m, int pitch, float sz) {
  static OncePerDevice limit;
  PT_TRY(allow_lds(c, limit, k_coarse_apply_wg, SMALL_LDS_BYTES));
  const size_t lds = sizeof(double) * (1 + CA_SEG) * c.nci;
  if (lds > SMALL_LDS_BYTES) {
    set_error("coarsest grid too large for the single-workgroup coarse operator");
    return PT_ERR_UNSUPPORTED;
  }
  hipLaunchKernelGGL(k_coarse_apply_wg, dim3(1), dim3(SMALL_THREADS), lds, c.stream, c.Gc, rhs, err, n, m, pitch, sz);
  return PT_OK;
}

// residual of the smoothed field (compute_residual, PS/iterative_solver.f90:415-448)
template <typename R>
static int smoothed_residual(Context& c, int l, dim3 grd, dim3 blk, bool fp32, bool l1_sum) {
  Level& L = c.L[l];
  StageArgs<R> a = stage_base<R>(c, l, fp32);
  a.Sx = fp32 ? (R*)L.ferr : (R*)L.err;
  R* res = fp32 ? (R*)L.fres : (R*)L.res;
  int nb = grd.x * grd.y;
  launch_residual<R>(c, grd, blk, a, res, c.red);
  if (l1_sum) {
    // the L1 norm of the residual into device memory; level1_residual copies
    // it to the host after the cycle's launches (or graph replay)
    hipLaunchKernelGGL(k_reduce_final, dim3(1), dim3(256), 0, c.stream, c.red, nb, (int)RED_SUM_ABS, c.red_out);
  }
  return PT_OK;
}

// iterate_stream (Nmulti sweeps) and the residual after it where it is read
// (PS/iterative_solver.f90:1418-1614, 415-448)
template <typename R>
static int iterate_stream_t(Context& c, int l, int p, bool fp32, bool l1_sum) {
  Level& L = c.L[l];
  const LevelGeom& g = L.g;
  dim3 blk(TX, TZ), grd((g.n - 1 + TX - 1) / TX, (g.m - 1 + TZ * PZ - 1) / (TZ * PZ));
  // the residual is read by the stop test (level 1) and by the restriction
  // when the cycle goes down from here
  const bool want_res = l1_sum || c.cyc[p + 1] > c.cyc[p];
  if constexpr (sizeof(R) == 8) {
    if (c.P.RKC1 == 0) {
      // RK1: per iteration F = stream_space(S0) into B, then the update
      const int tk = l == 1 ? PT_K_RKC_STAGE_L1 : PT_K_RKC_STAGE_COARSE;
      const int dir = c.cyc[p + 1] > c.cyc[p] ? 0 : 1;
      dim3 b16(64, 4), gi((g.n - 1 + 63) / 64, (g.m - 1 + 3) / 4);
      for (int it = 1; it <= c.P.Nmulti; it++) {
        const int ntemp = c.P.Nmulti - it + 1;
        const double temp = std::cos((double)(2 * ntemp - 1) * 3.1415926535897932 / (double)(2 * c.P.Nmulti));
        StageArgs<R> a = stage_base<R>(c, l, false);
        a.Sx = L.err;
        if (c.timing) timer_begin(c, tk, (int64_t)(g.n - 1) * (g.m - 1));
        launch_residual<R>(c, grd, blk, a, L.bufB, c.red);
        hipLaunchKernelGGL(k_rk1_update, gi, b16, 0, c.stream, L.err, (const double*)L.bufB, L.dts, L.ratio, g.n,
                           g.m, g.pitch, temp, dir, (double)a.sz);
        if (c.timing) timer_end(c, tk);
      }
      return smoothed_residual<R>(c, l, grd, blk, fp32, l1_sum);
    }
  }
  const LevelRkc rk = level_rkc(c, l, fp32);
  // the residual of levels >= 2 comes out of the sweep's last launch; level
  // 1's carries the L1 sum, and that of the larger levels in the factorised form
  // is the unfactorised form's (a matter of its rounding, as in sweep_form)
  const bool fuse = want_res && l >= 2 && !(sweep_form(c, l, fp32) == 2 && (g.n - 1) * (g.m - 1) > 4096);
  R* res = fp32 ? (R*)L.fres : (R*)L.res;
  for (int it = 1; it <= c.P.Nmulti; it++) {
    int ntemp = c.P.Nmulti - it + 1;
    double temp = (c.P.Nmulti > 1) ? (c.P.c_2 - c.P.c_1) * (double)(ntemp - 1) / (double)(1 - c.P.Nmulti) : 0.0;
    PT_TRY(sweep_level<R>(c, l, fp32, rk, temp + c.P.c_2, fuse && it == c.P.Nmulti ? res : nullptr));
  }
  return want_res && !fuse ? smoothed_residual<R>(c, l, grd, blk, fp32, l1_sum) : PT_OK;
}

// smoother_vis (PS/smoother.f90:454-580) on the field set `vs` of level l
static int smoother_vis(Context& c, int l, VisSet& vs, int interpolate) {
  Level& L = c.L[l];
  const LevelGeom& g = L.g;
  const Tables& t = c.T;
  auto bcs = [&]() {
    int rows = (g.m + 7) * 3;
    hipLaunchKernelGGL(k_vis_bcs_side, dim3((rows + 255) / 256), dim3(256), 0, c.stream, vs.vis, g.n, g.m, g.pitch);
    int cols = (g.n + 1) * 3;
    hipLaunchKernelGGL(k_vis_bcs_tb, dim3((cols + 255) / 256), dim3(256), 0, c.stream, vs.vis, g.n, g.m, g.pitch);
  };
  int option, Niter;
  double lb, la;
  if (interpolate == 0) { option = 1; Niter = 3; lb = -3.0; la = -2.0; }
  else { option = 0; Niter = c.P.vis_iter; lb = -2.0; la = -1.0; }
  int Nvis_store = 0, nn_store = 1, n = 0;
  bool trigger = false;
  double ratio_min = 1.0e100;
  dim3 b16(64, 4);
  dim3 gnodes = grid2(g.n + 1, g.m + 1, b16);
  dim3 gint = grid2(g.n - 1, g.m - 1, b16);
  const int ivis0 = c.P.ivis == 0;
  // dt_stream for the level's own RKC1 stage count (the mixed path's coarse
  // levels may use fewer stages than nstageS)
  const LevelRkc rk = level_rkc(c, l, c.P.precision == PT_PREC_MIXED);
  double ae = -(rk.stability / 2.0), be = (double)rk.s;
  double ctemp = c.P.courant_stream * (rk.stability / (ae * ae));
  if (c.P.RKC1 == 0) {
    // RK1 (PS/iterative_solver.f90:1173-1186): dt = -2 courant eR/(eR^2+eI^2),
    // k_test_eig's RKC1 form with unit ellipse axes (eR/1 and eI/1 are exact)
    ae = 1.0; be = 1.0;
    ctemp = -(c.P.courant_stream * 2.0);
  }
  auto factor = [&](int nn) {
    const int ntemp = Niter - nn + 1;
    const double cc = 2.0 / (-lb - la + (lb - la) * std::cos((double)(2 * ntemp - 1) * 3.1415926535897932 / (double)(2 * Niter)));
    return 0.99 * cc;
  };
  // the first pass asks nothing of the gradients: its updates go several to a
  // launch, from vis to vsmooth (scratch until the gradients are taken) and
  // back.  (A grid less than 3 wide mirrors ghosts of ghosts.)
  if (!ivis0 && Niter >= 2 && g.n >= 3 && g.m >= 3) {
    VisSmooth a;
    a.dr2 = g.dr2; a.ds2 = g.ds2; a.rdr2 = 1.0 / g.dr2; a.rds2 = 1.0 / g.ds2; a.dtv = t.dt_vis[l];
    a.n = g.n; a.m = g.m; a.p = g.pitch;
    const int launches = 2 * ((Niter + 2 * VIS_ITS - 1) / (2 * VIS_ITS));
    for (int k = 0, nn = 1; k < launches; k++, nn += a.its) {
      a.its = (Niter - nn + 1 + launches - k - 1) / (launches - k);
      for (int q = 0; q < a.its; q++) a.cc[q] = factor(nn + q);
      a.in = k & 1 ? vs.vsmooth : vs.vis;
      a.out = k & 1 ? vs.vis : vs.vsmooth;
      a.ghosts = k + 1 == launches;
      const dim3 grid((g.n + 64 - 2 * a.its) / (64 - 2 * a.its), (g.m + VIS_TZ) / VIS_TZ);
      if (pow2(g.dr2) && pow2(g.ds2)) hipLaunchKernelGGL(k_vis_smooth<true>, grid, dim3(256), 0, c.stream, a);
      else hipLaunchKernelGGL(k_vis_smooth<false>, grid, dim3(256), 0, c.stream, a);
    }
    Nvis_store++;
    if (option == 1) { Niter = 6; lb = -2.0; la = -1.0; }
    n++;
  } else {
    bcs();
  }
  for (;;) {
    for (int nn = nn_store; nn <= Niter; nn++) {
      hipLaunchKernelGGL(k_vis_grad, gnodes, b16, 0, c.stream, vs, g.n, g.m, g.pitch, Nvis_store >= 1 ? 1 : 0, ivis0,
                         g.dr, g.ds, g.dr2, g.ds2, g.drds, t.dt_vis[l]);
      if (interpolate == 0 && (Nvis_store >= 1 || ivis0)) {
        hipLaunchKernelGGL(k_test_eig, gint, b16, 0, c.stream, vs, L.ratio, L.dts, g.n, g.m, g.pitch, t.SR1[l],
                           t.SR2[l], t.SR4[l], t.SR5[l], t.SR6[l], t.SI1[l], t.SI2[l], t.SI4[l], t.SI5[l], t.SI6[l],
                           ae, be, ctemp, c.red);
        int nb = gint.x * gint.y;
        hipLaunchKernelGGL(k_reduce_final, dim3(1), dim3(256), 0, c.stream, c.red, nb, (int)RED_MIN, c.red_out);
        PT_HIP(hipMemcpyAsync(c.h_red, c.red_out, sizeof(double), hipMemcpyDeviceToHost, c.stream));
        PT_HIP(hipStreamSynchronize(c.stream));
        // the reference's loop starts from 1e100 and keeps it where every
        // ratio is +Inf (eigI = 0, isoviscous): PS/smoother.f90:501-506
        ratio_min = std::min(1.0e100, c.h_red[0]);
      }
      if (option == 1) {
        if ((Nvis_store >= 1 && ratio_min > c.P.eig_ratio_min) || ivis0 || n > 20) {
          c.eig_fine = ratio_min;   // module variables eig_fine, n_eta: last call wins
          c.n_eta = n;
          trigger = true;
          break;
        }
      } else if (interpolate >= 1 && (Nvis_store >= 1 || ivis0)) {
        trigger = true;
        break;
      }
      hipLaunchKernelGGL(k_vis_update, gnodes, b16, 0, c.stream, vs.vis, vs.vsmooth, g.n, g.m, g.pitch, factor(nn));
      if (g.n < 3 || g.m < 3) bcs();
    }
    if (trigger) break;
    Nvis_store++;
    nn_store = 1;
    if (option == 1) { Niter = 6; lb = -2.0; la = -1.0; }
    n++;
  }
  return PT_OK;
}

// compute_viscosity (Newtonian, static=1): PS/iterative_solver.f90:560-634.
// The reference saves and restores the finer level's fields around the
// restriction; here the finer level is smoothed in its scratch set instead.
static int compute_viscosity(Context& c, int l) {
  Level& L = c.L[l];
  const LevelGeom& g = L.g;
  dim3 b16(64, 4);
  size_t bytes = sizeof(double) * L.nelem;
  if (l == 1) {
    const double lvT = std::log(c.P.visT), lvC = std::log(c.P.visC), lvP = std::log(c.P.visP);
    hipLaunchKernelGGL(k_visf, grid2(g.n + 1, g.m + 1, b16), b16, 0, c.stream, c.Tvis, c.Cvis, L.vis_static, g.n, g.m,
                       g.pitch, g.n + 11, c.P.ivis, lvT, lvC, lvP, c.T.ds, c.P.RaT != 0.0 ? 1 : 0);
    PT_HIP(hipMemcpyAsync(L.v.vis, L.vis_static, bytes, hipMemcpyDeviceToDevice, c.stream));
    return smoother_vis(c, 1, L.v, 0);
  }
  Level& F = c.L[l - 1];
  size_t fbytes = sizeof(double) * F.nelem;
  PT_HIP(hipMemcpyAsync(F.vs.vis, F.vis_static, fbytes, hipMemcpyDeviceToDevice, c.stream));
  PT_TRY(smoother_vis(c, l - 1, F.vs, 1));
  hipLaunchKernelGGL((k_restrict<double, double>), grid2(g.n - 1, g.m - 1, b16), b16, 0, c.stream, F.vs.vis,
                     F.g.pitch, L.v.vis, g.n, g.m, g.pitch);
  int tmax = std::max(g.n + 1, g.m - 1);
  hipLaunchKernelGGL(k_vis_bcs_init_boundary, dim3((tmax + 255) / 256), dim3(256), 0, c.stream, L.v.vis, F.vs.vis,
                     g.n, g.m, g.pitch, F.g.n, F.g.m, F.g.pitch);
  int ts = (g.m + 1) * 3;
  hipLaunchKernelGGL(k_vis_bcs_init_side, dim3((ts + 255) / 256), dim3(256), 0, c.stream, L.v.vis, g.n, g.m, g.pitch);
  int tt = (g.n + 7) * 3;
  hipLaunchKernelGGL(k_vis_bcs_init_tb, dim3((tt + 255) / 256), dim3(256), 0, c.stream, L.v.vis, g.n, g.m, g.pitch);
  PT_HIP(hipMemcpyAsync(L.vis_static, L.v.vis, bytes, hipMemcpyDeviceToDevice, c.stream));
  return smoother_vis(c, l, L.v, 0);
}

int launch_equilibrate(Context& c, double* ab, double* row, int n, int kl, int ku) {
  hipLaunchKernelGGL(k_coarse_equilibrate, dim3((n + 127) / 128), dim3(128), 0, c.stream, ab, row, n, kl, ku);
  return PT_OK;
}

static int coarse_factor(Context& c) {
  const Tables& t = c.T;
  Level& G = c.L[t.grids];
  CoarseArgs a;
  a.vis = G.v.vis; a.vxm = G.v.vxxmzz; a.vxz = G.v.vxz; a.vx = G.v.vx; a.vz = G.v.vz;
  a.nxc = G.g.n; a.nzc = G.g.m; a.p = G.g.pitch; a.kl = t.kl; a.ku = t.ku; a.ngc = t.ngc;
  a.ivis0 = c.P.ivis == 0; a.Vbc = c.P.Vbc;
  std::memcpy(a.SM1, t.SM1, sizeof a.SM1); std::memcpy(a.SM2, t.SM2, sizeof a.SM2);
  std::memcpy(a.SM4, t.SM4, sizeof a.SM4); std::memcpy(a.SM5, t.SM5, sizeof a.SM5);
  std::memcpy(a.SM6, t.SM6, sizeof a.SM6);
  size_t mbytes = sizeof(double) * (size_t)(2 * t.kl + t.ku + 1) * t.ngc;
  PT_HIP(hipMemsetAsync(c.Mc, 0, mbytes, c.stream));
  hipLaunchKernelGGL(k_coarse_assemble, dim3((t.ngc + 127) / 128), dim3(128), 0, c.stream, a, c.Mc, c.RowB);
  hipLaunchKernelGGL(k_coarse_equilibrate, dim3((t.ngc + 127) / 128), dim3(128), 0, c.stream, c.Mc, c.RowB, t.ngc,
                     t.kl, t.ku);
  hipLaunchKernelGGL(k_band_lu, dim3(1), dim3(64), 0, c.stream, c.Mc, c.ipiv, t.ngc, t.kl, t.ku, c.d_info);
  int32_t info = 0;
  PT_HIP(hipMemcpyAsync(&info, c.d_info, sizeof(int32_t), hipMemcpyDeviceToHost, c.stream));
  PT_HIP(hipStreamSynchronize(c.stream));
  if (info != 0) {
    set_error("coarse-grid band LU: zero pivot at column " + std::to_string(info));
    return PT_ERR_SINGULAR_COARSE;
  }
  hipLaunchKernelGGL(k_coarse_inverse, dim3(c.nci), dim3(64), sizeof(double) * t.ngc, c.stream, c.Mc, c.ipiv,
                     c.RowB, c.Gc, t.ngc, t.kl, t.ku, G.g.n, G.g.m);
  return PT_OK;
}

int compute_rhs1(Context& c) {
  Level& L = c.L[1];
  dim3 b16(64, 4);
  const double* D1 = c.T.D1;
  hipLaunchKernelGGL(k_rhs1, grid2(c.T.nx - 1, c.T.nz - 1, b16), b16, 0, c.stream, c.Tbuoy, c.Cbuoy, L.rhs, c.T.nx,
                     c.T.nz, L.g.pitch, c.T.nx + 11, c.T.dr, c.P.RaT, c.P.RaC, D1[1], D1[2], D1[3], D1[4], D1[5]);
  return PT_OK;
}

// FP64 copies of the FP32 mirrors (mixed precision): coefficients per solve
__global__ void k_to_f32(const double* a, float* b, long n) {
  long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t < n) b[t] = (float)a[t];
}
__global__ void k_add_f32_to_f64(double* psi, const float* e, int n, int m, int p, double sz) {
  int i = 1 + blockIdx.x * blockDim.x + threadIdx.x, k = 1 + blockIdx.y * blockDim.y + threadIdx.y;
  if (i > n - 1 || k > m - 1) return;
  double y = psi[IDX(i, k, p)] + (double)e[IDX(i, k, p)];
  store_with_ghosts<double>(psi, i, k, n, m, p, y, sz);
}

static int to_f32(Context& c, const double* a, float* b, size_t n) {
  hipLaunchKernelGGL(k_to_f32, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, c.stream, a, b, (long)n);
  return PT_OK;
}

__global__ void k_fill_f32(float* v, long n) {
  long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t < n) v[t] = 0.0f;
}

// schedule entry p of the cycle (PS/iterative_solver.f90:143-340): the
// restriction into its level when the schedule descends, the visit (RKC1
// smoothing + residual, or the coarse solve), and the prolongation when it
// ascends next.  Kernel launches only (so a captured cycle holds kernel nodes
// and nothing else): a level-1 visit leaves the residual's L1 norm in
// device memory (red_out), which level1_residual copies to the host.
static int visit(Context& c, int p, bool mixed) {
  const Tables& t = c.T;
  const int* multi = c.cyc;
  dim3 b16(64, 4);
  const double sz = c.P.Vbc == 0 ? -1.0 : 1.0;
  const int l = multi[p];
  Level& L = c.L[l];
  if (multi[p - 1] < multi[p] && l >= 2 && mixed && c.coarse_zero && l < t.grids)
    hipLaunchKernelGGL(k_fill_f32, dim3((unsigned)((L.nelem + 255) / 256)), dim3(256), 0, c.stream, L.ferr,
                       (long)L.nelem);
  if (multi[p - 1] < multi[p] && l >= 2) {
    // compute_RHS(l) = restrict(residual(l-1))
    Level& F = c.L[l - 1];
    if (!mixed)
      hipLaunchKernelGGL((k_restrict<double, double>), grid2(L.g.n - 1, L.g.m - 1, b16), b16, 0, c.stream, F.res,
                         F.g.pitch, L.rhs, L.g.n, L.g.m, L.g.pitch);
    else if (l == 2)
      hipLaunchKernelGGL((k_restrict<double, float>), grid2(L.g.n - 1, L.g.m - 1, b16), b16, 0, c.stream, F.res,
                         F.g.pitch, L.frhs, L.g.n, L.g.m, L.g.pitch);
    else
      hipLaunchKernelGGL((k_restrict<float, float>), grid2(L.g.n - 1, L.g.m - 1, b16), b16, 0, c.stream, F.fres,
                         F.g.pitch, L.frhs, L.g.n, L.g.m, L.g.pitch);
  }
  if (l < t.grids) {
    if (!mixed) {
      PT_TRY(iterate_stream_t<double>(c, l, p, false, l == 1));
    } else if (l == 1) {
      // FP64 defect -> FP32 RKC1 smoothing of the correction -> FP64 update
      StageArgs<double> a = stage_base<double>(c, 1, false);
      a.Sx = L.err;
      dim3 blk(TX, TZ), grd((L.g.n - 1 + TX - 1) / TX, (L.g.m - 1 + TZ * PZ - 1) / (TZ * PZ));
      launch_residual<double>(c, grd, blk, a, c.dres64, c.red);
      PT_TRY(to_f32(c, c.dres64, L.frhs, L.nelem));
      hipLaunchKernelGGL(k_fill_f32, dim3((unsigned)((L.nelem + 255) / 256)), dim3(256), 0, c.stream, L.ferr,
                         (long)L.nelem);
      PT_TRY(iterate_stream_t<float>(c, 1, p, true, false));
      hipLaunchKernelGGL(k_add_f32_to_f64, grid2(L.g.n - 1, L.g.m - 1, b16), b16, 0, c.stream, L.err, L.ferr,
                         L.g.n, L.g.m, L.g.pitch, sz);
      launch_residual<double>(c, grd, blk, a, L.res, c.red);
      int nb = grd.x * grd.y;
      hipLaunchKernelGGL(k_reduce_final, dim3(1), dim3(256), 0, c.stream, c.red, nb, (int)RED_SUM_ABS, c.red_out);
    } else if (l >= c.presmooth_from && c.coarse_zero && multi[p - 1] < multi[p] && multi[p + 1] > multi[p]) {
      // no smoothing on the way down: a level entered from the finer one
      // and left for the coarser one starts its correction from zero, so
      // the residual restricted next is the level's right-hand side (the
      // turning visits of F- and W-cycles, entered from a coarser level,
      // carry a prolonged correction and are smoothed)
      StageArgs<float> a = stage_base<float>(c, l, true);
      a.Sx = L.ferr;
      dim3 blk(TX, TZ), grd((L.g.n - 1 + TX - 1) / TX, (L.g.m - 1 + TZ * PZ - 1) / (TZ * PZ));
      launch_residual<float>(c, grd, blk, a, L.fres, c.red);
    } else {
      PT_TRY(iterate_stream_t<float>(c, l, p, true, false));
    }
  } else {
    // Compute_coarse_vector + DGBTRS + Stream_grid_coarse + enforceBCs_stream
    // as one dense matvec with the operator built from the LU factors
    dim3 gb((c.nci + 255) / 256);
    size_t sh = sizeof(double) * c.nci;
    if (!mixed)
      hipLaunchKernelGGL((k_coarse_apply<double, double>), gb, dim3(256), sh, c.stream, c.Gc, L.rhs, L.err, L.g.n,
                         L.g.m, L.g.pitch, sz);
    else
      PT_TRY(launch_coarse_apply_wg(c, L.frhs, L.ferr, L.g.n, L.g.m, L.g.pitch, (float)sz));
  }
  if (l > 1 && multi[p + 1] < multi[p]) {
    Level& F = c.L[l - 1];
    dim3 gp = grid2(F.g.n - 1, F.g.m - 1, b16);
    if (!mixed)
      hipLaunchKernelGGL((k_prolong<double, double>), gp, b16, 0, c.stream, L.err, L.g.pitch, F.err, F.g.n, F.g.m,
                         F.g.pitch, sz);
    else if (l - 1 == 1)
      hipLaunchKernelGGL((k_prolong<float, double>), gp, b16, 0, c.stream, L.ferr, L.g.pitch, F.err, F.g.n,
                         F.g.m, F.g.pitch, sz);
    else
      hipLaunchKernelGGL((k_prolong<float, float>), gp, b16, 0, c.stream, L.ferr, L.g.pitch, F.ferr, F.g.n,
                         F.g.m, F.g.pitch, (float)sz);
  }
  return PT_OK;
}

// FP64 residual RHS - L psi of a level-1 iterate (compute_residual's operator
// with the level's current viscosity set) into res, and sum |res| on the host
int level1_residual_of(Context& c, const double* psi, double* res, double* l1) {
  Level& L = c.L[1];
  StageArgs<double> a = stage_base<double>(c, 1, false);
  a.Sx = psi;
  dim3 blk(TX, TZ), grd((L.g.n - 1 + TX - 1) / TX, (L.g.m - 1 + TZ * PZ - 1) / (TZ * PZ));
  launch_residual<double>(c, grd, blk, a, res, c.red);
  const int nb = grd.x * grd.y;
  hipLaunchKernelGGL(k_reduce_final, dim3(1), dim3(256), 0, c.stream, c.red, nb, (int)RED_SUM_ABS, c.red_out);
  PT_HIP(hipMemcpyAsync(c.h_red, c.red_out, sizeof(double), hipMemcpyDeviceToHost, c.stream));
  PT_HIP(hipStreamSynchronize(c.stream));
  *l1 = c.h_red[0];
  return PT_OK;
}

// residual_mag(1) of the level-1 visit just enqueued, and the abnormal-
// residual stop (PS/iterative_solver.f90:438-447)
static int level1_residual(Context& c, double* resmag1) {
  PT_HIP(hipMemcpyAsync(c.h_red, c.red_out, sizeof(double), hipMemcpyDeviceToHost, c.stream));
  PT_HIP(hipStreamSynchronize(c.stream));
  const LevelGeom& g = c.L[1].g;
  *resmag1 = c.h_red[0] / (double)(g.n - 2) / (double)(g.m - 2);
  if (*resmag1 > 1.0e10 * c.res_ref1) {
    set_error("residual " + std::to_string(*resmag1) + " > 1e10 * res_ref");
    return PT_ERR_HIGH_RESIDUAL;
  }
  return PT_OK;
}

// The level buffers whose roles rotate: a sweep of several tiles swaps its
// level's error buffer with a work buffer, so a cycle may start from one of a few
// arrangements, and a replay must leave the pointers as the eager launches
// would have.
static void buffer_roles(Context& c, std::vector<void*>& out) {
  out.clear();
  for (int l = 1; l <= c.T.grids; l++) {
    Level& L = c.L[l];
    out.insert(out.end(), {(void*)L.ferr, (void*)L.fB, (void*)L.fC, (void*)L.fD, (void*)L.fE, (void*)L.err,
                           (void*)L.bufB, (void*)L.bufC, (void*)L.bufD, (void*)L.bufE});
  }
}
static void restore_roles(Context& c, const std::vector<void*>& v) {
  size_t j = 0;
  for (int l = 1; l <= c.T.grids; l++) {
    Level& L = c.L[l];
    float** f[5] = {&L.ferr, &L.fB, &L.fC, &L.fD, &L.fE};
    double** d[5] = {&L.err, &L.bufB, &L.bufC, &L.bufD, &L.bufE};
    for (float** q : f) *q = (float*)v[j++];
    for (double** q : d) *q = (double*)v[j++];
  }
}

// visits 2..nsteps of a cycle and visit 1 of the next.  After one eager run
// the sequence is captured as a HIP graph (kernel nodes only) per starting
// arrangement of the rotating buffers (at most MAX_CYCLE_GRAPHS) and
// replayed; the graphs' kernel arguments (buffers, level constants) do not
// change between cycles or solves of a context.  PT_GRAPH=0 at pt_create,
// per-kernel timing, a failed capture or more arrangements keep the launches
// eager; the results are the same either way.
static constexpr size_t MAX_CYCLE_GRAPHS = 4;
static int rest_and_next_level1(Context& c, bool mixed) {
  auto enqueue = [&]() -> int {
    for (int p = 2; p <= c.cyc_n; p++) PT_TRY(visit(c, p, mixed));
    return visit(c, 1, mixed);
  };
  if (!c.use_graph || c.timing || c.graph_state < 0) return enqueue();
  if (c.graph_state == 0) {
    c.graph_state = 1;   // the first run is eager (sets the kernels' attributes)
    return enqueue();
  }
  c.graph_state = 2;
  std::vector<void*> before;
  buffer_roles(c, before);
  for (const Context::CycleGraph& cg : c.cycle_graphs) {
    if (cg.before != before) continue;
    PT_HIP(hipGraphLaunch(cg.exec, c.stream));
    restore_roles(c, cg.after);
    return PT_OK;
  }
  if (c.cycle_graphs.size() >= MAX_CYCLE_GRAPHS) {
    c.graph_state = -1;
    return enqueue();
  }
  // capture: the launches are recorded, not run, while the host-side pointer
  // swaps take effect; the replay below then runs them
  Context::CycleGraph cg;
  cg.before = before;
  PT_HIP(hipStreamBeginCapture(c.stream, hipStreamCaptureModeThreadLocal));
  const int rc = enqueue();
  hipError_t e = hipStreamEndCapture(c.stream, &cg.graph);
  if (rc != PT_OK || e != hipSuccess) {
    if (cg.graph) (void)hipGraphDestroy(cg.graph);
    restore_roles(c, before);
    c.graph_state = -1;
    if (rc != PT_OK) return rc;
    return enqueue();
  }
  buffer_roles(c, cg.after);
  e = hipGraphInstantiate(&cg.exec, cg.graph, nullptr, nullptr, 0);
  if (e != hipSuccess) {
    // nothing of the capture ran: back to the starting arrangement, eager from now on
    (void)hipGraphDestroy(cg.graph);
    restore_roles(c, before);
    c.graph_state = -1;
    return enqueue();
  }
  c.cycle_graphs.push_back(std::move(cg));
  PT_HIP(hipGraphLaunch(c.cycle_graphs.back().exec, c.stream));
  return PT_OK;
}

// multigrid: PS/iterative_solver.f90:124-341
static int multigrid_body(Context& c);
int multigrid(Context& c) {
  if (c.timing) timer_begin(c, PT_K_SOLVE);
  const int rc = multigrid_body(c);
  if (c.timing) timer_end(c, PT_K_SOLVE);
  return rc;
}

static int multigrid_body(Context& c) {
  const Tables& t = c.T;
  const bool mixed = c.P.precision == PT_PREC_MIXED;
  Level& L1 = c.L[1];
  size_t b1 = sizeof(double) * L1.nelem;
  PT_HIP(hipMemcpyAsync(L1.err, c.SF, b1, hipMemcpyDeviceToDevice, c.stream));
  PT_TRY(compute_rhs1(c));
  double rr;
  PT_TRY(reduce_to_host(c, L1.rhs, t.nx - 1, t.nz - 1, L1.g.pitch, 4, RED_SUM_ABS, &rr));
  c.res_ref1 = rr / (double)(t.nx - 2) / (double)(t.nz - 2);
  for (int l = 1; l <= t.grids; l++) PT_TRY(compute_viscosity(c, l));
  if (c.first_solve || c.P.ivis > 0) {
    PT_TRY(coarse_factor(c));
    c.first_solve = false;
  }
  if (mixed) {
    for (int l = 1; l <= t.grids; l++) {
      Level& L = c.L[l];
      PT_TRY(to_f32(c, L.v.vis, L.fvis, L.nelem)); PT_TRY(to_f32(c, L.v.vxxmzz, L.fvxm, L.nelem));
      PT_TRY(to_f32(c, L.v.vxz, L.fvxz, L.nelem)); PT_TRY(to_f32(c, L.v.vx, L.fvx, L.nelem));
      PT_TRY(to_f32(c, L.v.vz, L.fvz, L.nelem)); PT_TRY(to_f32(c, L.dts, L.fdts, L.nelem));
      // coarse corrections of the mixed path start each solve from zero
      if (l >= 2)
        hipLaunchKernelGGL(k_fill_f32, dim3((unsigned)((L.nelem + 255) / 256)), dim3(256), 0, c.stream, L.ferr,
                           (long)L.nelem);
    }
  }
  if (c.guess_net) PT_TRY(learned_before_solve(c));
  int q = 1;
  double resmag1 = 0.0;
  // cycle q: visit 1 (level 1, ends with its residual's L1 norm on the host),
  // then visits 2..nsteps; the stop test follows every level-1 visit
  PT_TRY(visit(c, 1, mixed));
  int rc = level1_residual(c, &resmag1);
  if (rc != PT_OK) { c.last_q = q; return rc; }
  while (!((resmag1 / c.res_ref1) <= c.P.tolerance)) {
    if (q + 1 > c.P.max_cycles) {
      for (int p = 2; p <= c.cyc_n; p++) PT_TRY(visit(c, p, mixed));
      c.cycles++;
      set_error("q > max_cycles = " + std::to_string(c.P.max_cycles));
      return PT_ERR_MAX_CYCLES;
    }
    PT_TRY(rest_and_next_level1(c, mixed));
    c.cycles++;
    q++;
    rc = level1_residual(c, &resmag1);
    if (rc != PT_OK) { c.last_q = q; return rc; }   // the cycle the reference stops at
  }
  c.cycles++;
  if (c.guess_net) PT_TRY(learned_after_solve(c));
  PT_HIP(hipMemcpyAsync(c.SF, L1.err, b1, hipMemcpyDeviceToDevice, c.stream));
  c.last_q = q;
  c.residual1 = resmag1;
  c.solves++;
  return PT_OK;
}

int stream_bcs(Context& c, double* S) {
  dim3 b16(64, 4);
  hipLaunchKernelGGL(k_stream_bcs, grid2(c.T.nx + 7, c.T.nz + 7, b16), b16, 0, c.stream, S, c.T.nx, c.T.nz,
                     c.T.nx + 7, c.P.Vbc == 0 ? -1.0 : 1.0);
  return PT_OK;
}

int compute_velocities(Context& c) {
  dim3 b16(64, 4);
  const double* D1 = c.T.D1;
  int p = c.T.nx + 7;
  hipLaunchKernelGGL(k_velocities, grid2(c.T.nx + 1, c.T.nz + 1, b16), b16, 0, c.stream, c.SF, c.u, c.w, c.T.nx,
                     c.T.nz, p, c.T.dr, c.T.ds, D1[1], D1[2], D1[3], D1[4], D1[5]);
  hipLaunchKernelGGL(k_velocity_bcs, grid2(c.T.nx + 7, c.T.nz + 7, b16), b16, 0, c.stream, c.u, c.w, c.T.nx, c.T.nz,
                     p, c.P.Vbc);
  return PT_OK;
}

// ---------------------------------------------------------------------------
// allocation
// ---------------------------------------------------------------------------
static int dalloc(void** p, size_t bytes) {
  PT_HIP(hipMalloc(p, bytes));
  PT_HIP(hipMemset(*p, 0, bytes));
  return PT_OK;
}
#define DALLOC(ptr, bytes) PT_TRY(dalloc((void**)&(ptr), (bytes)))

int solver_alloc(Context& c) {
  const Tables& t = c.T;
  for (int l = 1; l <= t.grids; l++) {
    Level& L = c.L[l];
    LevelGeom& g = L.g;
    g.n = t.nxg[l]; g.m = t.nzg[l]; g.pitch = g.n + 7;
    g.dr = t.drg[l]; g.ds = t.dsg[l]; g.dr2 = t.dr2g[l]; g.ds2 = t.ds2g[l]; g.dr3 = t.dr3g[l]; g.ds3 = t.ds3g[l];
    g.dr4 = t.dr4g[l]; g.ds4 = t.ds4g[l]; g.drds = t.drdsg[l]; g.drds2 = t.drds2g[l]; g.dr2ds = t.dr2dsg[l];
    g.dr2ds2 = t.dr2ds2g[l];
    L.nelem = (size_t)(g.n + 7) * (g.m + 7);
    size_t b = sizeof(double) * L.nelem, f = sizeof(float) * L.nelem;
    DALLOC(L.err, b); DALLOC(L.bufB, b); DALLOC(L.bufC, b); DALLOC(L.bufD, b); DALLOC(L.bufE, b); DALLOC(L.rhs, b); DALLOC(L.res, b);
    DALLOC(L.dts, b); DALLOC(L.ratio, b); DALLOC(L.vis_static, b);
    VisSet* sets[2] = {&L.v, &L.vs};
    for (VisSet* s : sets) {
      DALLOC(s->vis, b); DALLOC(s->vx, b); DALLOC(s->vz, b); DALLOC(s->vxx, b); DALLOC(s->vzz, b);
      DALLOC(s->vxz, b); DALLOC(s->vxxpzz, b); DALLOC(s->vxxmzz, b); DALLOC(s->vsmooth, b);
    }
    if (c.P.precision == PT_PREC_MIXED) {
      DALLOC(L.ferr, f); DALLOC(L.fB, f); DALLOC(L.fC, f); DALLOC(L.fD, f); DALLOC(L.fE, f); DALLOC(L.fres, f); DALLOC(L.frhs, f);
      DALLOC(L.fdts, f); DALLOC(L.fvis, f); DALLOC(L.fvxm, f); DALLOC(L.fvxz, f); DALLOC(L.fvx, f); DALLOC(L.fvz, f);
    }
  }
  const bool f32 = c.P.precision == PT_PREC_MIXED;
  for (int l = 1; l < t.grids && c.P.iterate == 1; l++) c.L[l].plan[f32] = sweep_plan(c, l, f32, level_rkc(c, l, f32).s);
  if (c.P.precision == PT_PREC_MIXED) DALLOC(c.dres64, sizeof(double) * c.L[1].nelem);
  DALLOC(c.d_info, sizeof(int32_t));
  if (c.P.iterate == 1) {   // the coarsest-grid operator of the multigrid path
    size_t mb = sizeof(double) * (size_t)(2 * t.kl + t.ku + 1) * t.ngc;
    if (t.ngc > 4096) {
      set_error("coarsest grid has more than 4096 unknowns");
      return PT_ERR_UNSUPPORTED;
    }
    DALLOC(c.Mc, mb); DALLOC(c.RowB, sizeof(double) * t.ngc); DALLOC(c.Bc, sizeof(double) * t.ngc);
    c.nci = (t.nxg[t.grids] - 1) * (t.nzg[t.grids] - 1);
    DALLOC(c.Gc, sizeof(double) * (size_t)c.nci * c.nci);
    DALLOC(c.ipiv, sizeof(int32_t) * t.ngc);
  }
  c.red_cap = 1 << 20;
  DALLOC(c.red, sizeof(double) * c.red_cap);
  DALLOC(c.red_out, sizeof(double) * 16);
  PT_HIP(hipHostMalloc((void**)&c.h_red, sizeof(double) * 16, hipHostMallocDefault));
  // stencil constants
  for (int q = 0; q < 5; q++) { c.st.D1[q] = t.D1[q + 1]; c.st.D2[q] = t.D2[q + 1]; }
  for (int q = 0; q < 7; q++) { c.st.D3[q] = t.D3[q]; c.st.D4[q] = t.D4[q]; }
  for (int b = 0; b < 5; b++)
    for (int q = 0; q < 5; q++) {
      c.st.Drs[b][q] = t.Drs[b + 1][q + 1]; c.st.Drss[b][q] = t.Drss[b + 1][q + 1];
      c.st.Drrs[b][q] = t.Drrs[b + 1][q + 1]; c.st.Drrss[b][q] = t.Drrss[b + 1][q + 1];
    }
  return PT_OK;
}

int solver_free(Context& c) {
  for (int l = 1; l <= c.T.grids; l++) {
    Level& L = c.L[l];
    void* ps[] = {L.err, L.bufB, L.bufC, L.bufD, L.bufE, L.fres, L.rhs, L.res, L.dts, L.ratio, L.vis_static, L.v.vis, L.v.vx, L.v.vz,
                  L.v.vxx, L.v.vzz, L.v.vxz, L.v.vxxpzz, L.v.vxxmzz, L.v.vsmooth, L.vs.vis, L.vs.vx, L.vs.vz,
                  L.vs.vxx, L.vs.vzz, L.vs.vxz, L.vs.vxxpzz, L.vs.vxxmzz, L.vs.vsmooth, L.ferr, L.fB, L.fC, L.fD, L.fE,
                  L.frhs, L.fdts, L.fvis, L.fvxm, L.fvxz, L.fvx, L.fvz};
    for (void* p : ps)
      if (p) (void)hipFree(p);
  }
  void* ps[] = {c.Mc, c.RowB, c.Bc, c.ipiv, c.d_info, c.red, c.red_out, c.dres64, c.Gc, c.lg_res, c.lg_res2, c.lg_psi, c.stats_rows,
                c.strain_buf};
  for (void* p : ps)
    if (p) (void)hipFree(p);
  if (c.h_red) (void)hipHostFree(c.h_red);
  for (Context::CycleGraph& cg : c.cycle_graphs) {
    if (cg.exec) (void)hipGraphExecDestroy(cg.exec);
    if (cg.graph) (void)hipGraphDestroy(cg.graph);
  }
  c.cycle_graphs.clear();
  return PT_OK;
}

}  // namespace pt
