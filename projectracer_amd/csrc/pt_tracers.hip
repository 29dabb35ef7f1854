// pt_tracers.hip -- Lagrangian tracer pipeline on gfx950.
//
//   k_bin            nint binning of tracer positions to node dual cells + domain
//                    check (PS/composition.f90:1002-1011)
//   k_cs_count/scan/fill  stable counting sort of (cell, slot) pairs that reads
//                    each cell's tracers from the storage order's neighbouring
//                    cells (the tracers move less than a cell per stage);
//                    (rocPRIM) stable radix sort when the storage order is not
//                    that of a previous projection or a tracer moved farther
//   k_cell_bounds    run bounds per cell after the radix sort (nempty = run length)
//   k_cell_reduce    per-cell sums of T*w, C*w, w for the 3x3 neighbour nodes
//                    (shape_func, PS/composition.f90:896-921), fixed order
//   k_node_combine   node = sum of its 9 cells' partials in a fixed order;
//                    Tratio/Cnew = ratio where sum w > 0 (PS/composition.f90:942-1070)
//   k_reorder        keeps the tracer SoA in cell order (ID map for host copies)
//   k_sym_* / k_t_*  enforceBCs / extendT / enforceBCs_comp
//                    (PS/energy.f90:558-630, PS/composition.f90:1279-1292)
//   k_filter_passes  smoother_time / smoother_time_T: checks and Richardson passes,
//                    several per launch on LDS tiles (PS/smoother.f90:582-672,
//                    75-139); k_smoothness / k_filter: the host-driven loop's
//   k_conduct_*      load_conductivity_array (PS/energy.f90:59-86)
//   k_source         tracer_space_uniform (PS/energy.f90:135-151)
//   k_itab           compute_derivatives for u, w and the source into one
//                    interleaved interpolation table (PS/composition.f90:1457-1478)
//   k_rk1..k_rk4     interpolate (x3) + the RK4 stage updates of energy_time
//                    (PS/composition.f90:1359-1393, PS/energy.f90:258-537)
#include <cmath>
#include <cstdint>
#include <cstring>
#include <algorithm>
#include "pt_internal.hpp"
#include "pt_quotient.hpp"

namespace pt {

#define I3(i, k, p) ((long)((k) + 3) * (p) + ((i) + 3))
#define I5(i, k, p) ((long)((k) + 5) * (p) + ((i) + 5))

static dim3 grid2(int ni, int nk, dim3 b) { return dim3((ni + b.x - 1) / b.x, (nk + b.y - 1) / b.y); }

// nint(x) for the reference's NINT: round half away from zero
__device__ __forceinline__ int nint(double x) { return (int)round(x); }

// ---------------------------------------------------------------------------
// binning, stable sort by cell, per-cell sums, node combine
// ---------------------------------------------------------------------------
// key = dual cell of nint(r/dr), nint(s/ds); positions outside the domain
// (or NaN) raise flag 0 and get the sentinel key ncell (sorted last).  With
// the storage order's cells (okey), a tracer whose cell is more than one
// cell from its slot's in either direction raises flag 1.
__global__ void k_bin(const double* r, const double* s, int64_t n, int nx, int nz, double dr, double ds,
                      double aspect, int32_t* key, int32_t* flags, const int32_t* okey) {
  // one flag store per wavefront that raises it: an under-resolved flow can
  // move half the tracers farther than a cell, and same-address atomics
  // from every one of them serialize
  const int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const bool live = j < n;
  const int ncell = (nx + 1) * (nz + 1);
  bool outside = false, far = false;
  if (live) {
    const double rv = r[j], sv = s[j];
    if (!(rv >= 0.0 && rv <= aspect && sv >= 0.0 && sv <= 1.0)) {
      outside = true;
      key[j] = ncell;
    } else {
      const int i = nint(rv / dr), k = nint(sv / ds);
      key[j] = k * (nx + 1) + i;
      if (okey) {
        const int o = okey[j], oi = o % (nx + 1), ok = o / (nx + 1);
        far = abs(oi - i) > 1 || abs(ok - k) > 1;
      }
    }
  }
  const unsigned long long bo = __ballot(outside), bf = __ballot(far);
  if ((threadIdx.x & 63) == 0) {
    if (bo) atomicOr(&flags[0], 1);
    if (bf) atomicOr(&flags[1], 1);
  }
}

// ---------------------------------------------------------------------------
// Stable counting sort of the (cell, slot) pairs when the tracers are stored
// in the cell order of an earlier projection and none moved more than one
// cell from its slot's cell.  A block owns CS_CELLS consecutive cells of one
// row; every tracer now in them is stored in the slot ranges of the cells of
// the three rows around, one column beyond the block's on each side.  Those
// three windows are read in ascending slot order, so each cell's tracers are
// found in ascending slot order: the result (perm, skey, cstart, cend) is the
// one the stable radix sort gives, element for element.
// ---------------------------------------------------------------------------
constexpr int CS_CELLS = 64;
constexpr int CS_THREADS = 256;

struct CsBlock {
  int cfirst, ncb, nwin, lo[3], hi[3];
};

// The block's cells and its windows: for each of the rows around (up to
// three), the slot range [lo, hi) of the cells ia..ib in the storage order,
// from the first non-empty cell's start to the last one's end (empty cells
// may hold any bounds).  One thread per (row, cell); ends with a barrier.
__device__ void cs_block(const int32_t* ostart, const int32_t* oend, int nx, int nz, CsBlock& b) {
  const int tid = threadIdx.x;
  const int k = blockIdx.y, i0 = blockIdx.x * CS_CELLS;
  const int ka = max(k - 1, 0), kb = min(k + 1, nz);
  const int ia = max(i0 - 1, 0), ib = min(i0 + min(CS_CELLS, nx + 1 - i0), nx);
  const int ncol = ib - ia + 1;   // at most CS_CELLS + 2
  if (tid == 0) {
    b.cfirst = k * (nx + 1) + i0;
    b.ncb = min(CS_CELLS, nx + 1 - i0);
    b.nwin = kb - ka + 1;
    for (int w = 0; w < 3; w++) {
      b.lo[w] = INT32_MAX;
      b.hi[w] = 0;
    }
  }
  __syncthreads();
  if (tid < 3 * ncol) {
    const int w = tid / ncol, i = ia + tid % ncol, kk = ka + w;
    if (kk <= kb) {
      const int c = kk * (nx + 1) + i;
      const int s0 = ostart[c], s1 = oend[c];
      if (s1 > s0) {
        atomicMin(&b.lo[w], s0);
        atomicMax(&b.hi[w], s1);
      }
    }
  }
  __syncthreads();
  if (tid < 3 && b.lo[tid] == INT32_MAX) {
    b.lo[tid] = 0;
    b.hi[tid] = 0;
  }
  __syncthreads();
}

// per-cell counts of the block's cells, and the block's total
__global__ void __launch_bounds__(CS_THREADS) k_cs_count(const int32_t* __restrict__ key,
                                                          const int32_t* __restrict__ ostart,
                                                          const int32_t* __restrict__ oend, int nx, int nz,
                                                          int32_t* __restrict__ ccount, int32_t* __restrict__ bsum) {
  __shared__ CsBlock sb;
  __shared__ int lcount[CS_CELLS];
  const int tid = threadIdx.x;
  if (tid < CS_CELLS) lcount[tid] = 0;
  cs_block(ostart, oend, nx, nz, sb);
  const int cfirst = sb.cfirst, ncb = sb.ncb;
  for (int w = 0; w < sb.nwin; w++)
    for (int q = sb.lo[w] + tid; q < sb.hi[w]; q += CS_THREADS) {
      const int lc = key[q] - cfirst;
      if (lc >= 0 && lc < ncb) atomicAdd(&lcount[lc], 1);
    }
  __syncthreads();
  if (tid < CS_CELLS) {
    int v = tid < ncb ? lcount[tid] : 0;
    if (tid < ncb) ccount[cfirst + tid] = v;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    if (tid == 0) bsum[blockIdx.y * gridDim.x + blockIdx.x] = v;
  }
}

// exclusive prefix sum of the block totals (one workgroup); flags[2] is
// raised when the total is not n (a tracer outside every window)
__global__ void __launch_bounds__(1024) k_cs_scan(int32_t* bsum, int nblk, int64_t n, int32_t* flags) {
  __shared__ int part[1024];
  const int t = threadIdx.x;
  const int per = (nblk + 1023) / 1024;
  const int a = min(t * per, nblk), b = min(a + per, nblk);
  int loc = 0;
  for (int u = a; u < b; u++) loc += bsum[u];
  part[t] = loc;
  __syncthreads();
  for (int off = 1; off < 1024; off <<= 1) {
    const int v = t >= off ? part[t - off] : 0;
    __syncthreads();
    part[t] += v;
    __syncthreads();
  }
  int run = part[t] - loc;   // exclusive
  for (int u = a; u < b; u++) {
    const int v = bsum[u];
    bsum[u] = run;
    run += v;
  }
  if (t == 1023 && (int64_t)part[1023] != n) atomicOr(&flags[2], 1);
}

// cell bounds, then the sorted (cell, slot) pairs: each window is read in
// chunks of CS_THREADS slots; within a wave a tracer's rank among the lanes
// before it with the same cell comes from ballots, across waves from the
// per-wave counts, across chunks from the running count per cell
__global__ void __launch_bounds__(CS_THREADS) k_cs_fill(const int32_t* __restrict__ key,
                                                         const int32_t* __restrict__ ostart,
                                                         const int32_t* __restrict__ oend, int nx, int nz,
                                                         const int32_t* __restrict__ ccount,
                                                         const int32_t* __restrict__ bsum, int32_t* __restrict__ cstart,
                                                         int32_t* __restrict__ cend, int32_t* __restrict__ perm,
                                                         int32_t* __restrict__ skey) {
  __shared__ CsBlock sb;
  __shared__ int lstart[CS_CELLS], running[CS_CELLS], cnt[CS_THREADS / 64][CS_CELLS];
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  cs_block(ostart, oend, nx, nz, sb);
  const int cfirst = sb.cfirst, ncb = sb.ncb;
  if (tid < CS_CELLS) {
    // the block's cell starts: its total's offset plus a wave prefix sum
    const int v = tid < ncb ? ccount[cfirst + tid] : 0;
    int incl = v;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int u = __shfl_up(incl, o, 64);
      if (lane >= o) incl += u;
    }
    const int st = bsum[blockIdx.y * gridDim.x + blockIdx.x] + incl - v;
    lstart[tid] = st;
    running[tid] = 0;
    if (tid < ncb) {
      cstart[cfirst + tid] = st;
      cend[cfirst + tid] = st + v;
    }
  }
  __syncthreads();
  const unsigned long long below = (1ull << lane) - 1ull;
  for (int w = 0; w < sb.nwin; w++) {
    const int lo = sb.lo[w], hi = sb.hi[w];
    for (int base = lo; base < hi; base += CS_THREADS) {
      cnt[wv][lane] = 0;
      const int q = base + tid;
      int lc = -1;
      if (q < hi) {
        const int d = key[q] - cfirst;
        if (d >= 0 && d < ncb) lc = d;
      }
      __syncthreads();
      int rank = 0;
      unsigned long long pending = __ballot(lc >= 0);
      while (pending) {
        const int leader = __ffsll((long long)pending) - 1;
        const int lv = __shfl(lc, leader, 64);
        const unsigned long long m = __ballot(lc == lv);
        if (lc == lv) rank = __popcll(m & below);
        if (lane == leader) cnt[wv][lv] = __popcll(m);
        pending &= ~m;
      }
      __syncthreads();
      if (lc >= 0) {
        int pos = lstart[lc] + running[lc] + rank;
        for (int u = 0; u < wv; u++) pos += cnt[u][lc];
        perm[pos] = q;
        skey[pos] = cfirst + lc;
      }
      __syncthreads();
      if (tid < CS_CELLS) {
        int add = 0;
        for (int u = 0; u < CS_THREADS / 64; u++) add += cnt[u][tid];
        running[tid] += add;
      }
      __syncthreads();
    }
  }
}

// segment bounds of each cell in the sorted key array (empty cells: 0,0)
__global__ void k_cell_bounds(const int32_t* skey, int64_t n, int ncell, int32_t* cstart, int32_t* cend) {
  int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= n) return;
  int c = skey[p];
  if (c >= ncell) return;
  if (p == 0 || skey[p - 1] != c) cstart[c] = (int32_t)p;
  if (p == n - 1 || skey[p + 1] != c) cend[c] = (int32_t)(p + 1);
}

// Per-cell partial sums of the projection.  A block owns PJ_CELLS
// consecutive cells; their tracers are one contiguous run of the
// (cell, slot)-sorted order, processed in chunks of PJ_CHUNK:
//  phase 1, one thread per tracer: coalesced loads through the permutation
//    (close to the identity, since the tracer arrays are kept in cell
//    order), the 3+3 hat factors max(0,1-|r-ri|/dr), max(0,1-|s-sk|/ds) of
//    shape_func (PS/composition.f90:896-921) for the nodes around the
//    tracer's cell, staged in LDS with T and C;
//  phase 2, one thread per (cell, neighbour node): w = wx*wz, and T*w, C*w,
//    w summed over the cell's tracers in ascending slot order (across
//    chunks too, so each sum is one sequential pass).
// Fixed summation order, no atomics: the result is deterministic.
constexpr int PJ_CELLS = 28;     // 28 cells x 9 neighbour nodes = 252 phase-2 threads
constexpr int PJ_THREADS = 256;
constexpr int PJ_CHUNK = 512;
static_assert(PJ_CHUNK % PJ_THREADS == 0, "a chunk is a whole number of tracers per thread");
__global__ void __launch_bounds__(PJ_THREADS) k_cell_reduce(const double* __restrict__ r, const double* __restrict__ s,
                                                            const double* __restrict__ Tt, const double* __restrict__ Ct,
                                                            const int32_t* __restrict__ perm,
                                                            const int32_t* __restrict__ skey, int64_t n,
                                                            const int32_t* __restrict__ cstart,
                                                            const int32_t* __restrict__ cend,
                                                            double* __restrict__ cellsum, int nx, int nz, double dr,
                                                            double ds) {
  // hat-factor rows padded by one double: an owner thread's row na (nb) is
  // then two LDS banks from its neighbours', not in the same bank
  __shared__ double hx[3][PJ_CHUNK + 1], hz[3][PJ_CHUNK + 1], sT[PJ_CHUNK], sC[PJ_CHUNK];
  __shared__ int32_t range[2];
  const int ncell = (nx + 1) * (nz + 1);
  const int cfirst = blockIdx.x * PJ_CELLS;
  const int clast = min(cfirst + PJ_CELLS, ncell);   // exclusive
  const int tid = threadIdx.x;
  // the block's tracers: from the first non-empty cell's segment start to
  // the last one's end (consecutive cells are consecutive in the sorted order)
  if (tid == 0) {
    range[0] = INT32_MAX;
    range[1] = 0;
  }
  __syncthreads();
  if (tid < clast - cfirst) {
    const int32_t b0 = cstart[cfirst + tid], b1 = cend[cfirst + tid];
    if (b1 > b0) {
      atomicMin(&range[0], b0);
      atomicMax(&range[1], b1);
    }
  }
  // phase-2 role: cell c, neighbour node (a, b) of the 3x3 around it
  const int c = cfirst + tid / 9, ab = tid % 9, na = ab / 3, nb = ab % 3;
  const bool owner = tid < 9 * PJ_CELLS && c < clast;
  int64_t b0 = 0, b1 = 0;
  if (owner) {
    b0 = cstart[c];
    b1 = cend[c];
  }
  double txs = 0.0, cxs = 0.0, ws = 0.0;
  __syncthreads();
  const int64_t t0 = range[0] == INT32_MAX ? 0 : range[0], t1 = range[0] == INT32_MAX ? 0 : range[1];
  for (int64_t base = t0; base < t1; base += PJ_CHUNK) {
    const int cnt = (int)min((int64_t)PJ_CHUNK, t1 - base);
    // the thread's PJ_Q tracers of the chunk: slot and permutation loads
    // (clamped into the chunk) for all of them, then their r, s, T, C, so
    // the chunk waits for two memory round trips
    constexpr int PJ_Q = PJ_CHUNK / PJ_THREADS;
    int32_t jq[PJ_Q], kq[PJ_Q];
#pragma unroll
    for (int u = 0; u < PJ_Q; u++) {
      const int q = min(tid + u * PJ_THREADS, cnt - 1);
      jq[u] = perm[base + q];
      kq[u] = skey[base + q];
    }
    double rq[PJ_Q], sq[PJ_Q], tq[PJ_Q], cq[PJ_Q];
#pragma unroll
    for (int u = 0; u < PJ_Q; u++) {
      rq[u] = r[jq[u]];
      sq[u] = s[jq[u]];
      tq[u] = Tt[jq[u]];
      cq[u] = Ct[jq[u]];
    }
#pragma unroll
    for (int u = 0; u < PJ_Q; u++) {
      const int q = tid + u * PJ_THREADS;
      if (q >= cnt) continue;
      const int key = kq[u];
      const int i = key % (nx + 1), k = key / (nx + 1);
#pragma unroll
      for (int e = 0; e < 3; e++) {
        const double tx = 1.0 - fabs(rq[u] - (double)(i + e - 1) * dr) / dr;
        hx[e][q] = tx < 0.0 ? 0.0 : tx;
        const double tz = 1.0 - fabs(sq[u] - (double)(k + e - 1) * ds) / ds;
        hz[e][q] = tz < 0.0 ? 0.0 : tz;
      }
      sT[q] = tq[u];
      sC[q] = cq[u];
    }
    __syncthreads();
    if (owner) {
      const int q0 = (int)(max(b0, base) - base), q1 = (int)(min(b1, base + cnt) - base);
      int q = q0;
      // four tracers' LDS operands in flight; the sums stay in slot order
      for (; q + 4 <= q1; q += 4) {
        double w[4], tv[4], cv[4];
#pragma unroll
        for (int u = 0; u < 4; u++) {
          w[u] = hx[na][q + u] * hz[nb][q + u];
          tv[u] = sT[q + u];
          cv[u] = sC[q + u];
        }
#pragma unroll
        for (int u = 0; u < 4; u++) {
          txs = txs + tv[u] * w[u];
          cxs = cxs + cv[u] * w[u];
          ws = ws + w[u];
        }
      }
      for (; q < q1; q++) {
        const double w = hx[na][q] * hz[nb][q];
        txs = txs + sT[q] * w;
        cxs = cxs + sC[q] * w;
        ws = ws + w;
      }
    }
    __syncthreads();
  }
  if (owner) {
    double* out = cellsum + (long)c * 27 + ab * 3;
    out[0] = txs;
    out[1] = cxs;
    out[2] = ws;
  }
}

// node (i,k) sums the partials of the 9 cells around it in a fixed order;
// Tratio, Cnew = ratio where the weight sum is positive, nempty = own count
__global__ void k_node_combine(const double* __restrict__ cellsum, const int32_t* cstart, const int32_t* cend,
                               double* Tratio, double* Cnew, int32_t* nempty, int nx, int nz) {
  int i = blockIdx.x * blockDim.x + threadIdx.x, k = blockIdx.y * blockDim.y + threadIdx.y;
  if (i > nx || k > nz) return;
  double txs = 0.0, cxs = 0.0, ssum = 0.0;
  for (int a = -1; a <= 1; a++) {
    int ic = i + a;
    if (ic < 0 || ic > nx) continue;
    for (int b = -1; b <= 1; b++) {
      int kc = k + b;
      if (kc < 0 || kc > nz) continue;
      long c = (long)kc * (nx + 1) + ic;
      int slot = ((-a) + 1) * 3 + ((-b) + 1);   // this node seen from cell (ic,kc)
      txs = txs + cellsum[c * 27 + slot * 3 + 0];
      cxs = cxs + cellsum[c * 27 + slot * 3 + 1];
      ssum = ssum + cellsum[c * 27 + slot * 3 + 2];
    }
  }
  long own = (long)k * (nx + 1) + i;
  nempty[own] = cend[own] - cstart[own];
  if (ssum > 0.0) {
    Tratio[I3(i, k, nx + 7)] = txs / ssum;
    Cnew[I5(i, k, nx + 11)] = cxs / ssum;
  }
}

// ---------------------------------------------------------------------------
// boundary conditions
// ---------------------------------------------------------------------------
// side ghosts (symmetric), rows 0..nz, for a field with halo h and pitch p
__global__ void k_sym_side(double* f, int nx, int nz, int h, int p) {
  int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= (nz + 1) * h) return;
  int k = t / h, i = 1 + t % h;
  long row = (long)(k + h) * p + h;
  f[row - i] = f[row + i];
  f[row + nx + i] = f[row + nx - i];
}
// enforceBCs_comp top/bottom: symmetric rows for all columns -h..nx+h
__global__ void k_sym_tb(double* f, int nx, int nz, int h, int p) {
  int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= (nx + 1 + 2 * h) * h) return;
  int i = -h + t / h, k = 1 + t % h;
  f[(long)(h - k) * p + (i + h)] = f[(long)(h + k) * p + (i + h)];
  f[(long)(h + nz + k) * p + (i + h)] = f[(long)(h + nz - k) * p + (i + h)];
}
// T wall rows: ghost = 2*Twall + (2/D2(0))*heating*ds2 - mirror (isothermal) or
// mirror (insulating bottom), then the wall rows themselves (enforceBCs/extendT)
__global__ void k_t_tb(double* f, const double* Cvis, int nx, int nz, int h, int p, int p5, int Tbot, double Tb,
                       double Tt, double two_over_d20, double ds2, double H, double Htype) {
  int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= (nx + 1 + 2 * h) * h) return;
  int i = -h + t / h, k = 1 + t % h;
  long ci = i + 5;
  double cb = Cvis[(long)(0 + 5) * p5 + ci], ct = Cvis[(long)(nz + 5) * p5 + ci];
  double hb = Htype * cb + H * (1.0 - (0.0 + cb));
  double ht = Htype * ct + H * (1.0 - (0.0 + ct));
  double in_b = f[(long)(h + k) * p + (i + h)];
  double in_t = f[(long)(h + nz - k) * p + (i + h)];
  if (Tbot == 0) f[(long)(h - k) * p + (i + h)] = 2.0 * Tb + two_over_d20 * hb * ds2 - in_b;
  else f[(long)(h - k) * p + (i + h)] = in_b;
  f[(long)(h + nz + k) * p + (i + h)] = 2.0 * Tt + two_over_d20 * ht * ds2 - in_t;
}
__global__ void k_t_walls(double* f, int nx, int nz, int h, int p, int Tbot, double Tb, double Tt) {
  int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= nx + 1 + 2 * h) return;
  int i = -h + t;
  if (Tbot == 0) f[(long)h * p + (i + h)] = Tb;
  f[(long)(h + nz) * p + (i + h)] = Tt;
}
__global__ void k_copy_nodes(const double* a, int pa, int ha, double* b, int pb, int hb, int nx, int nz) {
  int i = blockIdx.x * blockDim.x + threadIdx.x, k = blockIdx.y * blockDim.y + threadIdx.y;
  if (i > nx || k > nz) return;
  b[(long)(k + hb) * pb + (i + hb)] = a[(long)(k + ha) * pa + (i + ha)];
}

static void launch1(Context& c, void (*kern)(double*, int, int, int, int), double* f, int nthreads, int nx, int nz,
                    int h, int p) {
  hipLaunchKernelGGL(kern, dim3((nthreads + 255) / 256), dim3(256), 0, c.stream, f, nx, nz, h, p);
}

// enforceBCs(T) on a halo-3 field
static void t_bcs(Context& c, double* f) {
  int nx = c.T.nx, nz = c.T.nz;
  launch1(c, k_sym_side, f, (nz + 1) * 3, nx, nz, 3, nx + 7);
  int n = (nx + 7) * 3;
  hipLaunchKernelGGL(k_t_tb, dim3((n + 255) / 256), dim3(256), 0, c.stream, f, c.Cvis, nx, nz, 3, nx + 7, nx + 11,
                     c.P.Tbot, c.Tbot_iso, c.Ttop_iso, 2.0 / c.T.D2[3], c.T.ds2, c.P.H, c.P.Htype);
  hipLaunchKernelGGL(k_t_walls, dim3((nx + 7 + 255) / 256), dim3(256), 0, c.stream, f, nx, nz, 3, nx + 7, c.P.Tbot,
                     c.Tbot_iso, c.Ttop_iso);
}
// enforceBCs_comp on a halo-5 field
static void c_bcs(Context& c, double* f) {
  int nx = c.T.nx, nz = c.T.nz;
  launch1(c, k_sym_side, f, (nz + 1) * 5, nx, nz, 5, nx + 11);
  launch1(c, k_sym_tb, f, (nx + 11) * 5, nx, nz, 5, nx + 11);
}
// extendT: Textend(0:nx,0:nz) = Tratio, halo-5 wall ghosts
static void extend_t(Context& c) {
  int nx = c.T.nx, nz = c.T.nz;
  dim3 b16(64, 4);
  hipLaunchKernelGGL(k_copy_nodes, grid2(nx + 1, nz + 1, b16), b16, 0, c.stream, c.Tratio, nx + 7, 3, c.Textend,
                     nx + 11, 5, nx, nz);
  launch1(c, k_sym_side, c.Textend, (nz + 1) * 5, nx, nz, 5, nx + 11);
  int n = (nx + 11) * 5;
  hipLaunchKernelGGL(k_t_tb, dim3((n + 255) / 256), dim3(256), 0, c.stream, c.Textend, c.Cvis, nx, nz, 5, nx + 11,
                     nx + 11, c.P.Tbot, c.Tbot_iso, c.Ttop_iso, 2.0 / c.T.D2[3], c.T.ds2, c.P.H, c.P.Htype);
  hipLaunchKernelGGL(k_t_walls, dim3((nx + 11 + 255) / 256), dim3(256), 0, c.stream, c.Textend, nx, nz, 5, nx + 11,
                     c.P.Tbot, c.Tbot_iso, c.Ttop_iso);
}

// ---------------------------------------------------------------------------
// filters
// ---------------------------------------------------------------------------
// smoothness (PS/smoother.f90:75-95): block maxima over i=0..nx-1, k=1..nz-1
__global__ void k_smoothness(const double* f, int nx, int nz, int h, int p, double* partial) {
  __shared__ double red[256];
  int tid = threadIdx.y * blockDim.x + threadIdx.x;
  int i = blockIdx.x * blockDim.x + threadIdx.x, k = 1 + blockIdx.y * blockDim.y + threadIdx.y;
  double d = 0.0;
  if (i <= nx - 1 && k <= nz - 1) {
    auto F = [&](int a, int b) { return f[(long)(b + h) * p + (a + h)]; };
    double t = F(i, k);
    double a1 = fabs(F(i, k - 1) - t), a2 = fabs(F(i + 1, k - 1) - t), a3 = fabs(F(i + 1, k) - t),
           a4 = fabs(F(i, k + 1) - t), a5 = fabs(F(i + 1, k + 1) - t);
    d = fmax(fmax(fmax(fmax(a1, a2), a3), a4), a5);
  }
  red[tid] = d;
  __syncthreads();
  for (int st = 128; st > 0; st >>= 1) {
    if (tid < st) red[tid] = fmax(red[tid], red[tid + st]);
    __syncthreads();
  }
  if (tid == 0) partial[blockIdx.y * gridDim.x + blockIdx.x] = red[0];
}

// one Richardson pass: out = T0 + (c*dts)*lap(T0) (clamped to [0,1] for C)
__global__ void k_filter(const double* T0, double* out, int nx, int nz, int h, int p, double cdts, int clamp01,
                         double dr, double ds, double dr2, double ds2, double d10, double d11, double d12, double d13,
                         double d14, double d20, double d21, double d22, double d23, double d24) {
  int i = blockIdx.x * blockDim.x + threadIdx.x, k = blockIdx.y * blockDim.y + threadIdx.y;
  if (i > nx || k > nz) return;
  const double D1[5] = {d10, d11, d12, d13, d14}, D2[5] = {d20, d21, d22, d23, d24};
  auto F = [&](int a, int b) { return T0[(long)(b + h) * p + (a + h)]; };
  double sr = 0.0, ss = 0.0, srr = 0.0, sss = 0.0;
  for (int q = -2; q <= 2; q++) sr = sr + D1[q + 2] * F(i + q, k);
  for (int q = -2; q <= 2; q++) ss = ss + D1[q + 2] * F(i, k + q);
  for (int q = -2; q <= 2; q++) srr = srr + D2[q + 2] * F(i + q, k);
  for (int q = -2; q <= 2; q++) sss = sss + D2[q + 2] * F(i, k + q);
  double Tr = sr / dr, Ts = ss / ds, Trr = srr / dr2, Tss = sss / ds2;
  double Tx = Tr / 1.0, Tz = Ts / 1.0;
  double Txx = (Trr - Tx * 0.0) / 1.0, Tzz = (Tss - Tz * 0.0) / 1.0;
  double temp = Txx + Tzz;
  double v = F(i, k) + cdts * temp;
  if (clamp01) {
    if (v < 0.0) v = 0.0;
    if (v > 1.0) v = 1.0;
  }
  out[(long)(k + h) * p + (i + h)] = v;
}

static int smoothness_host(Context& c, const double* f, int h, int p, double* out) {
  dim3 b16(64, 4);
  dim3 g = grid2(c.T.nx, c.T.nz - 1, b16);
  hipLaunchKernelGGL(k_smoothness, g, b16, 0, c.stream, f, c.T.nx, c.T.nz, h, p, c.red);
  hipLaunchKernelGGL(k_reduce_final, dim3(1), dim3(256), 0, c.stream, c.red, (int)(g.x * g.y), (int)RED_MAX, c.red_out);
  PT_HIP(hipMemcpyAsync(c.h_red, c.red_out, sizeof(double), hipMemcpyDeviceToHost, c.stream));
  PT_HIP(hipStreamSynchronize(c.stream));
  *out = c.h_red[0];
  return PT_OK;
}

static void filter_pass(Context& c, const double* T0, double* out, int h, double cdts, int clamp01) {
  dim3 b16(64, 4);
  const double* D1 = c.T.D1;
  const double* D2 = c.T.D2;
  hipLaunchKernelGGL(k_filter, grid2(c.T.nx + 1, c.T.nz + 1, b16), b16, 0, c.stream, T0, out, c.T.nx, c.T.nz, h,
                     c.T.nx + 1 + 2 * h, cdts, clamp01, c.T.dr, c.T.ds, c.T.dr2, c.T.ds2, D1[1], D1[2], D1[3], D1[4],
                     D1[5], D2[1], D2[2], D2[3], D2[4], D2[5]);
}

// ---------------------------------------------------------------------------
// Filter loops driven on the device.  The reference checks the field's
// smoothness before every pass and stops at the first check below the
// threshold (PS/smoother.f90:582-672).  k_filter_passes makes K passes per
// launch on tiles of the nodes in LDS (temporal blocking): pass t of a launch
// is made on the tile's core widened by 2 nodes for every pass still to come,
// so tiles exchange nothing within a launch, and the check before each pass
// (a maximum, so its order is free) is taken on the tile's own nodes and left
// as one partial maximum per tile and pass.  Every tile of the next launch
// reduces those maxima.  When one of the K checks is below the threshold, the
// launch repeats the previous launch's passes up to that check from the field
// it started from, which is the field the reference stops with, and raises
// the done flag; otherwise it makes the next K passes.  Three buffers rotate,
// so the field a launch started from is intact in the next.  The host
// enqueues launches in batches without waiting.
//
// Only the nodes 0..nx x 0..nz are read: ghost values are the mirror images of
// node values (enforceBCs_comp; T: 2 T_wall + heating - image below and above),
// formed where they are used, and written with the last pass's result.
//
// The reference checks C (halo 5) through a dummy with the halo-3 shape
// (PS/smoother.f90:79, :602): sequence association makes it read the storage
// with row length nx+7 instead of P = nx+11, so a check point and its
// neighbours one row away lie 4 columns apart per row, and points in the
// ghost columns are compared with the other end of their row.  A tile checks
// its nodes (and the ghost rows below them); the ghost columns are checked by
// one extra tile per band of rows, which keeps a strip along each side wall.
//
// One pass per launch (latency-bound: a launch to launch gap, a round trip
// to memory for the field and one for the previous check) took 5.6 us and 1.5
// us of gap at 1024x256.  Eight passes per launch take 2.9 us each: 20.3 us a
// launch, of which vector instructions take 50% of the issue slots and LDS is
// active 41% (by counters; 2.4 times the nodes for the overlap), and the gap.
// ---------------------------------------------------------------------------
constexpr int FILTER_KMAX = 8;      // passes per launch
constexpr int FILTER_RB = 5;        // nodes per thread, vertically adjacent
constexpr int FILTER_THREADS = 1024;
constexpr int FILTER_LDS_BYTES = 158 * 1024;   // dynamic: two windows and the checks
constexpr int FILTER_MAX_PART = 1024;   // tiles whose partial maxima every tile reduces itself

struct FilterArgs {
  int nx, nz, h, p;
  double dr2, ds2, rdr2, rds2;
  double d2[3];         // D2 at offsets 0, 1, 2
  double dr, ds, d1[5]; // for the general form of a pass
  double limit;         // values below it stay finite through a launch's passes
  // T: enforceBCs with the isothermal / insulating walls
  int Tbot;
  double Tb, Tt, two_over_d20, H, Htype;
  const double* Cvis;   // halo 5, for the heating term of the T wall ghosts
  double delta;
  // tiles: core cw x ch, nbx x nbz of them, then (C) nbz edge tiles of two
  // strips of `strip` columns
  int cw, ch, nbx, nbz, strip, ntile;
  int K;                // passes per launch
  int pitch, rows;      // LDS window
  int w1, nrb;          // columns and row blocks of the first pass's region
};

struct FilterLaunch {
  const double *in, *prev;      // this launch's field; the one the previous launch started from
  double* out;
  int32_t* ctl;                 // deciding launch (0: none yet), passes made, buffer of the result
  const double* part_prev;      // the previous launch's partial maxima, K per tile (one set when reduced)
  double* part;
  int nprev;                    // sets in part_prev; 0: first launch
  int k, kprev;                 // passes of this launch and of the previous one, at most FilterArgs::K
  int jprev;                    // passes made before the previous launch
  int launch, out_id, prev_id;  // launch number from 1; buffer numbers
  double cd[FILTER_KMAX], cdp[FILTER_KMAX];   // c dts of this launch's and of the previous launch's passes
};

__device__ __forceinline__ int mirror(int i, int n) { return n - abs(n - abs(i)); }   // -n <= i <= 2 n

// maximum over a wavefront, in every lane
__device__ __forceinline__ double wave_max_f64(double d) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) d = fmax(d, __shfl_xor(d, o, 64));
  return d;
}

// what a thread of k_filter_passes keeps for its passes: LDS offsets of the
// rows k0-2 .. k0+RB+1 at its column, of the columns a pass and a check read
// (relative), the nodes it checks and its ghost cell's check
struct FilterThread {
  int ro[FILTER_RB + 4], oc[4], os[4], xo[6];
  unsigned chk, last;   // nodes checked; those on the check's last row
  bool extra;
  double Ab, At;        // T: the ghost rows' constants
  bool lowz, highz;     // the window holds rows that read them
};

// one pass (and the check before it) at a thread's nodes.  FINITE: nothing that
// the launch forms from the window is an infinity or NaN; otherwise the
// stretched-grid form's Txx = Trr - Tx*0 decides what becomes of them, so it is
// evaluated as written.
template <bool COMP, bool PW2, bool FINITE>
__device__ __forceinline__ double filter_nodes(const FilterArgs& a, const FilterThread& th, const double* X, double* Y,
                                               int k0, double cdts, double* yv) {
  constexpr int RB = FILTER_RB;
  const int nz = a.nz;
  double d = 0.0, col[RB + 4];
#pragma unroll
  for (int j = 0; j < RB + 4; j++) {
    double v = X[th.ro[j]];
    if constexpr (!COMP) {
      if (th.lowz && k0 + j - 2 < 0) v = th.Ab - v;
      if (th.highz && k0 + j - 2 > nz) v = th.At - v;
    }
    col[j] = v;
  }
#pragma unroll
  for (int r = 0; r < RB; r++) {
    const double* x = X + th.ro[r + 2];
    const double e0 = x[th.oc[0]], e1 = x[th.oc[1]], v = col[r + 2], e3 = x[th.oc[2]], e4 = x[th.oc[3]];
    double srr = a.d2[2] * e0;
    srr = srr + a.d2[1] * e1;
    srr = srr + a.d2[0] * v;
    srr = srr + a.d2[1] * e3;
    srr = srr + a.d2[2] * e4;
    double sss = a.d2[2] * col[r];
    sss = sss + a.d2[1] * col[r + 1];
    sss = sss + a.d2[0] * v;
    sss = sss + a.d2[1] * col[r + 3];
    sss = sss + a.d2[2] * col[r + 4];
    double Txx, Tzz;
    if constexpr (FINITE) {
      Txx = quot<PW2>(srr, a.dr2, a.rdr2);
      Tzz = quot<PW2>(sss, a.ds2, a.rds2);
    } else {
      double sr = a.d1[0] * e0;
      sr = sr + a.d1[1] * e1;
      sr = sr + a.d1[2] * v;
      sr = sr + a.d1[3] * e3;
      sr = sr + a.d1[4] * e4;
      double ss = a.d1[0] * col[r];
      ss = ss + a.d1[1] * col[r + 1];
      ss = ss + a.d1[2] * v;
      ss = ss + a.d1[3] * col[r + 3];
      ss = ss + a.d1[4] * col[r + 4];
      Txx = srr / a.dr2 - sr / a.dr * 0.0;
      Tzz = sss / a.ds2 - ss / a.ds * 0.0;
    }
    double y = v + cdts * (Txx + Tzz);
    const int k = k0 + r;
    if constexpr (COMP) {
      if constexpr (FINITE) {
        y = fmin(fmax(y, 0.0), 1.0);
      } else {
        if (y < 0.0) y = 0.0;
        if (y > 1.0) y = 1.0;
      }
    } else {
      if (k == 0 && a.Tbot == 0) y = a.Tb;
      if (k == nz) y = a.Tt;
    }
    yv[r] = y;
    if (k <= nz) Y[th.ro[r + 2]] = y;
    if (th.chk >> r & 1) {
      // the jumps to the row below, to the right, and across to the row
      // above; the jump straight up is the next row's jump down, so only the
      // check's last row takes its own
      double n1, n2, n4;
      if constexpr (COMP) {
        n1 = X[th.ro[r + 1] + th.os[0]];
        n2 = X[th.ro[r + 1] + th.os[1]];
        n4 = X[th.ro[r + 3] + th.os[2]];
      } else {
        n1 = col[r + 1];
        n2 = X[th.ro[r + 1] + th.oc[2]];
        n4 = X[th.ro[r + 3] + th.oc[2]];
      }
      d = fmax(d, fmax(fmax(fabs(n1 - v), fabs(n2 - v)), fmax(fabs(e3 - v), fabs(n4 - v))));
    }
  }
  if (th.last) {
#pragma unroll
    for (int r = 0; r < RB; r++)
      if (th.last >> r & 1) d = fmax(d, fabs((COMP ? X[th.ro[r + 3] + th.os[3]] : col[r + 3]) - col[r + 2]));
  }
  if constexpr (COMP) {
    if (th.extra) {
      const double v = X[th.xo[0]];
#pragma unroll
      for (int q = 1; q < 6; q++) d = fmax(d, fabs(X[th.xo[q]] - v));
    }
  }
  return d;
}

template <bool COMP, bool PW2>
__global__ void __launch_bounds__(FILTER_THREADS) k_filter_passes(FilterArgs a, FilterLaunch f) {
  extern __shared__ double fsm[];
  __shared__ int s_ok[FILTER_KMAX], s_bad[FILTER_THREADS / 64];
  constexpr int RB = FILTER_RB;
  const int nx = a.nx, nz = a.nz, K = a.K, tid = threadIdx.x, nthr = blockDim.x;
  const int lane = tid & 63, wave = tid >> 6, nwave = nthr >> 6;
  const int W = a.pitch, ne = a.pitch * a.rows;
  double* const dmax = fsm + 2 * ne;   // [K][nthr]: every thread's part of each check
  // XCD-aware tiles: workgroups are dealt round-robin over the 8 XCDs; each
  // XCD gets one contiguous band of tiles, the same in every launch, so that
  // most of what a tile reads is in its own L2
  const int ntile = a.ntile, q8 = ntile / 8, r8 = ntile % 8, xcd = blockIdx.x % 8;
  const int tile = xcd * q8 + min(xcd, r8) + blockIdx.x / 8;
  const bool edge = COMP && tile >= a.nbx * a.nbz;
  const int bz = edge ? tile - a.nbx * a.nbz : tile / a.nbx;
  const int bx = edge ? 0 : tile - bz * a.nbx;
  const int cz0 = bz * a.ch, cz1 = min(cz0 + a.ch, nz + 1);
  const int cx0 = edge ? 0 : bx * a.cw, cx1 = edge ? nx + 1 : min(cx0 + a.cw, nx + 1);
  constexpr int EX = COMP ? 3 : 0;   // the C check reads 5 columns to the side, the pass 2
  const int S = a.strip;
  const int xlo = edge ? 0 : max(0, cx0 - 2 * K - EX);
  const int ncol = edge ? 2 * S : min(nx, cx1 - 1 + 2 * K + EX) - xlo + 1;
  const int zlo = max(0, cz0 - 2 * K), nrow = min(nz, cz1 - 1 + 2 * K) - zlo + 1;
  // window: element e = row * ncol + column, threads nthr apart
  const int er0 = tid / ncol, ec0 = tid - er0 * ncol, dr = nthr / ncol, dc = nthr - dr * ncol;
  bool bad = false;
  auto load = [&](const double* src) {
    int er = er0, ec = ec0;
    while (er < nrow) {
      constexpr int FB = 5;
      double v[FB];
      int at[FB];
#pragma unroll
      for (int u = 0; u < FB; u++) {
        const int i = edge ? (ec < S ? ec : nx - (2 * S - 1 - ec)) : xlo + ec;
        v[u] = src[(long)(min(zlo + er, nz) + a.h) * a.p + (i + a.h)];
        at[u] = er < nrow ? er * W + ec : -1;
        er += dr;
        ec += dc;
        if (ec >= ncol) { ec -= ncol; er++; }
      }
#pragma unroll
      for (int u = 0; u < FB; u++)
        if (at[u] >= 0) {
          fsm[at[u]] = v[u];
          bad |= !(fabs(v[u]) < a.limit);
        }
    }
  };
  // each wavefront leaves what it found in a word of its own, so the flags need
  // no initial value; read after the barrier that follows
  auto report = [&]() {
    const bool any = __ballot(bad) != 0;
    if (lane == 0) s_bad[wave] = any;
  };
  // the control word, the previous launch's checks (wavefront t takes check
  // t) and the window are loaded together, before the decision
  const int decided = f.ctl[0];
  double pm[4];
  const bool mine = f.nprev > 0 && wave < f.kprev;
#pragma unroll
  for (int u = 0; u < 4; u++)
    pm[u] = mine && lane + u * 64 < f.nprev ? f.part_prev[(long)wave * f.nprev + lane + u * 64] : 0.0;
  load(f.in);
  if (decided != 0 && decided < f.launch) return;
  if (f.nprev > 0) {
    double d = fmax(fmax(pm[0], pm[1]), fmax(pm[2], pm[3]));
    for (int t = wave; t < f.kprev; t += nwave) {
      if (t != wave) d = 0.0;
      for (int b = lane + (t == wave ? 256 : 0); b < f.nprev; b += 64) d = fmax(d, f.part_prev[(long)t * f.nprev + b]);
      d = wave_max_f64(d);
      if (lane == 0) s_ok[t] = d < a.delta ? 1 : 0;
    }
  }
  // LDS column of a grid column (mirrored into the grid; clamped where a
  // thread outside its pass's region asks for a column the window lacks)
  auto strip_col = [&](int m, bool right) { return right ? max(2 * S - 1 - (nx - m), S) : min(m, S - 1); };
  auto lcol = [&](int i, bool right) {
    const int m = mirror(i, nx);
    return min(max(edge ? strip_col(m, right) : m - xlo, 0), ncol - 1);
  };
  auto lrow = [&](int k) { return min(max(mirror(k, nz) - zlo, 0), nrow - 1); };
  // this thread's nodes: column ic, rows k0 .. k0+RB-1 of the first pass's region
  const int x1 = edge ? 0 : max(0, cx0 - 2 * (K - 1) - EX), z1 = max(0, cz0 - 2 * (K - 1));
  const int w1 = edge ? 2 * S : a.w1;
  const int rb = tid / w1, cc = tid - rb * w1;
  const int ic = edge ? (cc < S ? cc : nx - (2 * S - 1 - cc)) : x1 + cc, k0 = z1 + rb * RB;
  const bool live = rb < a.nrb && ic <= nx && k0 <= nz, right = edge && cc >= S;
  // columns beyond the core (edge tiles: beyond the 6 columns at a wall)
  const int dx = edge ? max(0, right ? nx - 5 - ic : ic - 5) : max(0, max(cx0 - ic, ic - (cx1 - 1)));
  const int c0 = edge ? cc : lcol(ic, false);
  FilterThread th;
  th.oc[0] = lcol(ic - 2, right) - c0;
  th.oc[1] = lcol(ic - 1, right) - c0;
  th.oc[2] = lcol(ic + 1, right) - c0;
  th.oc[3] = lcol(ic + 2, right) - c0;
#pragma unroll
  for (int j = 0; j < RB + 4; j++) th.ro[j] = lrow(k0 + j - 2) * W + c0;
  th.chk = th.last = 0;
  if (!edge && live && dx == 0) {
    // the check's own (row, column) of the node, C: in rows of nx+7 values
    int kk = k0, ii = ic;
    const int Q = nx + 7;
    if constexpr (COMP) {
      const int L = (k0 + 5) * (Q + 4) + ic + 5;
      kk = L / Q;
      ii = L - kk * Q - 3;
      kk -= 3;
    }
#pragma unroll
    for (int r = 0; r < RB; r++) {
      const int k = k0 + r;
      if (k >= cz0 && k < cz1 && kk >= 1 && kk <= nz - 1 && ii >= 0 && ii <= nx - 1) {
        th.chk |= 1u << r;
        if (kk == nz - 1) th.last |= 1u << r;
      }
      kk++;
      if constexpr (COMP) {
        ii += 4;
        if (ii >= Q - 3) { ii -= Q; kk++; }
      }
    }
  }
  th.os[0] = th.os[1] = th.os[2] = th.os[3] = 0;
  if constexpr (COMP) {
    th.os[0] = lcol(ic + 4, right) - c0;
    th.os[1] = lcol(ic + 5, right) - c0;
    th.os[2] = lcol(ic - 3, right) - c0;
    th.os[3] = lcol(ic - 4, right) - c0;
  }
  // one ghost cell's check (C): the ghost rows below a bottom tile's columns,
  // or the ghost columns of an edge tile's rows
  th.extra = false;
#pragma unroll
  for (int q = 0; q < 6; q++) th.xo[q] = 0;
  if constexpr (COMP) {
    if (edge || cz0 == 0) {
      int col, row;
      bool cell;
      if (edge) {
        const int r0 = bz == 0 ? -5 : cz0, r1 = cz1 == nz + 1 ? nz + 5 : cz1 - 1;
        const int rr = tid / 10, q = tid - rr * 10;
        col = q < 5 ? q - 5 : nx + q - 4;
        row = r0 + rr;
        cell = row <= r1;
      } else {
        const int rr = tid / a.cw;
        col = cx0 + tid - rr * a.cw;
        row = -1 - rr;
        cell = rr < 5 && col < cx1;
      }
      if (cell) {
        const int P = nx + 11, Q = nx + 7, L = (row + 5) * P + col + 5;
        const int kk = L / Q - 3, ii = L - (kk + 3) * Q - 3;
        th.extra = kk >= 1 && kk <= nz - 1 && ii >= 0 && ii <= nx - 1;
        const int nb[6] = {0, -Q, -Q + 1, 1, Q, Q + 1};
#pragma unroll
        for (int q = 0; q < 6; q++) {
          const int Lq = th.extra ? L + nb[q] : 5 * P + 5;
          const int i = Lq % P - 5;
          th.xo[q] = lrow(Lq / P - 5) * W + lcol(i, edge && 2 * i >= nx);
        }
      }
    }
  }
  // T: the ghost rows' constants
  th.Ab = th.At = 0.0;
  th.lowz = th.highz = false;
  if constexpr (!COMP) {
    const int i = min(max(ic, 0), nx);
    const double cb = a.Cvis[(long)5 * (nx + 11) + (i + 5)], ct = a.Cvis[(long)(nz + 5) * (nx + 11) + (i + 5)];
    th.Ab = 2.0 * a.Tb + a.two_over_d20 * (a.Htype * cb + a.H * (1.0 - (0.0 + cb))) * a.ds2;
    th.At = 2.0 * a.Tt + a.two_over_d20 * (a.Htype * ct + a.H * (1.0 - (0.0 + ct))) * a.ds2;
    th.lowz = a.Tbot == 0 && zlo == 0;
    th.highz = zlo + nrow > nz;
    bad |= !(fabs(th.Ab) < a.limit && fabs(th.At) < a.limit);
  }
  report();
  __syncthreads();
  int np = f.k;           // passes this launch makes
  bool final = false;
  if (f.nprev > 0) {
    int t = 0;
    while (t < f.kprev && !s_ok[t]) t++;
    if (t < f.kprev) {
      final = true;
      np = t;
      if (blockIdx.x == 0 && tid == 0) {
        f.ctl[1] = f.jprev + t;
        f.ctl[2] = t == 0 ? f.prev_id : f.out_id;
        f.ctl[0] = f.launch;
      }
      if (t == 0 || edge) return;
      load(f.prev);
      report();
      __syncthreads();
    }
  }
  const bool finite = __ballot(lane < nwave && s_bad[lane < nwave ? lane : 0] != 0) == 0;
  int at0 = 0;
  double yv[RB];
#pragma unroll
  for (int r = 0; r < RB; r++) yv[r] = 0.0;
  for (int t = 1; t <= np; t++) {
    const double cdts = final ? f.cdp[t - 1] : f.cd[t - 1];
    const int left = np - t, hz = 2 * left;
    const int hx = edge ? 2 * (left - 1) : (left > 0 ? 2 * left + EX : 0);
    const double* X = fsm + at0;
    double* Y = fsm + (ne - at0);
    double d = 0.0;
    const bool pass = live && dx <= hx && k0 < cz1 + hz && k0 + RB > cz0 - hz;
    if (pass) {
      d = finite ? filter_nodes<COMP, PW2, true>(a, th, X, Y, k0, cdts, yv)
                 : filter_nodes<COMP, PW2, false>(a, th, X, Y, k0, cdts, yv);
    } else if (COMP && th.extra) {
      const double v = X[th.xo[0]];
#pragma unroll
      for (int q = 1; q < 6; q++) d = fmax(d, fabs(X[th.xo[q]] - v));
    }
    if (!final) dmax[(t - 1) * nthr + tid] = d;
    __syncthreads();
    at0 = ne - at0;
  }
  if (!final)
    for (int t = wave; t < np; t += nwave) {
      double d = 0.0;
      for (int u = lane; u < nthr; u += 64) d = fmax(d, dmax[t * nthr + u]);
      d = wave_max_f64(d);
      if (lane == 0) f.part[(long)t * ntile + tile] = d;
    }
  if (edge || !live || dx > 0) return;
  // the core's nodes and their ghost images: the columns whose images equal
  // this node's column are itself and its mirrors beyond the side walls
  const int h = a.h, p = a.p;
#pragma unroll
  for (int r = 0; r < RB; r++) {
    const int k = k0 + r;
    if (k < cz0 || k >= cz1) continue;
    const double y = yv[r];
    auto column = [&](int c) {
      auto put = [&](int row, double v) { f.out[(long)(row + h) * p + (c + h)] = v; };
      put(k, y);
      if (k >= 1 && k <= h) put(-k, !COMP && a.Tbot == 0 ? th.Ab - y : y);
      if (k >= nz - h && k <= nz - 1) put(2 * nz - k, COMP ? y : th.At - y);
    };
    column(ic);
    if (ic >= 1 && ic <= h) column(-ic);
    if (ic >= nx - h && ic <= nx - 1) column(2 * nx - ic);
  }
}

// partial maxima of many tiles to one set (grids whose tiles are too many for
// every tile of the next launch to reduce them itself)
__global__ void __launch_bounds__(1024) k_filter_reduce(const double* part, int n, double* out) {
  __shared__ double red[16];
  const int t = blockIdx.x, tid = threadIdx.x;
  double d = 0.0;
  for (int b = tid; b < n; b += 1024) d = fmax(d, part[(long)t * n + b]);
  d = wave_max_f64(d);
  if ((tid & 63) == 0) red[tid >> 6] = d;
  __syncthreads();
  if (tid == 0) {
    for (int w = 1; w < 16; w++) d = fmax(d, red[w]);
    out[t] = d;
  }
}

// a tiling's part of the arguments
static FilterArgs filter_shape(int nx, int nz, bool comp, const FilterPlan& p) {
  FilterArgs a;
  const int EX = comp ? 3 : 0;
  a.nx = nx; a.nz = nz; a.h = comp ? 5 : 3; a.p = nx + 1 + 2 * a.h;
  a.K = p.K; a.cw = p.cw; a.ch = p.ch;
  a.nbx = (nx + a.cw) / a.cw; a.nbz = (nz + a.ch) / a.ch;
  a.strip = std::min(nx + 1, 6 + 2 * (a.K - 1));
  a.ntile = a.nbx * a.nbz + (comp ? a.nbz : 0);
  a.pitch = std::min(a.cw + 2 * (2 * a.K + EX), nx + 1);
  if (comp) a.pitch = std::max(a.pitch, 2 * a.strip);
  a.rows = std::min(a.ch + 4 * a.K, nz + 1);
  a.w1 = std::min(a.cw + 2 * (2 * (a.K - 1) + EX), nx + 1);
  a.nrb = (std::min(a.ch + 4 * (a.K - 1), nz + 1) + FILTER_RB - 1) / FILTER_RB;
  return a;
}
static int filter_threads(const FilterArgs& a, bool comp) {
  int n = a.w1 * a.nrb;
  // an edge tile's strips, its ghost cells, a bottom tile's ghost cells
  if (comp) n = std::max({n, 2 * a.strip * a.nrb, 10 * (a.ch + 10), 5 * a.cw});
  return (n + 63) & ~63;
}
static size_t filter_lds(const FilterArgs& a, int threads) {
  return sizeof(double) * (2 * (size_t)a.pitch * a.rows + (size_t)a.K * threads);
}

// Tiles and passes per launch of a grid's filter loops: the tiling with the
// least modelled time per pass.  A launch costs 8 us (gap, window load, setup,
// stores), an evaluation 0.22 us and 0.51 ns per node and tile of a CU, fitted
// to 64x64 (43x4 cores: 2.0 us a pass), 384x128 (32x8: 2.2) and 1024x256
// (69x17: 2.9); one pass per launch took 3.3, 3.9 and 5.6 us and the gap.
static FilterPlan filter_plan(int nx, int nz, bool comp) {
  constexpr int CUS = 256;
  const int EX = comp ? 3 : 0;
  FilterPlan best = {8, 4, 1};
  double best_us = INFINITY;
  for (int K = 2; K <= FILTER_KMAX; K += 2)
    for (int ch = 4; ch <= 34; ch++)
      for (int nbx = 1; nbx <= (nx + 8) / 8; nbx++) {
        const int cw = (nx + nbx) / nbx;
        const FilterArgs a = filter_shape(nx, nz, comp, {cw, ch, K});
        const int threads = filter_threads(a, comp);
        if (threads > FILTER_THREADS || filter_lds(a, threads) > FILTER_LDS_BYTES) continue;
        double us = 0.0;
        for (int h = 0; h < K; h++) {
          const int w = std::min(cw + 2 * (2 * h + (h ? EX : 0)), nx + 1);
          const int rows = std::min(ch + 4 * h + FILTER_RB - 1, nz + FILTER_RB);
          us += 0.22 + 0.51e-3 * w * rows;
        }
        us = (8.0 + us * ((a.ntile + CUS - 1) / CUS)) / K;
        if (us < best_us) {
          best_us = us;
          best = {cw, ch, K};
        }
      }
  return best;
}

static double cdts_comp(const Context& c, int j);
static double cdts_temp(const Context& c, int j);
static FilterArgs filter_args(const Context& c, bool comp) {
  FilterArgs a = filter_shape(c.T.nx, c.T.nz, comp, c.filter[comp]);
  a.dr2 = c.T.dr2; a.ds2 = c.T.ds2; a.rdr2 = 1.0 / c.T.dr2; a.rds2 = 1.0 / c.T.ds2;
  for (int q = 0; q < 3; q++) a.d2[q] = c.T.D2[3 + q];
  a.dr = c.T.dr; a.ds = c.T.ds;
  for (int q = 0; q < 5; q++) a.d1[q] = c.T.D1[q + 1];
  // a derivative is at most `quotient` times the values it is formed from (the
  // weights of D1 and D2 sum to 1.5 and 16/3), a pass's result at most `growth`
  // times them and the ghost rows' constants
  double step = 0.0;
  for (int j = 1; j <= 11; j++) step = std::max(step, std::fabs((comp ? cdts_comp : cdts_temp)(c, j)));
  const double quotient = 6.0 * std::max({1.0, a.rdr2, a.rds2}), growth = 2.0 * (1.0 + 2.0 * step * quotient);
  a.limit = 0x1p1000 / quotient / std::pow(growth, FILTER_KMAX);
  a.Tbot = c.P.Tbot; a.Tb = c.Tbot_iso; a.Tt = c.Ttop_iso; a.two_over_d20 = 2.0 / c.T.D2[3];
  a.H = c.P.H; a.Htype = c.P.Htype; a.Cvis = c.Cvis;
  a.delta = comp ? c.T.delta_C : c.T.delta_T;
  return a;
}
template <bool COMP, bool PW2>
static int launch_filter(Context& c, const FilterArgs& a, const FilterLaunch& f, int threads, size_t lds) {
  static OncePerDevice limit;
  PT_TRY(allow_lds(c, limit, k_filter_passes<COMP, PW2>, FILTER_LDS_BYTES));
  hipLaunchKernelGGL((k_filter_passes<COMP, PW2>), dim3(a.ntile), dim3(threads), lds, c.stream, a, f);
  return PT_OK;
}

__global__ void k_filter_init(int32_t* ctl) {
  if (threadIdx.x < 4) ctl[threadIdx.x] = 0;
}

// one device-driven filter loop on x0 (x1, x2: the other buffers).
// cdts_of(j) is pass j's c*dts; on return x0 holds the filtered field with
// its ghosts and *passes the number of passes made before the successful check
static int filter_loop(Context& c, double* x0, double* x1, double* x2, bool comp,
                       double (*cdts_of)(const Context&, int), int* passes, int* hint) {
  const FilterArgs a = filter_args(c, comp);
  const int threads = filter_threads(a, comp);
  const size_t lds = filter_lds(a, threads);
  double* const buf[3] = {x0, x1, x2};
  double* const parts[2] = {c.d_fpart, c.d_fpart + (size_t)a.ntile * FILTER_KMAX};
  const bool reduced = a.ntile > FILTER_MAX_PART, pw2 = pow2(a.dr2) && pow2(a.ds2);
  if (c.timing) timer_begin(c, PT_K_FILTER);
  hipLaunchKernelGGL(k_filter_init, dim3(1), dim3(64), 0, c.stream, c.d_fctl);
  const int cap = 100000;
  // the first batch covers the previous call's pass count (consecutive
  // projections need similar counts) and the launch that decides on its last
  // check; later batches double.  The first launch makes no more passes than
  // that count's check needs.
  const int k1 = std::min(a.K, *hint + 1);
  int n = 0, done = 0, batch = std::min((*hint + 1 - k1 + a.K - 1) / a.K + 2, 1024 / a.K);
  FilterLaunch f;
  f.ctl = c.d_fctl;
  f.k = f.jprev = 0;
  for (;;) {
    for (int b = 0; b < batch; b++) {
      n++;
      f.kprev = f.k;
      f.k = n == 1 ? k1 : a.K;
      f.jprev = done - f.kprev;
      f.in = buf[(n - 1) % 3]; f.prev = buf[(n + 1) % 3]; f.out = buf[n % 3];
      f.part = parts[n % 2]; f.part_prev = reduced ? c.d_fred : parts[(n + 1) % 2];
      f.nprev = n == 1 ? 0 : reduced ? 1 : a.ntile;
      f.launch = n; f.out_id = n % 3; f.prev_id = (n + 1) % 3;
      for (int t = 0; t < FILTER_KMAX; t++) {
        f.cd[t] = t < f.k ? cdts_of(c, done + t + 1) : 0.0;
        f.cdp[t] = t < f.kprev ? cdts_of(c, f.jprev + t + 1) : 0.0;
      }
      done += f.k;
      if (comp) PT_TRY(pw2 ? (launch_filter<true, true>(c, a, f, threads, lds)) : (launch_filter<true, false>(c, a, f, threads, lds)));
      else PT_TRY(pw2 ? (launch_filter<false, true>(c, a, f, threads, lds)) : (launch_filter<false, false>(c, a, f, threads, lds)));
      if (reduced)
        hipLaunchKernelGGL(k_filter_reduce, dim3(f.k), dim3(1024), 0, c.stream, f.part, a.ntile, c.d_fred);
    }
    PT_HIP(hipMemcpyAsync(c.h_fctl, c.d_fctl, 3 * sizeof(int32_t), hipMemcpyDeviceToHost, c.stream));
    PT_HIP(hipStreamSynchronize(c.stream));
    if (c.h_fctl[0]) break;
    if (done > cap) {
      set_error("filter did not reach its smoothness threshold in 100000 passes");
      return PT_ERR_INVALID;
    }
    batch = std::min(2 * batch, 256 / a.K);
  }
  if (c.timing) timer_end(c, PT_K_FILTER);
  *passes = c.h_fctl[1];
  *hint = *passes;
  if (c.h_fctl[2] != 0) {
    const size_t bytes = sizeof(double) * (size_t)(c.T.nx + 1 + 2 * a.h) * (c.T.nz + 1 + 2 * a.h);
    PT_HIP(hipMemcpyAsync(x0, buf[c.h_fctl[2]], bytes, hipMemcpyDeviceToDevice, c.stream));
  }
  return PT_OK;
}

// C passes: the first ten with the Chebyshev-ordered steps that damp the
// unresolved frequencies first, then c = 1 (PS/smoother.f90:596-617)
static double cdts_comp(const Context& c, int j) {
  double cc = 1.0;
  if (j <= 10) {
    const int Niter = 10, ntemp = Niter - j + 1;
    const double lb = -5.0, la = -1.0;
    cc = 2.0 / (-lb - la + (lb - la) * std::cos((double)(2 * ntemp - 1) * 3.1415926535897932 / (double)(2 * Niter)));
  }
  return cc * (c.T.dts * c.P.courantC);
}
static double cdts_temp(const Context& c, int) { return c.T.dts * c.P.courantT; }

static int smoother_time_host(Context& c);

// smoother_time (C): PS/smoother.f90:582-636
static int smoother_time(Context& c) {
  size_t b5 = sizeof(double) * (size_t)(c.T.nx + 11) * (c.T.nz + 11);
  PT_HIP(hipMemcpyAsync(c.Cvis, c.Cnew, b5, hipMemcpyDeviceToDevice, c.stream));
  PT_HIP(hipMemcpyAsync(c.Cbuoy, c.Cnew, b5, hipMemcpyDeviceToDevice, c.stream));
  if (!c.filter_on_device) return smoother_time_host(c);
  // the reference passes the halo-5 C array to smoothness, whose dummy has
  // the halo-3 shape (PS/smoother.f90:79, :602): sequence association makes
  // it read the C storage with the halo-3 row length
  int P = 0;
  PT_TRY(filter_loop(c, c.Cvis, c.TxS, c.CxS, true, cdts_comp, &P, &c.hint_comp));
  // n_comp counts the outer iterations after the first ten-pass one
  c.n_comp = P < 10 ? 0 : P - 9;
  return PT_OK;
}

// smoother_time with a host round trip per check, the loop as the reference
// writes it (kept as the cross-check of the device-driven loop)
static int smoother_time_host(Context& c) {
  size_t b5 = sizeof(double) * (size_t)(c.T.nx + 11) * (c.T.nz + 11);
  int Niter = 10, nn = 0;
  double lb = -5.0, la = -1.0;
  bool trigger = false;
  for (;;) {
    if (nn > 100000) {
      set_error("smoother_time: C filter did not reach delta_C");
      return PT_ERR_INVALID;
    }
    for (int n = 1; n <= Niter; n++) {
      // the reference passes the halo-5 C array to smoothness, whose dummy has
      // the halo-3 shape (PS/smoother.f90:79, :602): sequence association
      // makes it read the C storage with the halo-3 row length
      double diff;
      PT_TRY(smoothness_host(c, c.Cvis, 3, c.T.nx + 7, &diff));
      if (diff < c.T.delta_C) { trigger = true; break; }
      double cc;
      if (nn == 0) {
        int ntemp = Niter - n + 1;
        cc = 2.0 / (-lb - la + (lb - la) * std::cos((double)(2 * ntemp - 1) * 3.1415926535897932 / (double)(2 * Niter)));
      } else {
        cc = 1.0;
      }
      // T0 = Cvis (copy), Cvis = filter(T0); c*dts*temp = (c*dts)*temp
      PT_HIP(hipMemcpyAsync(c.TxS, c.Cvis, b5, hipMemcpyDeviceToDevice, c.stream));
      filter_pass(c, c.TxS, c.Cvis, 5, cc * (c.T.dts * c.P.courantC), 1);
      c_bcs(c, c.Cvis);
    }
    if (trigger) break;
    Niter = 1;
    nn++;
  }
  c.n_comp = nn;
  return PT_OK;
}

// smoother_time_T: PS/smoother.f90:638-672 (Tin = Tratio)
static int smoother_time_T(Context& c) {
  size_t b3 = sizeof(double) * (size_t)(c.T.nx + 7) * (c.T.nz + 7);
  PT_HIP(hipMemcpyAsync(c.Tvis, c.Tratio, b3, hipMemcpyDeviceToDevice, c.stream));
  PT_HIP(hipMemcpyAsync(c.Tbuoy, c.Tratio, b3, hipMemcpyDeviceToDevice, c.stream));
  if (c.P.RaT == 0.0 || c.P.ivis == 0) return PT_OK;
  if (c.filter_on_device) {
    int P = 0;
    PT_TRY(filter_loop(c, c.Tvis, c.CxS, c.TxS, false, cdts_temp, &P, &c.hint_temp));
    c.n_temp = P;
    return PT_OK;
  }
  int n = 0;
  for (;;) {
    if (n > 100000) {
      set_error("smoother_time_T: T filter did not reach delta_T");
      return PT_ERR_INVALID;
    }
    double diff;
    PT_TRY(smoothness_host(c, c.Tvis, 3, c.T.nx + 7, &diff));
    if (diff < c.T.delta_T) { c.n_temp = n; break; }
    PT_HIP(hipMemcpyAsync(c.CxS, c.Tvis, b3, hipMemcpyDeviceToDevice, c.stream));
    filter_pass(c, c.CxS, c.Tvis, 3, c.T.dts * c.P.courantT, 0);
    t_bcs(c, c.Tvis);
    n++;
  }
  return PT_OK;
}

// load_conductivity_array: PS/energy.f90:59-86
__global__ void k_conduct_nodes(const double* Cvis, double* cond, int nx, int nz, double cf) {
  int i = blockIdx.x * blockDim.x + threadIdx.x, k = blockIdx.y * blockDim.y + threadIdx.y;
  if (i > nx || k > nz) return;
  cond[I5(i, k, nx + 11)] = 1.0 + Cvis[I5(i, k, nx + 11)] * (cf - 1.0);
}
__global__ void k_conduct_grad(const double* cond, double* cr, double* cs, int nx, int nz, double dr, double ds,
                               double d0, double d1, double d2, double d3, double d4) {
  int i = -3 + (int)(blockIdx.x * blockDim.x + threadIdx.x), k = -3 + (int)(blockIdx.y * blockDim.y + threadIdx.y);
  if (i > nx + 3 || k > nz + 3) return;
  const double D[5] = {d0, d1, d2, d3, d4};
  double sr = 0.0, ss = 0.0;
  for (int q = -2; q <= 2; q++) sr = sr + D[q + 2] * cond[I5(i + q, k, nx + 11)];
  for (int q = -2; q <= 2; q++) ss = ss + D[q + 2] * cond[I5(i, k + q, nx + 11)];
  cr[I3(i, k, nx + 7)] = sr / dr;
  cs[I3(i, k, nx + 7)] = ss / ds;
}
static void load_conductivity(Context& c) {
  int nx = c.T.nx, nz = c.T.nz;
  dim3 b16(64, 4);
  hipLaunchKernelGGL(k_conduct_nodes, grid2(nx + 1, nz + 1, b16), b16, 0, c.stream, c.Cvis, c.cond, nx, nz,
                     c.P.conduct_factor);
  launch1(c, k_sym_side, c.cond, (nz + 1) * 5, nx, nz, 5, nx + 11);
  launch1(c, k_sym_tb, c.cond, (nx + 11) * 5, nx, nz, 5, nx + 11);
  const double* D1 = c.T.D1;
  hipLaunchKernelGGL(k_conduct_grad, grid2(nx + 7, nz + 7, b16), b16, 0, c.stream, c.cond, c.cond_r, c.cond_s, nx, nz,
                     c.T.dr, c.T.ds, D1[1], D1[2], D1[3], D1[4], D1[5]);
}

// tracers_to_corners: PS/composition.f90:923-1087.  filters = false is the
// reference's smooth_vis=0 (no smoother_time / smoother_time_T).  With
// discrete types (iC_continuous=0, tracers_to_corners_OG :1090-1276 with
// shape_function=1) Ct holds Ttype as 0.0 / 1.0: the type-1 weight sum over
// the weight sum is count_type_real(1)/nempty_real, the same weighted
// average, and nempty counts the same nearest-node tracers.
int tracers_to_corners(Context& c, const double* r, const double* s, const double* Tt, bool filters) {
  const int nx = c.T.nx, nz = c.T.nz, ncell = (nx + 1) * (nz + 1);
  const int64_t n = c.T.ntr;
  size_t b3 = sizeof(double) * (size_t)(nx + 7) * (nz + 7);
  if (c.timing) timer_begin(c, PT_K_PROJECT);
  PT_HIP(hipMemcpyAsync(c.Tratio, c.T0, b3, hipMemcpyDeviceToDevice, c.stream));
  PT_HIP(hipMemsetAsync(c.d_flags, 0, sizeof(int32_t) * 4, c.stream));
  unsigned nbt = (unsigned)((n + 255) / 256);
  // The windowed sort needs the storage order of an earlier projection and
  // no tracer more than one cell from its slot's cell.  Under-resolved flows
  // move tracers several cells per stage; after such a projection the next
  // WINDOW_BACKOFF projections take the radix sort without asking.
  constexpr int WINDOW_BACKOFF = 8;
  const bool try_window = c.order_valid && !c.project_radix_only && c.window_skip == 0;
  if (c.window_skip > 0) c.window_skip--;
  hipLaunchKernelGGL(k_bin, dim3(nbt), dim3(256), 0, c.stream, r, s, n, nx, nz, c.T.dr, c.T.ds, c.T.aspect,
                     c.cellkey, c.d_flags, try_window ? c.okey : nullptr);
  bool windowed = false;
  if (try_window) {
    // the domain check first, as the reference's binning loop does
    // (PS/composition.f90:1002-1011); then the sort the order allows
    PT_HIP(hipMemcpyAsync(c.h_fctl, c.d_flags, 2 * sizeof(int32_t), hipMemcpyDeviceToHost, c.stream));
    PT_HIP(hipStreamSynchronize(c.stream));
    if (c.h_fctl[0]) {
      if (c.timing) timer_end(c, PT_K_PROJECT);
      set_error("tracer position outside [0,aspect]x[0,1]");
      return PT_ERR_TRACER_OUTSIDE;
    }
    windowed = c.h_fctl[1] == 0;
    if (!windowed) c.window_skip = WINDOW_BACKOFF;
  }
  if (windowed) {
    const dim3 gcs((unsigned)((nx + 1 + CS_CELLS - 1) / CS_CELLS), (unsigned)(nz + 1));
    const int nblk = (int)(gcs.x * gcs.y);
    hipLaunchKernelGGL(k_cs_count, gcs, dim3(CS_THREADS), 0, c.stream, c.cellkey, c.ostart, c.oend, nx, nz, c.ccount,
                       c.bsum);
    hipLaunchKernelGGL(k_cs_scan, dim3(1), dim3(1024), 0, c.stream, c.bsum, nblk, n, c.d_flags);
    hipLaunchKernelGGL(k_cs_fill, gcs, dim3(CS_THREADS), 0, c.stream, c.cellkey, c.ostart, c.oend, nx, nz, c.ccount,
                       c.bsum, c.cstart, c.cend, c.perm, c.skey);
    c.proj_window++;
  } else {
    PT_HIP(hipMemsetAsync(c.cstart, 0, sizeof(int32_t) * ncell, c.stream));
    PT_HIP(hipMemsetAsync(c.cend, 0, sizeof(int32_t) * ncell, c.stream));
    PT_TRY(sort_pairs(c.sort_tmp, c.sort_bytes, c.cellkey, c.skey, c.iota, c.perm, n, c.sort_bits, c.stream));
    hipLaunchKernelGGL(k_cell_bounds, dim3(nbt), dim3(256), 0, c.stream, c.skey, n, ncell, c.cstart, c.cend);
    c.proj_fallback++;
  }
  hipLaunchKernelGGL(k_cell_reduce, dim3((ncell + PJ_CELLS - 1) / PJ_CELLS), dim3(PJ_THREADS), 0, c.stream, r, s, Tt,
                     c.Ct, c.perm, c.skey, n, c.cstart, c.cend, c.cellsum, nx, nz, c.T.dr, c.T.ds);
  dim3 b16(64, 4);
  hipLaunchKernelGGL(k_node_combine, grid2(nx + 1, nz + 1, b16), b16, 0, c.stream, c.cellsum, c.cstart, c.cend,
                     c.Tratio, c.Cnew, c.nempty, nx, nz);
  if (c.timing) timer_end(c, PT_K_PROJECT);
  PT_HIP(hipMemcpyAsync(c.h_fctl, c.d_flags, 3 * sizeof(int32_t), hipMemcpyDeviceToHost, c.stream));
  PT_HIP(hipStreamSynchronize(c.stream));
  if (c.h_fctl[0]) {
    set_error("tracer position outside [0,aspect]x[0,1]");
    return PT_ERR_TRACER_OUTSIDE;
  }
  if (c.h_fctl[2]) {
    set_error("projection: the windowed counting sort did not place every tracer");
    return PT_ERR_INVALID;
  }
  c_bcs(c, c.Cnew);
  if (filters) PT_TRY(smoother_time(c));
  t_bcs(c, c.Tratio);
  if (filters) PT_TRY(smoother_time_T(c));
  load_conductivity(c);
  return PT_OK;
}

// ---------------------------------------------------------------------------
// source term, derivative tables, RK stages
// ---------------------------------------------------------------------------
__global__ void k_source(const double* Tx_, const double* cond, const double* cr, const double* cs, const double* Cvis,
                         double* src, int nx, int nz, double dr, double ds, double dr2, double ds2, double H,
                         double Htype, double d10, double d11, double d12, double d13, double d14, double d20,
                         double d21, double d22, double d23, double d24) {
  int i = -3 + (int)(blockIdx.x * blockDim.x + threadIdx.x), k = -3 + (int)(blockIdx.y * blockDim.y + threadIdx.y);
  if (i > nx + 3 || k > nz + 3) return;
  const double D1[5] = {d10, d11, d12, d13, d14}, D2[5] = {d20, d21, d22, d23, d24};
  const int p5 = nx + 11;
  double sx = 0, sz = 0, sxx = 0, szz = 0;
  for (int q = -2; q <= 2; q++) sx = sx + D1[q + 2] * Tx_[I5(i + q, k, p5)];
  for (int q = -2; q <= 2; q++) sz = sz + D1[q + 2] * Tx_[I5(i, k + q, p5)];
  for (int q = -2; q <= 2; q++) sxx = sxx + D2[q + 2] * Tx_[I5(i + q, k, p5)];
  for (int q = -2; q <= 2; q++) szz = szz + D2[q + 2] * Tx_[I5(i, k + q, p5)];
  double Tx = sx / dr, Tz = sz / ds, Txx = sxx / dr2, Tzz = szz / ds2;
  double kx = cr[I3(i, k, nx + 7)], kz = cs[I3(i, k, nx + 7)];
  double cv = Cvis[I5(i, k, p5)];
  double h = Htype * cv + H * (1.0 - (0.0 + cv));
  src[I3(i, k, nx + 7)] = cond[I5(i, k, p5)] * (Txx + Tzz) + (kx * Tx + kz * Tz) + h;
}

// interpolation table: tab[((i*(nz+7)) + (k+3))*12 + f*4 + d], f in {u,w,src},
// d = {value, DERr(1), DERr(2), DERr(3)}; i in 0..nx, k in -3..nz+3
__global__ void k_itab(const double* u, const double* w, const double* src, double* tab, int nx, int nz,
                       const double* Dm, double p1, double p2, double p3) {
  int k = -3 + (int)(blockIdx.x * blockDim.x + threadIdx.x), i = blockIdx.y * blockDim.y + threadIdx.y;
  if (i > nx || k > nz + 3) return;
  const double* fs[3] = {u, w, src};
  const double pw[3] = {p1, p2, p3};
  long base = ((long)i * (nz + 7) + (k + 3)) * 12;
  for (int f = 0; f < 3; f++) {
    const double* F = fs[f];
    tab[base + f * 4] = F[I3(i, k, nx + 7)];
    for (int jj = 1; jj <= 3; jj++) {
      double sacc = 0.0;
      for (int a = -3; a <= 3; a++) sacc = sacc + Dm[(jj - 1) * 7 + a + 3] * F[I3(i + a, k, nx + 7)];
      tab[base + f * 4 + jj] = sacc / pw[jj - 1];
    }
  }
}

// hr**3 as the correctly rounded cube (the reference evaluates hr**real(3,8)
// with libm pow); FMA-based double-double product, rounded once
__device__ __forceinline__ double cube_cr(double x) {
  double p = x * x;
  double e = __fma_rn(x, x, -p);
  double t = p * x;
  double te = __fma_rn(p, x, -t);
  return t + (te + e * x);
}

struct InterpConst {
  int nx, nz;
  double dr, ds, f3;             // factorial(3)
};
struct InterpConstTab {
  double dsp1, dsp2, dsp3;       // ds_power(1..3)
  double Dm[3][7];               // D(1..3, -3..3)
};

// Per-node coefficient table of the interpolation polynomial.  interpolate
// (PS/composition.f90:1359-1393) evaluates, around the tracer's node (i,k),
//   fR(jj) = T0(jj) + a1 T1(jj) + a2 T2(jj) + a3 T3(jj),   jj = k-3..k+3,
//   out    = fR(k) + b1 d1 + b2 d2 + b3 d3,  d_q = sum_jj D(q,jj) fR(jj) / ds^q,
// with T_p = DERr(p) (T_0 = f), a_p = hr^p/p!, b_q = hs^q/q!.  That is the
// bicubic  out = sum_q b_q sum_p a_p C_pq  with  C_p0 = T_p(k),
// C_pq = sum_jj D(q,jj) T_p(jj) / ds^q.  The C_pq depend on the node only, so
// they are formed once per stage here (16 per field) and a tracer evaluates
// 4+1 short sums instead of 7 rows of Taylor sums and three derivative sums
// with their divisions.  Same polynomial; the rounding differs from the
// reference's order at the level of the last bit.
// ctab[node*48 + f*16 + q*4 + p], node = k*(nx+1) + i, f in {u, w, source}.
// One thread per coefficient, in ctab order, so a wave's stores are one
// contiguous run; the 7-row sums keep the order jj = 0..6.
__global__ void k_ctab(const double* __restrict__ tab, double* __restrict__ ctab, int nx, int nz, InterpConstTab C) {
  const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
  const long nnode = (long)(nx + 1) * (nz + 1);
  if (t >= nnode * 48) return;
  const int node = (int)(t / 48), e = (int)(t - (long)node * 48);
  const int k = node / (nx + 1), i = node - k * (nx + 1);
  const int f = e >> 4, q = (e >> 2) & 3, p = e & 3;
  const double* col = tab + ((long)i * (nz + 7) + k) * 12 + f * 4 + p;   // row kk = k-3 at offset 0
  double v;
  if (q == 0) {
    v = col[3 * 12];
  } else {
    const double* D = C.Dm[q - 1];
    double acc = 0.0;
#pragma unroll
    for (int jj = 0; jj < 7; jj++) acc = acc + D[jj] * col[jj * 12];
    v = acc / (q == 1 ? C.dsp1 : (q == 2 ? C.dsp2 : C.dsp3));
  }
  ctab[t] = v;
}

// ---- interpolation at the tracers ------------------------------------------
// A workgroup holds RK_THREADS consecutive tracers of the cell-ordered SoA.
// Sorted by nearest node at the step's start, they reach a small box of
// nodes (at 1024x256 and 50 tracers per node: 6-7 nodes at stage 1, 14-24
// at the drifted stage positions).  The workgroup reduces the box, copies
// its coefficients from ctab into LDS with contiguous loads, and every lane
// reads its node's 48 coefficients (384 B) there, so the vector-memory path
// carries the tracer streams and one copy of the box per workgroup.  A box
// larger than RK_BOX nodes (a workgroup that wraps a grid row, or positions
// spread far) reads ctab directly.  Same coefficients in the same order:
// the results do not depend on the path.
constexpr int RK_THREADS = 256;
constexpr int RK_BOX = 42;     // staged nodes: 42 * 24 double2 fit 4 loads per thread
constexpr int RK_NODE = 25;    // double2 per staged node: 24 + 1 pad spreads nodes over LDS banks
static_assert(RK_BOX * 24 <= 4 * RK_THREADS, "box copy is 4 double2 per thread");

struct Located {
  int i, k;                      // nearest node
  double a1, a2, a3, b1, b2, b3; // hr^p/p!, hs^q/q!
};
__device__ __forceinline__ Located locate(const InterpConst& C, double r, double s) {
  Located p;
  int i = (int)round(r / C.dr), k = (int)round(s / C.ds);
  // positions reaching this point passed the projection's domain check;
  // the clamp only guards the table reads
  i = i < 0 ? 0 : (i > C.nx ? C.nx : i);
  k = k < 0 ? 0 : (k > C.nz ? C.nz : k);
  // factorial(1) = 1 and factorial(2) = 2 exactly, so h/factorial(1) = h and
  // h^2/factorial(2) = h^2 * 0.5 are the reference's quotients bit for bit
  const double hr = r - (double)i * C.dr;
  p.a1 = hr; p.a2 = (hr * hr) * 0.5; p.a3 = cube_cr(hr) / C.f3;
  const double hs = s - (double)k * C.ds;
  p.b1 = hs; p.b2 = (hs * hs) * 0.5; p.b3 = cube_cr(hs) / C.f3;
  p.i = i; p.k = k;
  return p;
}
// the bicubic from one node's 24 double2 of C_pq (LDS or global pointer)
template <typename P>
__device__ __forceinline__ void eval3(P cf, const Located& p, double out[3]) {
#pragma unroll
  for (int f = 0; f < 3; f++) {
    double g[4];
#pragma unroll
    for (int q = 0; q < 4; q++) {
      const double2 lo = cf[f * 8 + q * 2], hi = cf[f * 8 + q * 2 + 1];
      double v = lo.x;
      v = v + lo.y * p.a1;
      v = v + hi.x * p.a2;
      v = v + hi.y * p.a3;
      g[q] = v;
    }
    double fi = g[0];
    fi = fi + g[1] * p.b1;
    fi = fi + g[2] * p.b2;
    fi = fi + g[3] * p.b3;
    out[f] = fi;
  }
}
// workgroup barrier that orders LDS only: global loads issued before it stay
// in flight
__device__ __forceinline__ void lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}
__device__ __forceinline__ int wave_min(int v) {
#pragma unroll
  for (int o = 32; o; o >>= 1) v = min(v, __shfl_xor(v, o));
  return v;
}
__device__ __forceinline__ int wave_max(int v) {
#pragma unroll
  for (int o = 32; o; o >>= 1) v = max(v, __shfl_xor(v, o));
  return v;
}
// interpolate for the three fields at (r, s).  Every thread of the workgroup
// calls it (threads past the last tracer pass that tracer's position), since
// it holds two workgroup barriers.
__device__ __forceinline__ void interp3(const double* __restrict__ ctab, const InterpConst& C, double r, double s,
                                        double out[3]) {
  __shared__ double2 box[RK_BOX * RK_NODE];
  __shared__ int bb[RK_THREADS / 64][4];
  const Located p = locate(C, r, s);
  const int i0w = wave_min(p.i), i1w = wave_max(p.i), k0w = wave_min(p.k), k1w = wave_max(p.k);
  if ((threadIdx.x & 63) == 0) {
    const int wv = threadIdx.x >> 6;
    bb[wv][0] = i0w; bb[wv][1] = i1w; bb[wv][2] = k0w; bb[wv][3] = k1w;
  }
  lds_sync();
  int i0 = bb[0][0], i1 = bb[0][1], k0 = bb[0][2], k1 = bb[0][3];
#pragma unroll
  for (int q = 1; q < RK_THREADS / 64; q++) {
    i0 = min(i0, bb[q][0]); i1 = max(i1, bb[q][1]); k0 = min(k0, bb[q][2]); k1 = max(k1, bb[q][3]);
  }
  // the box [i0,i1] x [k0,k1] holds every thread's node; `staged` is the
  // same in all threads
  const int w = i1 - i0 + 1, h = k1 - k0 + 1;
  const bool staged = w * h <= RK_BOX;
  const double2* g2 = reinterpret_cast<const double2*>(ctab);
  if (staged) {
    // box rows are contiguous runs of w nodes in ctab; loads are clamped to
    // the box so they can all be issued before the first store
    const int total = w * h * 24, per = w * 24;
    double2 v[4];
    int dst[4];
#pragma unroll
    for (int u = 0; u < 4; u++) {
      const int t = threadIdx.x + u * RK_THREADS;
      const int tc = t < total ? t : total - 1;
      const int row = tc / per, rem = tc - row * per;
      const int nd = rem / 24, q = rem - nd * 24;
      v[u] = g2[((long)(k0 + row) * (C.nx + 1) + i0) * 24 + rem];
      dst[u] = t < total ? (row * w + nd) * RK_NODE + q : -1;
    }
#pragma unroll
    for (int u = 0; u < 4; u++)
      if (dst[u] >= 0) box[dst[u]] = v[u];
  }
  lds_sync();
  if (staged)
    eval3(box + ((p.k - k0) * w + (p.i - i0)) * RK_NODE, p, out);
  else
    eval3(g2 + ((long)p.k * (C.nx + 1) + p.i) * 24, p, out);
}

struct RkArgs {
  double *r, *s, *T;                 // r, s, Ttr (accumulators after stage 1)
  double *r0, *s0, *T0;              // step-start copies
  double *r1, *s1, *T1, *r2, *s2, *T2;
  const double* tab;                 // ctab (per-node polynomial coefficients)
  int64_t n;
  double dtstage;                    // stage-specific step
  InterpConst C;
};

// The tracer streams are read and written once per stage kernel:
// nontemporal loads and stores keep them from displacing the coefficient
// table in the caches.  Each kernel issues all of its stream loads before
// the interpolation's barriers; threads past the last tracer load that
// tracer (j clamped) and store nothing.
#define NT_LD(x) __builtin_nontemporal_load(&(x))
#define NT_ST(x, v) __builtin_nontemporal_store((v), &(x))

// stage 1: PS/energy.f90:258-301
__global__ void __launch_bounds__(RK_THREADS) k_rk1(RkArgs a) {
  const int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x, jc = j < a.n ? j : a.n - 1;
  const double rv = NT_LD(a.r[jc]), sv = NT_LD(a.s[jc]), Tv = NT_LD(a.T[jc]);
  double o[3];
  interp3(a.tab, a.C, rv, sv, o);
  if (j >= a.n) return;
  NT_ST(a.r0[j], rv); NT_ST(a.s0[j], sv); NT_ST(a.T0[j], Tv);
  NT_ST(a.r[j], o[0]); NT_ST(a.s[j], o[1]); NT_ST(a.T[j], o[2]);
  NT_ST(a.r1[j], rv + a.dtstage * o[0]);
  NT_ST(a.s1[j], sv + a.dtstage * o[1]);
  NT_ST(a.T1[j], Tv + a.dtstage * o[2]);
}
// stage 2: PS/energy.f90:350-402
__global__ void __launch_bounds__(RK_THREADS) k_rk2(RkArgs a) {
  const int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x, jc = j < a.n ? j : a.n - 1;
  const double rv = NT_LD(a.r[jc]), sv = NT_LD(a.s[jc]), Tv = NT_LD(a.T[jc]);
  const double r0 = NT_LD(a.r0[jc]), s0 = NT_LD(a.s0[jc]), T0 = NT_LD(a.T0[jc]);
  double o[3];
  interp3(a.tab, a.C, NT_LD(a.r1[jc]), NT_LD(a.s1[jc]), o);
  if (j >= a.n) return;
  NT_ST(a.r[j], rv + 2.0 * o[0]);
  NT_ST(a.s[j], sv + 2.0 * o[1]);
  NT_ST(a.T[j], Tv + 2.0 * o[2]);
  NT_ST(a.r2[j], r0 + a.dtstage * o[0]);
  NT_ST(a.s2[j], s0 + a.dtstage * o[1]);
  NT_ST(a.T2[j], T0 + a.dtstage * o[2]);
}
// stage 3: PS/energy.f90:450-473
__global__ void __launch_bounds__(RK_THREADS) k_rk3(RkArgs a) {
  const int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x, jc = j < a.n ? j : a.n - 1;
  const double rv = NT_LD(a.r[jc]), sv = NT_LD(a.s[jc]), Tv = NT_LD(a.T[jc]);
  const double r0 = NT_LD(a.r0[jc]), s0 = NT_LD(a.s0[jc]), T0 = NT_LD(a.T0[jc]);
  double o[3];
  interp3(a.tab, a.C, NT_LD(a.r2[jc]), NT_LD(a.s2[jc]), o);
  if (j >= a.n) return;
  NT_ST(a.r[j], rv + 2.0 * o[0]);
  NT_ST(a.r1[j], r0 + a.dtstage * o[0]);
  NT_ST(a.s[j], sv + 2.0 * o[1]);
  NT_ST(a.s1[j], s0 + a.dtstage * o[1]);
  NT_ST(a.T[j], Tv + 2.0 * o[2]);
  NT_ST(a.T1[j], T0 + a.dtstage * o[2]);
}
// stage 4: PS/energy.f90:517-537 (dtstage = dt/6)
__global__ void __launch_bounds__(RK_THREADS) k_rk4(RkArgs a) {
  const int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x, jc = j < a.n ? j : a.n - 1;
  const double rv = NT_LD(a.r[jc]), sv = NT_LD(a.s[jc]), Tv = NT_LD(a.T[jc]);
  const double r0 = NT_LD(a.r0[jc]), s0 = NT_LD(a.s0[jc]), T0 = NT_LD(a.T0[jc]);
  double o[3];
  interp3(a.tab, a.C, NT_LD(a.r1[jc]), NT_LD(a.s1[jc]), o);
  if (j >= a.n) return;
  NT_ST(a.r[j], r0 + a.dtstage * (rv + o[0]));
  NT_ST(a.s[j], s0 + a.dtstage * (sv + o[1]));
  NT_ST(a.T[j], T0 + a.dtstage * (Tv + o[2]));
}

static int source_and_tables(Context& c, bool velocity_too) {
  int nx = c.T.nx, nz = c.T.nz;
  dim3 b16(64, 4);
  (void)velocity_too;
  extend_t(c);
  const double *D1 = c.T.D1, *D2 = c.T.D2;
  hipLaunchKernelGGL(k_source, grid2(nx + 7, nz + 7, b16), b16, 0, c.stream, c.Textend, c.cond, c.cond_r, c.cond_s,
                     c.Cvis, c.src, nx, nz, c.T.dr, c.T.ds, c.T.dr2, c.T.ds2, c.P.H, c.P.Htype, D1[1], D1[2], D1[3],
                     D1[4], D1[5], D2[1], D2[2], D2[3], D2[4], D2[5]);
  return PT_OK;
}

static int build_tables(Context& c, const double* u, const double* w, const double* src) {
  int nx = c.T.nx, nz = c.T.nz;
  dim3 b(64, 4);
  hipLaunchKernelGGL(k_itab, grid2(nz + 7, nx + 1, b), b, 0, c.stream, u, w, src, c.itab, nx, nz,
                     (const double*)c.dtab, c.T.dr_power[1], c.T.dr_power[2], c.T.dr_power[3]);
  InterpConstTab C;
  C.dsp1 = c.T.ds_power[1]; C.dsp2 = c.T.ds_power[2]; C.dsp3 = c.T.ds_power[3];
  for (int m = 0; m < 3; m++)
    for (int q = 0; q < 7; q++) C.Dm[m][q] = c.T.D[m + 1][q];
  const long ncoef = (long)(nx + 1) * (nz + 1) * 48;
  hipLaunchKernelGGL(k_ctab, dim3((unsigned)((ncoef + 255) / 256)), dim3(256), 0, c.stream, c.itab, c.ctab, nx, nz, C);
  return PT_OK;
}
static int build_itab(Context& c) { return build_tables(c, c.u, c.w, c.src); }

static RkArgs rk_args(Context& c) {
  RkArgs a;
  a.r = c.r; a.s = c.s; a.T = c.Tt; a.r0 = c.r0; a.s0 = c.s0; a.T0 = c.T0t;
  a.r1 = c.r1; a.s1 = c.s1; a.T1 = c.T1t; a.r2 = c.r2; a.s2 = c.s2; a.T2 = c.T2t;
  a.tab = c.ctab; a.n = c.T.ntr;
  a.C.nx = c.T.nx; a.C.nz = c.T.nz;
  a.C.dr = c.T.dr; a.C.ds = c.T.ds; a.C.f3 = c.T.factorial[3];
  return a;
}

// stability_RK4 with tracers (CFL=0): PS/energy.f90:756-810
__global__ void k_eig_max(const double* cond, const double* cr, const double* cs, int nx, int nz, double Tr_max,
                          double Ts_max, double Trr_max, double Tss_max, double* partial) {
  __shared__ double ra[256], rd[256];
  int tid = threadIdx.y * blockDim.x + threadIdx.x;
  int i = blockIdx.x * blockDim.x + threadIdx.x, k = blockIdx.y * blockDim.y + threadIdx.y;
  double eA = 0.0, eD = 0.0;
  if (i <= nx && k <= nz) {
    double cd = cond[I5(i, k, nx + 11)];
    eA = fabs(-(cd * 0.0 / 1.0) + cr[I3(i, k, nx + 7)] / 1.0) * Tr_max +
         fabs(-(cd * 0.0 / 1.0) + cs[I3(i, k, nx + 7)] / 1.0) * Ts_max;
    eD = cd * (fabs(Trr_max / 1.0) + fabs(Tss_max / 1.0));
  }
  ra[tid] = eA; rd[tid] = eD;
  __syncthreads();
  for (int st = 128; st > 0; st >>= 1) {
    if (tid < st) { ra[tid] = fmax(ra[tid], ra[tid + st]); rd[tid] = fmax(rd[tid], rd[tid + st]); }
    __syncthreads();
  }
  if (tid == 0) {
    int b = blockIdx.y * gridDim.x + blockIdx.x;
    partial[2 * b] = ra[0];
    partial[2 * b + 1] = rd[0];
  }
}
__global__ void k_eig_final(const double* partial, int nb, double* out) {
  if (threadIdx.x == 0) {
    double a = 0.0, d = 0.0;
    for (int b = 0; b < nb; b++) { a = fmax(a, partial[2 * b]); d = fmax(d, partial[2 * b + 1]); }
    out[0] = a; out[1] = d;
  }
}
static int stability_rk4(Context& c) {
  const Tables& t = c.T;
  double Ts_max = t.Tr_base / t.ds, Tss_max = -t.Trr_base / t.ds2, Tr_max = t.Tr_base / t.dr,
         Trr_max = -t.Trr_base / t.dr2;
  dim3 b16(64, 4);
  dim3 g = grid2(t.nx + 1, t.nz + 1, b16);
  hipLaunchKernelGGL(k_eig_max, g, b16, 0, c.stream, c.cond, c.cond_r, c.cond_s, t.nx, t.nz, Tr_max, Ts_max, Trr_max,
                     Tss_max, c.red);
  hipLaunchKernelGGL(k_eig_final, dim3(1), dim3(64), 0, c.stream, c.red, (int)(g.x * g.y), c.red_out);
  PT_HIP(hipMemcpyAsync(c.h_red, c.red_out, 2 * sizeof(double), hipMemcpyDeviceToHost, c.stream));
  PT_HIP(hipStreamSynchronize(c.stream));
  double eA = c.h_red[0], eD = c.h_red[1];
  double dtA = 2.8 / eA, dtD = 2.8 / eD, dt;
  if (eA == 0.0) dt = dtD;
  else dt = 1.0 / (1.0 / dtA + 1.0 / dtD);
  c.dt = c.P.courant * dt;
  return PT_OK;
}

static int update_velocities(Context& c) {
  PT_TRY(solve_stream(c));
  return compute_velocities(c);
}

// `which` names the stage's own timer (PT_K_TRACER_RK2 for stage 2, else -1);
// every stage also counts towards PT_K_TRACER_STAGE
static void rk_launch(Context& c, void (*kern)(RkArgs), RkArgs a, int which = -1) {
  unsigned nb = (unsigned)((a.n + RK_THREADS - 1) / RK_THREADS);
  if (c.timing) timer_begin(c, PT_K_TRACER_STAGE);
  if (c.timing && which >= 0) timer_begin(c, which);
  hipLaunchKernelGGL(kern, dim3(nb), dim3(RK_THREADS), 0, c.stream, a);
  if (c.timing && which >= 0) timer_end(c, which);
  if (c.timing) timer_end(c, PT_K_TRACER_STAGE);
}

// energy_time: PS/energy.f90:181-556 (tracer=1, comp=1, torder=4, RK_update=1)
static int reorder_tracers(Context& c);

int energy_time(Context& c) {
  PT_TRY(stability_rk4(c));
  if (c.P.equalize == 1) PT_TRY(equalize_tracers(c));   // PS/energy.f90:198-204
  const double dt = c.dt;
  const int nx = c.T.nx, nz = c.T.nz;
  size_t b3 = sizeof(double) * (size_t)(nx + 7) * (nz + 7), b5 = sizeof(double) * (size_t)(nx + 11) * (nz + 11);
  PT_HIP(hipMemcpyAsync(c.C0, c.Cnew, b5, hipMemcpyDeviceToDevice, c.stream));
  PT_HIP(hipMemcpyAsync(c.T0, c.Tratio, b3, hipMemcpyDeviceToDevice, c.stream));
  RkArgs a = rk_args(c);
  // stage 1
  PT_TRY(source_and_tables(c, true));
  PT_TRY(build_itab(c));
  a.dtstage = 0.5 * dt;
  rk_launch(c, k_rk1, a);
  // stage 2
  PT_TRY(tracers_to_corners(c, c.r1, c.s1, c.T1t));
  PT_TRY(source_and_tables(c, false));
  PT_TRY(update_velocities(c));
  PT_TRY(build_itab(c));
  a.dtstage = 0.5 * dt;
  rk_launch(c, k_rk2, a, PT_K_TRACER_RK2);
  // stage 3
  PT_HIP(hipMemcpyAsync(c.Cnew, c.C0, b5, hipMemcpyDeviceToDevice, c.stream));
  PT_TRY(tracers_to_corners(c, c.r2, c.s2, c.T2t));
  PT_TRY(source_and_tables(c, false));
  PT_TRY(update_velocities(c));
  PT_TRY(build_itab(c));
  a.dtstage = dt;
  rk_launch(c, k_rk3, a);
  // stage 4
  PT_HIP(hipMemcpyAsync(c.Cnew, c.C0, b5, hipMemcpyDeviceToDevice, c.stream));
  PT_TRY(tracers_to_corners(c, c.r1, c.s1, c.T1t));
  PT_TRY(source_and_tables(c, false));
  PT_TRY(update_velocities(c));
  PT_TRY(build_itab(c));
  a.dtstage = dt / 6.0;
  rk_launch(c, k_rk4, a);
  // wrap up
  PT_HIP(hipMemcpyAsync(c.Cnew, c.C0, b5, hipMemcpyDeviceToDevice, c.stream));
  PT_TRY(tracers_to_corners(c, c.r, c.s, c.Tt));
  PT_TRY(reorder_tracers(c));
  c.t_initial = false;   // T = Tratio (PS/energy.f90:552)
  return PT_OK;
}

// initial state: PS/basics.f90:352-359, PS/composition.f90:848, PS/main.f90:228-229
__global__ void k_load_T(const double* Tn, double* T, int nx, int nz) {
  int i = blockIdx.x * blockDim.x + threadIdx.x, k = blockIdx.y * blockDim.y + threadIdx.y;
  if (i > nx || k > nz) return;
  T[I3(i, k, nx + 7)] = Tn[(long)k * (nx + 1) + i];
}

// Storage order of the tracers: after the projection of the step's final
// positions the SoA arrays are permuted into that projection's cell order
// (stable: ascending slot within a cell), so the next step's interpolation
// gathers and projection reads walk the grid cell by cell.
__global__ void k_reorder(const int32_t* __restrict__ perm, int64_t n, const double* __restrict__ r,
                          const double* __restrict__ s, const double* __restrict__ T, const double* __restrict__ C,
                          const int32_t* __restrict__ id, double* __restrict__ r2, double* __restrict__ s2,
                          double* __restrict__ T2, double* __restrict__ C2, int32_t* __restrict__ id2) {
  int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= n) return;
  const int32_t q = perm[j];
  r2[j] = r[q];
  s2[j] = s[q];
  T2[j] = T[q];
  C2[j] = C[q];
  id2[j] = id[q];
}
static int reorder_tracers(Context& c) {
  const int64_t n = c.T.ntr;
  hipLaunchKernelGGL(k_reorder, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, c.stream, c.perm, n, c.r, c.s,
                     c.Tt, c.Ct, c.tid, c.r1, c.s1, c.T1t, c.r2, c.tid_tmp);
  std::swap(c.r, c.r1);
  std::swap(c.s, c.s1);
  std::swap(c.Tt, c.T1t);
  std::swap(c.Ct, c.r2);
  std::swap(c.tid, c.tid_tmp);
  // the new storage order is the last projection's cell order
  std::swap(c.okey, c.skey);
  std::swap(c.ostart, c.cstart);
  std::swap(c.oend, c.cend);
  c.order_valid = true;
  return PT_OK;
}
__global__ void k_to_id_order(const int32_t* __restrict__ id, int64_t n, const double* __restrict__ a,
                              double* __restrict__ out) {
  int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (j < n) out[id[j]] = a[j];
}
// the RK4 registers r1, s1, T1t, r2 are free between steps and hold the result
int tracers_in_id_order(Context& c, double** r, double** s, double** Tt, double** Ct) {
  const int64_t n = c.T.ntr;
  const dim3 g((unsigned)((n + 255) / 256)), b(256);
  if (r) { hipLaunchKernelGGL(k_to_id_order, g, b, 0, c.stream, c.tid, n, c.r, c.r1); *r = c.r1; }
  if (s) { hipLaunchKernelGGL(k_to_id_order, g, b, 0, c.stream, c.tid, n, c.s, c.s1); *s = c.s1; }
  if (Tt) { hipLaunchKernelGGL(k_to_id_order, g, b, 0, c.stream, c.tid, n, c.Tt, c.T1t); *Tt = c.T1t; }
  if (Ct) { hipLaunchKernelGGL(k_to_id_order, g, b, 0, c.stream, c.tid, n, c.Ct, c.r2); *Ct = c.r2; }
  return PT_OK;
}

// ---- helpers of the tracer redistribution (pt_equalize.hip) ----------------
// The storage order as the cell order of the current positions (ostart /
// oend per cell, okey per slot).  Every projection of a step's final
// positions leaves it so; otherwise bin, sort and reorder here.
int ensure_cell_order(Context& c) {
  if (c.order_valid) return PT_OK;
  const int nx = c.T.nx, nz = c.T.nz, ncell = (nx + 1) * (nz + 1);
  const int64_t n = c.T.ntr;
  const unsigned nbt = (unsigned)((n + 255) / 256);
  PT_HIP(hipMemsetAsync(c.d_flags, 0, sizeof(int32_t) * 4, c.stream));
  hipLaunchKernelGGL(k_bin, dim3(nbt), dim3(256), 0, c.stream, c.r, c.s, n, nx, nz, c.T.dr, c.T.ds, c.T.aspect,
                     c.cellkey, c.d_flags, nullptr);
  PT_HIP(hipMemsetAsync(c.cstart, 0, sizeof(int32_t) * ncell, c.stream));
  PT_HIP(hipMemsetAsync(c.cend, 0, sizeof(int32_t) * ncell, c.stream));
  PT_TRY(sort_pairs(c.sort_tmp, c.sort_bytes, c.cellkey, c.skey, c.iota, c.perm, n, c.sort_bits, c.stream));
  hipLaunchKernelGGL(k_cell_bounds, dim3(nbt), dim3(256), 0, c.stream, c.skey, n, ncell, c.cstart, c.cend);
  PT_HIP(hipMemcpyAsync(c.h_fctl, c.d_flags, sizeof(int32_t), hipMemcpyDeviceToHost, c.stream));
  PT_HIP(hipStreamSynchronize(c.stream));
  if (c.h_fctl[0]) {
    set_error("tracer position outside [0,aspect]x[0,1]");
    return PT_ERR_TRACER_OUTSIDE;
  }
  return reorder_tracers(c);
}

// Textend(-3:nx+3,-3:nz+3) into a halo-3 field (the reference's Tdumb)
__global__ void k_window3(const double* T5, double* T3, int nx, int nz) {
  int i = -3 + (int)(blockIdx.x * blockDim.x + threadIdx.x), k = -3 + (int)(blockIdx.y * blockDim.y + threadIdx.y);
  if (i > nx + 3 || k > nz + 3) return;
  T3[I3(i, k, nx + 7)] = T5[I5(i, k, nx + 11)];
}
// T at the listed tracer slots from the coefficient table of one field
__global__ void k_interp_slots(const double* __restrict__ ctab, InterpConst C, const int32_t* __restrict__ slots,
                               int64_t n, const double* __restrict__ r, const double* __restrict__ s,
                               double* __restrict__ T) {
  const int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= n) return;
  const int32_t q = slots[j];
  const Located p = locate(C, r[q], s[q]);
  double o[3];
  eval3(reinterpret_cast<const double2*>(ctab) + ((long)p.k * (C.nx + 1) + p.i) * 24, p, o);
  T[q] = o[0];
}
// Ttr of redistributed tracers: extendT(Tratio), compute_derivatives of
// Textend(-3:nx+3,-3:nz+3) and interpolate (PS/composition.f90:174-177,
// 245-251).  src, itab and ctab are scratch here: stage 1 of the RK4
// rebuilds them.
int interpolate_T_at(Context& c, const int32_t* slots, int64_t n) {
  const int nx = c.T.nx, nz = c.T.nz;
  extend_t(c);
  dim3 b16(64, 4);
  hipLaunchKernelGGL(k_window3, grid2(nx + 7, nz + 7, b16), b16, 0, c.stream, c.Textend, c.src, nx, nz);
  PT_TRY(build_tables(c, c.src, c.src, c.src));
  InterpConst C;
  C.nx = nx; C.nz = nz; C.dr = c.T.dr; C.ds = c.T.ds; C.f3 = c.T.factorial[3];
  if (n > 0)
    hipLaunchKernelGGL(k_interp_slots, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, c.stream, c.ctab, C, slots, n,
                       c.r, c.s, c.Tt);
  return PT_OK;
}
// The projection that ends the redistribution: tracers_to_corners(rtr, str,
// Ttr, T) with smooth_vis=0 (PS/composition.f90:257-259); nodes without
// tracers keep the module T (the initial field before the first
// energy_time, Tratio after it).  The storage order then follows the new
// positions.
int equalize_projection(Context& c, bool moved) {
  const size_t b3 = sizeof(double) * (size_t)(c.T.nx + 7) * (c.T.nz + 7);
  if (!c.t_initial) PT_HIP(hipMemcpyAsync(c.T0, c.Tratio, b3, hipMemcpyDeviceToDevice, c.stream));
  if (moved) c.order_valid = false;
  PT_TRY(tracers_to_corners(c, c.r, c.s, c.Tt, false));
  return reorder_tracers(c);
}

// tracers (reference ID order) onto the device, projected onto the nodes, in cell order
static int place_tracers(Context& c, const double* rtr, const double* str, const double* Ttr, const double* Ctr) {
  size_t tb = sizeof(double) * (size_t)c.T.ntr;
  c.order_valid = false;
  c.window_skip = 0;
  PT_HIP(hipMemcpyAsync(c.r, rtr, tb, hipMemcpyHostToDevice, c.stream));
  PT_HIP(hipMemcpyAsync(c.s, str, tb, hipMemcpyHostToDevice, c.stream));
  PT_HIP(hipMemcpyAsync(c.Tt, Ttr, tb, hipMemcpyHostToDevice, c.stream));
  PT_HIP(hipMemcpyAsync(c.Ct, Ctr, tb, hipMemcpyHostToDevice, c.stream));
  PT_HIP(hipMemcpyAsync(c.tid, c.iota, sizeof(int32_t) * (size_t)c.T.ntr, hipMemcpyDeviceToDevice, c.stream));
  PT_TRY(tracers_to_corners(c, c.r, c.s, c.Tt));
  return reorder_tracers(c);
}

static int clear_coarse_errors(Context& c) {
  for (int l = 2; l <= c.T.grids; l++) {
    PT_HIP(hipMemsetAsync(c.L[l].err, 0, sizeof(double) * c.L[l].nelem, c.stream));
    if (c.L[l].ferr) PT_HIP(hipMemsetAsync(c.L[l].ferr, 0, sizeof(float) * c.L[l].nelem, c.stream));
  }
  return PT_OK;
}

// restart=1 start (PS/grid.f90:55-103, PS/main.f90:204-209, :226-229): T,
// Cnew and SF as print_restart wrote them (whole arrays with halos), the
// tracers in ID order.  T and Cnew are the values kept at nodes without
// tracers; the module T becomes the re-projected field.  The walls take
// Tbot/Ttop: the reference leaves Tbot_iso/Ttop_iso at 0 on this path.
int restart_state(Context& c, const double* T3, const double* C5, const double* SF3, double Tbot, double Ttop,
                  const double* rtr, const double* str, const double* Ttr, const double* Ctr) {
  const int nx = c.T.nx, nz = c.T.nz;
  c.Tbot_iso = Tbot; c.Ttop_iso = Ttop; c.time = 0.0; c.first_solve = true;
  c.t_initial = true; c.mass_set = false;
  const size_t b3 = sizeof(double) * (size_t)(nx + 7) * (nz + 7), b5 = sizeof(double) * (size_t)(nx + 11) * (nz + 11);
  PT_HIP(hipMemcpyAsync(c.T0, T3, b3, hipMemcpyHostToDevice, c.stream));
  hipLaunchKernelGGL(k_t_walls, dim3((nx + 7 + 255) / 256), dim3(256), 0, c.stream, c.T0, nx, nz, 3, nx + 7, 0, Tbot,
                     Ttop);
  t_bcs(c, c.T0);
  PT_HIP(hipMemcpyAsync(c.Cnew, C5, b5, hipMemcpyHostToDevice, c.stream));
  c_bcs(c, c.Cnew);
  PT_TRY(place_tracers(c, rtr, str, Ttr, Ctr));
  PT_HIP(hipMemcpyAsync(c.T0, c.Tratio, b3, hipMemcpyDeviceToDevice, c.stream));
  PT_HIP(hipMemcpyAsync(c.SF, SF3, b3, hipMemcpyHostToDevice, c.stream));
  if (c.P.iterate == 1) PT_TRY(stream_bcs(c, c.SF));   // PS/grid.f90:68
  PT_TRY(clear_coarse_errors(c));
  PT_HIP(hipStreamSynchronize(c.stream));
  return PT_OK;
}

int load_state(Context& c, const double* T_nodes, double Tbot, double Ttop, const double* rtr, const double* str,
               const double* Ttr, const double* Ctr) {
  const int nx = c.T.nx, nz = c.T.nz;
  c.Tbot_iso = Tbot; c.Ttop_iso = Ttop; c.time = 0.0; c.first_solve = true;
  c.t_initial = true; c.mass_set = false;
  size_t nb = sizeof(double) * (size_t)(nx + 1) * (nz + 1);
  double* dTn = c.src;   // staging (src is rebuilt every stage)
  PT_HIP(hipMemcpyAsync(dTn, T_nodes, nb, hipMemcpyHostToDevice, c.stream));
  PT_HIP(hipMemsetAsync(c.T0, 0, sizeof(double) * (size_t)(nx + 7) * (nz + 7), c.stream));
  dim3 b16(64, 4);
  hipLaunchKernelGGL(k_load_T, grid2(nx + 1, nz + 1, b16), b16, 0, c.stream, dTn, c.T0, nx, nz);
  hipLaunchKernelGGL(k_t_walls, dim3((nx + 7 + 255) / 256), dim3(256), 0, c.stream, c.T0, nx, nz, 3, nx + 7, 0, Tbot,
                     Ttop);
  t_bcs(c, c.T0);
  PT_HIP(hipMemsetAsync(c.Cnew, 0, sizeof(double) * (size_t)(nx + 11) * (nz + 11), c.stream));
  PT_TRY(place_tracers(c, rtr, str, Ttr, Ctr));
  PT_HIP(hipMemsetAsync(c.SF, 0, sizeof(double) * (size_t)(nx + 7) * (nz + 7), c.stream));
  PT_TRY(clear_coarse_errors(c));
  PT_HIP(hipStreamSynchronize(c.stream));
  return PT_OK;
}

// ---------------------------------------------------------------------------
static int dalloc(void** p, size_t bytes) {
  PT_HIP(hipMalloc(p, bytes));
  PT_HIP(hipMemset(*p, 0, bytes));
  return PT_OK;
}
#define DALLOC(ptr, bytes) PT_TRY(dalloc((void**)&(ptr), (bytes)))

__global__ void k_iota(int32_t* v, int64_t n) {
  int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (j < n) v[j] = (int32_t)j;
}

int tracers_alloc(Context& c) {
  const int nx = c.T.nx, nz = c.T.nz, ncell = (nx + 1) * (nz + 1);
  size_t b3 = sizeof(double) * (size_t)(nx + 7) * (nz + 7), b5 = sizeof(double) * (size_t)(nx + 11) * (nz + 11);
  double** f3[] = {&c.SF, &c.Tratio, &c.T0, &c.Tvis, &c.Tbuoy, &c.u, &c.w, &c.src, &c.cond_r, &c.cond_s};
  for (double** p : f3) DALLOC(*p, b3);
  double** f5[] = {&c.Cnew, &c.C0, &c.Cvis, &c.Cbuoy, &c.cond, &c.Textend, &c.TxS, &c.CxS};
  for (double** p : f5) DALLOC(*p, b5);
  DALLOC(c.itab, sizeof(double) * (size_t)(nx + 1) * (nz + 7) * 12);
  DALLOC(c.ctab, sizeof(double) * (size_t)(nx + 1) * (nz + 1) * 48);
  // D(1..3,-3..3) table for k_itab
  DALLOC(c.dtab, sizeof(double) * 21);
  double Dm[21];
  for (int m = 0; m < 3; m++)
    for (int q = 0; q < 7; q++) Dm[m * 7 + q] = c.T.D[m + 1][q];
  PT_HIP(hipMemcpy(c.dtab, Dm, sizeof Dm, hipMemcpyHostToDevice));
  size_t tb = sizeof(double) * (size_t)c.T.ntr;
  double** tr[] = {&c.r, &c.s, &c.Tt, &c.Ct, &c.r0, &c.s0, &c.T0t, &c.r1, &c.s1, &c.T1t, &c.r2, &c.s2, &c.T2t};
  for (double** p : tr) DALLOC(*p, tb);
  size_t ib = sizeof(int32_t) * (size_t)c.T.ntr;
  DALLOC(c.cellkey, ib); DALLOC(c.skey, ib); DALLOC(c.iota, ib); DALLOC(c.perm, ib);
  DALLOC(c.tid, ib); DALLOC(c.tid_tmp, ib);
  DALLOC(c.cstart, sizeof(int32_t) * ncell); DALLOC(c.cend, sizeof(int32_t) * ncell);
  DALLOC(c.okey, ib); DALLOC(c.ostart, sizeof(int32_t) * ncell); DALLOC(c.oend, sizeof(int32_t) * ncell);
  DALLOC(c.ccount, sizeof(int32_t) * ncell);
  DALLOC(c.bsum, sizeof(int32_t) * (size_t)((nx + 1 + CS_CELLS - 1) / CS_CELLS) * (nz + 1));
  DALLOC(c.nempty, sizeof(int32_t) * ncell);
  DALLOC(c.cellsum, sizeof(double) * 27 * (size_t)ncell);
  DALLOC(c.d_flags, sizeof(int32_t) * 4);
  DALLOC(c.d_fctl, sizeof(int32_t) * 4);
  size_t tiles = 0;
  for (int comp = 0; comp < 2; comp++) {
    c.filter[comp] = filter_plan(nx, nz, comp != 0);
    tiles = std::max(tiles, (size_t)filter_args(c, comp != 0).ntile);
  }
  DALLOC(c.d_fpart, sizeof(double) * FILTER_KMAX * 2 * tiles);
  DALLOC(c.d_fred, sizeof(double) * FILTER_KMAX);
  PT_HIP(hipHostMalloc((void**)&c.h_fctl, sizeof(int32_t) * 4, hipHostMallocDefault));
  hipLaunchKernelGGL(k_iota, dim3((unsigned)((c.T.ntr + 255) / 256)), dim3(256), 0, 0, c.iota, c.T.ntr);
  c.sort_bits = 1;
  while ((1 << c.sort_bits) <= ncell) c.sort_bits++;
  PT_TRY(sort_pairs_temp_bytes(c.T.ntr, c.sort_bits, &c.sort_bytes));
  DALLOC(c.sort_tmp, c.sort_bytes + 256);
  PT_HIP(hipDeviceSynchronize());
  return PT_OK;
}

int tracers_free(Context& c) {
  void* ps[] = {c.SF, c.Tratio, c.T0, c.Tvis, c.Tbuoy, c.u, c.w, c.src, c.cond_r, c.cond_s, c.Cnew, c.C0, c.Cvis,
                c.Cbuoy, c.cond, c.Textend, c.TxS, c.CxS, c.itab, c.ctab, c.dtab, c.r, c.s, c.Tt, c.Ct, c.r0, c.s0, c.T0t,
                c.r1, c.s1, c.T1t, c.r2, c.s2, c.T2t, c.cellkey, c.skey, c.iota, c.perm, c.tid, c.tid_tmp, c.cstart, c.cend,
                c.nempty, c.cellsum, c.d_flags, c.sort_tmp, c.d_fctl, c.d_fpart, c.d_fred, c.okey, c.ostart, c.oend, c.ccount,
                c.bsum};
  for (void* p : ps)
    if (p) (void)hipFree(p);
  if (c.h_fctl) (void)hipHostFree(c.h_fctl);
  equalize_free(c);
  return PT_OK;
}

}  // namespace pt
