// pm.hip -- the particle-grid steps either side of the PM solve, on the
// device: the cloud-in-cell deposit (Particles::cic, Particles.cxx:589-641)
// and its interpolation back to the particles (Particles::inverse_cic,
// Particles.cxx:645-714).
//
// Both follow the reference's arithmetic exactly: the weights ab, de, gh
// are 1.0 + (ix - x) with a float difference and a double sum stored as
// float; of the eight corner terms the first is a float product and the
// other seven are double from their first (1.0 - w) factor on, and each is
// added to its float accumulator in that precision.  That is the
// reference's own use of double (its literals 1.0 promote the arithmetic);
// compiled without FMA contraction.
//
// The deposit is a scatter whose result depends on the order of the float
// additions into each cell.  To reproduce the reference's sequential order
// in parallel it sorts the particles stably by base cell; a grid cell's
// contributions are then the merge, by particle index, of the particle
// lists of its eight neighbouring base cells.  A cell with at most 64 is
// merged and added by its own thread; a longer cell (dense clumps) by a
// workgroup, which forms its terms in merged order into LDS and adds them,
// 256 at a time, through exact fixed-grid maps of the float accumulation;
// the slot for corners outside the grid gets its contributions in
// (particle, corner) order and a workgroup.  The interpolation is a gather, one thread per
// particle.
#include "hsr_internal.h"

#include <hipcub/hipcub.hpp>

#include <algorithm>
#include <climits>

namespace {

inline unsigned nblk(int64_t n, int t) { return (unsigned)((n + t - 1) / t); }

// (int)floorf(x) as the reference's x86 build converts it: NaN and values
// outside the int range become INT_MIN (the conversion's indefinite value).
__device__ __forceinline__ int x86_floor_int(float x) {
  const float f = floorf(x);
  return (f >= -2147483648.0f && f < 2147483648.0f) ? (int)f : INT_MIN;
}

struct Grid {
  int ng0, ng1, ng2;
  uint32_t safe;  // ng0 * ng1 * ng2: the slot of corners outside the grid
};

// Particles.cxx:371-395 with lo = 0, hi = ng.
__device__ __forceinline__ uint32_t cell_of(int ix, int iy, int iz, const Grid &g) {
  if (ix >= 0 && ix < g.ng0 && iy >= 0 && iy < g.ng1 && iz >= 0 && iz < g.ng2)
    return ((uint32_t)ix * (uint32_t)g.ng1 + (uint32_t)iy) * (uint32_t)g.ng2 + (uint32_t)iz;
  return g.safe;
}

struct Corners {
  uint32_t cell[8];
  float ab, de, gh;
};

// Particles.cxx:617-640: corners in the reference's order.
__device__ __forceinline__ Corners corners(float xx, float yy, float zz, const Grid &g) {
  Corners c;
  const int ix = x86_floor_int(xx), iy = x86_floor_int(yy), iz = x86_floor_int(zz);
  const int ip = ix + 1, jp = iy + 1, kp = iz + 1;
  c.ab = (float)(1.0 + (double)((float)ix - xx));
  c.de = (float)(1.0 + (double)((float)iy - yy));
  c.gh = (float)(1.0 + (double)((float)iz - zz));
  c.cell[0] = cell_of(ix, iy, iz, g);
  c.cell[1] = cell_of(ix, jp, iz, g);
  c.cell[2] = cell_of(ix, jp, kp, g);
  c.cell[3] = cell_of(ix, iy, kp, g);
  c.cell[4] = cell_of(ip, iy, kp, g);
  c.cell[5] = cell_of(ip, jp, kp, g);
  c.cell[6] = cell_of(ip, jp, iz, g);
  c.cell[7] = cell_of(ip, iy, iz, g);
  return c;
}

// Corner q's term with lead factor s, evaluated as the reference's
// expression is: float products until the first (1.0 - w), double after.
__device__ __forceinline__ double corner_term(int q, float s, float ab, float de, float gh) {
  switch (q) {
  case 0: return (double)(s * ab * de * gh);
  case 1: return (double)(s * ab) * (1.0 - (double)de) * (double)gh;
  case 2: return (double)(s * ab) * (1.0 - (double)de) * (1.0 - (double)gh);
  case 3: return (double)(s * ab * de) * (1.0 - (double)gh);
  case 4: return (double)s * (1.0 - (double)ab) * (double)de * (1.0 - (double)gh);
  case 5: return (double)s * (1.0 - (double)ab) * (1.0 - (double)de) * (1.0 - (double)gh);
  case 6: return (double)s * (1.0 - (double)ab) * (1.0 - (double)de) * (double)gh;
  default: return (double)s * (1.0 - (double)ab) * (double)de * (double)gh;
  }
}

// The reference's accumulation step for one contribution
// (Particles.cxx:632-639): corner 0 adds a float term in float, the others
// add a double term and round to float.  The float addition r + t equals
// (float)((double)r + t) for float r and t (double rounding through a
// format of at least 2 * 24 + 2 bits is innocuous for a sum), so every
// corner takes the one form below.
__device__ __forceinline__ float cic_add(float r, double t) {
  return (float)((double)r + t);
}

__device__ __forceinline__ double readlane_f64(double v, int i) {
  const int lo = __builtin_amdgcn_readlane(__double2loint(v), i);
  const int hi = __builtin_amdgcn_readlane(__double2hiint(v), i);
  return __hiloint2double(hi, lo);
}

// Fixed-grid maps of the accumulation r <- (float)((double)r + t), t >= 0.
// While r stays in one binade [2^E, 2^(E+1)) (E >= -125) it is R u with
// u = 2^(E-23) and R an integer below 2^24, and one step is R <- R + D where
// D depends on t and on the parity of R alone: the double sum rounds to the
// grid u 2^-29 (its ulp in that binade, ties to even independent of R), the
// float to the grid u with ties to the even significand.  Maps (d0, d1) =
// (D for even R, D for odd R) compose associatively, so a wave scans the
// maps of 64 terms and applies the longest prefix that stays in the binade;
// the term that leaves it is added directly.  Totals past 2^26 saturate
// (they leave the binade anyway).
struct PMap {
  int d0, d1;
};
constexpr int PMAP_SAT = 1 << 26;

// a, then b.  Both are in [0, PMAP_SAT]: their sum fits an int and
// saturates with either.
__device__ __forceinline__ PMap pmap_compose(PMap a, PMap b) {
  PMap m;
  m.d0 = min(a.d0 + ((a.d0 & 1) ? b.d1 : b.d0), PMAP_SAT);
  m.d1 = min(a.d1 + ((a.d1 & 1) ? b.d0 : b.d1), PMAP_SAT);
  return m;
}

template <int CTRL, int ROWS>
__device__ __forceinline__ PMap pmap_dpp_step(PMap mp) {
  PMap pv;  // lanes without a source, and rows left out, get the identity
  pv.d0 = __builtin_amdgcn_update_dpp(0, mp.d0, CTRL, ROWS, 0xf, false);
  pv.d1 = __builtin_amdgcn_update_dpp(0, mp.d1, CTRL, ROWS, 0xf, false);
  return pmap_compose(pv, mp);
}

// Inclusive scan over a wave's lanes, all of them active: shifts within rows
// of 16, then the rows' totals passed on (lane moves in the vector pipe
// instead of 12 LDS permutes in a dependent chain).
__device__ __forceinline__ PMap pmap_scan(PMap mp) {
  mp = pmap_dpp_step<0x111, 0xf>(mp);  // row_shr 1, 2, 4, 8
  mp = pmap_dpp_step<0x112, 0xf>(mp);
  mp = pmap_dpp_step<0x114, 0xf>(mp);
  mp = pmap_dpp_step<0x118, 0xf>(mp);
  mp = pmap_dpp_step<0x142, 0xa>(mp);  // row_bcast 15 into rows 1 and 3
  return pmap_dpp_step<0x143, 0xc>(mp);  // row_bcast 31 into rows 2 and 3
}

__device__ __forceinline__ PMap pmap_term(double t, int E) {
  PMap m;
  const double q = ldexp(t, 23 - E);                 // t / u, exact
  if (!(q < 16777216.0)) {
    m.d0 = m.d1 = PMAP_SAT;
    return m;
  }
  const double qq = ldexp(rint(ldexp(q, 29)), -29);  // the double sum's rounding
  const double a = floor(qq), f = qq - a;
  const int ai = (int)a;
  const int up = f > 0.5 ? 1 : 0;
  const bool tie = f == 0.5;
  m.d0 = ai + up + ((tie && (ai & 1)) ? 1 : 0);
  m.d1 = ai + up + ((tie && !(ai & 1)) ? 1 : 0);
  return m;
}

// One wave adds 64 LT terms of a cell's contributions in order: lane l
// holds terms LT l .. LT l + LT - 1, the first cnt of the step live.  With
// all terms nonnegative (the deposit's weights are) it applies them by the
// map scan above -- each lane composes its LT terms in order, then the
// lanes' maps are scanned -- and applies the longest prefix that stays in
// the binade; in the lane where the sum leaves it the terms are stepped one
// at a time to the crossing term, which is added directly.  Otherwise the
// terms are added in order, reading them with v_readlane.  r is the same in
// every lane.
constexpr int LT = 4;
constexpr int WAVE_HEAD = 32;

__device__ __forceinline__ double pick(const double (&t)[LT], int k) {
  return k == 0 ? t[0] : k == 1 ? t[1] : k == 2 ? t[2] : t[3];
}

// HEAD: the sum starts here, and its first terms, where it leaves a binade
// every few of them, are added directly (a pass of the scan costs about as
// much as 32 additions).
template <bool HEAD>
__device__ __forceinline__ float wave_add_step(float r, const double (&t)[LT], int cnt) {
  static_assert(LT == 4, "pick() reads four terms per lane");
  const int l = threadIdx.x & 63;
  bool neg = false;
#pragma unroll
  for (int k = 0; k < LT; ++k) {
    const int i = LT * l + k;
    neg = neg || (i < cnt && !(t[k] >= 0.0));
  }
  if (__ballot(neg) != 0ull) {
    for (int i = 0; i < cnt; ++i) r = cic_add(r, readlane_f64(pick(t, i % LT), i / LT));
    return r;
  }
  int s = 0;
  if constexpr (HEAD) {
#pragma unroll
    for (int i = 0; i < WAVE_HEAD; ++i) r = cic_add(r, readlane_f64(t[i % LT], i / LT));  // zeros past cnt
    s = WAVE_HEAD;
  }
  while (s < cnt) {
    if (!(r >= 0x1p-125f)) {  // zero or subnormal: the double sum's grid varies
      r = cic_add(r, readlane_f64(pick(t, s % LT), s / LT));
      ++s;
      continue;
    }
    const int E = ilogbf(r);
    const double u = ldexp(1.0, E - 23);
    const int R = (int)((double)r / u);
    PMap mp = PMap{0, 0};
#pragma unroll
    for (int k = 0; k < LT; ++k) {
      const int i = LT * l + k;
      if (i >= s && i < cnt) mp = pmap_compose(mp, pmap_term(t[k], E));
    }
    mp = pmap_scan(mp);
    const int d = (R & 1) ? mp.d1 : mp.d0;
    const int Rl = d >= PMAP_SAT ? PMAP_SAT : R + d;
    // R only grows: the lanes past the crossing one cross too
    const unsigned long long cross = __ballot(Rl >= (1 << 24));
    if (!cross) {
      r = (float)((double)__shfl(Rl, 63) * u);
      s = cnt;
      continue;
    }
    const int j = __ffsll((long long)cross) - 1;
    // the lanes before j applied, then lane j's terms one at a time
    int Rj = j > 0 ? __shfl(Rl, j - 1) : R;
    for (int k = 0; k < LT; ++k) {  // uniform
      const int i = LT * j + k;
      if (i < s || i >= cnt) continue;
      const double tk = readlane_f64(pick(t, k), j);
      const PMap m1 = pmap_term(tk, E);
      const int dk = (Rj & 1) ? m1.d1 : m1.d0;
      if (dk >= PMAP_SAT || Rj + dk >= (1 << 24)) {  // the crossing term
        r = cic_add((float)((double)Rj * u), tk);
        s = i + 1;
        break;
      }
      Rj += dk;
    }
  }
  return r;
}

constexpr int TAIL_THREADS = 1024;

// The outside slot's terms [0, m) by one workgroup: LT TAIL_THREADS terms per step, LT
// per thread composed in order, maps scanned within each wave and across
// the 16 waves through LDS, the longest prefix that stays in the binade
// applied; the thread holding the crossing term steps its terms to it and
// adds it directly.
__global__ void __launch_bounds__(TAIL_THREADS)
k_cic_tail(int64_t m, const uint32_t *__restrict__ key, const double *__restrict__ ts,
           float *__restrict__ rho) {
  __shared__ PMap wtot[TAIL_THREADS / 64];
  __shared__ float r_sh;
  __shared__ int j_sh, neg_sh, s_sh, rj_sh;
  const int64_t p0 = 0;
  const int tid = threadIdx.x, l = tid & 63, w = tid >> 6;
  if (tid == 0) r_sh = 0.f;
  __syncthreads();
  for (int64_t base = p0; base < m; base += LT * TAIL_THREADS) {
    const int cnt = (int)min<int64_t>(LT * TAIL_THREADS, m - base);
    double t[LT];
    bool neg = false;
#pragma unroll
    for (int k = 0; k < LT; ++k) {
      const int i = LT * tid + k;
      t[k] = i < cnt ? ts[base + i] : 0.0;
      neg = neg || (i < cnt && !(t[k] >= 0.0));
    }
    if (tid == 0) neg_sh = 0;
    __syncthreads();
    if (neg) neg_sh = 1;
    __syncthreads();
    if (neg_sh) {
      if (tid == 0) {
        float r = r_sh;
        for (int i = 0; i < cnt; ++i) r = cic_add(r, ts[base + i]);
        r_sh = r;
      }
      __syncthreads();
      continue;
    }
    int s = 0;
    while (s < cnt) {
      const float r = r_sh;
      if (!(r >= 0x1p-125f)) {
        __syncthreads();
        if (tid == 0) r_sh = cic_add(r, ts[base + s]);
        __syncthreads();
        ++s;
        continue;
      }
      const int E = ilogbf(r);
      const double u = ldexp(1.0, E - 23);
      const int R = (int)((double)r / u);
      PMap mp = PMap{0, 0};
#pragma unroll
      for (int k = 0; k < LT; ++k) {
        const int i = LT * tid + k;
        if (i >= s && i < cnt) mp = pmap_compose(mp, pmap_term(t[k], E));
      }
      mp = pmap_scan(mp);
      if (l == 63) wtot[w] = mp;
      if (tid == 0) j_sh = TAIL_THREADS;
      __syncthreads();
      if (w == 0) {  // exclusive prefix of the wave totals, in wave order
        PMap tv = l < TAIL_THREADS / 64 ? wtot[l] : PMap{0, 0};
#pragma unroll
        for (int off = 1; off < TAIL_THREADS / 64; off <<= 1) {
          PMap pv;
          pv.d0 = __shfl_up(tv.d0, off);
          pv.d1 = __shfl_up(tv.d1, off);
          if (l >= off) tv = pmap_compose(pv, tv);
        }
        PMap ex;
        ex.d0 = __shfl_up(tv.d0, 1);
        ex.d1 = __shfl_up(tv.d1, 1);
        if (l == 0) ex = PMap{0, 0};
        if (l < TAIL_THREADS / 64) wtot[l] = ex;
      }
      __syncthreads();
      const PMap ex = wtot[w];  // the waves before this one
      const PMap inc = pmap_compose(ex, mp);
      const int d = (R & 1) ? inc.d1 : inc.d0;
      const int Rl = d >= PMAP_SAT ? PMAP_SAT : R + d;
      // R only grows: the threads past the crossing one cross too
      if (Rl >= (1 << 24)) atomicMin(&j_sh, tid);
      __syncthreads();
      const int j = j_sh;
      if (j == TAIL_THREADS) {  // no crossing: all applied
        if (tid == TAIL_THREADS - 1) r_sh = (float)((double)Rl * u);
        s = cnt;
        __syncthreads();
        continue;
      }
      // the threads before j applied: R after them is thread j - 1's
      // inclusive value; then thread j steps its own terms to the crossing
      if (tid == j - 1) rj_sh = Rl;
      if (j == 0 && tid == 0) rj_sh = R;
      __syncthreads();
      if (tid == j) {
        int Rj = rj_sh;
        for (int k = 0; k < LT; ++k) {
          const int i = LT * tid + k;
          if (i < s || i >= cnt) continue;
          const PMap m1 = pmap_term(t[k], E);
          const int dk = (Rj & 1) ? m1.d1 : m1.d0;
          if (dk >= PMAP_SAT || Rj + dk >= (1 << 24)) {  // the crossing term
            r_sh = cic_add((float)((double)Rj * u), t[k]);
            s_sh = i + 1;
            break;
          }
          Rj += dk;
        }
      }
      __syncthreads();
      s = s_sh;
      __syncthreads();
    }
  }
  if (tid == 0) rho[key[p0]] = r_sh;
}

// ------------------------------------------------- deposit by base cells
// A particle with floor coordinates (ix, iy, iz) deposits into the cells
// (ix, iy, iz) + d_q for its eight corners q (corners()), so a grid cell c
// receives, from each q, the particles whose base cell is c - d_q.  With
// the particles sorted stably by base cell, each such list is in particle
// order, and c's contributions in the reference's order (particle by
// particle; one particle reaches c through one corner at most) are the
// merge of its eight lists by particle index.  Base cells run over
// [-1, ng - 1] per axis (an extended grid, shifted by one); a particle
// outside it has all its corners outside the grid.  Corners outside the
// grid go to the outside slot, in (particle, corner) order.

// corner offsets d_q in corners()' order
__constant__ int kCornerDx[8] = {0, 0, 0, 0, 1, 1, 1, 1};
__constant__ int kCornerDy[8] = {0, 1, 1, 0, 0, 1, 1, 0};
__constant__ int kCornerDz[8] = {0, 0, 1, 1, 1, 1, 0, 0};

struct Ext {
  uint32_t e1, e2;  // extended sizes ng1 + 1, ng2 + 1 (ng0 + 1 along x)
  uint32_t out;     // (ng0 + 1)(ng1 + 1)(ng2 + 1): the key of particles outside
};

// The weights of corners() alone.
__device__ __forceinline__ void weights(float xx, float yy, float zz, float &ab, float &de,
                                        float &gh) {
  const int ix = x86_floor_int(xx), iy = x86_floor_int(yy), iz = x86_floor_int(zz);
  ab = (float)(1.0 + (double)((float)ix - xx));
  de = (float)(1.0 + (double)((float)iy - yy));
  gh = (float)(1.0 + (double)((float)iz - zz));
}

// Per particle: its extended base-cell key, its index (the sort's value) and
// the number of its corners outside the grid.
__global__ void __launch_bounds__(256)
k_cic_base(int64_t n, const float *__restrict__ x, const float *__restrict__ y,
           const float *__restrict__ z, Grid g, Ext ex, uint32_t *__restrict__ key,
           int32_t *__restrict__ idx, int32_t *__restrict__ nout, int32_t *__restrict__ unsorted) {
  const int64_t nn = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (nn >= n) return;
  auto base_key = [&](float xx, float yy, float zz) {
    const int ix = x86_floor_int(xx), iy = x86_floor_int(yy), iz = x86_floor_int(zz);
    const bool in = ix >= -1 && ix < g.ng0 && iy >= -1 && iy < g.ng1 && iz >= -1 && iz < g.ng2;
    return in ? (((uint32_t)(ix + 1) * ex.e1 + (uint32_t)(iy + 1)) * ex.e2 + (uint32_t)(iz + 1)) : ex.out;
  };
  const float xx = x[nn], yy = y[nn], zz = z[nn];
  const Corners cc = corners(xx, yy, zz, g);
  int no = 0;
#pragma unroll
  for (int q = 0; q < 8; ++q) no += cc.cell[q] == g.safe;
  const uint32_t k = base_key(xx, yy, zz);
  // whether the keys are in order already: the lane before's, or for a
  // wave's first lane the particle before's
  uint32_t prev = (uint32_t)__shfl_up((int)k, 1);
  if ((threadIdx.x & 63) == 0) prev = nn > 0 ? base_key(x[nn - 1], y[nn - 1], z[nn - 1]) : 0u;
  if (prev > k) unsorted[0] = 1;  // every writer stores the same value
  key[nn] = k;
  idx[nn] = (int32_t)nn;
  nout[nn] = no;
}

// [beg, end) of every base cell in the sorted order (left 0 when empty).
__global__ void __launch_bounds__(256)
k_cic_ranges(int64_t n, const uint32_t *__restrict__ key, Ext ex, int32_t *__restrict__ beg,
             int32_t *__restrict__ end) {
  const int64_t p = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (p >= n) return;
  const uint32_t k = key[p];
  if (k == ex.out) return;
  if (p == 0 || key[p - 1] != k) beg[k] = (int32_t)p;
  if (p == n - 1 || key[p + 1] != k) end[k] = (int32_t)(p + 1);
}

constexpr int CELL_SHORT = 64;  // contributions a cell's own thread merges and adds

// The eight source lists of grid cell c = (i, j, k).
__device__ __forceinline__ void cell_lists(int i, int j, int k, const Ext &ex,
                                           const int32_t *beg, const int32_t *end,
                                           int32_t (&s)[8], int32_t (&e)[8]) {
#pragma unroll
  for (int q = 0; q < 8; ++q) {
    const uint32_t b = ((uint32_t)(i - kCornerDx[q] + 1) * ex.e1 + (uint32_t)(j - kCornerDy[q] + 1)) * ex.e2 +
                       (uint32_t)(k - kCornerDz[q] + 1);
    s[q] = beg[b];
    e[q] = end[b];
  }
}

// The next contribution of the merge: the list whose head particle comes
// first (lists never share a particle).
__device__ __forceinline__ int merge_pick(const int32_t (&hv)[8]) {
  int qs = 0;
  int32_t best = hv[0];
#pragma unroll
  for (int q = 1; q < 8; ++q)
    if (hv[q] < best) {
      best = hv[q];
      qs = q;
    }
  return qs;
}

__device__ __forceinline__ void merge_advance(int qs, int32_t (&s)[8], const int32_t (&e)[8],
                                              int32_t (&hv)[8], const int32_t *idx) {
#pragma unroll
  for (int q = 0; q < 8; ++q)
    if (q == qs) {
      ++s[q];
      hv[q] = s[q] < e[q] ? idx[s[q]] : INT_MAX;
    }
}

// What the host reads, in one copy: the outside slot's contributions, and
// whether the keys are out of order.
__global__ void k_cic_totals(const int32_t *out_last, const int32_t *nout_last, const int32_t *unsorted,
                             int64_t *totals) {
  if (threadIdx.x == 0) {
    totals[0] = (int64_t)*out_last + *nout_last;
    totals[1] = *unsorted;
  }
}

// The corners in the order of their base cells' keys, for any cell: with the
// particles in base-cell order (k_cic_base) a cell's contributions are its
// eight lists one after another in this order.
constexpr int kCornerByKey[8] = {5, 6, 4, 7, 2, 1, 3, 0};
__constant__ int kCornerByKeyDev[8] = {5, 6, 4, 7, 2, 1, 3, 0};

// One thread per grid cell: at most CELL_SHORT contributions are merged and
// added here; longer cells are queued with their counts for k_cic_long_sum.
// INORDER: the particles are in base-cell order, so that nothing is merged
// and a list's particles are read where they lie, not through the order
// (18M clustered particles at 256^3: 0.84 ms merged,
// 0.50).  CELL_SHORT 128, 256 and 512 here gave the deposit 0, 1 and 4% more.
template <bool INORDER>
__global__ void __launch_bounds__(256)
k_cic_cells(Grid g, Ext ex, const int32_t *__restrict__ beg, const int32_t *__restrict__ end,
            const int32_t *__restrict__ idx, const float *__restrict__ x,
            const float *__restrict__ y, const float *__restrict__ z, float c,
            float *__restrict__ rho, uint32_t *__restrict__ long_cell,
            int64_t *__restrict__ long_k, unsigned long long *__restrict__ nlong) {
  const int64_t cid = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (cid >= (int64_t)g.safe) return;
  const int k = (int)(cid % g.ng2);
  const int64_t ij = cid / g.ng2;
  const int j = (int)(ij % g.ng1), i = (int)(ij / g.ng1);
  int32_t s[8], e[8];
  cell_lists(i, j, k, ex, beg, end, s, e);
  int K = 0;
#pragma unroll
  for (int q = 0; q < 8; ++q) K += e[q] - s[q];
  if (K == 0) return;
  if (K > CELL_SHORT) {
    const unsigned long long slot = atomicAdd(nlong, 1ull);
    long_cell[slot] = (uint32_t)cid;
    long_k[slot] = K;
    return;
  }
  float r = 0.f;
  if constexpr (INORDER) {
#pragma unroll
    for (int o = 0; o < 8; ++o) {
      const int q = kCornerByKey[o];
      for (int32_t nn = s[q]; nn < e[q]; ++nn) {
        float ab, de, gh;
        weights(x[nn], y[nn], z[nn], ab, de, gh);
        r = cic_add(r, corner_term(q, c, ab, de, gh));
      }
    }
    rho[cid] = r;
    return;
  }
  int32_t hv[8];
#pragma unroll
  for (int q = 0; q < 8; ++q) hv[q] = s[q] < e[q] ? idx[s[q]] : INT_MAX;
  for (int t = 0; t < K; ++t) {
    const int qs = merge_pick(hv);
    const int32_t nn = hv[qs];
    float ab, de, gh;
    weights(x[nn], y[nn], z[nn], ab, de, gh);
    r = cic_add(r, corner_term(qs, c, ab, de, gh));
    merge_advance(qs, s, e, hv, idx);
  }
  rho[cid] = r;
}

// One wave per long cell: its contributions' terms formed in merged order
// into LDS, LC_CHUNK at a time, and added in order (wave_add_step).  When
// the eight lists hold disjoint index ranges -- the particles of a base
// cell are contiguous when the input is in cell order, as the resort leaves
// it -- the merge is the lists in the order of their first particles, and
// all lanes form the terms; otherwise a window of each list is merged by
// counting (18M clustered particles with 1% of them out of order: 34.9 ms a
// deposit with a merge by lane 0, 6.6).  A wave per workgroup
// keeps many cells' latency-bound sums in flight on each CU.  INORDER: as in
// k_cic_cells, the lists follow each other in kCornerByKey's order, and each
// lane forms its own terms, without LDS.  18M clustered particles at 256^3
// (73,000 long cells, 70M contributions, the longest cell 33,600): 1.91 ms
// merged with lane 0's setup and the scan by LDS permutes, 1.48 with the
// lists in order, 0.98 with the scan by lane moves, the first terms added
// directly and the next particles' loads in flight.
constexpr int LC_CHUNK = 2 * 64 * LT;

template <bool INORDER>
__global__ void __launch_bounds__(64)
k_cic_long_sum(Grid g, Ext ex, const int32_t *__restrict__ beg, const int32_t *__restrict__ end,
               const int32_t *__restrict__ idx, const uint32_t *__restrict__ long_cell,
               const int64_t *__restrict__ long_k, const unsigned long long *__restrict__ nlong,
               const float *__restrict__ x, const float *__restrict__ y, const float *__restrict__ z,
               float c, float *__restrict__ rho) {
  __shared__ double tb[LC_CHUNK];
  __shared__ int32_t ss[8], se[8], soff[8];
  __shared__ int32_t win[INORDER ? 1 : 8][64];
  __shared__ int disjoint;
  const int tid = threadIdx.x;
  const int64_t nl = (int64_t)*nlong;
  for (int64_t t = blockIdx.x; t < nl; t += gridDim.x) {
    const uint32_t cid = long_cell[t];
    const int64_t K = long_k[t];
    int32_t s[8], e[8];  // the merge's state, the same in every lane
    if constexpr (INORDER) {
      if (tid < 8) {
        const int q = kCornerByKeyDev[tid];
        const int k = (int)(cid % (uint32_t)g.ng2);
        const uint32_t ij = cid / (uint32_t)g.ng2;
        const int j = (int)(ij % (uint32_t)g.ng1), i = (int)(ij / (uint32_t)g.ng1);
        const uint32_t b = ((uint32_t)(i - kCornerDx[q] + 1) * ex.e1 + (uint32_t)(j - kCornerDy[q] + 1)) * ex.e2 +
                           (uint32_t)(k - kCornerDz[q] + 1);
        const int32_t sb = beg[b], len = end[b] - sb;
        int32_t off = len;
#pragma unroll
        for (int d = 1; d < 8; d <<= 1) {
          const int32_t o = __shfl_up(off, d);
          if (tid >= d) off += o;
        }
        ss[q] = sb;
        se[q] = sb + len;
        soff[q] = off - len;
      }
    } else if (tid == 0) {
      const int k = (int)(cid % (uint32_t)g.ng2);
      const uint32_t ij = cid / (uint32_t)g.ng2;
      const int j = (int)(ij % (uint32_t)g.ng1), i = (int)(ij / (uint32_t)g.ng1);
      cell_lists(i, j, k, ex, beg, end, s, e);
      // each non-empty list's first and last particle; the lists ordered by
      // their first (a selection sort of eight)
      int32_t first[8], last[8], ord[8];
      int nq = 0;
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        ss[q] = s[q];
        se[q] = e[q];
        soff[q] = 0;
        first[q] = s[q] < e[q] ? idx[s[q]] : INT_MAX;
        last[q] = s[q] < e[q] ? idx[e[q] - 1] : INT_MAX;
      }
      for (int q = 0; q < 8; ++q)
        if (s[q] < e[q]) ord[nq++] = q;
      for (int a2 = 0; a2 < nq; ++a2)
        for (int b2 = a2 + 1; b2 < nq; ++b2)
          if (first[ord[b2]] < first[ord[a2]]) {
            const int tq = ord[a2];
            ord[a2] = ord[b2];
            ord[b2] = tq;
          }
      int dj = 1, off = 0;
      for (int a2 = 0; a2 < nq; ++a2) {
        const int q = ord[a2];
        if (a2 + 1 < nq && !(last[q] < first[ord[a2 + 1]])) dj = 0;
        soff[q] = off;
        off += e[q] - s[q];
      }
      disjoint = dj;
    }
    __syncthreads();
    if constexpr (!INORDER) {
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        s[q] = ss[q];
        e[q] = se[q];
      }
    }
    float r = 0.f;
    if constexpr (INORDER) {
      // a lane's terms straight from the lists; the next step's particles
      // are on their way while this one's terms are added
      float px[LT], py[LT], pz[LT];
      int pq[LT];
      auto fetch = [&](int64_t c0) {
#pragma unroll
        for (int k = 0; k < LT; ++k) {
          const int64_t pos = c0 + LT * tid + k;
          int q = -1;
          int32_t nn = 0;
#pragma unroll
          for (int qq = 0; qq < 8; ++qq) {
            const int64_t at = pos - soff[qq];
            if (at >= 0 && at < se[qq] - ss[qq]) {
              q = qq;
              nn = ss[qq] + (int32_t)at;
            }
          }
          pq[k] = q;  // -1 past the last
          px[k] = x[nn];
          py[k] = y[nn];
          pz[k] = z[nn];
        }
      };
      fetch(0);
      for (int64_t c0 = 0; c0 < K; c0 += 64 * LT) {
        const int cnt = (int)min<int64_t>(64 * LT, K - c0);
        double tt[LT];
#pragma unroll
        for (int k = 0; k < LT; ++k) {
          float ab, de, gh;
          weights(px[k], py[k], pz[k], ab, de, gh);
          tt[k] = pq[k] >= 0 ? corner_term(pq[k], c, ab, de, gh) : 0.0;
        }
        if (c0 + 64 * LT < K) fetch(c0 + 64 * LT);
        r = c0 == 0 ? wave_add_step<true>(r, tt, cnt) : wave_add_step<false>(r, tt, cnt);
      }
      if (tid == 0) rho[cid] = r;
      __syncthreads();  // the lists are rewritten for the next cell
      continue;
    }
    for (int64_t c0 = 0; c0 < K;) {
      int cl = (int)min<int64_t>(LC_CHUNK, K - c0);
      if (disjoint) {
        for (int u = tid; u < cl; u += blockDim.x) {
          const int pos = (int)c0 + u;
          // the list whose merged range holds pos (the ranges tile [0, K))
          int q = -1;
#pragma unroll
          for (int qq = 0; qq < 8; ++qq)
            if (pos >= soff[qq] && pos < soff[qq] + (se[qq] - ss[qq])) q = qq;
          double term = 0.0;
          if (q >= 0) {
            const int32_t nn = idx[ss[q] + (pos - soff[q])];
            float ab, de, gh;
            weights(x[nn], y[nn], z[nn], ab, de, gh);
            term = corner_term(q, c, ab, de, gh);
          }
          tb[u] = term;
        }
      } else {
        // each list's next 64 particles; those up to the least last one of
        // the windows that their lists go on past are the next of the merge
        // (at least 64 then, else all that are left), a particle's place
        // the count of smaller ones in every window
        int32_t v[8], bound = INT_MAX;
#pragma unroll
        for (int q = 0; q < 8; ++q) {
          v[q] = s[q] + tid < e[q] ? idx[s[q] + tid] : INT_MAX;
          win[q][tid] = v[q];
          if (e[q] - s[q] > 64) bound = min(bound, __builtin_amdgcn_readlane(v[q], 63));
        }
        __syncthreads();
        cl = 0;
#pragma unroll
        for (int q = 0; q < 8; ++q) {
          const bool live = v[q] <= bound && s[q] + tid < e[q];
          if (live) {
            int pos = tid;  // a list's particles ascend
            for (int p = 0; p < 8; ++p) {
              if (p == q || win[p][0] == INT_MAX) continue;
              int lo = 0;
#pragma unroll
              for (int d = 32; d > 0; d >>= 1)
                if (win[p][lo + d - 1] < v[q]) lo += d;
              pos += lo + (win[p][lo] < v[q] ? 1 : 0);
            }
            float ab, de, gh;
            weights(x[v[q]], y[v[q]], z[v[q]], ab, de, gh);
            tb[pos] = corner_term(q, c, ab, de, gh);
          }
          const int taken = __popcll(__ballot(live));
          s[q] += taken;
          cl += taken;
        }
      }
      __syncthreads();
      {
        for (int b = 0; b < cl; b += 64 * LT) {
          const int cnt = min(64 * LT, cl - b);
          double tt[LT];
#pragma unroll
          for (int k = 0; k < LT; ++k) {
            const int i = LT * tid + k;
            tt[k] = i < cnt ? tb[b + i] : 0.0;
          }
          r = c0 + b == 0 ? wave_add_step<true>(r, tt, cnt) : wave_add_step<false>(r, tt, cnt);
        }
      }
      c0 += cl;
      __syncthreads();  // tb and the windows are rewritten by the next chunk
    }
    if (tid == 0) rho[cid] = r;
  }
}

// The outside slot's contributions in (particle, corner) order, from
// position base (out_base: exclusive prefix of the particles' counts).
__global__ void __launch_bounds__(256)
k_cic_out_terms(int64_t n, const float *__restrict__ x, const float *__restrict__ y,
                const float *__restrict__ z, Grid g, float c, const int32_t *__restrict__ nout,
                const int32_t *__restrict__ out_base, int64_t base, uint32_t *__restrict__ skey,
                double *__restrict__ ts) {
  const int64_t nn = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (nn >= n || nout[nn] == 0) return;
  const Corners cc = corners(x[nn], y[nn], z[nn], g);
  int64_t p = base + out_base[nn];
#pragma unroll
  for (int q = 0; q < 8; ++q)
    if (cc.cell[q] == g.safe) {
      skey[p] = g.safe;
      ts[p] = corner_term(q, c, cc.ab, cc.de, cc.gh);
      ++p;
    }
}


// Particles.cxx:682-711, one component: f accumulated as the deposit's runs
// are (grid[safe] read as 0), then v += f * fscal * tau in float.
__global__ void __launch_bounds__(256)
k_inverse_cic(int64_t n, const float *__restrict__ x, const float *__restrict__ y,
              const float *__restrict__ z, Grid g, const float *__restrict__ grid,
              float tau, float fscal, float *__restrict__ v) {
  const int64_t nn = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (nn >= n) return;
  const Corners cc = corners(x[nn], y[nn], z[nn], g);
  float f = 0.f;
#pragma unroll
  for (int q = 0; q < 8; ++q) {
    const float s = cc.cell[q] == g.safe ? 0.f : grid[cc.cell[q]];
    const double t = corner_term(q, s, cc.ab, cc.de, cc.gh);
    if (q == 0) f = f + (float)t;
    else f = (float)((double)f + t);
  }
  v[nn] = v[nn] + f * fscal * tau;
}

__global__ void k_zero_u64(unsigned long long *p) {
  if (threadIdx.x == 0) p[0] = 0ull;
}

__global__ void k_fill0(int64_t n, float *a) {
  const int64_t k = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (k < n) a[k] = 0.f;
}

Grid make_grid(const int32_t ng[3]) {
  Grid g;
  g.ng0 = ng[0];
  g.ng1 = ng[1];
  g.ng2 = ng[2];
  g.safe = (uint32_t)((uint64_t)ng[0] * ng[1] * ng[2]);
  return g;
}

}  // namespace

namespace {

__global__ void k_fill_i32(int64_t n, int32_t *a) {
  const int64_t k = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (k < n) a[k] = 0;
}

template <class T>
hsr_status pm_excl_scan(hsr_ctx *c, const T *in, T *out, int64_t n) {
  size_t tmp = 0;
  HSR_HIP(hipcub::DeviceScan::ExclusiveSum(nullptr, tmp, in, out, (int)n, c->stream));
  HSR_HIP(dbuf_reserve(c->s.cub, tmp + 256));
  HSR_HIP(hipcub::DeviceScan::ExclusiveSum(c->s.cub.p, tmp, in, out, (int)n, c->stream));
  return HSR_OK;
}

}  // namespace

hsr_status cic_run(hsr_ctx *c, int64_t n, const float *x, const float *y, const float *z,
                   const int32_t ng[3], float gpscal, float *rho) {
  hipStream_t st = c->stream;
  const Grid g = make_grid(ng);
  const int64_t ncell = (int64_t)g.safe + 1;
  const uint64_t ext = (uint64_t)(ng[0] + 1) * (uint64_t)(ng[1] + 1) * (uint64_t)(ng[2] + 1);
  if (ext >= 0xffffffffull) {
    hsr_set_error("hsr_cic: (ng[0]+1)(ng[1]+1)(ng[2]+1) must be below 2^32 - 1");
    return HSR_ERR_ARG;
  }
  k_fill0<<<nblk(ncell, 256), 256, 0, st>>>(ncell, rho);
  HSR_HIP(hipGetLastError());
  if (n <= 0) return HSR_OK;
  const float cc = gpscal * gpscal * gpscal;  // Particles.cxx:606
  Ext ex;
  ex.e1 = (uint32_t)ng[1] + 1u;
  ex.e2 = (uint32_t)ng[2] + 1u;
  ex.out = (uint32_t)ext;
  int bits = 1;
  while (bits < 32 && ((uint64_t)ex.out >> bits) != 0) ++bits;
  // layout (8-byte arrays first): per grid cell the long-cell count (8 B);
  // per staged contribution of the outside slot its term (8 B; at most 8
  // per particle); then 4-byte arrays: per particle its key, sorted key,
  // index, sorted index, outside count and its prefix; per base cell its
  // range; per grid cell the long cell's id; per staged contribution its
  // run key; the long-cell counter
  const size_t nn = (size_t)n, nc = (size_t)g.safe, ms = 8 * nn, ne = (size_t)ex.out;
  // (each array starts on a 256-byte boundary: 14 arrays)
  const size_t bytes = 8 * (nc + ms) + 4 * (6 * nn + 2 * ne + nc + ms) + 32 + 14 * 256;
  HSR_HIP(dbuf_reserve(c->sub.keys, bytes));
  char *bp = (char *)c->sub.keys.p;
  auto take = [&bp](size_t b) {
    char *r = bp;
    bp += (b + 255) & ~(size_t)255;
    return r;
  };
  int64_t *long_k = (int64_t *)take(8 * nc);
  double *ts = (double *)take(8 * ms);
  uint32_t *key = (uint32_t *)take(4 * nn);
  uint32_t *key2 = (uint32_t *)take(4 * nn);
  int32_t *idx = (int32_t *)take(4 * nn);
  int32_t *idx2 = (int32_t *)take(4 * nn);
  int32_t *nout = (int32_t *)take(4 * nn);
  int32_t *out_base = (int32_t *)take(4 * nn);
  int32_t *beg = (int32_t *)take(4 * ne);
  int32_t *end = (int32_t *)take(4 * ne);
  uint32_t *long_cell = (uint32_t *)take(4 * nc);
  uint32_t *skey = (uint32_t *)take(4 * ms);
  unsigned long long *nlong = (unsigned long long *)take(32);  // and the unsorted flag, the host's totals
  int32_t *unsorted = (int32_t *)(nlong + 1);
  if ((size_t)(bp - (char *)c->sub.keys.p) > c->sub.keys.bytes) {
    hsr_set_error("hsr_cic: staging layout exceeds its buffer");
    return HSR_ERR_STATE;
  }
  k_zero_u64<<<1, 64, 0, st>>>(nlong);
  k_zero_u64<<<1, 64, 0, st>>>(nlong + 1);
  // particles by base cell (stable)
  k_cic_base<<<nblk(n, 256), 256, 0, st>>>(n, x, y, z, g, ex, key, idx, nout, unsorted);
  // the outside slot's contributions, and whether there is anything to sort:
  // one host round trip, which the contributions' count takes anyway
  hsr_status s;
  if ((s = pm_excl_scan(c, nout, out_base, n)) != HSR_OK) return s;
  int64_t *totals = (int64_t *)(nlong + 2);
  k_cic_totals<<<1, 64, 0, st>>>(out_base + n - 1, nout + n - 1, unsorted, totals);
  int64_t last[2] = {0, 0};
  HSR_HIP(hipMemcpyAsync(last, totals, sizeof(last), hipMemcpyDeviceToHost, st));
  HSR_HIP(stream_wait(st));
  const int64_t m = last[0];
  if ((size_t)m > ms) {
    hsr_set_error("hsr_cic: staged contributions exceed 8 per particle");
    return HSR_ERR_STATE;
  }
  if (last[1]) {
    size_t tmp = 0;
    HSR_HIP(hipcub::DeviceRadixSort::SortPairs(nullptr, tmp, key, key2, idx, idx2, (int)n, 0, bits, st));
    HSR_HIP(dbuf_reserve(c->s.cub, tmp + 256));
    HSR_HIP(hipcub::DeviceRadixSort::SortPairs(c->s.cub.p, tmp, key, key2, idx, idx2, (int)n, 0, bits, st));
  } else {
    // as the resort leaves them: particles in cell order have their base
    // cells in order, and a stable sort would move nothing (18M particles at
    // 256^3: 0.8 ms)
    key2 = key;
    idx2 = idx;
  }
  k_fill_i32<<<nblk((int64_t)ne, 256), 256, 0, st>>>((int64_t)ne, beg);
  k_fill_i32<<<nblk((int64_t)ne, 256), 256, 0, st>>>((int64_t)ne, end);
  k_cic_ranges<<<nblk(n, 256), 256, 0, st>>>(n, key2, ex, beg, end);
  // short cells summed, long ones queued and summed a workgroup each (the
  // grid loops over the device-side count)
  const auto cells = last[1] ? &k_cic_cells<false> : &k_cic_cells<true>;
  cells<<<nblk((int64_t)nc, 256), 256, 0, st>>>(g, ex, beg, end, idx2, x, y, z, cc, rho, long_cell, long_k,
                                                nlong);
  const unsigned lgrid = (unsigned)std::max(1, c->num_cus) * 32;
  const auto long_sum = last[1] ? &k_cic_long_sum<false> : &k_cic_long_sum<true>;
  long_sum<<<lgrid, 64, 0, st>>>(g, ex, beg, end, idx2, long_cell, long_k, nlong, x, y, z, cc, rho);
  // the outside slot: its contributions in (particle, corner) order
  if (m > 0) {
    k_cic_out_terms<<<nblk(n, 256), 256, 0, st>>>(n, x, y, z, g, cc, nout, out_base, 0, skey, ts);
    k_cic_tail<<<1, TAIL_THREADS, 0, st>>>(m, skey, ts, rho);
  }
  HSR_HIP(hipGetLastError());
  return HSR_OK;
}

hsr_status inverse_cic_run(hsr_ctx *c, int64_t n, const float *x, const float *y,
                           const float *z, const int32_t ng[3], const float *grid, float tau,
                           float fscal, float *v) {
  if (n <= 0) return HSR_OK;
  const Grid g = make_grid(ng);
  k_inverse_cic<<<nblk(n, 256), 256, 0, c->stream>>>(n, x, y, z, g, grid, tau, fscal, v);
  HSR_HIP(hipGetLastError());
  return HSR_OK;
}
