// force.hip -- short-range leaf kernel for gfx950 (FP32 VALU; no MFMA: the
// pair force is not a dense contraction).
//
// Pair law (BGQStep16.c:167-187, the 5th-order polynomial of ForceLaw.cxx
// :107-116 at POLY_ORDER 5):
//     f(r2) = m_j * [ (r2 + rsm^2)^(-3/2) - P(r2) ] * [r2 < rc2] (* [r2 > 0])
//     F_i  += f * (x_j - x_i)
// summed over every entry j of leaf i's interaction list (nbody1,
// RCBForceTree.cxx:599-619).  The polynomial is evaluated in s = r2 + rsm^2
// (coefficients re-expanded on the host), so s serves the power, the
// polynomial and the cutoff test.
//
// Work: one persistent launch walks a queue of work items -- a listed leaf,
// or a chunk of a long list -- sorted by decreasing pair count.  A wave
// takes an item: the leaf's i-particles sit in registers, R per lane, in G
// lane groups; the j-entries are staged in LDS per tile, each group owning a
// contiguous, padded slice (stride = 1 mod 8 entries, so the groups' 16-byte
// reads fall in distinct banks).  Chunk partials of long lists are summed in
// chunk order afterwards, so results are bitwise reproducible.
#include "hsr_internal.h"
#include "passes.h"
#include "queue.h"
#include "wave.h"

#include <hipcub/hipcub.hpp>

#include <algorithm>
#include <vector>

namespace {

// Kernel shapes: RR i-particles per lane, UU j entries per unrolled step,
// TT j entries staged per LDS tile.  The default (2, 2, 256) is the fastest
// measured at 256^3; the others are built for the tuner (hsr_tuning
// i_per_lane, unroll, tile).
constexpr int DEF_R = 2, DEF_U = 2, DEF_T = 256;
constexpr int GMAX = 16;      // at most 16 lane groups (>= 4 lanes each)
// Passes hold a power of two of at least 4 R target slots, so the group
// count G = 64 / (slots / R) is 1, 2, 4, 8 or 16;
// the staged slices of a full tile must fit for each of them.  A group's
// slice holds its unmasked entries (a multiple of UU) and its masked ones
// rounded up to UU: at most ceil(entries / G) + UU - 1 slots.
template <int UU>
__host__ __device__ constexpr int slice_slots(int nt, int G) { return (nt + G - 1) / G + UU; }
template <int UU, int TT>
constexpr int staged_entries(int G) {
  const int tg = slice_slots<UU>(TT, G);
  return G * (tg + ((9 - (tg & 7)) & 7));
}
template <int UU, int TT>
constexpr int lds_entries() {
  int m = 0;
  for (int G = 1; G <= GMAX; G *= 2) m = staged_entries<UU, TT>(G) > m ? staged_entries<UU, TT>(G) : m;
  return m;
}

struct Item {
  int32_t leaf;     // listed-leaf index
  int32_t cls;      // work class (0 = heaviest)
  int64_t e0, e1;   // list entry range
  int64_t pbase;    // partial-force offset (-1: write F directly)
};

// Degree of the fitted grid force's polynomial in r (fit_poly).
constexpr int FITN = 15;

struct LawArgs {
  float c[7];      // polynomial in s (degree 5 or 6)
  float rcs;       // s cutoff: pairs with s < rcs contribute
  float eps2;
  int guard;
  int cull;        // drop entries farther than the cutoff from the leaf's box
  float cull2;     // squared box distance beyond which every pair is masked
  int pmax;        // targets per pass (64 R or 32 R)
  int thin;        // few waves share a SIMD: fewer, wider passes (pass_slots)
  float in2;       // squared farthest box distance below which every pair of
                   // the pass is inside the cutoff (the unmasked class)
  int unmasked;    // 1: unit-mass entries inside the cutoff skip mask and mass
  // ForceLawSR with FGridEvalFit or FGridEvalInterp: f = s^-3/2 - g(r2),
  // pairs with r2 < rc2 contribute
  float rc2;
  float fit[FITN + 1];  // FGrid::fgor as a polynomial in t = fit_a r - 1
  float fit_a;          // 2 / rmax
  const float4 *bins;                        // {r2[i], f[i], f[i+1] - f[i], 0}
  float t_r2min, t_r2max, t_oodr2;
  int t_last;                                // last bin index (n_interp - 2)
};

// FGrid::fgor(r), the fitted grid force over r (ForceLaw.cxx:39-51), for r in
// [0, rmax]: the polynomial of fit_poly by Horner's rule.  Beyond rmax it is
// meaningless (the pair is masked by a select).
__device__ __forceinline__ float fgor_fit(const LawArgs &L, float r) {
  const float t = fmaf(r, L.fit_a, -1.f);
  float q = L.fit[FITN];
#pragma unroll
  for (int k = FITN - 1; k >= 0; --k) q = fmaf(q, t, L.fit[k]);
  return q;
}

// FGridEvalInterp::eval(r2) (ForceLaw.cxx:160-171): linear interpolation in
// the caller's table, zero outside (r2min, r2max).  The bin index is kept
// below the last point, which the reference's index can only reach through
// rounding just under r2max.
__device__ __forceinline__ float fgor_interp(const LawArgs &L, float r2) {
  const bool in = r2 > L.t_r2min && r2 < L.t_r2max;
  int k = in ? (int)((r2 - L.t_r2min) * L.t_oodr2) : 0;
  k = min(k, L.t_last);
  const float4 q = L.bins[k];
  const float v = q.y + (r2 - q.x) * L.t_oodr2 * q.z;
  return in ? v : 0.f;
}

// Squared distance from p to the box [lo, hi] (0 inside).
__device__ __forceinline__ float box_d2(const float *lo, const float *hi, float x, float y,
                                        float z) {
  const float dx = fmaxf(0.f, fmaxf(lo[0] - x, x - hi[0]));
  const float dy = fmaxf(0.f, fmaxf(lo[1] - y, y - hi[1]));
  const float dz = fmaxf(0.f, fmaxf(lo[2] - z, z - hi[2]));
  return dx * dx + dy * dy + dz * dz;
}

// Squared distance from p to the farthest point of the box [lo, hi].
__device__ __forceinline__ float box_far2(const float *lo, const float *hi, float x, float y,
                                          float z) {
  const float dx = fmaxf(fabsf(x - lo[0]), fabsf(x - hi[0]));
  const float dy = fmaxf(fabsf(y - lo[1]), fabsf(y - hi[1]));
  const float dz = fmaxf(fabsf(z - lo[2]), fabsf(z - hi[2]));
  return dx * dx + dy * dy + dz * dz;
}

template <int ORDER>
__device__ __forceinline__ float poly_tail(const LawArgs &L, float s) {
  // q(s) = c1 + c2 s + ... ; f = y^3 - c0 - s q(s)
  float q;
  if (ORDER == 6) {
    q = fmaf(L.c[6], s, L.c[5]);
    q = fmaf(q, s, L.c[4]);
  } else {
    q = fmaf(L.c[5], s, L.c[4]);
  }
  q = fmaf(q, s, L.c[3]);
  q = fmaf(q, s, L.c[2]);
  q = fmaf(q, s, L.c[1]);
  return q;
}

// Waves per SIMD the register allocation of the leaf kernel targets (0: the
// compiler's choice: 94 VGPRs, 5 waves, with the four pairs of an unrolled
// step interleaved; a cap of 6 waves fits 80 VGPRs but serialises them and
// measured 2.7% slower at 256^3).
#ifndef HSR_FORCE_WAVES
#define HSR_FORCE_WAVES 0
#endif
#if HSR_FORCE_WAVES > 0
#define HSR_FORCE_ATTR __attribute__((amdgpu_waves_per_eu(HSR_FORCE_WAVES, HSR_FORCE_WAVES)))
#else
#define HSR_FORCE_ATTR
#endif

// One pair: F_i += m_j f(r2) (x_j - x_i).  MASKED applies the cutoff (and
// the r2 > 0 guard) and the source mass; unmasked entries are known to have
// unit mass and every pair inside the cutoff, where both are exact no-ops.
template <int LAWK, int ORDER, bool GUARD, bool MASKED>
__device__ __forceinline__ void pair(const LawArgs &L, float c0, float rcs, const float4 p,
                                     float xi, float yi, float zi, float &ax, float &ay,
                                     float &az) {
  const float dx = p.x - xi;
  const float dy = p.y - yi;
  const float dz = p.z - zi;
  float f;
  if constexpr (LAWK == LAWK_POLY) {
    float s = fmaf(dx, dx, L.eps2);
    s = fmaf(dy, dy, s);
    s = fmaf(dz, dz, s);
    const float y = __builtin_amdgcn_rsqf(s);
    const float y2 = y * y;
    const float t3 = fmaf(y2, y, -c0);
    const float q = poly_tail<ORDER>(L, s);
    f = fmaf(-s, q, t3);
    if constexpr (MASKED) {
      float mm = (s < rcs) ? p.w : 0.f;
      if (GUARD) mm = (s > L.eps2) ? mm : 0.f;
      f *= mm;
    }
  } else {
    const float r2 = fmaf(dz, dz, fmaf(dy, dy, dx * dx));
    const float s = r2 + L.eps2;
    const float y = __builtin_amdgcn_rsqf(s);
    const float gr = LAWK == LAWK_FIT ? fgor_fit(L, __builtin_amdgcn_sqrtf(r2)) : fgor_interp(L, r2);
    f = y * y * y - gr;
    if constexpr (MASKED) {
      // a select, not a product: the fit's polynomial overflows at the padding
      // entries' distance
      bool in = r2 < L.rc2;
      if (GUARD) in = in && r2 > 0.f;
      f = in ? f * p.w : 0.f;
    }
  }
  ax = fmaf(f, dx, ax);
  ay = fmaf(f, dy, ay);
  az = fmaf(f, dz, az);
}

template <int LAWK, int ORDER, bool GUARD, int R, int UNROLL, int TILE>
__global__ void __launch_bounds__(64) HSR_FORCE_ATTR
k_force(const hsr_node *__restrict__ cn, const int32_t *__restrict__ leaves,
        const Item *__restrict__ items, const int64_t *__restrict__ nitems_p,
        const int32_t *__restrict__ jidx, const PJ *__restrict__ pj,
        const int32_t *__restrict__ iperm, LawArgs L,
        unsigned long long *__restrict__ qctr, float *__restrict__ fx,
        float *__restrict__ fy, float *__restrict__ fz, float *__restrict__ part,
        unsigned long long *__restrict__ evals) {
  static_assert(R == 1 || R == 2 || R == 4, "i-particles per lane");
  static_assert(UNROLL >= 1 && UNROLL <= 8, "j entries per unrolled step");
  static_assert(TILE % 64 == 0 && TILE <= 512, "tile of 64-entry chunks");
  constexpr int NCH = TILE / 64;  // 64-entry chunks per tile
  constexpr int LDS_ENT = lds_entries<UNROLL, TILE>();
  // the tile doubles as the reduction buffer once the j-walk is done
  __shared__ float4 tile[LDS_ENT];
  static_assert(3 * 64 * R <= 4 * LDS_ENT, "reduction buffer fits the tile");
  float (*red)[64 * R] = reinterpret_cast<float (*)[64 * R]>(&tile[0]);
  const int l = lane_id();
  const int64_t nitems = *nitems_p;
  const float c0 = L.c[0], rcs = L.rcs;
  __shared__ QueueState qs;
  queue_begin(&qs);
  for (;;) {
    const int64_t it = queue_pop(qctr, nitems, &qs);
    if (it >= nitems) break;
    const Item I = items[it];
    const hsr_node &nd = cn[leaves[I.leaf]];
    const int64_t off = nd.offset, cnt = nd.count;
    int64_t ev = 0;   // pairs evaluated for this item (culled entries excluded)
    int64_t evu = 0;  // of which unmasked
    // padding entries: far enough to be masked, near enough to keep every
    // intermediate finite
    const float4 pad = make_float4(nd.xc[0] + 1000.f, nd.xc[1], nd.xc[2], 0.f);
    // passes over the targets, each of a power of two of slots in groups of
    // lpg = slots / R lanes
    for (int64_t ib = 0, nib = 0; ib < cnt; ib += nib) {
      const int slots = pass_slots<R>(cnt - ib, L.pmax, L.thin);
      nib = min<int64_t>(slots, cnt - ib);
      const int ni = (int)nib;
      const int lpg = slots / R;
      const int G = 64 / lpg;
      const int g = l / lpg, tq = l & (lpg - 1);
      float xi[R], yi[R], zi[R], ax[R], ay[R], az[R];
      // the pass's targets (in the leaf's target order) and their box
      float bmin[3] = {INFINITY, INFINITY, INFINITY}, bmax[3] = {-INFINITY, -INFINITY, -INFINITY};
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const int ii = tq + r * lpg;
        const bool v = ii < ni;
        const PJ p = pj[iperm[off + ib + (v ? ii : 0)]];
        xi[r] = v ? p.x : 1e30f;
        yi[r] = v ? p.y : 1e30f;
        zi[r] = v ? p.z : 1e30f;
        ax[r] = ay[r] = az[r] = 0.f;
        if (v) {
          bmin[0] = fminf(bmin[0], p.x); bmax[0] = fmaxf(bmax[0], p.x);
          bmin[1] = fminf(bmin[1], p.y); bmax[1] = fmaxf(bmax[1], p.y);
          bmin[2] = fminf(bmin[2], p.z); bmax[2] = fmaxf(bmax[2], p.z);
        }
      }
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) {
#pragma unroll
        for (int d = 0; d < 3; ++d) {
          bmin[d] = fminf(bmin[d], __shfl_xor(bmin[d], o));
          bmax[d] = fmaxf(bmax[d], __shfl_xor(bmax[d], o));
        }
      }
      // the box is uniform across the wave: keep it in scalar registers
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        bmin[d] = __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, bmin[d])));
        bmax[d] = __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, bmax[d])));
      }
      const int lg = __builtin_ctz(G);  // G is a power of two
      for (int64_t t0 = I.e0; t0 < I.e1; t0 += TILE) {
        const int nt = (int)min<int64_t>(TILE, I.e1 - t0);
        int tgmax = slice_slots<UNROLL>(nt, G);
        const int stride = tgmax + ((9 - (tgmax & 7)) & 7);
        // Classify the tile's entries.  Culled: farther than the cutoff from
        // the pass's target box, every pair masked.  Unmasked: unit mass and
        // the farthest point of the box inside the cutoff, so every pair
        // passes the cutoff test and m_j = 1.  Masked: the rest.
        float4 v[NCH];
        uint64_t bk[NCH], ba[NCH];
#pragma unroll
        for (int k = 0; k < NCH; ++k) {
          v[k] = pad;
          bk[k] = ba[k] = 0;
          if (k * 64 < nt) {
            const int q = k * 64 + l;
            bool keep = false, um = false;
            if (q < nt) {
              const PJ p = pj[jidx[t0 + q]];
              v[k] = make_float4(p.x, p.y, p.z, p.m);
              keep = !L.cull || box_d2(bmin, bmax, p.x, p.y, p.z) <= L.cull2;
              um = keep && L.unmasked && p.m == 1.f &&
                   box_far2(bmin, bmax, p.x, p.y, p.z) < L.in2;
            }
            bk[k] = __ballot(keep);
            ba[k] = __ballot(um);
          }
        }
        int nA = 0, nK = 0;
#pragma unroll
        for (int k = 0; k < NCH; ++k) {
          nA += __popcll(ba[k]);
          nK += __popcll(bk[k]);
        }
        // Unmasked entries fill the first tA slots of every group (a multiple
        // of UNROLL, entry a -> group a % G, slot a / G); the unmasked ones
        // beyond G tA and the masked ones follow as masked entries m -> group
        // m % G, slot tA + m / G, padded to tM slots.
        const int tA = (nA >> lg) / UNROLL * UNROLL;
        const int splitA = tA << lg;
        const int nM = nK - splitA;
        const int tM = (((nM + G - 1) >> lg) + UNROLL - 1) / UNROLL * UNROLL;
        __syncthreads();
        const uint64_t lt = lanemask_lt();
        int pa = 0, pb = nA - splitA;
#pragma unroll
        for (int k = 0; k < NCH; ++k) {
          const uint64_t bm = bk[k] & ~ba[k];
          if ((bk[k] >> l) & 1ull) {
            int slot, grp;
            if ((ba[k] >> l) & 1ull) {
              const int a = pa + __popcll(ba[k] & lt);
              const int m = a - splitA;
              grp = (a < splitA ? a : m) & (G - 1);
              slot = a < splitA ? (a >> lg) : tA + (m >> lg);
            } else {
              const int m = pb + __popcll(bm & lt);
              grp = m & (G - 1);
              slot = tA + (m >> lg);
            }
            tile[grp * stride + slot] = v[k];
          }
          pa += __popcll(ba[k]);
          pb += __popcll(bm);
        }
        for (int m = nM + l; m < (tM << lg); m += 64) tile[(m & (G - 1)) * stride + tA + (m >> lg)] = pad;
        ev += (int64_t)nK * ni;
        evu += (int64_t)splitA * ni;
        __syncthreads();
        {
          const float4 *tp = tile + g * stride;
          // 0 .. 7: 152.5, 154.1, 152.8, 155.3, 152.6, 154.4, 151.7 and 155.4 ms
          // for shape (2, 2, 128), 151.3, 153.4, 151.7, 154.9, 151.8, 153.5,
          // 151.1 and 154.9 for (2, 2, 256) (256^3, leaves of 512)
          loop_offset<6>();
          for (int k = 0; k < tA; k += UNROLL) {
#pragma unroll
            for (int u = 0; u < UNROLL; ++u) {
              const float4 p = tp[k + u];
#pragma unroll
              for (int r = 0; r < R; ++r)
                pair<LAWK, ORDER, GUARD, false>(L, c0, rcs, p, xi[r], yi[r], zi[r], ax[r], ay[r], az[r]);
            }
          }
          for (int k = tA; k < tA + tM; k += UNROLL) {
#pragma unroll
            for (int u = 0; u < UNROLL; ++u) {
              const float4 p = tp[k + u];
#pragma unroll
              for (int r = 0; r < R; ++r)
                pair<LAWK, ORDER, GUARD, true>(L, c0, rcs, p, xi[r], yi[r], zi[r], ax[r], ay[r], az[r]);
            }
          }
        }
      }
      // fixed-order reduction over the G groups
      __syncthreads();
      for (int q = l; q < 64 * R; q += 64) red[0][q] = red[1][q] = red[2][q] = 0.f;
      __syncthreads();
      for (int gg = 0; gg < G; ++gg) {
        if (g == gg) {
#pragma unroll
          for (int r = 0; r < R; ++r) {
            const int ii = tq + r * lpg;
            if (ii < ni) {
              red[0][ii] += ax[r];
              red[1][ii] += ay[r];
              red[2][ii] += az[r];
            }
          }
        }
        __syncthreads();
      }
      if (I.pbase < 0) {
        for (int ii = l; ii < ni; ii += 64) {
          const int32_t q = iperm[off + ib + ii];
          fx[q] = red[0][ii];
          fy[q] = red[1][ii];
          fz[q] = red[2][ii];
        }
      } else {
        float *pp = part + I.pbase;
        for (int ii = l; ii < ni; ii += 64) {
          pp[3 * (ib + ii) + 0] = red[0][ii];
          pp[3 * (ib + ii) + 1] = red[1][ii];
          pp[3 * (ib + ii) + 2] = red[2][ii];
        }
      }
    }
    // into the wave's own slots, summed by k_reduce_chunks: atomics of all
    // waves on one address would pass one at a time; here nothing waits
    if (l == 0) {
      atomicAdd(evals + 2 * (int64_t)blockIdx.x, (unsigned long long)ev);
      atomicAdd(evals + 2 * (int64_t)blockIdx.x + 1, (unsigned long long)evu);
    }
  }
}

// Sum the chunk partials of long lists in chunk order; the last COUNT_BLOCKS
// workgroups sum the waves' pair counts: of every wave, since one past the
// items' number pops items too while the queue's owners (half the waves) are
// fewer than the items; with no more items than owners nothing is popped and
// the waves past the items counted none.  (One workgroup reads the 8192 waves'
// counts in 16 dependent batches, the kernel's time where there are few
// partials: 7.5 us at 32^3 with leaves of 32, 4.4 with 16.)
constexpr int COUNT_BLOCKS = 16;

__global__ void __launch_bounds__(256)
k_reduce_chunks(const hsr_node *cn, const int32_t *leaves,
                const int64_t *multi, const int64_t *nmulti_p,
                const int64_t *leaf_pbase, const int32_t *leaf_nchunk,
                const int32_t *iperm, const float *part, float *fx, float *fy, float *fz,
                const int64_t *nitems_p, int64_t nwaves, const unsigned long long *evals,
                unsigned long long *totals) {
  const int64_t nred = gridDim.x - COUNT_BLOCKS;  // workgroups for the partials
  if (blockIdx.x >= nred) {
    if (threadIdx.x >= 64) return;
    const int64_t nw = *nitems_p <= nwaves / 2 ? *nitems_p : nwaves;
    uint64_t a = 0, b = 0;
#pragma unroll 8
    for (int64_t w = 64 * (blockIdx.x - nred) + threadIdx.x; w < nw; w += 64 * COUNT_BLOCKS) {
      a += evals[2 * w];
      b += evals[2 * w + 1];
    }
    a = wave_sum_u64(a);
    b = wave_sum_u64(b);
    if (threadIdx.x == 0 && a) {
      atomicAdd(&totals[0], (unsigned long long)a);
      atomicAdd(&totals[1], (unsigned long long)b);
    }
    return;
  }
  // a fixed grid over the device-resident count, so a captured force phase
  // serves every list build
  for (int64_t k = blockIdx.x; k < *nmulti_p; k += nred) {
    const int64_t lf = multi[k];
    const hsr_node &nd = cn[leaves[lf]];
    const int64_t cnt = nd.count, off = nd.offset;
    const int nc = leaf_nchunk[lf];
    const float *p0 = part + leaf_pbase[lf];
    // a leaf's targets side by side and four chunks in flight: the loads bound it
    // (0.33 -> 0.21 ms at 256^3)
    for (int64_t i = threadIdx.x; i < cnt; i += blockDim.x) {
      float sx = 0.f, sy = 0.f, sz = 0.f;
#pragma unroll 4
      for (int c = 0; c < nc; ++c) {
        const float *p = p0 + (int64_t)c * 3 * cnt + 3 * i;
        sx += p[0];
        sy += p[1];
        sz += p[2];
      }
      const int32_t q = iperm[off + i];  // partials are kept in target order
      fx[q] = sx;
      fy[q] = sy;
      fz[q] = sz;
    }
  }
}

// Work items: chunk counts per leaf.
__global__ void k_item_count(int64_t nleaves, const int64_t *ent_ptr,
                             int64_t chunk, int32_t *nchunk, int64_t *nitem,
                             int64_t *multi_flag, const hsr_node *cn,
                             const int32_t *leaves, int64_t *psize) {
  int64_t k = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (k >= nleaves) return;
  int64_t L = ent_ptr[k + 1] - ent_ptr[k];
  int64_t c = std::max<int64_t>(1, (L + chunk - 1) / chunk);
  nchunk[k] = (int32_t)c;
  nitem[k] = c;
  multi_flag[k] = c > 1 ? 1 : 0;
  psize[k] = c > 1 ? c * 3 * cn[leaves[k]].count : 0;
}

// The plan's totals: items, leaves with several, partial floats; the counts
// the force phase reads are its first two.
__global__ void k_plan_totals(int64_t nl, const int64_t *item_base, const int64_t *nitem,
                              const int64_t *mpos, const int64_t *mflag, const int64_t *pbase,
                              const int64_t *psize, int64_t *counts) {
  if (threadIdx.x == 0) {
    counts[0] = item_base[nl - 1] + nitem[nl - 1];
    counts[1] = mpos[nl - 1] + mflag[nl - 1];
    counts[2] = pbase[nl - 1] + psize[nl - 1];
  }
}

// Work classes of the queue, heaviest first: four to the octave.
constexpr int NCLASS = 256;

__device__ __forceinline__ int work_class(int64_t targets, int64_t entries) {
  const int64_t passes = (targets + 64 * DEF_R - 1) / (64 * DEF_R);
  const float w = (float)(passes * entries + 1);
  const int b = (int)(__float_as_uint(w) >> 21) - (127 << 2);
  return NCLASS - 1 - min(NCLASS - 1, b);
}

__global__ void __launch_bounds__(256)
k_item_fill(int64_t nleaves, const int64_t *ent_ptr, int64_t chunk, const int32_t *nchunk,
            const int64_t *item_base, const int64_t *pbase, const hsr_node *cn,
            const int32_t *leaves, Item *items, uint32_t *hist, int64_t *multi,
            const int64_t *multi_pos, const int64_t *multi_flag) {
  __shared__ uint32_t h[NCLASS];
  h[threadIdx.x] = 0;
  __syncthreads();
  const int64_t k = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (k < nleaves) {
    const int64_t e0 = ent_ptr[k], e1 = ent_ptr[k + 1];
    const int nc = nchunk[k];
    const int64_t cnt = cn[leaves[k]].count;
    for (int c = 0; c < nc; ++c) {
      Item I;
      I.leaf = (int32_t)k;
      I.e0 = e0 + (int64_t)c * chunk;
      I.e1 = std::min<int64_t>(e1, I.e0 + chunk);
      I.pbase = nc > 1 ? pbase[k] + (int64_t)c * 3 * cnt : -1;
      I.cls = work_class(cnt, I.e1 - I.e0);
      items[item_base[k] + c] = I;
      atomicAdd(&h[I.cls], 1u);
    }
    if (multi_flag[k]) multi[multi_pos[k]] = k;
  }
  __syncthreads();
  if (h[threadIdx.x]) atomicAdd(&hist[threadIdx.x], h[threadIdx.x]);
}

// The queue in class order: a workgroup reserves its items' slots class by
// class (hist: items per class; next: slots given out).  The order inside a
// class, which no result depends on, is whichever workgroup came first.
__global__ void __launch_bounds__(256)
k_item_order(int64_t n, const Item *in, const uint32_t *hist, uint32_t *next, Item *out) {
  __shared__ uint32_t base[NCLASS], cnt[NCLASS];
  const int t = threadIdx.x;
  const uint32_t mine = hist[t];
  base[t] = mine;
  cnt[t] = 0;
  __syncthreads();
  for (int o = 1; o < NCLASS; o <<= 1) {  // inclusive scan
    const uint32_t v = t >= o ? base[t - o] : 0;
    __syncthreads();
    base[t] += v;
    __syncthreads();
  }
  const int64_t k = blockIdx.x * (int64_t)blockDim.x + t;
  Item I;
  uint32_t rank = 0;
  if (k < n) {
    I = in[k];
    rank = atomicAdd(&cnt[I.cls], 1u);
  }
  __syncthreads();
  const uint32_t first = base[t] - mine + (cnt[t] ? atomicAdd(&next[t], cnt[t]) : 0u);
  __syncthreads();
  base[t] = first;
  __syncthreads();
  if (k < n) out[base[I.cls] + rank] = I;
}

// The queue's class counts and slots start from zero.
__global__ void __launch_bounds__(256) k_zero_classes(uint32_t *hist) {
  hist[threadIdx.x] = hist[NCLASS + threadIdx.x] = 0;
}

// Forces and the waves' pair counts start from zero, the work queue from its
// first items.
__global__ void k_fill3(int64_t n, float *a, float *b, float *c, unsigned long long *qctr,
                        int64_t grid) {
  int64_t k = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (k < n) a[k] = b[k] = c[k] = 0.f;
  if (!qctr) return;
  if (blockIdx.x == 0) queue_reset(qctr, (int)threadIdx.x, grid);
  unsigned long long *evals = qctr + FORCE_TOTALS;  // the totals and the counts
  for (int64_t j = k; j < 2 * grid + 2; j += (int64_t)gridDim.x * blockDim.x) evals[j] = 0;
}

__global__ void k_kick(int64_t nleaves, const hsr_node *cn,
                       const int32_t *leaves, const float *fx,
                       const float *fy, const float *fz, const float *ms,
                       float fcoeff, int mul_mass, float *vx, float *vy,
                       float *vz) {
  int64_t k = blockIdx.x;
  if (k >= nleaves) return;
  const hsr_node &nd = cn[leaves[k]];
  for (int64_t i = threadIdx.x; i < nd.count; i += blockDim.x) {
    int64_t p = nd.offset + i;
    float cfac = mul_mass ? fcoeff * ms[p] : fcoeff;
    vx[p] = vx[p] + fx[p] * cfac;
    vy[p] = vy[p] + fy[p] * cfac;
    vz[p] = vz[p] + fz[p] * cfac;
  }
}

inline unsigned nblk(int64_t n, int t) { return (unsigned)((n + t - 1) / t); }

template <class T>
hsr_status excl_scan(hsr_ctx *c, const T *in, T *out, int64_t n) {
  size_t tmp = 0;
  HSR_HIP(hipcub::DeviceScan::ExclusiveSum(nullptr, tmp, in, out, (int)n, c->stream));
  HSR_HIP(dbuf_reserve(c->s.cub, tmp + 256));
  HSR_HIP(hipcub::DeviceScan::ExclusiveSum(c->s.cub.p, tmp, in, out, (int)n, c->stream));
  return HSR_OK;
}

// FGrid::fgor(r) = [tanh(br) - br/cosh^2(br) + cc r^3 (1 + d r^2) e^(-d r^2) +
// e r^2 (ff r^2 + g r^4 + l r^6) e^(-h r^2)] / r^3 on [0, rmax]
// (ForceLaw.cxx:23-51) as a polynomial of degree FITN in t = 2 r / rmax - 1:
// its interpolant at the Chebyshev points of the first kind, in double.
//
// fgor is analytic in r -- the first term's nearest singularities are the
// poles of tanh at r = +-i pi / (2 b) -- so the interpolants converge
// geometrically (about 3.6x per degree); at degree 15 the interpolant is
// within 2.4e-9 of fgor, below the float rounding of Horner's rule (3.6e-8
// at most, 7e-9 rms, against 0.26 at r = 0).  The expression itself in float
// loses up to 7e-5 for r > 0.05 and everything below r = 1e-3, where its
// first two terms cancel, and costs a coshf, a tanhf, two expf and three
// divisions per pair.  The pair is bound by VALU issue: 16 FMA and a square
// root in place of these took the leaf kernel from 6.88 to 1.00 ms on a
// 60^3 Plummer mix (216k particles, leaves of 128, 3.1e8 pairs).
struct FitPoly {
  float c[FITN + 1], scale;
};

FitPoly fit_poly() {
  const double b = 0.72f, cc = 0.01f, d = 0.27f, e = 0.0001f, ff = 360.0f, g = 100.0f, h = 0.67f,
               l = 17.0f, rmax = 3.116326355f;
  auto fgor = [&](double r) {
    const double r2 = r * r, u = b * r, u2 = u * u;
    // (tanh u - u / cosh^2 u) / u^3: from tanh's series where the terms cancel
    double th;
    if (u < 0.1) {
      th = 2.0 / 3.0 - u2 * (8.0 / 15.0 - u2 * (34.0 / 105.0 - u2 * (496.0 / 2835.0 -
           u2 * (13820.0 / 155925.0))));
    } else {
      const double ch = std::cosh(u);
      th = (std::tanh(u) - u / (ch * ch)) / (u2 * u);
    }
    return b * b * b * th + cc * (1.0 + d * r2) * std::exp(-d * r2) +
           e * r * (ff + g * r2 + l * r2 * r2) * std::exp(-h * r2);
  };
  constexpr int n = FITN + 1;
  const double pi = std::acos(-1.0);
  double cheb[n], mono[n] = {}, tp[n] = {}, tc[n] = {}, tn[n];
  double f[n];
  for (int i = 0; i < n; ++i) f[i] = fgor(0.5 * rmax * (std::cos(pi * (i + 0.5) / n) + 1.0));
  for (int k = 0; k < n; ++k) {
    cheb[k] = 0.0;
    for (int i = 0; i < n; ++i) cheb[k] += f[i] * std::cos(pi * k * (i + 0.5) / n);
    cheb[k] *= (k == 0 ? 1.0 : 2.0) / n;
  }
  // T_0 = 1, T_1 = t, T_(k+1) = 2 t T_k - T_(k-1), summed into powers of t
  tp[0] = 1.0;
  tc[1] = 1.0;
  for (int i = 0; i < n; ++i) mono[i] = cheb[0] * tp[i] + cheb[1] * tc[i];
  for (int k = 2; k < n; ++k) {
    for (int i = 0; i < n; ++i) tn[i] = (i ? 2.0 * tc[i - 1] : 0.0) - tp[i];
    for (int i = 0; i < n; ++i) {
      mono[i] += cheb[k] * tn[i];
      tp[i] = tc[i];
      tc[i] = tn[i];
    }
  }
  FitPoly P;
  for (int i = 0; i < n; ++i) P.c[i] = (float)mono[i];
  P.scale = (float)(2.0 / rmax);
  return P;
}

// P(r2) = sum a_k r2^k re-expanded in s = r2 + eps2 (host, double).
LawArgs law_args(const ForceLawDev &D) {
  LawArgs A = {};
  double a[7] = {0, 0, 0, 0, 0, 0, 0}, b[7] = {0, 0, 0, 0, 0, 0, 0};
  for (int k = 0; k <= 6; ++k) a[k] = D.c[k];
  const double e = D.eps2;
  // P(s - e) = sum_k a_k (s - e)^k
  for (int k = 0; k <= 6; ++k) {
    double binom = 1.0;
    for (int i = 0; i <= k; ++i) {
      // coefficient of s^i in (s - e)^k: C(k,i) (-e)^(k-i)
      double cki = binom;
      double term = cki * std::pow(-e, k - i);
      b[i] += a[k] * term;
      binom = binom * (double)(k - i) / (double)(i + 1);
    }
  }
  for (int k = 0; k <= 6; ++k) A.c[k] = (float)b[k];
  // r2 < rc2  <=>  s < rc2 + eps2 up to rounding at the boundary, where the
  // short-range force is ~1e-5 of its r = 1 value
  A.rcs = (float)((double)D.rc2 + e);
  A.eps2 = D.eps2;
  A.guard = D.guard;
  // a relative margin far above the few-ulp rounding of r2 keeps every pair
  // the kernel's own s < rcs test would accept
  A.cull = 1;
  A.cull2 = (float)((double)D.rc2 * (1.0 + 1e-4));
  A.pmax = 64 * DEF_R;
  A.thin = 0;
  // the same relative margin the other way: every pair of an entry whose
  // farthest box point is inside in2 passes the kernel's cutoff test
  A.in2 = (float)((double)D.rc2 * (1.0 - 1e-4));
  A.unmasked = D.guard ? 0 : 1;
  A.rc2 = D.rc2;
  if (D.kind == LAWK_FIT) {
    static const FitPoly P = fit_poly();  // of constants alone (3 us)
    std::copy(P.c, P.c + FITN + 1, A.fit);
    A.fit_a = P.scale;
  }
  A.bins = D.bins;
  A.t_r2min = D.t_r2min;
  A.t_r2max = D.t_r2max;
  A.t_oodr2 = D.t_oodr2;
  A.t_last = std::max(0, D.n_interp - 2);
  return A;
}

}  // namespace

// Target order inside each listed leaf: positions sorted along the leaf's
// longest box edge (ties x > y > z; equal coordinates by position), so that
// a pass's 128 targets span a slab of the leaf and the entries its box is
// beyond the cutoff of can be skipped.  iperm[off + k] = position of the
// k-th target; leaves above SORT_MAX keep their order.
constexpr int SORT_MAX = 1024;

__global__ void k_iota32(int64_t n, int32_t *a) {
  const int64_t k = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (k < n) a[k] = (int32_t)k;
}

// Every target's place is the number of smaller keys in its leaf: n broadcast
// LDS reads a target and no barriers, where a bitonic sort took log^2 n of
// them (0.70 -> 0.53 ms at 256^3 with leaves of 512).  The keys are whole
// coordinates: their leading 22 bits, with the position in the other ten, took
// 0.41 ms, but leave targets that agree in them in tree order (evaluated pairs
// 4.1216e11 against 4.1205e11 there, 0.03%: 0.05 ms of the leaf kernel, and
// three times that of the adjoint).
__global__ void __launch_bounds__(256)
k_leaf_sort(int64_t nl, const int32_t *__restrict__ leaves, const hsr_node *__restrict__ cn,
            const PJ *__restrict__ pj, int32_t *__restrict__ iperm) {
  __shared__ uint32_t key[SORT_MAX];
  const int64_t k = blockIdx.x;
  if (k >= nl) return;
  const hsr_node &nd = cn[leaves[k]];
  const int64_t off = nd.offset;
  if (nd.count < 2 || nd.count > SORT_MAX) return;
  const int cnt = (int)nd.count;
  const float e0 = nd.xmax[0] - nd.xmin[0], e1 = nd.xmax[1] - nd.xmin[1],
              e2 = nd.xmax[2] - nd.xmin[2];
  const int d = (e0 >= e1 && e0 >= e2) ? 0 : (e1 >= e2 ? 1 : 2);
  for (int i = threadIdx.x; i < cnt; i += 256) {
    const PJ p = pj[off + i];
    const uint32_t u = __float_as_uint(d == 0 ? p.x : (d == 1 ? p.y : p.z));
    // an unsigned number in the order of the floats
    key[i] = u ^ ((uint32_t)((int32_t)u >> 31) | 0x80000000u);
  }
  __syncthreads();
  for (int i = threadIdx.x; i < cnt; i += 256) {
    const uint32_t mine = key[i];
    // equal coordinates by position: those before count, those after do not
    const int w0 = i & ~63, w1 = min(w0 + 64, cnt);  // the wave's own
    int rank = 0;
#pragma unroll 8
    for (int q = 0; q < w0; ++q) rank += key[q] <= mine ? 1 : 0;
#pragma unroll 8
    for (int q = w0; q < w1; ++q) rank += key[q] < mine || (key[q] == mine && q < i) ? 1 : 0;
#pragma unroll 8
    for (int q = w1; q < cnt; ++q) rank += key[q] < mine ? 1 : 0;
    iperm[off + rank] = (int32_t)(off + i);
  }
}

// Shapes built for every polynomial law without the r2 > 0 guard (the
// production laws); the other laws run the default shape only.
struct Shape {
  int r, u, t;
};
constexpr Shape kShapes[] = {{2, 2, 256}, {2, 1, 256}, {2, 4, 256}, {1, 2, 256},
                             {1, 4, 256}, {4, 1, 256}, {2, 2, 128}, {2, 2, 512}};

void force_shape(const hsr_tuning &t, int *r, int *u, int *tile) {
  *r = t.i_per_lane ? t.i_per_lane : DEF_R;
  *u = t.unroll ? t.unroll : DEF_U;
  *tile = t.tile ? t.tile : DEF_T;
}

bool force_shape_built(int law_kind, bool guard, int r, int u, int tile) {
  if (r == DEF_R && u == DEF_U && tile == DEF_T) return true;
  if (law_kind != LAWK_POLY || guard) return false;
  for (const Shape &sh : kShapes)
    if (sh.r == r && sh.u == u && sh.t == tile) return true;
  return false;
}

std::string force_shapes_built() {
  std::string out;
  for (const Shape &sh : kShapes)
    out += (out.empty() ? "" : ", ") + std::string("(") + std::to_string(sh.r) + ", " +
           std::to_string(sh.u) + ", " + std::to_string(sh.t) + ")";
  return out;
}

// List entries per work item when the caller sets none: CHUNK_MAX, halved
// while the lists would give the chip fewer than ITEMS_PER_CU items per
// compute unit, down to one tile.  A wave works through its item alone, so a
// load whose leaves are few or short leaves most of the chip idle, and the
// rest waiting for the longest list, unless the lists are cut finer; above
// the line the items outnumber the resident waves (20 per compute unit)
// several times and a finer cut only adds target loads and partial sums
// (8192 measured 0.5% faster for the leaf kernel and 2% for the adjoint than
// 16384 at 256^3).  Leaf kernel and fused adjoint with 8192 and with this
// rule (queue.h's queue both times): 0.62 and 0.18, 1.31 and 0.46 ms on a
// 50^3 Plummer mix with leaves of 128; 0.87 and 0.47 ms (leaf kernel) at 64^3.
// The partial sums the cut makes (12 bytes per target and item of a leaf
// with several) stay below PART_MAX bytes.
constexpr int64_t CHUNK_MIN = 256, ITEMS_PER_CU = 160;
constexpr int64_t PART_MAX = (int64_t)1 << 28;

static int64_t auto_chunk(const hsr_ctx *c) {
  const int64_t want = (int64_t)std::max(1, c->num_cus) * ITEMS_PER_CU;
  int64_t chunk = CHUNK_MAX;
  while (chunk > CHUNK_MIN && c->lists.nentries / chunk < want &&
         c->lists.pairs / (chunk / 2) <= PART_MAX / 12)
    chunk >>= 1;
  return chunk;
}

// (full: an allocation found no room)
static hsr_status force_plan_chunk(hsr_ctx *c, int64_t chunk, bool *full);

hsr_status force_plan(hsr_ctx *c) {
  bool full = false;
  if (c->tuning.chunk > 0) return force_plan_chunk(c, c->tuning.chunk, &full);
  const int64_t chunk = auto_chunk(c);
  hsr_status s = force_plan_chunk(c, chunk, &full);
  // what the finer cut takes more may exceed the caller's cap or the device
  if (s != HSR_OK && chunk < CHUNK_MAX && (s == HSR_ERR_NOMEM || full)) {
    if (full) {
      dbuf_free(c->lists.items);
      dbuf_free(c->lists.part);
    }
    s = force_plan_chunk(c, CHUNK_MAX, &full);
  }
  return s;
}

static hsr_status force_plan_chunk(hsr_ctx *c, int64_t chunk, bool *full) {
  hipStream_t st = c->stream;
  auto reserve = [full](DBuf &b, size_t bytes) {
    const hipError_t e = dbuf_reserve(b, bytes);
    *full = e == hipErrorOutOfMemory;
    return e;
  };
  ListState &LS = c->lists;
  const int64_t nl = LS.nleaves;
  LS.chunk = chunk;
  // the lists were short of items for the chip: what waves there are run
  // with few others on their SIMD
  LS.thin = LS.nentries / CHUNK_MAX < (int64_t)std::max(1, c->num_cus) * 16;
  if (nl == 0) {
    LS.nitems = 0;
    return HSR_OK;
  }
  // scratch layout (int64 unless noted), arrays at a stride that only grows,
  // so their addresses (held by a captured force phase) survive list builds
  if (nl + 3 > LS.plan_stride) LS.plan_stride = std::max<int64_t>(nl + 3, LS.plan_stride + LS.plan_stride / 4);
  const int64_t ps = LS.plan_stride;
  HSR_HIP(reserve(LS.plan, sizeof(int64_t) * 8 * ps + sizeof(int32_t) * ps + 256));
  int64_t *nitem = dptr<int64_t>(LS.plan);
  int64_t *item_base = nitem + ps;
  int64_t *mflag = item_base + ps;
  int64_t *mpos = mflag + ps;
  int64_t *psize = mpos + ps;
  int64_t *pbase = psize + ps;
  int64_t *multi = pbase + ps;
  int64_t *counts = multi + ps;  // [0] nitems, [1] nmulti, [2] partial floats
  int32_t *nchunk = reinterpret_cast<int32_t *>(counts + ps);
  const hsr_node *cn = dptr<hsr_node>(c->tree.canon_nodes);
  const int32_t *leaves = dptr<int32_t>(LS.leaves);
  const int64_t *ent_ptr = dptr<int64_t>(LS.ent_ptr);
  k_item_count<<<nblk(nl, 256), 256, 0, st>>>(nl, ent_ptr, chunk, nchunk, nitem, mflag, cn, leaves, psize);
  hsr_status s;
  if ((s = excl_scan(c, nitem, item_base, nl)) != HSR_OK) return s;
  if ((s = excl_scan(c, mflag, mpos, nl)) != HSR_OK) return s;
  if ((s = excl_scan(c, psize, pbase, nl)) != HSR_OK) return s;
  // (the arrays' stride leaves counts room for its three words)
  k_plan_totals<<<1, 64, 0, st>>>(nl, item_base, nitem, mpos, mflag, pbase, psize, counts);
  int64_t tail[3];
  HSR_HIP(hipMemcpyAsync(tail, counts, sizeof(tail), hipMemcpyDeviceToHost, st));
  HSR_HIP(stream_wait(st));
  const int64_t nitems = tail[0], nmulti = tail[1], npart = tail[2];
  // the item ids are 32-bit
  if (nitems >= (int64_t)INT32_MAX) {
    hsr_set_error("force plan: " + std::to_string(nitems) +
                  " work items (2^31 or more); raise tuning.chunk");
    return HSR_ERR_NOMEM;
  }
  const int64_t plan_bytes = (int64_t)sizeof(Item) * 2 * (nitems + 1) + (int64_t)sizeof(float) * npart;
  if (c->tuning.max_plan_bytes > 0 && plan_bytes > c->tuning.max_plan_bytes) {
    hsr_set_error("force plan: needs " + std::to_string(plan_bytes) + " bytes, above tuning.max_plan_bytes (" +
                  std::to_string(c->tuning.max_plan_bytes) + ")");
    return HSR_ERR_NOMEM;
  }
  LS.nitems = nitems;
  LS.nmulti = nmulti;
  HSR_HIP(reserve(LS.items, sizeof(Item) * 2 * (nitems + 1)));
  HSR_HIP(reserve(LS.item_keys, sizeof(uint32_t) * 2 * NCLASS));
  HSR_HIP(reserve(LS.part, sizeof(float) * std::max<int64_t>(npart, 1)));
  Item *items_tmp = dptr<Item>(LS.items) + (nitems + 1);
  Item *items = dptr<Item>(LS.items);
  uint32_t *hist = dptr<uint32_t>(LS.item_keys);
  k_zero_classes<<<1, NCLASS, 0, st>>>(hist);
  k_item_fill<<<nblk(nl, 256), 256, 0, st>>>(nl, ent_ptr, chunk, nchunk, item_base, pbase, cn, leaves,
                                             items_tmp, hist, multi, mpos, mflag);
  // heaviest items first
  k_item_order<<<nblk(nitems, 256), 256, 0, st>>>(nitems, items_tmp, hist, hist + NCLASS, items);
  LS.multi = multi;
  LS.counts = counts;
  LS.leaf_pbase = pbase;
  LS.leaf_nchunk = nchunk;
  // target order inside the listed leaves
  const int64_t n = c->tree.n;
  HSR_HIP(reserve(LS.iperm, sizeof(int32_t) * std::max<int64_t>(n, 1)));
  int32_t *iperm = dptr<int32_t>(LS.iperm);
  if (n) k_iota32<<<nblk(n, 256), 256, 0, st>>>(n, iperm);
  if (!c->tuning.tree_order_targets)
    k_leaf_sort<<<(unsigned)nl, 256, 0, st>>>(nl, leaves, cn, dptr<PJ>(c->tree.pj), iperm);
  HSR_HIP(hipGetLastError());
  return HSR_OK;
}

static hsr_status force_enqueue(hsr_ctx *c, float *fx, float *fy, float *fz,
                                bool timed);

static_assert(FORCE_TOTALS >= QWORDS, "pair totals lie behind the queue's counters");

// The persistent grid does not depend on the item count (waves beyond the
// items leave at once), so a captured launch fits any list.
static int64_t force_grid(const hsr_ctx *c) {
  const int wpc = c->tuning.waves_per_cu > 0 ? c->tuning.waves_per_cu : 32;
  return (int64_t)std::max(1, c->num_cus) * wpc;
}

static unsigned reduce_grid(const hsr_ctx *c) {
  unsigned g = 256;
  while ((int64_t)g < c->lists.nmulti) g <<= 1;
  return g;
}

// The force phase: zero F, reset the work queue, persistent leaf kernel,
// chunk reduction.  With tuning.use_graph the launches are captured once and
// replayed as one graph across list builds: their grids are fixed (the
// persistent kernel and the chunk reduction read their counts from device
// memory), so a new capture is needed only when an address they use, the
// particle count or the settings change.
hsr_status force_run(hsr_ctx *c, float *fx, float *fy, float *fz) {
  hipStream_t st = c->stream;
  if (c->law.kind == LAWK_INTERP && !c->law.bins) {
    hsr_set_error("HSR_LAW_SR_INTERP: no table (call hsr_set_law_table first)");
    return HSR_ERR_STATE;
  }
  HSR_HIP(dbuf_reserve(c->s.qctr, sizeof(unsigned long long) * (FORCE_TOTALS + 2 + 2 * (size_t)force_grid(c))));
  if (!c->tuning.use_graph) return force_enqueue(c, fx, fy, fz, true);
  const ListState &LS = c->lists;
  const uintptr_t sig[20] = {(uintptr_t)fx, (uintptr_t)fy, (uintptr_t)fz, (uintptr_t)c->tree.n,
                             (uintptr_t)(LS.nleaves == 0 || LS.nitems == 0), (uintptr_t)c->tree.canon_nodes.p,
                             (uintptr_t)LS.leaves.p, (uintptr_t)LS.items.p, (uintptr_t)LS.counts,
                             (uintptr_t)LS.jidx.p, (uintptr_t)c->tree.pj.p, (uintptr_t)LS.iperm.p,
                             (uintptr_t)LS.part.p, (uintptr_t)LS.multi, (uintptr_t)LS.leaf_pbase,
                             (uintptr_t)LS.leaf_nchunk, (uintptr_t)c->s.qctr.p, (uintptr_t)reduce_grid(c), (uintptr_t)LS.thin, 0};
  bool same = c->graph_exec != nullptr && c->graph_gen != -1;
  for (int k = 0; k < 20 && same; ++k) same = c->graph_sig[k] == sig[k];
  const bool stale = !same;
  if (stale) {
    if (c->graph_exec) {
      HSR_HIP(hipGraphExecDestroy(c->graph_exec));
      c->graph_exec = nullptr;
    }
    if (c->graph) {
      HSR_HIP(hipGraphDestroy(c->graph));
      c->graph = nullptr;
    }
    HSR_HIP(hipStreamBeginCapture(st, hipStreamCaptureModeThreadLocal));
    hsr_status s = force_enqueue(c, fx, fy, fz, false);
    hipGraph_t g = nullptr;
    hipError_t e = hipStreamEndCapture(st, &g);
    if (s != HSR_OK) {
      if (g) (void)hipGraphDestroy(g);
      return s;
    }
    HSR_HIP(e);
    c->graph = g;
    HSR_HIP(hipGraphInstantiate(&c->graph_exec, g, nullptr, nullptr, 0));
    c->graph_gen = 0;
    for (int k = 0; k < 20; ++k) c->graph_sig[k] = sig[k];
    c->graph_captures++;
  }
  HSR_HIP(hipEventRecord(c->ev[6], st));
  HSR_HIP(hipGraphLaunch(c->graph_exec, st));
  HSR_HIP(hipEventRecord(c->ev[7], st));
  c->kernel_timed = true;
  c->graph_launches++;
  return HSR_OK;
}

static hsr_status force_enqueue(hsr_ctx *c, float *fx, float *fy, float *fz,
                                bool timed) {
  hipStream_t st = c->stream;
  const int64_t n = c->tree.n;
  ListState &LS = c->lists;
  if (timed) c->kernel_timed = false;
  const bool work = LS.nleaves > 0 && LS.nitems > 0;
  const int64_t grid = force_grid(c);
  unsigned long long *qctr = dptr<unsigned long long>(c->s.qctr);
  if (n > 0 || work)
    k_fill3<<<(unsigned)std::max<int64_t>(1, (n + 255) / 256), 256, 0, st>>>(n, fx, fy, fz,
                                                                             work ? qctr : nullptr, grid);
  if (!work) return HSR_OK;
  unsigned long long *totals = qctr + FORCE_TOTALS, *evals = totals + 2;
  LawArgs A = law_args(c->law);
  A.cull = c->tuning.cull_off ? 0 : 1;
  int R, U, T;
  force_shape(c->tuning, &R, &U, &T);
  A.pmax = c->tuning.force_pass == 32 * R ? 32 * R : 64 * R;
  A.thin = LS.thin;
  const hsr_node *cn = dptr<hsr_node>(c->tree.canon_nodes);
  const int32_t *leaves = dptr<int32_t>(LS.leaves);
  const Item *items = dptr<Item>(LS.items);
  float *part = dptr<float>(LS.part);
  // events bracket the leaf-kernel launch alone (the roofline's duration)
  if (timed) HSR_HIP(hipEventRecord(c->ev[6], st));
#define LAUNCH(LK, ORD, GRD, RR, UU, TT)                                              \
  k_force<LK, ORD, GRD, RR, UU, TT><<<(unsigned)grid, 64, 0, st>>>(cn, leaves, items, LS.counts, \
      dptr<int32_t>(LS.jidx), dptr<PJ>(c->tree.pj), dptr<int32_t>(LS.iperm), A, qctr, fx, fy, fz, \
      part, evals)
#define SHAPES(ORD)                                                                      \
  if (R == 2 && U == 1 && T == 256) LAUNCH(LAWK_POLY, ORD, false, 2, 1, 256);            \
  else if (R == 2 && U == 4 && T == 256) LAUNCH(LAWK_POLY, ORD, false, 2, 4, 256);       \
  else if (R == 1 && U == 2 && T == 256) LAUNCH(LAWK_POLY, ORD, false, 1, 2, 256);       \
  else if (R == 1 && U == 4 && T == 256) LAUNCH(LAWK_POLY, ORD, false, 1, 4, 256);       \
  else if (R == 4 && U == 1 && T == 256) LAUNCH(LAWK_POLY, ORD, false, 4, 1, 256);       \
  else if (R == 2 && U == 2 && T == 128) LAUNCH(LAWK_POLY, ORD, false, 2, 2, 128);       \
  else if (R == 2 && U == 2 && T == 512) LAUNCH(LAWK_POLY, ORD, false, 2, 2, 512);       \
  else LAUNCH(LAWK_POLY, ORD, false, DEF_R, DEF_U, DEF_T)
  if (c->law.kind == LAWK_FIT) {
    if (A.guard) LAUNCH(LAWK_FIT, 0, true, DEF_R, DEF_U, DEF_T);
    else LAUNCH(LAWK_FIT, 0, false, DEF_R, DEF_U, DEF_T);
  } else if (c->law.kind == LAWK_INTERP) {
    if (A.guard) LAUNCH(LAWK_INTERP, 0, true, DEF_R, DEF_U, DEF_T);
    else LAUNCH(LAWK_INTERP, 0, false, DEF_R, DEF_U, DEF_T);
  } else if (c->law.order == 6) {
    if (A.guard) LAUNCH(LAWK_POLY, 6, true, DEF_R, DEF_U, DEF_T);
    else { SHAPES(6); }
  } else {
    if (A.guard) LAUNCH(LAWK_POLY, 5, true, DEF_R, DEF_U, DEF_T);
    else { SHAPES(5); }
  }
#undef SHAPES
#undef LAUNCH
  HSR_HIP(hipGetLastError());
  if (timed) {
    HSR_HIP(hipEventRecord(c->ev[7], st));
    c->kernel_timed = true;
  }
  // a grid over the device-resident multi-chunk count (which may be 0): a
  // workgroup per multi-chunk leaf, the grid rounded up to a power of two so a
  // captured force phase serves later lists unless their count outgrows it
  k_reduce_chunks<<<reduce_grid(c) + COUNT_BLOCKS, leaf_threads(c), 0, st>>>(
      cn, leaves, LS.multi, LS.counts + 1, LS.leaf_pbase, LS.leaf_nchunk, dptr<int32_t>(LS.iperm), part,
      fx, fy, fz, LS.counts, grid, evals, totals);
  HSR_HIP(hipGetLastError());
  return HSR_OK;
}

hsr_status kick_run(hsr_ctx *c, float fcoeff, float *vx, float *vy, float *vz,
                    const float *mass_sorted) {
  int64_t n = c->tree.n;
  HSR_HIP(dbuf_reserve(c->force, sizeof(float) * 3 * std::max<int64_t>(n, 1)));
  float *f = dptr<float>(c->force);
  hsr_status s = force_run(c, f, f + n, f + 2 * n);
  if (s != HSR_OK) return s;
  if (c->lists.nleaves == 0) return HSR_OK;
  // Step16 path: v += fcoeff * a (BGQStep16 caller, RCBForceTree.cxx:594-596);
  // ForceLaw path: nbody1 multiplies by m_i (RCBForceTree.cxx:610).
  int mul_mass = c->p.law == HSR_LAW_STEP16 ? 0 : 1;
  k_kick<<<(unsigned)c->lists.nleaves, 256, 0, c->stream>>>(
      c->lists.nleaves, dptr<hsr_node>(c->tree.canon_nodes),
      dptr<int32_t>(c->lists.leaves), f, f + n, f + 2 * n, mass_sorted, fcoeff,
      mul_mass, vx, vy, vz);
  HSR_HIP(hipGetLastError());
  return HSR_OK;
}
