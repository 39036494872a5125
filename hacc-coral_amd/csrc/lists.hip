// lists.hip -- bit-exact per-leaf interaction lists on the GPU.
//
// Restates RCBForceTree<TDPTS>::calcInternodeForces / calcInternodeForce
// (RCBForceTree.cxx:924-1197, useRealOA = false): for every leaf inside the
// force box, a right-child-first LIFO walk from the root that
//   * expands the leaf's ancestors to their children (except the leaf),
//   * accepts a node whose angular size passes the tan(oa) test and drops
//     it if its centre is farther than fsrrmax; an accepted node with
//     count <= TDPTS contributes its particles, else its TDPTS
//     pseudo-particles (TDPTS = 1 or 12),
//   * takes a not-accepted leaf's particles,
//   * pushes the children of a not-accepted internal node whose L-infinity
//     gap to the target leaf is <= fsrrmax,
// and finally appends the leaf's own particles.  One wave walks one leaf's
// list, up to 64 nodes of its LIFO stack (in LDS) at a time.
//
// Compiled with -ffp-contract=off so dist2, l2, dtt2 and the corner
// diagonals round exactly as the reference's x86 float code does.
#include "hsr_internal.h"
#include "wave.h"

#include <hipcub/hipcub.hpp>

#include <algorithm>
#include <cstring>
#include <vector>

namespace {

struct ListParams {
  float fsrrmax, fsrrmax2, tan_oa;
  int tdpts;                 // pseudo-particles per node (1 or 12)
  int stack_cap;             // nodes the wave's LDS stack holds
  int stack_reserve;         // of which the last ones are for one-by-one walking
  int64_t *overflow;
  // the count pass keeps each leaf's first `cache` segments (offset or node
  // id, count or -1) at cache_seg[leaf * cache + i]; only longer lists are
  // walked again to be filled in
  int cache;
  int2 *cache_seg;
};

// Leaf of box b in the right-first order gets slot leaf_base[b] + leaf_rank.
__global__ void k_leaf_slots(const BNode *nodes, int64_t nb,
                             const int32_t *box_of, const int64_t *leaf_base,
                             const float *fmin, const float *fmax,
                             int32_t *slot_canon, const int64_t *cbase) {
  int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (t >= nb) return;
  const BNode &n = nodes[t];
  if (n.kind == NODE_SPLIT) return;
  int b = box_of[t];
  const float *lo = fmin + 3 * b, *hi = fmax + 3 * b;
  // RCBForceTree.cxx:1166-1170 (strict open interval on either face)
  bool inside = true;
  for (int i = 0; i < 3; ++i) {
    inside &= (n.xmax[i] < hi[i] && n.xmax[i] > lo[i]) ||
              (n.xmin[i] < hi[i] && n.xmin[i] > lo[i]);
  }
  slot_canon[leaf_base[b] + n.leaf_rank] =
      inside ? (int32_t)(cbase[b] + n.canon) : -1;
}

__global__ void k_flag_valid(const int32_t *slot, int64_t n, int32_t *flag) {
  int64_t k = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (k <= n) flag[k] = k < n && slot[k] >= 0 ? 1 : 0;  // flag[n]: the scan ends with the total
}

__global__ void k_compact(const int32_t *slot, const int32_t *flag,
                          const int32_t *pos, int64_t n, int32_t *out,
                          int32_t *out_box, const int32_t *slot_box) {
  int64_t k = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (k < n && flag[k]) {
    out[pos[k]] = slot[k];
    out_box[pos[k]] = slot_box[k];
  }
}

__global__ void k_slot_box(int64_t nboxes, const int64_t *leaf_base,
                           int32_t *slot_box) {
  int64_t b = blockIdx.x;
  if (b >= nboxes) return;
  for (int64_t k = leaf_base[b] + threadIdx.x; k < leaf_base[b + 1];
       k += blockDim.x)
    slot_box[k] = (int32_t)b;
}

// What a stack slot of the walk holds: a node still to be looked at (a node
// reached from a not-accepted one must first pass the distance test; an
// ancestor's child need not) or a decided segment, waiting for those that
// come before it in the list.
enum { W_NODE = 0, W_NODE_GAP = 1, W_RANGE = 2, W_PSEUDO = 3 };

// Whether node N, seen from leaf L's centre, is too large to be accepted
// (RCBForceTree.cxx:975-1030: the shortest edge, then the four space
// diagonals with z fixed min to max, against dist2 tan^2 oa).
__device__ __forceinline__ bool looks_big(const hsr_node &N, const float *lxc, float dist2,
                                          float tanOA) {
  const float sx = N.xmax[0] - N.xmin[0];
  const float sy = N.xmax[1] - N.xmin[1];
  const float sz = N.xmax[2] - N.xmin[2];
  const float sx2 = sx * sx, sy2 = sy * sy, sz2 = sz * sz;
  const float syz = (sz2 < sy2) ? sz2 : sy2;
  const float l2 = (syz < sx2) ? syz : sx2;
  const float dtt2 = dist2 * tanOA * tanOA;
  bool big = l2 > dtt2;
  for (int i = 0; i < 2; ++i)
    for (int j = 0; j < 2; ++j) {
      const float x1 = (i == 0 ? N.xmin[0] : N.xmax[0]) - lxc[0];
      const float y1 = (j == 0 ? N.xmin[1] : N.xmax[1]) - lxc[1];
      const float z1 = N.xmin[2] - lxc[2];
      const float x2 = (i == 0 ? N.xmax[0] : N.xmin[0]) - lxc[0];
      const float y2 = (j == 0 ? N.xmax[1] : N.xmin[1]) - lxc[1];
      const float z2 = N.xmax[2] - lxc[2];
      const float ddx = x1 - x2, ddy = y1 - y2, ddz = z1 - z2;
      const float dh2 = ddx * ddx + ddy * ddy + ddz * ddz;
      big = big || dh2 > dtt2;
    }
  return big;
}

// The list of one leaf by one wave.  The reference walks a LIFO one node at a
// time; what becomes of a node depends on the node and the leaf alone, so a
// wave takes the top 64 slots at once, decides all of them, puts the children
// of the opened nodes in their parent's place (right child on top, as the
// LIFO pops it first) and emits the segments above the first opened node --
// everything below it has to wait for that node's subtree and goes back on
// the stack, decided.  The segments come out in the LIFO's order, and the
// number of rounds is about the depth of the tree plus a 64th of the nodes
// looked at, each round one dependent node load, where one thread per walk
// took a round per node and the longest walk set the time (latency-bound
// still, but with every lane of a round in flight).  Count pass, before and
// now: 1.35 and 0.055 ms at 48^3 clustered with leaves of 128, 1.38 and 0.35
// ms at 256^3 with leaves of 512; the list phase 4.45 and 2.59 ms there.
//
// A round replaces k slots by at most 2 k, so the stack could grow by 64 a
// round; when fewer than stack_reserve slots are free above it, the wave
// walks one node at a time, whose height grows by at most one per level of
// the tree (stack_reserve covers the tree's depth).
template <bool FILL>
__global__ void __launch_bounds__(64)
k_walk(const hsr_node *__restrict__ t, const int32_t *__restrict__ leaves,
       const int32_t *__restrict__ leaf_box, const int64_t *__restrict__ cbase,
       const int32_t *__restrict__ nleaves, ListParams lp, int64_t *nseg_out, int64_t *nent_out,
       const int64_t *seg_ptr, int64_t *seg_a, int64_t *seg_b) {
  extern __shared__ int32_t stk[];
  uint8_t *kind = reinterpret_cast<uint8_t *>(stk + lp.stack_cap);
  const int64_t k = blockIdx.x;
  if (k >= *nleaves) {
    // slots past the listed leaves, and the one the scans end with, hold none
    if (!FILL && threadIdx.x == 0) nseg_out[k] = nent_out[k] = 0;
    return;
  }
  // fill pass: only the lists the cache does not hold whole
  if (FILL && nseg_out[k] - 1 <= lp.cache) return;
  const int l = lane_id();
  const int32_t tl = leaves[k];
  const int32_t root = (int32_t)cbase[leaf_box[k]];
  const hsr_node &L = t[tl];
  const int64_t toff = L.offset, tend = L.offset + L.count;
  const float lxc[3] = {L.xc[0], L.xc[1], L.xc[2]};
  const float lmin[3] = {L.xmin[0], L.xmin[1], L.xmin[2]};
  const float lmax[3] = {L.xmax[0], L.xmax[1], L.xmax[2]};
  const int64_t so = FILL ? seg_ptr[k] : 0;
  int64_t nseg = 0;   // emitted so far (uniform)
  int64_t nent = 0;   // this lane's share of their entries
  int h = 1;          // stack height (uniform)
  if (l == 0) {
    stk[0] = root;
    kind[0] = W_NODE;
  }
  __syncthreads();
  while (h > 0) {
    const int room = lp.stack_cap - h - lp.stack_reserve;
    const int b = room > 0 ? min(min(64, h), room) : 1;
    if (h >= lp.stack_cap) {  // unreachable while the reserve covers the depth
      if (l == 0) atomicAdd((unsigned long long *)lp.overflow, 1ull);
      break;
    }
    // this lane's slot, its outcome (the children to push or a segment)
    int nout = 0, k0 = W_RANGE, k1 = W_RANGE;
    int32_t v0 = 0, v1 = 0;
    int64_t sa = 0, sb = 0;
    if (l < b) {
      const int32_t id = stk[h - 1 - l];
      const int kd = kind[h - 1 - l];
      const hsr_node &N = t[id];
      const int64_t cnt = N.count, noff = N.offset;
      const int32_t cl = (int32_t)N.cl, cr = (int32_t)N.cr;
      v0 = id;
      if (kd >= W_RANGE) {
        nout = 1;
        k0 = kd;
      } else if (id < tl && noff <= toff && tend <= noff + cnt) {
        // an ancestor of the leaf: its children but the leaf
        if (cr > 0 && cr != tl) {
          v0 = cr;
          k0 = W_NODE;
          nout = 1;
        }
        if (cl > 0 && cl != tl) {
          (nout ? v1 : v0) = cl;
          (nout ? k1 : k0) = W_NODE;
          ++nout;
        }
      } else {
        bool near = cnt > 0 || id == root;  // the root of an empty box is looked at
        if (kd == W_NODE_GAP) {
          for (int i = 0; i < 3; ++i) {
            float dist = 0;
            if (lmax[i] < N.xmin[i]) dist = N.xmin[i] - lmax[i];
            else if (lmin[i] > N.xmax[i]) dist = lmin[i] - N.xmax[i];
            if (dist > lp.fsrrmax) near = false;
          }
        }
        if (near) {
          const float dx = N.xc[0] - lxc[0];
          const float dy = N.xc[1] - lxc[1];
          const float dz = N.xc[2] - lxc[2];
          const float dist2 = dx * dx + dy * dy + dz * dz;
          if (!looks_big(N, lxc, dist2, lp.tan_oa)) {
            if (!(dist2 > lp.fsrrmax2)) {
              nout = 1;
              k0 = cnt <= lp.tdpts ? W_RANGE : W_PSEUDO;
            }
          } else if (cr == 0 && cl == 0) {
            nout = 1;
            k0 = W_RANGE;
          } else {
            if (cr > 0) {
              v0 = cr;
              k0 = W_NODE_GAP;
              nout = 1;
            }
            if (cl > 0) {
              (nout ? v1 : v0) = cl;
              (nout ? k1 : k0) = W_NODE_GAP;
              ++nout;
            }
          }
        }
      }
      sa = k0 == W_PSEUDO ? (int64_t)id : noff;
      sb = k0 == W_PSEUDO ? -1 : cnt;
    }
    // the lanes before the first one that opened a node are done
    const uint64_t opened = __ballot(nout > 0 && k0 < W_RANGE);
    const int first = opened ? (int)__builtin_ctzll(opened) : 64;
    const bool emit = l < first && nout == 1;
    const uint64_t em = __ballot(emit);
    if (emit) {
      const int64_t s = nseg + __popcll(em & lanemask_lt());
      if (FILL) {
        seg_a[so + s] = sa;
        seg_b[so + s] = sb;
      } else {
        if (s < lp.cache) lp.cache_seg[k * lp.cache + s] = make_int2((int)sa, (int)sb);
        nent += sb < 0 ? lp.tdpts : sb;
      }
    }
    nseg += __popcll(em);
    // the rest go back on the stack, the first lane's on top
    const int np = l >= first ? nout : 0;
    const uint64_t p1 = __ballot(np >= 1), p2 = __ballot(np == 2);
    const int total = __popcll(p1) + __popcll(p2);
    const int before = __popcll(p1 & lanemask_lt()) + __popcll(p2 & lanemask_lt());
    __syncthreads();  // every slot has been read
    const int base = h - b + total - 1 - before;
    if (np >= 1) {
      stk[base] = v0;
      kind[base] = (uint8_t)k0;
    }
    if (np == 2) {
      stk[base - 1] = v1;
      kind[base - 1] = (uint8_t)k1;
    }
    h += total - b;
    __syncthreads();
  }
  if (!FILL) {
    nent = wave_sum_i64(nent);
    if (l == 0) {
      nseg_out[k] = nseg + 1;  // and the leaf's own particles
      nent_out[k] = nent + L.count;
    }
  }
}

// The segments of every listed leaf in place, with their entry offsets, and
// expanded into j indices (one wave per leaf): particle ranges by all lanes,
// the T pseudo-particles of node a as indices count + T a + j
// (RCBForceTree.cxx:1051-1060).  The segments come from the count pass's
// cache, or for the lists it does not hold whole from where the second walk
// left them; the leaf's own particles are the last segment.
__global__ void __launch_bounds__(64)
k_expand(int64_t nleaves, int64_t n, ListParams lp, const hsr_node *__restrict__ t,
         const int32_t *__restrict__ leaves, const int64_t *__restrict__ seg_ptr,
         int64_t *__restrict__ seg_a, int64_t *__restrict__ seg_b, int64_t *__restrict__ seg_e,
         const int64_t *__restrict__ ent_ptr, int32_t *__restrict__ jidx) {
  const int64_t k = blockIdx.x;
  if (k >= nleaves) return;
  const int l = lane_id();
  const int tdpts = lp.tdpts;
  const int64_t e0 = ent_ptr[k];
  const int64_t s0 = seg_ptr[k], s1 = seg_ptr[k + 1];
  const bool cached = s1 - s0 - 1 <= lp.cache;
  int64_t e = 0;
  // 64 segments at a time: lane i reads segment s + i, a wave prefix of
  // their entry counts places them, then they are written one by one
  for (int64_t s = s0; s < s1; s += 64) {
    const int64_t sl = s + l;
    int64_t a = 0, b = 0;
    if (sl == s1 - 1) {
      const hsr_node &L = t[leaves[k]];
      a = L.offset;
      b = L.count;
    } else if (sl < s1 && cached) {
      const int2 q = lp.cache_seg[k * lp.cache + (sl - s0)];
      a = q.x;
      b = q.y;
    } else if (sl < s1) {
      a = seg_a[sl];
      b = seg_b[sl];
    }
    const int64_t len = b < 0 ? (int64_t)tdpts : b;
    int64_t inc = len;  // inclusive prefix over the lanes
    for (int o = 1; o < 64; o <<= 1) {
      const int64_t y = (int64_t)__shfl_up((long long)inc, o);
      if (l >= o) inc += y;
    }
    if (sl < s1) {
      seg_a[sl] = a;
      seg_b[sl] = b;
      seg_e[sl] = e + inc - len;
    }
    const int m = (int)min<int64_t>(64, s1 - s);
    for (int j = 0; j < m; ++j) {
      const int32_t aj = readlane_i32((int32_t)a, j), bj = readlane_i32((int32_t)b, j);
      int32_t *out = jidx + e0 + e + (int64_t)readlane_u64((uint64_t)(inc - len), j);
      if (bj < 0) {
        if (l < tdpts) out[l] = (int32_t)(n + (int64_t)tdpts * aj + l);
      } else {
        for (int i = l; i < bj; i += 64) out[i] = aj + i;
      }
    }
    e += (int64_t)readlane_u64((uint64_t)inc, 63);
  }
}

__global__ void k_pairs(const int32_t *nleaves, const hsr_node *t, const int32_t *leaves,
                        const int64_t *nent, int64_t *pairs_out) {
  int64_t k = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  int64_t v = 0;
  if (k < *nleaves) v = t[leaves[k]].count * nent[k];
  v = wave_sum_i64(v);
  if (lane_id() == 0 && v)
    atomicAdd((unsigned long long *)pairs_out, (unsigned long long)v);
}

// What the host needs of the count pass, in one place: listed leaves,
// segments, entries (behind pairs and overflow).
__global__ void k_totals(const int32_t *nleaves, const int64_t *seg_total, const int64_t *ent_total,
                         int64_t *out) {
  if (threadIdx.x == 0) {
    out[2] = *nleaves;
    out[3] = *seg_total;
    out[4] = *ent_total;
  }
}

__global__ void k_zero_i64(int64_t *p, int64_t n) {
  int64_t k = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (k < n) p[k] = 0;
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

}  // namespace

// BFS node table -> listed leaves, per-leaf lists (segments + j indices).
hsr_status lists_build_device(hsr_ctx *c, const float *min_force_h,
                              const float *max_force_h) {
  hipStream_t st = c->stream;
  TreeState &T = c->tree;
  ListState &LS = c->lists;
  Scratch &S = c->s;
  const int64_t nb = T.nnodes_bfs, nboxes = T.nboxes, n = T.n;
  BNode *nodes = dptr<BNode>(T.bnodes);

  std::vector<int64_t> leaf_base(nboxes + 1, 0);
  for (int64_t b = 0; b < nboxes; ++b) leaf_base[b + 1] = leaf_base[b] + T.box_leaves[b];
  const int64_t nslots = leaf_base[nboxes];

  // device scratch: leaf_base, cbase, force boxes, slot arrays
  size_t need = sizeof(int64_t) * 2 * (nboxes + 1) + sizeof(float) * 6 * nboxes +
                sizeof(int32_t) * 4 * (nslots + 1) + 256;
  HSR_HIP(dbuf_reserve(S.g, need));
  int64_t *d_leaf_base = dptr<int64_t>(S.g);
  int64_t *d_cbase = d_leaf_base + nboxes + 1;
  float *d_fmin = reinterpret_cast<float *>(d_cbase + nboxes + 1);
  float *d_fmax = d_fmin + 3 * nboxes;
  int32_t *slot = reinterpret_cast<int32_t *>(d_fmax + 3 * nboxes);
  int32_t *flag = slot + nslots + 1;
  int32_t *pos = flag + nslots + 1;
  int32_t *slot_box = pos + nslots + 1;
  // one copy: the four tables lie behind one another
  const size_t nb1 = sizeof(int64_t) * (nboxes + 1), nf = sizeof(float) * 3 * nboxes;
  std::vector<char> tables(2 * nb1 + 2 * nf);
  memcpy(tables.data(), leaf_base.data(), nb1);
  memcpy(tables.data() + nb1, T.box_root.data(), nb1);
  memcpy(tables.data() + 2 * nb1, min_force_h, nf);
  memcpy(tables.data() + 2 * nb1 + nf, max_force_h, nf);
  HSR_HIP(hipMemcpyAsync(d_leaf_base, tables.data(), tables.size(), hipMemcpyHostToDevice, st));
  const int32_t *box_of = dptr<int32_t>(S.f);  // from the build

  // The number of listed leaves stays on the device (pos[nslots]) through the
  // count pass: its launches and buffers take a slot for every leaf, and the
  // host reads all totals once, before the fill.  (A host round trip costs
  // about 25 us, a small copy 8; the list and plan phases made five and
  // sixteen of them, now two and three: 0.28 -> 0.14 ms for 12k particles,
  // 0.35 -> 0.23 ms for 365k.)
  k_leaf_slots<<<nblk(nb, 256), 256, 0, st>>>(nodes, nb, box_of, d_leaf_base, d_fmin, d_fmax, slot, d_cbase);
  k_slot_box<<<(unsigned)nboxes, 256, 0, st>>>(nboxes, d_leaf_base, slot_box);
  k_flag_valid<<<nblk(nslots + 1, 256), 256, 0, st>>>(slot, nslots, flag);
  if (excl_scan(c, flag, pos, nslots + 1) != HSR_OK) return HSR_ERR_HIP;
  const int32_t *d_nl = pos + nslots;
  HSR_HIP(dbuf_reserve(LS.leaves, sizeof(int32_t) * (2 * nslots + 2)));
  int32_t *leaves = dptr<int32_t>(LS.leaves);
  int32_t *leaf_box = leaves + nslots + 1;
  k_compact<<<nblk(nslots, 256), 256, 0, st>>>(slot, flag, pos, nslots, leaves, leaf_box, slot_box);

  // ---- pass 1: counts
  HSR_HIP(dbuf_reserve(LS.seg_ptr, sizeof(int64_t) * (nslots + 1)));
  HSR_HIP(dbuf_reserve(LS.ent_ptr, sizeof(int64_t) * (nslots + 1)));
  HSR_HIP(dbuf_reserve(S.h, sizeof(int64_t) * 2 * (nslots + 1) + 64));
  int64_t *nseg = dptr<int64_t>(S.h);
  int64_t *nent = nseg + nslots + 1;
  ListParams lp;
  lp.fsrrmax = c->p.fsrrmax;
  lp.fsrrmax2 = c->p.fsrrmax * c->p.fsrrmax;
  lp.tan_oa = c->p.tan_oa;
  lp.tdpts = c->p.tdpts;
  // 1024 slots beside the reserve: 5.2 KB of LDS a wave
  lp.stack_reserve = (int)std::min<int64_t>(T.max_depth + 4, 8192);
  lp.stack_cap = 1024 + lp.stack_reserve;
  const size_t lds = ((sizeof(int32_t) + 1) * (size_t)lp.stack_cap + 15) / 16 * 16;
  // segment cache: up to 512 per leaf within 2 GiB (at 256^3, 0.2 GB)
  lp.cache = (int)std::min<int64_t>(512, ((int64_t)1 << 31) / ((int64_t)sizeof(int2) * std::max<int64_t>(1, nslots)));
  HSR_HIP(dbuf_reserve(LS.segcache, sizeof(int2) * (size_t)std::max(lp.cache, 1) * (size_t)std::max<int64_t>(1, nslots)));
  lp.cache_seg = dptr<int2>(LS.segcache);
  HSR_HIP(dbuf_reserve(S.counters, 256));
  int64_t *d_tot = dptr<int64_t>(S.counters) + 16;  // pairs, overflow, leaves, segments, entries
  lp.overflow = d_tot + 1;
  k_zero_i64<<<1, 64, 0, st>>>(d_tot, 2);
  const hsr_node *cn = dptr<hsr_node>(T.canon_nodes);
  k_walk<false><<<(unsigned)(nslots + 1), 64, lds, st>>>(cn, leaves, leaf_box, d_cbase, d_nl, lp, nseg, nent,
                                                         nullptr, nullptr, nullptr);
  if (excl_scan(c, nseg, dptr<int64_t>(LS.seg_ptr), nslots + 1) != HSR_OK) return HSR_ERR_HIP;
  if (excl_scan(c, nent, dptr<int64_t>(LS.ent_ptr), nslots + 1) != HSR_OK) return HSR_ERR_HIP;
  k_pairs<<<nblk(nslots, 64), 64, 0, st>>>(d_nl, cn, leaves, nent, d_tot);
  k_totals<<<1, 64, 0, st>>>(d_nl, dptr<int64_t>(LS.seg_ptr) + nslots, dptr<int64_t>(LS.ent_ptr) + nslots,
                             d_tot);
  int64_t tot[5];
  HSR_HIP(hipMemcpyAsync(tot, d_tot, sizeof(tot), hipMemcpyDeviceToHost, st));
  HSR_HIP(stream_wait(st));
  LS.pairs = tot[0];
  const int64_t nl = tot[2];
  LS.nleaves = nl;
  LS.nsegs = tot[3];
  LS.nentries = tot[4];
  if (tot[1]) {
    hsr_set_error("interaction-list walk exceeded its stack bound");
    return HSR_ERR_STATE;
  }
  // ---- pass 2: fill
  HSR_HIP(dbuf_reserve(LS.seg, sizeof(int64_t) * 3 * (LS.nsegs + 1)));
  int64_t *seg_a = dptr<int64_t>(LS.seg);
  int64_t *seg_b = seg_a + LS.nsegs + 1;
  int64_t *seg_e = seg_b + LS.nsegs + 1;
  HSR_HIP(dbuf_reserve(LS.jidx, sizeof(int32_t) * (LS.nentries + 1)));
  if (nl > 0) {
    k_walk<true><<<(unsigned)nl, 64, lds, st>>>(cn, leaves, leaf_box, d_cbase, d_nl, lp, nseg, nullptr,
                                                dptr<int64_t>(LS.seg_ptr), seg_a, seg_b);
    k_expand<<<(unsigned)nl, 64, 0, st>>>(nl, n, lp, cn, leaves, dptr<int64_t>(LS.seg_ptr), seg_a, seg_b,
                                          seg_e, dptr<int64_t>(LS.ent_ptr), dptr<int32_t>(LS.jidx));
  }
  HSR_HIP(hipGetLastError());
  return HSR_OK;
}
