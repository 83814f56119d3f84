// Adaptive octree (reference: include/build_tree_tbb.h:36-374), built on the
// device from sorted path keys.  Compiled with -ffp-contract=off.
//
// Reference semantics reproduced:
//   * a node with more than ncrit bodies is split; its bodies are partitioned
//     stably by octant (x > Xc) + ((y > Yc) << 1) + ((z > Zc) << 2)
//     (CountBodies/MoveBodies, :52-116, a stable out-of-place scatter);
//   * child centres are X +- R0 / 2^(level+1) (:199-203), empty octants get
//     no node;
//   * cells are numbered as Nodes2cells does (:250-294): root 0, each node's
//     children form one block at the running cursor, and child i's subtree
//     block follows the blocks of children 0..i-1;
//   * R = R0 / 2^level, ICELL = level offset + Morton interleave of the
//     centre (:240-249; computed in 64 bits, the reference's int overflows
//     beyond level 10).
//
// A node's centre depends on its path alone, so every body finds the octants
// of its whole path by itself, with the operations that a level-by-level
// partition would use, as a key of 3 bits per level.  One stable sort by the
// key puts every node's bodies side by side; a node's children are the digit
// boundaries in its range (found by bisection), level by level on the device;
// and since a stable partition keeps the input order inside a leaf, each
// leaf's bodies are finally put in the order of their indices.  (A stable sort
// of the active bodies per level, with a read-back, took 12 to 25 launches a
// level.  Build times by HIP events with the profiler attached: 250 000 Plummer
// bodies, 9 levels, 4.1 -> 0.43 ms; 4 M, 11 levels, 5.0 -> 0.71 ms.)
#include <algorithm>
#include <cmath>

#include "device_util.h"
#include "internal.h"

namespace exafmm {

namespace {

constexpr int kDepth = 20;      // splits along a path (60 key bits)
constexpr int kTreeGrid = 512;  // workgroups of the level kernels
constexpr int kTreeBlock = 256;
constexpr int kTreeSmall = 128;  // levels of up to this many splitting nodes run in one workgroup

constexpr int kPinTree = 128;   // words of Handle::hpin that receive the state

// The build's progress, on the device.  A level's splitting nodes ("active")
// are act[sel]; act[1 - sel] receives the next level's.
struct TreeState {
  int total, nact, lev, sel;
  int overflow;     // the node arrays or lists were too small
  int done_blocks;  // k_tree_emit workgroups finished (the last one advances the level)
  int bad;          // cells that failed the structural check
  int pad;
  double R0;
  int first[kDepth + 2];   // first node of each level (the last entry used: total)
  int nsplit[kDepth + 2];  // splitting nodes of each level
};
static_assert(kPinTree * sizeof(int) + sizeof(TreeState) <= Handle::kPinBounds * sizeof(int), "pinned words");

// Nodes in creation order: level by level, (parent, octant) within a level.
struct Nodes {
  double4 *X;
  int *start, *count, *parent, *level, *first, *nchild;
  int *act[2];
  int *lo;  // first body of each octant of the active nodes
  int cap, cap_act;
};

// bounds2box (build_tree_tbb.h:298-310): box = centre, R0 (after the bounds).
__global__ void k_tree_init(const double *__restrict__ bb, double *__restrict__ box, int n, int ncrit, Nodes nd,
                            TreeState *__restrict__ st) {
  double Xc[3], R0 = 0;
  for (int d = 0; d < 3; d++) Xc[d] = (bb[3 + d] + bb[d]) / 2;
  for (int d = 0; d < 3; d++) {  // std::max(a, R0) = a < R0 ? R0 : a
    const double a = Xc[d] - bb[d], b = bb[3 + d] - Xc[d];
    R0 = a < R0 ? R0 : a;
    R0 = b < R0 ? R0 : b;
  }
  R0 *= 1.00001;
  for (int d = 0; d < 3; d++) box[d] = Xc[d];
  box[3] = R0;
  nd.X[0] = make_double4(Xc[0], Xc[1], Xc[2], 0);
  nd.start[0] = 0;
  nd.count[0] = n;
  nd.parent[0] = -1;
  nd.level[0] = 0;
  nd.first[0] = 0;
  nd.nchild[0] = 0;
  nd.act[0][0] = 0;
  st->total = 1;
  st->nact = n > ncrit ? 1 : 0;
  st->lev = st->sel = st->overflow = st->done_blocks = st->bad = 0;
  st->R0 = R0;
  for (int l = 0; l < kDepth + 2; l++) st->first[l] = st->nsplit[l] = 0;
  st->first[1] = 1;
  st->nsplit[0] = st->nact;
}

// Octants of the body's path, the root's in the highest of the 60 bits.
__global__ void __launch_bounds__(256)
    k_path_keys(const double4 *__restrict__ body, int n, const double *__restrict__ box, int levels,
                uint64_t *__restrict__ key, int *__restrict__ idx) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const double4 x = body[i];
  double cx = box[0], cy = box[1], cz = box[2], r = box[3];
  uint64_t k = 0;
  for (int l = 0; l < levels; l++) {
    r *= 0.5;
    const int ox = x.x > cx, oy = x.y > cy, oz = x.z > cz;
    k = k << 3 | (uint64_t)(ox + (oy << 1) + (oz << 2));
    cx = cx + r * (ox * 2 - 1);
    cy = cy + r * (oy * 2 - 1);
    cz = cz + r * (oz * 2 - 1);
  }
  key[i] = k << 3 * (kDepth - levels);
  idx[i] = i;
}

// First body of octant o of the node with bodies [b, e) at level lev: the
// range shares its higher digits, so it is sorted by this one.
__device__ inline int octant_begin(const uint64_t *__restrict__ key, int b, int e, int lev, int o) {
  const int shift = 3 * (kDepth - 1 - lev);
  while (b < e) {
    const int mid = (b + e) >> 1;
    if ((int)(key[mid] >> shift & 7) < o)
      b = mid + 1;
    else
      e = mid;
  }
  return b;
}

__device__ inline void put_child(const Nodes &nd, int parent, int o, int b, int cnt, int lev, double r, int child,
                                 bool split, int *next_act, int at) {
  const double4 P = nd.X[parent];
  nd.X[child] = make_double4(P.x + r * ((o & 1) * 2 - 1), P.y + r * (((o >> 1) & 1) * 2 - 1),
                             P.z + r * (((o >> 2) & 1) * 2 - 1), 0);
  nd.start[child] = b;
  nd.count[child] = cnt;
  nd.parent[child] = parent;
  nd.level[child] = lev + 1;
  nd.first[child] = 0;
  nd.nchild[child] = 0;
  if (split) next_act[at] = child;
}

// 8 lanes per active node, one per octant: the octant's bodies [lo, lo + cnt).
__device__ inline void octant_range(const Nodes &nd, const uint64_t *__restrict__ key, int node, int lev, int o,
                                    int &lo, int &cnt) {
  const int b = nd.start[node], e = b + nd.count[node];
  lo = o == 0 ? b : octant_begin(key, b, e, lev, o);
  const int hi = __shfl_down(lo, 1);
  cnt = (o == 7 ? e : hi) - lo;
}

// The first levels, while they have 1 to kTreeSmall splitting nodes (and
// another digit was sorted), in one workgroup.
__global__ void __launch_bounds__(8 * kTreeSmall)
    k_tree_small(Nodes nd, const uint64_t *__restrict__ key, int ncrit, int levels, TreeState *__restrict__ st) {
  __shared__ TreeState s;
  if (threadIdx.x == 0) s = *st;
  __syncthreads();
  const int r = threadIdx.x / 8, o = threadIdx.x % 8;
  while (s.nact > 0 && s.nact <= kTreeSmall && s.lev < levels) {
    const int lev = s.lev, sel = s.sel, total = s.total, nact = s.nact;
    const double rad = s.R0 / (double)(1 << (lev + 1));
    const bool on = r < nact;
    const int node = on ? nd.act[sel][r] : 0;
    int lo = 0, cnt = 0;
    octant_range(nd, key, node, lev, o, lo, cnt);
    const bool child = on && cnt > 0, split = on && cnt > ncrit;
    int4 tot;
    const int4 at = block_exscan4<8 * kTreeSmall>(make_int4(child, split, 0, 0), &tot);
    if (total + tot.x > nd.cap || tot.y > nd.cap_act) {
      if (threadIdx.x == 0) {
        s.overflow = 1;
        s.nact = 0;
      }
      __syncthreads();
      break;
    }
    if (child) put_child(nd, node, o, lo, cnt, lev, rad, total + at.x, split, nd.act[1 - sel], at.y);
    const int nch = (int)__popcll(__ballot(child) >> (threadIdx.x / 8 * 8 & 63) & 255);
    if (on && o == 0) {
      nd.first[node] = total + at.x;
      nd.nchild[node] = nch;
    }
    __threadfence_block();
    __syncthreads();
    if (threadIdx.x == 0) {
      s.total = total + tot.x;
      s.nact = tot.y;
      s.lev = lev + 1;
      s.sel = 1 - sel;
      s.first[lev + 2] = s.total;
      s.nsplit[lev + 1] = tot.y;
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) *st = s;
}

// One level over kTreeGrid workgroups, each with a contiguous chunk of the
// active nodes: the octants' bodies and the workgroup's child and split
// counts, then (second kernel) the children at offsets from those counts.
__device__ inline void tree_chunk(int nact, int &i0, int &i1) {
  constexpr int kPer = kTreeBlock / 8;
  const int c = ((nact + kTreeGrid - 1) / kTreeGrid + kPer - 1) / kPer * kPer;
  i0 = min(nact, (int)blockIdx.x * c);
  i1 = min(nact, i0 + c);
}

__global__ void __launch_bounds__(kTreeBlock)
    k_tree_split(Nodes nd, const uint64_t *__restrict__ key, int ncrit, int levels, const TreeState *__restrict__ st,
                 int2 *__restrict__ blk) {
  const int nact = st->lev < levels ? st->nact : 0, lev = st->lev;
  const int *act = nd.act[st->sel];
  int i0, i1;
  tree_chunk(nact, i0, i1);
  const int o = threadIdx.x % 8;
  int4 sum = make_int4(0, 0, 0, 0);
  for (int i = i0; i < i1; i += kTreeBlock / 8) {
    const int r = i + threadIdx.x / 8;
    const bool on = r < i1;
    int lo = 0, cnt = 0;
    octant_range(nd, key, on ? act[r] : act[i0], lev, o, lo, cnt);
    if (on) {
      nd.lo[8 * r + o] = lo;
      sum.x += cnt > 0;
      sum.y += cnt > ncrit;
    }
  }
  int4 tot;
  block_exscan4<kTreeBlock>(sum, &tot);
  if (threadIdx.x == 0) blk[blockIdx.x] = make_int2(tot.x, tot.y);
}

__global__ void __launch_bounds__(kTreeBlock)
    k_tree_emit(Nodes nd, int ncrit, int levels, TreeState *__restrict__ st, const int2 *__restrict__ blk) {
  __shared__ int4 sbase;
  __shared__ int slast;
  const int nact = st->lev < levels ? st->nact : 0, lev = st->lev, sel = st->sel, total = st->total;
  const double rad = st->R0 / (double)(1 << (lev + 1));
  const int *act = nd.act[sel];
  int4 tot;
  {
    constexpr int kPer = kTreeGrid / kTreeBlock;
    int4 v[kPer], sum = make_int4(0, 0, 0, 0);
    for (int k = 0; k < kPer; k++) {
      const int2 b = blk[threadIdx.x * kPer + k];
      v[k] = make_int4(b.x, b.y, 0, 0);
      sum = add4(sum, v[k]);
    }
    int4 r = block_exscan4<kTreeBlock>(sum, &tot);
    for (int k = 0; k < kPer; k++) {
      if (threadIdx.x * kPer + k == (int)blockIdx.x) sbase = r;
      r = add4(r, v[k]);
    }
  }
  __syncthreads();
  const bool ok = total + tot.x <= nd.cap && tot.y <= nd.cap_act;
  int i0, i1;
  tree_chunk(nact, i0, i1);
  if (!ok) i1 = i0;
  const int o = threadIdx.x % 8;
  int4 run = sbase;
  for (int i = i0; i < i1; i += kTreeBlock / 8) {
    const int r = i + threadIdx.x / 8;
    const bool on = r < i1;
    const int node = on ? act[r] : act[i0];
    const int lo = on ? nd.lo[8 * r + o] : 0, hi = __shfl_down(lo, 1);
    const int cnt = on ? (o == 7 ? nd.start[node] + nd.count[node] : hi) - lo : 0;
    const bool child = cnt > 0, split = cnt > ncrit;
    int4 t;
    const int4 at = add4(block_exscan4<kTreeBlock>(make_int4(child, split, 0, 0), &t), run);
    run = add4(run, t);
    if (child) put_child(nd, node, o, lo, cnt, lev, rad, total + at.x, split, nd.act[1 - sel], at.y);
    const int nch = (int)__popcll(__ballot(child) >> (threadIdx.x / 8 * 8 & 63) & 255);
    if (on && o == 0) {
      nd.first[node] = total + at.x;
      nd.nchild[node] = nch;
    }
  }
  __syncthreads();
  if (threadIdx.x == 0) slast = atomicAdd(&st->done_blocks, 1) == (int)gridDim.x - 1;
  __syncthreads();
  if (slast && threadIdx.x == 0) {  // every workgroup has read the state by now
    st->done_blocks = 0;
    if (!ok) {
      st->overflow = 1;
      st->nact = 0;
    } else if (nact > 0) {
      st->total = total + tot.x;
      st->nact = tot.y;
      st->lev = lev + 1;
      st->sel = 1 - sel;
      st->first[lev + 2] = total + tot.x;
      st->nsplit[lev + 1] = tot.y;
    }
  }
}

// Nodes2cells lays the blocks of children out in depth-first order of their
// parents, which is the order of (first body, level).  So a node's block
// starts after the blocks of all splitting nodes that begin at an earlier
// body (a prefix sum over the bodies) and of its ancestors that begin at its
// own first body.
//
// These kernels are launched before the host knows the number of nodes: they
// take it from the state of a finished build (0 otherwise), up to what the
// cell arrays hold.
__device__ inline int node_count(const TreeState *st, int room) {
  return st->nact == 0 && !st->overflow && st->total <= room ? st->total : 0;
}

__global__ void k_block_sizes(Nodes nd, const TreeState *__restrict__ st, int room, int *__restrict__ size) {
  const int g = blockIdx.x * blockDim.x + threadIdx.x;
  if (g < node_count(st, room) && nd.nchild[g] > 0) atomicAdd(&size[nd.start[g]], nd.nchild[g]);
}

__device__ inline int block_begin(const Nodes &nd, const int *__restrict__ before, int g) {
  const int s = nd.start[g];
  int at = 1 + before[s];
  for (int p = nd.parent[g]; p >= 0 && nd.start[p] == s; p = nd.parent[p]) at += nd.nchild[p];
  return at;
}

__global__ void k_emit_cells(Nodes nd, const TreeState *__restrict__ st, int room, const int *__restrict__ before,
                             const double *__restrict__ box,
                             double4 *__restrict__ cX, double *__restrict__ cRb, int *__restrict__ cParent,
                             int *__restrict__ cChild, int *__restrict__ cNChild, int *__restrict__ cBody,
                             int *__restrict__ cNBody, uint64_t *__restrict__ cKey, int *__restrict__ cLevel,
                             int *__restrict__ lvl_cells) {
  const int g = blockIdx.x * blockDim.x + threadIdx.x, total = node_count(st, room);
  if (g >= total) return;
  // The cell of a node: its parent's block, then its place among the siblings.
  auto cell_of = [&](int v) {
    const int p = nd.parent[v];
    return p < 0 ? 0 : block_begin(nd, before, p) + (v - nd.first[p]);
  };
  const int c = cell_of(g);
  if (c < 0 || c >= total) return;  // caught by k_validate
  const int lev = nd.level[g];
  const double R0 = box[3], x0 = box[0] - R0, y0 = box[1] - R0, z0 = box[2] - R0;
  const double R = R0 / (1 << lev);
  double4 Xc = nd.X[g];
  Xc.w = R;
  cX[c] = Xc;
  cRb[c] = R;
  cParent[c] = nd.parent[g] >= 0 ? cell_of(nd.parent[g]) : 0;
  const int nch = nd.nchild[g];
  cChild[c] = nch > 0 ? block_begin(nd, before, g) : 0;
  cNChild[c] = nch;
  cBody[c] = nd.start[g];
  cNBody[c] = nd.count[g];
  cLevel[c] = lev;
  // getKey (:240-249), 64-bit.
  const double diameter = 2 * R;
  int64_t ix = (int64_t)(int)((Xc.x - x0) / diameter);
  int64_t iy = (int64_t)(int)((Xc.y - y0) / diameter);
  int64_t iz = (int64_t)(int)((Xc.z - z0) / diameter);
  uint64_t index = ((1ULL << (3 * lev)) - 1) / 7;
  for (int l = 0; l < lev; l++) {
    index += (uint64_t)(ix & 1) << (3 * l);
    index += (uint64_t)(iy & 1) << (3 * l + 1);
    index += (uint64_t)(iz & 1) << (3 * l + 2);
    ix >>= 1;
    iy >>= 1;
    iz >>= 1;
  }
  cKey[c] = index;
  lvl_cells[g] = c;
}

// Structural check of a finished tree: every cell written, parent and child
// ranges inside the cell array, body ranges inside the body array, and the
// cell's children pointing back to it.  Violations are counted.
__global__ void k_validate(TreeState *__restrict__ st, int room, int n, const int *__restrict__ cParent,
                           const int *__restrict__ cChild, const int *__restrict__ cNChild,
                           const int *__restrict__ cBody, const int *__restrict__ cNBody) {
  const int c = blockIdx.x * blockDim.x + threadIdx.x, nc = node_count(st, room);
  if (c >= nc) return;
  const int p = cParent[c], ch = cChild[c], nch = cNChild[c], b = cBody[c], nb = cNBody[c];
  bool ok = p >= 0 && p < nc && nch >= 0 && nch <= 8 && b >= 0 && nb >= 0 && b + nb <= n;
  if (ok && nch > 0) {
    ok = ch > c && ch + nch <= nc;
    for (int k = 0; ok && k < nch; k++) ok = cParent[ch + k] == c;
  }
  if (!ok) atomicAdd(&st->bad, 1);
}

// Each leaf's bodies in the order of their indices, one wave a leaf, where no
// leaf is larger than that takes well (kRangeRank).
__global__ void __launch_bounds__(64)
    k_leaf_bodies(int g0, Nodes nd, const TreeState *__restrict__ st, int room, int bits, int *__restrict__ idx,
                  int *__restrict__ aux, const double4 *__restrict__ in, double4 *__restrict__ body,
                  int *__restrict__ bidx) {
  __shared__ RangeSortLds sh;
  const int g = g0 + blockIdx.x;
  if (g >= node_count(st, room) || nd.nchild[g] != 0) return;
  const int b = nd.start[g];
  sort_range(idx + b, aux + b, nd.count[g], bits, sh, [&](int rank, int e) {
    body[b + rank] = in[e];
    bidx[b + rank] = e;
  });
}

// Larger leaves: key[e] = the first body of body e's leaf, for a stable sort of
// (key, e) in input order.  (100000 bodies, a leaf for all or ncrit = 20000: 3650
// and 570 us a build by one wave a leaf, 71 and 170 so.)
__global__ void __launch_bounds__(256)
    k_leaf_keys(Nodes nd, const TreeState *__restrict__ st, int room, const int *__restrict__ idx,
                int *__restrict__ key, int *__restrict__ val) {
  const int total = node_count(st, room);
  for (int g = blockIdx.x; g < total; g += gridDim.x) {
    if (nd.nchild[g] != 0) continue;
    const int b = nd.start[g], n = nd.count[g];
    for (int i = threadIdx.x; i < n; i += 256) {
      const int e = idx[b + i];
      key[e] = b;
      val[e] = e;
    }
  }
}

// The bodies in the order ord (only written for a finished build).
__global__ void __launch_bounds__(256)
    k_body_gather(const TreeState *__restrict__ st, int room, const int *__restrict__ ord, int n,
                  const double4 *__restrict__ in, double4 *__restrict__ body, int *__restrict__ bidx) {
  const int p = blockIdx.x * 256 + threadIdx.x;
  if (p >= n || node_count(st, room) == 0) return;
  const int e = ord[p];
  body[p] = in[e];
  bidx[p] = e;
}

constexpr const char *kDegenerate = "build_tree: degenerate bounds (box radius 0)";

}  // namespace

void run_build_adaptive(Handle &h) {
  const int n = h.n, ncrit = h.cfg.ncrit;
  const int T = 256;
  if (!h.bounds_pending) {  // (otherwise the device's radius is read back)
    bool extent = false;
    for (int d = 0; d < 3; d++) extent = extent || h.xmax[d] > h.xmin[d];
    if (!extent) throw Error(EXAFMM_HIP_EINVAL, kDegenerate);
  }
  h.drop_tree();
  upload_bounds(h);
  h.body4.resize(n);
  h.bidx.resize(n);
  h.trg4.resize(n);
  h.k64a.reserve(n + 1);
  h.k64b.reserve(n + 1);
  h.ia.reserve(n + 1);
  h.ib.reserve(n + 1);
  h.at_blk.reserve(2 * kTreeGrid);
  h.at_state.reserve(sizeof(TreeState));
  TreeState *st = reinterpret_cast<TreeState *>(h.at_state.p);
  int2 *blk = reinterpret_cast<int2 *>(h.at_blk.p);
  double *box = h.box.p + 8;
  size_t cap = std::max<size_t>(2 * (size_t)(n / std::max(ncrit, 1)) * 8 + 1024, h.at_cap);
  // Digits to sort: all of them, or one more than the last tree of this handle
  // split (fewer sort passes); a deeper tree is built again with all.
  int levels = h.at_depth > 0 ? std::min(kDepth, h.at_depth + 1) : kDepth;
  TreeState hs;
  Nodes nd;
  int bits = 1;
  while (((int64_t)1 << bits) < n) bits++;
  const uint64_t *key = nullptr;
  uint64_t *spare = nullptr;  // the keys' other buffer
  int *idx = nullptr, *aux = nullptr;
  const bool one = n <= ncrit;  // the root is a leaf: its bodies stay in input order
  // The cells of up to `room` nodes, the bodies in tree order and the check.
  auto emit = [&](int room) {
    h.cX.reserve(room);
    h.cRb.reserve(room);
    h.cParent.reserve(room);
    h.cChild.reserve(room);
    h.cNChild.reserve(room);
    h.cBody.reserve(room);
    h.cNBody.reserve(room);
    h.cKey.reserve(room);
    h.cLevel.reserve(room);
    h.lvl_cells.reserve(room);
    h.ic.reserve((size_t)n + 2);
    h.id.reserve((size_t)n + 2);
    const int *ord = idx;
    if (!one && ncrit <= kRangeRank) {
      launch_ranges(room, 64, [&](int g, int cnt) {
        hipLaunchKernelGGL(k_leaf_bodies, dim3(cnt), dim3(64), 0, h.stream, g, nd, st, room, bits, idx, aux, h.in4.p,
                           h.body4.p, h.bidx.p);
      });
      ord = nullptr;
    } else if (!one) {
      int *k = reinterpret_cast<int *>(spare);
      h.ie.reserve(n + 1);
      hipLaunchKernelGGL(k_leaf_keys, dim3(std::min(room, 1 << 20)), dim3(T), 0, h.stream, nd, st, room, idx, k, aux);
      bool alt = false;
      sort_pairs_int_int(k, k + n + 1, aux, h.ie.p, n, bits, alt, h.stream, h.tmp);
      ord = alt ? h.ie.p : aux;
    }
    if (ord)
      hipLaunchKernelGGL(k_body_gather, dim3(div_up(n, T)), dim3(T), 0, h.stream, st, room, ord, n, h.in4.p, h.body4.p,
                         h.bidx.p);
    if (!one) {
      zero_device(h.ic.p, ((size_t)n + 1) / 2 * 8, h.stream);
      hipLaunchKernelGGL(k_block_sizes, dim3(div_up(room, T)), dim3(T), 0, h.stream, nd, st, room, h.ic.p);
      exclusive_scan_int(h, h.ic.p, h.id.p, n);
    }
    EXA_HIP(hipMemsetAsync(h.cNChild.p, 0xff, room * sizeof(int), h.stream));  // -1: not written
    hipLaunchKernelGGL(k_emit_cells, dim3(div_up(room, T)), dim3(T), 0, h.stream, nd, st, room, h.id.p, box, h.cX.p,
                       h.cRb.p, h.cParent.p, h.cChild.p, h.cNChild.p, h.cBody.p, h.cNBody.p, h.cKey.p, h.cLevel.p,
                       h.lvl_cells.p);
    hipLaunchKernelGGL(k_validate, dim3(div_up(room, T)), dim3(T), 0, h.stream, st, room, n, h.cParent.p, h.cChild.p,
                       h.cNChild.p, h.cBody.p, h.cNBody.p);
    EXA_HIP(hipGetLastError());
  };
  auto read_state = [&] {
    EXA_HIP(hipMemcpyAsync(h.hpin + kPinTree, st, sizeof(TreeState), hipMemcpyDeviceToHost, h.stream));
    EXA_HIP(hipStreamSynchronize(h.stream));
    hs = *reinterpret_cast<const TreeState *>(h.hpin + kPinTree);
  };
  bool emitted = false;
  while (true) {
    if (cap > INT_MAX) throw Error(EXAFMM_HIP_EUNSUP, "adaptive tree: too many nodes");
    h.at_X.reserve(cap);
    for (auto *b : {&h.at_start, &h.at_count, &h.at_parent, &h.at_level, &h.at_first, &h.at_nchild, &h.at_act0,
                    &h.at_act1})
      b->reserve(cap);
    h.at_lo.reserve(8 * cap);
    nd = Nodes{h.at_X.p, h.at_start.p, h.at_count.p, h.at_parent.p, h.at_level.p, h.at_first.p, h.at_nchild.p,
               {h.at_act0.p, h.at_act1.p}, h.at_lo.p, (int)cap, (int)cap};
    hipLaunchKernelGGL(k_tree_init, dim3(1), dim3(1), 0, h.stream, h.box.p, box, n, ncrit, nd, st);
    hipLaunchKernelGGL(k_path_keys, dim3(div_up(n, T)), dim3(T), 0, h.stream, h.in4.p, n, box, levels, h.k64a.p,
                       h.ia.p);
    bool alt = false;
    if (!one) sort_pairs_u64_int(h, h.k64a.p, h.k64b.p, h.ia.p, h.ib.p, n, 3 * (kDepth - levels), 3 * kDepth, alt);
    key = alt ? h.k64b.p : h.k64a.p;
    spare = alt ? h.k64a.p : h.k64b.p;
    idx = alt ? h.ib.p : h.ia.p;
    aux = alt ? h.ia.p : h.ib.p;
    hipLaunchKernelGGL(k_tree_small, dim3(1), dim3(8 * kTreeSmall), 0, h.stream, nd, key, ncrit, levels, st);
    // The other levels without waiting for any: as many as the last tree had
    // after its small ones, and then the cells, for as many as the last tree
    // had and a quarter more; what was not enough is done after the read-back.
    int batch = h.at_depth > 0 ? h.at_big : 4;
    const int room = h.at_total > 0 ? (int)std::min<int64_t>(h.at_total + h.at_total / 4 + 64, INT_MAX) : 0;
    while (true) {
      for (int l = 0; l < batch; l++) {
        hipLaunchKernelGGL(k_tree_split, dim3(kTreeGrid), dim3(kTreeBlock), 0, h.stream, nd, key, ncrit, levels, st,
                           blk);
        hipLaunchKernelGGL(k_tree_emit, dim3(kTreeGrid), dim3(kTreeBlock), 0, h.stream, nd, ncrit, levels, st, blk);
      }
      if (room > 0) emit(room);
      read_state();
      emitted = room > 0 && hs.nact == 0 && !hs.overflow && hs.total <= room;
      if (hs.overflow || hs.nact == 0 || hs.lev >= levels) break;
      batch = 4;
    }
    if (!(hs.R0 > 0)) throw Error(EXAFMM_HIP_EINVAL, kDegenerate);
    if (hs.overflow) {
      cap *= 2;
      continue;
    }
    if (hs.nact == 0) break;
    if (levels == kDepth)
      throw Error(EXAFMM_HIP_EUNSUP, "adaptive tree deeper than 20 levels (more than ncrit coincident bodies?)");
    levels = kDepth;
  }
  const int total = hs.total;
  if (!emitted) {
    emit(total);
    read_state();
  }
  h.at_cap = cap;
  h.at_depth = std::max(1, hs.lev);
  h.at_total = total;
  h.at_big = 0;
  for (int l = 0; l < hs.lev && h.at_big == 0; l++)
    if (hs.nsplit[l] > kTreeSmall) h.at_big = hs.lev - l;
  h.ncells = total;
  h.nlevels = hs.lev + 1;
  h.lvl_off.assign(h.nlevels + 1, 0);
  h.lvl_par.assign(h.nlevels, 0);
  for (int l = 0; l < h.nlevels; l++) {
    h.lvl_off[l + 1] = hs.first[l + 1];
    h.lvl_par[l] = hs.nsplit[l];
  }
  h.leaf_level = 0;
  h.cX.resize(total);
  h.cRb.resize(total);
  h.cParent.resize(total);
  h.cChild.resize(total);
  h.cNChild.resize(total);
  h.cBody.resize(total);
  h.cNBody.resize(total);
  h.cKey.resize(total);
  h.cLevel.resize(total);
  h.lvl_cells.resize(total);
  if (hs.bad)
    throw Error(EXAFMM_HIP_EDEVICE, "adaptive tree failed its structural check (" + std::to_string(hs.bad) + " cells)");
}

}  // namespace exafmm
