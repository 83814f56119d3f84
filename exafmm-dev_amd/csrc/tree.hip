// Bounds and the uniform Morton-key tree (reference: include/bound_box.h and
// include/build_tree_omp.h).  Compiled with -ffp-contract=off: keys, cell
// centres and radii must round exactly as the reference does on x86-64.
//
// Layout produced (identical to build_tree_omp.h after reverseOrder,
// :200-211): cells are level-contiguous, root first; inside a level they run
// in descending Morton order; bodies run in ascending Morton order (stable).
#include <algorithm>
#include <climits>
#include <cmath>

#include "device_util.h"
#include "internal.h"

namespace exafmm {

// ---------------------------------------------------------------------------
// Bounds: grid-stride min/max, one partial per block, then one block.
constexpr int kBoundsBlocks = 512;
constexpr int kBoundsOne = 4096;  // bodies up to which one block is no slower than a second launch

// (host: with one block, the pinned copy of the result.)
__global__ void __launch_bounds__(256) k_bounds_partial(const double4 *__restrict__ b, int n, double *__restrict__ part,
                                                        double *__restrict__ host) {
  __shared__ double s[6][256];
  double mn[3] = {b[0].x, b[0].y, b[0].z};
  double mx[3] = {mn[0], mn[1], mn[2]};
  for (int i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256) {
    const double4 v = b[i];
    mn[0] = v.x < mn[0] ? v.x : mn[0];
    mn[1] = v.y < mn[1] ? v.y : mn[1];
    mn[2] = v.z < mn[2] ? v.z : mn[2];
    mx[0] = v.x > mx[0] ? v.x : mx[0];
    mx[1] = v.y > mx[1] ? v.y : mx[1];
    mx[2] = v.z > mx[2] ? v.z : mx[2];
  }
  for (int d = 0; d < 3; d++) {
    s[d][threadIdx.x] = mn[d];
    s[3 + d][threadIdx.x] = mx[d];
  }
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) {
      for (int d = 0; d < 3; d++) {
        const double a = s[d][threadIdx.x + w];
        s[d][threadIdx.x] = a < s[d][threadIdx.x] ? a : s[d][threadIdx.x];
        const double c = s[3 + d][threadIdx.x + w];
        s[3 + d][threadIdx.x] = c > s[3 + d][threadIdx.x] ? c : s[3 + d][threadIdx.x];
      }
    }
    __syncthreads();
  }
  if (threadIdx.x < 6) part[blockIdx.x * 6 + threadIdx.x] = s[threadIdx.x][0];
  if (host && threadIdx.x < 6) host[threadIdx.x] = s[threadIdx.x][0];
}

__global__ void __launch_bounds__(256) k_bounds_final(const double *__restrict__ part, int nb, double *__restrict__ out,
                                                      double *__restrict__ host) {
  __shared__ double s[6][256];
  double r[6];
  for (int d = 0; d < 6; d++) r[d] = part[d];
  for (int i = threadIdx.x; i < nb; i += 256)
    for (int d = 0; d < 3; d++) {
      const double a = part[6 * i + d], c = part[6 * i + 3 + d];
      r[d] = a < r[d] ? a : r[d];
      r[3 + d] = c > r[3 + d] ? c : r[3 + d];
    }
  for (int d = 0; d < 6; d++) s[d][threadIdx.x] = r[d];
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w)
      for (int d = 0; d < 3; d++) {
        const double a = s[d][threadIdx.x + w], c = s[3 + d][threadIdx.x + w];
        s[d][threadIdx.x] = a < s[d][threadIdx.x] ? a : s[d][threadIdx.x];
        s[3 + d][threadIdx.x] = c > s[3 + d][threadIdx.x] ? c : s[3 + d][threadIdx.x];
      }
    __syncthreads();
  }
  if (threadIdx.x < 6) out[threadIdx.x] = host[threadIdx.x] = s[threadIdx.x][0];
}

// The bounds stay on the device for the builder; the host copy (xmin,
// xmax) arrives behind ev_bounds and is read by sync_bounds when needed.
void run_bounds(Handle &h) {
  h.box.reserve(16);
  h.bounds_dev_stale = h.bounds_given = false;
  if (h.n == 0) {
    sync_bounds(h);
    for (int d = 0; d < 3; d++) h.xmin[d] = h.xmax[d] = 0;
    h.bounds_dev_stale = true;
    h.have_bounds = true;
    return;
  }
  double *host = reinterpret_cast<double *>(h.hpin + Handle::kPinBounds);
  if (h.n <= kBoundsOne) {
    hipLaunchKernelGGL(k_bounds_partial, dim3(1), dim3(256), 0, h.stream, h.in4.p, h.n, h.box.p, host);
  } else {
    const int nb = std::min(kBoundsBlocks, div_up(h.n, 256));
    h.red.reserve(6 * nb);
    hipLaunchKernelGGL(k_bounds_partial, dim3(nb), dim3(256), 0, h.stream, h.in4.p, h.n, h.red.p, nullptr);
    hipLaunchKernelGGL(k_bounds_final, dim3(1), dim3(256), 0, h.stream, h.red.p, nb, h.box.p, host);
  }
  EXA_HIP(hipEventRecord(h.ev_bounds, h.stream));
  h.bounds_pending = true;
  h.have_bounds = true;
}

void sync_bounds(Handle &h) {
  if (!h.bounds_pending) return;
  EXA_HIP(hipEventSynchronize(h.ev_bounds));
  const double *r = reinterpret_cast<const double *>(h.hpin + Handle::kPinBounds);
  for (int d = 0; d < 3; d++) {
    h.xmin[d] = r[d];
    h.xmax[d] = r[3 + d];
  }
  h.bounds_pending = false;
}

// The device bounds set from the host values (bounds given by the caller).
void upload_bounds(Handle &h) {
  h.box.reserve(16);
  if (!h.bounds_dev_stale) return;
  const double v[6] = {h.xmin[0], h.xmin[1], h.xmin[2], h.xmax[0], h.xmax[1], h.xmax[2]};
  EXA_HIP(hipMemcpyAsync(h.box.p, v, sizeof(v), hipMemcpyHostToDevice, h.stream));
  EXA_HIP(hipStreamSynchronize(h.stream));  // v lives on this stack frame
  h.bounds_dev_stale = false;
}

// ---------------------------------------------------------------------------
// Uniform trees: one system, or a forest of independent systems (batched
// evaluation).  System s owns bodies [begin, end) of the input and gets its own
// bounds, depth L and Morton keys; level t holds the level-t cells of every
// system with L >= t, and a system's cells come in the order of its
// single-system build.
//
// A tree of depth L has 8^L possible leaves, at most 8 per ncrit bodies, so a
// cell of any level is a run of leaves: where the leaves' first bodies are known,
// they say whether a cell holds bodies, and a prefix sum over the possible cells
// of all levels numbers those that do (no key sort, scan and compaction over the
// bodies for every level, which took 24 launches and more).
// The bodies come into leaf order, those of a leaf in input order, as a stable
// sort by key gives, in one of two ways:
//   up to kCountMost bodies by counting, in 9 to 12 launches: bodies per leaf
//   (atomic counts), a prefix sum for the leaves' first bodies, bodies scattered
//   into their leaves in any order, and each body's rank among its leaf's.
//   2000 bodies 30 us (75 by sorts per level), 100k 46 (124), 400k 81 (165).
//   With a leaf beyond kLeafRank bodies the sort follows, and it comes at once in
//   the handle's next build.
//   beyond, by a stable sort of (leaf, body), the starts found by bisection: 400k
//   bodies 130 us, 1 M 150, 4 M 330, however clustered (1 M and 4 M by counting 147
//   and 468, and 4 M clustered bodies 900 us and more: the atomic counts of few
//   leaves follow each other).
constexpr int kMaxUniformLevels = 10;  // the reference's int keys hold 3 x 10 bits

struct ForestSys {
  double x0, y0, z0;  // bounds minimum (the key origin)
  float d;            // leaf cell size, 2 R0 / 2^L
  int L;              // depth
  int leaf0;          // first of its possible leaves
};

// Possible cells: level t's are [lev0[t], lev0[t + 1]), system s's part of it
// from base[t (S + 1) + s] on (8^t of them, none if L < t).
struct TreeShape {
  int S, nlev, nleaf, ncell;
  int lev0[kMaxUniformLevels + 2];
  const int *base;
};

// bounds2box (build_tree_omp.h:21-33) and the leaf cell size (:218-220), a
// float, with the reference's double operations.
__device__ inline void set_box(const double *mn, const double *mx, ForestSys &f) {
  double R0 = 0;
  for (int d = 0; d < 3; d++) {  // std::max(a, R0) = a < R0 ? R0 : a
    const double Xc = (mx[d] + mn[d]) / 2;
    const double a = Xc - mn[d], b = mx[d] - Xc;
    R0 = a < R0 ? R0 : a;
    R0 = b < R0 ? R0 : b;
  }
  R0 *= 1.00001;
  f.x0 = mn[0];
  f.y0 = mn[1];
  f.z0 = mn[2];
  f.d = 2 * R0 / (1 << f.L);
}

// Per-system min/max: chunks (system, first, last body), one workgroup each,
// then one workgroup per system over its chunks [chunk0[s], chunk0[s + 1]).
__device__ inline void block_minmax(double *mn, double *mx, double (*s)[256]) {
  for (int d = 0; d < 3; d++) {
    s[d][threadIdx.x] = mn[d];
    s[3 + d][threadIdx.x] = mx[d];
  }
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w)
      for (int d = 0; d < 3; d++) {
        const double a = s[d][threadIdx.x + w];
        s[d][threadIdx.x] = a < s[d][threadIdx.x] ? a : s[d][threadIdx.x];
        const double c = s[3 + d][threadIdx.x + w];
        s[3 + d][threadIdx.x] = c > s[3 + d][threadIdx.x] ? c : s[3 + d][threadIdx.x];
      }
    __syncthreads();
  }
}

constexpr int kBoundsChunk = 4096;

__global__ void __launch_bounds__(256)
    k_bounds_chunks(const double4 *__restrict__ b, const int2 *__restrict__ chunk, double *__restrict__ out) {
  __shared__ double s[6][256];
  const int i0 = chunk[blockIdx.x].x, i1 = chunk[blockIdx.x].y;
  double mn[3] = {b[i0].x, b[i0].y, b[i0].z};
  double mx[3] = {mn[0], mn[1], mn[2]};
  for (int i = i0 + threadIdx.x; i < i1; i += 256) {
    const double4 v = b[i];
    mn[0] = v.x < mn[0] ? v.x : mn[0];
    mn[1] = v.y < mn[1] ? v.y : mn[1];
    mn[2] = v.z < mn[2] ? v.z : mn[2];
    mx[0] = v.x > mx[0] ? v.x : mx[0];
    mx[1] = v.y > mx[1] ? v.y : mx[1];
    mx[2] = v.z > mx[2] ? v.z : mx[2];
  }
  block_minmax(mn, mx, s);
  if (threadIdx.x < 6) out[6 * blockIdx.x + threadIdx.x] = s[threadIdx.x][0];
}

__global__ void __launch_bounds__(256)
    k_bounds_systems(const double *__restrict__ part, const int *__restrict__ chunk0, ForestSys *__restrict__ fs) {
  __shared__ double s[6][256];
  const int c0 = chunk0[blockIdx.x], c1 = chunk0[blockIdx.x + 1];
  double mn[3], mx[3];
  for (int d = 0; d < 3; d++) {
    mn[d] = part[6 * c0 + d];
    mx[d] = part[6 * c0 + 3 + d];
  }
  for (int c = c0 + threadIdx.x; c < c1; c += 256)
    for (int d = 0; d < 3; d++) {
      const double a = part[6 * c + d], b = part[6 * c + 3 + d];
      mn[d] = a < mn[d] ? a : mn[d];
      mx[d] = b > mx[d] ? b : mx[d];
    }
  block_minmax(mn, mx, s);
  if (threadIdx.x == 0) {
    const double a[3] = {s[0][0], s[1][0], s[2][0]}, b[3] = {s[3][0], s[4][0], s[5][0]};
    set_box(a, b, fs[blockIdx.x]);
  }
}

// Largest s with v[s] <= x, 0 <= s < n (v ascending, v[0] <= x).
__device__ inline int last_le(const int *__restrict__ v, int n, int x) {
  int lo = 0, hi = n;
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (v[mid] <= x)
      lo = mid;
    else
      hi = mid;
  }
  return lo;
}

// getKey (build_tree_omp.h:36-57): float cell size promoted to double for the
// division, truncation to int, bit interleave in int.  The body's leaf among
// all systems' possible ones.
__device__ inline int body_leaf(const double4 *__restrict__ in, int b, const double *__restrict__ box,
                                ForestSys *__restrict__ fs, int S, const int *__restrict__ begin) {
  ForestSys f = fs[S > 1 ? last_le(begin, S, b) : 0];
  if (box) {  // one system: its box, for the kernels behind this one too
    set_box(box, box + 3, f);
    if (b == 0) {
      fs->x0 = f.x0;
      fs->y0 = f.y0;
      fs->z0 = f.z0;
      fs->d = f.d;
    }
  }
  const double4 v = in[b];
  const double dd = (double)f.d;
  int ix = (int)((v.x - f.x0) / dd);
  int iy = (int)((v.y - f.y0) / dd);
  int iz = (int)((v.z - f.z0) / dd);
  int id = 0;
  for (int l = 0; l != f.L; ++l) {
    id += (ix & 1) << (3 * l);
    id += (iy & 1) << (3 * l + 1);
    id += (iz & 1) << (3 * l + 2);
    ix >>= 1;
    iy >>= 1;
    iz >>= 1;
  }
  return f.leaf0 + id;
}

// leaf[b] and slot[b], the body's place in it.  A workgroup counts its bodies
// per leaf in an LDS table first (open addressing, half full at most) and adds
// one count per leaf: additions to one line of counters follow each other, and
// 65536 bodies in one leaf took 745 us with an addition each, 10 with one per
// workgroup.
constexpr int kCountTable = 512;

__global__ void __launch_bounds__(256)
    k_leaf_count(const double4 *__restrict__ in, int n, const double *__restrict__ box, ForestSys *__restrict__ fs,
                 int S, const int *__restrict__ begin, int *__restrict__ leaf, int *__restrict__ slot,
                 int *__restrict__ cnt) {
  __shared__ int key[kCountTable], num[kCountTable];
  const int tid = threadIdx.x, b = blockIdx.x * 256 + tid;
  for (int i = tid; i < kCountTable; i += 256) {
    key[i] = -1;
    num[i] = 0;
  }
  __syncthreads();
  int at = 0, before = 0;
  if (b < n) {
    const int id = body_leaf(in, b, box, fs, S, begin);
    leaf[b] = id;
    at = (int)(((unsigned)id * 2654435761u >> 16) % kCountTable);
    while (true) {
      const int k = atomicCAS(&key[at], -1, id);
      if (k == -1 || k == id) break;
      at = (at + 1) % kCountTable;
    }
    before = atomicAdd(&num[at], 1);
  }
  __syncthreads();
  for (int i = tid; i < kCountTable; i += 256)
    if (num[i] > 0) num[i] = atomicAdd(&cnt[key[i]], num[i]);
  __syncthreads();
  if (b < n) slot[b] = num[at] + before;
}

// leaf[b] and the bodies' indices, for the sort by leaf.
__global__ void __launch_bounds__(256)
    k_leaf_keys(const double4 *__restrict__ in, int n, const double *__restrict__ box, ForestSys *__restrict__ fs,
                int S, const int *__restrict__ begin, int *__restrict__ leaf, int *__restrict__ ord) {
  const int b = blockIdx.x * 256 + threadIdx.x;
  if (b >= n) return;
  leaf[b] = body_leaf(in, b, box, fs, S, begin);
  ord[b] = b;
}

// First of the n sorted keys that is not below v, in [lo, hi].
__device__ inline int first_not_below(const int *__restrict__ key, int lo, int hi, int v) {
  while (lo < hi) {
    const int mid = (lo + hi) >> 1;
    if (key[mid] < v)
      lo = mid + 1;
    else
      hi = mid;
  }
  return lo;
}

// start[l] = first body of leaf l (l = nleaf: n) among the sorted keys, PER leaves
// a thread; the two ends of a workgroup's leaves bound the others' search.
template <int PER>
__global__ void __launch_bounds__(256)
    k_leaf_starts(const int *__restrict__ key, int n, int nleaf, int *__restrict__ start) {
  __shared__ int ends[2];
  const int64_t l0 = (int64_t)blockIdx.x * 256 * PER;
  if (threadIdx.x < 2)
    ends[threadIdx.x] = first_not_below(key, 0, n, (int)min<int64_t>(nleaf, l0 + 256 * PER * threadIdx.x));
  __syncthreads();
#pragma unroll
  for (int j = 0; j < PER; j++) {
    const int64_t l = l0 + 256 * j + threadIdx.x;
    if (l <= nleaf) start[l] = first_not_below(key, ends[0], ends[1], (int)l);
  }
}

// Level, system and index of possible cell e.
__device__ inline void cell_of(const TreeShape &sh, int e, int &t, int &s, int &k) {
  t = 0;
#pragma unroll
  for (int l = 1; l <= kMaxUniformLevels; l++) t += e >= sh.lev0[l];  // (ncell from lev0[nlev] on)
  const int *b = sh.base + t * (sh.S + 1);
  s = sh.S > 1 ? last_le(b, sh.S, e) : 0;
  k = e - b[s];
}

// First body and end of the run of leaves that cell (t, s, k) covers.
__device__ inline void cell_bodies(const ForestSys &f, const int *__restrict__ start, int t, int k, int &b0, int &b1) {
  const int sh = 3 * (f.L - t);
  b0 = start[f.leaf0 + (k << sh)];
  b1 = start[f.leaf0 + ((k + 1) << sh)];
}

// Prefix sums in chunks of kScanChunk: totals per chunk, then each chunk's
// offsets from the totals before it.  USED: of the cells' flags, else of the
// counts.
constexpr int kScanChunk = 4096;

template <bool USED>
__device__ inline int4 scan_load(const TreeShape &sh, const ForestSys *__restrict__ fs, const int *src, int i, int n) {
  int v[4] = {0, 0, 0, 0};
  if (USED) {  // a cell's end is the next one's first body, within its level and system
    int t, s, k, end = 0, step = 0, at = 0, b = 0;
    for (int j = 0; j < 4 && i + j < n; j++, at += step) {
      if (i + j >= end) {
        cell_of(sh, i + j, t, s, k);
        end = sh.base[t * (sh.S + 1) + s + 1];
        step = 1 << 3 * (fs[s].L - t);
        at = fs[s].leaf0 + k * step;
        b = src[at];
      }
      const int e = src[at + step];
      v[j] = e > b;
      b = e;
    }
  } else {
    for (int k = 0; k < 4; k++) v[k] = i + k >= n ? 0 : src[i + k];
  }
  return make_int4(v[0], v[1], v[2], v[3]);
}

// The counts, read for the last time, are left at zero for the next build.
__device__ inline void clear_counts(int *cnt, int i, int n) {
  for (int k = 0; k < 4; k++)
    if (i + k < n) cnt[i + k] = 0;
}

__device__ inline void scan_store(int *__restrict__ out, int i, int n, int at, int4 v) {
  const int w[4] = {v.x, v.y, v.z, v.w};
  for (int k = 0; k < 4; k++) {
    if (i + k <= n) out[i + k] = at;  // out[n]: the total
    at += w[k];
  }
}

template <bool USED>
__global__ void __launch_bounds__(1024)
    k_tree_totals(TreeShape sh, const ForestSys *__restrict__ fs, const int *__restrict__ src, int n,
                  int *__restrict__ tot) {
  const int4 v = scan_load<USED>(sh, fs, src, blockIdx.x * kScanChunk + 4 * threadIdx.x, n);
  int4 sum;
  block_exscan4<1024>(make_int4(v.x + v.y + v.z + v.w, 0, 0, 0), &sum);
  if (threadIdx.x == 0) tot[blockIdx.x] = sum.x;
}

template <bool USED>
__global__ void __launch_bounds__(1024)
    k_tree_offsets(TreeShape sh, const ForestSys *__restrict__ fs, int *src, int n,
                   const int *__restrict__ tot, int *__restrict__ out) {
  int before = 0;
  for (int b = threadIdx.x; b < (int)blockIdx.x; b += 1024) before += tot[b];
  int4 base, sum;
  block_exscan4<1024>(make_int4(before, 0, 0, 0), &base);
  const int i = blockIdx.x * kScanChunk + 4 * threadIdx.x;
  const int4 v = scan_load<USED>(sh, fs, src, i, n);
  if (!USED) clear_counts(src, i, n);
  const int4 at = block_exscan4<1024>(make_int4(v.x + v.y + v.z + v.w, 0, 0, 0), &sum);
  scan_store(out, i, n, base.x + at.x, v);
}

// Both prefix sums of a small tree in one workgroup.
constexpr int kScanSmall = 4 * kScanChunk;
// Cells up to which the cell arrays are sized by what is possible, about 100
// bytes each, to spare the host a wait for the count.
constexpr int kCellsUnread = 1 << 21;

__global__ void __launch_bounds__(1024)
    k_tree_scan_small(TreeShape sh, const ForestSys *__restrict__ fs, int *__restrict__ cnt, int *start,
                      int *rank) {
  for (int pass = 0; pass < 2; pass++) {
    const int n = pass ? sh.ncell : sh.nleaf;
    int run = 0;
    for (int c = 0; c <= n; c += kScanChunk) {
      const int i = c + 4 * threadIdx.x;
      const int4 v = pass ? scan_load<true>(sh, fs, start, i, n) : scan_load<false>(sh, fs, cnt, i, n);
      if (!pass) clear_counts(cnt, i, n);
      int4 sum;
      const int4 at = block_exscan4<1024>(make_int4(v.x + v.y + v.z + v.w, 0, 0, 0), &sum);
      scan_store(pass ? rank : start, i, n, run + at.x, v);
      run += sum.x;
    }
    __threadfence_block();
    __syncthreads();
  }
}

// Bodies into their leaves' ranges.
__global__ void __launch_bounds__(256)
    k_leaf_scatter(const int *__restrict__ leaf, const int *__restrict__ slot, int n, const int *__restrict__ start,
                   int *__restrict__ ord) {
  const int b = blockIdx.x * 256 + threadIdx.x;
  if (b < n) ord[start[leaf[b]] + slot[b]] = b;
}

// Every leaf's bodies in input order, a thread per place: its body's rank in the
// leaf is the number of the leaf's bodies with a smaller index.  Work follows
// the bodies, whatever the number of possible leaves (with a workgroup for each,
// 262144 bodies at ncrit = 1, 2.1 M possible leaves, took 565 us a build, now
// 121; 2^26 and more were not launched at all).  Leaves beyond kLeafRank bodies,
// where the quadratic count costs more than a sort of all bodies, are left to it.
constexpr int kLeafRank = 1024, kLeafFew = 8;

__global__ void __launch_bounds__(256)
    k_leaf_order(const int *__restrict__ leaf, const int *__restrict__ start, int n, const int *__restrict__ ord,
                 const double4 *__restrict__ in, double4 *__restrict__ body, int *__restrict__ bidx) {
  const int p = min(blockIdx.x * 256 + (int)threadIdx.x, n - 1);  // (the last place may be done more than once)
  const int e = ord[p], l = leaf[e], s = start[l], t = start[l + 1];
  bool todo = t - s <= kLeafRank;
  int rank = 0;
  if (todo && t - s <= kLeafFew) {  // by lane
    for (int k = s; k < t; k++) rank += ord[k] < e;
    todo = false;
  }
  // The wave's larger leaves one by one, their indices by scalar loads.
  while (__any(todo)) {
    const int who = __ffsll(__ballot(todo)) - 1;
    const int s0 = __builtin_amdgcn_readlane(s, who), t0 = __builtin_amdgcn_readlane(t, who);
    int r = 0, k = s0;
    for (; k + 16 <= t0; k += 16)
#pragma unroll
      for (int u = 0; u < 16; u++) r += ord[k + u] < e;
    for (; k < t0; k++) r += ord[k] < e;
    if (todo && s == s0) {
      rank = r;
      todo = false;
    }
  }
  if (t - s > kLeafRank) return;
  body[s + rank] = in[e];
  bidx[s + rank] = e;
}

// The bodies in the order ord (a stable sort by leaf).
__global__ void __launch_bounds__(256)
    k_body_gather(const int *__restrict__ ord, int n, const double4 *__restrict__ in, double4 *__restrict__ body,
                  int *__restrict__ bidx) {
  const int p = blockIdx.x * 256 + threadIdx.x;
  if (p >= n) return;
  const int e = ord[p];
  body[p] = in[e];
  bidx[p] = e;
}

// bodies2leafs / leafs2cells (build_tree_omp.h:130-198) fused with the index
// arithmetic of reverseOrder: the r-th cell of a level in ascending order
// lands at the level's offset + count - 1 - r.  rank: prefix sum of the cells'
// flags, so rank[lev0[t]] is the offset of level t.  Runs before the host
// knows the number of cells (kCellsUnread).  *host_big: a leaf has more than
// kLeafRank bodies.
__global__ void k_uniform_cells(TreeShape sh, const ForestSys *__restrict__ fs, const int *__restrict__ start,
                                const int *__restrict__ rank, const double4 *__restrict__ body,
                                double4 *__restrict__ cX, double *__restrict__ cRb, int *__restrict__ cParent,
                                int *__restrict__ cChild, int *__restrict__ cNChild, int *__restrict__ cBody,
                                int *__restrict__ cNBody, uint64_t *__restrict__ cKey, int *__restrict__ cLevel,
                                int *__restrict__ lvl_cells, int *__restrict__ host_off, int *__restrict__ host_big) {
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e <= sh.nlev) host_off[e] = rank[sh.lev0[e]];
  if (e >= sh.ncell || rank[e + 1] == rank[e]) return;
  int t, s, k, b0, b1;
  cell_of(sh, e, t, s, k);
  const ForestSys f = fs[s];
  cell_bodies(f, start, t, k, b0, b1);
  const int nc = rank[sh.ncell];
  const int c = rank[sh.lev0[t]] + rank[sh.lev0[t + 1]] - 1 - rank[e];
  const double4 v = body[b0];
  float dt = f.d;
  for (int l = 0; l < f.L - t; l++) dt *= 2;  // leafs2cells doubles d per level (:166)
  const double dd = (double)dt;
  const int ix = (int)((v.x - f.x0) / dd);
  const int iy = (int)((v.y - f.y0) / dd);
  const int iz = (int)((v.z - f.z0) / dd);
  double4 X;
  X.x = dd * (ix + .5) + f.x0;
  X.y = dd * (iy + .5) + f.y0;
  X.z = dd * (iz + .5) + f.z0;
  X.w = dd * .5;
  cX[c] = X;
  cRb[c] = X.w;
  cBody[c] = b0;
  cNBody[c] = b1 - b0;
  cKey[c] = (uint64_t)(int64_t)k;
  cLevel[c] = t;
  lvl_cells[c] = c;  // level order: the layout is already level-contiguous
  if (t == f.L) {
    if (b1 - b0 > kLeafRank) *host_big = 1;
    cNChild[c] = 0;
    cChild[c] = nc;  // reverseOrder maps ICHILD = 0 of a leaf to numCells
  } else {
    const int e0 = sh.base[(t + 1) * (sh.S + 1) + s] + 8 * k;
    const int lo = rank[e0], hi = rank[e0 + 8];
    cNChild[c] = hi - lo;
    cChild[c] = rank[sh.lev0[t + 1]] + rank[sh.lev0[t + 2]] - hi;
  }
  if (t == 0) {
    cParent[c] = nc - 1;  // reverseOrder maps the root's IPARENT = 0 to numCells-1
  } else {
    const int rp = rank[sh.base[(t - 1) * (sh.S + 1) + s] + (k >> 3)];
    cParent[c] = rank[sh.lev0[t - 1]] + rank[sh.lev0[t]] - 1 - rp;
  }
}

// Depth of a system of n bodies (build_tree_omp.h:218, integer n / ncrit
// inside the log).
static int uniform_depth(int n, int ncrit) {
  const int L = n >= ncrit ? 1 + int(std::log((double)(n / ncrit)) / M_LN2 / 3) : 0;
  if (L > kMaxUniformLevels)
    throw Error(EXAFMM_HIP_EUNSUP, "uniform tree deeper than 10 levels overflows the reference's int keys");
  return L;
}

// Bodies up to which the leaves are counted (see above); leaves from which a
// thread finds the starts of several.
constexpr int kCountMost = 1 << 20, kStartsMany = 1 << 21;

// The trees of the systems [off[s], off[s + 1]): with given bounds (one
// system), or each with its own.
static void build_uniform(Handle &h, const int *off, int S, bool own_bounds) {
  const int n = h.n, T = 256;
  // Shape and host tables, uploaded when they change.
  std::vector<int> L(S);
  int Lmax = 0, Lmin = kMaxUniformLevels;
  for (int s = 0; s < S; s++) {
    L[s] = uniform_depth(off[s + 1] - off[s], h.cfg.ncrit);
    Lmax = std::max(Lmax, L[s]);
    Lmin = std::min(Lmin, L[s]);
  }
  TreeShape sh{};
  sh.S = S;
  sh.nlev = Lmax + 1;
  // Words: base [nlev][S + 1], begin [S], chunk0 [S + 1], chunks [][2] at an even word.
  const size_t begin0 = (size_t)sh.nlev * (S + 1), chunk00 = begin0 + S, chunks0 = (chunk00 + S + 2) / 2 * 2;
  std::vector<int> tab(chunks0);
  int64_t e = 0;
  for (int t = 0; t <= Lmax; t++) {
    sh.lev0[t] = (int)e;
    for (int s = 0; s <= S; s++) {
      tab[(size_t)t * (S + 1) + s] = (int)e;
      if (s < S && L[s] >= t) e += (int64_t)1 << (3 * t);
    }
    if (e > INT_MAX) throw Error(EXAFMM_HIP_EUNSUP, "build_tree: too many cells");
  }
  sh.ncell = (int)e;
  for (int t = Lmax + 1; t < kMaxUniformLevels + 2; t++) sh.lev0[t] = (int)e;
  std::vector<ForestSys> fs(S);
  int64_t leaf0 = 0;
  for (int s = 0; s < S; s++) {
    fs[s] = ForestSys{0, 0, 0, 0, L[s], (int)leaf0};
    leaf0 += (int64_t)1 << (3 * L[s]);
  }
  if (leaf0 > INT_MAX) throw Error(EXAFMM_HIP_EUNSUP, "build_tree: too many leaves");
  sh.nleaf = (int)leaf0;
  for (int s = 0; s < S; s++) {
    tab[begin0 + s] = off[s];
    tab[chunk00 + s] = (int)((tab.size() - chunks0) / 2);
    for (int b = off[s]; own_bounds && b < off[s + 1]; b += kBoundsChunk) {
      tab.push_back(b);
      tab.push_back(std::min(off[s + 1], b + kBoundsChunk));
    }
  }
  const int nchunk = (int)((tab.size() - chunks0) / 2);
  tab[chunk00 + S] = nchunk;
  h.drop_tree();
  if (tab != h.ut_tab_host) {
    h.ut_tab_host.clear();
    h.ut_tab.resize(tab.size() + 1);
    h.ut_sys.resize(S * sizeof(ForestSys) / sizeof(double));
    EXA_HIP(hipMemcpyAsync(h.ut_tab.p, tab.data(), tab.size() * sizeof(int), hipMemcpyHostToDevice, h.stream));
    EXA_HIP(hipMemcpyAsync(h.ut_sys.p, fs.data(), S * sizeof(ForestSys), hipMemcpyHostToDevice, h.stream));
    EXA_HIP(hipStreamSynchronize(h.stream));
    h.ut_tab_host = std::move(tab);
  }
  sh.base = h.ut_tab.p;
  ForestSys *fsd = reinterpret_cast<ForestSys *>(h.ut_sys.p);
  if (own_bounds) {
    h.red.reserve(6 * (size_t)nchunk);
    const int *chunk = h.ut_tab.p + chunks0;
    hipLaunchKernelGGL(k_bounds_chunks, dim3(nchunk), dim3(256), 0, h.stream, h.in4.p,
                       reinterpret_cast<const int2 *>(chunk), h.red.p);
    hipLaunchKernelGGL(k_bounds_systems, dim3(S), dim3(256), 0, h.stream, h.red.p, h.ut_tab.p + chunk00, fsd);
  } else {
    upload_bounds(h);
  }
  h.body4.resize(n);
  h.bidx.resize(n);
  h.trg4.resize(n);
  h.ia.reserve(n + 1);
  h.ib.reserve(n + 1);
  h.ic.reserve(n + 1);
  h.ut_start.resize((size_t)sh.nleaf + 1);
  h.ut_rank.resize((size_t)sh.ncell + 1);
  const int nchl = div_up((int64_t)sh.nleaf + 1, kScanChunk), nchc = div_up((int64_t)sh.ncell + 1, kScanChunk);
  h.ut_tot.reserve(std::max(nchl, nchc));
  int *leaf = h.ic.p, *ord = h.ia.p, *aux = h.ib.p, *start = h.ut_start.p, *rank = h.ut_rank.p;
  const double *box = own_bounds ? nullptr : h.box.p;
  const int *begin = h.ut_tab.p + begin0;
  const int nb = div_up(n, 256);
  // Bodies by a stable sort, and the leaves' starts from the sorted keys.
  auto sort_bodies = [&] {
    int bits = 1;
    while (((int64_t)1 << bits) < sh.nleaf) bits++;
    h.id.reserve(n + 1);
    hipLaunchKernelGGL(k_leaf_keys, dim3(nb), dim3(256), 0, h.stream, h.in4.p, n, box, fsd, S, begin, leaf, ord);
    bool alt = false;
    sort_pairs_int_int(leaf, h.id.p, ord, aux, n, bits, alt, h.stream, h.tmp);
    auto starts = [&](auto kernel, int per) {
      hipLaunchKernelGGL(kernel, dim3(div_up((int64_t)sh.nleaf + 1, 256 * per)), dim3(256), 0, h.stream,
                         alt ? h.id.p : leaf, n, sh.nleaf, start);
    };
    // (16.7 M leaves: 250 us with one leaf a thread, 132 with four; 262144: 13 and 25.)
    sh.nleaf >= kStartsMany ? starts(k_leaf_starts<4>, 4) : starts(k_leaf_starts<1>, 1);
    hipLaunchKernelGGL(k_body_gather, dim3(nb), dim3(256), 0, h.stream, alt ? aux : ord, n, h.in4.p, h.body4.p,
                       h.bidx.p);
  };
  const bool sort = n > kCountMost || h.ut_sort;
  if (sort) {
    sort_bodies();
  } else {
    if (!h.ut_zero || (size_t)sh.nleaf >= h.ut_cnt.cap) {
      h.ut_cnt.reserve((size_t)sh.nleaf + 1);
      zero_device(h.ut_cnt.p, h.ut_cnt.cap / 2 * 8, h.stream);
    }
    h.ut_zero = false;
    hipLaunchKernelGGL(k_leaf_count, dim3(nb), dim3(256), 0, h.stream, h.in4.p, n, box, fsd, S, begin, leaf, aux,
                       h.ut_cnt.p);
  }
  if (!sort && sh.ncell <= kScanSmall) {
    hipLaunchKernelGGL(k_tree_scan_small, dim3(1), dim3(1024), 0, h.stream, sh, fsd, h.ut_cnt.p, start, rank);
  } else {
    if (!sort) {
      hipLaunchKernelGGL(k_tree_totals<false>, dim3(nchl), dim3(1024), 0, h.stream, sh, fsd, h.ut_cnt.p, sh.nleaf,
                         h.ut_tot.p);
      hipLaunchKernelGGL(k_tree_offsets<false>, dim3(nchl), dim3(1024), 0, h.stream, sh, fsd, h.ut_cnt.p, sh.nleaf,
                         h.ut_tot.p, start);
    }
    hipLaunchKernelGGL(k_tree_totals<true>, dim3(nchc), dim3(1024), 0, h.stream, sh, fsd, start, sh.ncell,
                       h.ut_tot.p);
    hipLaunchKernelGGL(k_tree_offsets<true>, dim3(nchc), dim3(1024), 0, h.stream, sh, fsd, start, sh.ncell,
                       h.ut_tot.p, rank);
  }
  if (!sort) {
    hipLaunchKernelGGL(k_leaf_scatter, dim3(nb), dim3(256), 0, h.stream, leaf, aux, n, start, ord);
    hipLaunchKernelGGL(k_leaf_order, dim3(nb), dim3(256), 0, h.stream, leaf, start, n, ord, h.in4.p, h.body4.p,
                       h.bidx.p);
    h.ut_zero = true;
  }
  int *host_off = h.hpin + 128;  // (the adaptive builder's words)
  int ncap = sh.ncell;           // the cell arrays hold every possible cell of trees up to kCellsUnread of them
  if (ncap > kCellsUnread) {
    EXA_HIP(hipMemcpyAsync(host_off, rank + ncap, sizeof(int), hipMemcpyDeviceToHost, h.stream));
    EXA_HIP(hipStreamSynchronize(h.stream));
    ncap = host_off[0];
  }
  for (DBuf<int> *v : {&h.cParent, &h.cChild, &h.cNChild, &h.cBody, &h.cNBody, &h.cLevel, &h.lvl_cells})
    v->reserve(ncap);
  h.cX.reserve(ncap);
  h.cRb.reserve(ncap);
  h.cKey.reserve(ncap);
  volatile int *host_big = host_off + sh.nlev + 1;
  auto cells = [&] {
    *host_big = 0;
    hipLaunchKernelGGL(k_uniform_cells, dim3(div_up(std::max(sh.ncell, sh.nlev + 1), T)), dim3(T), 0, h.stream, sh,
                       fsd, start, rank, h.body4.p, h.cX.p, h.cRb.p, h.cParent.p, h.cChild.p, h.cNChild.p, h.cBody.p,
                       h.cNBody.p, h.cKey.p, h.cLevel.p, h.lvl_cells.p, host_off, const_cast<int *>(host_big));
    EXA_HIP(hipGetLastError());
    EXA_HIP(hipStreamSynchronize(h.stream));
  };
  cells();
  h.ut_sort = *host_big != 0;
  if (h.ut_sort && !sort) {  // the large leaves' bodies, and the cells again (a cell's centre comes from its first)
    sort_bodies();
    cells();
  }
  const int nc = host_off[sh.nlev];
  h.ncells = nc;
  h.nlevels = sh.nlev;
  h.lvl_off.assign(host_off, host_off + sh.nlev + 1);
  h.lvl_par.assign(sh.nlev, 0);
  // All cells above the leaves have children; in a forest a bound, as
  // shallower systems end above.
  for (int t = 0; t < sh.nlev; t++) h.lvl_par[t] = h.lvl_off[t + 1] - h.lvl_off[t];
  h.leaf_level = Lmin;
  for (DBuf<int> *v : {&h.cParent, &h.cChild, &h.cNChild, &h.cBody, &h.cNBody, &h.cLevel, &h.lvl_cells})
    v->resize(nc);
  h.cX.resize(nc);
  h.cRb.resize(nc);
  h.cKey.resize(nc);
}

void run_build_uniform(Handle &h) {
  const int off[2] = {0, h.n};
  build_uniform(h, off, 1, false);
  sync_bounds(h);  // (arrived before the cells)
}

void run_build_forest(Handle &h) { build_uniform(h, h.sys_off.data(), h.nsys, true); }

}  // namespace exafmm
