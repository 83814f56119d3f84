// Workgroup scans and the sort of short index ranges shared by the tree build
// and the list grouping.
#pragma once
#include <hip/hip_runtime.h>

#include <climits>

namespace exafmm {

// Orders the LDS accesses of one wave (its stores before its later loads by
// other lanes), where waves of a workgroup use separate parts of LDS.
__device__ inline void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

__device__ inline int4 add4(int4 a, int4 b) { return make_int4(a.x + b.x, a.y + b.y, a.z + b.z, a.w + b.w); }

// Exclusive prefix of v over the NT threads of the block (wave scans, then
// the wave totals); *total receives the block sum.
template <int NT = 256>
__device__ inline int4 block_exscan4(int4 v, int4 *total) {
  __shared__ int4 wsum[NT / 64];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  int4 inc = v;
  for (int d = 1; d < 64; d <<= 1) {
    const int4 t = make_int4(__shfl_up(inc.x, d), __shfl_up(inc.y, d), __shfl_up(inc.z, d), 0);
    if (lane >= d) inc = add4(inc, t);
  }
  if (lane == 63) wsum[w] = inc;
  __syncthreads();
  int4 base = make_int4(0, 0, 0, 0), tot = make_int4(0, 0, 0, 0);
  if (NT <= 256) {
    for (int k = 0; k < NT / 64; k++) {
      if (k < w) base = add4(base, wsum[k]);
      tot = add4(tot, wsum[k]);
    }
  } else {  // many waves: the first wave scans the wave totals in place
    if (w == 0) {
      int4 x = lane < NT / 64 ? wsum[lane] : make_int4(0, 0, 0, 0);
      for (int d = 1; d < NT / 64; d <<= 1) {
        const int4 t = make_int4(__shfl_up(x.x, d), __shfl_up(x.y, d), __shfl_up(x.z, d), 0);
        if (lane >= d) x = add4(x, t);
      }
      if (lane < NT / 64) wsum[lane] = x;
    }
    __syncthreads();
    if (w > 0) base = wsum[w - 1];
    tot = wsum[NT / 64 - 1];
  }
  __syncthreads();
  *total = tot;
  return make_int4(base.x + inc.x - v.x, base.y + inc.y - v.y, base.z + inc.z - v.z, 0);
}

// Sorts n distinct whole numbers below 2^bits held in a[0 .. n) by one wave (a
// workgroup of 64) and hands each with its place to emit(place, value).  A
// value's place is the number of smaller ones: up to 64 values by lane reads,
// up to kRangeRank through LDS (quadratic: 1 us at 30 to 100 values); longer
// ranges by a stable radix sort, 5 bits at a time, between a and b.
constexpr int kRangeRank = 1024;
struct RangeSortLds {
  __attribute__((aligned(16))) int e[kRangeRank];
  int hist[32];
};

template <typename Emit>
__device__ inline void sort_range(int *a, int *b, int n, int bits, RangeSortLds &sh, Emit emit) {
  const int lane = threadIdx.x;
  if (n <= 64) {
    const int e = lane < n ? a[lane] : INT_MAX;
    int rank = 0;
    for (int k = 0; k < n; k++) rank += __builtin_amdgcn_readlane(e, k) < e;
    if (lane < n) emit(rank, e);
    return;
  }
  if (n <= kRangeRank) {
    for (int k = lane; k < (n + 3) / 4 * 4; k += 64) sh.e[k] = k < n ? a[k] : INT_MAX;
    __syncthreads();
    const int4 *s4 = reinterpret_cast<const int4 *>(sh.e);
    for (int i = lane; i < n; i += 64) {
      const int e = sh.e[i];
      int rank = 0;
      for (int k = 0; k < (n + 3) / 4; k++) {
        const int4 v = s4[k];
        rank += (v.x < e) + (v.y < e) + (v.z < e) + (v.w < e);
      }
      emit(rank, e);
    }
    return;
  }
  for (int shift = 0; shift < bits; shift += 5) {
    if (lane < 32) sh.hist[lane] = 0;
    __syncthreads();
    for (int i = lane; i < n; i += 64) atomicAdd(&sh.hist[(a[i] >> shift) & 31], 1);
    __syncthreads();
    const int h = lane < 32 ? sh.hist[lane] : 0;
    int inc = h;
    for (int d = 1; d < 32; d <<= 1) {
      const int t = __shfl_up(inc, d);
      if (lane >= d) inc += t;
    }
    __syncthreads();
    if (lane < 32) sh.hist[lane] = inc - h;  // where the digit's next value goes
    __syncthreads();
    for (int i0 = 0; i0 < n; i0 += 64) {
      const int i = i0 + lane;
      const int e = i < n ? a[i] : 0, d = (e >> shift) & 31;
      unsigned long long same = __ballot(i < n);
      for (int k = 0; k < 5; k++) {
        const unsigned long long m = __ballot((d >> k) & 1);
        same &= (d >> k) & 1 ? m : ~m;
      }
      const int before = (int)__popcll(same & ((1ull << lane) - 1));
      const int at = i < n ? sh.hist[d] : 0;
      __syncthreads();
      if (i < n && before == 0) sh.hist[d] = at + (int)__popcll(same);
      if (i < n) b[at + before] = e;
      __syncthreads();
    }
    __threadfence_block();
    __syncthreads();
    int *t = a;
    a = b;
    b = t;
  }
  for (int i = lane; i < n; i += 64) emit(i, a[i]);
}

}  // namespace exafmm
