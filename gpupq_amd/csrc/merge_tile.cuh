// merge_tile.cuh -- one tile of a merge of two sorted record sequences, by one block: the
// block's share of both by merge-path searches, merged through LDS.  Used by the merge launches
// of the global queues (sortprim.hip, queue_hq.hip).
#pragma once

#include "sortprim.h"

namespace gpq {

constexpr int kPerThread = 8;                          // records per thread in the merge

// A = a1[0:n1) ++ a2[...]
struct ASrc {
  const Event* a1;
  const Event* a2;
  uint32_t n1;
  __device__ __forceinline__ const Event* at(uint32_t i) const { return i < n1 ? a1 + i : a2 + (i - n1); }
  __device__ __forceinline__ Event get(uint32_t i) const { return load_event(at(i)); }
};

struct OutMap {
  Event* out[3];
  uint32_t end[3];
  __device__ __forceinline__ Event* at(uint32_t o) const {
    if (o < end[0]) return out[0] + o;
    if (o < end[1]) return out[1] + (o - end[0]);
    return out[2] + (o - end[1]);
  }
};

// Merge-path split: the number of A records among the first d outputs of the stable merge
// (ties: A first) is the smallest i in [max(0, d - nb), min(d, na)] with B[d-1-i] < A[i].
// Found for the block's two diagonals d0 and d1 at once, each by half of the block: every
// round the kT / 2 threads of a half probe as many evenly spaced points of the remaining range and
// keep the gap where the predicate turns true, so a range of n shrinks to nothing in
// ceil(log n / log(kT / 2)) rounds of one load each, not log_2 n dependent loads.
template <int kT>
__device__ __forceinline__ void block_merge_splits(const ASrc& A, uint32_t na, const Event* B, uint32_t nb, uint32_t d0, uint32_t d1,
                                   uint32_t* s_split) {
  constexpr uint32_t kProbes = kT / 2;
  __shared__ uint32_t s_lo[2], s_hi[2], s_first[2];
  const uint32_t h = threadIdx.x / kProbes, k = threadIdx.x % kProbes;
  const uint32_t d = h ? d1 : d0;
  if (k == 0) {
    s_lo[h] = d > nb ? d - nb : 0u;
    s_hi[h] = d < na ? d : na;
  }
  __syncthreads();
  while (s_lo[0] < s_hi[0] || s_lo[1] < s_hi[1]) {   // uniform: read after a barrier
    const uint32_t lo = s_lo[h], hi = s_hi[h];
    const uint32_t step = (hi - lo + kProbes - 1) / kProbes;
    if (k == 0) s_first[h] = 0xFFFFFFFFu;
    __syncthreads();
    if (lo < hi) {
      const uint32_t i = lo + k * step;
      if (i < hi && key_less(load_event(B + (d - 1u - i)), A.get(i))) atomicMin(&s_first[h], k);
    }
    __syncthreads();
    if (k == 0 && lo < hi) {
      const uint32_t f = s_first[h];
      if (f == 0xFFFFFFFFu) {
        s_lo[h] = lo + (hi - lo - 1u) / step * step + 1u;   // past the last probe
      } else {
        s_hi[h] = lo + f * step;
        if (f) s_lo[h] = lo + (f - 1u) * step + 1u;
      }
    }
    __syncthreads();
  }
  if (k == 0) s_split[h] = s_lo[h];
  __syncthreads();
}

// LDS slot of tile element i: one pad record after every 8, so the 8-record runs that
// consecutive threads merge start in different banks.
__device__ __forceinline__ uint32_t pad8(uint32_t i) { return i + (i >> 3); }

// Merges output ranks [t0, t0 + kMergeTile) of merge(A, B) through LDS: the block's input
// ranges are located by two merge-path searches, staged in LDS, each thread merges 8
// outputs, and the results leave through LDS in coalesced 16-byte stores.
// With `pre` set, the block's splits were computed before the launch (merge_partition_kernel):
// pre[0] and pre[1] are those of its first and last output rank.
template <int kT>
__device__ __forceinline__ void merge_tile(const ASrc& A, uint32_t na, const Event* B, uint32_t nb, uint32_t t0,
                                           const OutMap& out, const uint32_t* pre = nullptr) {
  constexpr uint32_t kTile = kT * kPerThread;
  __shared__ Event s[kTile + kTile / 8 + 2 * kPerThread];   // heads are read up to kPerThread past the tile
  __shared__ uint32_t s_split[2];
  const uint32_t total = na + nb;
  const uint32_t t1 = t0 + kTile < total ? t0 + kTile : total;
  uint32_t i0, i1;
  if (pre) {
    i0 = pre[0];
    i1 = pre[1];
  } else {
    block_merge_splits<kT>(A, na, B, nb, t0, t1, s_split);
    i0 = s_split[0];
    i1 = s_split[1];
  }
  const uint32_t j0 = t0 - i0;
  const uint32_t ca = i1 - i0, cb = (t1 - t0) - ca;
  const uint32_t len = t1 - t0;
  // the thread's loads are all in flight at once: one after the other, each waits for memory (100,003
  // LPs in the HQ 175 ms, 166 so, with the heads below in registers)
  uint4 res[kPerThread];
#pragma unroll
  for (int q = 0; q < kPerThread; ++q) {
    const uint32_t i = threadIdx.x + (uint32_t)q * kT, x = i < len ? i : len - 1u;
    res[q] = *reinterpret_cast<const uint4*>(x < ca ? A.at(i0 + x) : B + (j0 + x - ca));
  }
#pragma unroll
  for (int q = 0; q < kPerThread; ++q) {
    const uint32_t i = threadIdx.x + (uint32_t)q * kT;
    if (i < len) s[pad8(i)] = Event{res[q].x, res[q].y, res[q].z, res[q].w};
  }
  __syncthreads();
  const uint32_t d = threadIdx.x * kPerThread;
  uint32_t got = 0;
  if (d < len) {
    uint32_t lo = d > cb ? d - cb : 0u, hi = d < ca ? d : ca;
    while (lo < hi) {
      const uint32_t mid = (lo + hi) >> 1;
      if (key_less(s[pad8(ca + (d - 1u - mid))], s[pad8(mid)])) hi = mid; else lo = mid + 1u;
    }
    uint32_t ia = lo, ib = ca + d - lo;                // of the two runs' heads, which stay in registers
    Event a = s[pad8(ia)], b = s[pad8(ib)];
#pragma unroll
    for (int q = 0; q < kPerThread; ++q) {
      const bool take_a = ib >= len || (ia < ca && !key_less(b, a));
      const Event r = take_a ? a : b;
      res[q] = make_uint4(r.ts, r.dst, r.src, r.seq);
      const Event next = s[pad8(take_a ? ++ia : ++ib)];
      if (take_a) a = next;
      else b = next;
    }
    got = len - d < (uint32_t)kPerThread ? len - d : (uint32_t)kPerThread;
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < kPerThread; ++q)
    if ((uint32_t)q < got) s[pad8(d + q)] = Event{res[q].x, res[q].y, res[q].z, res[q].w};
  __syncthreads();
  for (uint32_t x = threadIdx.x; x < len; x += kT) store_event(out.at(t0 + x), s[pad8(x)]);
}

}  // namespace gpq
