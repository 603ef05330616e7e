// sortprim.hip -- record sort (tile sort in LDS, then levels of up to 128-way merges),
// multi-task merge-path merges, and the parallel one-safe-event-per-LP selection.
#include <algorithm>

#include "merge_tile.cuh"
#include "sortprim.h"

namespace gpq {
namespace {

constexpr int kThreads = 256;                       // selection blocks; merge blocks: kT of 128, 256 or
                                                    // 512 threads (tiles of 8 kT records)
constexpr uint32_t kSelectTile = 1024;              // records per selection tile (256 threads x 4)
constexpr uint32_t kSelectBlocks = 1024;            // blocks of a selection launch, at most
constexpr uint32_t kSplitLanes = 8;                 // lanes per tile boundary in the merge partition

__device__ __forceinline__ Event sentinel() { return Event{0xFFFFFFFFu, 0xFFFFFFFFu, 0xFFFFFFFFu, 0xFFFFFFFFu}; }

// The same split for diagonal d by a group of P lanes (P a power of two dividing the wave; every
// lane of a group passes the same d, `active` false for a group with no diagonal): P probes per
// round, ceil(log_P n) rounds.  The loop runs while any group of the wave is searching.
template <int P>
__device__ __forceinline__ uint32_t group_merge_split(const ASrc& A, uint32_t na, const Event* B, uint32_t nb,
                                                      uint32_t d, bool active) {
  const uint32_t lane = (uint32_t)lane_id(), k = lane % P, gbase = lane - k;
  const uint64_t gmask = (P == kWave ? ~0ull : ((1ull << P) - 1ull)) << gbase;
  uint32_t lo = active && d > nb ? d - nb : 0u, hi = active ? (d < na ? d : na) : 0u;
  while (__ballot(lo < hi)) {
    const bool run = lo < hi;                         // uniform within the group
    const uint32_t step = run ? (hi - lo + P - 1u) / P : 1u;
    const uint32_t i = lo + k * step;
    const bool p = run && i < hi && key_less(load_event(B + (d - 1u - i)), A.get(i));
    const uint64_t m = (__ballot(p) & gmask) >> gbase;
    if (run) {
      if (m == 0) {
        lo = lo + (hi - lo - 1u) / step * step + 1u;  // past the last probe
      } else {
        const uint32_t f = (uint32_t)__ffsll((unsigned long long)m) - 1u;
        hi = lo + f * step;
        if (f) lo = lo + (f - 1u) * step + 1u;
      }
    }
  }
  return lo;
}

// --- sort -------------------------------------------------------------------------
//
// A run of up to kRun records is sorted by one block (tile_sort_kernel); a level then merges up to
// fan_of() sorted runs at once: every kSampleth record of a run is a sample (from an offset of the run's
// own: the same quantiles sampled in every run would leave gaps without samples, and blocks with
// three times the others' records), sample_rank_kernel ranks
// all samples of the runs against each other, and bucket_merge_kernel takes bucket_samples()
// consecutive samples' worth of records per block -- its share of every run, found by searching
// each run for two samples -- and merges the shares in LDS.  Between two samples of a run lie fewer
// than kSample records, so a block's shares hold at most (kBucketSamples + kFan) * kSample =
// kBucketCap records whatever the data.  One level sorts 2^17 records, two 2^24.
//
// What bounds it at the global queues' sizes (10^4 to 10^6 records) is the chain of launches and
// of dependent LDS and L2 accesses, not bytes: 100,003 records took 59 us in a bitonic tile sort
// of 66 stages and 10 us in each of six pairwise merge passes, 120 us in all; the three launches
// here take 16, 9 and 28 us, 52 us in all.
// Tiles and buckets are small (1024 records, two or one per thread) so that they spread over the
// CUs: with tiles and buckets of 2048 records and eight or four per thread the launches took 38
// and 39 us, most of it LDS reads and index arithmetic of one wave per SIMD.
//
// Order: (ts, src, seq), then dst, so that records compare equal only if they are identical.
constexpr uint32_t kRun = 1024;
constexpr uint32_t kTilePer = 2;
constexpr int kTileThreads = kRun / kTilePer;
constexpr uint32_t kFan = 128;
constexpr uint32_t kSample = 32;
constexpr uint32_t kBucketSamples = 24;
constexpr uint32_t kBucketCap = (kBucketSamples + kFan) * kSample;
constexpr int kBucketThreads = 1024;
constexpr uint32_t kBucketPer = (kBucketCap + kBucketThreads - 1) / kBucketThreads;
constexpr uint32_t kFindLanes = kBucketThreads / (2 * kFan);   // lanes that search one run for one sample
static_assert(kRun % kSample == 0, "whole runs have the same number of samples");

// Samples of run r (in its group): records off, off + kSample, ... with off = sample_offset(r).
__device__ __forceinline__ uint32_t sample_offset(uint32_t r) { return (r * 21u + 5u) % kSample; }
__device__ __forceinline__ uint32_t samples_of(uint32_t r, uint32_t len) {
  const uint32_t off = sample_offset(r);
  return len > off ? (len - off - 1u) / kSample + 1u : 0u;
}
// Record index of sample s of a level's input: the samples of whole runs are numbered run by run.
__device__ __forceinline__ uint32_t sample_record(uint32_t s, uint32_t w, uint32_t fan) {
  const uint32_t run = s / (w / kSample);
  return run * w + (s % (w / kSample)) * kSample + sample_offset(run % fan);
}

// Runs merged at once, for n records.  Two levels of 32 (up to 2^20 records) or 64 (2^22) runs each, with up
// to 64 samples a block, where 128 runs leave a block room for 24 (all shares have to fit), so that a level
// takes several rounds of blocks, and leave the second level few runs: 200,003 records 85 us and 93 with 128,
// 500,009 133 and 163, 1,000,003 202 and 300.
__host__ __device__ __forceinline__ uint32_t fan_of(uint64_t n) {
  return n <= (uint64_t)kRun * kFan ? kFan : (n <= kRun << 10 ? 32u : (n <= kRun << 12 ? 64u : kFan));
}
// Samples per block of bucket_merge_kernel: as many blocks as the chip runs at once, two per CU.
__device__ __forceinline__ uint32_t bucket_samples(uint32_t n, uint32_t fan) {
  const uint32_t even = (n / kSample + 511u) / 512u;
  return fan == kFan || even < kBucketSamples ? kBucketSamples : (even < 64u ? even : 64u);
}
static_assert((64u + 64u) * kSample <= kBucketCap, "a block of the narrower levels fits");
// Records per run of a level's input.
__device__ __forceinline__ uint32_t level_width(uint32_t level, uint32_t fan) {
  uint32_t w = kRun;
  for (uint32_t i = 1; i < level; ++i) w *= fan;
  return w;
}

// A record as two words whose pair order is the sort order.
struct Rec {
  uint64_t hi, lo;
};
__device__ __forceinline__ Rec load_rec(const Event* p) {
  const Event e = load_event(p);
  return Rec{((uint64_t)e.ts << 32) | e.src, ((uint64_t)e.seq << 32) | e.dst};
}
__device__ __forceinline__ bool rec_less(uint64_t ahi, uint64_t alo, uint64_t bhi, uint64_t blo) {
  return ahi != bhi ? ahi < bhi : alo < blo;
}

// Records in LDS by word: searches read timestamps alone (4-byte reads, 32-bit comparisons), and
// the other words only where timestamps tie.  One pad word per 32: the probes of a binary search
// lie powers of two apart, which would put them all in one bank.
template <uint32_t N>
struct LdsRecs {
  static constexpr uint32_t kSize = N + N / 32u;
  uint64_t lo[kSize];
  uint32_t ts[kSize], src[kSize];
  static __device__ __forceinline__ uint32_t at(uint32_t i) { return i + (i >> 5); }
  __device__ __forceinline__ uint32_t time(uint32_t i) const { return ts[at(i)]; }
  __device__ __forceinline__ void put(uint32_t i, uint64_t h, uint64_t l) {
    const uint32_t a = at(i);
    ts[a] = (uint32_t)(h >> 32);
    src[a] = (uint32_t)h;
    lo[a] = l;
  }
  __device__ __forceinline__ Event get(uint32_t i) const {
    const uint32_t a = at(i);
    const uint64_t l = lo[a];
    return Event{ts[a], (uint32_t)l, src[a], (uint32_t)(l >> 32)};
  }
  // record i comes before (h, l), or equals it with `equal`
  __device__ __forceinline__ bool before(uint32_t i, uint64_t h, uint64_t l, bool equal) const {
    const uint32_t a = at(i);
    const uint64_t oh = ((uint64_t)ts[a] << 32) | src[a], ol = lo[a];
    return oh != h ? oh < h : (equal ? ol <= l : ol < l);
  }
};

// Levels that n records take.
__host__ __device__ __forceinline__ uint32_t sort_levels(uint64_t n) {
  uint32_t k = 0;
  for (uint64_t w = kRun; w < n; w *= kFan) ++k;
  return k;
}

// Sorted runs of kRun records; written to buf1 when the levels that follow are odd in number, to
// buf0 otherwise, so that the last level leaves the result in buf0.
// seg_pre (optional): `in` is a striped insert area (core.cuh) whose segment k holds records
// [seg_pre[k], seg_pre[k + 1]) of the input (k < kInsertStripes: at k * seg_cap; the spill
// segment k = kInsertStripes after the stripes).
__global__ __launch_bounds__(kTileThreads) void tile_sort_kernel(const Event* in, Event* buf0, Event* buf1,
                                                                 const uint32_t* d_n, uint32_t cap,
                                                                 const uint32_t* seg_pre, uint32_t seg_cap) {
  __shared__ LdsRecs<kRun> s;
  __shared__ uint32_t s_pre[kInsertStripes + 2];
  const uint32_t n = d_n ? *d_n : cap;
  const uint32_t base = blockIdx.x * kRun;
  if (base >= n) return;
  if (seg_pre) {
    for (uint32_t k = threadIdx.x; k < kInsertStripes + 2u; k += kTileThreads) s_pre[k] = seg_pre[k];
    __syncthreads();
  }
  const uint32_t have = n - base < kRun ? n - base : kRun;
  uint64_t hi[kTilePer], lo[kTilePer];
  uint32_t pos[kTilePer];
#pragma unroll
  for (uint32_t q = 0; q < kTilePer; ++q) {
    pos[q] = threadIdx.x * kTilePer + q;
    hi[q] = lo[q] = ~0ull;                            // past the end: never placed or looked at
    if (pos[q] < have) {
      const uint32_t g = base + pos[q];
      const Event* p = in + g;
      if (seg_pre) {
        uint32_t a = 0, b = kInsertStripes;           // the last segment k with s_pre[k] <= g
        while (a < b) {
          const uint32_t mid = (a + b + 1u) >> 1;
          if (s_pre[mid] <= g) a = mid; else b = mid - 1u;
        }
        p = in + (size_t)a * seg_cap + (g - s_pre[a]);
      }
      const Rec r = load_rec(p);
      hi[q] = r.hi;
      lo[q] = r.lo;
    }
  }
  static_assert(kTilePer == 2, "one exchange sorts a thread's records");
  if (rec_less(hi[1], lo[1], hi[0], lo[0])) {
    const uint64_t h = hi[0], l = lo[0];
    hi[0] = hi[1]; lo[0] = lo[1];
    hi[1] = h; lo[1] = l;
  }
#pragma unroll
  for (uint32_t q = 0; q < kTilePer; ++q)
    if (pos[q] < have) s.put(pos[q], hi[q], lo[q]);
  __syncthreads();
  // runs of w pair up: a record's place is its place in its run plus its rank in the other
  for (uint32_t w = kTilePer; w < kRun; w *= 2) {
    uint32_t cnt[kTilePer];
    const uint32_t own = threadIdx.x * kTilePer & ~(w - 1u);   // the thread's records lie in one run
    const uint32_t other = own ^ w;
    const uint32_t len = other < have ? (have - other < w ? have - other : w) : 0u;
    const bool right = (own & w) != 0;                // ties: the left run's records first
#pragma unroll
    for (uint32_t q = 0; q < kTilePer; ++q) cnt[q] = 0;
    for (uint32_t bit = w; bit; bit >>= 1) {
      uint32_t ot[kTilePer];
      bool tie = false;
#pragma unroll
      for (uint32_t q = 0; q < kTilePer; ++q) {       // a probe past the run reads slot 0 and is not used
        const uint32_t c = cnt[q] + bit;
        ot[q] = s.time(c <= len ? other + c - 1u : 0u);
      }
#pragma unroll
      for (uint32_t q = 0; q < kTilePer; ++q) tie |= cnt[q] + bit <= len && ot[q] == (uint32_t)(hi[q] >> 32);
      if (__any(tie)) {                               // a branch of the whole wave, rarely taken
#pragma unroll
        for (uint32_t q = 0; q < kTilePer; ++q) {
          const uint32_t c = cnt[q] + bit;
          if (c <= len && s.before(other + c - 1u, hi[q], lo[q], right)) cnt[q] = c;
        }
      } else {
#pragma unroll
        for (uint32_t q = 0; q < kTilePer; ++q) {
          const uint32_t c = cnt[q] + bit;
          if (c <= len && ot[q] < (uint32_t)(hi[q] >> 32)) cnt[q] = c;
        }
      }
    }
    __syncthreads();
    const uint32_t pair = own & ~(2u * w - 1u);
#pragma unroll
    for (uint32_t q = 0; q < kTilePer; ++q) {
      if (pos[q] < have) {
        pos[q] = pair + (pos[q] - own) + cnt[q];
        s.put(pos[q], hi[q], lo[q]);
      }
    }
    __syncthreads();
  }
  Event* out = (sort_levels(n) & 1u) ? buf1 : buf0;
  for (uint32_t i = threadIdx.x; i < kRun; i += kTileThreads)
    if (base + i < n) store_event(out + base + i, s.get(i));
}

// Number of the cnt elements a[0], a[stride], ... that come before (hi, lo) -- or equal it, with
// `equal` -- in a sorted sequence.
__device__ __forceinline__ uint32_t count_before(const Event* a, uint32_t cnt, uint32_t stride, uint64_t hi, uint64_t lo,
                                                 bool equal) {
  uint32_t c = 0;
  for (uint32_t bit = cnt ? 1u << (31 - __builtin_clz(cnt)) : 0u; bit; bit >>= 1) {
    const uint32_t t = c + bit;
    if (t > cnt) continue;
    const Rec r = load_rec(a + (size_t)(t - 1u) * stride);
    if (rec_less(r.hi, r.lo, hi, lo) || (equal && r.hi == hi && r.lo == lo)) c = t;
  }
  return c;
}

// The same count for stride 1 by a group of kFindLanes lanes (all of them call with the same
// arguments): each round probes kFindLanes points that cut the remaining range evenly.
__device__ __forceinline__ uint32_t count_before_lanes(const Event* a, uint32_t cnt, uint64_t hi, uint64_t lo, bool equal) {
  const uint32_t lane = (uint32_t)lane_id(), k = lane % kFindLanes, first = lane - k;
  uint32_t from = 0, to = cnt;                                     // the count lies in [from, to]
  while (__ballot(from < to)) {
    const uint32_t len = to - from;
    bool before = false;
    if (len) {
      const Rec r = load_rec(a + from + len * (k + 1u) / (kFindLanes + 1u));
      before = rec_less(r.hi, r.lo, hi, lo) || (equal && r.hi == hi && r.lo == lo);
    }
    const uint32_t m = (uint32_t)__popcll((__ballot(before) >> first) & ((1ull << kFindLanes) - 1ull));
    if (len) {
      const uint32_t f = from;
      if (m < kFindLanes) to = f + len * (m + 1u) / (kFindLanes + 1u);
      if (m) from = f + len * m / (kFindLanes + 1u) + 1u;
    }
  }
  return from;
}

// Source and destination of level `level` (1, 2, ...) for n records; false when n needs fewer.
__device__ __forceinline__ bool level_buffers(uint32_t n, uint32_t level, Event* buf0, Event* buf1, const Event** src,
                                              Event** dst) {
  const uint32_t k = sort_levels(n);
  if (level > k) return false;
  const bool odd = ((k - level) & 1u) != 0;
  *dst = odd ? buf1 : buf0;
  *src = odd ? buf0 : buf1;
  return true;
}

// Level input: runs of w records, groups of kFan runs.  Every sample is ranked
// among the samples of its group, a lane per run of the group (the lanes per sample rounded up to
// a power of two, at most a wave's, which then takes two runs each), and order[group's first
// sample + rank] = the sample's index.
__global__ __launch_bounds__(256) void sample_rank_kernel(Event* buf0, Event* buf1, const uint32_t* d_n, uint32_t cap,
                                                          uint32_t level, uint32_t most, uint32_t* order) {
  const uint32_t n = d_n ? *d_n : cap;
  const uint32_t fan = fan_of(n), w = level_width(level, fan);
  const Event* in;
  Event* out;
  if (!level_buffers(n, level, buf0, buf1, &in, &out)) return;
  const uint32_t ns = (n + kSample - 1u) / kSample;
  const uint64_t group = (uint64_t)w * fan;                        // records per group
  uint32_t lanes = 1;                                              // lanes per sample, `most` at most
  while (lanes < most && lanes < fan && (uint64_t)lanes * w < n) lanes *= 2;
  const uint32_t t = blockIdx.x * 256u + threadIdx.x;
  const uint64_t s = (uint64_t)t / lanes;
  const uint32_t k = t % lanes;
  if (((uint64_t)t & ~63ull) / lanes >= ns) return;                // the whole wave is past the samples
  uint32_t rank = 0;
  const uint32_t i = sample_record((uint32_t)s, w, fan);
  const uint32_t g0 = (uint32_t)(i / group * group);               // first record of its group
  const bool is = s < ns && i < n;                                 // the last run may be short of its last sample
  if (is) {
    const uint32_t own = (i - g0) / w;
    const Rec me = load_rec(in + i);
    for (uint32_t r = k; r < fan; r += lanes) {
      const uint64_t r0 = (uint64_t)g0 + (uint64_t)r * w;          // first record of run r
      if (r0 >= n) break;
      const uint32_t len = (uint32_t)(n - r0 < w ? n - r0 : w);
      rank += r == own ? (uint32_t)(i - r0) / kSample
                       : count_before(in + r0 + sample_offset(r), samples_of(r, len), kSample, me.hi, me.lo, r < own);
    }
  }
  for (uint32_t off = lanes / 2u; off > 0; off >>= 1) rank += (uint32_t)__shfl_xor((int)rank, (int)off, kWave);
  if (is && k == 0) order[g0 / kSample + rank] = (uint32_t)s;
}

// A block merges, for bucket_samples of its group from rank b0 on (in sample order), the
// records from the first of them up to the first of the next block (the group's first block:
// from its first record; the last: to its end).
__global__ __launch_bounds__(kBucketThreads) void bucket_merge_kernel(Event* buf0, Event* buf1, const uint32_t* d_n,
                                                                      uint32_t cap, uint32_t level,
                                                                      const uint32_t* order) {
  __shared__ LdsRecs<kBucketCap> s;
  __shared__ uint32_t s_from[kFan], s_off[kFan + 1];
  const uint32_t n = d_n ? *d_n : cap;
  const Event* in;
  Event* out;
  if (!level_buffers(n, level, buf0, buf1, &in, &out)) return;
  const uint32_t fan = fan_of(n), w = level_width(level, fan), samples = bucket_samples(n, fan);
  const uint64_t group = (uint64_t)w * fan;
  const uint64_t per = (group / kSample + samples - 1u) / samples;  // blocks per group
  const uint64_t start = blockIdx.x / per * group;                 // first record of the block's group
  if (start >= n) return;
  const uint32_t g0 = (uint32_t)start;
  const uint32_t glen = (uint32_t)(n - g0 < group ? n - g0 : group);
  const uint32_t runs = (glen + w - 1u) / w;
  const uint32_t last = (runs - 1u) * w;                           // the group's last run may be short
  const uint32_t gs = last / kSample + samples_of(runs - 1u, glen - last);   // samples of the group
  const uint32_t b0 = (uint32_t)(blockIdx.x % per) * samples;
  if (b0 && b0 >= gs) return;
  // kFindLanes lanes each: the block's first record in run r, and the record past its last
  {
    const uint32_t job = threadIdx.x / kFindLanes, r = job >> 1, at = b0 + (job & 1u) * samples;
    const uint32_t r0 = g0 + r * w;
    const uint32_t len = r < runs ? (n - r0 < w ? n - r0 : w) : 0u;
    uint32_t c = at ? len : 0u, find = 0;
    Rec me{0, 0};
    uint32_t own = 0;
    if (at && at < gs) {
      const uint32_t i = sample_record(order[g0 / kSample + at], w, fan);   // the splitting record
      own = (i - g0) / w;
      if (r == own) {
        c = i - r0;
      } else {
        me = load_rec(in + i);
        find = len;
      }
    }
    const uint32_t f = count_before_lanes(in + r0, find, me.hi, me.lo, r < own);
    if (find) c = f;
    const uint32_t end = (uint32_t)__shfl_xor((int)c, (int)kFindLanes, kWave);
    if (threadIdx.x % (2u * kFindLanes) == 0) {
      s_from[r] = c;
      s_off[r + 1] = end - c;
    }
  }
  __syncthreads();
  // the run shares one after the other; the records of the group before the block's
  __shared__ uint32_t s_before;
  if (threadIdx.x < (uint32_t)kWave) {
    static_assert(kFan == 2 * kWave, "two runs per lane");
    const uint32_t r = 2u * threadIdx.x;
    const uint32_t l0 = s_off[r + 1], l1 = s_off[r + 2];
    uint32_t x = l0 + l1;
#pragma unroll
    for (int off = 1; off < kWave; off <<= 1) {
      const uint32_t y = (uint32_t)__shfl_up((int)x, off, kWave);
      if ((int)threadIdx.x >= off) x += y;
    }
    s_off[r + 1] = x - l1;
    s_off[r + 2] = x;
    const uint32_t f = wave_sum_u32(s_from[r] + s_from[r + 1]);
    if (threadIdx.x == 0) {
      s_off[0] = 0;
      s_before = f;
    }
  }
  __syncthreads();
  const uint32_t total = s_off[kFan];
  // records per thread, nearly always 1 (a uniform value, so that the loops over them branch as a wave)
  const uint32_t slots = __builtin_amdgcn_readfirstlane((total + kBucketThreads - 1u) / kBucketThreads);
  uint64_t hi[kBucketPer], lo[kBucketPer];
  uint32_t pos[kBucketPer], run[kBucketPer];
#pragma unroll
  for (uint32_t q = 0; q < kBucketPer; ++q) {
    if (q >= slots) break;
    const uint32_t i = threadIdx.x + q * kBucketThreads;
    pos[q] = i;
    run[q] = 0;
    hi[q] = lo[q] = ~0ull;
    if (i < total) {
      uint32_t a = 0, b = kFan - 1u;                               // the run r with s_off[r] <= i < s_off[r + 1]
      while (a < b) {
        const uint32_t mid = (a + b) >> 1;
        if (s_off[mid + 1] > i) b = mid; else a = mid + 1u;
      }
      run[q] = a;
      const Rec r = load_rec(in + g0 + (size_t)a * w + s_from[a] + (i - s_off[a]));
      hi[q] = r.hi;
      lo[q] = r.lo;
      s.put(i, r.hi, r.lo);
    }
  }
  __syncthreads();
  for (uint32_t m = 0; (1u << m) < runs; ++m) {                    // 2^m runs' shares are merged so far
    uint32_t cnt[kBucketPer], from[kBucketPer], len[kBucketPer], top = 0;
    bool right[kBucketPer];
#pragma unroll
    for (uint32_t q = 0; q < kBucketPer; ++q) {
      if (q >= slots) break;
      const uint32_t g = run[q] >> m, a = (g ^ 1u) << m, b = a + (1u << m);   // kFan is a power of two
      from[q] = s_off[a];
      len[q] = pos[q] < total ? s_off[b] - s_off[a] : 0u;
      right[q] = (g & 1u) != 0;
      cnt[q] = 0;
      top = len[q] > top ? len[q] : top;
    }
    for (uint32_t bit = top ? 1u << (31 - __builtin_clz(top)) : 0u; bit; bit >>= 1) {
      uint32_t ot[kBucketPer];
      bool tie = false;
#pragma unroll
      for (uint32_t q = 0; q < kBucketPer; ++q) {      // a probe past the share reads slot 0 and is not used
        if (q >= slots) break;
        const uint32_t c = cnt[q] + bit;
        ot[q] = s.time(c <= len[q] ? from[q] + c - 1u : 0u);
      }
#pragma unroll
      for (uint32_t q = 0; q < kBucketPer; ++q) {
        if (q >= slots) break;
        tie |= cnt[q] + bit <= len[q] && ot[q] == (uint32_t)(hi[q] >> 32);
      }
      if (__any(tie)) {                                // a branch of the whole wave, rarely taken
#pragma unroll
        for (uint32_t q = 0; q < kBucketPer; ++q) {
          if (q >= slots) break;
          const uint32_t c = cnt[q] + bit;
          if (c <= len[q] && s.before(from[q] + c - 1u, hi[q], lo[q], right[q])) cnt[q] = c;
        }
      } else {
#pragma unroll
        for (uint32_t q = 0; q < kBucketPer; ++q) {
          if (q >= slots) break;
          const uint32_t c = cnt[q] + bit;
          if (c <= len[q] && ot[q] < (uint32_t)(hi[q] >> 32)) cnt[q] = c;
        }
      }
    }
    __syncthreads();
#pragma unroll
    for (uint32_t q = 0; q < kBucketPer; ++q) {
      if (q >= slots) break;
      if (pos[q] < total) {
        // the left share's records move by those of the right one before them, and vice versa
        pos[q] = right[q] ? pos[q] - len[q] + cnt[q] : pos[q] + cnt[q];
        s.put(pos[q], hi[q], lo[q]);
      }
    }
    __syncthreads();
  }
  Event* to = out + g0 + s_before;
  for (uint32_t i = threadIdx.x; i < total; i += kBucketThreads) store_event(to + i, s.get(i));
}

// splits (optional): task y's splits at splits[y * stride + x], for tile x's first output rank
// (x <= the task's tile count; the last one is that of the task's total).
template <int kT>
__global__ __launch_bounds__(kT) void merge_tasks_kernel(const MergeTask* tasks, const uint32_t* splits,
                                                         uint32_t stride) {
  constexpr uint32_t kTile = kT * kPerThread;
  const MergeTask t = tasks[blockIdx.y];
  const uint32_t na = t.n_a1 + t.n_a2;
  const uint32_t total = na + t.n_b;
  const uint32_t t0 = blockIdx.x * kTile;
  if (t0 >= total) return;
  const ASrc A{t.a1, t.a2, t.n_a1};
  const OutMap om{{t.out[0], t.out[1], t.out[2]}, {t.end[0], t.end[1], t.end[2]}};
  merge_tile<kT>(A, na, t.b, t.n_b, t0, om, splits ? splits + (size_t)blockIdx.y * stride + blockIdx.x : nullptr);
}

// The merge-path splits of every tile boundary of every task, kSplitLanes lanes per boundary,
// so that the merge blocks start loading at once.  Boundary x of task y is output rank
// min(x * kTile, total); grid (ceil(boundaries / (256 / kSplitLanes)), ntasks) of 256 threads.
// Fewer lanes per boundary take more rounds but far fewer loads, which is what limits this
// launch: thousands of boundaries search at once and their probes are scattered lines.
template <int kT>
__global__ __launch_bounds__(256) void merge_partition_kernel(const MergeTask* tasks, uint32_t boundaries,
                                                              uint32_t* splits, uint32_t stride) {
  constexpr uint32_t kTile = kT * kPerThread;
  constexpr uint32_t kPer = 256u / kSplitLanes;         // boundaries per block
  const uint32_t x = blockIdx.x * kPer + threadIdx.x / kSplitLanes;
  if (blockIdx.x * kPer >= boundaries) return;          // the whole block is past the boundaries
  const MergeTask t = tasks[blockIdx.y];
  const uint32_t na = t.n_a1 + t.n_a2;
  const uint32_t total = na + t.n_b;
  // boundaries past the task's last tile boundary do not search (their groups stay in the loop)
  const bool active = x < boundaries && (uint64_t)x * kTile <= total + (uint64_t)kTile;
  const uint32_t d = (uint64_t)x * kTile < total ? x * kTile : total;
  const ASrc A{t.a1, t.a2, t.n_a1};
  const uint32_t s = group_merge_split<kSplitLanes>(A, na, t.b, t.n_b, d, active);
  if (active && threadIdx.x % kSplitLanes == 0) splits[(size_t)blockIdx.y * stride + x] = s;
}

// One wave: lane k < kInsertStripes + 1 takes segment k's record count (a stripe counter past
// seg_cap also counts the lanes that spilled), the segments' offsets are a wave prefix sum,
// and every offset is capped at max_total.
__global__ __launch_bounds__(64) void gather_inserts_kernel(uint32_t* seg_m, uint32_t seg_cap, uint32_t spill_cap,
                                                            uint32_t max_total, uint32_t* seg_pre, uint32_t* d_m,
                                                            WindowState* ws) {
  const uint32_t k = threadIdx.x;
  uint32_t n = 0;
  if (k <= kInsertStripes) {
    const uint32_t c = seg_m[k * kStripeWords], cap = k < kInsertStripes ? seg_cap : spill_cap;
    n = c < cap ? c : cap;
    seg_m[k * kStripeWords] = 0;
  }
  uint32_t inc = n;
  for (int off = 1; off < kWave; off <<= 1) {
    const uint32_t t = (uint32_t)__shfl_up((int)inc, off, kWave);
    if (k >= (uint32_t)off) inc += t;
  }
  const uint32_t exc = inc - n;
  const uint32_t total = (uint32_t)__shfl((int)inc, (int)kInsertStripes, kWave);
  const uint32_t m = total < max_total ? total : max_total;
  if (k <= kInsertStripes) seg_pre[k] = exc < max_total ? exc : max_total;
  if (k == 0) {
    seg_pre[kInsertStripes + 1] = m;
    *d_m = m;
    if (total > max_total) atomicOr(&ws->error, kErrQueueOverflow);
  }
}

// --- selection --------------------------------------------------------------------

__device__ __forceinline__ bool in_prefix(const Event& e, uint32_t wend, bool bounded, const Event& bound) {
  return e.ts < wend && (!bounded || !key_less(bound, e));
}

// The length of the prefix, by one wave: 64 probes a round.
__device__ __forceinline__ uint32_t wave_prefix(const Event* s, uint32_t n, uint32_t wend, bool bounded, const Event& bound) {
  uint32_t lo = 0, hi = n;                             // the prefix ends in [lo, hi]
  while (lo < hi) {
    const uint32_t step = (hi - lo + kWave - 1u) / kWave, i = lo + (uint32_t)lane_id() * step;
    const uint64_t out = __ballot(i < hi && !in_prefix(load_event(s + (i < hi ? i : lo)), wend, bounded, bound));
    if (out == 0) {
      lo = lo + (hi - lo - 1u) / step * step + 1u;     // past the last probe
    } else {
      const uint32_t f = (uint32_t)__ffsll((unsigned long long)out) - 1u;
      hi = lo + f * step;
      if (f) lo = lo + (f - 1u) * step + 1u;
    }
  }
  return lo;
}

// Each block finds the prefix's length for itself (four rounds of loads; as a launch of its own, by
// one thread's binary search, it took 6 us), and marks the first record of every LP in it.
__global__ __launch_bounds__(kThreads) void select_mark_kernel(const Event* const* d_s, const uint32_t* d_n,
                                                               const uint32_t* d_wend, const Event* d_bound,
                                                               const uint32_t* d_bound_valid, uint32_t* d_prefix,
                                                               uint32_t* first) {
  __shared__ uint32_t s_p;
  const Event* s = *d_s;
  if (threadIdx.x < (uint32_t)kWave) {
    const bool bounded = d_bound_valid && *d_bound_valid;
    const Event bound = bounded ? *d_bound : sentinel();
    const uint32_t p = wave_prefix(s, *d_n, *d_wend, bounded, bound);
    if (threadIdx.x == 0) {
      s_p = p;
      if (blockIdx.x == 0) *d_prefix = p;
    }
  }
  __syncthreads();
  const uint32_t p = s_p;
  for (uint32_t i = blockIdx.x * kThreads + threadIdx.x; i < p; i += gridDim.x * kThreads) atomicMin(&first[s[i].dst], i);
}

// The marked records of every tile of the prefix.
__global__ __launch_bounds__(kThreads) void select_count_kernel(const Event* const* d_s, const uint32_t* d_prefix,
                                                                const uint32_t* first, uint32_t* counts) {
  __shared__ uint32_t s_w[kThreads / kWave];
  const Event* s = *d_s;
  const uint32_t p = *d_prefix;
  for (uint32_t tile = blockIdx.x; (uint64_t)tile * kSelectTile < p; tile += gridDim.x) {
    const uint32_t base = tile * kSelectTile;
    uint32_t c = 0;
#pragma unroll
    for (uint32_t q = 0; q < kSelectTile / kThreads; ++q) {
      const uint32_t i = base + q * kThreads + threadIdx.x, x = i < p ? i : base;
      c += first[s[x].dst] == i ? 1u : 0u;             // i >= p is no record's place
    }
    c = wave_sum_u32(c);
    if (lane_id() == 0) s_w[threadIdx.x / kWave] = c;
    __syncthreads();
    if (threadIdx.x == 0) counts[tile] = s_w[0] + s_w[1] + s_w[2] + s_w[3];
    __syncthreads();
  }
}

// The prefix's records to deq and rest, a tile at a time; a block adds up the counts of the tiles
// before its own (as a launch of its own the scan of all counts took 5 us, which is more than the
// reading of a few hundred words by every block), and the one with the last tile publishes the totals.
__global__ __launch_bounds__(kThreads) void select_scatter_kernel(const Event* const* d_s, const uint32_t* d_prefix,
                                                                  uint32_t* first, const uint32_t* counts,
                                                                  Event* deq, Event* rest, uint32_t* d_deq_n,
                                                                  uint32_t* d_rest_n) {
  constexpr uint32_t kWaves = kThreads / kWave;
  __shared__ uint32_t s_w[kWaves], s_c[kWaves];
  const Event* s = *d_s;
  const uint32_t p = *d_prefix;
  constexpr uint32_t kItems = kSelectTile / kThreads;   // 4 consecutive records per thread
  const uint32_t wv = threadIdx.x / kWave;
  uint32_t earlier = 0, counted = 0;                    // marked records of the tiles before `counted`
  for (uint32_t tile = blockIdx.x; (uint64_t)tile * kSelectTile < p; tile += gridDim.x) {
    uint32_t c = 0;
    for (uint32_t i = counted + threadIdx.x; i < tile; i += kThreads) c += counts[i];
    counted = tile;
    const uint32_t i0 = tile * kSelectTile + threadIdx.x * kItems;
    bool mark[kItems];
    Event e[kItems];
    uint32_t mine = 0;
#pragma unroll
    for (uint32_t q = 0; q < kItems; ++q) {
      const uint32_t i = i0 + q;
      e[q] = load_event(s + (i < p ? i : p - 1u));
    }
#pragma unroll
    for (uint32_t q = 0; q < kItems; ++q) {
      mark[q] = first[e[q].dst] == i0 + q;              // i >= p is no record's place
      mine += mark[q] ? 1u : 0u;
    }
    uint32_t x = mine;   // inclusive scan over the block, in thread order
    for (int off = 1; off < kWave; off <<= 1) {
      const uint32_t y = (uint32_t)__shfl_up((int)x, off, kWave);
      if (lane_id() >= off) x += y;
    }
    c = wave_sum_u32(c);
    if (lane_id() == kWave - 1) s_w[wv] = x;
    if (lane_id() == 0) s_c[wv] = c;
    __syncthreads();
    uint32_t in_tile = 0, wave_off = 0;
#pragma unroll
    for (uint32_t w = 0; w < kWaves; ++w) {
      earlier += s_c[w];
      if (w < wv) wave_off += s_w[w];
      in_tile += s_w[w];
    }
    uint32_t before = earlier + wave_off + x - mine;   // marked records before i0
#pragma unroll
    for (uint32_t q = 0; q < kItems; ++q) {
      const uint32_t i = i0 + q;
      if (i < p) {
        if (mark[q]) {
          store_event(deq + before, e[q]);
          first[e[q].dst] = 0xFFFFFFFFu;
          ++before;
        } else {
          store_event(rest + (i - before), e[q]);
        }
      }
    }
    if (threadIdx.x == 0 && (uint64_t)(tile + 1u) * kSelectTile >= p) {
      *d_deq_n = earlier + in_tile;
      *d_rest_n = p - (earlier + in_tile);
    }
    __syncthreads();                                   // s_w and s_c are rewritten
  }
  if (p == 0 && blockIdx.x == 0 && threadIdx.x == 0) {
    *d_deq_n = 0;
    *d_rest_n = 0;
  }
}

uint32_t grid_of(uint64_t items, uint32_t per_block) {
  const uint64_t g = (items + per_block - 1) / per_block;
  return g ? (uint32_t)g : 1u;
}

// Work accounting (queues created with collect_stats): one small launch after a primitive
// adds the records it handled to a counter, so the primitive's own kernels are unchanged.
__global__ void acct_count_kernel(const uint32_t* d_n, uint32_t cap, unsigned long long* acct) {
  if (threadIdx.x == 0) atomicAdd(acct, (unsigned long long)min(*d_n, cap));
}

__global__ __launch_bounds__(256) void acct_tasks_kernel(const MergeTask* tasks, uint32_t ntasks,
                                                         unsigned long long* acct) {
  unsigned long long s = 0;
  for (uint32_t t = threadIdx.x; t < ntasks; t += blockDim.x)
    s += (unsigned long long)tasks[t].n_a1 + tasks[t].n_a2 + tasks[t].n_b;
  if (s) atomicAdd(acct, s);
}

}  // namespace

bool valid_sort_tile(uint32_t tile) { return tile == 1024 || tile == 2048 || tile == 4096; }

size_t sort_order_words(uint64_t cap) { return (size_t)((cap + kSample - 1) / kSample) + 1; }

gpq_status sort_records(const Event* in, Event* buf0, Event* buf1, uint32_t* order, const uint32_t* d_n, uint32_t cap,
                        hipStream_t stream, unsigned long long* acct, const uint32_t* seg_pre, uint32_t seg_cap) {
  hipLaunchKernelGGL(tile_sort_kernel, dim3(grid_of(cap, kRun)), dim3(kTileThreads), 0, stream, in, buf0, buf1,
                     d_n, cap, seg_pre, seg_cap);
  // Grids for any number of records up to cap, and so for either width of the levels: a group's blocks hold 768
  // records or more on average, and its last one may hold fewer.
  const uint64_t blocks = cap / 762u + 45u;
  for (uint32_t level = 1; level <= sort_levels(cap); ++level) {
    const uint64_t w = level == 1 ? kRun : (level == 2 ? (uint64_t)kRun * fan_of(cap) : (uint64_t)kRun * kFan * kFan);
    const uint64_t runs = std::min<uint64_t>((cap + w - 1) / w, kWave);
    const uint32_t lanes = 1u << log2u(runs);
    hipLaunchKernelGGL(sample_rank_kernel, dim3(grid_of(((uint64_t)cap + kSample - 1) / kSample * lanes, 256)), dim3(256),
                       0, stream, buf0, buf1, d_n, cap, level, lanes, order);
    hipLaunchKernelGGL(bucket_merge_kernel, dim3((uint32_t)blocks), dim3(kBucketThreads), 0, stream, buf0, buf1, d_n, cap,
                       level, order);
  }
  GPQ_HIP(hipGetLastError());
  if (!acct) return GPQ_OK;
  hipLaunchKernelGGL(acct_count_kernel, dim3(1), dim3(64), 0, stream, d_n, cap, acct);
  GPQ_HIP(hipGetLastError());
  return GPQ_OK;
}

uint32_t merge_split_words(uint64_t max_total, uint32_t tile) {
  return (uint32_t)((max_total + tile - 1) / tile) + 2u;
}

namespace {
template <int kT>
gpq_status merge_tasks_t(const MergeTask* d_tasks, uint32_t ntasks, uint64_t max_total, hipStream_t stream,
                         uint32_t* splits, uint32_t stride) {
  constexpr uint32_t kTile = kT * kPerThread;
  const uint32_t gx = grid_of(max_total, kTile);
  if (splits) {
    GPQ_CHECK_ARG(stride >= gx + 1u, "merge_tasks: split buffer stride below the tile count + 1");
    hipLaunchKernelGGL(merge_partition_kernel<kT>, dim3(ceil_div(gx + 1u, 256u / kSplitLanes), ntasks), dim3(256), 0,
                       stream, d_tasks, gx + 1u, splits, stride);
  }
  hipLaunchKernelGGL(merge_tasks_kernel<kT>, dim3(gx, ntasks), dim3(kT), 0, stream, d_tasks,
                     static_cast<const uint32_t*>(splits), stride);
  return GPQ_OK;
}
}  // namespace

gpq_status merge_tasks(const MergeTask* d_tasks, uint32_t ntasks, uint64_t max_total, hipStream_t stream,
                       uint32_t tile, unsigned long long* acct, uint32_t* splits, uint32_t stride,
                       uint64_t partition_min) {
  if (ntasks == 0) return GPQ_OK;
  // Below 2^20 records a task's blocks search their splits themselves: the partition launch
  // would cost about what it saves (four heaps of a quarter of the LPs each measured 2.5e8 events/s
  // without it and 1.7e8 with it at 2^20 LPs; one heap and the GAQ gain).
  if (max_total < partition_min) splits = nullptr;
  switch (tile) {
    case 1024: GPQ_TRY(merge_tasks_t<128>(d_tasks, ntasks, max_total, stream, splits, stride)); break;
    case 2048: GPQ_TRY(merge_tasks_t<256>(d_tasks, ntasks, max_total, stream, splits, stride)); break;
    case 4096: GPQ_TRY(merge_tasks_t<512>(d_tasks, ntasks, max_total, stream, splits, stride)); break;
    default:
      set_error("merge tile must be 1024, 2048 or 4096 records");
      return GPQ_ERR_INVALID;
  }
  GPQ_HIP(hipGetLastError());
  if (acct) {
    hipLaunchKernelGGL(acct_tasks_kernel, dim3(1), dim3(256), 0, stream, d_tasks, ntasks, acct);
    GPQ_HIP(hipGetLastError());
  }
  return GPQ_OK;
}

gpq_status select_safe(const Event* const* s, const uint32_t* d_n, uint32_t cap, const uint32_t* d_wend,
                       const Event* d_bound, const uint32_t* d_bound_valid, const SelectBufs& b, Event* deq,
                       Event* rest, hipStream_t stream, unsigned long long* acct) {
  const uint32_t nblk = grid_of(cap, kSelectTile);
  uint32_t* counts = b.scratch;
  const uint32_t blocks = std::min(nblk, kSelectBlocks);
  hipLaunchKernelGGL(select_mark_kernel, dim3(std::min(grid_of(cap, kThreads), kSelectBlocks)), dim3(kThreads), 0, stream,
                     s, d_n, d_wend, d_bound, d_bound_valid, b.d_prefix, b.first);
  hipLaunchKernelGGL(select_count_kernel, dim3(blocks), dim3(kThreads), 0, stream, s, b.d_prefix, b.first, counts);
  hipLaunchKernelGGL(select_scatter_kernel, dim3(blocks), dim3(kThreads), 0, stream, s, b.d_prefix, b.first, counts, deq,
                     rest, b.d_deq_n, b.d_rest_n);
  GPQ_HIP(hipGetLastError());
  if (acct) {
    hipLaunchKernelGGL(acct_count_kernel, dim3(1), dim3(64), 0, stream, b.d_prefix, cap, acct);
    GPQ_HIP(hipGetLastError());
  }
  return GPQ_OK;
}

gpq_status gather_inserts(uint32_t* seg_m, uint32_t seg_cap, uint32_t spill_cap, uint32_t max_total, uint32_t* seg_pre,
                          uint32_t* d_m, WindowState* ws, hipStream_t stream) {
  static_assert(kInsertStripes + 1 <= kWave, "one wave gathers the stripes");
  hipLaunchKernelGGL(gather_inserts_kernel, dim3(1), dim3(kWave), 0, stream, seg_m, seg_cap, spill_cap, max_total,
                     seg_pre, d_m, ws);
  GPQ_HIP(hipGetLastError());
  return GPQ_OK;
}

}  // namespace gpq
