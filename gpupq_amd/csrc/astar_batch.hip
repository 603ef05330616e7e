// astar_batch.hip -- batched A*: many independent grid queries, one workgroup per query.
//
// The reference runs one block per agent and pulls agents from an atomic counter
// (get_new_agent, src/a_star.cu:149-164); thread 0 pops up to 8 vertices, the block expands
// them, deduplicates, and thread 0 inserts or updates (src/a_star.cu:325-374,441-569).  Here
// the open list of a query is a row of buckets by f: bucket i holds the pending entries with
// f in [i * 2^s, (i + 1) * 2^s), a stack, for the kBuckets buckets from the lowest pending one on;
// entries beyond them (or for a full bucket) wait in an unsorted far store, which is scanned when
// its smallest f comes up.  Each iteration the workgroup's K threads take K entries of the lowest
// buckets, the newest of each first, and expand them in parallel; g is relaxed with atomicMin, so
// entries made stale by a cheaper path are recognised when taken.
// Newest first, because among cells of one f the deepest are nearest to the goal: with 4 neighbours
// and few obstacles most of the grid has the goal's own f, and oldest first expanded all of it.  64
// queries of side 2048, 4-connected, no obstacles: 102 ms oldest first, 42 newest first (73 with the
// binary heaps named below); 512 queries of side 256 to 2048, 8-connected, 256 threads: 19.3 and 12.7 ms.
// An entry's successors have f at least its own (consistent heuristic), so no entry is ever
// appended below the lowest bucket.  The search of a query ends when the best goal cost found is
// <= the smallest f that may be pending, which makes the result the optimal cost.
//
// What bounds it: the latency of an iteration (three barriers and four dependent accesses: bucket
// entry, g and obstacle bits, relaxations, append), times the longest query's iterations, which its
// path's steps bound from below.  Expanding an entry's best successor in the same iteration (2
// to 16 of a chain) made iterations longer by more than it saved (15 to 29 ms where without it was 12).  The
// list this replaced, a binary heap per thread, moved some 3 KB per expansion in sifts over
// scattered lines and took 19 us per iteration against 7 us here: 512 queries of side 256 to
// 2048, 8-connected, in 512-thread workgroups 39.0 -> 14.6 ms, in 256-thread ones 30.4 -> 12.8.
//
// Entry = f << 22 | cell.  Limits that follow: side <= 2048 (cell < 2^22), f < 2^26.
//
// g entries carry a generation tag so that a slot is not cleared per query: entry =
// tag << 26 | g, where the tag of the slot's current query is smaller than every tag written
// before (tags count down from 62; 63 = never written), so atomicMin still relaxes and an
// entry of an older query compares as infinite.  After tag 0 the slot is cleared once.
#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstring>
#include <thread>

#include "astar.h"

namespace gpq {

namespace {

constexpr uint32_t kMaxSide = 2048;
constexpr uint32_t kNoCost = 0xFFFFFFFFu;
constexpr int kMaxWaves = 16;

// Buckets of a query's open list: one per lane of the wave that plans an iteration.
constexpr uint32_t kBuckets = 64;
// f values per bucket, as a power of two: f - h(source) is even on both kinds of grid, so a bucket
// is one f value.  Wider buckets expand more cells out of order: 512 queries of side 256 to 2048,
// 8-connected, 512 threads each, took 14.7 ms at width 2, 16.0 at 4 and 17.4 at 8.  Taking entries of
// the lowest 32, 16 or 8 buckets only (fewer expansions, idler iterations) took 13.4, 12.8 and 15.1 ms;
// with 64 threads and 256 queries 20.5, 21.5 and 24.0 against 20.9 without a limit.
constexpr uint32_t kShift = 1;
constexpr uint32_t kNoBucket = 0xFFFFFFFFu;

struct BatchQuery {
  uint32_t side, conn, sx, sy, tx, ty;
  uint64_t bit_off;                     // first bitmap word of the query in the pool
};

constexpr uint32_t kTagShift = 26;
constexpr uint32_t kTagNever = 63;

// Per-slot state: the generation tag of the slot's query, and (plain drive) the search
// state between launches.
struct SlotState {
  uint32_t best;
  uint32_t overflow;
  uint32_t tag;
  uint32_t pad;
  unsigned long long expanded;
};

// A query's open list between the launches of the plain drive.
struct SlotList {
  uint32_t cnt[kBuckets];
  uint32_t base, far_n, far_min, pad;
};

struct BatchDev {
  const BatchQuery* q;
  const uint32_t* bits;                 // pooled obstacle bitmaps
  uint32_t* g;                          // [slot][g_stride]
  uint64_t* far;                        // [slot][far_cap]
  uint64_t* bucket;                     // [slot][kBuckets][bucket_cap]
  SlotList* list;                       // [slot] (plain drive)
  SlotState* slot;
  long long* cost;                      // [query]
  unsigned long long* expanded;         // [query]
  uint32_t* flags;                      // [query] 1 = open-list overflow
  unsigned long long* clk;              // [query][2] device wall clock at pickup and at completion
  const uint32_t* ids;                  // queries of this launch
  uint32_t n;
  uint32_t* counter;                    // work counter of the persistent launch
  uint32_t slot_base;                   // workgroup b of the launch uses slot slot_base + b
  uint64_t g_stride;
  uint64_t far_cap;
  uint32_t bucket_cap;
};

__device__ __forceinline__ uint64_t make_entry(uint32_t f, uint32_t cell) { return ((uint64_t)f << 22) | cell; }
__device__ __forceinline__ uint32_t entry_f(uint64_t e) { return (uint32_t)(e >> 22); }
__device__ __forceinline__ uint32_t entry_cell(uint64_t e) { return (uint32_t)(e & 0x3FFFFFu); }

struct Shared {
  uint32_t best;
  uint32_t overflow;
  uint32_t qi;
  uint32_t base;                 // the lowest bucket that may hold an entry (f >> shift)
  uint32_t cnt[kBuckets];        // entries in bucket b (at b mod kBuckets)
  uint32_t pre[kBuckets + 1];    // this iteration: entries taken from the buckets before base + i
  uint32_t from[kBuckets];       // and the first one taken from base + i
  uint32_t far_n, far_min, far_keep;
  uint32_t act;                  // this iteration: kTake, kScan or kFinish
  unsigned long long expanded[kMaxWaves];
};
enum : uint32_t { kTake = 0, kScan = 1, kFinish = 2 };

// Where a query's open list lives.
struct OpenList {
  uint64_t* far;
  uint64_t* bucket;
  uint64_t far_cap;
  uint32_t bucket_cap;
};

// Appends e to its bucket, or to the far store when the bucket is full or beyond the row.
__device__ __forceinline__ void open_push(Shared& sh, const OpenList& o, uint64_t e) {
  const uint32_t f = entry_f(e), b = f >> kShift;
  if (b - sh.base < kBuckets) {
    const uint32_t pos = atomicAdd(&sh.cnt[b % kBuckets], 1u);
    if (pos < o.bucket_cap) {
      o.bucket[(uint64_t)(b % kBuckets) * o.bucket_cap + pos] = e;
      return;
    }
  }
  const uint32_t pos = atomicAdd(&sh.far_n, 1u);
  if (pos < o.far_cap) {
    o.far[pos] = e;
    atomicMin(&sh.far_min, f);
  } else {
    sh.overflow = 1;
  }
}

// One wave, lane i for bucket base + i: retires what the last iteration took, moves base to the
// lowest bucket with entries and lists the first K pending entries.  Asks for a scan of the
// far store when that holds an entry below every bucket's, and ends the search when nothing
// pending can be below `best`.
__device__ __forceinline__ void open_plan(Shared& sh, const OpenList& o, uint32_t K) {
  const uint32_t lane = (uint32_t)lane_id();
  uint32_t base = sh.base;
  uint32_t b = (base + lane) % kBuckets;
  const uint32_t n = min(sh.cnt[b], o.bucket_cap);
  sh.cnt[b] = n;
  const uint64_t some = __ballot(n != 0);
  const uint32_t skip = some ? (uint32_t)__builtin_ctzll(some) : kBuckets;
  const uint32_t far_n = sh.far_n < o.far_cap ? sh.far_n : (uint32_t)o.far_cap;
  const uint32_t far_b = far_n ? sh.far_min >> kShift : kNoBucket;
  const uint32_t low = some ? base + skip : kNoBucket;   // the lowest bucket with entries
  const uint32_t lowest = far_b < low ? far_b : low;
  const uint32_t best = sh.best;
  if (lowest == kNoBucket || (lowest << kShift) >= best) {
    if (lane == 0) sh.act = kFinish;
    return;
  }
  if (far_b < low) {
    if (lane == 0) {
      sh.act = kScan;
      sh.base = far_b;
      sh.far_n = far_n;
    }
    return;
  }
  // bucket base + skip + lane
  const uint32_t src = lane + skip;
  const uint32_t n2 = (uint32_t)__shfl((int)n, (int)(src & 63u), kWave);
  const uint32_t mine = src < kBuckets ? n2 : 0u;
  uint32_t inc = mine;
#pragma unroll
  for (int off = 1; off < kWave; off <<= 1) {
    const uint32_t t = (uint32_t)__shfl_up((int)inc, off, kWave);
    if (lane >= (uint32_t)off) inc += t;
  }
  const uint32_t before = inc - mine < K ? inc - mine : K, last = inc < K ? inc : K;
  const uint32_t left = mine - (last - before);      // the newest entries are taken
  sh.pre[lane + 1] = last;
  sh.from[lane] = left;
  if (src < kBuckets) sh.cnt[(base + src) % kBuckets] = left;
  if (lane == 0) {
    sh.pre[0] = 0;
    sh.base = base + skip;
    sh.act = kTake;
    sh.far_n = far_n;
  }
}

// The far store's entries that the row of buckets now covers move into it; those that cannot
// beat the goal found are dropped, the others stay, closed up in place: a chunk is read whole
// before any of it is written, and never to a place past what has been read.
__device__ void open_scan(Shared& sh, const OpenList& o, uint32_t far_n) {
  constexpr uint32_t kU = 4;
  const uint32_t K = blockDim.x, lane = (uint32_t)lane_id();
  if (threadIdx.x == 0) {
    sh.far_min = kNoBucket;
    sh.far_keep = 0;
  }
  __syncthreads();
  const uint32_t best = sh.best, base = sh.base;
  uint32_t kept_min = kNoBucket;
  for (uint32_t c0 = 0; c0 < far_n; c0 += kU * K) {
    uint64_t e[kU];
    bool keep[kU];
#pragma unroll
    for (uint32_t u = 0; u < kU; ++u) {
      const uint32_t i = c0 + u * K + threadIdx.x;
      e[u] = i < far_n ? o.far[i] : ~0ull;
    }
    __syncthreads();                                 // the chunk is in registers
    uint32_t n_keep = 0;
#pragma unroll
    for (uint32_t u = 0; u < kU; ++u) {
      const uint32_t i = c0 + u * K + threadIdx.x;
      keep[u] = i < far_n && entry_f(e[u]) < best;
      const uint32_t b = entry_f(e[u]) >> kShift;
      if (keep[u] && b - base < kBuckets) {
        const uint32_t pos = atomicAdd(&sh.cnt[b % kBuckets], 1u);
        if (pos < o.bucket_cap) {
          o.bucket[(uint64_t)(b % kBuckets) * o.bucket_cap + pos] = e[u];
          keep[u] = false;
        }
      }
      n_keep += (uint32_t)__popcll(__ballot(keep[u]));
    }
    uint32_t at = 0;
    if (lane == 0 && n_keep) at = atomicAdd(&sh.far_keep, n_keep);
    at = (uint32_t)__shfl((int)at, 0, kWave);
#pragma unroll
    for (uint32_t u = 0; u < kU; ++u) {
      const uint64_t m = __ballot(keep[u]);
      if (keep[u]) {
        o.far[at + (uint32_t)__popcll(m & ((1ull << lane) - 1ull))] = e[u];
        kept_min = min(kept_min, entry_f(e[u]));
      }
      at += (uint32_t)__popcll(m);
    }
  }
  if (kept_min != kNoBucket) atomicMin(&sh.far_min, kept_min);
  __syncthreads();
  if (threadIdx.x == 0) sh.far_n = sh.far_keep;
  __syncthreads();
}

// Searches query `qidx` in `slot`.  max_iters = 0: to the end; otherwise at most that many
// iterations, keeping the state in the slot (resume continues it).  Returns true when done.
__device__ bool search_query(const BatchDev& d, Shared& sh, uint32_t qidx, uint32_t slot, uint32_t max_iters,
                             bool resume) {
  const uint32_t tid = threadIdx.x, K = blockDim.x;
  const BatchQuery Q = d.q[qidx];
  const uint32_t W = Q.side;
  const uint32_t* bits = d.bits + Q.bit_off;
  uint32_t* g = d.g + (uint64_t)slot * d.g_stride;
  const OpenList o{d.far + (uint64_t)slot * d.far_cap, d.bucket + (uint64_t)slot * kBuckets * d.bucket_cap, d.far_cap,
                   d.bucket_cap};
  const uint32_t source = Q.sy * W + Q.sx, target = Q.ty * W + Q.tx;

  unsigned long long expanded = 0;
  uint32_t tag;
  if (!resume) {
    if (tid == 0) d.clk[2 * qidx] = wall_clock64();
    const uint32_t prev = d.slot[slot].tag;
    if (prev == 0) {                                   // tags exhausted: clear the slot once
      // the whole slot, not only this query's cells: a later, larger query in the slot would
      // otherwise meet entries of older queries whose tags are below its own
      for (uint64_t c = tid; c < d.g_stride; c += K) g[c] = 0xFFFFFFFFu;
    }
    tag = prev == 0 ? kTagNever - 1 : prev - 1;
    if (tid < kBuckets) sh.cnt[tid] = 0;
    if (tid == 0) {
      sh.best = source == target ? 0u : kNoCost;
      sh.overflow = 0;
      sh.far_n = 0;
      sh.far_min = kNoBucket;
      sh.base = grid_heur(Q.conn, (int)Q.sx, (int)Q.sy, (int)Q.tx, (int)Q.ty) >> kShift;
    }
    __syncthreads();
    if (tid == 0) {
      d.slot[slot].tag = tag;
      if (source != target) {
        __hip_atomic_store(&g[source], tag << kTagShift, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        open_push(sh, o, make_entry(grid_heur(Q.conn, (int)Q.sx, (int)Q.sy, (int)Q.tx, (int)Q.ty), source));
      }
    }
  } else {
    tag = d.slot[slot].tag;
    if (tid < kBuckets) sh.cnt[tid] = d.list[slot].cnt[tid];
    if (tid == 0) {
      sh.best = d.slot[slot].best;
      sh.overflow = d.slot[slot].overflow;
      sh.base = d.list[slot].base;
      sh.far_n = d.list[slot].far_n;
      sh.far_min = d.list[slot].far_min;
    }
  }
  const uint32_t tag_bits = tag << kTagShift;
  __syncthreads();

  bool finished = false;
  uint32_t it = 0;
  for (;;) {
    if (tid < (uint32_t)kWave) open_plan(sh, o, K);
    __syncthreads();
    const uint32_t act = sh.act;
    if (act == kFinish) { finished = true; break; }
    if (act == kScan) {
      open_scan(sh, o, sh.far_n);
      continue;
    }
    // --- take and expand ------------------------------------------------------------------
    const bool some = tid < sh.pre[kBuckets];
    uint32_t cell = 0, f = 0, g0 = 0, g_now = 0, nbr = 0;
    int x = 0, y = 0;
    if (some) {
      uint32_t lo = 0, hi = kBuckets - 1;              // the bucket i with pre[i] <= tid < pre[i + 1]
      while (lo < hi) {
        const uint32_t mid = (lo + hi) >> 1;
        if (sh.pre[mid + 1] > tid) hi = mid; else lo = mid + 1;
      }
      const uint64_t e = o.bucket[(uint64_t)((sh.base + lo) % kBuckets) * o.bucket_cap + sh.from[lo] + (tid - sh.pre[lo])];
      cell = entry_cell(e);
      f = entry_f(e);
      x = (int)(cell % W);
      y = (int)(cell / W);
      g0 = f - grid_heur(Q.conn, x, y, (int)Q.tx, (int)Q.ty);
      g_now = __hip_atomic_load(&g[cell], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      nbr = free_neighbours(bits, Q.conn, x, y, (int)W, (int)W);
    }
    __syncthreads();                                   // every entry is read: its place may be taken
    if (some) {
      if ((tag_bits | g0) == g_now && f < *(volatile uint32_t*)&sh.best) {
        ++expanded;
        // all relaxations in flight at once: a neighbour's improvement does not depend on another's
        uint32_t old[8];
#pragma unroll
        for (uint32_t k = 0; k < 8; ++k) {
          const uint32_t v = (uint32_t)(y + nbr_dy(k)) * W + (uint32_t)(x + nbr_dx(k));
          old[k] = ((nbr >> k) & 1u) && v != target ? atomicMin(&g[v], tag_bits | (g0 + nbr_cost(Q.conn, k))) : 0u;
        }
#pragma unroll
        for (uint32_t k = 0; k < 8; ++k) {
          if (!((nbr >> k) & 1u)) continue;
          const int nx = x + nbr_dx(k), ny = y + nbr_dy(k);
          const uint32_t v = (uint32_t)ny * W + (uint32_t)nx;
          const uint32_t g2 = g0 + nbr_cost(Q.conn, k);
          if (v == target) {
            atomicMin(&sh.best, g2);
            continue;
          }
          if (old[k] <= (tag_bits | g2)) continue;
          const uint32_t f2 = g2 + grid_heur(Q.conn, nx, ny, (int)Q.tx, (int)Q.ty);
          if (f2 >= *(volatile uint32_t*)&sh.best) continue;   // cannot beat the goal found
          open_push(sh, o, make_entry(f2, v));
        }
      }
    }
    __syncthreads();
    ++it;
    if (max_iters && it >= max_iters) break;
  }

  // --- results or saved state ---------------------------------------------------------------
  unsigned long long e = expanded;
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) e += __shfl_xor(e, off, kWave);
  if (lane_id() == 0) sh.expanded[tid / kWave] = e;
  __syncthreads();
  if (!finished && tid < kBuckets) d.list[slot].cnt[tid] = min(sh.cnt[tid], o.bucket_cap);
  if (tid == 0) {
    unsigned long long tot = 0;
    for (uint32_t w = 0; w < K / kWave; ++w) tot += sh.expanded[w];
    if (resume) tot += d.slot[slot].expanded;
    if (finished) {
      d.clk[2 * qidx + 1] = wall_clock64();
      d.cost[qidx] = sh.best == kNoCost ? -1ll : (long long)sh.best;
      d.expanded[qidx] = tot;
      d.flags[qidx] = sh.overflow;
    } else {
      d.slot[slot] = SlotState{sh.best, sh.overflow, tag, 0u, tot};
      d.list[slot].base = sh.base;
      d.list[slot].far_n = sh.far_n;
      d.list[slot].far_min = sh.far_min;
    }
  }
  __syncthreads();
  return finished;
}

// Persistent drive: each workgroup owns slot blockIdx.x and pulls queries until none is left.
__global__ __launch_bounds__(1024) void astar_batch_kernel(BatchDev d) {
  __shared__ Shared sh;
  for (;;) {
    if (threadIdx.x == 0) sh.qi = atomicAdd(d.counter, 1u);
    __syncthreads();
    const uint32_t qi = sh.qi;
    __syncthreads();
    if (qi >= d.n) break;
    search_query(d, sh, d.ids[qi], d.slot_base + blockIdx.x, 0, false);
  }
}

// Plain drive: one iteration of query ids[0] in slot slot_base per launch.
__global__ __launch_bounds__(1024) void astar_batch_step_kernel(BatchDev d, uint32_t resume, uint32_t* done) {
  __shared__ Shared sh;
  const bool fin = search_query(d, sh, d.ids[0], d.slot_base, 1, resume != 0);
  if (threadIdx.x == 0) *done = fin ? 1u : 0u;
}

__global__ void zero_u32_kernel(uint32_t* p) { *p = 0; }

// threads * (8 * stage_capacity + 4) accepted: the bound that stage_capacity has always had, though the open
// list needs no staging now and takes any number of inserts per iteration.
constexpr size_t kStageLimit = 64 * 1024;

// Entries a bucket holds: half of the list's capacity over the row, within [256, 8192] (64 KiB); a fuller bucket spills into the far store.
uint32_t bucket_cap_for(const gpq_batch_tuning& t) {
  const uint64_t c = (uint64_t)t.heap_capacity * t.threads_per_query / (2u * kBuckets);
  return (uint32_t)std::min<uint64_t>(std::max<uint64_t>(c, 256), 8192);
}

__global__ void init_slots_kernel(SlotState* s, uint32_t n) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) s[i] = SlotState{kNoCost, 0u, kTagNever, 0u, 0ull};
}

uint32_t gen_blocks(uint64_t n) {
  const uint64_t g = (n + 255) / 256;
  return (uint32_t)std::min<uint64_t>(std::max<uint64_t>(g, 1), 65536);
}

bool host_blocked(uint32_t seed, uint32_t tag, uint32_t query, uint32_t threshold, uint64_t c) {
  const uint4 r = philox4x32_10(make_uint4((uint32_t)(c >> 2), query, tag, 2u), make_uint2(seed, 0u));
  const uint32_t rr[4] = {r.x, r.y, r.z, r.w};
  return rr[c & 3] < threshold;
}

}  // namespace

struct AstarBatch::Dev : BatchDev {};

// Query q of the synthetic batch: shape from Philox({q, 0, 3, 0}), source and target from
// the first free candidates of Philox({a, q, 4 | 5, 0}), obstacles from stream tag 1.
gpq_status query_synthetic(uint32_t seed, uint32_t q, gpq_query_spec* out) {
  const uint4 r = philox4x32_10(make_uint4(q, 0u, 3u, 0u), make_uint2(seed, 0u));
  const double u0 = (double)r.x * 0x1p-32, u1 = (double)r.y * 0x1p-32;
  gpq_query_spec s{};
  s.side = (uint32_t)std::floor(256.0 * std::exp2(3.0 * u0) + 0.5);
  s.threshold = (uint32_t)((0.1 + 0.2 * u1) * 4294967296.0);
  s.connectivity = 8;
  s.seed = seed;
  s.stream_tag = 1;
  s.query = q;
  for (int which = 0; which < 2; ++which) {
    for (uint32_t a = 0;; ++a) {
      const uint4 p = philox4x32_10(make_uint4(a, q, 4u + (uint32_t)which, 0u), make_uint2(seed, 0u));
      const uint32_t x = (uint32_t)(((uint64_t)p.x * s.side) >> 32), y = (uint32_t)(((uint64_t)p.y * s.side) >> 32);
      if (!host_blocked(seed, s.stream_tag, q, s.threshold, (uint64_t)y * s.side + x)) {
        if (which == 0) { s.sx = x; s.sy = y; } else { s.tx = x; s.ty = y; }
        break;
      }
      if (a > (1u << 20)) {
        set_error("query_synthetic: no free cell found");
        return GPQ_ERR_INVALID;
      }
    }
  }
  *out = s;
  return GPQ_OK;
}

gpq_status AstarBatch::create(const gpq_query_spec* sp, uint32_t count, const gpq_batch_tuning& t, AstarBatch** out) {
  GPQ_CHECK_ARG(sp && count >= 1, "batch: no queries");
  gpq_batch_tuning tu = t;
  if (!tu.threads_per_query) tu.threads_per_query = 256;
  if (!tu.heap_capacity) tu.heap_capacity = 2048;
  if (!tu.stage_capacity) tu.stage_capacity = 8;
  GPQ_CHECK_ARG(tu.threads_per_query >= 64 && tu.threads_per_query <= 1024 && is_pow2(tu.threads_per_query),
                "batch: threads_per_query must be a power of two in [64, 1024]");
  GPQ_CHECK_ARG(tu.heap_capacity >= 16 && tu.heap_capacity <= (1u << 20), "batch: heap_capacity out of range");
  GPQ_CHECK_ARG(tu.stage_capacity >= 1 && tu.stage_capacity <= 64, "batch: stage_capacity must be in [1, 64]");
  GPQ_CHECK_ARG((size_t)tu.threads_per_query * (tu.stage_capacity * 8 + 4) <= kStageLimit,
                "batch: threads_per_query * (8 * stage_capacity + 4) must be <= 65536");
  uint64_t max_cells = 0, words = 0;
  std::vector<BatchQuery> hq(count);
  std::vector<uint64_t> off(count);
  for (uint32_t i = 0; i < count; ++i) {
    const gpq_query_spec& s = sp[i];
    GPQ_CHECK_ARG(s.side >= 1 && s.side <= kMaxSide, "batch: side must be in [1, 2048]");
    GPQ_CHECK_ARG(s.connectivity == 4 || s.connectivity == 8, "batch: connectivity must be 4 or 8");
    GPQ_CHECK_ARG(s.sx < s.side && s.sy < s.side && s.tx < s.side && s.ty < s.side, "batch: endpoint outside grid");
    const uint64_t cells = (uint64_t)s.side * s.side;
    max_cells = std::max(max_cells, cells);
    off[i] = words;
    hq[i] = BatchQuery{s.side, s.connectivity, s.sx, s.sy, s.tx, s.ty, words};
    words += ((cells + 31) / 32 + 3) & ~3ull;
  }
  int dev = 0, cus = 0;
  GPQ_HIP(hipGetDevice(&dev));
  GPQ_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
  int per_cu = 0;
  GPQ_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, astar_batch_kernel, (int)tu.threads_per_query, 0));
  // a slot holds a whole grid's g values, so the slots grow with the workgroups per CU; an
  // iteration is bound by latency, and two 512-thread workgroups per CU already overlap theirs
  per_cu = std::min(per_cu, std::min<int>(8, 512 / (int)tu.threads_per_query + 1));
  uint32_t resident = tu.max_resident ? tu.max_resident : (uint32_t)std::max(1, cus * std::max(per_cu, 1));
  resident = std::min(resident, count);
  tu.max_resident = resident;

  AstarBatch* b = new AstarBatch();
  b->specs.assign(sp, sp + count);
  b->tuning = tu;
  b->resident = resident;
  b->cell_off = off;
  auto fail = [&](gpq_status s) { delete b; return s; };
  if (hipStreamCreateWithFlags(&b->stream, hipStreamNonBlocking) != hipSuccess) {
    set_error("hipStreamCreate failed");
    return fail(GPQ_ERR_HIP);
  }
  Dev* d = new Dev();
  b->dev = d;
  BatchQuery* dq = nullptr;
  uint32_t* bits = nullptr;
  gpq_status s;
  const uint64_t slots = std::max<uint32_t>(resident, 1);
  // the far store alone holds every entry that the open list may (heap_capacity per thread); the
  // buckets come on top
  d->far_cap = (uint64_t)tu.heap_capacity * tu.threads_per_query;
  d->bucket_cap = bucket_cap_for(tu);
  if ((s = b->arena.alloc(&dq, count)) != GPQ_OK || (s = b->arena.alloc(&bits, words ? words : 1)) != GPQ_OK ||
      (s = b->arena.alloc(&d->g, slots * max_cells)) != GPQ_OK ||
      (s = b->arena.alloc(&d->far, slots * d->far_cap)) != GPQ_OK ||
      (s = b->arena.alloc(&d->bucket, slots * kBuckets * d->bucket_cap)) != GPQ_OK ||
      (s = b->arena.alloc(&d->list, slots)) != GPQ_OK ||
      (s = b->arena.alloc(&d->slot, slots)) != GPQ_OK || (s = b->arena.alloc(&d->cost, count)) != GPQ_OK ||
      (s = b->arena.alloc(&d->expanded, count)) != GPQ_OK || (s = b->arena.alloc(&d->flags, count)) != GPQ_OK ||
      (s = b->arena.alloc(&d->clk, 2 * (size_t)count)) != GPQ_OK ||
      (s = b->arena.alloc(&b->d_ids_all, count)) != GPQ_OK || (s = b->arena.alloc(&b->counter, 2)) != GPQ_OK)
    return fail(s);
  d->q = dq;
  d->bits = bits;
  d->g_stride = max_cells;
  d->counter = b->counter;
  std::vector<uint32_t> ids(count);
  for (uint32_t i = 0; i < count; ++i) ids[i] = i;
  if (hipMemcpyAsync(dq, hq.data(), sizeof(BatchQuery) * count, hipMemcpyHostToDevice, b->stream) != hipSuccess ||
      hipMemcpyAsync(b->d_ids_all, ids.data(), sizeof(uint32_t) * count, hipMemcpyHostToDevice, b->stream) !=
          hipSuccess) {
    set_error("batch: upload failed");
    return fail(GPQ_ERR_HIP);
  }
  hipLaunchKernelGGL(fill_u32_kernel, dim3(gen_blocks(slots * max_cells)), dim3(256), 0, b->stream, d->g,
                     slots * max_cells, 0xFFFFFFFFu);
  hipLaunchKernelGGL(init_slots_kernel, dim3(gen_blocks(slots)), dim3(256), 0, b->stream, d->slot, (uint32_t)slots);
  for (uint32_t i = 0; i < count; ++i) {
    const gpq_query_spec& q = sp[i];
    const uint64_t cells = (uint64_t)q.side * q.side;
    const uint64_t src = (uint64_t)q.sy * q.side + q.sx, tgt = (uint64_t)q.ty * q.side + q.tx;
    hipLaunchKernelGGL(grid_generate_kernel, dim3(gen_blocks((cells + 31) / 32)), dim3(256), 0, b->stream,
                       bits + off[i], cells, q.seed, q.stream_tag, q.query, q.threshold, src, tgt);
  }
  if (hipGetLastError() != hipSuccess || hipStreamSynchronize(b->stream) != hipSuccess) {
    set_error("batch: grid generation failed");
    return fail(GPQ_ERR_HIP);
  }
  *out = b;
  return GPQ_OK;
}

AstarBatch::~AstarBatch() {
  if (stream) (void)hipStreamSynchronize(stream);
  if (graph_exec) (void)hipGraphExecDestroy(graph_exec);
  if (graph) (void)hipGraphDestroy(graph);
  delete static_cast<Dev*>(dev);
  if (stream) (void)hipStreamDestroy(stream);
}

gpq_status AstarBatch::launch(const uint32_t* d_ids, uint32_t n, uint32_t slot_base, uint32_t slots,
                              uint32_t* d_counter, hipStream_t s) {
  GPQ_CHECK_ARG(slots >= 1 && slot_base + slots <= resident, "batch: slot range outside the resident slots");
  Dev d = *static_cast<Dev*>(dev);
  d.ids = d_ids;
  d.n = n;
  d.counter = d_counter;
  d.slot_base = slot_base;
  const uint32_t K = tuning.threads_per_query;
  hipLaunchKernelGGL(zero_u32_kernel, dim3(1), dim3(1), 0, s, d_counter);
  hipLaunchKernelGGL(astar_batch_kernel, dim3(std::max<uint32_t>(1, std::min(slots, n))), dim3(K), 0, s,
                     static_cast<BatchDev>(d));
  GPQ_HIP(hipGetLastError());
  return GPQ_OK;
}

// The one-query-per-launch path: query ids[0] (device) alone in `slot`, one launch per
// iteration, each followed by a host synchronization that reads the done flag.
gpq_status AstarBatch::plain_one(const uint32_t* d_id, uint32_t spec_index, uint32_t slot, uint32_t* d_done,
                                 uint32_t* h_done, hipStream_t s) {
  GPQ_CHECK_ARG(slot < resident, "batch: slot outside the resident slots");
  Dev d = *static_cast<Dev*>(dev);
  d.ids = d_id;
  d.n = 1;
  d.slot_base = slot;
  const uint32_t K = tuning.threads_per_query;
  const uint64_t step_cap = 64ull * specs[spec_index].side * specs[spec_index].side + 1024;
  for (uint64_t step = 0;; ++step) {
    if (step > step_cap) {
      set_error("batch plain: step bound exceeded");
      return GPQ_ERR_STATE;
    }
    hipLaunchKernelGGL(astar_batch_step_kernel, dim3(1), dim3(K), 0, s, static_cast<BatchDev>(d), step ? 1u : 0u,
                       d_done);
    GPQ_HIP(hipGetLastError());
    GPQ_HIP(hipMemcpyAsync(h_done, d_done, sizeof(uint32_t), hipMemcpyDeviceToHost, s));
    GPQ_HIP(hipStreamSynchronize(s));
    if (*h_done) return GPQ_OK;
  }
}

gpq_status AstarBatch::run(gpq_drive_mode mode, double* seconds) {
  const uint32_t n = (uint32_t)specs.size();
  GPQ_HIP(hipStreamSynchronize(stream));
  const auto t0 = std::chrono::steady_clock::now();
  if (mode == GPQ_DRIVE_GRAPH) {
    if (!graph_exec) {
      GPQ_HIP(hipStreamBeginCapture(stream, hipStreamCaptureModeThreadLocal));
      const gpq_status st = launch(d_ids_all, n, 0, resident, counter, stream);
      hipGraph_t gph = nullptr;
      const hipError_t e = hipStreamEndCapture(stream, &gph);
      if (st != GPQ_OK) return st;
      GPQ_HIP(e);
      graph = gph;
      GPQ_HIP(hipGraphInstantiate(&graph_exec, graph, nullptr, nullptr, 0));
    }
    GPQ_HIP(hipGraphLaunch(graph_exec, stream));
    GPQ_HIP(hipStreamSynchronize(stream));
  } else {
    uint32_t* h_done = nullptr;
    GPQ_HIP(hipHostMalloc(reinterpret_cast<void**>(&h_done), sizeof(uint32_t), hipHostMallocDefault));
    gpq_status st = GPQ_OK;
    for (uint32_t qi = 0; qi < n && st == GPQ_OK; ++qi) st = plain_one(d_ids_all + qi, qi, 0, counter + 1, h_done, stream);
    (void)hipHostFree(h_done);
    if (st != GPQ_OK) return st;
  }
  const auto t1 = std::chrono::steady_clock::now();
  if (seconds) *seconds = std::chrono::duration<double>(t1 - t0).count();
  return GPQ_OK;
}

// Times every workgroup size on the first `sample` queries (two persistent runs each, the second
// timed) and returns the fastest; heap_capacity and max_resident are kept from `base`.  Candidates
// whose open lists overflow are skipped.
gpq_status batch_autotune(const gpq_query_spec* sp, uint32_t count, uint32_t sample, const gpq_batch_tuning& base,
                          gpq_batch_tuning* out, double* best_seconds) {
  GPQ_CHECK_ARG(sp && count >= 1, "autotune: no queries");
  const uint32_t n = sample ? std::min(sample, count) : count;
  static const uint32_t kThreads[] = {64, 128, 256, 512};   // stage_capacity 8 excludes 1024
  double best = 1e300;
  gpq_batch_tuning pick{};
  for (uint32_t k : kThreads) {
    gpq_batch_tuning t = base;
    t.threads_per_query = k;
    t.stage_capacity = 8;
    AstarBatch* b = nullptr;
    if (AstarBatch::create(sp, n, t, &b) != GPQ_OK) continue;
    double sec = 0.0;
    gpq_status s = b->run(GPQ_DRIVE_GRAPH, &sec);
    if (s == GPQ_OK) s = b->run(GPQ_DRIVE_GRAPH, &sec);
    if (s == GPQ_OK) s = b->results(nullptr, nullptr);
    const gpq_batch_tuning used = b->tuning;
    delete b;
    if (s == GPQ_OK && sec < best) {
      best = sec;
      pick = used;
      pick.max_resident = base.max_resident;
    }
  }
  if (best == 1e300) {
    set_error("autotune: no candidate completed");
    return GPQ_ERR_CAPACITY;
  }
  *out = pick;
  if (best_seconds) *best_seconds = best;
  return GPQ_OK;
}

gpq_status AstarBatch::results(int64_t* costs, uint64_t* expanded) {
  const Dev* d = static_cast<const Dev*>(dev);
  const size_t n = specs.size();
  std::vector<uint32_t> flags(n);
  if (costs) GPQ_HIP(hipMemcpyAsync(costs, d->cost, sizeof(int64_t) * n, hipMemcpyDeviceToHost, stream));
  if (expanded) GPQ_HIP(hipMemcpyAsync(expanded, d->expanded, sizeof(uint64_t) * n, hipMemcpyDeviceToHost, stream));
  GPQ_HIP(hipMemcpyAsync(flags.data(), d->flags, sizeof(uint32_t) * n, hipMemcpyDeviceToHost, stream));
  GPQ_HIP(hipStreamSynchronize(stream));
  for (size_t i = 0; i < n; ++i)
    if (flags[i]) {
      set_error("batch: query " + std::to_string(i) + " overflowed its open lists (raise heap_capacity)");
      return GPQ_ERR_CAPACITY;
    }
  return GPQ_OK;
}

uint64_t AstarBatch::open_list_bytes() const {
  const Dev* d = static_cast<const Dev*>(dev);
  return 8ull * (d->far_cap + (uint64_t)kBuckets * d->bucket_cap);
}

gpq_status AstarBatch::timing(double* start_us, double* finish_us) {
  const Dev* d = static_cast<const Dev*>(dev);
  const size_t n = specs.size();
  std::vector<unsigned long long> clk(2 * n);
  GPQ_HIP(hipMemcpyAsync(clk.data(), d->clk, sizeof(unsigned long long) * 2 * n, hipMemcpyDeviceToHost, stream));
  GPQ_HIP(hipStreamSynchronize(stream));
  int dev_id = 0, khz = 0;
  GPQ_HIP(hipGetDevice(&dev_id));
  GPQ_HIP(hipDeviceGetAttribute(&khz, hipDeviceAttributeWallClockRate, dev_id));
  GPQ_CHECK_ARG(khz > 0, "batch: device wall clock rate unknown");
  unsigned long long t0 = ~0ull;
  for (size_t i = 0; i < n; ++i) t0 = std::min(t0, clk[2 * i]);
  const double us_per_tick = 1000.0 / khz;
  for (size_t i = 0; i < n; ++i) {
    if (start_us) start_us[i] = (double)(clk[2 * i] - t0) * us_per_tick;
    if (finish_us) finish_us[i] = (double)(clk[2 * i + 1] - t0) * us_per_tick;
  }
  return GPQ_OK;
}

// An optimal path of query q: q searched again alone in slot 0 (one persistent launch of one
// workgroup), then the closed-list backtrack of src/a_star.cu:90-94,417-438 over that slot's
// g values on the host: from the target (whose g is the query's cost), a free neighbour whose g
// (of the slot's current tag) plus the step cost equals the current cell's g.  Along such a
// chain every g is the optimal distance (the target's is; a neighbour meeting the equality
// cannot be above its optimum), so the neighbour that relaxed a cell last always qualifies and
// the chain reaches the source.
gpq_status AstarBatch::path(uint32_t q, uint32_t* cells, uint32_t cap, uint32_t* len) {
  GPQ_CHECK_ARG(q < specs.size(), "batch: query index out of range");
  GPQ_CHECK_ARG(len && (cells || cap == 0), "batch path: null output");
  const Dev* d = static_cast<const Dev*>(dev);
  const gpq_query_spec& sp = specs[q];
  const uint32_t side = sp.side;
  const uint64_t n = (uint64_t)side * side;
  GPQ_HIP(hipStreamSynchronize(stream));
  GPQ_TRY(launch(d_ids_all + q, 1, 0, 1, counter, stream));
  long long cost = -1;
  SlotState st{};
  std::vector<uint32_t> g(n);
  GPQ_HIP(hipMemcpyAsync(&cost, d->cost + q, sizeof(cost), hipMemcpyDeviceToHost, stream));
  GPQ_HIP(hipMemcpyAsync(&st, d->slot, sizeof(st), hipMemcpyDeviceToHost, stream));
  GPQ_HIP(hipMemcpyAsync(g.data(), d->g, sizeof(uint32_t) * n, hipMemcpyDeviceToHost, stream));
  GPQ_HIP(hipStreamSynchronize(stream));
  *len = 0;
  if (cost < 0) return GPQ_OK;
  std::vector<uint8_t> blocked(n);
  GPQ_TRY(grid_bytes(q, blocked.data()));
  const uint32_t mask = (1u << kTagShift) - 1u;
  auto gval = [&](uint64_t c, uint32_t* out) {
    if ((g[c] >> kTagShift) != st.tag) return false;
    *out = g[c] & mask;
    return true;
  };
  static const int dx[8] = {1, -1, 0, 0, 1, -1, 1, -1}, dy[8] = {0, 0, 1, -1, 1, 1, -1, -1};
  const uint64_t source = (uint64_t)sp.sy * side + sp.sx;
  uint64_t cur = (uint64_t)sp.ty * side + sp.tx;
  uint32_t gc = (uint32_t)cost;          // the search records the target's cost, not its g entry
  std::vector<uint32_t> rev{(uint32_t)cur};
  while (cur != source) {
    const int x = (int)(cur % side), y = (int)(cur / side);
    bool found = false;
    for (uint32_t k = 0; k < sp.connectivity && !found; ++k) {
      const int nx = x + dx[k], ny = y + dy[k];
      if (nx < 0 || ny < 0 || nx >= (int)side || ny >= (int)side) continue;
      const uint64_t nc = (uint64_t)ny * side + (uint64_t)nx;
      const uint32_t step = sp.connectivity == 4 ? 1u : (k < 4 ? 10u : 14u);
      uint32_t gn = 0;
      if (blocked[nc] || !gval(nc, &gn) || gn + step != gc) continue;
      cur = nc;
      gc = gn;
      found = true;
    }
    if (!found || rev.size() > n) {
      set_error("batch path: no predecessor with a matching g");
      return GPQ_ERR_STATE;
    }
    rev.push_back((uint32_t)cur);
  }
  *len = (uint32_t)rev.size();
  for (uint32_t i = 0; i < *len && i < cap; ++i) cells[i] = rev[*len - 1 - i];
  return GPQ_OK;
}

gpq_status AstarBatch::grid_bytes(uint32_t q, uint8_t* out) {
  GPQ_CHECK_ARG(q < specs.size(), "batch: query index out of range");
  const Dev* d = static_cast<const Dev*>(dev);
  const uint64_t cells = (uint64_t)specs[q].side * specs[q].side;
  uint8_t* tmp = nullptr;
  GPQ_HIP(hipMalloc(&tmp, cells));
  hipLaunchKernelGGL(grid_to_bytes_kernel, dim3(gen_blocks(cells)), dim3(256), 0, stream, d->bits + cell_off[q], tmp,
                     cells);
  hipError_t e = hipMemcpyAsync(out, tmp, cells, hipMemcpyDeviceToHost, stream);
  if (e == hipSuccess) e = hipStreamSynchronize(stream);
  (void)hipFree(tmp);
  GPQ_HIP(e);
  return GPQ_OK;
}

}  // namespace gpq
