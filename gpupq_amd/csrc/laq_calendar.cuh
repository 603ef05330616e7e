// laq_calendar.cuh -- calendar mode of the local array queue and the PHOLD step on it.
//
// The merge-and-commit PHOLD step (drain mode 2) ends window k at w_k = min(w_{k-1} + lookahead,
// end time) in float arithmetic, so every window end is known as soon as the first one is.  In
// calendar mode the queue uses that: it keeps one append log per upcoming window (a calendar
// queue, R. Brown, CACM 31(10), 1988, with one day per window), split by the block of LPs the
// events are for, and an event is appended to the log of its window and LP block.  Step c is one
// launch with two kinds of blocks that run side by side:
//   * commit blocks, one per block of kBlock LPs: the block's log of window c is grouped by LP and
//     put in key order in LDS, its events are committed, and their successors are appended to the
//     logs of their windows and LP blocks;
//   * a few list blocks: the events beyond the calendar (over[(c + 1) & 1]) whose window the
//     calendar now reaches move into the logs.
// No sorted run is kept, merged or shifted, and no separate pass groups the events by LP.  Calendars of
// LaqQueue::kGroupedMinLps LPs or more have logs with one writer instead (laq_calendar_groups.cuh); what the two
// share is here.
//
// Layout (B = cal_windows, a power of two; L = num_lps; K = kBlock LPs per block):
//   wlog   [B][blocks][sub_cap]  Event   window x, LP block b: count wlog_n[((x mod B) * blocks + b) * 16]
//   over   [2][over_cap]         Event   events beyond the calendar: appended to over[c & 1] by step
//                                        c, read (and moved on) by step c + 1
//   parked [parked_cap]          Event   events at or past the end time: never committed, only kept
//   cal_st                               `cur` (the window the next step commits) and the ends of
//                                        windows x in [cur, cur + B] at w[x mod 2B]
// A step appends only to windows c + 1 .. c + B - 1, so the log slot of window c (the one its
// commit blocks read and then empty) takes no appends during the step.
//
// Reference: the per-LP queue of src/local_array_queue.cu and its heap-backed far tier
// (:515-681); the step is handle_next_event (src/phold.cu:81-117) for every event of a window.
#pragma once

#include "phold_fused.cuh"

namespace gpq {
namespace cal {

// LPs per commit block, and so per log.  Smaller blocks mean more logs and shorter runs of the
// self-addressed successors, larger ones fewer blocks in flight: with a thread per LP and at 2^20 LPs, 64
// LPs 1.37e10, 128 LPs 1.59-1.66e10, 256 LPs 1.74-1.83e10, 512 LPs 1.60e10, 1024 LPs 1.42e10 events/s.
constexpr int kBlock = 256;
constexpr uint32_t kLpMost = 64;  // events of one LP in one window
constexpr uint32_t kPer = 4;      // events of one thread in a pass over the log
constexpr int kGroupBlocks = 2048;        // blocks of the standalone filing launch
constexpr uint32_t kStepListBlocks = 32;  // blocks of a step that move the beyond-the-calendar events

// Window offset of timestamp bits ts: the smallest o in [o_min, n) with ts < sw[o], where
// sw[o] is the end of window x + o; n when ts >= sw[n - 1] (beyond the windows looked at).  The
// ends lie one lookahead apart (inv = 1 / lookahead), the last ones at the end time, so the search
// starts at the window that the difference to the first end gives: it is off by at most a
// few, where a binary search made six dependent LDS reads at 64 windows.
__device__ __forceinline__ uint32_t find_window(const uint32_t* sw, uint32_t n, uint32_t ts, uint32_t o_min, float inv) {
  if (!(ts < sw[n - 1])) return n;
  const float d = (bits_to_f(ts) - bits_to_f(sw[0])) * inv;
  uint32_t o = d > 0.0f ? (uint32_t)fminf(d, (float)(n - 1u)) + 1u : 0u;
  o = o < o_min ? o_min : (o < n ? o : n - 1u);
  while (o > o_min && ts < sw[o - 1u]) --o;
  while (!(ts < sw[o])) ++o;                           // ends: ts < sw[n - 1]
  return o;
}

// Where an event goes, seen from window x with n windows looked at: a window offset o < n
// (the log of window x + o), kOver (beyond them) or kParked (at or past the end time).
struct Route {
  static constexpr uint32_t kOver = kCalMaxWindows;
  static constexpr uint32_t kParked = kCalMaxWindows + 1;
  static constexpr uint32_t kNone = kCalMaxWindows + 2;   // no record
};
constexpr uint32_t kRemote = 0x1000u;    // flag on a window route: the event is for another block's LPs

__device__ __forceinline__ uint32_t route_of(const uint32_t* sw, uint32_t n, uint32_t ts, uint32_t end_bits,
                                             uint32_t o_min, float inv) {
  if (!(ts < end_bits)) return Route::kParked;
  const uint32_t o = find_window(sw, n, ts, o_min, inv);
  return o < n ? o : Route::kOver;
}

// The log of window x for LP block b: its counter and its first record.  Counters sit 16 words
// (64 bytes) apart: packed, the counters of one window for 32 neighbouring LP blocks shared a
// 128-byte line, and every block's successors for those blocks' logs met on it (about 2,000
// atomics per line and step at 2^20 LPs).  Spread out, the step took 154 against 159 us (nine
// A/B pairs at 2^20 LPs) and the instances of one calendar ran 9% faster; 32 words apart gave no
// more.
constexpr uint32_t kLogCountShift = 4;
__device__ __forceinline__ uint32_t* log_count(const LaqView& q, uint32_t x, uint32_t b) {
  return &q.wlog_n[((size_t)(x & (q.cal_windows - 1u)) * q.cal_blocks + b) << kLogCountShift];
}
__device__ __forceinline__ Event* log_base(const LaqView& q, uint32_t x, uint32_t b) {
  return q.wlog + (size_t)(x & (q.cal_windows - 1u)) * q.wlog_cap + (size_t)b * q.cal_sub_cap;
}

// e appended to the log of window x for its LP's block, by its own atomic.
__device__ __forceinline__ void log_append(const LaqView& q, uint32_t x, const Event& e) {
  const uint32_t b = e.dst >> q.cal_block_log2;
  const uint32_t pos = atomicAdd(log_count(q, x, b), 1u);
  if (pos < q.cal_sub_cap) store_event(log_base(q, x, b) + pos, e);
  else atomicOr(&q.ws->error, kErrQueueOverflow);
}

// The lists: beyond the calendar (over[op]) and parked.
__device__ __forceinline__ uint32_t* list_count(const LaqView& q, uint32_t op, uint32_t r) {
  return r == Route::kParked ? q.parked_n : &q.over_n[op];
}
__device__ __forceinline__ void list_store(const LaqView& q, uint32_t op, uint32_t r, uint32_t pos, const uint4& e) {
  const bool parked = r == Route::kParked;
  if (pos < (parked ? q.parked_cap : q.over_cap))
    *reinterpret_cast<uint4*>(parked ? q.parked + pos : q.over + (size_t)op * q.over_cap + pos) = e;
  else
    atomicOr(&q.ws->error, kErrQueueOverflow);
}

// One event filed by its own atomic: route r seen from window x (a window offset, kOver: the
// list over[op], or kParked).
__device__ __forceinline__ void append_one(const LaqView& q, uint32_t x, uint32_t op, uint32_t r, const Event& e) {
  if (r < kCalMaxWindows) {
    log_append(q, x + r, e);
    return;
  }
  list_store(q, op, r, atomicAdd(list_count(q, op, r), 1u), make_uint4(e.ts, e.dst, e.src, e.seq));
}

// Block-wide filing of at most one event per thread: a window route goes to its log by the
// event's own atomic; the list routes take a rank in the block's LDS count of their list, one
// thread per list reserves the block's run with a single atomic, and the events are written
// into the runs.  op is block-uniform; every thread of the block calls.
struct ListAppend {
  uint32_t cnt[2];
  uint32_t base[2];
};

__device__ __forceinline__ void block_file(const LaqView& q, uint32_t x, uint32_t op, uint32_t r, const Event& e,
                                           ListAppend& la) {
  if (threadIdx.x < 2) la.cnt[threadIdx.x] = 0u;
  __syncthreads();
  const bool list = r == Route::kOver || r == Route::kParked;
  const uint32_t li = r == Route::kParked ? 1u : 0u;
  uint32_t rank = 0;
  if (r < kCalMaxWindows) log_append(q, x + r, e);
  else if (list) rank = atomicAdd(&la.cnt[li], 1u);
  __syncthreads();
  if (threadIdx.x < 2) {
    const uint32_t n = la.cnt[threadIdx.x];
    la.base[threadIdx.x] = n ? atomicAdd(list_count(q, op, threadIdx.x ? Route::kParked : Route::kOver), n) : 0u;
  }
  __syncthreads();
  if (list) list_store(q, op, r, la.base[li] + rank, make_uint4(e.ts, e.dst, e.src, e.seq));
  __syncthreads();
}

// Block-wide: the ends of windows x .. x + B - 1 into sw (every thread of the block calls).
__device__ __forceinline__ void load_windows(const LaqView& q, uint32_t x, uint32_t* sw) {
  const uint32_t B = q.cal_windows, M = 2u * B - 1u;
  for (uint32_t i = threadIdx.x; i < B; i += blockDim.x) sw[i] = q.cal_st->w[(x + i) & M];
}

// The successor of a committed event (src/phold.cu:93-116): draw {n, local, 0, 0}, destination
// self with probability p_self else uniform over the instance, ts' = (ts + lookahead) + Exp(1).
__device__ __forceinline__ Event successor(const FusedModel& m, uint32_t lp, uint32_t n, uint32_t ts) {
  const uint32_t local = lp - m.base;
  const uint4 r = philox4x32_10(make_uint4(n, local, 0u, 0u), make_uint2(m.seed, 0u));
  const uint32_t dst = r.y < m.p_self ? lp : m.base + (uint32_t)(((uint64_t)r.z * m.lps) >> 32);
  const float t_new = (bits_to_f(ts) + m.lookahead) + exp_from_u32(r.x);
  return Event{f_to_bits(t_new), dst, local, m.init_per_lp + n};
}

// ---- the parts of a commit that every size of calendar shares ---------------------------------
// U threads, one per LP, take a window's events from one log, U * PER at a time.
template <int U, uint32_t PER>
struct CommitLds {
  static constexpr uint32_t kPass = U * PER;
  uint32_t cnt[U], off[U + 1], fill[U], n0[U];         // per LP: events, their first place, and its count before
  uint32_t ts[kPass], src[kPass], seq[kPass];          // the events of the pass in LP order, then in key order
  uint16_t lp[kPass];
  uint32_t wave[U / kWave];
};

// The log's n events counted per LP, the counts' prefix sum, and with n <= kPass the events placed in
// LP order; e[0 .. loaded) hold the thread's first ones already.  Returns the events of the
// thread's LP.  cnt is clear before, and the caller synchronizes after.
template <int U, uint32_t PER>
__device__ __forceinline__ uint32_t group_log(CommitLds<U, PER>& s, const LaqView& q, const Event* lg, uint32_t n,
                                              uint32_t lp0, Event* e, uint32_t loaded) {
  const uint32_t t = threadIdx.x;
  uint32_t l[PER], k[PER];
#pragma unroll
  for (uint32_t j = 0; j < PER; ++j) {
    const uint32_t i = t + j * U;
    l[j] = U;
    k[j] = 0;
    if (i < n) {
      if (j >= loaded) e[j] = load_event(&lg[i]);
      l[j] = e[j].dst - lp0;                           // < U: these LPs only
      if (l[j] < (uint32_t)U) k[j] = atomicAdd(&s.cnt[l[j]], 1u);
      else atomicOr(&q.ws->error, kErrBadState);
    }
  }
  for (uint32_t i = t + CommitLds<U, PER>::kPass; i < n; i += U) {
    const uint32_t x = lg[i].dst - lp0;
    if (x < (uint32_t)U) atomicAdd(&s.cnt[x], 1u);
    else atomicOr(&q.ws->error, kErrBadState);
  }
  __syncthreads();
  const uint32_t mine = s.cnt[t];
  if (mine > kLpMost) atomicOr(&q.ws->error, kErrStageOverflow);
  uint32_t inc = mine;
#pragma unroll
  for (int off = 1; off < kWave; off <<= 1) {
    const uint32_t y = (uint32_t)__shfl_up((int)inc, off, kWave);
    if (lane_id() >= off) inc += y;
  }
  if (lane_id() == kWave - 1) s.wave[t / kWave] = inc;
  __syncthreads();
  for (uint32_t w = 0; w < t / kWave; ++w) inc += s.wave[w];
  s.off[t + 1u] = inc;
  if (t == 0) s.off[0] = 0u;
  __syncthreads();
  if (n <= CommitLds<U, PER>::kPass) {                 // from registers
#pragma unroll
    for (uint32_t j = 0; j < PER; ++j) {
      if (l[j] >= (uint32_t)U) continue;
      const uint32_t p = s.off[l[j]] + k[j];
      s.ts[p] = e[j].ts;
      s.src[p] = e[j].src;
      s.seq[p] = e[j].seq;
      s.lp[p] = (uint16_t)l[j];
    }
  }
  return mine;
}

// The pass over the LPs from `first` on: *last past its last LP.  A log of more than kPass events is
// taken in several, each over the LPs whose events fit; false when LP `first` alone does not (it was
// refused: kPass > kLpMost), and the caller goes on with the next one.  Uniform; the caller
// synchronizes after.
template <int U, uint32_t PER>
__device__ __forceinline__ bool begin_pass(CommitLds<U, PER>& s, uint32_t n, uint32_t first, uint32_t* last) {
  const uint32_t t = threadIdx.x;
  *last = U;
  if (n <= CommitLds<U, PER>::kPass) return true;
  *last = first + (uint32_t)__syncthreads_count(t >= first && s.off[t + 1u] - s.off[first] <= CommitLds<U, PER>::kPass);
  s.fill[t] = 0u;
  return *last != first;
}

// With n > kPass: the pass's events from the log into LP order.
template <int U, uint32_t PER>
__device__ __forceinline__ void fill_pass(CommitLds<U, PER>& s, const Event* lg, uint32_t n, uint32_t lp0, uint32_t first,
                                          uint32_t last) {
  if (n <= CommitLds<U, PER>::kPass) return;
  __syncthreads();
  for (uint32_t i = threadIdx.x; i < n; i += U) {
    const Event x = load_event(&lg[i]);
    const uint32_t xl = x.dst - lp0;
    if (xl < first || xl >= last) continue;
    const uint32_t p = s.off[xl] - s.off[first] + atomicAdd(&s.fill[xl], 1u);
    s.ts[p] = x.ts;
    s.src[p] = x.src;
    s.seq[p] = x.seq;
    s.lp[p] = (uint16_t)xl;
  }
}

// A thread per event: its rank among its LP's events, and the events moved into key order.  The
// caller synchronizes before and after.
template <int U, uint32_t PER>
__device__ __forceinline__ void order_pass(CommitLds<U, PER>& s, uint32_t base, uint32_t take) {
  const uint32_t t = threadIdx.x;
  uint32_t ets[PER], esrc[PER], eseq[PER], to[PER];
#pragma unroll
  for (uint32_t j = 0; j < PER; ++j) {
    const uint32_t p = t + j * U;
    if (p >= take) continue;
    const uint32_t el = s.lp[p], o = s.off[el] - base, kk = s.cnt[el];
    ets[j] = s.ts[p];
    esrc[j] = s.src[p];
    eseq[j] = s.seq[p];
    uint32_t rank = 0;
    for (uint32_t i = 0; i < kk; ++i) {
      const uint32_t ot = s.ts[o + i];
      bool before = ot < ets[j];
      if (ot == ets[j] && o + i != p) {                // equal times: by source, then number, then arrival
        const uint32_t os = s.src[o + i], oq = s.seq[o + i];
        before = os != esrc[j] ? os < esrc[j] : (oq != eseq[j] ? oq < eseq[j] : o + i < p);
      }
      rank += before ? 1u : 0u;
    }
    to[j] = o + rank;
  }
  __syncthreads();                                     // every rank is taken
#pragma unroll
  for (uint32_t j = 0; j < PER; ++j) {
    if (t + j * U >= take) continue;
    s.ts[to[j]] = ets[j];
    s.src[to[j]] = esrc[j];
    s.seq[to[j]] = eseq[j];
  }
}

// A thread per LP: the trace hash over its k events in key order, at place o.
template <int U, uint32_t PER>
__device__ __forceinline__ uint64_t hash_events(const CommitLds<U, PER>& s, const LaqView& q, const FusedModel& m, uint32_t lp,
                                                uint32_t o, uint32_t k, uint64_t h) {
  uint32_t prev = m.last_ts ? m.last_ts[lp] : 0u;
  for (uint32_t i = 0; i < k; ++i) {
    const uint32_t xt = s.ts[o + i];
    h = trace_step(h, xt, s.src[o + i], s.seq[o + i]);
    if (m.last_ts) {
      if (xt < prev) atomicOr(&q.ws->error, kErrBadState);
      prev = xt;
    }
  }
  if (m.last_ts && k) m.last_ts[lp] = prev;
  return h;
}

// Commit block `blk` of step c (window c).  The block's log of the window is grouped by LP in LDS
// (a count per LP, its prefix sum, the records in LP order), and then worked on event by event, a
// thread per event: its rank among its LP's events (compared one by one: three on average),
// which gives its draw number, its successor and where that goes.  Only the trace hash, a chain
// over an LP's events in key order, is left to a thread per LP; it runs while the successors' slot
// atomics are in flight.  A successor for one of this block's LPs (half of them in PHOLD: the
// self-addressed ones) and one for a list take a rank in the block's LDS count of their window or
// list, one thread per window and list reserves the block's run, and they are written into
// the runs; a successor for another block goes to that block's log by its own atomic.  The log is
// emptied at the end.  A log of more than kPer events per thread is taken in passes over ranges of LPs.
//
// What bounds it: a block's chain of loads, LDS phases and the atomics' round trips, and the launch: 10.1
// us a step at 1024 LPs x 16 events (four blocks), 21.4 at 65,536 x 32 (one block per CU), 30.2 at 131,072
// x 32, where 7 us of it are the 190,000 atomics on other blocks' log counters (performed at the memory
// side, at 26.6 G/s whatever lines they meet on).  At 2^20 LPs they were 64 us of 126, which is why large
// calendars are kept otherwise.
// With a thread per LP and its events in eight register slots (sorted by a network), a wave ran
// all eight slots' draws for LPs that hold three events on average, and an LP with more was
// committed by a wave of its own afterwards: 152 us per step (and 15.7 us at 1024 LPs, now 10.1).
// Registers do not bind: 4, 5 and 6 waves per SIMD (105, 81 and 79 registers) took the same time.
__device__ __forceinline__ void commit_block(const LaqView& q, const FusedModel& m, float end_time, float inv, uint32_t c,
                                             uint32_t blk) {
  __shared__ uint32_t sw[kCalMaxWindows];
  __shared__ CommitLds<kBlock, kPer> s;
  __shared__ uint32_t s_lcnt[2], s_lbase[2];
  __shared__ uint32_t s_wcnt[kCalMaxWindows], s_wbase[kCalMaxWindows];
  const uint32_t t = threadIdx.x;
  const uint32_t lp0 = blk << q.cal_block_log2;
  const uint32_t lp = lp0 + t;
  const bool in_range = lp < q.num_lps && lp - m.base < m.lps;
  const Event* lg = log_base(q, c, blk);
  // issued together with the window ends' load: the log's length, the first two of the thread's
  // records (the slots exist, or the second is not read; used only below the length) and the
  // thread's LP state, so that their latencies overlap
  const uint32_t n0 = *log_count(q, c, blk);
  Event e[kPer];
  e[0] = load_event(&lg[t]);
  e[1] = Event{};
  if (q.cal_sub_cap >= 2u * kBlock) e[1] = load_event(&lg[t + kBlock]);
  const uint32_t cnt_pre = in_range ? m.count[lp] : 0u;
  const uint64_t h_pre = in_range ? m.hash[lp] : 0ull;
  load_windows(q, c, sw);
  const uint32_t B = q.cal_windows;
  const uint32_t end_bits = f_to_bits(end_time);
  s.cnt[t] = 0u;
  s.n0[t] = cnt_pre;
  __syncthreads();
  const uint32_t n = n0 < q.cal_sub_cap ? n0 : q.cal_sub_cap;
  const uint32_t mine = group_log(s, q, lg, n, lp0, e, 2u);
  for (uint32_t first = 0, last; first < (uint32_t)kBlock; first = last) {   // one pass unless the log is long
    if (!begin_pass(s, n, first, &last)) {
      ++last;
      continue;
    }
    const uint32_t base = s.off[first], take = s.off[last] - base;
    for (uint32_t i = t; i < B; i += kBlock) s_wcnt[i] = 0u;
    if (t < 2) s_lcnt[t] = 0u;
    fill_pass(s, lg, n, lp0, first, last);
    __syncthreads();
    order_pass(s, base, take);
    __syncthreads();
    if (in_range && mine && t >= first && t < last) {
      m.hash[lp] = hash_events(s, q, m, lp, s.off[t] - base, mine, h_pre);
      m.count[lp] = cnt_pre + mine;
    }
    __syncthreads();                                   // the events' words now hold their successors
    // a thread per event, one after the other (side by side they take 108 registers, four waves per
    // SIMD): the successor's time and destination, and its route with its rank in this
    // block's run of that window or list
#pragma unroll 1
    for (uint32_t p = t; p < take; p += kBlock) {
      const uint32_t el = s.lp[p], elp = lp0 + el;
      uint32_t way = Route::kNone;
      if (elp < q.num_lps && elp - m.base < m.lps) {
        const Event sc = successor(m, elp, s.n0[el] + (p - (s.off[el] - base)), s.ts[p]);
        const uint32_t r = route_of(sw, B, sc.ts, end_bits, 1u, inv);
        s.ts[p] = sc.ts;
        s.src[p] = sc.dst;
        if (r >= kCalMaxWindows) way = r | (atomicAdd(&s_lcnt[r == Route::kParked ? 1u : 0u], 1u) << 16);
        else if ((sc.dst >> q.cal_block_log2) == blk) way = r | (atomicAdd(&s_wcnt[r], 1u) << 16);
        else way = r | kRemote;
      }
      s.seq[p] = way;
    }
    // successors for other blocks' logs: every slot atomic of the thread in flight at once
    uint32_t pos[kPer];
#pragma unroll
    for (uint32_t j = 0; j < kPer; ++j) {
      const uint32_t p = t + j * kBlock;
      const uint32_t way = p < take ? s.seq[p] : (uint32_t)Route::kNone;
      pos[j] = way & kRemote ? atomicAdd(log_count(q, c + (way & 0xFFFu), s.src[p] >> q.cal_block_log2), 1u) : 0u;
    }
    __syncthreads();
    // one run per window (this block's own log) and per list for the block
    for (uint32_t i = t; i < B; i += kBlock) {
      const uint32_t x = s_wcnt[i];
      s_wbase[i] = x ? atomicAdd(log_count(q, c + i, blk), x) : 0u;
    }
    if (t < 2) {
      const uint32_t x = s_lcnt[t];
      s_lbase[t] = x ? atomicAdd(list_count(q, c & 1u, t ? Route::kParked : Route::kOver), x) : 0u;
    }
    auto record = [&](uint32_t p) {
      const uint32_t el = s.lp[p];
      return make_uint4(s.ts[p], s.src[p], lp0 + el - m.base, m.init_per_lp + s.n0[el] + (p - (s.off[el] - base)));
    };
#pragma unroll
    for (uint32_t j = 0; j < kPer; ++j) {
      const uint32_t p = t + j * kBlock;
      const uint32_t way = p < take ? s.seq[p] : (uint32_t)Route::kNone;
      if (!(way & kRemote)) continue;
      if (pos[j] < q.cal_sub_cap)
        *reinterpret_cast<uint4*>(log_base(q, c + (way & 0xFFFu), s.src[p] >> q.cal_block_log2) + pos[j]) = record(p);
      else
        atomicOr(&q.ws->error, kErrQueueOverflow);
    }
    __syncthreads();
    for (uint32_t p = t; p < take; p += kBlock) {
      const uint32_t way = s.seq[p], r = way & 0xFFFu, rank = way >> 16;
      if ((way & kRemote) || r == Route::kNone) continue;
      if (r < kCalMaxWindows) {
        const uint32_t i = s_wbase[r] + rank;
        if (i < q.cal_sub_cap) *reinterpret_cast<uint4*>(log_base(q, c + r, blk) + i) = record(p);
        else atomicOr(&q.ws->error, kErrQueueOverflow);
      } else {
        list_store(q, c & 1u, r, s_lbase[r == Route::kParked ? 1u : 0u] + rank, record(p));
      }
    }
    if (last < (uint32_t)kBlock) __syncthreads();      // the next pass clears the counts
  }
  if (t == 0) *log_count(q, c, blk) = 0u;              // the block's log of window c is consumed
}

// The end of the step that committed window c (its logs emptied by the commit blocks): the list
// the step's list blocks read is emptied; the window advances by the lookahead (capped at the end
// time) and the end of window c + 1 + B joins the ring; the window that reached the end time ends
// the run.  Only the fields it owns are written: other blocks of the step may be setting the
// error flag.
__device__ __forceinline__ void publish(const LaqView& q, float lookahead, float end_time) {
  WindowState* ws = q.ws;
  CalState* st = q.cal_st;
  const uint32_t B = q.cal_windows, M = 2u * B - 1u;
  const uint32_t c = st->cur;
  const uint32_t wend = ws->wend;
  q.over_n[(c + 1u) & 1u] = 0;
  ws->windows += 1;
  ws->gmin = wend;                                 // a lower bound of the pending minimum
  if (!(bits_to_f(wend) < end_time)) {
    ws->done = 1;
  } else {
    const uint32_t nc = c + 1u;
    st->cur = nc;
    float nw = bits_to_f(st->w[(nc + B - 1u) & M]) + lookahead;
    if (end_time < nw) nw = end_time;
    st->w[(nc + B) & M] = f_to_bits(nw);
    ws->wend = st->w[nc & M];
  }
}

// Called by thread 0 of every block of a step once the block is done: the last block publishes.
// No fence is needed: the words publish() reads are written by no block of the step, the list it
// empties was read (and the values used) by the list blocks before they counted themselves, the
// error flag it leaves alone, and its writes reach the next step across the kernel boundary.
__device__ __forceinline__ void block_done(const LaqView& q, float lookahead, float end_time) {
  if (atomicAdd(&q.cal_st->fin, 1u) == gridDim.x - 1u) {
    publish(q, lookahead, end_time);
    q.cal_st->fin = 0u;
  }
}

// List block `blk` of `nblk` in the step that commits window x - 1: the events of over[x & 1]
// (beyond the windows the step before could reach) are seen from window x over its first B - 1
// windows -- x .. x + B - 2, all of them beyond the window being committed and short of the
// one whose log slot it is reading -- and go to the log of their window, on to over[(x + 1) & 1],
// or with the parked ones.
__device__ __forceinline__ void list_block(const LaqView& q, float end_time, float inv, uint32_t x, uint32_t blk,
                                           uint32_t nblk) {
  __shared__ uint32_t sw[kCalMaxWindows];
  __shared__ ListAppend la;
  load_windows(q, x, sw);
  __syncthreads();
  const uint32_t B = q.cal_windows;
  const uint32_t rp = x & 1u, wp = rp ^ 1u;
  const uint32_t no0 = q.over_n[rp];
  const uint32_t no = no0 < q.over_cap ? no0 : q.over_cap;
  const Event* ov = q.over + (size_t)rp * q.over_cap;
  const uint32_t end_bits = f_to_bits(end_time);
  const uint32_t stride = nblk * blockDim.x;
  for (uint32_t base = blk * blockDim.x; base < no; base += stride) {   // block-uniform trip count
    const uint32_t i = base + threadIdx.x;
    const bool has = i < no;
    const Event e = has ? load_event(&ov[i]) : Event{};
    const uint32_t r = has ? route_of(sw, B - 1u, e.ts, end_bits, 0u, inv) : Route::kNone;
    block_file(q, x, wp, r, e, la);
  }
}

}  // namespace cal
}  // namespace gpq
