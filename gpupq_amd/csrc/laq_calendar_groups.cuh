// laq_calendar_groups.cuh -- the calendar step for large queues: logs with one writer.
//
// In laq_calendar.cuh a successor for another block's LPs takes its slot in that block's log with
// an atomic, and atomics are performed at the memory side at 26.6 G/s for the whole card: 1.7 M
// per step at 2^20 LPs x 32 events, half of the step's time.  Here every log has one writer at a
// time and its count is a plain word.  A step is two launches:
//   * cal_file_kernel, a workgroup per group of units: the events that the last step sent to the
//     group, and the group's events beyond the calendar whose window has come into reach, go to
//     the logs of their windows and units, with the logs' counts in LDS;
//   * the commit step, a workgroup per unit of kUnit LPs (commit_unit): window c's events are
//     committed as in laq_calendar.cuh; a successor for the unit's own LPs goes to the unit's log of
//     its window, any other to the unit's outbox, whose events lie in the order of the groups they
//     are for, with the group's offsets beside them.
// An event for another unit is written and read once more than with an atomic, both in runs.  At 2^20
// LPs x 32 events the two launches take 24 and 62 us against 126 for the one with atomics.
//
// Layout (B = calendar windows, U = units, G = groups <= kMaxGroups of 2^group_shift LPs):
//   wlog  [U][B][log_cap]  Event      window x, unit u at [u][x mod B]: wlog_n[u * B + x mod B] events
//   out   [U][passes][kUnitPass]      outbox of each pass of a unit's last step
//   parts [U][passes][kMaxGroups]     the part of group g in it: first event | number << 16
//   npass [U]                         passes of the unit's last step
//   over  [G][own_cap], [G * own_cap] the groups' events beyond the calendar.  Half of the room is the
//                                     groups' own, far_per_lp records per LP; the other half is dealt
//                                     out at the start (cal_start_groups_kernel): to each group what its
//                                     initial events need beyond its own, and the rest evenly, so that
//                                     initial events may lie anywhere, as in the one list of a small
//                                     calendar.  Until then the shared half holds them unsorted.
// The outboxes of the last step are part of the queue's contents.
#pragma once

#include "calendar_groups.h"
#include "laq_calendar.cuh"

namespace gpq {
namespace cal {

constexpr uint32_t kUnitPer = 4;         // events of one thread in a pass over the log
constexpr uint32_t kUnitPass = kUnitPer * kUnit;
constexpr int kFileThreads = 1024;
constexpr uint32_t kFileUnits = 2 * kFileThreads;   // units whose outboxes are looked at together
constexpr uint32_t kFileCap = 8192;      // inbox events filed at once
constexpr uint32_t kFileBurst = 4;       // of a thread
constexpr uint32_t kToGroup = 0x1000u;   // flag on a way: to a group's part of the outbox

__device__ __forceinline__ Event* unit_log(const LaqView& q, const Groups& g, uint32_t unit, uint32_t x) {
  return g.wlog + ((size_t)unit * q.cal_windows + (x & (q.cal_windows - 1u))) * g.log_cap;
}
// A group's events beyond the calendar: `cap` places at most, of which the first are its own.
struct OverList {
  Event* own;
  Event* more;
  uint32_t own_cap, cap;
  __device__ __forceinline__ Event* at(uint32_t p) const { return p < own_cap ? own + p : more + (p - own_cap); }
};
__device__ __forceinline__ Event* shared_over(const Groups& g) { return g.over + (size_t)g.groups * g.own_cap; }
__device__ __forceinline__ OverList over_list(const Groups& g, uint32_t grp) {
  const uint32_t* w = g.over_n + grp * kOverWords;
  return OverList{g.over + (size_t)grp * g.own_cap, shared_over(g) + w[kOverFrom], g.own_cap, g.own_cap + w[kOverMore]};
}

__device__ __forceinline__ uint32_t* unit_count(const LaqView& q, const Groups& g, uint32_t unit, uint32_t x) {
  return g.wlog_n + (size_t)unit * q.cal_windows + (x & (q.cal_windows - 1u));
}

// Commit of window c for the kUnit LPs of `unit`; see commit_block in laq_calendar.cuh, whose
// passes, ranks and hash are the same.
__device__ __forceinline__ void commit_unit(const LaqView& q, const Groups& g, const FusedModel& m, float end_time,
                                            float inv, uint32_t c, uint32_t unit) {
  __shared__ uint32_t sw[kCalMaxWindows];
  __shared__ CommitLds<kUnit, kUnitPer> s;
  __shared__ uint32_t s_wcnt[kCalMaxWindows], s_wbase[kCalMaxWindows];
  __shared__ uint32_t s_gcnt[kMaxGroups], s_goff[kMaxGroups];
  __shared__ uint32_t s_pcnt, s_pbase;
  const uint32_t t = threadIdx.x;
  const uint32_t lp0 = unit << kUnitLog2;
  const uint32_t lp = lp0 + t;
  const bool in_range = lp < q.num_lps && lp - m.base < m.lps;
  const Event* lg = unit_log(q, g, unit, c);
  const uint32_t n0 = *unit_count(q, g, unit, c);
  Event e[kUnitPer];
  e[0] = load_event(&lg[t]);                           // the slots exist (log_cap >= kUnit); used below n only
  e[1] = Event{};
  if (g.log_cap >= 2u * kUnit) e[1] = load_event(&lg[t + kUnit]);
  const uint32_t cnt_pre = in_range ? m.count[lp] : 0u;
  const uint64_t h_pre = in_range ? m.hash[lp] : 0ull;
  load_windows(q, c, sw);
  const uint32_t B = q.cal_windows;
  const uint32_t end_bits = f_to_bits(end_time);
  s.cnt[t] = 0u;
  s.n0[t] = cnt_pre;
  __syncthreads();
  const uint32_t n = n0 < g.log_cap ? n0 : g.log_cap;
  const uint32_t mine = group_log(s, q, lg, n, lp0, e, 2u);
  uint32_t pass = 0;
  for (uint32_t first = 0, last; first < (uint32_t)kUnit && n; first = last) {   // one pass unless the log is long
    if (!begin_pass(s, n, first, &last)) {
      ++last;
      continue;
    }
    if (pass >= g.passes) {                            // only after an LP was refused: others fill their passes
      if (t == 0) atomicOr(&q.ws->error, kErrStageOverflow);
      break;
    }
    const uint32_t base = s.off[first], take = s.off[last] - base;
    if (t < B) s_wcnt[t] = 0u;
    if (t < kMaxGroups) s_gcnt[t] = 0u;
    if (t == 0) s_pcnt = 0u;
    static_assert(kCalMaxWindows <= (uint32_t)kUnit && kMaxGroups <= (uint32_t)kUnit, "one thread clears each count");
    fill_pass(s, lg, n, lp0, first, last);
    __syncthreads();
    order_pass(s, base, take);
    __syncthreads();
    if (in_range && mine && t >= first && t < last) {
      m.hash[lp] = hash_events(s, q, m, lp, s.off[t] - base, mine, h_pre);
      m.count[lp] = cnt_pre + mine;
    }
    __syncthreads();                                   // the events' words now hold their successors
    // a thread per event: the successor's time and destination, and its way with its rank on it
#pragma unroll 1
    for (uint32_t p = t; p < take; p += kUnit) {
      const uint32_t el = s.lp[p], elp = lp0 + el;
      uint32_t way = Route::kNone;
      if (elp < q.num_lps && elp - m.base < m.lps) {
        const Event sc = successor(m, elp, s.n0[el] + (p - (s.off[el] - base)), s.ts[p]);
        s.ts[p] = sc.ts;
        s.src[p] = sc.dst;
        if (!(sc.ts < end_bits)) {
          way = Route::kParked | (atomicAdd(&s_pcnt, 1u) << 16);
        } else {
          uint32_t r = B;
          if ((sc.dst >> kUnitLog2) == unit) r = find_window(sw, B, sc.ts, 1u, inv);
          if (r < B) {
            way = r | (atomicAdd(&s_wcnt[r], 1u) << 16);
          } else {                                     // another unit's, or beyond the calendar
            const uint32_t to = sc.dst >> g.group_shift;
            way = kToGroup | to | (atomicAdd(&s_gcnt[to], 1u) << 16);
          }
        }
      }
      s.seq[p] = way;
    }
    __syncthreads();
    if (t < B) {                                       // the unit's runs in its own logs
      const uint32_t x = s_wcnt[t];
      if (x) {
        uint32_t* cn = unit_count(q, g, unit, c + t);
        const uint32_t at = *cn;
        s_wbase[t] = at;
        *cn = at + x;
      }
    }
    if (t >= (uint32_t)kUnit - kWave) {                // the last wave: offsets of the groups' parts
      const uint32_t ln = (uint32_t)lane_id();
      static_assert(kMaxGroups == 4 * kWave, "four groups per lane");
      uint32_t v[4], sum = 0;
#pragma unroll
      for (uint32_t i = 0; i < 4; ++i) {
        v[i] = s_gcnt[4u * ln + i];
        sum += v[i];
      }
      uint32_t x = sum;
#pragma unroll
      for (int off = 1; off < kWave; off <<= 1) {
        const uint32_t y = (uint32_t)__shfl_up((int)x, off, kWave);
        if ((int)ln >= off) x += y;
      }
      uint32_t run = x - sum;
#pragma unroll
      for (uint32_t i = 0; i < 4; ++i) {
        s_goff[4u * ln + i] = run;
        run += v[i];
      }
      if (ln == 0) s_pbase = s_pcnt ? atomicAdd(q.parked_n, s_pcnt) : 0u;
    }
    __syncthreads();
    const size_t slot = (size_t)unit * g.passes + pass;
    if (t < kMaxGroups) g.parts[slot * kMaxGroups + t] = s_goff[t] | (s_gcnt[t] << 16);
    Event* out = g.out + slot * kUnitPass;
    for (uint32_t p = t; p < take; p += kUnit) {
      const uint32_t way = s.seq[p], r = way & 0xFFFu, rank = way >> 16;
      if (!(way & kToGroup) && r == Route::kNone) continue;
      const uint32_t el = s.lp[p];
      const uint4 ne = make_uint4(s.ts[p], s.src[p], lp0 + el - m.base, m.init_per_lp + s.n0[el] + (p - (s.off[el] - base)));
      if (way & kToGroup) {
        *reinterpret_cast<uint4*>(out + s_goff[r] + rank) = ne;
      } else if (r < kCalMaxWindows) {
        const uint32_t i = s_wbase[r] + rank;
        if (i < g.log_cap) *reinterpret_cast<uint4*>(unit_log(q, g, unit, c + r) + i) = ne;
        else atomicOr(&q.ws->error, kErrQueueOverflow);
      } else {
        list_store(q, 0u, Route::kParked, s_pbase + rank, ne);
      }
    }
    ++pass;
    if (last < (uint32_t)kUnit) __syncthreads();       // the next pass clears the counts
  }
  if (n == 0 && t < kMaxGroups) g.parts[(size_t)unit * g.passes * kMaxGroups + t] = 0u;   // an empty first part
  if (t == 0) {
    g.npass[unit] = pass;
    *unit_count(q, g, unit, c) = 0u;                   // the unit's log of window c is consumed
  }
}

// Files an event of the group in the log of its window, seen from window x over all B windows, or
// behind the group's events beyond the calendar.  s_n: the counts of the group's logs.
__device__ __forceinline__ void file_event(const LaqView& q, const Groups& g, const uint32_t* sw, uint32_t x, float inv,
                                           uint32_t unit0, uint32_t nu, uint32_t* s_n, uint32_t* s_over, const OverList& over,
                                           const Event& e) {
  const uint32_t B = q.cal_windows;
  const uint32_t u = (e.dst >> kUnitLog2) - unit0;
  if (u >= nu) {                                       // the group's LPs only
    atomicOr(&q.ws->error, kErrBadState);
    return;
  }
  const uint32_t r = find_window(sw, B, e.ts, 0u, inv);
  if (r < B) {
    const uint32_t pos = atomicAdd(&s_n[u * B + ((x + r) & (B - 1u))], 1u);
    if (pos < g.log_cap) store_event(unit_log(q, g, unit0 + u, x + r) + pos, e);
    else atomicOr(&q.ws->error, kErrQueueOverflow);
  } else {
    const uint32_t pos = atomicAdd(s_over, 1u);
    if (pos < over.cap) store_event(over.at(pos), e);
    else atomicOr(&q.ws->error, kErrQueueOverflow);
  }
}

// The filing launch of the step that commits window cur (and of the start, when every initial event
// lies beyond the calendar): a workgroup of kFileThreads per group.  s_n: units per group x B counts
// in LDS.  Neighbouring groups' parts lie side by side in every outbox, some 50 bytes each, so the
// workgroups of one XCD (dispatched round robin, blockIdx mod 8) take a run of groups and share
// the lines in its L2: with group = blockIdx the launch fetched each line several times over, and
// took 29 us instead of 24 at 2^20 LPs.
constexpr uint32_t kXcds = 8;
__device__ __forceinline__ void file_group(const LaqView& q, const Groups& g, float end_time, float inv, uint32_t* s_n) {
  __shared__ uint32_t sw[kCalMaxWindows];
  __shared__ uint16_t s_from[kFileCap];                // the source of each inbox event of a chunk
  __shared__ int s_shift[kFileUnits];
  __shared__ uint32_t s_wave[kFileThreads / kWave];
  __shared__ uint32_t s_over, s_pn, s_pb;
  const uint32_t run = (g.groups + kXcds - 1u) / kXcds;
  const uint32_t grp = blockIdx.x % kXcds * run + blockIdx.x / kXcds;
  if (q.ws->done || grp >= g.groups) return;
  const uint32_t t = threadIdx.x, B = q.cal_windows, x = q.cal_st->cur;
  const uint32_t per = 1u << (g.group_shift - kUnitLog2);
  const uint32_t unit0 = grp * per;
  const uint32_t nu = g.units - unit0 < per ? g.units - unit0 : per;
  const uint32_t end_bits = f_to_bits(end_time);
  const OverList over = over_list(g, grp);
  const uint32_t no0 = g.over_n[grp * kOverWords];
  const uint32_t no = no0 < over.cap ? no0 : over.cap;
  // issued first: the parts of the first units' first passes (always valid) and their pass counts
  uint32_t np[2], part[2];
  auto load_parts = [&](uint32_t u0) {
#pragma unroll
    for (uint32_t h = 0; h < 2; ++h) {
      const uint32_t u = u0 + 2u * t + h;
      np[h] = u < g.units ? g.npass[u] : 0u;
      part[h] = u < g.units ? g.parts[(size_t)u * g.passes * kMaxGroups + grp] : 0u;
    }
  };
  load_parts(0u);
  for (uint32_t i = t; i < nu * B; i += kFileThreads) s_n[i] = g.wlog_n[(size_t)unit0 * B + i];
  load_windows(q, x, sw);
  if (t == 0) s_over = s_pn = 0u;
  __syncthreads();
  // the group's events beyond the calendar: filed, parked, or kept, closed up in place (a chunk is
  // in registers before any of it is written, and never to a place past what has been read)
  for (uint32_t c0 = 0; c0 < no; c0 += kFileThreads) {
    const bool has = c0 + t < no;
    const Event e = has ? load_event(over.at(c0 + t)) : Event{};
    __syncthreads();
    const bool parked = has && !(e.ts < end_bits);
    const bool keep = has && !parked && !(e.ts < sw[B - 1u]);
    uint32_t rank = 0;
    if (parked) rank = atomicAdd(&s_pn, 1u);
    else if (has && !keep) file_event(q, g, sw, x, inv, unit0, nu, s_n, &s_over, over, e);
    const uint64_t mk = __ballot(keep);
    uint32_t at = 0;
    if (mk && lane_id() == 0) at = atomicAdd(&s_over, (uint32_t)__popcll(mk));
    at = (uint32_t)__shfl((int)at, 0, kWave);
    if (keep) store_event(over.at(at + (uint32_t)__popcll(mk & ((1ull << lane_id()) - 1ull))), e);
    __syncthreads();
    if (s_pn) {                                        // uniform: read after a barrier
      if (t == 0) s_pb = atomicAdd(q.parked_n, s_pn);
      __syncthreads();
      if (parked) list_store(q, 0u, Route::kParked, s_pb + rank, make_uint4(e.ts, e.dst, e.src, e.seq));
      __syncthreads();
      if (t == 0) s_pn = 0u;
      __syncthreads();
    }
  }
  // the group's parts of the units' outboxes: two units per thread, then a thread per event
  for (uint32_t u0 = 0; u0 < g.units; u0 += kFileUnits) {
    if (u0) load_parts(u0);
    for (uint32_t pass = 0; pass == 0 || __syncthreads_or(pass < np[0] || pass < np[1]); ++pass) {
      uint32_t o0[2], len[2];
#pragma unroll
      for (uint32_t h = 0; h < 2; ++h) {
        if (pass)
          part[h] = pass < np[h] ? g.parts[((size_t)(u0 + 2u * t + h) * g.passes + pass) * kMaxGroups + grp] : 0u;
        o0[h] = part[h] & 0xFFFFu;
        len[h] = part[h] >> 16;
      }
      uint32_t inc = len[0] + len[1];
#pragma unroll
      for (int off = 1; off < kWave; off <<= 1) {
        const uint32_t y = (uint32_t)__shfl_up((int)inc, off, kWave);
        if (lane_id() >= off) inc += y;
      }
      if (lane_id() == kWave - 1) s_wave[t / kWave] = inc;
      __syncthreads();
      uint32_t total = 0, before = 0;
      for (uint32_t w = 0; w < kFileThreads / kWave; ++w) {
        before += w < t / kWave ? s_wave[w] : 0u;
        total += s_wave[w];
      }
      uint32_t at[2];
      at[0] = before + inc - len[0] - len[1];
      at[1] = at[0] + len[0];
#pragma unroll
      for (uint32_t h = 0; h < 2; ++h) s_shift[2u * t + h] = (int)o0[h] - (int)at[h];   // place in the part, from the chunk's
      for (uint32_t p0 = 0; p0 < total; p0 += kFileCap) {
        const uint32_t p1 = total - p0 < kFileCap ? total : p0 + kFileCap;
#pragma unroll
        for (uint32_t h = 0; h < 2; ++h)
          for (uint32_t i = at[h] < p0 ? p0 : at[h]; i < at[h] + len[h] && i < p1; ++i) s_from[i - p0] = (uint16_t)(2u * t + h);
        __syncthreads();
        for (uint32_t i0 = p0; i0 < p1; i0 += kFileBurst * kFileThreads) {   // a thread's loads in flight together
          Event e[kFileBurst];
#pragma unroll
          for (uint32_t j = 0; j < kFileBurst; ++j) {
            const uint32_t i = i0 + j * kFileThreads + t;
            if (i < p1) {
              const uint32_t k = s_from[i - p0];
              e[j] = load_event(g.out + ((size_t)(u0 + k) * g.passes + pass) * kUnitPass + (uint32_t)((int)i + s_shift[k]));
            }
          }
#pragma unroll
          for (uint32_t j = 0; j < kFileBurst; ++j)
            if (i0 + j * kFileThreads + t < p1) file_event(q, g, sw, x, inv, unit0, nu, s_n, &s_over, over, e[j]);
        }
        __syncthreads();
      }
    }
  }
  __syncthreads();
  for (uint32_t i = t; i < nu * B; i += kFileThreads) g.wlog_n[(size_t)unit0 * B + i] = s_n[i];
  if (t == 0) g.over_n[grp * kOverWords] = s_over;
}

}  // namespace cal
}  // namespace gpq
