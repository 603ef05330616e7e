// queue_hq.hip -- global parallel heap with r-record nodes (Deo and Prasad, "Parallel
// heap: an optimal parallel priority queue", J. Supercomputing 6, 1992), restated for a
// device-resident schedule.  The reference (src/heap_queue.cu) drives each node merge
// from host pthreads with device-side launches, cudaStreamSynchronize and D2H copies per
// level; here every step is a fixed launch sequence whose kernels read the sizes and
// node choices from device memory.
//
// What bounds a step is that sequence and the latency of each merge: at 10^5 LPs a merge's bytes
// take 1 us and its launch 4.  So a merge launch plans for itself -- every block derives the tasks
// from the heap's counts, and one commits what they change -- and deals the tiles of those that
// have records out to its blocks; no node is copied back after a merge, since nodes are reached
// through a table of slots and a merge writes a free slot that then becomes the node's; the refill is
// part of the merge that fills the root; and the insert chunks follow one another down the heap, a level
// behind the one before.  100,003 LPs, 16 events each: 320 us a step with 39 merges and 30
// planners, 219 us with the 18 merges here; 200 with the selection in three launches and the tickets on
// several words as well.
//
// queue_post:
//  1. sort the step's inserts; M = merge(root, inserts)            (src/heap_queue.cu:1541-1553, 1448-1470)
//  2. publish the window from M[0]; select one safe record per LP of M with ts < window
//     end and key <= max(root) while nodes exist below the root -> dequeue buffer
//                                                                   (:478-547, 1560-1604)
//  3. R = M minus the selection: the first r records become the root, the rest are
//     carried down as insert chunks                                 (:418-466, 1097-1249)
//  4. a short root is refilled from the last node (copy_last, :975-1094)
//  5. delete-update, level by level: every dirty node whose largest record exceeds a
//     child's smallest merges with both children; it keeps the smallest records, the
//     child with the larger maximum (or the non-full right child) takes the largest,
//     the other the middle, and both children are checked at the next level
//                                                                   (:631-784)
//  6. insert-update: each chunk travels root -> target node, every node on the path
//     keeping its smallest records                                  (:817-960)
#include <algorithm>

#include "merge_tile.cuh"
#include "queues.h"

namespace gpq {
namespace {

__device__ __forceinline__ uint32_t depth_of(uint32_t v) { return 31u - __clz(v + 1u); }

}  // namespace

// One heap's arrays.  Node v's records are at store + slot[v] * r; spare[0 .. spares) are the slots
// that no node has: one per task of the widest delete-update level, then one per insert chunk.
constexpr uint32_t kTickets = 8, kTicketWords = 32;
struct HqHeap {
  HqState* st;
  uint32_t* counts;      // by node
  uint32_t* slot;
  uint32_t* spare;
  Event* store;
  uint32_t* ticket;      // kTickets + 1 counts of blocks that have planned, a line each; 0 between launches
  uint32_t* dirty;       // per parity of a level, `slots` nodes whose children are to be looked at
  uint32_t* dirty_n;     // ... and their number; dirty_n[2]: the tasks of `second`
  MergeTask* second;     // a level's merges of parents with their children
  uint32_t* second_v;    // ... and the parents
  WindowState* ws;
  unsigned long long* acct;
  uint32_t r, nodes, slots;
  __device__ __forceinline__ Event* at(uint32_t v) const { return store + (size_t)slot[v] * r; }
  __device__ __forceinline__ Event* at_spare(uint32_t i) const { return store + (size_t)spare[i] * r; }
  __device__ __forceinline__ void swap(uint32_t v, uint32_t i) const {   // node v takes spare slot i
    const uint32_t x = slot[v];
    slot[v] = spare[i];
    spare[i] = x;
  }
};

namespace {

using Heap = HqHeap;

__global__ void hq_init_kernel(Heap p, uint32_t spares, uint32_t* first, uint32_t num_lps, const Event* merged) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < p.nodes) {
    p.counts[i] = 0;
    p.slot[i] = i;
  }
  if (i < spares) p.spare[i] = p.nodes + i;
  if (i < num_lps) first[i] = 0xFFFFFFFFu;
  if (i == 0) {
    HqState s{};
    s.mptr = merged;
    *p.st = s;
    for (uint32_t x = 0; x <= kTickets; ++x) p.ticket[x * kTicketWords] = 0;
    *p.ws = WindowState{kInfBits, 0u, 0u, 0u, 0ull, 0u, 0u};
  }
}

// The window that starts at the smallest pending time g.
__device__ __forceinline__ void set_window(WindowState* ws, uint32_t g, float lookahead, float horizon) {
  float wend = bits_to_f(g) + lookahead;
  if (horizon < wend) wend = horizon;
  ws->gmin = g;
  ws->wend = f_to_bits(wend);
  ws->done = (g == kInfBits || !(bits_to_f(g) < horizon)) ? 1u : 0u;
  ws->windows += 1;
}

__device__ __forceinline__ void set_select(HqState* st, uint32_t select) {
  st->select = select;
  if (select) return;
  st->prefix = 0;
  st->deq_n = 0;
  st->rest_n = 0;
}

// Step 2, window over several heaps (heap h's merged buffer at merged + h * mstride): the smallest
// record starts it; the reference takes the minimum over its heaps' dequeue
// buffers (src/heap_queue.cu:1783-1806).
__global__ void hq_window_kernel(HqState* st, uint32_t heaps, const Event* merged, size_t mstride, WindowState* ws,
                                 float lookahead, float horizon, uint32_t select) {
  uint32_t g = kInfBits;
  for (uint32_t h = 0; h < heaps; ++h) {
    const uint32_t v = st[h].mcount ? merged[h * mstride].ts : kInfBits;
    g = v < g ? v : g;
    set_select(st + h, select);
  }
  set_window(ws, g, lookahead, horizon);
}

// The merges of a step.  A launch has tasks() = n of them; plan(y, n) is the y-th (empty for y >= n),
// place(t, k) completes it when k tasks before it are not empty, commit(y, t, k) makes its
// changes to the heap, and finish(k) runs once with the number of tasks that are not empty.  Where plan reads
// what commit changes (kTicket: at most a wave of tasks), commit waits until every block has planned.
struct MergeOp {
  __device__ void place(MergeTask&, uint32_t) const {}
  __device__ void finish(uint32_t) const {}
};

// Step 1: M = merge(root, sorted inserts); the selection bound is the root's maximum.  With one
// heap the window is published here as well.
struct InsertMerge : MergeOp {
  Heap p;
  const Event* ins;
  Event* merged;
  uint32_t enq_cap, publish, select;
  float lookahead, horizon;
  static constexpr bool kTicket = true, kAlways = true;
  __device__ uint32_t tasks() const { return 1u; }
  __device__ MergeTask plan(uint32_t y, uint32_t n) const {
    if (y >= n) return MergeTask{};
    const uint32_t m = p.st->m < enq_cap ? p.st->m : enq_cap;
    const uint32_t c0 = p.counts[0];
    MergeTask t{};
    t.a1 = t.a2 = p.at(0);
    t.n_a1 = c0;
    t.b = ins;
    t.n_b = m;
    t.out[0] = t.out[1] = t.out[2] = merged;
    t.end[0] = t.end[1] = t.end[2] = c0 + m;
    return t;
  }
  __device__ void commit(uint32_t, const MergeTask& t, uint32_t) const {
    HqState* st = p.st;
    st->mcount = t.n_a1 + t.n_b;
    st->m = 0;
    st->bound_valid = st->last > 0 ? 1u : 0u;
    st->bound = t.n_a1 ? t.a1[t.n_a1 - 1] : Event{0u, 0u, 0u, 0u};
    if (!publish) return;
    const uint32_t a = t.n_a1 ? t.a1[0].ts : kInfBits, b = t.n_b ? t.b[0].ts : kInfBits;
    set_select(st, select);
    set_window(p.ws, a < b ? a : b, lookahead, horizon);
  }
};

// Steps 3 and 4: R = (unselected part of the scanned prefix) ++ M[prefix:]; root <- R[0:r), carry <-
// rest.  A short root takes records from the tail of the last node (copy_last).  Then the
// set-up of step 6: carried records are cut into chunks, each targeting the last node's free
// space or a new node at the end of the heap (the delete-update changes no count).
struct RootMerge : MergeOp {
  Heap p;
  const Event* merged;
  const Event* rest;
  Event* carry;
  static constexpr bool kTicket = true, kAlways = true;
  __device__ uint32_t tasks() const { return 1u; }
  __device__ MergeTask plan(uint32_t y, uint32_t n) const {
    if (y >= n) return MergeTask{};
    const HqState* st = p.st;
    const uint32_t prefix = st->prefix, rest_n = st->rest_n, last = st->last;
    const uint32_t tail = st->mcount - prefix;
    const uint32_t rn = rest_n + tail;
    const uint32_t root_n = rn < p.r ? rn : p.r;
    const uint32_t have = p.counts[last];
    const uint32_t take = root_n < p.r && last > 0 ? min(p.r - root_n, have) : 0u;
    MergeTask t{};
    t.a1 = rest;
    t.n_a1 = rest_n;
    t.a2 = merged + prefix;
    t.n_a2 = tail;
    t.b = p.at(last) + (have - take);
    t.n_b = take;
    t.out[0] = p.at(0);
    t.out[1] = t.out[2] = carry;
    t.end[0] = root_n + take;
    t.end[1] = t.end[2] = rn + take;
    return t;
  }
  __device__ void commit(uint32_t, const MergeTask& t, uint32_t) const {
    HqState* st = p.st;
    uint32_t last = st->last;
    uint32_t have = p.counts[last] - t.n_b;          // before the root's count is set: last may be 0
    if (last > 0) p.counts[last] = have;
    while (last > 0 && have == 0) have = p.counts[--last];
    p.counts[0] = t.end[0];
    const uint32_t carry_n = t.end[2] - t.end[0];
    uint32_t off = 0;
    for (uint32_t c = 0; c < (uint32_t)kHqMaxChunks; ++c) {
      uint32_t n = 0;
      if (off < carry_n) {
        if (last == 0 || have >= p.r) {
          if (last + 1u >= p.nodes) {
            off = carry_n;                           // the rest does not fit
            atomicOr(&p.ws->error, kErrHeapOverflow);
          } else {
            ++last;
            have = 0;
          }
        }
        if (off < carry_n) n = min(p.r - have, carry_n - off);
      }
      st->chunk_target[c] = last;
      st->chunk_n[c] = n;
      st->chunk_off[c] = off;
      have += n;
      off += n;
    }
    st->last = last;
    if (off < carry_n) atomicOr(&p.ws->error, kErrHeapOverflow);
  }
};

// Step 5, a level's first merge, a task per node of the level's list: the node's children into one
// sequence, if one of them begins before the node ends.  The merge of the node with that is planned
// now, while the children's ends can be read, and the children are the next level's list.
struct ChildrenMerge : MergeOp {
  Heap p;
  uint32_t level;
  Event* both;                                       // 2 r records per task that is not empty
  static constexpr bool kTicket = false, kAlways = false;
  __device__ const uint32_t* list() const { return p.dirty + (level & 1u) * p.slots; }
  __device__ uint32_t tasks() const { return level ? p.dirty_n[level & 1u] : 1u; }
  // One exit, and loads that do not depend on one another: with a return from between the two
  // comparisons the compiler (hipcc of ROCm 7.2.0, clang 22, -O3) lost the children's addresses on the way
  // from the second one: in its assembly that path cleared their registers and went on with the counts.
  // Keep it so, or read the assembly of what replaces it.
  __device__ MergeTask plan(uint32_t y, uint32_t n) const {
    const uint32_t top = p.nodes - 1u;
    const uint32_t v0 = level ? list()[min(y, p.slots - 1u)] : 0u, v = min(v0, top);   // any node for y >= n
    const uint32_t l = min(2u * v + 1u, top), rr = min(2u * v + 2u, top);
    const uint32_t cv = p.counts[v], nl = p.counts[l], nr = p.counts[rr];
    const Event* L = p.at(l);
    const Event* R = p.at(rr);
    const Event* V = p.at(v);
    const uint32_t cl = 2u * v + 1u < p.nodes ? nl : 0u, cr = 2u * v + 2u < p.nodes ? nr : 0u;
    // an empty node's record is not used
    const Event maxv = load_event(V + (cv ? cv - 1u : 0u)), minl = load_event(L), minr = load_event(R);
    const uint32_t out = ((cl ? 1u : 0u) & (key_less(minl, maxv) ? 1u : 0u)) |
                         ((cr ? 1u : 0u) & (key_less(minr, maxv) ? 1u : 0u));
    const uint32_t on = y < n && v == v0 && cv ? 0u - out : 0u;
    MergeTask a;
    a.a1 = a.a2 = L;
    a.n_a1 = cl & on;
    a.n_a2 = 0;
    a.b = R;
    a.n_b = cr & on;
    a.out[0] = a.out[1] = a.out[2] = both;           // task k's part of it: place()
    a.end[0] = a.end[1] = a.end[2] = a.n_a1 + a.n_b;
    return a;
  }
  __device__ void place(MergeTask& a, uint32_t k) const {
    a.out[0] = a.out[1] = a.out[2] = both + (size_t)k * 2u * p.r;
  }
  __device__ void commit(uint32_t y, const MergeTask& a, uint32_t k) const {
    const uint32_t cl = a.n_a1, cr = a.n_b;
    const uint32_t v = level ? list()[y] : 0u;
    const uint32_t cv = p.counts[v];
    Event* L = const_cast<Event*>(a.a1);
    Event* R = const_cast<Event*>(a.b);
    // the non-full right child, or the child with the larger maximum, takes the largest records
    const Event maxl = load_event(L + (cl ? cl - 1u : 0u)), maxr = load_event(R + (cr ? cr - 1u : 0u));
    const bool big_right = cr != 0 && (cl == 0 || cr < p.r || key_less(maxl, maxr));
    MergeTask b{};
    b.a1 = b.a2 = p.at(v);
    b.n_a1 = cv;
    b.b = a.out[0];
    b.n_b = cl + cr;
    b.out[0] = p.at_spare(k);
    b.out[1] = big_right ? L : R;
    b.out[2] = big_right ? R : L;
    b.end[0] = cv;
    b.end[1] = cv + (big_right ? cl : cr);
    b.end[2] = cv + cl + cr;
    p.second[k] = b;
    p.second_v[k] = v;
    uint32_t* next = p.dirty + (~level & 1u) * p.slots;
    if (2u * k + 1u < p.slots) {                     // the lowest level's children have none
      next[2u * k] = 2u * v + 1u;
      next[2u * k + 1u] = 2u * v + 2u;               // may be past the last node
    }
  }
  __device__ void finish(uint32_t tasks_on) const {
    p.dirty_n[~level & 1u] = min(2u * tasks_on, p.slots);
    p.dirty_n[2] = tasks_on;
  }
};

// ... and its second: the node keeps the smallest records, the children take the others in place.
struct ParentMerge : MergeOp {
  Heap p;
  static constexpr bool kTicket = false, kAlways = false;
  __device__ uint32_t tasks() const { return p.dirty_n[2]; }
  __device__ MergeTask plan(uint32_t y, uint32_t n) const {
    MergeTask t = p.second[min(y, p.slots - 1u)];
    const uint32_t on = y < n ? 0xFFFFFFFFu : 0u;
    t.n_a1 &= on;
    t.n_a2 &= on;
    t.n_b &= on;
    return t;
  }
  __device__ void commit(uint32_t y, const MergeTask&, uint32_t) const { p.swap(p.second_v[y], y); }
};

// Step 6: chunk c = first + y at level diag - c of its path from the root to its target node (the root
// is skipped: carried records are never smaller than the root's).  A node on the path keeps its
// smallest records and the others move on; the target takes the chunk.
struct PathMerge : MergeOp {
  Heap p;
  Event* carry;
  Event* chunk_buf;                                  // r records per chunk
  uint32_t first, diag, chunks;                      // chunks: of this launch
  static constexpr bool kTicket = true, kAlways = false;
  __device__ uint32_t tasks() const { return chunks; }
  __device__ MergeTask plan(uint32_t y, uint32_t n_tasks) const {
    if (y >= n_tasks) return MergeTask{};
    const uint32_t c = first + y, level = diag - c;
    const HqState* st = p.st;
    const uint32_t n = st->chunk_n[c], target = st->chunk_target[c], dt = depth_of(target);
    MergeTask t{};
    if (n == 0 || level > dt) return t;
    const uint32_t v = ((target + 1u) >> (dt - level)) - 1u;
    const uint32_t cv = p.counts[v];
    Event* x = carry + st->chunk_off[c];             // the chunk goes to and fro between two places
    Event* z = chunk_buf + (size_t)c * p.r;
    t.a1 = t.a2 = p.at(v);
    t.n_a1 = cv;
    t.b = level & 1u ? x : z;
    t.n_b = n;
    t.out[0] = p.at_spare(p.slots + c);
    t.out[1] = t.out[2] = level & 1u ? z : x;
    t.end[0] = level < dt ? cv : cv + n;
    t.end[1] = t.end[2] = cv + n;
    return t;
  }
  __device__ void commit(uint32_t y, const MergeTask& t, uint32_t) const {
    const uint32_t c = first + y, level = diag - c;
    const uint32_t target = p.st->chunk_target[c];
    const uint32_t v = ((target + 1u) >> (depth_of(target) - level)) - 1u;
    p.counts[v] = t.end[0];
    p.swap(v, p.slots + c);
  }
};

__device__ __forceinline__ uint32_t total_of(const MergeTask& t) { return t.n_a1 + t.n_a2 + t.n_b; }

// One wave plans the tasks g .. g + 63 of a launch of n; *k: the tasks before this lane's, from *on, that are not
// empty.  (InsertMerge and RootMerge are committed when they are empty as well.)
template <typename Op>
__device__ __forceinline__ MergeTask plan_lane(const Op& op, uint32_t g, uint32_t n, uint32_t* k, uint32_t* on) {
  MergeTask m = op.plan(g + (uint32_t)lane_id(), n);
  const bool some = total_of(m) != 0;
  const uint64_t mask = __ballot(some);
  *k = *on + (uint32_t)__popcll(mask & ((1ull << lane_id()) - 1ull));
  *on += (uint32_t)__popcll(mask);
  if (some) op.place(m, *k);
  return m;
}

template <typename Op>
__device__ __forceinline__ void commit_lane(const Op& op, uint32_t y, uint32_t n, const MergeTask& m, uint32_t k) {
  if (y >= n) return;
  const uint32_t total = total_of(m);
  if (total || Op::kAlways) op.commit(y, m, k);
  if (op.p.acct && total) atomicAdd(op.p.acct, (unsigned long long)total);
}

// The tiles of a launch's tasks, dealt out to its blocks.  Every block plans all tasks, a lane each
// (a wave of them at a time), so that only tasks with records take tiles.  With a grid slot per tile
// of every node of a level, 2352 blocks on the fifth level at 100,003 LPs, most found nothing to do: a
// ParentMerge took 18 us on average and takes 10, a step went from 288 us to 219.
template <typename Op, int kT>
__global__ __launch_bounds__(kT) void hq_merge_kernel(Op op) {
  constexpr uint32_t kTile = kT * kPerThread;
  __shared__ MergeTask t[kWave];
  __shared__ uint32_t first[kWave + 1];
  const uint32_t n = op.tasks(), lane = threadIdx.x;
  uint32_t g = 0, before = 0, on = 0, k = 0, ticket = 0;
  do {
    if (threadIdx.x < (uint32_t)kWave) {
      const MergeTask m = plan_lane(op, g, n, &k, &on);
      uint32_t inc = (total_of(m) + kTile - 1u) / kTile;
#pragma unroll
      for (int off = 1; off < kWave; off <<= 1) {
        const uint32_t x = (uint32_t)__shfl_up((int)inc, off, kWave);
        if (lane >= (uint32_t)off) inc += x;
      }
      t[lane] = m;
      first[lane + 1u] = inc;
      if (lane == 0) first[0] = 0;
      if (!Op::kTicket && blockIdx.x == 0) commit_lane(op, g + lane, n, m, k);
    }
    __syncthreads();
    // the plan's loads have returned: they decided what is in LDS
    if (Op::kTicket && threadIdx.x == 0) ticket = atomicAdd(&op.p.ticket[(1u + blockIdx.x % kTickets) * kTicketWords], 1u);
    const uint32_t all = first[kWave];
    for (uint32_t x = (blockIdx.x + gridDim.x - before % gridDim.x) % gridDim.x; x < all; x += gridDim.x) {
      uint32_t j = 0;                                  // the task of tile x: first[j] <= x < first[j + 1]
#pragma unroll
      for (uint32_t w = kWave / 2; w; w >>= 1)
        if (first[j + w] <= x) j += w;
      const MergeTask m = t[j];
      const OutMap om{{m.out[0], m.out[1], m.out[2]}, {m.end[0], m.end[1], m.end[2]}};
      merge_tile<kT>(ASrc{m.a1, m.a2, m.n_a1}, m.n_a1 + m.n_a2, m.b, m.n_b, (x - first[j]) * kTile, om);
    }
    before += all;
    g += kWave;
    if (g < n) __syncthreads();                        // the next wave of tasks replaces these
  } while (g < n);
  if (threadIdx.x >= (uint32_t)kWave) return;
  if (Op::kTicket) {
    // Counted on kTickets words and by the last of each on another one: on one word, where the blocks
    // arrive together, a step took 5 us longer (100,003 LPs).
    const uint32_t c = blockIdx.x % kTickets, mine = (gridDim.x - c + kTickets - 1u) / kTickets;
    if ((uint32_t)__shfl((int)ticket, 0, kWave) != mine - 1u) return;
    if (lane == 0) {
      op.p.ticket[(1u + c) * kTicketWords] = 0;
      ticket = atomicAdd(op.p.ticket, 1u);
    }
    if ((uint32_t)__shfl((int)ticket, 0, kWave) != min(gridDim.x, kTickets) - 1u) return;
    if (lane == 0) *op.p.ticket = 0;
    commit_lane(op, lane, n, t[lane], k);
  } else if (blockIdx.x == 0 && lane == 0) {
    op.finish(on);
  }
}

// The same tasks for merges with a partition launch, by one wave: written out (`slots` of them, the ones past
// the last empty) and committed at once.
template <typename Op>
__global__ __launch_bounds__(64) void hq_plan_kernel(Op op, MergeTask* tasks, uint32_t slots) {
  const uint32_t n = op.tasks();
  uint32_t on = 0;
  for (uint32_t g = 0; g < slots; g += kWave) {
    const uint32_t y = g + threadIdx.x;
    uint32_t k;
    const MergeTask m = plan_lane(op, g, n, &k, &on);
    if (y < slots) tasks[y] = m;
    commit_lane(op, y, n, m, k);
  }
  if (threadIdx.x == 0) op.finish(on);
}

__global__ void hq_pending_kernel(const uint32_t* counts, uint32_t num_nodes, unsigned long long* out) {
  if (threadIdx.x || blockIdx.x) return;
  unsigned long long s = 0;
  for (uint32_t v = 0; v < num_nodes; ++v) s += counts[v];
  *out = s;
}

// One launch of `ntasks` merges of up to max_total records each.  From kMergePartitionMin records on,
// three: the plans, the partition and the merges.
template <typename Op>
gpq_status launch_merges(const Op& op, uint32_t ntasks, uint64_t max_total, uint32_t tile, MergeTask* tasks,
                         uint32_t* splits, uint32_t stride, hipStream_t s) {
  if (max_total >= kMergePartitionMin) {
    hipLaunchKernelGGL(hq_plan_kernel<Op>, dim3(1), dim3(64), 0, s, op, tasks, ntasks);
    return merge_tasks(tasks, ntasks, max_total, s, tile, nullptr, splits, stride);
  }
  // three blocks per CU fit (LDS)
  const dim3 grid((uint32_t)std::min<uint64_t>((uint64_t)ceil_div(max_total, tile) * ntasks, 768));
  switch (tile) {
    case 1024: hipLaunchKernelGGL((hq_merge_kernel<Op, 128>), grid, dim3(128), 0, s, op); break;
    case 2048: hipLaunchKernelGGL((hq_merge_kernel<Op, 256>), grid, dim3(256), 0, s, op); break;
    default: hipLaunchKernelGGL((hq_merge_kernel<Op, 512>), grid, dim3(512), 0, s, op); break;
  }
  GPQ_HIP(hipGetLastError());
  return GPQ_OK;
}

uint32_t levels_with_children(uint32_t nodes) {
  uint32_t lv = 0;
  while (((1u << lv) - 1u) < nodes && 2u * ((1u << lv) - 1u) + 1u < nodes) ++lv;
  return lv;   // levels 0 .. lv-1 contain a node with a child
}

}  // namespace

HqHeap HqQueue::heap(uint32_t h) const {
  uint32_t* dirty = dirty_ + (size_t)h * dirty_words();
  return HqHeap{v_.st + h, counts_ + (size_t)h * nodes_, slot_ + (size_t)h * nodes_, spare_ + (size_t)h * spares_,
                nodes_buf_ + (size_t)h * (nodes_ + spares_) * r_, ticket_ + (size_t)h * (kTickets + 1) * kTicketWords, dirty, dirty + 2 * (size_t)slots_,
                second_ + (size_t)h * slots_, second_v_ + (size_t)h * slots_, ws, acct(kStatMerged), r_, nodes_, slots_};
}

template <typename Op>
gpq_status HqQueue::merges(uint32_t h, const Op& op, uint32_t ntasks, uint64_t max_total, hipStream_t s) const {
  return launch_merges(op, ntasks, max_total, tile_, tasks_ + (size_t)h * tasks_n_,
                       splits_ + (size_t)h * tasks_n_ * split_stride_, split_stride_, s);
}

const Event* HqQueue::node_at(uint32_t v, uint32_t slot) const {
  return nodes_buf_ + ((size_t)(v / nodes_) * (nodes_ + spares_) + slot) * r_;
}

gpq_status HqQueue::init() {
  GPQ_CHECK_ARG(cfg.node_size >= 1, "HQ: node_size (r) must be >= 1");
  heaps_ = cfg.heaps ? cfg.heaps : 1u;
  GPQ_CHECK_ARG(heaps_ <= cfg.num_lps && heaps_ <= 1024, "HQ: heaps must be in [1, min(num_lps, 1024)]");
  lps_per_heap_ = (uint32_t)ceil_div(cfg.num_lps, heaps_);
  const uint64_t total = (uint64_t)lps_per_heap_ * (cfg.capacity_per_lp ? cfg.capacity_per_lp : 1);
  const uint64_t nodes = cfg.heap_nodes ? cfg.heap_nodes : (total + cfg.node_size - 1) / cfg.node_size + 1;
  GPQ_CHECK_ARG(nodes >= 1 && nodes < (1u << 20), "HQ: bad heap_nodes");
  r_ = cfg.node_size;
  tile_ = cfg.sort_tile ? cfg.sort_tile : kMergeTile;
  GPQ_CHECK_ARG(valid_sort_tile(tile_), "HQ: sort_tile must be 0, 1024, 2048 or 4096");
  nodes_ = (uint32_t)nodes;
  // every heap takes a whole step's inserts (the events of one step may all go to one heap)
  const uint64_t enq_cap = (uint64_t)cfg.num_lps * (cfg.stage_per_lp ? cfg.stage_per_lp : 1);
  GPQ_CHECK_ARG(enq_cap + r_ < (1ull << 31), "HQ: num_lps * stage_per_lp + node_size must be < 2^31");
  GPQ_CHECK_ARG(enq_cap <= (uint64_t)(kHqMaxChunks - 1) * r_, "HQ: num_lps * stage_per_lp must be <= 7 * node_size");
  GPQ_CHECK_ARG((uint64_t)heaps_ * nodes_ * r_ < (1ull << 34), "HQ: heap too large");
  v_.num_lps = cfg.num_lps;
  v_.enq_cap = (uint32_t)enq_cap;
  v_.heaps = heaps_;
  v_.lps_per_heap = lps_per_heap_;
  levels_ = levels_with_children(nodes_);
  slots_ = levels_ ? (1u << (levels_ - 1)) : 1u;
  depth_ = 0;
  while ((1u << (depth_ + 1)) - 1u < nodes_) ++depth_;   // deepest level index of any node
  mcap_ = r_ + enq_cap;
  chunks_ = std::min<uint32_t>(kHqMaxChunks, (uint32_t)ceil_div(enq_cap, r_) + 1);
  spares_ = slots_ + chunks_;
  GPQ_TRY(arena.alloc(&nodes_buf_, (size_t)heaps_ * (nodes_ + spares_) * r_));
  GPQ_TRY(arena.alloc(&slot_, (size_t)heaps_ * nodes_));
  GPQ_TRY(arena.alloc(&spare_, (size_t)heaps_ * spares_));
  GPQ_TRY(arena.alloc(&ticket_, (size_t)heaps_ * (kTickets + 1) * kTicketWords));
  GPQ_TRY(arena.alloc(&counts_, (size_t)heaps_ * nodes_));
  GPQ_TRY(arena.alloc(&dirty_, (size_t)heaps_ * dirty_words()));
  v_.seg_cap = insert_stripe_cap(enq_cap);
  v_.area = (uint64_t)kInsertStripes * v_.seg_cap + enq_cap;
  GPQ_TRY(arena.alloc(&v_.enq, (size_t)heaps_ * v_.area));
  GPQ_TRY(arena.alloc(&v_.seg_m, (size_t)heaps_ * kStripeCounterWords));
  GPQ_TRY(arena.alloc(&seg_pre_, (size_t)heaps_ * (kInsertStripes + 2)));
  GPQ_HIP(hipMemsetAsync(v_.seg_m, 0, sizeof(uint32_t) * heaps_ * kStripeCounterWords, stream));
  // working buffers, one set per heap so that the heaps' steps can run concurrently
  scratch_n_ = ceil_div(mcap_, 1024);
  tasks_n_ = spares_;   // the tasks of one launch
  GPQ_TRY(arena.alloc(&sort_[0], (size_t)heaps_ * enq_cap));
  GPQ_TRY(arena.alloc(&sort_[1], (size_t)heaps_ * enq_cap));
  GPQ_TRY(arena.alloc(&order_, (size_t)heaps_ * sort_order_words(enq_cap)));
  GPQ_TRY(arena.alloc(&merged_, (size_t)heaps_ * mcap_));
  GPQ_TRY(arena.alloc(&rest_, (size_t)heaps_ * mcap_));
  GPQ_TRY(arena.alloc(&carry_, (size_t)heaps_ * mcap_));
  GPQ_TRY(arena.alloc(&chunk_buf_, (size_t)heaps_ * kHqMaxChunks * r_));
  GPQ_TRY(arena.alloc(&tmp2_, (size_t)heaps_ * slots_ * 2u * r_));
  GPQ_TRY(arena.alloc(&v_.deq, (size_t)heaps_ * lps_per_heap_));
  GPQ_TRY(arena.alloc(&v_.st, heaps_));
  GPQ_TRY(arena.alloc(&first_, cfg.num_lps));   // by LP: the heaps' LP ranges are disjoint
  GPQ_TRY(arena.alloc(&scratch_, (size_t)heaps_ * scratch_n_));
  GPQ_TRY(arena.alloc(&tasks_, (size_t)heaps_ * tasks_n_));
  GPQ_TRY(arena.alloc(&second_, (size_t)heaps_ * slots_));
  GPQ_TRY(arena.alloc(&second_v_, (size_t)heaps_ * slots_));
  split_stride_ = merge_split_words(std::max<uint64_t>(mcap_, 3ull * r_), tile_);
  GPQ_TRY(arena.alloc(&splits_, (size_t)heaps_ * tasks_n_ * split_stride_));
  if (heaps_ > 1) {
    // one stream per heap (default priority), forked from and joined back into the queue's
    // stream twice per step; a hipGraph capture of the step records the branches
    hs_.assign(heaps_, nullptr);
    ev_.assign(2 * heaps_ + 2, nullptr);
    for (auto& x : hs_) {
      GPQ_HIP(hipStreamCreateWithFlags(&x, hipStreamNonBlocking));
      arena.on(x);
    }
    for (auto& e : ev_) GPQ_HIP(hipEventCreateWithFlags(&e, hipEventDisableTiming));
  }
  GPQ_TRY(arena.alloc(&sum_, 1));
  v_.ws = ws;
  partial_slots = 1;
  GPQ_TRY(arena.alloc(&partial, 1));
  const uint32_t n = std::max({nodes_, cfg.num_lps, spares_});
  for (uint32_t h = 0; h < heaps_; ++h) {
    hipLaunchKernelGGL(hq_init_kernel, dim3(ceil_div(n, 256)), dim3(256), 0, stream, heap(h), spares_, first_, cfg.num_lps,
                       merged_ + (size_t)h * mcap_);
    GPQ_HIP(hipGetLastError());
  }
  return GPQ_OK;
}

HqQueue::~HqQueue() {
  arena.release();   // waits for the streams: a step that failed half way has not joined the heaps' to the queue's
  for (auto e : ev_) if (e) (void)hipEventDestroy(e);
  for (auto x : hs_) if (x) (void)hipStreamDestroy(x);
}

// One post over every heap: the merges of inserts into the roots, the global window, then per
// heap the selection and the heap maintenance.  With several heaps each heap's part runs on
// its own stream (the reference runs one host pthread per heap, src/heap_queue.cu:1721-1757).
gpq_status HqQueue::step(bool select) {
  if (heaps_ == 1) {
    GPQ_TRY(merge_root(0, select, stream));
    return step_heap(0, select, stream);
  }
  for (int phase = 0; phase < 2; ++phase) {
    hipEvent_t fork = ev_[2 * heaps_ + phase];
    GPQ_HIP(hipEventRecord(fork, stream));
    for (uint32_t h = 0; h < heaps_; ++h) {
      GPQ_HIP(hipStreamWaitEvent(hs_[h], fork, 0));
      GPQ_TRY(phase ? step_heap(h, select, hs_[h]) : merge_root(h, select, hs_[h]));
      hipEvent_t join = ev_[phase * heaps_ + h];
      GPQ_HIP(hipEventRecord(join, hs_[h]));
      GPQ_HIP(hipStreamWaitEvent(stream, join, 0));
    }
    if (!phase)
      hipLaunchKernelGGL(hq_window_kernel, dim3(1), dim3(1), 0, stream, v_.st, heaps_, merged_, (size_t)mcap_, ws,
                         cfg.lookahead, cfg.horizon, select ? 1u : 0u);
  }
  GPQ_HIP(hipGetLastError());
  return GPQ_OK;
}

// Step 1 for heap h: M = merge(root, sorted inserts).
gpq_status HqQueue::merge_root(uint32_t h, bool select, hipStream_t s) {
  HqState* st = v_.st + h;
  Event* sorted = sort_[0] + (size_t)h * v_.enq_cap;
  uint32_t* pre = seg_pre_ + (size_t)h * (kInsertStripes + 2);
  GPQ_TRY(gather_inserts(v_.seg_m + (size_t)h * kStripeCounterWords, v_.seg_cap, v_.enq_cap, v_.enq_cap, pre, &st->m,
                         ws, s));
  GPQ_TRY(sort_records(v_.enq + (size_t)h * v_.area, sorted, sort_[1] + (size_t)h * v_.enq_cap,
                       order_ + (size_t)h * sort_order_words(v_.enq_cap), &st->m, v_.enq_cap, s, acct(kStatSorted), pre,
                       v_.seg_cap));
  return merges(h, InsertMerge{{}, heap(h), sorted, merged_ + (size_t)h * mcap_, v_.enq_cap, heaps_ == 1 ? 1u : 0u,
                               select ? 1u : 0u, cfg.lookahead, cfg.horizon}, 1, mcap_, s);
}

// Steps 2 (selection) to 6 for heap h, after the window is published.
gpq_status HqQueue::step_heap(uint32_t h, bool select, hipStream_t s) {
  HqState* st = v_.st + h;
  const Heap p = heap(h);
  Event* merged = merged_ + (size_t)h * mcap_;
  Event* rest = rest_ + (size_t)h * mcap_;
  Event* carry = carry_ + (size_t)h * mcap_;
  Event* chunk_buf = chunk_buf_ + (size_t)h * kHqMaxChunks * r_;
  if (select) {
    const SelectBufs b{first_, scratch_ + (size_t)h * scratch_n_, &st->prefix, &st->deq_n, &st->rest_n};
    GPQ_TRY(select_safe(&st->mptr, &st->mcount, (uint32_t)mcap_, &ws->wend, &st->bound, &st->bound_valid, b,
                        v_.deq + (size_t)h * lps_per_heap_, rest, s, acct(kStatSelected)));
  }
  GPQ_TRY(merges(h, RootMerge{{}, p, merged, rest, carry}, 1, mcap_, s));
  for (uint32_t lv = 0; lv < levels_; ++lv) {
    GPQ_TRY(merges(h, ChildrenMerge{{}, p, lv, tmp2_ + (size_t)h * slots_ * 2u * r_}, 1u << lv, 2ull * r_, s));
    GPQ_TRY(merges(h, ParentMerge{{}, p}, 1u << lv, 3ull * r_, s));
  }
  // chunk c is at level d - c of its path in launch d: the chunks follow one another
  for (uint32_t d = 1; depth_ && d < depth_ + chunks_; ++d) {
    const uint32_t first = d > depth_ ? d - depth_ : 0u, end = std::min(d, chunks_);
    GPQ_TRY(merges(h, PathMerge{{}, p, carry, chunk_buf, first, d, end - first}, end - first, 2ull * r_, s));
  }
  GPQ_HIP(hipGetLastError());
  return GPQ_OK;
}

gpq_status HqQueue::post() { return step(true); }
gpq_status HqQueue::post_init() { return step(false); }

gpq_status HqQueue::pending(uint64_t* n) {
  hipLaunchKernelGGL(hq_pending_kernel, dim3(1), dim3(1), 0, stream, counts_, heaps_ * nodes_,
                     reinterpret_cast<unsigned long long*>(sum_));
  GPQ_HIP(hipGetLastError());
  GPQ_HIP(hipMemcpyAsync(n, sum_, sizeof(uint64_t), hipMemcpyDeviceToHost, stream));
  GPQ_HIP(hipStreamSynchronize(stream));
  return GPQ_OK;
}

gpq_status HqQueue::snapshot(std::vector<Event>* out, std::vector<uint32_t>* counts) {
  const uint32_t all = heaps_ * nodes_;   // node v of heap h is number h * nodes_ + v
  std::vector<uint32_t> slots(all);
  GPQ_HIP(hipMemcpyAsync(slots.data(), slot_, sizeof(uint32_t) * all, hipMemcpyDeviceToHost, stream));
  counts->resize(all);
  GPQ_HIP(hipMemcpyAsync(counts->data(), counts_, sizeof(uint32_t) * all, hipMemcpyDeviceToHost, stream));
  GPQ_HIP(hipStreamSynchronize(stream));
  out->clear();
  for (uint32_t v = 0; v < all; ++v) {
    const uint32_t c = (*counts)[v];
    if (!c) continue;
    const size_t at = out->size();
    out->resize(at + c);
    GPQ_HIP(hipMemcpyAsync(out->data() + at, node_at(v, slots[v]), sizeof(Event) * c, hipMemcpyDeviceToHost, stream));
  }
  GPQ_HIP(hipStreamSynchronize(stream));
  return GPQ_OK;
}

gpq_status HqQueue::node_contents(uint32_t v, Event* out, uint32_t cap, uint32_t* n) {
  GPQ_CHECK_ARG(v < heaps_ * nodes_, "node out of range");
  uint32_t c = 0, x = 0;
  GPQ_HIP(hipMemcpyAsync(&c, counts_ + v, 4, hipMemcpyDeviceToHost, stream));
  GPQ_HIP(hipMemcpyAsync(&x, slot_ + v, 4, hipMemcpyDeviceToHost, stream));
  GPQ_HIP(hipStreamSynchronize(stream));
  *n = c;
  const uint32_t k = std::min(c, cap);
  if (k) {
    GPQ_HIP(hipMemcpyAsync(out, node_at(v, x), sizeof(Event) * k, hipMemcpyDeviceToHost, stream));
    GPQ_HIP(hipStreamSynchronize(stream));
  }
  return GPQ_OK;
}

gpq_status HqQueue::length(uint32_t lp, uint32_t* n) {
  GPQ_CHECK_ARG(lp < cfg.num_lps, "lp out of range");
  std::vector<Event> all;
  std::vector<uint32_t> counts;
  GPQ_TRY(snapshot(&all, &counts));
  *n = (uint32_t)std::count_if(all.begin(), all.end(), [lp](const Event& e) { return e.dst == lp; });
  return GPQ_OK;
}

gpq_status HqQueue::clear_lp(uint32_t) {
  set_error("HQ: per-LP clear is not provided for the shared heap");
  return GPQ_ERR_UNSUPPORTED;
}

gpq_status HqQueue::lp_contents(uint32_t lp, Event* out, uint32_t cap, uint32_t* n) {
  GPQ_CHECK_ARG(lp < cfg.num_lps, "lp out of range");
  std::vector<Event> all;
  std::vector<uint32_t> counts;
  GPQ_TRY(snapshot(&all, &counts));
  std::vector<Event> mine;
  for (const Event& e : all)
    if (e.dst == lp) mine.push_back(e);
  std::sort(mine.begin(), mine.end(), [](const Event& a, const Event& b) {
    if (a.ts != b.ts) return a.ts < b.ts;
    if (a.src != b.src) return a.src < b.src;
    return a.seq < b.seq;
  });
  *n = (uint32_t)mine.size();
  for (uint32_t i = 0; i < mine.size() && i < cap; ++i) out[i] = mine[i];
  return GPQ_OK;
}

}  // namespace gpq
