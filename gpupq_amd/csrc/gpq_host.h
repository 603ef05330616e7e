// gpq_host.h -- host-side internals: error plumbing, device buffers, the queue
// base class every queue kind derives from, and the window state shared with
// the model kernels.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdio>
#include <string>
#include <utility>
#include <vector>

#include "../../include/gpupq.h"
#include "devmem.h"
#include "gpq_device.h"

namespace gpq {

void set_error(const std::string& msg);
const std::string& last_error();

#define GPQ_HIP(call)                                                                   \
  do {                                                                                  \
    hipError_t e_ = (call);                                                             \
    if (e_ != hipSuccess) {                                                             \
      ::gpq::set_error(std::string(#call) + ": " + hipGetErrorString(e_));              \
      return GPQ_ERR_HIP;                                                               \
    }                                                                                   \
  } while (0)

#define GPQ_TRY(expr)                                                                   \
  do {                                                                                  \
    gpq_status s_ = (expr);                                                             \
    if (s_ != GPQ_OK) return s_;                                                        \
  } while (0)

#define GPQ_CHECK_ARG(cond, msg)                                                        \
  do {                                                                                  \
    if (!(cond)) { ::gpq::set_error(msg); return GPQ_ERR_INVALID; }                     \
  } while (0)

// Device memory tracked by its owner, given back in the owner's destructor (devmem.h keeps it for
// the next owner, whose stream knows nothing of this owner's work: the work must have ended by
// then).  The streams named with on() are waited for; the device as a whole is not, as that
// would break a graph capture on another host thread.
class DeviceArena {
 public:
  ~DeviceArena() { release(); }
  void on(hipStream_t s) { streams_.push_back(s); }
  // Blocks of no more than is asked for, for an owner whose memory has a stated bound.
  void exact() { exact_ = true; }
  template <class T>
  gpq_status alloc(T** p, size_t count) {
    const size_t bytes = count * sizeof(T) > 0 ? count * sizeof(T) : 16;
    size_t size = 0;
    void* raw = mem_get(MemKind::kDevice, bytes, &size, exact_);
    if (!raw) {
      set_error("hipMalloc of " + std::to_string(bytes) + " bytes failed");
      return GPQ_ERR_NOMEM;
    }
    blocks_.push_back({raw, size});
    bytes_ += size;
    *p = static_cast<T*>(raw);
    return GPQ_OK;
  }
  size_t bytes() const { return bytes_; }     // of the blocks held
  void release() {
    for (hipStream_t s : streams_) (void)hipStreamSynchronize(s);
    streams_.clear();
    for (const auto& b : blocks_) mem_put(MemKind::kDevice, b.first, b.second);
    blocks_.clear();
    bytes_ = 0;
  }

 private:
  std::vector<std::pair<void*, size_t>> blocks_;
  std::vector<hipStream_t> streams_;
  size_t bytes_ = 0;
  bool exact_ = false;
};

// Pinned host memory of one owner, which ends every copy to or from it first.
class PinnedBlock {
 public:
  PinnedBlock() = default;
  PinnedBlock(const PinnedBlock&) = delete;
  PinnedBlock& operator=(const PinnedBlock&) = delete;
  ~PinnedBlock() { release(); }
  template <class T>
  gpq_status alloc(T** p, size_t count) {
    release();
    p_ = mem_get(MemKind::kPinned, count * sizeof(T) > 0 ? count * sizeof(T) : 16, &size_);
    if (!p_) {
      set_error("hipHostMalloc of " + std::to_string(count * sizeof(T)) + " bytes failed");
      return GPQ_ERR_HIP;
    }
    *p = static_cast<T*>(p_);
    return GPQ_OK;
  }
  void release() {
    if (!p_) return;
    mem_put(MemKind::kPinned, p_, size_);
    p_ = nullptr;
  }

 private:
  void* p_ = nullptr;
  size_t size_ = 0;
};

inline uint32_t ceil_div(uint64_t a, uint64_t b) { return (uint32_t)((a + b - 1) / b); }
inline bool is_pow2(uint64_t x) { return x && !(x & (x - 1)); }
inline uint32_t log2u(uint64_t x) { uint32_t r = 0; while ((1ull << r) < x) ++r; return r; }

// Common part of every queue handle.  The window (gmin, safe-window end, done flag)
// lives in device memory and is published by the queue's post kernels.
class QueueBase {
 public:
  explicit QueueBase(const gpq_queue_config& c) : cfg(c) {}
  virtual ~QueueBase() {
    arena.release();                         // waits for the stream
    if (stream) (void)hipStreamDestroy(stream);
  }
  gpq_status init_common();

  virtual gpq_status init() = 0;
  virtual gpq_status pre() { return GPQ_OK; }
  virtual gpq_status post() = 0;
  virtual gpq_status post_init() { return post(); }
  virtual gpq_status lp_contents(uint32_t lp, Event* out, uint32_t cap, uint32_t* n) = 0;
  virtual gpq_status pending(uint64_t* n) = 0;
  virtual gpq_status length(uint32_t lp, uint32_t* n) = 0;
  virtual gpq_status clear_lp(uint32_t lp) = 0;
  // Per-LP queues: every LP emptied on the queue's stream (a new search on the same open lists).
  virtual gpq_status empty_all() {
    set_error("empty_all is provided for the per-LP queues");
    return GPQ_ERR_UNSUPPORTED;
  }
  // Number of queue_peek() slots the model iterates over.
  virtual uint32_t peek_slots() const { return cfg.num_lps; }

  // Folds partial[0 .. partial_slots) into the window state (one small kernel on stream), unless
  // the post kernel has published the window (alloc_partial, publish_args).
  gpq_status publish_window();
  // partial[0 .. partial_slots), and the words by which up to kFoldMost blocks fold their minima in the
  // post kernel itself.
  gpq_status alloc_partial();
  WindowPublish publish_args() const;
  // A search's end, decided where the window is published: between set_search and the post.  False when the
  // queue publishes it by a launch of its own.
  bool set_search(const uint32_t* best, uint32_t* done, unsigned long long* steps);
  gpq_status window(WindowState* out);   // synchronous copy of the device window state
  gpq_status error_flags(uint32_t* flags);
  gpq_status stats_get(gpq_queue_stats* out);
  // *out = sum of a device u32 array (synchronous); tmp is one device u64.
  gpq_status sum_u32(const uint32_t* d_values, uint32_t count, uint64_t* tmp, uint64_t* out);

  gpq_queue_config cfg;
  hipStream_t stream = nullptr;
  DeviceArena arena;
  WindowState* ws = nullptr;          // device
  WindowState* host_ws = nullptr;     // pinned mirror for polling
  PinnedBlock host_ws_block;
  hipEvent_t profile_mark = nullptr;  // when set, recorded just before the window publication
  uint32_t* partial = nullptr;        // device, one slot per reduction block
  uint32_t partial_slots = 0;
  uint32_t* fold = nullptr;           // device, two words after the partials; nullptr: publish by a launch
  const uint32_t* search_best = nullptr;
  uint32_t* search_done = nullptr;
  unsigned long long* search_steps = nullptr;
  uint32_t threads = 256;
  // Work counters (device, kStatSlots u64) when cfg.collect_stats; nullptr otherwise.
  // Slots: 0 inserted, 1 displaced, 2 merged LPs, 3 scanned LPs, 4 aux bytes, 5 records
  // sorted, 6 records merged, 7 records scanned by the safe-event selection.
  unsigned long long* stats = nullptr;
  unsigned long long* acct(int slot) const { return stats ? stats + slot : nullptr; }
};

constexpr int kStatSlots = 8;
constexpr int kStatSorted = 5, kStatMerged = 6, kStatSelected = 7;

}  // namespace gpq

struct gpq_queue {
  gpq::QueueBase* impl;
};
