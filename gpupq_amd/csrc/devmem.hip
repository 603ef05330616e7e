// devmem.hip -- see devmem.h.
#include "devmem.h"

#include <hip/hip_runtime.h>

#include <map>
#include <mutex>
#include <set>
#include <tuple>
#include <unordered_map>
#include <vector>

namespace gpq {
namespace {

struct Block {
  void* p;
  size_t size;
  int dev;                       // kDevice: the device it lies on; kPinned: -1
  MemKind kind;
};

// Kept blocks by kind: by age, and by device and size, kMostBlocks of a kind.  A process that had 1500 small
// queues at once kept 13,000 blocks, and making the next queue took 1.4 ms, of which searching one list of
// them took 1.0 and the runtime's own search among its allocations 0.2 (0.12 with none kept).  Never destroyed: the HIP runtime may be gone when static objects end.
constexpr size_t kMostBlocks = 1024;
struct Kept {
  std::mutex mu;
  std::map<uint64_t, Block> by_age[2];                            // the oldest first
  std::set<std::tuple<int, size_t, uint64_t>> by_size[2];         // device, size, age
  uint64_t next_age = 0;
  std::unordered_map<void*, int> dev_of;     // device of every block handed out or kept
  size_t bytes[2] = {0, 0};

  void add(const Block& b) {
    const int i = (int)b.kind;
    by_age[i].emplace(next_age, b);
    by_size[i].emplace(b.dev, b.size, next_age);
    ++next_age;
    bytes[i] += b.size;
  }
  Block take(MemKind kind, uint64_t age) {
    const int i = (int)kind;
    const auto it = by_age[i].find(age);
    const Block b = it->second;
    by_age[i].erase(it);
    by_size[i].erase(std::make_tuple(b.dev, b.size, age));
    bytes[i] -= b.size;
    return b;
  }
};

Kept& kept() {
  static Kept* k = new Kept;
  return *k;
}

// Kept bytes: an eighth of the device's memory (36 GiB of 288), so that the largest simulations' logs
// (15 to 20 GB) are kept and the rest of the card stays with the process's other users; 1 GiB
// of pinned memory.
size_t bound(MemKind kind) {
  if (kind == MemKind::kPinned) return (size_t)1 << 30;
  static const size_t b = [] {
    size_t free_b = 0, total = 0;
    if (hipMemGetInfo(&free_b, &total) != hipSuccess) {
      (void)hipGetLastError();
      return (size_t)0;
    }
    return total / 8;
  }();
  return b;
}

void free_block(const Block& b) {
  if (b.kind == MemKind::kPinned) (void)hipHostFree(b.p);
  else (void)hipFree(b.p);
}

// Sizes are rounded up so that handles of nearly the same size can take each other's blocks: to a
// power of two up to 1 MiB, to a sixteenth of one above.
size_t rounded(size_t n) {
  size_t p = 256;
  while (p < n) p *= 2;
  if (p <= ((size_t)1 << 20)) return p;
  const size_t step = p / 32;                // p/2 < n <= p: at most a sixteenth of n is added
  return (n + step - 1) / step * step;
}

void* fresh(MemKind kind, size_t size) {
  void* p = nullptr;
  const hipError_t e = kind == MemKind::kPinned ? hipHostMalloc(&p, size, hipHostMallocDefault) : hipMalloc(&p, size);
  if (e == hipSuccess) return p;
  (void)hipGetLastError();
  return nullptr;
}

}  // namespace

void* mem_get(MemKind kind, size_t bytes, size_t* size, bool exact) {
  int dev = -1;
  if (kind == MemKind::kDevice && hipGetDevice(&dev) != hipSuccess) {
    (void)hipGetLastError();
    return nullptr;
  }
  const size_t want = exact ? (bytes + 255) / 256 * 256 : rounded(bytes), most = exact ? want : 2 * want + 1;
  Kept& k = kept();
  {
    std::lock_guard<std::mutex> lock(k.mu);
    const auto& sizes = k.by_size[(int)kind];          // the smallest that fits without wasting half of it
    const auto best = sizes.lower_bound(std::make_tuple(dev, want, (uint64_t)0));
    if (best != sizes.end() && std::get<0>(*best) == dev && std::get<1>(*best) <= most) {
      const Block b = k.take(kind, std::get<2>(*best));
      *size = b.size;
      return b.p;
    }
  }
  void* p = fresh(kind, want);
  if (!p) {                                  // the kept blocks may be what is missing
    mem_release_kept();
    p = fresh(kind, want);
  }
  size_t got = want;
  if (!p && want != bytes) {                 // or the rounding
    got = bytes;
    p = fresh(kind, got);
  }
  if (!p) return nullptr;
  *size = got;
  std::lock_guard<std::mutex> lock(k.mu);
  k.dev_of[p] = dev;
  return p;
}

void mem_put(MemKind kind, void* p, size_t size) {
  if (!p) return;
  Kept& k = kept();
  const size_t most = bound(kind);
  std::vector<Block> out;
  {
    std::lock_guard<std::mutex> lock(k.mu);
    const Block b{p, size, k.dev_of[p], kind};
    if (size > most) {
      out.push_back(b);
    } else {
      k.add(b);
      while (k.bytes[(int)kind] > most || k.by_age[(int)kind].size() > kMostBlocks)
        out.push_back(k.take(kind, k.by_age[(int)kind].begin()->first));
    }
    for (const Block& x : out) k.dev_of.erase(x.p);
  }
  for (const Block& x : out) free_block(x);
}

void mem_release_kept() {
  Kept& k = kept();
  std::vector<Block> out;
  {
    std::lock_guard<std::mutex> lock(k.mu);
    for (int i = 0; i < 2; ++i) {
      for (const auto& x : k.by_age[i]) out.push_back(x.second);
      k.by_age[i].clear();
      k.by_size[i].clear();
      k.bytes[i] = 0;
    }
    for (const Block& x : out) k.dev_of.erase(x.p);
  }
  for (const Block& x : out) free_block(x);
}

}  // namespace gpq

extern "C" gpq_status gpq_release_kept_memory(void) {
  gpq::mem_release_kept();
  return GPQ_OK;
}
