// devmem.hip -- see devmem.h.
#include "devmem.h"

#include <hip/hip_runtime.h>

#include <list>
#include <mutex>
#include <unordered_map>

namespace gpq {
namespace {

struct Block {
  void* p;
  size_t size;
  int dev;                       // kDevice: the device it lies on; kPinned: -1
  MemKind kind;
};

// Kept blocks, oldest first.  A process keeps a few hundred at most, so a linear search is cheap
// next to any launch.  Never destroyed: the HIP runtime may be gone when static objects end.
struct Kept {
  std::mutex mu;
  std::list<Block> blocks;
  std::unordered_map<void*, int> dev_of;     // device of every block handed out or kept
  size_t bytes[2] = {0, 0};
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
    auto best = k.blocks.end();              // the smallest that fits without wasting half of it
    for (auto it = k.blocks.begin(); it != k.blocks.end(); ++it)
      if (it->kind == kind && it->dev == dev && it->size >= want && it->size <= most &&
          (best == k.blocks.end() || it->size < best->size))
        best = it;
    if (best != k.blocks.end()) {
      void* p = best->p;
      *size = best->size;
      k.bytes[(int)kind] -= best->size;
      k.blocks.erase(best);
      return p;
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
  std::list<Block> out;
  {
    std::lock_guard<std::mutex> lock(k.mu);
    const Block b{p, size, k.dev_of[p], kind};
    if (size > most) {
      out.push_back(b);
    } else {
      k.blocks.push_back(b);
      k.bytes[(int)kind] += size;
      for (auto it = k.blocks.begin(); k.bytes[(int)kind] > most && it != k.blocks.end();) {
        if (it->kind != kind) { ++it; continue; }
        k.bytes[(int)kind] -= it->size;
        out.push_back(*it);
        it = k.blocks.erase(it);
      }
    }
    for (const Block& x : out) k.dev_of.erase(x.p);
  }
  for (const Block& x : out) free_block(x);
}

void mem_release_kept() {
  Kept& k = kept();
  std::list<Block> out;
  {
    std::lock_guard<std::mutex> lock(k.mu);
    out.swap(k.blocks);
    k.bytes[0] = k.bytes[1] = 0;
    for (const Block& x : out) k.dev_of.erase(x.p);
  }
  for (const Block& x : out) free_block(x);
}

}  // namespace gpq

extern "C" gpq_status gpq_release_kept_memory(void) {
  gpq::mem_release_kept();
  return GPQ_OK;
}
