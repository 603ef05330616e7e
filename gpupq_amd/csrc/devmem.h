// devmem.h -- device and pinned host memory of the handles, kept for the next handle.
//
// The driver wipes device memory after it is freed, at about 33 GB/s: once a process has handed out
// the card's clean pages, every byte a simulation allocates and frees costs it 30 ms per GiB (15
// GiB per 2^20-LP simulation).  Blocks that handles give back are therefore kept, up to a bound,
// and the next handle takes them.
#pragma once

#include <cstddef>

#include "../../include/gpupq.h"

namespace gpq {

enum class MemKind { kDevice, kPinned };

// A block of at least `bytes` (> 0) on the current device (kDevice) or in pinned host memory;
// nullptr when there is none.  Its contents are undefined.  *size receives the block's own size: up
// to twice `bytes` when it was kept, or with `exact` no more than `bytes` rounded up to 256.
void* mem_get(MemKind kind, size_t bytes, size_t* size, bool exact = false);
// Gives a block back.  No work that uses it may be pending: the callers synchronize first.
void mem_put(MemKind kind, void* p, size_t size);
// Frees every kept block.
void mem_release_kept();

}  // namespace gpq
