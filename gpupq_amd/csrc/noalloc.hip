// noalloc.hip -- the record sort for callers that cannot allocate device memory (code under
// HIP graph capture, tight serving loops, harnesses that forbid hipMalloc).
//
// gpq_sort_events_noalloc sorts caller-owned device records with the same kernels as
// gpq_selftest_sort (one tile sort, then levels of up to 128-way merges), but its ping-pong
// partner buffer and its sample order live in `scratch`, a file-scope device array of
// kScratchBytes that every GPU the library runs on holds until the process ends.
// The array's address on the current device is looked up once per device with
// hipGetSymbolAddress and kept; host code only ever passes that address to kernels.
//
// Every call on one GPU shares that GPU's array, so calls that overlap on one GPU (on
// different streams, or from different host threads) race on it and must be serialised by
// the caller.  The array keeps the last call's contents; every word that a call reads it has
// written before, so nothing needs clearing.
#include <array>
#include <mutex>

#include "sortprim.h"

namespace gpq {
namespace {

constexpr uint32_t kNoAllocMaxRecords = 1u << 20;       // 16 MiB of partner buffer
constexpr size_t kOrderBytes = 128 * 1024 + 256;        // sample order: a word per 32 records and one more
constexpr size_t kScratchBytes = kOrderBytes + sizeof(Event) * (size_t)kNoAllocMaxRecords;
constexpr int kMaxDevices = 64;

static __device__ __align__(256) unsigned char scratch[kScratchBytes];

std::mutex g_scratch_mu;
std::array<unsigned char*, kMaxDevices> g_scratch_ptr{};   // per device, from hipGetSymbolAddress

// The current device's address of `scratch`, looked up on the first call on that device.
gpq_status scratch_on_current_device(unsigned char** out) {
  int dev = -1;
  GPQ_HIP(hipGetDevice(&dev));
  GPQ_CHECK_ARG(dev >= 0 && dev < kMaxDevices, "noalloc: device index out of range");
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    void* p = nullptr;
    GPQ_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    GPQ_CHECK_ARG(p != nullptr, "noalloc: no device address for the scratch array");
    g_scratch_ptr[dev] = static_cast<unsigned char*>(p);
  }
  *out = g_scratch_ptr[dev];
  return GPQ_OK;
}

}  // namespace
}  // namespace gpq

extern "C" gpq_status gpq_sort_events_noalloc(const gpq_event* d_in, uint32_t n, gpq_event* d_out, void* stream) {
  using gpq::Event;
  if (n == 0) return GPQ_OK;
  if (!d_in || !d_out) {
    gpq::set_error("sort_events_noalloc: null record pointer");
    return GPQ_ERR_INVALID;
  }
  if (n > gpq::kNoAllocMaxRecords) {
    gpq::set_error("sort_events_noalloc: " + std::to_string(n) + " records exceed the scratch limit of " +
                   std::to_string(gpq::kNoAllocMaxRecords));
    return GPQ_ERR_CAPACITY;
  }
  const uintptr_t in0 = reinterpret_cast<uintptr_t>(d_in), out0 = reinterpret_cast<uintptr_t>(d_out);
  const uintptr_t bytes = sizeof(Event) * (uintptr_t)n;
  if (in0 != out0 && in0 < out0 + bytes && out0 < in0 + bytes) {
    gpq::set_error("sort_events_noalloc: input and output overlap without being the same array");
    return GPQ_ERR_INVALID;
  }
  if ((in0 | out0) % alignof(Event) != 0) {
    gpq::set_error("sort_events_noalloc: records must be 16-byte aligned");
    return GPQ_ERR_INVALID;
  }
  unsigned char* base = nullptr;
  GPQ_TRY(gpq::scratch_on_current_device(&base));
  Event* partner = reinterpret_cast<Event*>(base + gpq::kOrderBytes);
  if (sizeof(uint32_t) * gpq::sort_order_words(n) > gpq::kOrderBytes) {
    gpq::set_error("sort_events_noalloc: sample order exceeds its scratch");
    return GPQ_ERR_STATE;
  }
  return gpq::sort_records(reinterpret_cast<const Event*>(d_in), reinterpret_cast<Event*>(d_out), partner,
                           reinterpret_cast<uint32_t*>(base), nullptr, n, static_cast<hipStream_t>(stream));
}
