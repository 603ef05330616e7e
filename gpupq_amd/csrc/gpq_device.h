// gpq_device.h -- the public device vocabulary (include/gpupq_device/core.cuh) plus the
// helpers only the library's own kernels use: the block-wide window minimum and the
// kernel that publishes it.
#pragma once

#include "../../include/gpupq_device/core.cuh"

namespace gpq {

// Block-wide min of one value per thread, written to partial[blockIdx.x].  No fence:
// a device-scope fence on gfx950 writes back the XCD's L2 (buffer_wbl2), far too
// costly per block; the partials are folded by window_publish_kernel, launched
// after the producing kernel on the same stream.  blockDim.x: multiple of 64, <= 1024.
__device__ __forceinline__ void block_min_to_partial(uint32_t v, uint32_t* partial) {
  __shared__ uint32_t s_wmin[16];
  v = wave_min_u32(v);
  if (lane_id() == 0) s_wmin[threadIdx.x / kWave] = v;
  __syncthreads();
  if (threadIdx.x == 0) {
    uint32_t m = s_wmin[0];
    for (int i = 1; i < (int)(blockDim.x / kWave); ++i) m = s_wmin[i] < m ? s_wmin[i] : m;
    partial[blockIdx.x] = m;
  }
}

// What a post kernel needs to publish the window by itself.  `fold`: the minimum so far, kInfBits between
// launches, and the blocks that have added to it, 0 between launches; null when a launch follows that
// folds the partials.  A search over the queue also has its end decided here (best .. steps; null without).
struct WindowPublish {
  uint32_t* fold;
  WindowState* ws;
  float lookahead, horizon;
  const uint32_t* best;
  uint32_t* search_done;
  unsigned long long* steps;
};

__device__ __forceinline__ void publish_window_at(const WindowPublish& w, uint32_t g) {
  float wend = bits_to_f(g) + w.lookahead;   // inf + lookahead stays inf
  if (w.horizon < wend) wend = w.horizon;
  w.ws->gmin = g;
  w.ws->wend = f_to_bits(wend);
  w.ws->done = (g == kInfBits || !(bits_to_f(g) < w.horizon)) ? 1u : 0u;
  w.ws->windows += 1;
  if (w.best) {                              // every list empty, or no f below the best goal cost
    *w.search_done = (g == kInfBits || (*w.best != 0xFFFFFFFFu && *w.best <= g)) ? 1u : 0u;
    *w.steps += 1;
  }
}

// block_min_to_partial, and with w.fold the window published by the block that comes last: the minima
// and the count are atomics, which are performed at memory and so need no fence.
__device__ __forceinline__ void block_min_publish(uint32_t v, uint32_t* partial, const WindowPublish& w) {
  __shared__ uint32_t s_wmin[16];
  v = wave_min_u32(v);
  if (lane_id() == 0) s_wmin[threadIdx.x / kWave] = v;
  __syncthreads();
  if (threadIdx.x != 0) return;
  uint32_t m = s_wmin[0];
  for (int i = 1; i < (int)(blockDim.x / kWave); ++i) m = s_wmin[i] < m ? s_wmin[i] : m;
  if (!w.fold) {
    partial[blockIdx.x] = m;
    return;
  }
  uint32_t before = atomicMin(&w.fold[0], m);
  asm volatile("s_waitcnt vmcnt(0)" : "+v"(before) : : "memory");   // done before this block is counted
  if (atomicAdd(&w.fold[1], 1u) != gridDim.x - 1u) return;
  w.fold[1] = 0;
  publish_window_at(w, atomicExch(&w.fold[0], kInfBits));
}

// A thread's inserts into the staging of LPs, each one's slot on its way while the thread works on the
// next event: the record is stored when the next slot has been asked for, and by flush().
struct StagedInserts {
  Event e;
  uint32_t pos;
  bool any = false;
  __device__ __forceinline__ void put(Event* stage, uint32_t* ins, uint32_t stage_cap, WindowState* ws, const Event& x) {
    const uint32_t p = atomicAdd(&ins[x.dst], 1u);
    flush(stage, stage_cap, ws);
    e = x;
    pos = p;
    any = true;
  }
  __device__ __forceinline__ void flush(Event* stage, uint32_t stage_cap, WindowState* ws) {
    if (!any) return;
    if (pos < stage_cap) store_event(&stage[(size_t)e.dst * stage_cap + pos], e);
    else atomicOr(&ws->error, kErrStageOverflow);
    any = false;
  }
};

// One block: folds the per-block minima and publishes gmin, the window end
// min(gmin + lookahead, horizon) and the done flag.
__global__ void window_publish_kernel(const uint32_t* partial, uint32_t count, WindowState* ws, float lookahead,
                                      float horizon);

}  // namespace gpq
