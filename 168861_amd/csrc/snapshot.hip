// Potentials of one neurite to host memory, in element order.
//
// A kernel gathers them (through the slot map of the tree solves' layouts) straight into
// pinned host memory and raises a flag there when the last block is done; the host polls
// the flag and copies to the caller. Before, a copy of the slots to pageable memory, a
// synchronisation and a loop over the elements on the host: 26 us (500 elements), 38 us
// (5,000), 997 us (902,037); here 11, 14 and 338 us. What is left is the launch, the write
// over the host link and the caller's own page faults.
#include <algorithm>
#include <atomic>
#include <chrono>
#include <cstring>
#include <mutex>
#include <vector>
#include "nrt_internal.hpp"

namespace nrt {

constexpr int kSnapChunk = 1 << 18;  // elements per staging buffer (2 MiB)
constexpr int kSnapBlock = 256;
constexpr int kSnapPer = 4;          // elements per thread
constexpr size_t kSnapKept = 4;      // staging sets kept for later calls (16 MiB of host memory)

__global__ __launch_bounds__(kSnapBlock) void k_snapshot(const double* __restrict__ x,
                                                         const int32_t* __restrict__ slot, int i0,
                                                         int n, double* __restrict__ host,
                                                         unsigned* count, unsigned* flag,
                                                         unsigned value) {
  const int b = blockIdx.x * (kSnapBlock * kSnapPer) + threadIdx.x;
#pragma unroll
  for (int k = 0; k < kSnapPer; k++) {
    const int i = b + k * kSnapBlock;
    if (i < n) host[i] = x[slot ? slot[i0 + i] : i0 + i];
  }
  __threadfence_system();
  __syncthreads();
  // the last block to come (the count wraps to 0 for the next launch) raises the flag
  if (threadIdx.x == 0 && atomicInc(count, gridDim.x - 1) == gridDim.x - 1)
    __hip_atomic_store(flag, value, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

namespace {
// Two staging buffers with their flags (pinned) and block counts (device).
struct Stage {
  int device = 0;
  double* host = nullptr;     // 2 x kSnapChunk, then the flags
  unsigned* flag = nullptr;   // [2]
  unsigned* count = nullptr;  // [2] device
  unsigned value[2] = {0, 0};
};
struct Stages {
  std::mutex mu;
  std::vector<Stage*> idle;
};
Stages& stages() {
  static Stages* s = new Stages;  // never destroyed: used until the process ends
  return *s;
}
void stage_free(Stage* s) {
  if (s->host) (void)hipHostFree(s->host);
  if (s->count) (void)hipFree(s->count);
  delete s;
}
Stage* stage_take(int device, hipStream_t stream) {
  Stages& all = stages();
  {
    std::lock_guard<std::mutex> g(all.mu);
    for (size_t i = 0; i < all.idle.size(); i++)
      if (all.idle[i]->device == device) {
        Stage* s = all.idle[i];
        all.idle.erase(all.idle.begin() + i);
        return s;
      }
  }
  auto* s = new Stage;
  s->device = device;
  try {
    NRT_HIP(hipHostMalloc((void**)&s->host, sizeof(double) * 2 * kSnapChunk + 64,
                          hipHostMallocDefault));
    s->flag = (unsigned*)(s->host + 2 * kSnapChunk);
    s->flag[0] = s->flag[1] = 0;
    NRT_HIP(hipMalloc((void**)&s->count, 2 * sizeof(unsigned)));
    NRT_HIP(hipMemsetAsync(s->count, 0, 2 * sizeof(unsigned), stream));
  } catch (...) {
    stage_free(s);
    throw;
  }
  return s;
}
// (a stage whose launches may not have ended is not kept: `whole` false)
void stage_give(Stage* s, bool whole) {
  Stages& all = stages();
  if (whole) {
    std::lock_guard<std::mutex> g(all.mu);
    if (all.idle.size() < kSnapKept) {
      all.idle.push_back(s);
      return;
    }
  }
  stage_free(s);
}
}  // namespace

// x (slot: null for element order) of n elements to `out`, after the work queued on s.
void snapshot_to_host(int device, const double* x, const int32_t* slot, int n, double* out,
                      hipStream_t s) {
  Stage* st = stage_take(device, s);
  bool whole = false;
  try {
    const int chunks = grid_for(n, kSnapChunk);
    auto start = [&](int c) {
      const int i0 = c * kSnapChunk, m = std::min(kSnapChunk, n - i0), b = c & 1;
      hipLaunchKernelGGL(k_snapshot, dim3(grid_for(m, kSnapBlock * kSnapPer)), dim3(kSnapBlock), 0,
                         s, x, slot, i0, m, st->host + (size_t)b * kSnapChunk, st->count + b,
                         st->flag + b, ++st->value[b]);
      NRT_HIP(hipGetLastError());
    };
    for (int c = 0; c < std::min(chunks, 2); c++) start(c);
    for (int c = 0; c < chunks; c++) {
      const int i0 = c * kSnapChunk, m = std::min(kSnapChunk, n - i0), b = c & 1;
      const auto* flag = (const std::atomic<unsigned>*)(st->flag + b);
      // poll for as long as a short wait lasts; a stream with more work ahead of the
      // gathering kernel (or an error) is waited for by the runtime
      const auto until = std::chrono::steady_clock::now() + std::chrono::microseconds(300);
      int polls = 0;
      while (flag->load(std::memory_order_acquire) != st->value[b]) {
        if ((++polls & 63) == 0 && std::chrono::steady_clock::now() > until) {
          NRT_HIP(hipStreamSynchronize(s));
          NRT_REQUIRE(flag->load(std::memory_order_acquire) == st->value[b], NRT_ERR_HIP,
                      "snapshot: the gathering kernel did not finish");
          break;
        }
      }
      memcpy(out + i0, st->host + (size_t)b * kSnapChunk, sizeof(double) * m);
      if (c + 2 < chunks) start(c + 2);
    }
    whole = true;
  } catch (...) {
    stage_give(st, whole);
    throw;
  }
  stage_give(st, whole);
}

}  // namespace nrt
