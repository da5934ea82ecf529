// The backward's step 3, the library's static scratch, and the host's shape functions (the workspace
// and schedule rules of the C ABI). The forward and step 2 are in fattn_pair.hip.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <mutex>
#include <stddef.h>
#include <stdint.h>

#include "fattn.h"
#include "fattn_device.h"
#include "fattn_internal.h"

// The backward workspace of fattn_bwd_f32_noalloc, for callers that cannot allocate: device memory
// of this library, one copy per GPU (each at its own address), held until the process ends. In
// host code the name is only a host-side handle: the device address comes from
// hipGetSymbolAddress (fattn::static_scratch below), never from the name itself.
static __device__ __align__(256) unsigned char scratch[FATTN_STATIC_SCRATCH_BYTES];

namespace fattn {
namespace {

constexpr int kQT = kBwdQueryTile;

// Backward, step 3: every 16-query tile whose done flag does not hold the epoch of the step 2 launch
// recorded in the workspace left its dQ there, unscaled ([tile][16][D]); times scale it goes to its
// rows. The flags are zeroed after use. Normally every flag is set and this only reads them.
template <int D>
__global__ void __launch_bounds__(kThreads) dq_kernel(const float* __restrict__ part,
                                                     unsigned long long* __restrict__ done,
                                                     const unsigned long long* __restrict__ epoch,
                                                     float* __restrict__ dqkv, int BH, int H, int S,
                                                     int ntile, float scale) {
  const int tid = threadIdx.x, tot = BH * ntile;
  const unsigned long long now = *epoch;
  for (int it = static_cast<int>(blockIdx.x); it < tot; it += static_cast<int>(gridDim.x)) {
    const bool written = done[it] == now;
    __syncthreads();  // every thread has read the flag
    if (tid == 0) done[it] = 0ull;
    if (written) continue;
    const int bh = it / ntile, b = bh / H, h = bh % H, q0 = it % ntile * kQT;
    const float* src = part + static_cast<int64_t>(it) * (kQT * D);
    for (int i = tid; i < kQT * D / 4; i += kThreads) {
      const int row = i / (D / 4), c = 4 * (i % (D / 4));
      if (q0 + row < S) {
        st4(dqkv + (static_cast<int64_t>(b) * S + q0 + row) * 3 * H * D +
                static_cast<int64_t>(h) * D + c,
            ld4(src + row * D + c) * scale);
      }
    }
  }
}

}  // namespace

bool head_dim_supported(int64_t d) { return d == 32 || d == 64 || d == 128; }

int64_t bwd_main_blocks(int64_t b, int64_t h, int64_t s) {
  return ((s + kBwdKeys - 1) / kBwdKeys) * h * b;
}
// (Step 1's grid when it had one; part of the range that calls are held to.)
int64_t bwd_prep_blocks(int64_t b, int64_t h, int64_t s, int d) {
  const int64_t rows_per_block = kThreads / (d / 4);
  return (b * h * s + rows_per_block - 1) / rows_per_block;
}
int64_t bwd_dq_blocks(int64_t b, int64_t h, int64_t s) { return b * h * ((s + kQT - 1) / kQT); }
namespace {
std::atomic<int> g_step2_sums{1};
std::atomic<int> g_sum_shift{0};
std::atomic<int> g_give_up_bh{-1};
}  // namespace
bool set_step2_sums(bool on) { return g_step2_sums.exchange(on ? 1 : 0) != 0; }
int set_sum_shift(int shift) { return g_sum_shift.exchange(shift & 7); }
int set_give_up_bh(int bh) { return g_give_up_bh.exchange(bh < 0 ? -1 : bh); }
bool step2_deferred() { return g_step2_sums.load(std::memory_order_relaxed) == 0; }
int give_up_pair() { return g_give_up_bh.load(std::memory_order_relaxed); }
void test_hook_state(int64_t out[3]) {
  out[0] = g_step2_sums.load(std::memory_order_relaxed);
  out[1] = g_sum_shift.load(std::memory_order_relaxed);
  out[2] = g_give_up_bh.load(std::memory_order_relaxed);
}

int bwd_split_keys(int64_t b, int64_t h, int64_t s, int d, int causal) {
  // (The rule of the size queries: 128-key blocks for non-causal launches that fill the chip with
  // them. The kernels' own blocks are 128 rows at every shape.)
  const int64_t blocks128 = (s + 2 * kBwdKeys - 1) / (2 * kBwdKeys) * b * h;
  if (causal) return kBwdKeys;
  if (d == 32) return blocks128 >= 1536 ? 2 * kBwdKeys : kBwdKeys;
  if (d != 64 || s < 512) return kBwdKeys;
  return blocks128 >= 512 ? 2 * kBwdKeys : kBwdKeys;
}
namespace {
// The plan of nbh (b, h) pairs with key blocks of `keys` keys.
bool step2_sums_of(int64_t nbh, int64_t s, int d, int causal, int keys) {
  if (g_step2_sums.load(std::memory_order_relaxed) == 0) return false;
  // The range check keeps b h s (hence every count below) inside int32.
  const int nkb = static_cast<int>((s + keys - 1) / keys);
  const int ntile = static_cast<int>((s + kQT - 1) / kQT);
  return sum_plan(static_cast<int>(nbh), nkb, ntile, d, causal).on != 0;
}
int64_t sum_blocks_of(int64_t nbh, int64_t s, int d, int causal, int keys) {
  if (causal || !step2_sums_of(nbh, s, d, causal, keys)) return 0;
  const int nkb = static_cast<int>((s + keys - 1) / keys);
  const int ntile = static_cast<int>((s + kQT - 1) / kQT);
  const SumPlan p = sum_plan(static_cast<int>(nbh), nkb, ntile, d, causal);
  return sum_blocks(p, static_cast<int>(nbh), causal);
}
}  // namespace
bool bwd_step2_sums(int64_t b, int64_t h, int64_t s, int d, int causal) {
  return step2_sums_of(b * h, s, d, causal, bwd_split_keys(b, h, s, d, causal));
}
int64_t bwd_sum_blocks(int64_t b, int64_t h, int64_t s, int d, int causal) {
  return sum_blocks_of(b * h, s, d, causal, bwd_split_keys(b, h, s, d, causal));
}

// The device address of `scratch` on the device that runs `stream` (the null stream: the current
// device), looked up with hipGetSymbolAddress once per device, with that device current, and kept.
int static_scratch(void* stream, void** out) {
  constexpr int kMaxDevices = 64;
  static std::atomic<void*> addr[kMaxDevices];
  static std::mutex mu;
  int dev = 0;
  hipError_t e = stream ? hipStreamGetDevice(static_cast<hipStream_t>(stream), &dev)
                        : hipGetDevice(&dev);
  if (e != hipSuccess) return static_cast<int>(e);
  if (dev < 0 || dev >= kMaxDevices) return static_cast<int>(hipErrorInvalidDevice);
  void* p = addr[dev].load(std::memory_order_acquire);
  if (p == nullptr) {
    std::lock_guard<std::mutex> lock(mu);
    p = addr[dev].load(std::memory_order_relaxed);
    if (p == nullptr) {
      int cur = 0;
      if ((e = hipGetDevice(&cur)) != hipSuccess) return static_cast<int>(e);
      if (cur != dev && (e = hipSetDevice(dev)) != hipSuccess) return static_cast<int>(e);
      e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
      if (cur != dev) {
        const hipError_t e2 = hipSetDevice(cur);
        if (e == hipSuccess) e = e2;
      }
      if (e != hipSuccess) return static_cast<int>(e);
      if (p == nullptr) return static_cast<int>(hipErrorInvalidSymbol);
      addr[dev].store(p, std::memory_order_release);
    }
  }
  *out = p;
  return 0;
}

int launch_bwd_dq(const float* part, unsigned long long* done, const unsigned long long* epoch_slot,
                  float* dqkv, int b, int h, int s, int d, float scale, void* stream) {
  int bh = b * h, ntile = (s + kQT - 1) / kQT;
  void* args[] = {&part, &done, &epoch_slot, &dqkv, &bh, &h, &s, &ntile, &scale};
  const void* fn = d == 32    ? reinterpret_cast<const void*>(dq_kernel<32>)
                   : d == 128 ? reinterpret_cast<const void*>(dq_kernel<128>)
                              : reinterpret_cast<const void*>(dq_kernel<64>);
  const int64_t blocks = std::min<int64_t>(bwd_dq_blocks(b, h, s), 1024);
  return static_cast<int>(hipLaunchKernel(fn, dim3(static_cast<unsigned>(blocks)), dim3(kThreads),
                                          args, 0, static_cast<hipStream_t>(stream)));
}

}  // namespace fattn
