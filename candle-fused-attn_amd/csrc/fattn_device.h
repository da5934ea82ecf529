// Device helpers shared by the kernel files (fattn_kernels.hip, fattn_pair.hip).
#ifndef FATTN_DEVICE_H
#define FATTN_DEVICE_H

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "fattn_internal.h"

namespace fattn {
namespace {

typedef float f4 __attribute__((ext_vector_type(4)));
// An int known at compile time, or not, behind the same call syntax.
template <int V>
struct Const {
  static constexpr int value = V;
  __device__ constexpr int operator()() const { return V; }
};
struct Var {
  int v;
  __device__ int operator()() const { return v; }
};

constexpr int kThreads = 256;  // 4 waves of 64
constexpr float kLog2e = 1.44269504088896340736f;
constexpr float kNegInf = -__builtin_inff();
// Forward lazy rescaling: a row's reference max moves only when a tile's max exceeds it by more
// than this many powers of two (unnormalised probabilities stay below 2^8).
constexpr float kRescaleLog2 = 8.0f;
// 2^x on the transcendental unit (v_exp_f32); 2^-inf = 0.
__device__ __forceinline__ float exp2_hw(float x) { return __builtin_amdgcn_exp2f(x); }
__device__ __forceinline__ f4 ld4(const float* p) { return *reinterpret_cast<const f4*>(p); }
__device__ __forceinline__ void st4(float* p, f4 v) { *reinterpret_cast<f4*>(p) = v; }
// Non-temporal store (nt): for outputs no kernel of the same pass reads again, so that they do not
// sit dirty in the L2s when the kernel ends (each XCD's L2 writes its dirty lines back then).
__device__ __forceinline__ void st4_nt(float* p, f4 v) {
  __builtin_nontemporal_store(v, reinterpret_cast<f4*>(p));
}
__device__ __forceinline__ f4 zero4() { return f4{0.0f, 0.0f, 0.0f, 0.0f}; }
// A lane of x through a DPP lane permutation (VALU, no LDS round trip).
template <int CTRL>
__device__ __forceinline__ float dpp(float x) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), CTRL, 0xF, 0xF, false));
}
// Sum over each aligned group of N = 8, 16 or 32 lanes, every lane of the group getting the same
// bits (each step adds a lane and its partner, and x + y == y + x): partner = lane ^ 1
// (quad_perm 1,0,3,2), lane ^ 2 (quad_perm 2,3,0,1), the other quad of the 8 (row_half_mirror),
// the other 8 of the 16 (row_mirror), the other 16 of the 32 (row swap).
template <int N>
__device__ __forceinline__ float lane_sum(float x) {
  static_assert(N == 8 || N == 16 || N == 32, "groups of 8, 16 or 32 lanes");
  x += dpp<0xB1>(x);
  x += dpp<0x4E>(x);
  x += dpp<0x141>(x);
  if constexpr (N >= 16) x += dpp<0x140>(x);
  if constexpr (N == 32) {
    const unsigned u = __float_as_uint(x);
    const auto p = __builtin_amdgcn_permlane16_swap(u, u, false, false);
    x = __uint_as_float(p[0]) + __uint_as_float(p[1]);
  }
  return x;
}

// max of two floats as one v_max_f32: fmaxf on values from a lane swap makes the compiler quiet
// both inputs first (two more v_max per call, 8 per forward tile), which NaN-free scores do not
// need.
__device__ __forceinline__ float vmax(float a, float b) {
  float r;
  asm("v_max_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
  return r;
}
// v_permlane16_swap / v_permlane32_swap on a pair of floats (16-lane rows: the first swaps odd
// rows of a with even rows of b, the second the upper 32 lanes of a with the lower 32 of b).
__device__ __forceinline__ void swap_rows16(float& a, float& b) {
  const auto p = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false,
                                                  false);
  a = __uint_as_float(p[0]);
  b = __uint_as_float(p[1]);
}
__device__ __forceinline__ void swap_rows32(float& a, float& b) {
  const auto p = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false,
                                                  false);
  a = __uint_as_float(p[0]);
  b = __uint_as_float(p[1]);
}
// s_waitcnt with vmcnt(n) and no lgkm / export wait (gfx9 encoding: vmcnt bits 3:0 and 15:14,
// expcnt 6:4, lgkmcnt 11:8). Issued through the builtin, not inline asm, so that the compiler
// knows which of its own loads have completed: otherwise it adds waits of its own at their first
// uses -- inside the loops, where they would also wait for the prefetch copies in flight. The
// empty asm keeps memory accesses from moving across the wait.
template <int N>
__device__ __forceinline__ void wait_vm() {
  static_assert(N >= 0 && N < 64, "vmcnt 0..63");
  __builtin_amdgcn_s_waitcnt(0x0F70 | (N & 15) | ((N >> 4) << 14));
  asm volatile("" ::: "memory");
}
// Waits until every vector memory operation of this wave has completed (loads returned, stores
// and direct copies landed).
__device__ __forceinline__ void wait_mem() { wait_vm<0>(); }

// Wave priority from the work left: 3 while more than three quarters of the walk remain, down to
// 0 for the last quarter. A SIMD otherwise issues from its oldest wave first, so the first of a
// CU's workgroups finishes well before the last, which then runs alone; with the priority falling
// as a wave progresses, co-resident waves progress together and end together.
__device__ __forceinline__ void prio_by_remaining(int rem, int total) {
  const int q = (4 * rem) / max(total, 1);
  if (q >= 3) {
    __builtin_amdgcn_s_setprio(3);
  } else if (q == 2) {
    __builtin_amdgcn_s_setprio(2);
  } else if (q == 1) {
    __builtin_amdgcn_s_setprio(1);
  } else {
    __builtin_amdgcn_s_setprio(0);
  }
}

struct FwdArgs {
  View q, k, v;
  float* o;
  float* lse;
  int B, H, S, nqb;
  float scale;
  int causal;
};

}  // namespace
}  // namespace fattn

#endif  // FATTN_DEVICE_H
