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

constexpr int kThreads = 256;  // 4 waves of 64
constexpr float kLog2e = 1.44269504088896340736f;
constexpr float kNegInf = -__builtin_inff();
// 2^x on the transcendental unit (v_exp_f32); 2^-inf = 0.
__device__ __forceinline__ float exp2_hw(float x) { return __builtin_amdgcn_exp2f(x); }
__device__ __forceinline__ f4 ld4(const float* p) { return *reinterpret_cast<const f4*>(p); }
__device__ __forceinline__ void st4(float* p, f4 v) { *reinterpret_cast<f4*>(p) = v; }
// Non-temporal store (nt): for outputs no kernel of the same pass reads again, so that they do not
// sit dirty in the L2s when the kernel ends (each XCD's L2 writes its dirty lines back then).
__device__ __forceinline__ void st4_nt(float* p, f4 v) {
  __builtin_nontemporal_store(v, reinterpret_cast<f4*>(p));
}
// A lane of x through a DPP lane permutation (VALU, no LDS round trip).
template <int CTRL>
__device__ __forceinline__ float dpp(float x) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), CTRL, 0xF, 0xF, false));
}
// max of two floats as one v_max_f32: fmaxf on values from a lane swap makes the compiler quiet
// both inputs first (two more v_max per call, 8 per forward tile), which NaN-free scores do not
// need.
__device__ __forceinline__ float vmax(float a, float b) {
  float r;
  asm("v_max_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
  return r;
}

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
