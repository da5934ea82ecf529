// Internal interface between the C-ABI layer (fattn_api.cpp) and the gfx950 kernels
// (fattn_pair.hip, fattn_kernels.hip), all compiled by hipcc.
#ifndef FATTN_INTERNAL_H
#define FATTN_INTERNAL_H

#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

namespace fattn {

// head_dim of the reference's kernels; the kernels here are built for 32, 64 and 128.
constexpr int kHeadDim = 64;
bool head_dim_supported(int64_t d);

// The units of the workspace's sizes (what callers plan with and saved plans hold), not of the
// kernels: key blocks of kBwdKeys, query tiles of kBwdQueryTile.
constexpr int kBwdKeys = 64;
#ifndef BWD_QT
#define BWD_QT 16
#endif
constexpr int kBwdQueryTile = BWD_QT;

// A [b, h, s, d] operand on the device: its first element and its (batch, head, seq) strides
// in floats, head_dim contiguous.
struct View {
  const float* p;
  int64_t sb, sh, ss;
};

// Workspace of the backward, in this order, each part 256-byte aligned:
//   ctrl   64 i32                           [32] guard word (first, so that its place does not
//                                           depend on the shape)
//   D      [b, h, s] f32                    (unused)
//   turn   [b, h, ntile] i32                (unused)
//   part   [nkb, b, h, ntile, kQT * d] f32  the first [b, h, ntile, kQT * d]: dQ left to step 3
//   arrive [b, h, nkb] u64                  (unused)
//   done   [b, h, ntile] u64                the epoch of the launch that wrote the tile's dQ rows
//   epoch  u64 (256 bytes)                  the epoch of the last step 2 launch on the workspace
// with ntile = ceil(s / kBwdQueryTile), nkb = ceil(s / kBwdKeys). The layout and its sizes are those
// of the ABI's size queries: `bytes_min` covers ctrl, D and turn, `bytes_split` all seven.
struct Workspace {
  size_t d_off, turn_off, ctrl_off, part_off, arrive_off, done_off, epoch_off, bytes_min,
      bytes_split;
};
Workspace workspace_layout(int64_t b, int64_t h, int64_t s, int64_t d);
constexpr int kCtrlGuard = 32;
// The schedule of dQ sums over key blocks, as the ABI's schedule queries describe it for a shape and
// a workspace (a plan over the units above). The kernels keep dQ in registers and sum nothing across
// workgroups; the queries keep their answers.
constexpr int kSumMaxBlocks = 256;
constexpr int kSumTiles = 3;  // query tiles per summing workgroup
// Causal: the query tiles whose last contributor is key block kb of `keys` keys (its diagonal
// tiles; keys / kBwdQueryTile of them, fewer at the end of the sequence).
__host__ __device__ inline void own_tiles(int kb, int keys, int ntile, int* j0, int* j1) {
  const int n = keys / kBwdQueryTile;
  *j0 = kb * n;
  *j1 = *j0 + n < ntile ? *j0 + n : ntile;
}

// Workgroups are dealt to the 8 XCDs round-robin (workgroup id % 8). xcd_remap gives each XCD a
// contiguous range of logical items, so logical neighbours (the key blocks of one (b, h)) share
// one L2: workgroup id runs item (id % 8) F + id / 8 with F = (total rounded down to a multiple
// of 8) / 8; the last total % 8 items run as themselves.
__host__ __device__ inline int xcd_remap(int id, int total) {
  const int full = total & ~7;
  if (id >= full) return id;
  return (id & 7) * (full >> 3) + (id >> 3);
}
// The XCD that runs logical item `item` of xcd_remap (its inverse, taken mod 8).
__host__ __device__ inline int item_xcd(int item, int total) {
  const int full = total & ~7;
  return item >= full ? (item & 7) : item / (full >> 3);
}

// The plan: non-causal, summing units after the key blocks of the grid; unit m < mc nchunk of XCD x
// takes chunk m % nchunk of the (m / nchunk)-th (b, h) whose last key block is among XCD x's, the
// units after those take, in (b, h) order, the (b, h)s whose last key block is among the rest.
// Causal: every key block sums the tiles it completes. on = 0: no sums (step 3 takes every tile).
struct SumPlan {
  int on;
  int nchunk;  // chunks of kSumTiles query tiles per (b, h)
  int nkb;     // key blocks per (b, h)
  int mc;      // (non-causal) the most (b, h)s one XCD's range holds
};
// The (b, h)s whose last key block lies in XCD x's range of key blocks: lo .. hi (empty if
// hi < lo); consecutive over x, from 0 to 8 F / nkb - 1.
__host__ __device__ inline int sum_range_lo(int x, int F, int nkb) {
  return (x * F + nkb) / nkb - 1;  // ceil((x F + 1) / nkb) - 1
}
__host__ __device__ inline int sum_range_hi(int x, int F, int nkb) { return (x + 1) * F / nkb - 1; }
__host__ __device__ inline SumPlan sum_plan(int BH, int nkb, int ntile, int d, int causal) {
  SumPlan p{0, (ntile + kSumTiles - 1) / kSumTiles, nkb, 0};
  if (nkb > kSumMaxBlocks || BH <= 0) return p;
  p.on = 1;
  if (!causal) {
    const int F = nkb * BH / 8;
    for (int x = 0; x < 8; ++x) {
      const int n = sum_range_hi(x, F, nkb) - sum_range_lo(x, F, nkb) + 1;
      p.mc = n > p.mc ? n : p.mc;
    }
  }
  return p;
}
// Units of the non-causal plan (a multiple of 8).
__host__ __device__ inline int sum_blocks(SumPlan p, int BH, int causal) {
  if (causal || !p.on) return 0;
  const int left = BH - 8 * (p.nkb * BH / 8) / p.nkb;
  return 8 * p.mc * p.nchunk + (left * p.nchunk + 7) / 8 * 8;
}
// Non-causal summing workgroup m of XCD x (workgroup n_main + 8 m + x): the (b, h) it sums and
// its first query tile. False for a workgroup with nothing to sum (past the plan or past b h),
// and always when causal (no summing workgroups).
__host__ __device__ inline bool sum_target(SumPlan p, int x, int m, int BH, int causal, int* bh,
                                           int* j0) {
  if (causal || !p.on) return false;
  const int F = p.nkb * BH / 8;
  if (m < p.mc * p.nchunk) {
    const int b0 = sum_range_lo(x, F, p.nkb) + m / p.nchunk;
    if (b0 > sum_range_hi(x, F, p.nkb) || b0 >= BH) return false;
    *bh = b0;
    *j0 = m % p.nchunk * kSumTiles;
    return true;
  }
  const int idx = (m - p.mc * p.nchunk) * 8 + x, left0 = 8 * F / p.nkb;
  if (idx >= (BH - left0) * p.nchunk) return false;
  *bh = left0 + idx / p.nchunk;
  *j0 = idx % p.nchunk * kSumTiles;
  return *bh < BH;
}
// Keys per key block of the plan: kBwdKeys, or twice that for large non-causal launches.
int bwd_split_keys(int64_t b, int64_t h, int64_t s, int d, int causal);
// Whether the plan has sums for this shape (and the hook has not turned them off).
bool bwd_step2_sums(int64_t b, int64_t h, int64_t s, int d, int causal);
// Units of the non-causal plan (0 when causal or without sums).
int64_t bwd_sum_blocks(int64_t b, int64_t h, int64_t s, int d, int causal);
// Test hooks (the C ABI lets a process use them only when it opted in at load). Off: step 2 leaves
// every dQ tile of a split-size workspace to step 3, in every later backward of the process; returns
// the previous setting (1, the default: on).
bool set_step2_sums(bool on);
// A setting of the plan's XCDs; kept and returned, the kernels do not read it.
int set_sum_shift(int shift);
// Step 2 gives up the dQ of (b, h) pair `bh` (of the whole backward; -1: none, the default) in every
// later launch: NaN and guard word 3 where no step 3 follows, else left to it; returns the previous
// pair.
int set_give_up_bh(int bh);
// What the hooks ask of a launch: dQ deferred to step 3 (step 2's sums off), the give-up pair.
bool step2_deferred();
int give_up_pair();
// The three hooks' current settings: step 2's sums on, the sum shift, the give-up pair.
void test_hook_state(int64_t out[3]);
// Launchers (step 3: fattn_kernels.hip, the others fattn_pair.hip). They assume validated arguments
// and return a hipError_t value as int (0 = launched).
int launch_forward(View q, View k, View v, float* o, float* lse, int b, int h, int s, int d,
                   float scale, int causal, void* stream);
// Backward, step 2 (fattn_pair.hip): dK, dV and dQ. part, done, epoch_slot (a split-size workspace,
// else null): with `defer` dQ goes to `part` for step 3, else to its rows, and `done` takes `epoch`
// per 16-query tile. last: no step 3 follows. give_up_bh: a test hook's pair (-1: none).
int launch_backward(View q, View k, View v, View d_o, const float* o, const float* lse, float* dqkv,
                    float* part, unsigned long long* done, unsigned long long* epoch_slot,
                    unsigned long long epoch, int* ctrl, int b, int h, int s, int d, float scale,
                    int causal, int defer, int last, int give_up_bh, void* stream);
// Step 3: dQ of every query tile that step 2 left in the workspace; the flags are zeroed.
int launch_bwd_dq(const float* part, unsigned long long* done, const unsigned long long* epoch_slot,
                  float* dqkv, int b, int h, int s, int d, float scale, void* stream);

// The device address of the library's static scratch (FATTN_STATIC_SCRATCH_BYTES, the workspace
// of fattn_bwd_f32_noalloc) on the device that runs `stream`; a hipError_t value as int.
int static_scratch(void* stream, void** out);

// Grid sizes the launchers will use (for range checks before launching).
int64_t bwd_main_blocks(int64_t b, int64_t h, int64_t s);
int64_t bwd_prep_blocks(int64_t b, int64_t h, int64_t s, int d);
int64_t bwd_dq_blocks(int64_t b, int64_t h, int64_t s);
}  // namespace fattn

#endif  // FATTN_INTERNAL_H
