// fp32 attention on the f16 matrix cores. Every fp32 operand, times a power of two, is held as the
// sum of two f16 terms, x 2^k = h + l (h rounded to nearest, l the rest rounded to nearest: 22 bits
// and the sign of l), and a product is accumulated in fp32 as three f16 products,
//   h l' + l h' + h h'
// (l l' is below 2^-22 of the product with a random sign, as is what l drops).
//
// Why: v_mfma_f32_32x32x16_f16 runs at 16 times the rate of the fp32 v_mfma_f32_16x16x4_f32
// (measured on MI355X, 4 waves per SIMD: 2.27 PFLOP/s against 151 TFLOP/s), so three of them take
// a fifth of the time, and unlike the fp32 one they run beside the VALU (six VALU instructions per
// MFMA are free with two waves per SIMD; beside the fp32 MFMA each adds its whole issue time). The
// sums are no less accurate, since one rounding covers 16 contracted values instead of 4: N(0, 1)
// dot products against fp64, normwise, 32 / 64 / 128 terms: 8.8e-8 / 9.5e-8 / 1.08e-7, the fp32
// instruction 1.02e-7 / 1.44e-7 / 2.03e-7. (Three bf16 terms with six products hold all 24 bits,
// 4.6e-8 at 64 terms, but twice the products run into the power limit: the clock fell to 1.82 GHz
// where the fp32 kernel holds 2.41, and the forward at b 16 h 16 s 1024 took 352 us against 524.)
//
// Scales. f16 spans 2^-14 .. 2^16 (normal), so every row of an operand carries its own exact power
// of two, from the largest magnitude in it: that is stored in [2^kTop, 2^(kTop + 1)), and an element
// keeps its 22 bits down to 2^-17 of its row's largest (below, an absolute error of 2^-39 of it). A
// wave's own rows hold theirs in a register; a staged row's is in LDS beside the tile (`unit`, 2^e)
// and multiplies back per accumulator row: into the scores' factor, and, where the product sums over
// the staged rows, into the weights (P, dS). The weights of a lane's own row follow a power of two
// of their own, which puts the largest term of the sum at 2^6 or more: 22 bits down to 2^-9 of it,
// below that an error of 2^-31 of it, and none that depends on a row that has no part in the sum. (One
// scale serves all D columns of it: where the heavy rows are exactly 0 in a column, the light ones' sum
// there has the error too.)
// One scale per tile, or the largest so far, costs less: forward b64 h6 s240 28.9 us against 30.3, b16
// h16 s1024 200 against 220, with inputs of deviation 2, whose weights move the scales more often, 203
// against 242; backward 92 against 94 and 792 against 808, d 128 228 against 235. But one large row,
// masked or not, or one key of large weight, takes the bits of all the others.
//
// For one v_mfma_f32_32x32x16_f16, lane l (j = l % 32, g = l / 32) supplies A[j][8 g + e] and
// B[8 g + e][j], e = 0..7, and holds D[8 (r / 4) + 4 g + r % 4][j], r = 0..15. As the contraction
// order is free (A and B alike), eight consecutive accumulator registers of one product are the B
// operand of the next one over 16 of its rows: step ks, element e is row
//   16 ks + 4 g + e (e < 4),  16 ks + 8 + 4 g + e - 4 (e >= 4).
// A operands are read from LDS, where a tile of 32 rows is held as two f16 planes [32][D]: by rows
// (ds_read_b128: 8 columns of row j), or transposed (two ds_read_b64_tr_b16: 4 + 4 rows of column
// j, in the order above). 16-byte chunk c of row r sits at chunk c ^ chunk_swz(r).
//
// Values the split cannot carry (infinities, NaN) show as a non-finite result; a wave that finds
// one computes its 32 rows again on the fp32 matrix instruction.
#include <hip/hip_runtime.h>
#include <math.h>
#include <stddef.h>
#include <stdint.h>

#include "fattn_device.h"
#include "fattn_internal.h"

namespace fattn {
namespace {

typedef float f16v __attribute__((ext_vector_type(16)));
typedef float f2 __attribute__((ext_vector_type(2)));
typedef _Float16 h2 __attribute__((ext_vector_type(2)));
typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef unsigned u4 __attribute__((ext_vector_type(4)));
typedef short s4 __attribute__((ext_vector_type(4)));

constexpr int kRows = 32;  // rows of a staged tile, and of a wave's own operand
constexpr int kTop = 13;   // the scaled maximum lies in [2^kTop, 2^(kTop + 1))

__device__ __forceinline__ f16v mma(h8 a, h8 b, f16v c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ f16v zero16() { return f16v{}; }

// 2^e, -126 <= e <= 127.
__device__ __forceinline__ float pow2(int e) { return __int_as_float((e + 127) << 23); }
// The exponent of a magnitude, within [kMinExp, kMaxExp] (0, subnormals, infinities): every 2^e,
// 2^-e and 2^(kTop - e) is a normal float, and the smallest normal one is still scaled to 1.
constexpr int kMinExp = kTop - 126, kMaxExp = 126;
__device__ __forceinline__ int exponent(float x) {
  return min(max(static_cast<int>(__float_as_uint(x) >> 23) - 127, kMinExp), kMaxExp);
}

// Eight values times a scale, in two terms.
struct Pair {
  h8 h, l;
};
__device__ __forceinline__ Pair make_pair8(const unsigned* h, const unsigned* l) {
  return Pair{__builtin_bit_cast(h8, u4{h[0], h[1], h[2], h[3]}),
              __builtin_bit_cast(h8, u4{l[0], l[1], l[2], l[3]})};
}
// x sc = h + l, two values: four instructions (v_fma_mixlo / mixhi_f16 scale, subtract and round in
// one). The empty asm makes the compiler take l's subtrahend from the packed h instead of
// converting each value a second time.
__device__ __forceinline__ void split2(float x, float y, float sc, unsigned& h, unsigned& l) {
  const h2 a{static_cast<_Float16>(fmaf(x, sc, 0.0f)), static_cast<_Float16>(fmaf(y, sc, 0.0f))};
  h = __builtin_bit_cast(unsigned, a);
  asm("" : "+v"(h));
  const h2 b = __builtin_bit_cast(h2, h);
  const h2 c{static_cast<_Float16>(fmaf(x, sc, -static_cast<float>(b.x))),
             static_cast<_Float16>(fmaf(y, sc, -static_cast<float>(b.y)))};
  l = __builtin_bit_cast(unsigned, c);
}
__device__ __forceinline__ Pair split8(f4 x, f4 y, float sc) {
  unsigned h[4], l[4];
  split2(x[0], x[1], sc, h[0], l[0]);
  split2(x[2], x[3], sc, h[1], l[1]);
  split2(y[0], y[1], sc, h[2], l[2]);
  split2(y[2], y[3], sc, h[3], l[3]);
  return make_pair8(h, l);
}
// Registers 8 KS .. 8 KS + 7 of an accumulator, times a scale, as a B operand.
template <int KS>
__device__ __forceinline__ Pair split_acc(const f16v& x, float sc) {
  unsigned h[4], l[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) split2(x[8 * KS + 2 * i], x[8 * KS + 2 * i + 1], sc, h[i], l[i]);
  return make_pair8(h, l);
}
__device__ __forceinline__ f16v mma_small(const Pair& a, const Pair& b, f16v c) {
  c = mma(a.h, b.l, c);
  return mma(a.l, b.h, c);
}
__device__ __forceinline__ f16v mma3(const Pair& a, const Pair& b, f16v c) {
  return mma(a.h, b.h, mma_small(a, b, c));
}

// --- LDS tiles ---------------------------------------------------------------------------------
// The 16-byte chunk a row's chunk 0 moves to, linear over xor in the row's low four bits: the maps
// that took the fewest cycles over all of them, measured for the two read patterns and the staging
// writes together (128 of each by four waves, D 64: row reads 5276 cycles, transposed 3648, writes
// 6636; bit-reversed low three bits: 6020, 4000, 6684).
template <int D>
constexpr int kSwz8 = D == 32 ? 3 : D == 64 ? 1 : 7;  // of row 8
template <int D>
__device__ __forceinline__ int chunk_swz(int row) {
  constexpr int f1 = D == 32 ? 1 : D == 64 ? 2 : 11, f2 = D == 32 ? 0 : D == 64 ? 5 : 15;
  constexpr int f4 = D == 32 ? 2 : D == 64 ? 6 : 10;
  return ((row & 1) ? f1 : 0) ^ ((row & 2) ? f2 : 0) ^ ((row & 4) ? f4 : 0) ^
         ((row & 8) ? kSwz8<D> : 0);
}
template <int D>
struct Tile {
  _Float16 p[2][kRows * D];  // planes h, l
};
template <int D>
constexpr int kPlane = kRows * D * 2;  // bytes

// Row j = lane % 32's columns 8 g .. + 7; those of step ks, 16 ks on, at this ^ row_step(ks).
template <int D>
__device__ __forceinline__ int row_off(int j, int g) {
  return j * (2 * D) + ((g ^ chunk_swz<D>(j)) << 4);
}
__device__ constexpr int row_step(int ks) { return ks << 5; }
template <int D>
__device__ __forceinline__ Pair ld_row(const Tile<D>& t, int off) {
  const char* p = reinterpret_cast<const char*>(&t) + off;
  return Pair{*reinterpret_cast<const h8*>(p), *reinterpret_cast<const h8*>(p + kPlane<D>)};
}
// The lane's base offset of the transposed read of columns lane % 32 (32 dt + those at this ^
// col_step(dt)): within each group of 16 lanes, lane i points at row i / 4 and columns 4 (i % 4) .. + 3
// of a 4 x 16 block and receives the block's column i. Rows 16 ks + 4 g + (0..3) at + 32 D ks bytes; 8 rows on, + 16 D bytes and
// the chunk of the offset changed by kSwz8.
template <int D>
__device__ __forceinline__ int col_off(int lane) {
  const int i = lane & 15, hi = (lane >> 4) & 1, g = lane >> 5;
  const int row = 4 * g + (i >> 2);
  const int chunk = 2 * hi + ((i & 3) >> 1);
  return row * (2 * D) + ((chunk ^ chunk_swz<D>(row)) << 4) + ((i & 1) << 3);
}
__device__ constexpr int col_step(int dt) { return dt << 6; }
template <int D>
__device__ __forceinline__ h8 ld_tr(const char* t, int off) {
  typedef __attribute__((address_space(3))) s4 lds_s4;
  const s4 a = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4*)(t + off));
  const s4 b = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
      (lds_s4*)(t + 16 * D + (off ^ (kSwz8<D> << 4))));
  return __builtin_bit_cast(h8, __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7));
}
template <int D>
__device__ __forceinline__ Pair ld_col(const Tile<D>& t, int off, int ks) {
  const char* p = reinterpret_cast<const char*>(&t) + 32 * D * ks;
  return Pair{ld_tr<D>(p, off), ld_tr<D>(p + kPlane<D>, off)};
}

// --- Lane exchanges ----------------------------------------------------------------------------
// The sum over a lane and lane ^ 32 (both get the same bits), and the max.
__device__ __forceinline__ float pair_sum(float x) {
  const unsigned u = __float_as_uint(x);
  const auto p = __builtin_amdgcn_permlane32_swap(u, u, false, false);
  return __uint_as_float(p[0]) + __uint_as_float(p[1]);
}
__device__ __forceinline__ float pair_max(float x) {
  const unsigned u = __float_as_uint(x);
  const auto p = __builtin_amdgcn_permlane32_swap(u, u, false, false);
  return vmax(__uint_as_float(p[0]), __uint_as_float(p[1]));
}
// The max of magnitudes over each aligned group of N lanes (4, 8 or 16), as integers: one
// instruction per step, where fmaxf quiets its inputs first.
template <int CTRL>
__device__ __forceinline__ unsigned max_dpp(unsigned x) {
  return max(x, static_cast<unsigned>(__builtin_amdgcn_update_dpp(0, static_cast<int>(x), CTRL, 0xF,
                                                                  0xF, true)));
}
template <int N>
__device__ __forceinline__ float group_max(float m) {
  // (The mask is an instruction between an asm's result and the lane move that reads it: the compiler
  // counts that wait from the instructions it knows.)
  unsigned x = __float_as_uint(m) & 0x7fffffffu;
  x = max_dpp<0xB1>(x);
  x = max_dpp<0x4E>(x);
  if constexpr (N >= 8) x = max_dpp<0x141>(x);
  if constexpr (N >= 16) x = max_dpp<0x140>(x);
  return __uint_as_float(x);
}
// max(m, |x|, |y|) over eight values: four v_max3_f32 with absolute operands (from fmaxf the
// compiler makes eight and quiets every input first). For loaded values; NaN is passed over.
__device__ __forceinline__ float abs_max8(f4 x, f4 y, float m) {
#pragma unroll
  for (int i = 0; i < 4; ++i) asm("v_max3_f32 %0, |%1|, |%2|, %0" : "+v"(m) : "v"(x[i]), "v"(y[i]));
  return m;
}
// No memory access moves across: a step's loads are issued before its LDS reads (left to itself the
// compiler sinks them to their first use, at the end of the step).
__device__ __forceinline__ void pin_loads() { asm volatile("" ::: "memory"); }
// x, as the compiler finds it here: what is formed from it (a walk's offsets in each step, the
// addresses used after it) is not formed earlier and held in registers, or memory, until then.
__device__ __forceinline__ int late(int x) {
  asm volatile("" : "+v"(x));
  return x;
}
// 0 where every value is finite, else NaN.
template <int N>
__device__ __forceinline__ float probe_finite(const f16v (&x)[N], float z) {
#pragma unroll
  for (int i = 0; i < N; ++i) {
#pragma unroll
    for (int r = 0; r < 16; ++r) z = fmaf(x[i][r], 0.0f, z);
  }
  return z;
}

// --- Staging -----------------------------------------------------------------------------------
// Two operands' tiles of 32 rows through the registers of a workgroup of W waves: wave w takes rows
// 32 / W w .. of both (D 32 with four waves: operand a in lanes 0..31, b in the others), eight
// columns per lane and access. A tile is loaded in one step of the walk; the next step takes each row's largest
// magnitude (over the lanes that hold the row), scales, splits and stores it.
struct Operand {
  const char* p;  // row 0 of the (b, h)
  unsigned ss4;   // row stride in bytes
};
template <int D, int W>
struct Stage {
  static constexpr int kC = D / 8;             // chunks per row
  static constexpr int kWaveRows = kRows / W;
  static constexpr bool kHalves = kWaveRows * kC == 32;  // one access holds both operands
  static constexpr int kPer = kHalves ? 1 : kWaveRows * kC / 64;  // accesses per lane and operand
  static constexpr int kN = kHalves ? 1 : 2 * kPer;               // in all: a's, then b's
  f4 x[kN][2];
  int e[kN];  // the access's row's exponent (after store)

  static __device__ __forceinline__ int row(int i, int w, int lane) {
    if constexpr (kHalves) return kWaveRows * w + (lane & 31) / kC;
    return kWaveRows * w + (64 / kC) * (i % kPer) + lane / kC;
  }
  // Rows past `last` repeat it (finite where the operand is; masked by the reader).
  __device__ __forceinline__ void load(const Operand& a, const Operand& b, int r0, int last, int w,
                                       int lane) {
#pragma unroll
    for (int i = 0; i < kN; ++i) {
      const bool is_b = kHalves ? lane >= 32 : i >= kPer;
      const unsigned r = static_cast<unsigned>(min(r0 + row(i, w, lane), last));
      const char* p = is_b ? b.p : a.p;
      const unsigned off =
          r * (is_b ? b.ss4 : a.ss4) + 32u * static_cast<unsigned>(lane % kC);
      x[i][0] = *reinterpret_cast<const f4*>(p + off);
      x[i][1] = *reinterpret_cast<const f4*>(p + off + 16);
    }
  }
  // The tiles and their rows' units: 2^(e - kTop) of operand a's, 2^e of b's. (a's meet the unit of a
  // wave's own row, 2^(e - kTop) too, in the factor of the scores: the product of a tiny and a huge row
  // passes through no subnormal, which 2^(-2 kTop) on one side would be from 2^-98 down.)
  __device__ __forceinline__ void store(Tile<D>& a, Tile<D>& b, float* ua, float* ub, int w,
                                        int lane) {
#pragma unroll
    for (int i = 0; i < kN; ++i) {
      const bool is_b = kHalves ? lane >= 32 : i >= kPer;
      const int r = row(i, w, lane);
      e[i] = exponent(group_max<kC>(abs_max8(x[i][0], x[i][1], 0.0f)));
      if (lane % kC == 0) (is_b ? ub : ua)[r] = pow2(is_b ? e[i] : e[i] - kTop);
      const Pair s = split8(x[i][0], x[i][1], pow2(kTop - e[i]));
      char* p = reinterpret_cast<char*>(is_b ? &b : &a) + r * (2 * D) +
                (((lane % kC) ^ chunk_swz<D>(r)) << 4);
      *reinterpret_cast<h8*>(p) = s.h;
      *reinterpret_cast<h8*>(p + kPlane<D>) = s.l;
    }
  }
};
// Beside a Stage whose operand b is dO: O's rows in the same lanes, and D = rowsum(dO o O) of the
// tile's 32 rows, in units of dO's rows and times 2^kTop (dS meets Q's unit). O's offsets are in
// elements: its rows of one (b, h) may span more than 4 GiB (the views' may not).
template <int D, int W>
struct RowDots {
  using S = Stage<D, W>;
  static constexpr int kC = S::kC, kN = S::kPer;
  f4 x[kN][2];
  __device__ __forceinline__ void load(const float* o, unsigned ss, int r0, int last, int w,
                                       int lane) {
#pragma unroll
    for (int i = 0; i < kN; ++i) {
      const unsigned r = static_cast<unsigned>(min(r0 + S::row(i, w, lane), last));
      const unsigned off = r * ss + 8u * static_cast<unsigned>(lane % kC);
      x[i][0] = ld4(o + off);
      x[i][1] = ld4(o + off + 4);
    }
  }
  __device__ __forceinline__ void put(const S& st, float* dst, int w, int lane) const {
#pragma unroll
    for (int i = 0; i < kN; ++i) {
      const f4(&y)[2] = st.x[S::kN / 2 + i];
      float t = x[i][0][0] * y[0][0];
#pragma unroll
      for (int e = 1; e < 8; ++e) t = fmaf(x[i][e / 4][e % 4], y[e / 4][e % 4], t);
      t += dpp<0xB1>(t);
      t += dpp<0x4E>(t);
      if constexpr (D >= 64) t += dpp<0x141>(t);
      if constexpr (D == 128) t += dpp<0x140>(t);
      if (lane % kC == 0 && (!S::kHalves || lane >= 32)) {
        dst[S::row(i, w, lane)] = t * pow2(kTop - st.e[S::kN / 2 + i]);
      }
    }
  }
};
// A wave's own 32 rows as B operands: row j, columns 16 ks + 8 g .. + 7 of each step, scaled per
// row (lanes j and j + 32 hold one row). Returns 1 / scale (without `sign`).
template <int D>
struct OwnRows {
  f4 x[D / 16][2];
  __device__ __forceinline__ void load(const float* row, int g) {
#pragma unroll
    for (int ks = 0; ks < D / 16; ++ks) {
      x[ks][0] = ld4(row + 16 * ks + 8 * g);
      x[ks][1] = ld4(row + 16 * ks + 8 * g + 4);
    }
  }
  __device__ __forceinline__ float split(float sign, Pair (&dst)[D / 16]) const {
    float m = 0.0f;
#pragma unroll
    for (int ks = 0; ks < D / 16; ++ks) m = abs_max8(x[ks][0], x[ks][1], m);
    const int e = exponent(pair_max(fmaxf(m, 0.0f)));
    const float sc = pow2(kTop - e) * sign;
#pragma unroll
    for (int ks = 0; ks < D / 16; ++ks) dst[ks] = split8(x[ks][0], x[ks][1], sc);
    return pow2(e - kTop);
  }
};

// 32 rows x D of an accumulator (times f f2, per lane), through the wave's part of LDS, to rows of
// `stride` floats. Two factors: their product may be below the least float, where it is 0 or, as a
// pow2() out of range, anything, while a sum times it is not.
template <int D, int N>
__device__ __forceinline__ void store_rows(const f16v (&acc)[N], float f, float f2, float* so,
                                           float* base, int64_t stride, int rows, int lane) {
  constexpr int kCols = D < 64 ? D : 64, kPitch = kCols + 4, kLanes = kCols / 4;
  const int j = lane & 31, g = lane >> 5;
#pragma unroll
  for (int c0 = 0; c0 < D; c0 += kCols) {
#pragma unroll
    for (int dt = c0 / 32; dt < (c0 + kCols) / 32; ++dt) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const f4 x{acc[dt][4 * i], acc[dt][4 * i + 1], acc[dt][4 * i + 2], acc[dt][4 * i + 3]};
        st4(so + j * kPitch + 32 * dt - c0 + 8 * i + 4 * g, x * f * f2);
      }
    }
#pragma unroll
    for (int i = 0; i < kRows; i += 64 / kLanes) {
      const int row = i + lane / kLanes, c = 4 * (lane % kLanes);
      const f4 x = ld4(so + row * kPitch + c);
      if (row < rows) st4_nt(base + row * stride + c0 + c, x);
    }
  }
}
// --- Rows in fp32 ------------------------------------------------------------------------------
// A wave's 32 rows from memory, on v_mfma_f32_32x32x2_f32 and with no part of the workgroup's
// staging (waves come here alone, past the last barrier). Lane (j, g) supplies A[j][g] and B[g][j]
// and holds D as above, so a product over columns takes 8 i + 4 g + e in step (i, e), and a sum over
// staged rows takes row 8 (r / 4) + 4 g + r % 4 in step r, with register r as its B operand. A row
// that a lane's own row does not see must not meet its weight of 0 there (0 times an infinity): a
// tile with masked rows sums its live ones row by row, the weights through the wave's part of LDS.
// With a NaN in V of every head, forward / backward us (one row at a time, lanes over keys, before;
// clean inputs in brackets): b64 h6 s240 132 / 477 (4186 / 19357; 36 / 106), b16 h16 s1024 1118 / 3939
// (60518 / 262624; 222 / 798).
__device__ __forceinline__ f16v mma32(float a, float b, f16v c) {
  return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
}
// The tile's row of register r, for the half g.
__device__ __forceinline__ int tile_row(int r, int g) { return 8 * (r >> 2) + 4 * g + (r & 3); }
// The products of a tile's row (one per lane j) with the lane's own row.
template <int D>
__device__ __forceinline__ f16v dots_fp32(const float* row, const float* own, int g) {
  f16v c = zero16();
#pragma clang loop unroll_count(4)
  for (int i = 4 * g; i < D; i += 8) {
    const f4 x = ld4(row + i), y = ld4(own + i);
#pragma unroll
    for (int e = 0; e < 4; ++e) c = mma32(x[e], y[e], c);
  }
  return c;
}
// acc^T += rows^T weights, over the tile's rows r0 .. (register r holds the weight of tile_row(r)).
// kFull: all 32 are live for every lane. Else those below `end` that live(row) lets through.
template <int D, bool kFull, typename Live>
__device__ __forceinline__ void sum_fp32(const f16v& weights, const float* base, int64_t stride,
                                         int r0, int end, Live live, float* so, f16v (&acc)[D / 32],
                                         int j, int g) {
  if constexpr (kFull) {
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const float* row = base + (r0 + tile_row(r, g)) * stride + j;
#pragma unroll
      for (int dt = 0; dt < D / 32; ++dt) acc[dt] = mma32(row[32 * dt], weights[r], acc[dt]);
    }
  } else {
#pragma unroll
    for (int r = 0; r < 16; ++r) so[tile_row(r, g) * 32 + j] = weights[r];
    const int n = min(kRows, end - r0);
#pragma clang loop unroll(disable)
    for (int i = 0; i < n; ++i) {
      const float w = so[i * 32 + j];
      const float* row = base + (r0 + i) * stride + 4 * g;
      if (live(r0 + i)) {
#pragma unroll
        for (int dt = 0; dt < D / 32; ++dt) {
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            acc[dt][r] = fmaf(w, row[32 * dt + 8 * (r >> 2) + (r & 3)], acc[dt][r]);
          }
        }
      }
    }
  }
}

// --- Forward -----------------------------------------------------------------------------------
// One workgroup = W waves of one (b, h), NQ groups of 32 queries per wave; key tiles of 32 keys,
// split into LDS by all its waves (each value split once per workgroup). Per wave, tile and group:
//   S^T = K Q^T (A = K rows, B = Q in registers): lane (j, g), register r holds the score of query
//   j and key 8 (r / 4) + 4 g + r % 4, so a query's online softmax is one lane's and lane ^ 32's;
//   O^T += V^T P^T (A = V transposed, B = P from S^T's registers).
// Two LDS buffers, one barrier per tile: a step works on tile t, stores tile t + 1 and loads tile
// t + 2. (Fewer than four waves have at most one tile each, and all are staged before the walk.)
// The softmax: p = 2^(s c2 - m), c2 = |scale| log2 e and the two rows' scales, m a reference that is
// kRefTop below the largest score seen when it was set. p is computed with the m in hand and its
// row sum is what is tested: only where it exceeds kRowTop (or m is not set yet) is the tile's
// largest score taken, m moved and p computed again, so that an ordinary tile pays no rescale.
// What enters O's product is p times the unit of its V row and the query's running power of two
// `wsc`, which puts the largest such weight at 2^kWTop when it is set, moves with m and falls where a
// weight would pass f16's limit: a key of large weight and small V (an attention sink), or a large V
// row of no weight, leaves the others' bits alone. (kWTop: 10 bits of room before a weight moves it.)
constexpr float kRefTop = 3.0f;
constexpr float kRowTop = 32768.0f;
constexpr int kWTop = 6;
constexpr float kMaxWeight = 61440.0f;  // of a scaled weight (f16 ends at 65504)
constexpr float kMaxScale = 0x1p127f;   // of a running scale, and where it starts

// O and L of 32 queries from qg in fp32. `store` takes O's sums and their factor.
template <int D, bool kCausal, typename Store>
__device__ __forceinline__ void fwd_rows_fp32(const FwdArgs& a, int b, int h, int qg, float* so,
                                              int lane, Store store) {
  const int j = lane & 31, g = lane >> 5, S = a.S, qi = qg + j;
  const float* qp = a.q.p + b * a.q.sb + h * a.q.sh + min(qi, S - 1) * a.q.ss;
  const float* kp = a.k.p + b * a.k.sb + h * a.k.sh;
  const float* vp = a.v.p + b * a.v.sb + h * a.v.sh;
  const float sign = a.scale < 0.0f ? -1.0f : 1.0f, c2 = fabsf(a.scale) * kLog2e;
  f16v acc[D / 32];
#pragma unroll
  for (int dt = 0; dt < D / 32; ++dt) acc[dt] = zero16();
  float m = kNegInf, l = 0.0f;
  auto tile = [&](auto fullc, int k0) {
    constexpr bool kFull = decltype(fullc)::value != 0;
    auto live = [&](int key) { return kFull || (key < S && !(kCausal && key > qi)); };
    f16v s = dots_fp32<D>(kp + min(k0 + j, S - 1) * a.k.ss, qp, g);
    float mn = m;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      s[r] = live(k0 + tile_row(r, g)) ? s[r] * sign : kNegInf;
      mn = fmaxf(mn, s[r]);
    }
    mn = pair_max(fmaxf(mn, kNegInf));
    const float alpha = mn == m ? 1.0f : m == kNegInf ? 0.0f : exp2_hw((m - mn) * c2);
    m = mn;
    l *= alpha;
#pragma unroll
    for (int dt = 0; dt < D / 32; ++dt) acc[dt] *= alpha;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      s[r] = s[r] == kNegInf ? 0.0f : exp2_hw(fmaf(s[r], c2, -(mn * c2)));
      l += s[r];
    }
    sum_fp32<D, kFull>(s, vp, a.v.ss, k0, S, live, so, acc, j, g);
  };
  const int kend = kCausal ? min(S, qg + kRows) : S;
  int k0 = 0;
  for (; k0 + kRows <= (kCausal ? min(S, qg + 1) : S); k0 += kRows) tile(Const<1>{}, k0);
  for (; k0 < kend; k0 += kRows) tile(Const<0>{}, k0);
  l = pair_sum(l);
  store(acc, 1.0f / l);
  if (g == 0 && qi < S) {
    a.lse[(static_cast<int64_t>(b) * a.H + h) * S + qi] = m * fabsf(a.scale) + logf(l);
  }
}

template <int D, bool kCausal, int NQ, int W, int WAVES>
__global__ void __launch_bounds__(64 * W) __attribute__((amdgpu_waves_per_eu(WAVES, WAVES)))
fwd_pair_kernel(FwdArgs a) {
  a.causal = kCausal ? 1 : 0;
  constexpr int kKS = D / 16;              // contraction steps of S
  constexpr int kDT = D / 32;              // 32-dim tiles of O
  constexpr int kOPitch = (D < 64 ? D : 64) + 4;  // store_rows'
  constexpr int kWaveQ = kRows * NQ, kQ = W * kWaveQ, kBufs = W == 1 ? 1 : 2;
  struct Kv {
    Tile<D> k, v;
  };
  union Tiles {
    Kv kv[kBufs];
    float o[W][kRows * kOPitch];
  };
  struct Smem {
    Tiles t;
    float uk[kBufs][kRows], uv[kBufs][kRows];
  };
  __shared__ __attribute__((aligned(16))) Smem sm;

  const int tid = threadIdx.x, lane = tid & 63, j = lane & 31, g = lane >> 5;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int S = a.S, BH = a.B * a.H;
  int qb, bh;
  if (kCausal) {
    qb = a.nqb - 1 - static_cast<int>(blockIdx.x) / BH;  // the most expensive first
    bh = static_cast<int>(blockIdx.x) % BH;
  } else {
    const int id = xcd_remap(static_cast<int>(blockIdx.x), a.nqb * BH);
    qb = id % a.nqb;
    bh = id / a.nqb;
  }
  const int b = bh / a.H, h = bh % a.H;
  const int q0 = qb * kQ, qw0 = q0 + w * kWaveQ;
  const float* qp = a.q.p + b * a.q.sb + h * a.q.sh;
  const Operand kop{reinterpret_cast<const char*>(a.k.p + b * a.k.sb + h * a.k.sh),
                    static_cast<unsigned>(a.k.ss) * 4u};
  const Operand vop{reinterpret_cast<const char*>(a.v.p + b * a.v.sb + h * a.v.sh),
                    static_cast<unsigned>(a.v.ss) * 4u};

  const int k_end = kCausal ? min(S, q0 + kQ) : S;
  const int ntiles = (k_end + kRows - 1) / kRows;
  const int kw_end = kCausal ? min(S, qw0 + kWaveQ) : S;  // keys this wave's queries can see
  const bool wave_live = qw0 < S;

  // The first tile, the wave's queries (negated for a negative scale, so that the raw scores' max
  // is the scaled scores'), and the second tile's loads.
  Stage<D, W> st;
  Pair q[NQ][kKS];
  float cq[NQ];  // |scale| log2 e over the query's scale
  {
    OwnRows<D> own[NQ];
    st.load(kop, vop, 0, S - 1, w, lane);
#pragma unroll
    for (int n = 0; n < NQ; ++n) own[n].load(qp + min(qw0 + kRows * n + j, S - 1) * a.q.ss, g);
    st.store(sm.t.kv[0].k, sm.t.kv[0].v, sm.uk[0], sm.uv[0], w, lane);
    if (W > 1) st.load(kop, vop, kRows, S - 1, w, lane);
#pragma unroll
    for (int n = 0; n < NQ; ++n) {
      cq[n] = own[n].split(a.scale < 0.0f ? -1.0f : 1.0f, q[n]) *
              (fabsf(a.scale) * kLog2e);
    }
    if constexpr (W == 2) st.store(sm.t.kv[1].k, sm.t.kv[1].v, sm.uk[1], sm.uv[1], w, lane);
  }

  f16v acc[NQ][kDT];  // O^T, in units of p / wsc and 2^-kTop
  float m[NQ], lsum[NQ], wsc[NQ];
#pragma unroll
  for (int n = 0; n < NQ; ++n) {
    m[n] = kNegInf;
    lsum[n] = 0.0f;
    wsc[n] = kMaxScale;
#pragma unroll
    for (int dt = 0; dt < kDT; ++dt) acc[n][dt] = zero16();
  }
  const int roff0 = row_off<D>(j, g), coff0 = col_off<D>(lane);

  // Stores tile t + 1 (loaded in the last step) and issues the loads of tile t + 2.
  auto stage = [&](int t) {
    if (W != 4) return;
    const int put = (t + 1) & 1;
    st.store(sm.t.kv[put].k, sm.t.kv[put].v, sm.uk[put], sm.uv[put], w, lane);
    st.load(kop, vop, (t + 2) * kRows, S - 1, w, lane);
    pin_loads();
  };
  // One tile: kFull, one with no mask. (Past the walk's end a step stages rows that repeat the last
  // one and nothing reads: tested for, the loaded registers would live across the whole step.)
  auto tile = [&](auto fullc, int t) {
    constexpr bool kFull = decltype(fullc)::value != 0;
    const int roff = late(roff0), coff = late(coff0), kt0 = t * kRows, cur = W == 1 ? 0 : t & 1;
    const Kv& kv = sm.t.kv[cur];
    stage(t);
    f16v s[NQ];
    {
      h8 kh[kKS];
#pragma unroll
      for (int n = 0; n < NQ; ++n) s[n] = zero16();
#pragma unroll
      for (int ks = 0; ks < kKS; ++ks) {
        const Pair k = ld_row<D>(kv.k, roff ^ row_step(ks));
        kh[ks] = k.h;
#pragma unroll
        for (int n = 0; n < NQ; ++n) s[n] = mma_small(k, q[n][ks], s[n]);
      }
#pragma unroll
      for (int ks = 0; ks < kKS; ++ks) {
#pragma unroll
        for (int n = 0; n < NQ; ++n) s[n] = mma(kh[ks], q[n][ks].h, s[n]);
      }
    }
    Pair p[NQ][2];
#pragma unroll
    for (int n = 0; n < NQ; ++n) {
      const int qi = qw0 + kRows * n + j;
      // Live: keys below S and, causal, not after the query.
      auto live = [&](int r) {
        const int key = kt0 + 8 * (r >> 2) + 4 * g + (r & 3);
        return kFull || (key < S && !(kCausal && key > qi));
      };
      f16v e;
      float psum = 0.0f, wmax = 0.0f;
      // The weights (e) and their largest.
      auto exps = [&] {
        wmax = 0.0f;
        int r0 = 4 * g;
        asm("" : "+v"(r0));  // (the units are read again the second time, not held)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const f4 uk = ld4(&sm.uk[cur][8 * i + r0]), uv = ld4(&sm.uv[cur][8 * i + r0]);
#pragma unroll
          for (int c = 0; c < 4; ++c) {
            const int r = 4 * i + c;
            const float x = exp2_hw(fmaf(s[n][r], cq[n] * uk[c], -m[n]));
            const float p = live(r) ? x : 0.0f;
            psum = r == 0 ? p : psum + p;
            e[r] = p * uv[c];
          }
          asm("v_max3_f32 %0, %1, %2, %0" : "+v"(wmax) : "v"(e[4 * i]), "v"(e[4 * i + 1]));
          asm("v_max3_f32 %0, %1, %2, %0" : "+v"(wmax) : "v"(e[4 * i + 2]), "v"(e[4 * i + 3]));
        }
      };
      exps();
      if (__builtin_amdgcn_ballot_w64(!(psum <= kRowTop && wmax * wsc[n] <= kMaxWeight)) != 0) {
        float tmax = kNegInf;
        int r0 = 4 * g;
        asm("" : "+v"(r0));
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const float x = s[n][r] * (cq[n] * sm.uk[cur][8 * (r >> 2) + r0 + (r & 3)]);
          tmax = fmaxf(tmax, live(r) ? x : kNegInf);
        }
        // (-inf: a row with no live key.)
        const float ref = pair_max(tmax) - kRefTop;
        // O's unit is p / wsc: where p falls by alpha, wsc rises and O stays as it is but for rounding.
        float to = wsc[n], alpha = 1.0f;
        if (!(pair_sum(psum) <= kRowTop) && ref > m[n]) {
          alpha = m[n] == kNegInf ? 0.0f : exp2_hw(m[n] - ref);
          to = alpha > 0.0f ? fminf(to * pow2(-exponent(alpha)), kMaxScale) : kMaxScale;
          m[n] = ref;
          lsum[n] *= alpha;
          exps();
        }
        wmax = pair_max(fmaxf(wmax, 0.0f));
        if (wmax * to > kMaxWeight) to = pow2(kWTop - exponent(wmax));
        const float f = alpha > 0.0f ? alpha * (to / wsc[n]) : 0.0f;
        wsc[n] = to;
#pragma unroll
        for (int dt = 0; dt < kDT; ++dt) acc[n][dt] *= f;
      }
      lsum[n] += psum;
      p[n][0] = split_acc<0>(e, wsc[n]);
      p[n][1] = split_acc<1>(e, wsc[n]);
    }
    const bool second = kFull || kt0 + 16 < kw_end;  // wave-uniform: the last 16 keys are live
#pragma unroll
    for (int dt = 0; dt < kDT; ++dt) {
      const Pair v0 = ld_col<D>(kv.v, coff ^ col_step(dt), 0);
#pragma unroll
      for (int n = 0; n < NQ; ++n) acc[n][dt] = mma3(v0, p[n][0], acc[n][dt]);
      if (second) {
        const Pair v1 = ld_col<D>(kv.v, coff ^ col_step(dt), 1);
#pragma unroll
        for (int n = 0; n < NQ; ++n) acc[n][dt] = mma3(v1, p[n][1], acc[n][dt]);
      }
    }
  };
  // Tiles wholly below S (and, causal, at or before the wave's first query) need no mask.
  const int full_end = (kCausal ? min(S, qw0 + 1) : S) / kRows;
  const int nfull = wave_live ? min(full_end, ntiles) : 0;
  __syncthreads();  // tile 0
  int t = 0;
  for (; t < nfull; ++t) {
    if (!kCausal) prio_by_remaining(ntiles - t, ntiles);
    tile(Const<1>{}, t);
    __syncthreads();  // tile t + 1 is staged; every wave is done with tile t
  }
  for (; t < ntiles; ++t) {
    if (!kCausal) prio_by_remaining(ntiles - t, ntiles);
    if (wave_live && t * kRows < kw_end) {
      tile(Const<0>{}, t);
    } else {
      stage(t);
    }
    __syncthreads();
  }

  // L = m / (log2 e as rounded into c2) + ln(l), to one rounding (in fp64, the logarithm of l's
  // significand aside): the backward takes exp(S scale - L), where an error of L scales a whole row
  // of P (logf(l), with log2 of some 8 taken at once, left -3.8e-7 on average and 4.9e-7 rms).
  const float as = fabsf(a.scale), cu = as * kLog2e;
  const double mr =
      as == 0.0f ? 0.6931471805599453 : static_cast<double>(as) / static_cast<double>(cu);
#pragma unroll
  for (int n = 0; n < NQ; ++n) {
    const int qg = qw0 + kRows * n, qi = qg + j;
    if (qg >= S) break;
    const float l = pair_sum(lsum[n]);
    // O through LDS (the wave's own part; every wave is past its last tile), so that each row is
    // written as whole 128-byte lines.
    float* so = sm.t.o[w];
    const int lane_e = late(lane);
    auto store = [&](const f16v (&x)[kDT], float f, float f2) {
      store_rows<D>(x, f, f2, so, a.o + ((static_cast<int64_t>(b) * S + qg) * a.H + h) * D,
                    static_cast<int64_t>(a.H) * D, S - qg, lane_e);
    };
    if (__builtin_amdgcn_ballot_w64(qi < S && !(probe_finite<kDT>(acc[n], l * 0.0f) == 0.0f)) !=
        0) {
      fwd_rows_fp32<D, kCausal>(a, b, h, qg, so, late(lane),
                                [&](const f16v (&x)[kDT], float inv) { store(x, inv, 1.0f); });
      continue;
    }
    // (Two factors: their product may be subnormal.)
    store(acc[n], 1.0f / l, pow2(-kTop) / wsc[n]);
    if (g == 0 && qi < S) {
      int le = exponent(l);
      float f = l * pow2(-le);  // [1, 2), then [0.75, 1.5)
      if (f > 1.5f) f *= 0.5f, ++le;
      const double L = fma(static_cast<double>(m[n]), mr, fma(le, 0.6931471805599453, logf(f)));
      __builtin_nontemporal_store(static_cast<float>(L), a.lse + static_cast<int64_t>(bh) * S + qi);
    }
  }
}

// --- Backward ----------------------------------------------------------------------------------
// One launch of two kinds of workgroup, W waves x 32 rows each, which share no sum, so that no
// workgroup waits for another and the results depend on nothing but the shape:
//   key blocks (of 128 keys with four waves) walk 32-query tiles and hold dK, dV (S, dP, dV, dK: four
//   products);
//   query blocks walk 32-key tiles and hold dQ (S, dP, dQ: three products).
// S and dP are computed in both: seven products where one kind of workgroup would need five, but
// then dQ's partial sums (4 s^2 b h bytes) would go through memory and dS through LDS, between
// barriers. Backward, against that scheme on the fp32 matrix instruction (five products): b64 h6 s240
// 92 us (147), causal 81 (93), causal b8 h12 s2048 630 (1096), b16 h16 s1024 808 (1373), d 128
// b64 h6 s240 234 (319). Where walks are short and the blocks many it loses at d 128: one wave per SIMD,
// so that nothing runs beside a block's first loads and last stores: causal, 1024 (b, h), s 65
// 192 us (132), s 128 277 (228), s 200 572 (466), even at s 400; without a mask even at s 65.
// (Workgroups of two waves that walk need 124 registers more than there are: s 200 669.)
// Bounds, b64 h6 s240 (per call): 8.8 us per 32-row step of the walk, about half of it the matrix
// cores, the rest the softmax, the splits and the staging between them; 35 us for the own rows in,
// the first tiles and the gradients out (past the L2s 239 MB are read, each operand by both kinds of
// block, and 77 MB written). Long walks are bound by power: at b16 h16 s1024 the clock falls from 2.4
// to about 1.95 GHz.
//   key block: S = Q K^T, dP = dO V^T (A = staged rows, B = the wave's keys in registers): lane
//   (j, g), register r holds key j and query 8 (r / 4) + 4 g + r % 4 of the tile;
//   P = exp(S scale - L), dS = P o (dP - D); dV^T += dO^T P, dK^T += Q^T dS (A = the staged tiles
//   transposed, B = P, dS from those registers). L comes from the forward, D = rowsum(dO o O) is
//   formed while dO is staged.
//   query block: S^T = K Q^T, dP^T = V dO^T, lane (j, g) holding query j; dQ^T += K^T dS^T.
// S takes the forward's products in the forward's order: exp(S scale - L) is 1 / l of the
// probabilities that L was summed from, and the rows of P sum to 1.
// Exponents: P is formed as P 2^k = 2^(S c2 + (k - L log2 e)), the sum in brackets (exact to one
// rounding) held per row and k about half of log2 s, so that the exponent stays near 0 whether a row
// is flat (P about 1 / s) or peaked (P about 1): exp((S scale - L)) rounds its argument twice, at
// -log2 s for a flat row, which was the largest error of the gradients.
// Weights: P 2^k and dS times the unit of the staged row enter their products times a running power
// of two per lane (its key, or query), lowered (and the sums with it) when a weight would pass f16's
// limit. D is staged in units of its dO row, so that the unit enters P alone: P u (dP / u - D / u).
struct BwdPairArgs {
  View q, k, v, d_o;
  const float* o;
  const float* lse;
  float* dqkv;
  // A split-size workspace: per 16-query tile, `done` takes the launch's epoch where dQ was written;
  // with `defer` (or for the pair `give_up_bh`, where no step 3 follows: NaN) dQ goes unscaled to
  // `part` ([b h][tile][16][D]) for step 3. Null: dQ is written.
  float* part;
  unsigned long long* done;
  unsigned long long* epoch_slot;
  unsigned long long epoch;
  int* ctrl;
  int B, H, S, nkv, nblk;  // nkv: key blocks in the grid; nblk: blocks of 32 W rows per (b, h)
  float scale;
  int causal, defer, last, give_up_bh;
};
// Where a new scale puts the largest weight: 9 bits of room before the next one moves it, which costs
// a pass over the sums (with 5, inputs of deviation 2: d 128 b64 h6 s240 259 us against 242, d 32 56.0 /
// 54.4, b16 h16 s1024 851 / 839), and no row error above 1.01 of that over 1580 checks.
constexpr int kDsTop = 7;

// The running scale of the weights in one lane: raises nothing, lowers `sc` (and the accumulators by
// the same factor) where a weight would exceed kMaxWeight. First the largest, then the test.
__device__ __forceinline__ float max_weight(const f16v& x) {
  float m = 0.0f;
#pragma unroll
  for (int r = 0; r < 16; r += 2) {
    asm("v_max3_f32 %0, |%1|, |%2|, %0" : "+v"(m) : "v"(x[r]), "v"(x[r + 1]));
  }
  return m;
}
template <int N>
__device__ __forceinline__ void fit_scale(float m, float& sc, f16v (&acc)[N]) {
  m = pair_max(fmaxf(m, 0.0f));
  if (m * sc > kMaxWeight) {
    const float to = pow2(kDsTop - exponent(m));
    const float f = to / sc;  // (a power of two, or 0)
    sc = to;
#pragma unroll
    for (int i = 0; i < N; ++i) acc[i] *= f;
  }
}
// D 128: the sums stay in accumulation registers across a branch that rescales them (the compiler
// otherwise keeps them, or what they displace, in memory).
template <int N>
__device__ __forceinline__ void pin_acc(f16v (&acc)[N]) {
  if constexpr (N == 4) {
#pragma unroll
    for (int i = 0; i < N; ++i) asm("" : "+a"(acc[i]));
  }
}
// k - L log2 e, log2 e in two terms.
constexpr float kLog2eLow = 1.925963033500e-8f;
__device__ __forceinline__ float shifted_l(float L, float k) {
  return fmaf(-L, kLog2eLow, fmaf(-L, kLog2e, k));
}
__device__ __forceinline__ int half_log2(int s) { return (32 - __builtin_clz(s)) / 2; }

// dK and dV of 32 keys from kw0, dQ of 32 queries from qw0, in fp32 (without the scale).
template <int D, bool kCausal>
__device__ __forceinline__ void bwd_keys_fp32(const BwdPairArgs& a, int b, int h, int kw0, float* so,
                                              f16v (&dk)[D / 32], f16v (&dv)[D / 32], int lane) {
  const int j = lane & 31, g = lane >> 5, S = a.S, key = kw0 + j;
  const float* kr = a.k.p + b * a.k.sb + h * a.k.sh + min(key, S - 1) * a.k.ss;
  const float* vr = a.v.p + b * a.v.sb + h * a.v.sh + min(key, S - 1) * a.v.ss;
  const float* qp = a.q.p + b * a.q.sb + h * a.q.sh;
  const float* gp = a.d_o.p + b * a.d_o.sb + h * a.d_o.sh;
  const float* op = a.o + (static_cast<int64_t>(b) * S * a.H + h) * D;
  const float* lp = a.lse + (static_cast<int64_t>(b) * a.H + h) * S;
#pragma unroll
  for (int dt = 0; dt < D / 32; ++dt) dk[dt] = zero16(), dv[dt] = zero16();
  auto tile = [&](auto fullc, int q0) {
    constexpr bool kFull = decltype(fullc)::value != 0;
    auto live = [&](int qi) { return kFull || (qi < S && !(kCausal && qi < key)); };
    const int64_t qr = min(q0 + j, S - 1);
    f16v s = dots_fp32<D>(qp + qr * a.q.ss, kr, g), dp = dots_fp32<D>(gp + qr * a.d_o.ss, vr, g);
    float dd = 0.0f;
#pragma clang loop unroll(disable)
    for (int c = 4 * g; c < D; c += 8) {
      const f4 x = ld4(gp + qr * a.d_o.ss + c), y = ld4(op + qr * a.H * D + c);
#pragma unroll
      for (int e = 0; e < 4; ++e) dd = fmaf(x[e], y[e], dd);
    }
    dd = pair_sum(dd);
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int t = tile_row(r, g), qi = min(q0 + t, S - 1);
      const float p = exp2_hw(fmaf(s[r], a.scale, -lp[qi]) * kLog2e);
      const float y = p * (dp[r] - __shfl(dd, t));  // (every lane takes part in the shuffle)
      s[r] = live(q0 + t) ? p : 0.0f;
      dp[r] = live(q0 + t) ? y : 0.0f;
    }
    sum_fp32<D, kFull>(s, gp, a.d_o.ss, q0, S, live, so, dv, j, g);
    sum_fp32<D, kFull>(dp, qp, a.q.ss, q0, S, live, so, dk, j, g);
  };
  int q0 = kCausal ? kw0 : 0;
  if (kCausal) tile(Const<0>{}, q0), q0 += kRows;
  for (; q0 + kRows <= S; q0 += kRows) tile(Const<1>{}, q0);
  if (q0 < S) tile(Const<0>{}, q0);
}
template <int D, bool kCausal>
__device__ __forceinline__ void bwd_queries_fp32(const BwdPairArgs& a, int b, int h, int qw0,
                                                 float* so, f16v (&dq)[D / 32], int lane) {
  const int j = lane & 31, g = lane >> 5, S = a.S, qi = qw0 + j;
  const int64_t qc = min(qi, S - 1);
  const float* qr = a.q.p + b * a.q.sb + h * a.q.sh + qc * a.q.ss;
  const float* gr = a.d_o.p + b * a.d_o.sb + h * a.d_o.sh + qc * a.d_o.ss;
  const float* kp = a.k.p + b * a.k.sb + h * a.k.sh;
  const float* vp = a.v.p + b * a.v.sb + h * a.v.sh;
  const float* orow = a.o + ((static_cast<int64_t>(b) * S + qc) * a.H + h) * D;
  const float L = a.lse[(static_cast<int64_t>(b) * a.H + h) * S + qc];
  float dd = 0.0f;
#pragma clang loop unroll(disable)
  for (int c = 4 * g; c < D; c += 8) {
    const f4 x = ld4(gr + c), y = ld4(orow + c);
#pragma unroll
    for (int e = 0; e < 4; ++e) dd = fmaf(x[e], y[e], dd);
  }
  dd = pair_sum(dd);
#pragma unroll
  for (int dt = 0; dt < D / 32; ++dt) dq[dt] = zero16();
  auto tile = [&](auto fullc, int k0) {
    constexpr bool kFull = decltype(fullc)::value != 0;
    auto live = [&](int key) { return kFull || (key < S && !(kCausal && key > qi)); };
    const int64_t kr = min(k0 + j, S - 1);
    const f16v s = dots_fp32<D>(kp + kr * a.k.ss, qr, g);
    f16v dp = dots_fp32<D>(vp + kr * a.v.ss, gr, g);
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const float x = exp2_hw(fmaf(s[r], a.scale, -L) * kLog2e) * (dp[r] - dd);
      dp[r] = live(k0 + tile_row(r, g)) ? x : 0.0f;
    }
    sum_fp32<D, kFull>(dp, kp, a.k.ss, k0, S, live, so, dq, j, g);
  };
  const int kend = kCausal ? min(S, qw0 + kRows) : S;
  int k0 = 0;
  for (; k0 + kRows <= (kCausal ? min(S, qw0 + 1) : S); k0 += kRows) tile(Const<1>{}, k0);
  for (; k0 < kend; k0 += kRows) tile(Const<0>{}, k0);
}

// LDS of a backward workgroup.
template <int D, int W>
struct BwdSmem {
  static constexpr int kBufs = W == 1 ? 1 : 2;  // (one wave has at most one tile, two have two)
  union {
    struct {
      Tile<D> a, b;
    } t[kBufs];
    float o[W][kRows * ((D < 64 ? D : 64) + 4)];
  };
  float ua[kBufs][kRows], ub[kBufs][kRows], l[kBufs][kRows], d[kBufs][kRows];  // (d over ub)
};

template <int D, bool kCausal, bool kSerial, int W>
__device__ __forceinline__ void bwd_keys(const BwdPairArgs& a, BwdSmem<D, W>& sm, int item) {
  constexpr int kKS = D / 16, kDT = D / 32;
  const int tid = threadIdx.x, lane = tid & 63, j = lane & 31, g = lane >> 5;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int S = a.S, bh = item / a.nblk, kb = item % a.nblk;
  const int b = bh / a.H, h = bh % a.H;
  const int k0 = kb * (W * kRows), kw0 = k0 + w * kRows, key = kw0 + j;
  const bool wave_live = kw0 < S;
  const Operand qop{reinterpret_cast<const char*>(a.q.p + b * a.q.sb + h * a.q.sh),
                    static_cast<unsigned>(a.q.ss) * 4u};
  const Operand gop{reinterpret_cast<const char*>(a.d_o.p + b * a.d_o.sb + h * a.d_o.sh),
                    static_cast<unsigned>(a.d_o.ss) * 4u};
  const float* op = a.o + (static_cast<int64_t>(b) * S * a.H + h) * D;
  const float* lp = a.lse + static_cast<int64_t>(bh) * S;
  // The walk: step u takes tile t0 + u (causal: from the block's diagonal, W tiles, on).
  const int ntiles = (S + kRows - 1) / kRows, t0 = kCausal ? k0 / kRows : 0;
  const int nsteps = ntiles - t0;

  const int kp = half_log2(S);
  Stage<D, W> st;
  RowDots<D, W> ro;
  float lreg;
  auto load = [&](int u) { st.load(qop, gop, (t0 + u) * kRows, S - 1, w, lane); };
  auto load_o = [&](int u) {
    const int r0 = (t0 + u) * kRows;
    ro.load(op, static_cast<unsigned>(a.H) * D, r0, S - 1, w, lane);
    lreg = lp[min(r0 + j, S - 1)];
  };
  auto store = [&](int put) {
    st.store(sm.t[put].a, sm.t[put].b, sm.ua[put], sm.ub[put], w, lane);
    ro.put(st, sm.d[put], w, lane);
    if (w == 0 && g == 0) sm.l[put][j] = shifted_l(lreg, kp);
  };
  Pair kB[kKS], vB[kKS];
  float uk, uv;  // 1 / the key's scales
  {
    OwnRows<D> ok, ov;
    load(0);
    load_o(0);
    ok.load(a.k.p + b * a.k.sb + h * a.k.sh + min(key, S - 1) * a.k.ss, g);
    ov.load(a.v.p + b * a.v.sb + h * a.v.sh + min(key, S - 1) * a.v.ss, g);
    uk = ok.split(1.0f, kB);
    uv = ov.split(1.0f, vB);
    store(0);
    if (W > 1) {
      load(1);
      load_o(1);
    }
    if (W == 2) store(1);
  }
  f16v dk[kDT], dv[kDT];
#pragma unroll
  for (int dt = 0; dt < kDT; ++dt) dk[dt] = zero16(), dv[dt] = zero16();
  const float cs = a.scale * kLog2e * uk, cg = uv;
  float psc = kSerial ? 1.0f : kMaxScale, dsc = kMaxScale;
  const int roff0 = row_off<D>(j, g), coff0 = col_off<D>(lane);

  // The next step's tile, and the loads of the one after it (four waves; fewer have at most two
  // tiles, and both are staged).
  constexpr bool kWalk = W == 4;
  auto tile = [&](auto fullc, int u) {
    constexpr bool kFull = decltype(fullc)::value != 0;
    const int roff = late(roff0), coff = late(coff0), cur = W == 1 ? 0 : u & 1, q0 = (t0 + u) * kRows;
    if (kFull && kWalk) store((u + 1) & 1);
    const Tile<D>&Q = sm.t[cur].a, &G = sm.t[cur].b;
    f16v s = zero16(), dp = zero16();
    {
      h8 x[kKS];
#pragma unroll
      for (int ks = 0; ks < kKS; ++ks) {
        const Pair q = ld_row<D>(Q, roff ^ row_step(ks));
        x[ks] = q.h;
        // (The forward's order: its A operand is this B.)
        s = mma(q.l, kB[ks].h, s);
        s = mma(q.h, kB[ks].l, s);
      }
#pragma unroll
      for (int ks = 0; ks < kKS; ++ks) s = mma(x[ks], kB[ks].h, s);
#pragma unroll
      for (int ks = 0; ks < kKS; ++ks) {
        const Pair y = ld_row<D>(G, roff ^ row_step(ks));
        x[ks] = y.h;
        dp = mma_small(y, vB[ks], dp);
      }
#pragma unroll
      for (int ks = 0; ks < kKS; ++ks) dp = mma(x[ks], vB[ks].h, dp);
    }
    // The loads of the step after next from here on (its O later still): held across the products
    // above as well, they do not fit.
    if (kFull && kWalk) {
      load(u + 2);
      pin_loads();
    }
    // Live: register r's query, q0 + 4 g + 8 i + e, below S and, causal, not before the key.
    const int hi = key < S ? S - q0 - 4 * g : 0, lo = kCausal ? key - q0 - 4 * g : 0;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const f4 L = ld4(&sm.l[cur][8 * i + 4 * g]), Dv = ld4(&sm.d[cur][8 * i + 4 * g]);
      const f4 uq = ld4(&sm.ua[cur][8 * i + 4 * g]), ug = ld4(&sm.ub[cur][8 * i + 4 * g]);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int r = 4 * i + e;
        const float x = exp2_hw(fmaf(s[r], cs * uq[e], L[e])) * ug[e];
        const bool live = kFull || (8 * i + e < hi && !(kCausal && 8 * i + e < lo));
        const float p = live ? x : 0.0f;
        const float y = p * fmaf(dp[r], cg, -Dv[e]) * uq[e];
        dp[r] = live ? y : 0.0f;
        s[r] = p;
      }
    }
    // (Both tests before either product: a second branch over accumulators spills at d 128.)
    pin_acc(dv);
    pin_acc(dk);
    const float mp = kSerial ? 0.0f : max_weight(s), md = max_weight(dp);
    if (__builtin_amdgcn_ballot_w64(mp * psc > kMaxWeight || md * dsc > kMaxWeight) != 0) {
      if constexpr (!kSerial) fit_scale(mp, psc, dv);
      fit_scale(md, dsc, dk);
      pin_acc(dv);
      pin_acc(dk);
    }
    if constexpr (kSerial) {
#pragma unroll
      for (int dt = 0; dt < kDT; ++dt) {
        const Pair g0 = ld_col<D>(G, coff ^ col_step(dt), 0), g1 = ld_col<D>(G, coff ^ col_step(dt), 1);
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const Pair& y = r < 8 ? g0 : g1;
          dv[dt] = mma32(static_cast<float>(y.h[r % 8]) + static_cast<float>(y.l[r % 8]), s[r],
                         dv[dt]);
        }
      }
    } else {
      const Pair p0 = split_acc<0>(s, psc), p1 = split_acc<1>(s, psc);
#pragma unroll
      for (int dt = 0; dt < kDT; ++dt) {
        dv[dt] = mma3(ld_col<D>(G, coff ^ col_step(dt), 0), p0, dv[dt]);
        dv[dt] = mma3(ld_col<D>(G, coff ^ col_step(dt), 1), p1, dv[dt]);
      }
    }
    if (kFull && kWalk) {
      load_o(u + 2);
      pin_loads();
    }
    {
      const Pair p0 = split_acc<0>(dp, dsc), p1 = split_acc<1>(dp, dsc);
#pragma unroll
      for (int dt = 0; dt < kDT; ++dt) {
        dk[dt] = mma3(ld_col<D>(Q, coff ^ col_step(dt), 0), p0, dk[dt]);
        dk[dt] = mma3(ld_col<D>(Q, coff ^ col_step(dt), 1), p1, dk[dt]);
      }
    }
  };
  // Steps with no mask: every query and key below S and, causal, past the diagonal. (In the others
  // the staging is outside the branch: in both its arms, the loaded registers and the accumulators
  // spill where they join.)
  const int full1 = kw0 + kRows <= S ? S / kRows - t0 : 0;
  auto masked = [&](int u) {
    if (kWalk) {
      store((u + 1) & 1);
      load(u + 2);
      load_o(u + 2);
      pin_loads();
    }
    if (wave_live && !(kCausal && (t0 + u) * kRows + kRows <= kw0)) tile(Const<0>{}, u);
    __syncthreads();
  };
  __syncthreads();
  int u = 0;
  if (kCausal) {
    for (; u < min(W, nsteps); ++u) masked(u);
  }
  for (; u < full1; ++u) {
    tile(Const<1>{}, u);
    __syncthreads();
  }
  for (; u < nsteps; ++u) masked(u);
  if (!wave_live) return;
  // The two factors of dK and of dV: the second is a power of two, exact where it is subnormal.
  float fk = pow2(-kTop) * a.scale, fk2 = pow2(-kp) / dsc, fv = pow2(-kTop - kp), fv2 = 1.0f / psc;
  const float z = probe_finite<kDT>(dk, probe_finite<kDT>(dv, fk * 0.0f));
  if (__builtin_amdgcn_ballot_w64(key < S && !(z == 0.0f)) != 0) {
    bwd_keys_fp32<D, kCausal>(a, b, h, kw0, sm.o[w], dk, dv, late(lane));
    fk = a.scale, fk2 = fv = fv2 = 1.0f;
  }
  const int64_t part = static_cast<int64_t>(a.H) * D;
  float* row = a.dqkv + (static_cast<int64_t>(b) * S + kw0) * 3 * part + static_cast<int64_t>(h) * D;
  const int lane_e = late(lane);
  store_rows<D>(dk, fk, fk2, sm.o[w], row + part, 3 * part, S - kw0, lane_e);
  store_rows<D>(dv, fv, fv2, sm.o[w], row + 2 * part, 3 * part, S - kw0, lane_e);
}

template <int D, bool kCausal, int W>
__device__ __forceinline__ void bwd_queries(const BwdPairArgs& a, BwdSmem<D, W>& sm, int item) {
  constexpr int kKS = D / 16, kDT = D / 32;
  const int tid = threadIdx.x, lane = tid & 63, j = lane & 31, g = lane >> 5;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int S = a.S, bh = item / a.nblk, qb = item % a.nblk;
  const int b = bh / a.H, h = bh % a.H;
  const int q0 = qb * (W * kRows), qw0 = q0 + w * kRows, qi = qw0 + j;
  const bool wave_live = qw0 < S;
  const Operand kop{reinterpret_cast<const char*>(a.k.p + b * a.k.sb + h * a.k.sh),
                    static_cast<unsigned>(a.k.ss) * 4u};
  const Operand vop{reinterpret_cast<const char*>(a.v.p + b * a.v.sb + h * a.v.sh),
                    static_cast<unsigned>(a.v.ss) * 4u};
  const int k_end = kCausal ? min(S, q0 + W * kRows) : S;
  const int ntiles = (k_end + kRows - 1) / kRows;
  const int kw_end = kCausal ? min(S, qw0 + kRows) : S;

  Stage<D, W> st;
  Pair qB[kKS], gB[kKS];
  const int kp = half_log2(S);
  float uq, ug, L, Dq;  // L: kp - L log2 e
  {
    OwnRows<D> oq, og, oo;
    const int qc = min(qi, S - 1);
    st.load(kop, vop, 0, S - 1, w, lane);
    oq.load(a.q.p + b * a.q.sb + h * a.q.sh + qc * a.q.ss, g);
    og.load(a.d_o.p + b * a.d_o.sb + h * a.d_o.sh + qc * a.d_o.ss, g);
    oo.load(a.o + ((static_cast<int64_t>(b) * S + qc) * a.H + h) * D, g);
    L = a.lse[static_cast<int64_t>(bh) * S + qc];
    Dq = 0.0f;
#pragma unroll
    for (int ks = 0; ks < kKS; ++ks) {
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        Dq = fmaf(og.x[ks][e / 4][e % 4], oo.x[ks][e / 4][e % 4], Dq);
      }
    }
    Dq = pair_sum(Dq) * pow2(kTop);  // (dP and D times 2^kTop meet K's unit)
    L = shifted_l(L, kp);
    uq = oq.split(1.0f, qB);
    ug = og.split(1.0f, gB);
    st.store(sm.t[0].a, sm.t[0].b, sm.ua[0], sm.ub[0], w, lane);
    if (W > 1) st.load(kop, vop, kRows, S - 1, w, lane);
    if constexpr (W == 2) st.store(sm.t[1].a, sm.t[1].b, sm.ua[1], sm.ub[1], w, lane);
  }
  f16v dq[kDT];
#pragma unroll
  for (int dt = 0; dt < kDT; ++dt) dq[dt] = zero16();
  const float cs = a.scale * kLog2e * uq, cg = ug;
  float dsc = kMaxScale;
  const int roff0 = row_off<D>(j, g), coff0 = col_off<D>(lane);

  auto stage = [&](int t) {  // (four waves, as above)
    if (W != 4) return;
    const int put = (t + 1) & 1;
    st.store(sm.t[put].a, sm.t[put].b, sm.ua[put], sm.ub[put], w, lane);
  };
  auto load = [&](int t) {
    if (W != 4) return;
    st.load(kop, vop, (t + 2) * kRows, S - 1, w, lane);
    pin_loads();
  };
  auto tile = [&](auto fullc, int t) {
    constexpr bool kFull = decltype(fullc)::value != 0;
    const int roff = late(roff0), coff = late(coff0), cur = W == 1 ? 0 : t & 1, kt0 = t * kRows;
    stage(t);
    const Tile<D>&K = sm.t[cur].a, &V = sm.t[cur].b;
    f16v s = zero16(), dp = zero16();
    {
      h8 x[kKS];
#pragma unroll
      for (int ks = 0; ks < kKS; ++ks) {
        const Pair k = ld_row<D>(K, roff ^ row_step(ks));
        x[ks] = k.h;
        s = mma_small(k, qB[ks], s);
      }
#pragma unroll
      for (int ks = 0; ks < kKS; ++ks) s = mma(x[ks], qB[ks].h, s);
#pragma unroll
      for (int ks = 0; ks < kKS; ++ks) {
        const Pair v = ld_row<D>(V, roff ^ row_step(ks));
        x[ks] = v.h;
        // (The key blocks' order: their A operand is this B.)
        dp = mma(v.l, gB[ks].h, dp);
        dp = mma(v.h, gB[ks].l, dp);
      }
#pragma unroll
      for (int ks = 0; ks < kKS; ++ks) dp = mma(x[ks], gB[ks].h, dp);
    }
    load(t);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const f4 uk = ld4(&sm.ua[cur][8 * i + 4 * g]), uv = ld4(&sm.ub[cur][8 * i + 4 * g]);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int r = 4 * i + e, key = kt0 + 8 * i + 4 * g + e;
        const float x =
            exp2_hw(fmaf(s[r], cs * uk[e], L)) * fmaf(dp[r], cg * uv[e], -Dq) * uk[e];
        dp[r] = kFull || (key < S && !(kCausal && key > qi)) ? x : 0.0f;
      }
    }
    pin_acc(dq);
    const float md = max_weight(dp);
    if (__builtin_amdgcn_ballot_w64(md * dsc > kMaxWeight) != 0) {
      fit_scale(md, dsc, dq);
      pin_acc(dq);
    }
    const Pair p0 = split_acc<0>(dp, dsc), p1 = split_acc<1>(dp, dsc);
#pragma unroll
    for (int dt = 0; dt < kDT; ++dt) {
      dq[dt] = mma3(ld_col<D>(K, coff ^ col_step(dt), 0), p0, dq[dt]);
      dq[dt] = mma3(ld_col<D>(K, coff ^ col_step(dt), 1), p1, dq[dt]);
    }
  };
  const int full_end = (kCausal ? min(S, qw0 + 1) : S) / kRows;
  const int nfull = wave_live ? min(full_end, ntiles) : 0;
  __syncthreads();
  int t = 0;
  for (; t < nfull; ++t) {
    tile(Const<1>{}, t);
    __syncthreads();
  }
  for (; t < ntiles; ++t) {
    if (wave_live && t * kRows < kw_end) {
      tile(Const<0>{}, t);
    } else {
      stage(t);
      load(t);
    }
    __syncthreads();
  }
  // Where dQ goes (uniform): its rows, or the workspace for step 3.
  const bool gave_up = bh == a.give_up_bh;
  const bool direct = a.part == nullptr || !(a.defer || (gave_up && !a.last));
  const int ntile16 = (S + kBwdQueryTile - 1) / kBwdQueryTile;
  if (a.done != nullptr && direct && tid < W * kRows / kBwdQueryTile) {
    const int j16 = q0 / kBwdQueryTile + tid;
    if (j16 < ntile16) a.done[static_cast<int64_t>(bh) * ntile16 + j16] = a.epoch;
  }
  if (!wave_live) return;
  const int64_t stride = direct ? static_cast<int64_t>(3) * a.H * D : D;
  float* row = direct ? a.dqkv + (static_cast<int64_t>(b) * S + qw0) * 3 * a.H * D +
                            static_cast<int64_t>(h) * D
                      : a.part + (static_cast<int64_t>(bh) * ntile16 * kBwdQueryTile + qw0) * D;
  const float factor = direct ? a.scale : 1.0f;
  float f = pow2(-kTop) * factor, f2 = pow2(-kp) / dsc;
  if (gave_up && direct) {
    // (The test hook, as a wait that ran out would: NaN and the guard word.)
    if (lane == 0) {
      __hip_atomic_store(a.ctrl + kCtrlGuard, 3, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    f = __builtin_nanf("");
  } else if (__builtin_amdgcn_ballot_w64(
                 qi < S && !(probe_finite<kDT>(dq, f * 0.0f) == 0.0f)) != 0) {
    bwd_queries_fp32<D, kCausal>(a, b, h, qw0, sm.o[w], dq, late(lane));
    f = factor, f2 = 1.0f;
  }
  store_rows<D>(dq, f, f2, sm.o[w], row, stride, S - qw0, late(lane));
}

template <int D, bool kCausal, bool kSerial, int W, int WAVES>
__global__ void __launch_bounds__(64 * W) __attribute__((amdgpu_waves_per_eu(WAVES, WAVES)))
bwd_pair_kernel(BwdPairArgs a) {
  a.causal = kCausal ? 1 : 0;
  __shared__ __attribute__((aligned(16))) BwdSmem<D, W> sm;
  const int id = static_cast<int>(blockIdx.x), BH = a.B * a.H;
  if (id == 0 && threadIdx.x == 0) {
    __hip_atomic_store(a.ctrl + kCtrlGuard, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (a.epoch_slot != nullptr) *a.epoch_slot = a.epoch;
  }
  if (W < 4) {
    // One workgroup of each kind per (b, h): side by side on one XCD, so that what both read comes
    // from memory once.
    const int item = xcd_remap(id, 2 * a.nkv);
    if (item & 1) {
      bwd_queries<D, kCausal, W>(a, sm, item >> 1);
    } else {
      bwd_keys<D, kCausal, kSerial, W>(a, sm, item >> 1);
    }
  } else if (id < a.nkv) {
    // Causal: the low blocks (they see every later query) first.
    bwd_keys<D, kCausal, kSerial, W>(a, sm, kCausal ? id % BH * a.nblk + id / BH : xcd_remap(id, a.nkv));
  } else {
    const int i = id - a.nkv;
    bwd_queries<D, kCausal, W>(a, sm, kCausal ? i % BH * a.nblk + a.nblk - 1 - i / BH : xcd_remap(i, a.nkv));
  }
}

template <int D, int WAVES>
const void* fwd_pair_fn(int causal, int waves) {
  auto fn = [&](auto w) {
    constexpr int W = decltype(w)::value;
    constexpr int kOcc = W == 2 && D == 64 ? 2 : WAVES;  // (two waves share two tiles' LDS)
    return causal ? reinterpret_cast<const void*>(fwd_pair_kernel<D, true, 1, W, kOcc>)
                  : reinterpret_cast<const void*>(fwd_pair_kernel<D, false, 1, W, kOcc>);
  };
  if constexpr (D != 128) {
    if (waves == 2) return fn(Const<2>{});
  }
  return waves == 1 ? fn(Const<1>{}) : fn(Const<4>{});
}

// Waves per workgroup, each of 32 rows. Four share the staging of a tile, but over a short sequence
// those past its end only stage and wait, and the tiles ahead of the walk are staged for nothing:
// where there are workgroups enough for every CU without them, one wave takes s <= 32 and two
// s <= 64, with every tile staged before the walk (and, backward, the two kinds of workgroup of one
// (b, h) side by side). Fewer waves against four, us, 1536 (b, h), forward / backward: D 64, s 16
// 9.5 / 18 (16.0 / 41), s 32 11.5 / 22 (17.0 / 47), s 64 22.8 / 47 (24.4 / 66), causal s 64 25.3 / 49
// (25.2 / 72); D 128 s 32 27 / 56 (31 / 148), s 64 backward 122 (209), forward 46 (44: four);
// D 32 s 64 13.4 / 27 (15.9 / 39). With 64 (b, h), where the time is one workgroup's: D 64 s 64
// 8.1 / 11.4 (7.2 / 10.1), D 128 s 32 9.2 / 14.1 (8.1 / 13.4).
int workgroup_waves(int bh, int s, bool two) {
  if (bh <= 256 || s > 64) return 4;
  return s <= 32 ? 1 : two ? 2 : 4;
}

// Causal, s up to kSerialLength and up to kSerialBlocks key blocks: dV summed over the queries one at a
// time, on the fp32 matrix instruction (kSerial). The first keys of a causal row sum hundreds of terms
// of one sign, and there a sum of one rounding per query, as the composed fp32 path makes, and one of
// three per 16 queries drift apart by more than the reference's band around that path (5e-6;
// tests/parity.rs:218): at b 2 h 6 s 240 the composed path's dV is 6.0e-6 from fp64, so a correctly
// rounded one misses the band too. Small grids of the lengths for which the reference states the band
// (up to 240; here two blocks) keep to it, at a few us per call; all others take the faster and more
// accurate sum. With it / without, backward us: s 64 12.3 / 10.7, s 128 19.3 / 16.1, s 240 30.5 / 23.5
// (b 2 h 6: 31.0 / 24.0), and what longer walks would pay: s 512 51.5 / 36.9, s 2048 179 / 119, s 8192
// 689 / 447; D 128 s 1024 180 / 125.
constexpr int kSerialBlocks = 64, kSerialLength = 256;
template <int D, int WAVES>
const void* bwd_pair_fn(int causal, bool serial, int waves) {
  auto fn = [&](auto w) {
    constexpr int W = decltype(w)::value;
    if constexpr (W == 4) {  // (fewer waves: more than 256 (b, h))
      if (serial) return reinterpret_cast<const void*>(bwd_pair_kernel<D, true, true, W, WAVES>);
    }
    return causal ? reinterpret_cast<const void*>(bwd_pair_kernel<D, true, false, W, WAVES>)
                  : reinterpret_cast<const void*>(bwd_pair_kernel<D, false, false, W, WAVES>);
  };
  return waves == 1 ? fn(Const<1>{}) : waves == 2 ? fn(Const<2>{}) : fn(Const<4>{});
}

}  // namespace

int launch_forward(View q, View k, View v, float* o, float* lse, int b, int h, int s, int d,
                   float scale, int causal, void* stream) {
  // 64 queries per wave (256 per workgroup) halve what a query pays for reading, splitting and
  // waiting for the key tiles, but hold 2 waves per SIMD instead of 3 (D 64; 3 instead of 4 at D 32)
  // and halve the workgroups. Taken where every workgroup walks all keys, 1024 of them keep every CU
  // busy for two rounds or more, and no more than an eighth of their queries is padding that 128 per
  // workgroup would not have. Measured, 64 against 32 queries per wave, us: D 64, b h 256 s 1024
  // (1024 workgroups) 224 / 247, 512 x 512 121 / 131, 1024 x 256 77 / 83; too few, 64 x 1280 (320)
  // 119 / 108, 256 x 256 26 / 23; padded, 1024 x 300 140 / 121, 1024 x 640 425 / 419, and below s 128
  // half of it is (1536 x 32: 29 / 17). D 32, 256 x 1024 145 / 150, 512 x 512 81 / 81, but 1024 x 200
  // 46 / 43: from s 257 on. At D 128 their registers do not fit.
  const int64_t wide = static_cast<int64_t>((s + 255) / 256) * b * h;
  const bool filled = 8 * 2 * ((s + 255) / 256) <= 9 * ((s + 127) / 128) && (d == 64 || s > 256);
  const int nq = d != 128 && !causal && wide >= 1024 && filled ? 2 : 1;
  const int waves = workgroup_waves(b * h, s, d != 128), qb = kRows * waves * nq, nqb = (s + qb - 1) / qb;
  FwdArgs a{q, k, v, o, lse, b, h, s, nqb, scale, causal ? 1 : 0};
  void* args[] = {&a};
  const void* fn;
  if (nq == 2) {
    fn = d == 32 ? reinterpret_cast<const void*>(fwd_pair_kernel<32, false, 2, 4, 3>)
                 : reinterpret_cast<const void*>(fwd_pair_kernel<64, false, 2, 4, 2>);
  } else {
    fn = d == 32    ? fwd_pair_fn<32, 4>(causal, waves)
         : d == 128 ? fwd_pair_fn<128, 2>(causal, waves)
                    : fwd_pair_fn<64, 3>(causal, waves);
  }
  return static_cast<int>(hipLaunchKernel(fn, dim3(static_cast<unsigned>(nqb) * b * h),
                                          dim3(64u * waves), args, 0,
                                          static_cast<hipStream_t>(stream)));
}

int launch_backward(View q, View k, View v, View d_o, const float* o, const float* lse, float* dqkv,
                    float* part, unsigned long long* done, unsigned long long* epoch_slot,
                    unsigned long long epoch, int* ctrl, int b, int h, int s, int d, float scale,
                    int causal, int defer, int last, int give_up_bh, void* stream) {
  const int waves = workgroup_waves(b * h, s, true), rows = kRows * waves, nblk = (s + rows - 1) / rows;
  BwdPairArgs a{q, k, v, d_o, o, lse, dqkv, part, done, epoch_slot, epoch, ctrl, b, h, s,
                nblk * b * h, nblk, scale, causal ? 1 : 0, defer, last, give_up_bh};
  void* args[] = {&a};
  const bool serial = causal && s <= kSerialLength && a.nkv <= kSerialBlocks;
  // Waves per SIMD: what the registers allow without spills to the loop. At d 32 the third fits once
  // the fp32 fallback's loops are not unrolled (they set the register count); with it b64 h6 s240
  // takes 63 us (67 with two), causal b8 h12 s2048 352 (375).
  const void* fn = d == 32    ? bwd_pair_fn<32, 3>(causal, serial, waves)
                   : d == 128 ? bwd_pair_fn<128, 1>(causal, serial, waves)
                              : bwd_pair_fn<64, 2>(causal, serial, waves);
  return static_cast<int>(hipLaunchKernel(fn, dim3(2u * static_cast<unsigned>(a.nkv)),
                                          dim3(64u * waves), args, 0,
                                          static_cast<hipStream_t>(stream)));
}

}  // namespace fattn
