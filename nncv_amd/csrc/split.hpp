// fp32 products on the bf16 matrix pipes (gfx950): an fp32 value is the exact sum of three bf16 pieces, and
//   a b = ah bh + (ah bm + am bh) + (ah bl + am bm + al bh) + what is below 2^-24 of it
// (G. Henry, P. T. P. Tang, A. Heinecke, Leveraging the bfloat16 Artificial Intelligence Datatype For Higher-Precision Computations, 2019).
// The six products are v_mfma_f32_32x32x16_bf16, sixteen times the rate of the fp32 instructions for six times the
// work; every one is exact and the sums are fp32.  The five small ones are summed in registers of their own, so the chain of
// roundings that carries the result's magnitude has one link for 16 k, where the fp32 instructions have one for every k: against
// 64 bits the error of a sum of normal products is 3.1e-8 at 16 of them (fp32 instructions 7.3e-8), 1.3e-7 at 576 (4.3e-7)
// and 4.2e-7 at 4608 (1.2e-6).  A sum that one product is all of is where the dropped ones show: off by 9.5e-8 at most, 2.6e-8 in the
// mean, where one fp32 rounding makes 6.0e-8 and 2.5e-8.  (Pieces that are cut off instead of rounded: 1.55e-7 with the second one,
// and with the first one the dropped products have a sign, a bias of 3e-8.)
//
// Range.  bf16 ends at 2^-133 (its normal numbers at 2^-126), fp32 at 2^-149: what is split is 2^24 times the value, so that every piece
// of every fp32 value is a normal number, and a sum is 2^48 times what it is worth.  (Unscaled, the error of a sum of products of one
// operand at 2^-112 was 2.6e-7, at 2^-118 1.8e-5, at 2^-126 2.4e-3.)  The two multiplications for a pair of values cost what a kernel's
// vector instructions bound: 2 to 11 % of a product (1024^3 14.9 -> 16.6 us, 1500x1001x777 22.7 -> 23.2, 4096^3 772 -> 817), 8 % of
// the 64 x 32 form of conv_direct, 2 to 7 % of igemm_fast's, 0 to 3 % of conv3x3_split, 1.7 % of a classification of six photographs.  To look
// for pieces that lose bits instead (an or for a pair) was slower: its register made the 64 x 64 products spill (4096^3 1142).
//
// What is not finite.  An infinity has a NaN for its second piece, and so has a value from 2^103 on, which 2^24 takes to infinity; a sum
// from 2^80 on is infinite.  Every result such an operand takes part in comes out not finite, and a wave whose sums are not all finite
// takes them again with the fp32 instructions (plain_products): one operand like that costs its tile's waves a second walk at a
// third of the rate, and inputs that are all NaN every wave.  Back to back, us a call, usual / one NaN / all NaN: 1500x1001x777
// 40 / 53 / 75 (one lane a sum: 40 / 90 / 693), a 3x3 layer 6x58x78x64 -> 64 31 / 83 / 119 (30 / 360 / 2038), a 1x1 one
// 23x88x24x128 -> 128 36 / 59 / 77 (36 / 305 / 1918).
#pragma once
#include "mfma_tile.hpp"

namespace nncv_hip {
namespace mt {

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx2 __attribute__((ext_vector_type(2)));
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));

constexpr float kSplitScale = 0x1p24f, kSplitWorth = 0x1p-48f;

// Two values -> their pieces, packed in pairs: thirteen instructions.  Two pieces are rounded to nearest even, what is left after them
// has eight bits: the third is exact.  (The second one cut off takes as many, and as long within 1 %.  v_dot2_f32_bf16 would take a piece off in one instruction instead of
// two, but it runs in the matrix pipe: the products wait for it.)
__device__ __forceinline__ void split_pair(float x, float y, unsigned (&p)[3]) {
  x *= kSplitScale;
  y *= kSplitScale;
  p[0] = __builtin_bit_cast(unsigned, __builtin_convertvector((floatx2{x, y}), bf16x2));
  x -= __builtin_bit_cast(float, p[0] << 16);
  y -= __builtin_bit_cast(float, p[0] & 0xffff0000u);
  p[1] = __builtin_bit_cast(unsigned, __builtin_convertvector((floatx2{x, y}), bf16x2));
  x -= __builtin_bit_cast(float, p[1] << 16);
  y -= __builtin_bit_cast(float, p[1] & 0xffff0000u);
  p[2] = __builtin_amdgcn_perm(__builtin_bit_cast(unsigned, y), __builtin_bit_cast(unsigned, x), 0x07060302u);
}

__device__ __forceinline__ floatx16 mma_bf16(const u32x4& a, const u32x4& b, const floatx16& c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

// eight values -> an operand in three pieces
__device__ __forceinline__ void split_eight(const u32x4& a, const u32x4& b, u32x4 (&out)[3]) {
  const floatx4 x = __builtin_bit_cast(floatx4, a), y = __builtin_bit_cast(floatx4, b);
  unsigned p[4][3];
  split_pair(x[0], x[1], p[0]);
  split_pair(x[2], x[3], p[1]);
  split_pair(y[0], y[1], p[2]);
  split_pair(y[2], y[3], p[3]);
#pragma unroll
  for (int c = 0; c < 3; ++c) out[c] = u32x4{p[0][c], p[1][c], p[2][c], p[3][c]};
}

// the six products of TM x TN blocks
template <int TM, int TN>
__device__ __forceinline__ void split_products(const u32x4 (&a)[TM][3], const u32x4 (&b)[TN][3], floatx16 (&big)[TM][TN], floatx16 (&low)[TM][TN]) {
  constexpr int kX[6] = {0, 0, 1, 0, 1, 2}, kY[6] = {0, 1, 0, 2, 1, 0};
#pragma unroll
  for (int c = 0; c < 6; ++c)
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        floatx16& s = c == 0 ? big[i][j] : low[i][j];
        s = mma_bf16(a[i][kX[c]], b[j][kY[c]], s);
      }
}

// what big + low are worth -> big; whether a sum of the wave is not finite
template <int TM, int TN>
__device__ __forceinline__ bool split_sums(floatx16 (&big)[TM][TN], const floatx16 (&low)[TM][TN]) {
  float t = 0.0f;  // a sum times zero is a zero or a NaN
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) {
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        big[i][j][v] = (big[i][j][v] + low[i][j][v]) * kSplitWorth;
        t = __builtin_fmaf(big[i][j][v], 0.0f, t);
      }
    }
  return __builtin_amdgcn_ballot_w64(!(t == 0.0f)) != 0;
}

// The sums of TM x TN blocks with the fp32 instructions, straight from memory.  load(s, a, b): step s, eight k, four of which a lane half has
// (lanes l < 32 the first ones); zeros for a step past the last.
template <int TM, int TN, typename Load>
__device__ __forceinline__ void plain_products(floatx16 (&acc)[TM][TN], int steps, const Load& load) {
  u32x4 a[2][TM], b[2][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.0f;
  load(0, a[0], b[0]);
#pragma unroll 1
  for (int s = 0; s < steps; s += 2)
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      load(s + h + 1, a[h ^ 1], b[h ^ 1]);
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) Mma<float>::run(a[h][i], b[h][j], acc[i][j]);
    }
}

}  // namespace mt
}  // namespace nncv_hip
