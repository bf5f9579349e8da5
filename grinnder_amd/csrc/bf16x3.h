// fp32 products on the bf16 matrix cores: every fp32 operand is split into
// three bf16 pieces and the six leading piece products are summed in fp32.
//
// x = h + m + l with h = bf16(x), m = bf16(x - h), l = bf16(x - h - m), each
// rounded to nearest: |m| <= 2^-9 |x|, |l| <= 2^-18 |x|, and since a bf16 has
// 8 significant bits the three hold all 24 of an fp32 (exactly, while l is
// above bf16's smallest denormal: for |x| below 2^-109 the absolute error is
// at most 2^-134).  x y is formed as h h' + h m' + m h' + m m' + h l' + l h';
// the dropped m l', l m', l l' are at most 2^-26 |x y|, a quarter of an fp32
// product's own rounding.  A bf16 product is exact in fp32, and the matrix
// core adds 16 of them per step where v_mfma_f32_32x32x2_f32 adds two, so a
// sum over K takes 6 K / 16 rounded additions instead of K / 2 (or K).
//
// Rate: v_mfma_f32_32x32x16_bf16 does 16 times the work of
// v_mfma_f32_32x32x2_f32 per cycle, six of them replace eight fp32 steps:
// 2.67 times the fp32 matrix peak per clock.  The clock falls under the load
// (1.3 to 1.8 GHz with random operands, 2.0 to 2.4 for the fp32 products), so
// what is left is 1.5 to 1.8 times.
//
// Error, relative 2-norm against 64 bits on N(0, 1) operands, this split
// against the fp32 matrix instructions: C[100k, 256] over K = 64, 256, 1024
// 1.1e-7, 2.4e-7, 4.9e-7 against 1.5e-7, 2.9e-7, 5.7e-7; 256 x 256 over 1M
// rows in 256 chunks 9.6e-7 against 1.15e-6.
//
// Bias: aligning the addends to the largest, the bf16 matrix core drops bits
// below its window toward minus infinity, so every sum comes out slightly low
// (mean error -1.5e-8 of the result's rms over K = 256, 6% of the rms error),
// whatever its sign.  Each result alone is no worse for it, but a later sum
// over many of them would collect it.  The products therefore sum the negated
// operand, and negate the result, for every other row (gemm_nt_bf3) or K
// chunk (gemm_tn_bf3): the low bias becomes a high one there, and sums over
// rows or chunks cancel it (mean error 1e-11 after, as for fp32; 256 x 256
// over 1M rows was 3.4e-6 without it).
//
// An infinite or NaN operand, or one that rounds up to infinity in bf16,
// gives inf - inf = NaN pieces.  Kernels that use the split therefore look
// for a non-finite sum and form such a block again with fp32 MFMAs, so
// infinities and NaN come out as in fp32.
#ifndef GR_BF16X3_H
#define GR_BF16X3_H

#include <hip/hip_runtime.h>

namespace gr_bf3 {

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx2 __attribute__((ext_vector_type(2)));
typedef float floatx16 __attribute__((ext_vector_type(16)));

// The three pieces of (x0, x1), packed (x0 in the low half).
__device__ __forceinline__ void split2(float x0, float x1, unsigned& h, unsigned& m,
                                       unsigned& l) {
  auto pack = [](float a, float b) {
    return __builtin_bit_cast(unsigned, __builtin_convertvector((floatx2){a, b}, bf16x2));
  };
  auto lo = [](unsigned p) { return __builtin_bit_cast(float, p << 16); };
  auto hi = [](unsigned p) { return __builtin_bit_cast(float, p & 0xffff0000u); };
  h = pack(x0, x1);
  const float r0 = x0 - lo(h), r1 = x1 - hi(h);
  m = pack(r0, r1);
  l = pack(r0 - lo(m), r1 - hi(m));
}

// The pieces of A and B in the order their products are summed: smallest first.
constexpr int kPieceA[6] = {2, 0, 1, 1, 0, 0};
constexpr int kPieceB[6] = {0, 2, 1, 0, 1, 0};

}  // namespace gr_bf3

#endif
