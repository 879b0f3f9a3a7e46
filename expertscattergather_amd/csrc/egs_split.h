// fp32 products on the bf16 matrix instruction.
//
// An fp32 value is the sum of three bf16 values exactly: h = bf16(x), m = bf16(x - h), l = x - h - m (8 bits of the 24 each; the
// subtractions are exact).  Of the nine products of two such sums six are taken, the smallest first,
//   x y = lh + hl + mm + mh + hm + hh   (the others are below 2^-25 of it),
// each exact in the fp32 accumulator's input, so that what is rounded is the accumulator, as with the fp32 matrix instruction -
// fewer times: 16x16x32 adds 32 products at a time where 16x16x4 adds four.  Measured against 64 bits, 64 problems of N(0,1) data:
// reduction 32 3.8e-8 (the fp32 instruction 1.0e-7), 64 0.94e-7 (1.44e-7), 128 1.5e-7 (2.0e-7), 1024 4.9e-7 (5.7e-7), 4096 1.00e-6
// (1.14e-6) of the result's root mean square.  Six instructions of 16 cycles stand for eight of 32, and at a higher clock:
// an instruction-only loop over all CUs does 320 to 400 TFLOP/s of fp32 work against 140 to 156, by its length.
//
// bf16 numbers end at 2^-133 (subnormal ones are kept by the conversion and by the matrix instruction), where an fp32 value may still
// have bits down to 2^-149.  So both operands are taken times 2^16, which makes the three pieces exact down to the smallest fp32 number,
// and sums times 2^-32.  What that brings near the other end - values from 2^112 on, sums from 2^96 - arrives as infinity or NaN, as
// infinities (inf - inf) and NaN do: a wavefront whose stored results are not all finite takes its tile again with the fp32 instruction.
// Without the factor the error grew below 2^-110: operands of 2^-115 1.1e-6, 2^-120 3.5e-5, 2^-125 1.1e-3.
#pragma once
#include "egs_device.h"

namespace egs {

constexpr float kSplitScale = 65536.f, kSplitUnscale = 0x1p-32f;       // of a value; of a sum of products of two

// the three pieces of two floats (times kSplitScale), packed in pairs
__device__ __forceinline__ void split_pair(float x, float y, uint32_t (&piece)[3])
{
    x *= kSplitScale; y *= kSplitScale;
    piece[0] = pack2<ElemBF16>(x, y);
    const float rx = x - bits_f32(piece[0] << 16), ry = y - bits_f32(piece[0] & 0xffff0000u);
    piece[1] = pack2<ElemBF16>(rx, ry);
    piece[2] = pack2<ElemBF16>(rx - bits_f32(piece[1] << 16), ry - bits_f32(piece[1] & 0xffff0000u));
}
// ... and of four
__device__ __forceinline__ void split_chunk(const u32x4 &v, u32x2 (&piece)[3])
{
    uint32_t lo[3], hi[3];
    split_pair(bits_f32(v[0]), bits_f32(v[1]), lo);
    split_pair(bits_f32(v[2]), bits_f32(v[3]), hi);
#pragma unroll
    for (int x = 0; x < 3; ++x) piece[x] = u32x2{lo[x], hi[x]};
}
// `t` if the first `live` elements are finite, else NaN
__device__ __forceinline__ float not_finite(const f32x4 &v, int live, float t)
{
#pragma unroll
    for (int x = 0; x < 4; ++x) t = fmaf(x < live ? v[x] : 0.f, 0.f, t);
    return t;
}
// sums of split products out of their scale; where one is not finite, the second take's result instead.  (Element by element: which
// bits a finite result has does not depend on its neighbours.)
__device__ __forceinline__ void split_result(f32x4 &v, const f32x4 &second)
{
#pragma unroll
    for (int x = 0; x < 4; ++x) v[x] = fabsf(v[x]) < __builtin_inff() ? v[x] * kSplitUnscale : second[x];
}

constexpr int kSplitP[6] = {2, 0, 1, 1, 0, 0}, kSplitQ[6] = {0, 2, 1, 0, 1, 0};   // pieces of the six products, the smallest first

}  // namespace egs
