// fp32 products on the bf16 matrix cores (gfx950).
//
// v_mfma_f32_16x16x4_f32 runs at 1/16 of the bf16 rate per contracted element, so an fp32 contraction
// is done as six bf16 products.  A value x is split into three bf16 parts that carry its 24 significand
// bits exactly: x0 = the upper 16 bits of x (never overflows), x1 = bf16(x - x0), x2 = x - x0 - x1 (both
// differences are exact, and the last one has at most 8 bits).  a b is then a0 b0 + (a0 b1 + a1 b0) +
// (a0 b2 + a1 b1 + a2 b0); what is left out, a1 b2 + a2 b1 + a2 b2, is below 2^-22 |a b| at worst
// (a = b = 1.0078) and 2^-25.5 |a b| rms over all significands, about one fp32 rounding of that product; the
// fp32 instruction rounds the growing sum instead, K times.  The bf16 products
// are exact in fp32.  The large term has an accumulator of its own (K / 32 roundings instead of the K / 4 or
// more of the fp32 instruction); the five correction terms, 2^-8 of it or less, go to a second one.
//
// An infinite operand has no such parts: its second is inf - inf = NaN, which enters the correction terms only.  The two
// accumulators are therefore added by joined(), which takes the large term alone where the corrections are NaN, so an
// infinity comes out where the fp32 instruction gives one.  (Not in the weight gradients of egnn_f32s.hip, which keep both
// in one accumulator, and not where NaN follows from SiLU(-inf) or SiLU'(inf) in any case.)
// A finite operand never becomes infinite, as x0 is truncated; a NaN whose payload has its lower 16 bits only (no arithmetic
// makes one) counts as an infinity.
#pragma once
#include "egnn_device.h"

namespace egnn {
namespace split {

// a chunk (8 values per lane) in three bf16 parts
struct Chunk3 { bf16x8 p0, p1, p2; };

__device__ __forceinline__ uint32_t fbits(float x) { return __builtin_bit_cast(uint32_t, x); }
__device__ __forceinline__ float bitsf(uint32_t u) { return __builtin_bit_cast(float, u); }

// parts of one value (weights, prepared once per call)
__device__ __forceinline__ void split1(float x, bf16& a, bf16& b, bf16& c) {
  const float x0 = bitsf(fbits(x) & 0xffff0000u);
  const float r = x - x0;
  a = (bf16)x0;
  b = (bf16)r;
  c = (bf16)(r - (float)b);
}

typedef __bf16 bf16x2_ __attribute__((ext_vector_type(2)));
// the upper halves of two values as one register, x in the low half
__device__ __forceinline__ uint32_t hi_pair(float x, float y) { return __builtin_amdgcn_perm(fbits(y), fbits(x), 0x07060302u); }

__device__ __forceinline__ Chunk3 split_chunk(const f32x4& lo, const f32x4& hi) {
  u32x4 q0, q1, q2;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float x = i < 2 ? lo[2 * i] : hi[2 * i - 4], y = i < 2 ? lo[2 * i + 1] : hi[2 * i - 3];
    q0[i] = hi_pair(x, y);
    const float rx = x - bitsf(fbits(x) & 0xffff0000u), ry = y - bitsf(fbits(y) & 0xffff0000u);
    bf16x2_ b;
    b[0] = (bf16)rx;
    b[1] = (bf16)ry;
    q1[i] = __builtin_bit_cast(uint32_t, b);
    bf16x2_ c;
    c[0] = (bf16)(rx - bitsf(q1[i] << 16));
    c[1] = (bf16)(ry - bitsf(q1[i] & 0xffff0000u));
    q2[i] = __builtin_bit_cast(uint32_t, c);
  }
  return Chunk3{__builtin_bit_cast(bf16x8, q0), __builtin_bit_cast(bf16x8, q1), __builtin_bit_cast(bf16x8, q2)};
}

// the six products of one 32-deep slice: hi += a0 b0, lo += the corrections (smallest first)
__device__ __forceinline__ void mma3(f32x4& hi, f32x4& lo, const Chunk3& a, const Chunk3& b) {
  mma(lo, a.p2, b.p0);
  mma(hi, a.p0, b.p0);
  mma(lo, a.p0, b.p2);
  mma(lo, a.p1, b.p1);
  mma(lo, a.p1, b.p0);
  mma(lo, a.p0, b.p1);
}
// the same for two row blocks, their products in turn (no product waits for the one just issued)
__device__ __forceinline__ void mma3x2(f32x4* hi, f32x4* lo, const Chunk3& a, const Chunk3& d, const Chunk3& b) {
  mma(lo[0], a.p2, b.p0);
  mma(lo[1], d.p2, b.p0);
  mma(hi[0], a.p0, b.p0);
  mma(hi[1], d.p0, b.p0);
  mma(lo[0], a.p0, b.p2);
  mma(lo[1], d.p0, b.p2);
  mma(lo[0], a.p1, b.p1);
  mma(lo[1], d.p1, b.p1);
  mma(lo[0], a.p1, b.p0);
  mma(lo[1], d.p1, b.p0);
  mma(lo[0], a.p0, b.p1);
  mma(lo[1], d.p0, b.p1);
}

// hi + lo, and hi alone where lo is NaN.  lo is NaN exactly where an infinite (or NaN) operand entered the sum, as such an
// operand has no second and third part; hi is then what the fp32 product gives.
__device__ __forceinline__ f32x4 joined(const f32x4& hi, const f32x4& lo) {
  f32x4 r;
#pragma unroll
  for (int i = 0; i < 4; ++i)
    r[i] = hi[i] + __builtin_amdgcn_fmed3f(lo[i], -3.40282347e+38f, lo[i]);   // NaN -> the finite bound: one instruction
  return r;
}

// The matrix instruction drops the low bits of its sums towards one side, so the errors of many results of one kind add up
// instead of averaging out where those are summed.  Reductions over edges or nodes therefore contract with -B in every
// other part and subtract: flip is the sign bit to change in B, sgn the factor of the part's result.  The chains of the
// edge kernels carry every other edge, and the node products every other row, with its sign changed (sg = -1): an edge's
// operand is sg y, its products come out as sg times the sum, and sg goes back in by the multiplication or the signed
// SiLU that follows, at no extra instruction.
__device__ __forceinline__ f32x4 flip_sign(const f32x4& v, uint32_t flip) {
  f32x4 r;
#pragma unroll
  for (int i = 0; i < 4; ++i) r[i] = bitsf(fbits(v[i]) ^ flip);
  return r;
}

// SiLU of the fp32 path: e^-x as 2^t (1 + d ln 2) with t = fl(-x log2 e) and d its rounding error (the
// product's by fma, and log2 e's own), so the exponential keeps the accuracy of v_exp_f32 (1 ulp) for every x.
// x is clamped in the exponent only, where the sigmoid is 0 or 1 to fp32 precision: an infinite x then gives
// no inf - inf in d (SiLU(inf) = inf, SiLU(-inf) = -inf * 0 = NaN as with expf).
// signed forms, sg = 1 or -1: sg sigmoid(x), sg SiLU(x), sg SiLU'(x)
__device__ __forceinline__ float sigmoid_f32(float x, float sg = 1.0f) {
  const float u = __builtin_amdgcn_fmed3f(x, -120.0f, 120.0f);
  const float t = u * -1.44269502e+0f;                                   // fl(log2 e)
  const float d = __builtin_fmaf(u, -1.92596303e-8f, __builtin_fmaf(u, -1.44269502e+0f, -t));
  const float e = __builtin_amdgcn_exp2f(t);
  return __builtin_amdgcn_rcpf(__builtin_fmaf(e, __builtin_fmaf(d, 0.693147182f * sg, sg), sg));   // e may be inf: rcp 0
}
__device__ __forceinline__ float silu_f32(float x, float sg = 1.0f) { return x * sigmoid_f32(x, sg); }
__device__ __forceinline__ YD silu_yd_f32(float x, float sg = 1.0f) {
  const float s = sigmoid_f32(x, sg);
  const float y = x * s;
  return YD{y, __builtin_fmaf(y, __builtin_fmaf(s, -sg, 1.0f), s)};
}
// v + sg x
__device__ __forceinline__ f32x4 add_signed(const f32x4& v, const f32x4& x, float sg) {
  f32x4 r;
#pragma unroll
  for (int i = 0; i < 4; ++i) r[i] = __builtin_fmaf(x[i], sg, v[i]);
  return r;
}

}  // namespace split
}  // namespace egnn
