// fp32 operands on the bf16 matrix cores.
#pragma once
#include "common.h"

namespace rfqmix {

// fp32 as a sum of three bf16, h + m + l, each the rounding of what is left: the sum is exact (8 bits each and two signs).
// Products of two such sums without m l, l m (up to 2^-25 of the whole product each) and l l, together up to 2^-24, fp32's own
// rounding, and a quarter of that on the average, take six products on the matrix cores, 2.7 times the rate of fp32 MFMA and,
// other than those, beside the vector instructions of other waves.  Packed in twos: a in the low half.
struct Split2 {
  uint32_t h, m, l;
};
__device__ __forceinline__ float lo_f(uint32_t x) { return __uint_as_float(x << 16); }
__device__ __forceinline__ float hi_f(uint32_t x) { return __uint_as_float(x & 0xffff0000u); }
__device__ __forceinline__ Split2 split3(float a, float b) {
  Split2 s;
  s.h = rfq::pack_bf16x2(a, b);
  a -= lo_f(s.h);
  b -= hi_f(s.h);
  s.m = rfq::pack_bf16x2(a, b);
  s.l = rfq::pack_bf16x2(a - lo_f(s.m), b - hi_f(s.m));
  return s;
}
// Sums of sizes from here on are not for products of parts: above 2^127 h itself may round to infinity, and a product of two
// h may pass the end of fp32 where that of the values does not (both 2^64 - 2^55).
constexpr float kSplitMost = 0x1p60f;
// Nor are sums below this that are not zero: bf16 end at 2^-133, and the third part of values below 2^-110 is cut there.
// What is lost, 2^-134 of an entry, is nothing beside the rest of a sum that is not as small (1e-36 for all entries of a
// product: 2.7e-5 of the result, from there on 2^-38).
constexpr float kSplitLeast = 0x1p-96f;
__device__ __forceinline__ bool split_fits(float sum) { return (sum < kSplitMost) & ((sum >= kSplitLeast) | (sum == 0.f)); }
__device__ __forceinline__ rfq::f32x4 mma32(const uint4& a, const uint4& b, const rfq::f32x4& c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(rfq::bf16x8, a), __builtin_bit_cast(rfq::bf16x8, b), c, 0, 0, 0);
}

}  // namespace rfqmix
