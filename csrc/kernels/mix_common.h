// Helpers of the layer-list models' kernels (mix_*.hip; library _C_mix.so).
//
// These kernels are templated on the activation type: bf16 (raw bits) for a model served
// in bf16, float for one served in full precision.  Norms, scores, softmax, the residual
// stream and the convolution state are fp32 in both.
#pragma once
#include <hip/hip_runtime.h>
#include <hip/hip_bf16.h>
#include <stdint.h>

namespace rfqmix {

typedef uint16_t bf16_t;

__device__ __forceinline__ float ldf(const float* p) { return *p; }
__device__ __forceinline__ float ldf(const bf16_t* p) {
  return __uint_as_float(((uint32_t)*p) << 16);
}
__device__ __forceinline__ void stf(float* p, float v) { *p = v; }
__device__ __forceinline__ void stf(bf16_t* p, float v) {
  __hip_bfloat16 b = __float2bfloat16(v);               // round to nearest even
  *p = __builtin_bit_cast(bf16_t, b);
}

__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}
__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o, 64));
  return v;
}

// 64 lanes' pieces of 16 bytes from base + offset (per lane) to LDS, one after another from byte `to` (the same for
// the wave) on.  Written out: behind the builtin the compiler waits for the copy before any later LDS read through a
// builtin.  The caller waits with s_waitcnt vmcnt(0).  M0 is named as overwritten, so that a builtin's copy behind it
// sets its own; the compiler warns of such a name because it saves no value there, and none is kept in M0 across.
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
__device__ __forceinline__ void lds_copy16(const void* base, uint32_t offset, uint32_t to) {
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1"
               ::"v"(offset), "s"(base), "s"(__builtin_amdgcn_readfirstlane(to)) : "memory", "m0");
#endif
}
#pragma clang diagnostic pop

// Sum over each aligned group of L neighbouring lanes (L = 4, 8, .. 64, the same for the whole wave);
// every lane of the group receives it.  The first four steps stay inside a row of 16 lanes.
__device__ __forceinline__ float group_sum(float v, int L) {
  v += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0xB1, 0xf, 0xf, true));              // lanes 1 0 3 2
  v += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x4E, 0xf, 0xf, true));              // lanes 2 3 0 1
  if (L > 4) v += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x141, 0xf, 0xf, true));  // half rows mirrored
  if (L > 8) v += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x140, 0xf, 0xf, true));  // rows mirrored
  if (L > 16) v += __shfl_xor(v, 16, 64);
  if (L > 32) v += __shfl_xor(v, 32, 64);
  return v;
}

// four neighbouring entries, 16- or 8-byte aligned
__device__ __forceinline__ float4 ld4(const float* p) { return *reinterpret_cast<const float4*>(p); }
__device__ __forceinline__ float4 ld4(const bf16_t* p) {
  const uint2 w = *reinterpret_cast<const uint2*>(p);
  return make_float4(__uint_as_float(w.x << 16), __uint_as_float(w.x & 0xffff0000u),
                     __uint_as_float(w.y << 16), __uint_as_float(w.y & 0xffff0000u));
}
__device__ __forceinline__ void st4(float* p, float4 v) { *reinterpret_cast<float4*>(p) = v; }
__device__ __forceinline__ void st4(bf16_t* p, float4 v) {
  union { bf16_t h[4]; uint2 w; } u;
  stf(u.h, v.x);
  stf(u.h + 1, v.y);
  stf(u.h + 2, v.z);
  stf(u.h + 3, v.w);
  *reinterpret_cast<uint2*>(p) = u.w;
}

// exp(x) for x <= 87, to about a unit in the last place: v_exp_f32 takes base 2, and the product's rounding,
// which grows with |x|, and the rest of log2 e follow as a factor near one.  Below e^-200: 0.  NaN stays NaN.
__device__ __forceinline__ float exp_c(float x) {
  x = x < -200.f ? -200.f : x;
  const float t = x * 1.44269502f, e = __builtin_amdgcn_exp2f(t);
  const float rest = fmaf(x, 1.92596299e-8f, fmaf(x, 1.44269502f, -t));
  return fmaf(e * 0.693147181f, rest, e);
}
// log(1 + e^y): log(1 + e) = 2 atanh(e / (2 + e)), the odd series fitted to a relative error of 5e-9
__device__ __forceinline__ float softplus_c(float y) {
  const float e = exp_c(-fabsf(y)), d = 2.f + e, r = __builtin_amdgcn_rcpf(d), s0 = e * r;
  const float s = fmaf(fmaf(-s0, d, e), r, s0), u = s * s;
  const float p = fmaf(fmaf(fmaf(0.140123978f, u, 0.139995337f), u, 0.200108513f), u, 0.333332062f);
  return fmaf(2.f, fmaf(s * u, p, s), fmaxf(y, 0.f));
}
__device__ __forceinline__ float sigmoid_c(float x) { return 1.0f / (1.0f + exp_c(x < -87.f ? 87.f : -x)); }

// Block-wide sum for blockDim.x a multiple of 64, at most 1024.  scratch >= 16 floats.
__device__ __forceinline__ float block_sum(float v, float* scratch) {
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const int nw = (blockDim.x + 63) >> 6;
  v = wave_sum(v);
  if (lane == 0) scratch[wid] = v;
  __syncthreads();
  float t = (lane < nw) ? scratch[lane] : 0.f;
  t = wave_sum(t);
  __syncthreads();
  return t;
}

}  // namespace rfqmix
