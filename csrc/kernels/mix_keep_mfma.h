// What the kernels of attn_keep_window on MFMA tiles share (mix_keep_attn_mfma.hip, mix_keep_latent.hip,
// mix_keep_streams.hip).
#pragma once
#include <utility>

#include "common.h"
#include "mix_common.h"

namespace rfqmix {

using rfq::as_bf16x8;
using rfq::f32x16;
using rfq::u32x4;
using rfq::f32x4;
using rfq::s16x4;
using rfq::s16x8;

namespace {
constexpr int WQB = 32;                 // queries per work item
constexpr int WBS = 32;                 // keys per tile = page size
constexpr float kNegInfW = -__builtin_huge_valf();
constexpr float kLog2e = 1.44269504088896f;
constexpr float kDeferW = 11.f;         // base 2

__device__ __forceinline__ void split_bf16w(const float* f, s16x8& hi, s16x8& lo) {
  float r[8];
  hi = rfq::pack8(f);
#pragma unroll
  for (int i = 0; i < 8; ++i) r[i] = f[i] - rfq::bf2f_s(hi[i]);
  lo = rfq::pack8(r);
}

// the value of the lane 32 away beside one's own
__device__ __forceinline__ float other_half_max(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float both_halves_sum(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
// the same over lanes 16 away
__device__ __forceinline__ float other_row_max(float x) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float both_rows_sum(float x) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

}  // namespace

struct KeepArgs {
  const float* q;
  const void *k_cache, *v_cache;
  int64_t vrs;
  const int32_t* bt;
  int maxb;
  const int32_t *q_start, *q_len, *kv_len, *work_seq, *work_qblk;
  int W;
  const float* head_bias;
  const void* gate;
  int64_t gate_stride;
  int gate_w;
  void* out;
  int64_t out_stride;
  float scale;
  int window, keep_first;
  bool sigmoid;
  int H, G;
  float softcap, out_mult;
  hipStream_t s;
  bool turned = false;                             // attn_keep_tile_kernel: a block's heads begin where the block says
};

__device__ __forceinline__ uint32_t lds_byte(const unsigned char* smem) {      // where the dynamic LDS begins
  return (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const unsigned char*)smem;
}

// f(0), f(1) .. f(N - 1) with constants: loops whose bodies have loops over parts of their index are unrolled for sure
template <int... I, typename F>
__device__ __forceinline__ void each_of(std::integer_sequence<int, I...>, F f) { (f(std::integral_constant<int, I>{}), ...); }
template <int N, typename F>
__device__ __forceinline__ void each(F f) { each_of(std::make_integer_sequence<int, N>{}, f); }

// lane (col, half) of a 32 x 32 tile holds value channels 32 m + 8 b + 4 half .. + 3 of its query: 8-byte stores.
// Tiles from channel c0 of vdim on, times mul and a gate per output.
template <int N>
__device__ __forceinline__ void store_tiles32(const KeepArgs& a, const f32x16 (&o)[N], float mul, int64_t t, int hh,
                                              int vdim, int c0, int half, bool qlive) {
  if (!qlive) return;
  const bf16_t* gate = static_cast<const bf16_t*>(a.gate);
  // a gate column per output: four neighbouring logits, 8-byte reads
  const int64_t at = (int64_t)hh * vdim + c0 + half * 4;
  const bool gated = gate != nullptr && a.gate_w > 1;
  const bf16_t* grow = gate + (gated ? t * a.gate_stride + at : 0);
  bf16_t* orow = static_cast<bf16_t*>(a.out) + t * a.out_stride + at;
#pragma unroll
  for (int m = 0; m < N; ++m)
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      float y[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) y[i] = o[m][4 * b + i] * mul;
      if (gated) {
        const uint2 gu = *reinterpret_cast<const uint2*>(grow + m * 32 + b * 8);
        y[0] /= 1.0f + __expf(-__uint_as_float(gu.x << 16));
        y[1] /= 1.0f + __expf(-__uint_as_float(gu.x & 0xffff0000u));
        y[2] /= 1.0f + __expf(-__uint_as_float(gu.y << 16));
        y[3] /= 1.0f + __expf(-__uint_as_float(gu.y & 0xffff0000u));
      }
      *reinterpret_cast<uint2*>(orow + m * 32 + b * 8) = make_uint2(rfq::pack_bf16x2(y[0], y[1]), rfq::pack_bf16x2(y[2], y[3]));
    }
}

// What a query's weighted values are multiplied by, given the sum of its weights: a gate per head.
template <int MODE>
__device__ __forceinline__ float row_factor(const KeepArgs& a, float l, int64_t t, int hh) {
  const bf16_t* gate = static_cast<const bf16_t*>(a.gate);
  float mul = MODE >= 2 ? a.out_mult : (l > 0.f ? a.out_mult / l : 0.f);
  if (gate != nullptr && a.gate_w == 1) mul /= 1.0f + __expf(-ldf(gate + t * a.gate_stride + hh));
  return mul;
}

// Rows of 320 and 576 entries lie unpadded in LDS, 16-byte pieces permuted inside each 128 bytes.
// Pieces that one LDS access takes together then lie on different banks: of a K read rows 0..3 and 12..15 of one
// piece with rows 4..11 of its neighbour, or the other way round (sixteen rows of one piece are not what it takes: a
// permutation that parts those alone cost 1,150 clocks a page of eight waves), of a transposed V read four
// neighbouring rows of a pair of pieces beside the next four.  The row's parity picks a half of the banks, bit 1 the
// half of that, the row's quad the order inside it.
__device__ __forceinline__ int wide_swizzle(int r) { return ((r >> 1) & 1) << 2 | ((4 - (r >> 2)) & 3); }

// prompt rows over 576-wide latents with 512 values, four heads a workgroup (mix_keep_latent.hip)
void launch_attn_keep_latent(const KeepArgs& a);

}  // namespace rfqmix
