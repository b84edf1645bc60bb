// What the kernels of attn_keep_window for decode rows share (mix_keep_split.hip, mix_keep_row.hip).
#pragma once
#include "common.h"
#include "mix_common.h"

namespace rfqmix {

using rfq::as_bf16x8;
using rfq::f32x4;
using rfq::s16x4;
using rfq::s16x8;

namespace {
constexpr int PG = 32;                  // tokens per page
constexpr float kNegInfS = -__builtin_huge_valf();
// The maximum that weights are taken against moves only when a score passes it by this much (weights
// stay below e^8): most turns then leave the accumulators alone.
constexpr float kDefer = 8.f;

// f as a sum of N bf16 values: three hold all 24 bits, two 16.  INF: f may be infinite, as one of them.
template <bool INF, int N>
__device__ __forceinline__ void split_parts(const float* f, s16x8 (&p)[N]) {
  float r[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) r[i] = f[i];
#pragma unroll
  for (int n = 0; n < N; ++n) {
    p[n] = rfq::pack8(r);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float h = rfq::bf2f_s(p[n][i]);
      r[i] = INF && fabsf(h) == -kNegInfS ? 0.f : r[i] - h;
    }
  }
}
template <bool EXACT>
__device__ __forceinline__ float exp_of(float x) { return EXACT ? expf(x) : __expf(x); }
// tanh to 1.6 units in the last place, without tanhf's branches (64 sequences of 300 - 900 tokens: 58.5 us a
// pass with it, 57.5 with this, 56.4 with the wide groups' form).  Below 0.7 an odd
// polynomial, fitted to a relative error of 1.6e-8; above, 1 - 2 / (exp(2 |x|) + 1).
__device__ __forceinline__ float tanh_of(float x) {
  const float u = x * x, ax = fabsf(x);
  float p = -0.0051386617f;
  p = p * u + 0.02009197f;
  p = p * u - 0.05355886f;
  p = p * u + 0.13329111f;
  p = p * u - 0.3333319f;
  const float big = 1.f - 2.f * __builtin_amdgcn_rcpf(__builtin_amdgcn_exp2f(ax * 2.88539008f) + 1.f);
  return ax < 0.7f ? x + x * u * p : copysignf(big, x);
}

// Lanes read here what others of their wave wrote to LDS.  The hardware keeps a wave's LDS accesses in
// order, this keeps the compiler's; no instruction comes of it.
__device__ __forceinline__ void wave_lds_order() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}
}  // namespace

struct KeepSplitArgs {
  const float* q;
  const bf16_t *k_cache, *v_cache;
  int64_t vrs;
  const int32_t* bt;
  int maxb;
  const int32_t *q_start, *q_len, *kv_len;
  const float* head_bias;
  const bf16_t* gate;
  int64_t gate_stride;
  int gate_w;
  bf16_t* out;
  int64_t out_stride;
  float scale, softcap, out_mult;
  int window, keep_first, sigmoid, H, G;
};

// Decode rows of groups of up to eight heads (mix_keep_row.hip): T rows of NA sequences, no more than these.
bool keep_row_ok(int T, int NA, int H, int G, int E, int vdim, bool shared);
void launch_attn_keep_row(const KeepSplitArgs& a, int T, int NA, int E, hipStream_t s);

}  // namespace rfqmix
