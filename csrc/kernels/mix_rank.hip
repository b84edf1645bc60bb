// Y[M, N] = X[M, K] . W[N, K]^T for short K (32, 64, 96 or 128; bf16 operands, fp32 sums, Y in bf16 or
// fp32): the second factor of a low-rank projection.
//
// For products where a launch and the host's work before it are what counts: an eager call takes 5 us
// against the library's 19, which bounded a decode step (64 rows of a delta rule layer: 64.7 -> 49.1 us
// a pass).  The lines lie where the device's time, all that a graph sees, is the library's: 2^21 entries
// (512 x 4,096, 4,096 x 512, 64 x 32,768: K = 32 3.1 - 3.9 us against 4.3 - 5.0, 64 4.6 - 5.3 against
// 4.6 - 5.6, 96 4.3 - 5.1 against 4.7 - 5.9), 2^20 for K = 128 (64 x 16,384 in bf16 4.3 us on both sides,
// at 2^21 6.7 against 4.9).  4,096 rows of 2,048 columns, K = 64: 15.4 us against 12.7.
//
// No LDS: a wave has the W rows of 64 columns, all K of them, and 16 rows of X straight from memory in
// 16-byte pieces.  Y comes out transposed in the accumulators (A = W, B = X), so a lane holds
// neighbouring entries of a row.
#include "common.h"
#include "mix_common.h"

namespace rfqmix {

using rfq::as_bf16x8;
using rfq::f32x4;
using rfq::s16x8;

template <typename TO, int KS>
__global__ __launch_bounds__(256) void rank_product_kernel(const bf16_t* __restrict__ x, int64_t xs,
                                                           const bf16_t* __restrict__ w, int64_t ws,
                                                           TO* __restrict__ y, int M, int N) {
  const int lane = threadIdx.x & 63, col = lane & 15, grp = lane >> 4;
  const int n0 = (blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6)) * 64;
  if (n0 >= N) return;
  // tile i's rows: fp32, the 16 columns from 16 i on, 64 bytes of a row per store; bf16, four columns
  // of each 16, so that a lane's four tiles are 16 neighbouring columns
  constexpr bool WIDE = sizeof(TO) == 2;
  s16x8 a[4][KS];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int n = n0 + (WIDE ? 16 * (col >> 2) + 4 * i + (col & 3) : 16 * i + col);
    const bf16_t* wr = w + (int64_t)min(n, N - 1) * ws + grp * 8;
#pragma unroll
    for (int k = 0; k < KS; ++k) a[i][k] = *reinterpret_cast<const s16x8*>(wr + 32 * k);
  }
  const int m = blockIdx.y * 16 + col;
  const bf16_t* xr = x + (int64_t)min(m, M - 1) * xs + grp * 8;
  f32x4 c[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) c[i] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int k = 0; k < KS; ++k) {
    const s16x8 b = *reinterpret_cast<const s16x8*>(xr + 32 * k);
#pragma unroll
    for (int i = 0; i < 4; ++i)
      c[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(a[i][k]), as_bf16x8(b), c[i], 0, 0, 0);
  }
  if (m >= M) return;
  TO* const to = y + (int64_t)m * N;
  const int nl = n0 + 16 * grp;
  if (WIDE && N % 8 == 0 && nl + 15 < N) {
#pragma unroll
    for (int i = 0; i < 4; i += 2) {
      const float f[8] = {c[i][0], c[i][1], c[i][2], c[i][3], c[i + 1][0], c[i + 1][1], c[i + 1][2], c[i + 1][3]};
      *reinterpret_cast<s16x8*>(to + nl + 4 * i) = rfq::pack8(f);
    }
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int n = WIDE ? nl + 4 * i : n0 + 16 * i + 4 * grp;        // N is a multiple of four
      if (n < N) st4(to + n, make_float4(c[i][0], c[i][1], c[i][2], c[i][3]));
    }
  }
}

// ------------------------------------------------------------------ launcher
bool rank_product_ok(int64_t M, int64_t N, int64_t K) {
  return M >= 1 && K >= 32 && K <= 128 && K % 32 == 0 && N >= 4 && N % 4 == 0 && M <= (1 << (K > 96 ? 20 : 21)) / N;
}

void launch_rank_product(bool out_f32, const void* x, int64_t xs, const void* w, int64_t ws, void* y, int M, int N,
                         int K, hipStream_t s) {
  const dim3 grid((N + 255) / 256, (M + 15) / 16);         // at most 2^15 blocks of rows
#define RANK_GO(TO, KS)                                                                                       \
  hipLaunchKernelGGL((rank_product_kernel<TO, KS>), grid, dim3(256), 0, s, (const bf16_t*)x, xs, (const bf16_t*)w, \
                     ws, (TO*)y, M, N)
#define RANK_ALL(TO)                \
  do {                              \
    if (K == 32) RANK_GO(TO, 1);    \
    else if (K == 64) RANK_GO(TO, 2); \
    else if (K == 96) RANK_GO(TO, 3); \
    else RANK_GO(TO, 4);            \
  } while (0)
  if (out_f32) RANK_ALL(float);
  else RANK_ALL(bf16_t);
#undef RANK_ALL
#undef RANK_GO
}

}  // namespace rfqmix
