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
#include <algorithm>
#include <type_traits>

#include "common.h"
#include "mix_common.h"
#include "mix_split.h"

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

// The same in fp32, X, W and Y.  Up to 64 terms an eager call takes 8 us for the library's 19, and the device's time is no
// longer either (K = 64: 64 x 2,048 3.2 us for 4.3, 1,000 x 2,048 6.8 for 7.2, 2,067 x 2,048 10.7 for 30.5, 4,096 x 4,096
// 23.9 for 31.0, 4,096 x 8,192 35.3 for 54.8; 4,096 x 1,024, the worst of 34 sizes, 11.3 for 11.1).  With more terms the
// library's tiles are better above 2^18 entries (1,000 x 2,048, K = 96 9.0 us for 13.1) and along sides beyond 2^14 (K = 128,
// 4 x 65,536 7.3 for 9.0).  Error against 64 bits: 4.6e-8 for the library's 1.4e-7 (K = 64).
// By operands of three bf16 parts (split3): six products on the matrix cores take 96 clocks for the 256
// that fp32 MFMA hold the vector unit.  A wave keeps its 16 NT columns' W rows as parts and goes through `blocks` times 16 rows
// of X, the next ones on their way meanwhile.  Infinities, NaN and rows too large or too small for products of parts go
// through fp32 MFMA.
template <int KS, int NT>
__global__ __launch_bounds__(256) void rank_product_f32_kernel(const float* __restrict__ x, int64_t xs, const float* __restrict__ w,
                                                               int64_t ws, float* __restrict__ y, int M, int N, int blocks) {
  const int lane = threadIdx.x & 63, col = lane & 15, grp = lane >> 4;
  const int n0 = (blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6)) * (16 * NT);
  if (n0 >= N) return;
  float4 next[2 * KS];                                       // a lane's K entries: 32 k + 8 grp ..
  auto parts = [](const float4& p, const float4& q, uint4 (&to)[3]) {
    const Split2 s0 = split3(p.x, p.y), s1 = split3(p.z, p.w), s2 = split3(q.x, q.y), s3 = split3(q.z, q.w);
    to[0] = make_uint4(s0.h, s1.h, s2.h, s3.h);
    to[1] = make_uint4(s0.m, s1.m, s2.m, s3.m);
    to[2] = make_uint4(s0.l, s1.l, s2.l, s3.l);
    return ((fabsf(p.x) + fabsf(p.y)) + (fabsf(p.z) + fabsf(p.w))) + ((fabsf(q.x) + fabsf(q.y)) + (fabsf(q.z) + fabsf(q.w)));
  };
  auto fetch = [&](int m) {
    const float* xr = x + (int64_t)min(m, M - 1) * xs + 8 * grp;
#pragma unroll
    for (int k = 0; k < 2 * KS; ++k) next[k] = ld4(xr + 32 * (k >> 1) + 4 * (k & 1));
  };
  const int first = blockIdx.y * blocks * 16 + col;
  fetch(first);
  uint4 a[NT][KS][3];
  bool fits = true;
#pragma unroll
  for (int i = 0; i < NT; ++i) {
    const float* wr = w + (int64_t)min(n0 + 16 * i + col, N - 1) * ws + 8 * grp;
    float size = 0.f;
#pragma unroll
    for (int k = 0; k < KS; ++k) size += parts(ld4(wr + 32 * k), ld4(wr + 32 * k + 4), a[i][k]);
    fits &= split_fits(size);
  }
  for (int t = 0; t < blocks; ++t) {
    const int m = first + 16 * t;
    uint4 b[KS][3];
    float size = 0.f;
#pragma unroll
    for (int k = 0; k < KS; ++k) size += parts(next[2 * k], next[2 * k + 1], b[k]);
    if (t + 1 < blocks) fetch(m + 16);
    f32x4 c[NT];
#pragma unroll
    for (int i = 0; i < NT; ++i) c[i] = (f32x4){0.f, 0.f, 0.f, 0.f};
    if (__builtin_amdgcn_ballot_w64(!(fits & split_fits(size))) == 0ull) {
      auto product = [&](int p, int q) {                     // the small ones first
#pragma unroll
        for (int k = 0; k < KS; ++k)
#pragma unroll
          for (int i = 0; i < NT; ++i) c[i] = mma32(a[i][k][p], b[k][q], c[i]);
      };
      product(2, 0);
      product(0, 2);
      product(1, 1);
      product(1, 0);
      product(0, 1);
      product(0, 0);
    } else {
      const float* xr = x + (int64_t)min(m, M - 1) * xs + 4 * grp;
#pragma unroll 1
      for (int k = 0; k < 32 * KS; k += 16) {
        const float4 xv = ld4(xr + k);
#pragma unroll
        for (int i = 0; i < NT; ++i) {
          const float4 wv = ld4(w + (int64_t)min(n0 + 16 * i + col, N - 1) * ws + 4 * grp + k);
          c[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(wv.x, xv.x, c[i], 0, 0, 0);
          c[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(wv.y, xv.y, c[i], 0, 0, 0);
          c[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(wv.z, xv.z, c[i], 0, 0, 0);
          c[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(wv.w, xv.w, c[i], 0, 0, 0);
        }
      }
    }
    if (m < M) {
      float* const to = y + (int64_t)m * N + n0 + 4 * grp;
#pragma unroll
      for (int i = 0; i < NT; ++i)
        if (n0 + 16 * i + 4 * grp < N) st4(to + 16 * i, make_float4(c[i][0], c[i][1], c[i][2], c[i][3]));   // N: a multiple of four
    }
  }
}

// Y[b] = X[b] . W[b] for a batch, W[b] [K, N] as it lies, bf16 operands, Y in fp32: queries of decode rows carried into a
// latent space, head by head, into slices of wider rows.  A wave makes 16 rows of 64 columns: their W passes through its
// piece of LDS, 64 terms at a time, and is read back transposed.  What bounds it: launch and three trips to memory, 4 - 5 us;
// the library's takes 5 - 6 and 18 us of the host, 9 here, which bounded a decode step (64 rows of 32 heads, 128 to
// 512: 5.6 -> 4.7 us, the pass 49 -> 41).  Up to 2^20 results (64 heads 7.9 us for the library's 6.8).
template <int KS>
__global__ __launch_bounds__(256) void batch_product_kernel(const bf16_t* __restrict__ x, int64_t xb, int64_t xs,
                                                            const bf16_t* __restrict__ w, int64_t wb, int64_t ws,
                                                            float* __restrict__ y, int64_t yb, int64_t ys, int M, int N) {
  constexpr int WR = 64 + 8, KH = KS < 2 ? 32 : 64;          // shorts per row in LDS, rows
  __shared__ __attribute__((aligned(16))) short slab[4][KH * WR];
  const int lane = threadIdx.x & 63, col = lane & 15, grp = lane >> 4, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n0 = (blockIdx.x * 4 + wave) * 64;
  if (n0 >= N) return;
  x += blockIdx.z * xb;
  w += blockIdx.z * wb + n0;
  y += blockIdx.z * yb + n0;
  const int m = blockIdx.y * 16 + col;
  const bf16_t* xr = x + (int64_t)min(m, M - 1) * xs + 8 * grp;
  s16x8 b[KS];
#pragma unroll
  for (int k = 0; k < KS; ++k) b[k] = *reinterpret_cast<const s16x8*>(xr + 32 * k);
  s16x8 a[4][KS];
  short* S = slab[wave];
#pragma unroll
  for (int h = 0; h < KS; h += 2) {
    constexpr int pieces = KH / 8;                           // eight rows to a load of the wave
    s16x8 raw[pieces];
#pragma unroll
    for (int i = 0; i < pieces; ++i)
      if (h * 32 + 8 * i < KS * 32)
        raw[i] = *reinterpret_cast<const s16x8*>(w + (int64_t)(h * 32 + 8 * i + (lane >> 3)) * ws + 8 * (lane & 7));
#pragma unroll
    for (int i = 0; i < pieces; ++i)
      if (h * 32 + 8 * i < KS * 32) *reinterpret_cast<s16x8*>(S + (8 * i + (lane >> 3)) * WR + 8 * (lane & 7)) = raw[i];
    // a wave's LDS accesses are in order: this keeps the compiler's
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
    for (int k = h; k < h + 2 && k < KS; ++k)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const short* p = S + (32 * (k - h) + 8 * grp + (col >> 2)) * WR + 16 * i + 4 * (col & 3);
        const rfq::s16x4 lo = rfq::ds_read_tr16(p), hi = rfq::ds_read_tr16(p + 4 * WR);
        a[i][k] = (s16x8){lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
      }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  }
  f32x4 c[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) c[i] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int k = 0; k < KS; ++k)
#pragma unroll
    for (int i = 0; i < 4; ++i)
      c[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(a[i][k]), as_bf16x8(b[k]), c[i], 0, 0, 0);
  if (m >= M) return;
  float* const to = y + (int64_t)m * ys + 4 * grp;
#pragma unroll
  for (int i = 0; i < 4; ++i) st4(to + 16 * i, make_float4(c[i][0], c[i][1], c[i][2], c[i][3]));
}

// The same for many rows: a wave keeps its 64 columns' W and goes through blocks of 16 rows, every gridDim.y-th, the next
// one's X on its way meanwhile; the workgroup's columns of a block leave by way of LDS, 1 KB to an access, many results past the
// caches (PAST).
// What bounds it: the results' bytes.  32 heads, 8,192 rows, 128 to 512 (537 MB): 97 us, 5.5 TB/s, as fast as they can be
// filled with a number (102); the library's product 153.  Stored as the tiles lie, 64 bytes of 16 rows to an access, 206; 256
// bytes of a row 171; 1 KB 158; past the caches 97.  2,067 rows 30.2 for 43.1, 1,031 18.3 for 23.1, 600 13.6 for 15.4.
constexpr int kBatchWaves = 8;
template <int KS, bool PAST>
__global__ __launch_bounds__(64 * kBatchWaves, 4) void batch_rows_kernel(const bf16_t* __restrict__ x, int64_t xb, int64_t xs,
                                                                         const bf16_t* __restrict__ w, int64_t wb, int64_t ws,
                                                                         float* __restrict__ y, int64_t yb, int64_t ys, int M) {
  constexpr int WR = 64 + 8;                                 // shorts per row of a wave's W in LDS
  extern __shared__ __attribute__((aligned(16))) float blocks[];     // [2][16][columns + 4]
  const int lane = threadIdx.x & 63, col = lane & 15, grp = lane >> 4, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int nthr = blockDim.x, n0 = blockIdx.x * nthr, FR = nthr + 4;      // a column per thread
  x += blockIdx.z * xb;
  w += blockIdx.z * wb + n0 + 64 * wave;
  y += blockIdx.z * yb + n0;
  auto fetch = [&](s16x8 (&b)[KS], int m) {
    const bf16_t* xr = x + (int64_t)min(m + col, M - 1) * xs + 8 * grp;
#pragma unroll
    for (int k = 0; k < KS; ++k) b[k] = *reinterpret_cast<const s16x8*>(xr + 32 * k);
  };
  const int step = 16 * gridDim.y;
  s16x8 b[KS];
  fetch(b, 16 * blockIdx.y);
  s16x8 a[4][KS];
  short* S = reinterpret_cast<short*>(blocks) + wave * 32 * WR;
#pragma unroll
  for (int k = 0; k < KS; ++k) {
    s16x8 raw[4];                                            // eight rows to a load of the wave
#pragma unroll
    for (int i = 0; i < 4; ++i)
      raw[i] = *reinterpret_cast<const s16x8*>(w + (int64_t)(k * 32 + 8 * i + (lane >> 3)) * ws + 8 * (lane & 7));
#pragma unroll
    for (int i = 0; i < 4; ++i) *reinterpret_cast<s16x8*>(S + (8 * i + (lane >> 3)) * WR + 8 * (lane & 7)) = raw[i];
    // a wave's LDS accesses are in order: this keeps the compiler's
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const short* p = S + (8 * grp + (col >> 2)) * WR + 16 * i + 4 * (col & 3);
      const rfq::s16x4 lo = rfq::ds_read_tr16(p), hi = rfq::ds_read_tr16(p + 4 * WR);
      a[i][k] = (s16x8){lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  }
  __syncthreads();                                           // every wave has its W: blocks take its place
  int buf = 0, m = 16 * blockIdx.y;
  auto block = [&](auto whole) {
    f32x4 c[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) c[i] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int k = 0; k < KS; ++k)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        c[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(a[i][k]), as_bf16x8(b[k]), c[i], 0, 0, 0);
    float* const F = blocks + buf * 16 * FR;
#pragma unroll
    for (int i = 0; i < 4; ++i) *reinterpret_cast<f32x4*>(F + col * FR + 64 * wave + 16 * i + 4 * grp) = c[i];
    if constexpr (whole) fetch(b, m + step);                 // past the last row: that one again
    __syncthreads();
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int p = threadIdx.x + j * nthr, r = p / (nthr / 4), e = (p - r * (nthr / 4)) * 4;
      f32x4* const to = reinterpret_cast<f32x4*>(y + (int64_t)(m + r) * ys + e);
      const f32x4 v = *reinterpret_cast<const f32x4*>(F + r * FR + e);
      if (!whole && m + r >= M) continue;
      if constexpr (PAST) __builtin_nontemporal_store(v, to);
      else *to = v;
    }
  };
  // only whole blocks in the loop: behind a store that may be left out the compiler waits for all of them, not for X alone
  for (; m + 16 <= M; m += step, buf ^= 1) block(std::true_type{});
  if (m < M) block(std::false_type{});
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

bool rank_product_f32_ok(int64_t M, int64_t N, int64_t K) {
  return M >= 1 && M <= 1 << (K > 64 ? 14 : 20) && K >= 32 && K <= 128 && K % 32 == 0 && N >= 4 && N % 4 == 0 &&
         (K <= 64 || N <= 1 << 14) && M <= (1 << (K > 64 ? 18 : 26)) / N;
}

void launch_rank_product_f32(const float* x, int64_t xs, const float* w, int64_t ws, float* y, int M, int N, int K, hipStream_t s) {
  // Tiles of 16 x 16 in one round of a wave to every SIMD where up to sixteen blocks of rows a wave allow it: a wave splits
  // its columns' W once, so 16 (K above 64: registers), 32 or 64 columns by what a wave then has, and as few blocks as
  // make the round.  K = 64, the library's times beside: 1,000 x 2,048 (columns 32, blocks 4) 6.7 us of the device for 7.2,
  // 300 x 4,096 (32, 3) 5.6 for 6.9, 2,067 x 2,048 (64, 5) 11 for 31, 65,536 x 16 (16, 4) 5.4 for 6.1, 4 x 2^20 48 for 75.
  // By waves alone, with blocks in place of rows that are not there: 8.6, 7.0, 12.7, 7.3 and 177.
  const int64_t tx = (N + 15) / 16, ty = (M + 15) / 16, want = tx * ty / 1024;
  const int nt = K > 64 || tx < 2 || want < 2 ? 1 : tx < 4 || want <= 8 ? 2 : 4;
  const int64_t across = (tx + nt - 1) / nt, down = std::max<int64_t>(1, 1024 / across);     // waves
  const int blocks = (int)std::min<int64_t>(16, (ty + down - 1) / down);
  const dim3 grid((N + 64 * nt - 1) / (64 * nt), (M + 16 * blocks - 1) / (16 * blocks));
#define RANK_GO(KS, NT) \
  hipLaunchKernelGGL((rank_product_f32_kernel<KS, NT>), grid, dim3(256), 0, s, x, xs, w, ws, y, M, N, blocks)
#define RANK_ALL(KS)              \
  do {                            \
    if (nt == 1) RANK_GO(KS, 1);  \
    else if (nt == 2) RANK_GO(KS, 2); \
    else RANK_GO(KS, 4);          \
  } while (0)
  if (K == 32) RANK_ALL(1);
  else if (K == 64) RANK_ALL(2);
  else if (K == 96) RANK_GO(3, 1);
  else RANK_GO(4, 1);
#undef RANK_ALL
#undef RANK_GO
}

// Up to 2^20 results a launch is what counts.  Above, the kernel for many rows is slower than the library's in two places,
// measured from 1 to 128 matrices, 64 to 4,096 columns, 64 to 8,192 rows: 128 terms with fewer rows or results than repay W's
// way into registers (32 x 512 columns, 300 rows 10.2 us for 9.4, 500 14.6 for 13.7, 700 17.2 for 17.1, 800 18.1 for 20.3;
// 16 x 512, 900 rows 12.7 for 11.0, 1,031 13.3 for 15.0; 8 x 512, 1,500 rows 10.4 for 9.8, 2,067 13.0 for 14.8; 64 x 512, 100
// rows 8.5 for 8.2, 500 19.9 for 20.3), and results of 2 GB (630 for 593).
static bool few_results(int64_t B, int64_t M, int64_t N) { return M <= (1 << 20) / N && B <= (1 << 20) / (M * N); }
bool batch_product_ok(int64_t B, int64_t M, int64_t N, int64_t K) {
  if (!(B >= 1 && B <= 65535 && M >= 1 && N >= 64 && N % 64 == 0 && N <= 1 << 20 && K >= 32 && K <= 128 && K % 32 == 0)) return false;
  return few_results(B, M, N) || (M <= (1 << 28) / N && B <= (1 << 28) / (M * N) && (K <= 96 || (M >= 500 && B * M * N > 1 << 23)));
}

void launch_batch_product(const void* x, int64_t xb, int64_t xs, const void* w, int64_t wb, int64_t ws, float* y, int64_t yb,
                          int64_t ys, int B, int M, int N, int K, hipStream_t s) {
  if (!few_results(B, M, N)) {
    // a workgroup of eight waves to a CU: two take 107 us for the 97
    int waves = kBatchWaves;
    while (N / 64 % waves != 0) --waves;
    const int across = N / 64 / waves;
    const int64_t down = std::max<int64_t>(1, 256 * kBatchWaves / waves / ((int64_t)across * B));
    const dim3 g2(across, std::min<int64_t>((M + 15) / 16, down), B);
    const size_t lds = std::max<size_t>((size_t)2 * 16 * (64 * waves + 4) * 4, (size_t)waves * 32 * 72 * 2);
    // more than half of the last cache holds go past it; of fewer the next kernel reads some there (a layer's passes with 64 -
    // 200 MB of results are 0 - 2 % shorter so, those with more 0 - 1.5 % longer)
    const bool past = (int64_t)B * M * N > 1 << 25;
#define ROWS_AS(KS, PAST)                                                                                                        \
  do {                                                                                                                           \
    static bool attr = false;                                                                                                    \
    if (!attr) {                                                                                                                 \
      (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&batch_rows_kernel<KS, PAST>),                                     \
                                hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);                                         \
      attr = true;                                                                                                               \
    }                                                                                                                            \
    hipLaunchKernelGGL((batch_rows_kernel<KS, PAST>), g2, dim3(64 * waves), lds, s, (const bf16_t*)x, xb, xs, (const bf16_t*)w, wb, \
                       ws, y, yb, ys, M);                                                                                        \
  } while (0)
#define ROWS_GO(KS) do { if (past) ROWS_AS(KS, true); else ROWS_AS(KS, false); } while (0)
    if (K == 32) ROWS_GO(1);
    else if (K == 64) ROWS_GO(2);
    else if (K == 96) ROWS_GO(3);
    else ROWS_GO(4);
#undef ROWS_GO
#undef ROWS_AS
    return;
  }
  const dim3 grid((N + 255) / 256, (M + 15) / 16, B);
#define BATCH_GO(KS)                                                                                                    \
  hipLaunchKernelGGL((batch_product_kernel<KS>), grid, dim3(256), 0, s, (const bf16_t*)x, xb, xs, (const bf16_t*)w, wb, \
                     ws, y, yb, ys, M, N)
  if (K == 32) BATCH_GO(1);
  else if (K == 64) BATCH_GO(2);
  else if (K == 96) BATCH_GO(3);
  else BATCH_GO(4);
#undef BATCH_GO
}

}  // namespace rfqmix
