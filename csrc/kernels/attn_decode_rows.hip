// Paged decode attention for steps of no more rows than work items (one decode row a sequence; captured steps, whose
// lists have an item for every row, of extends too): the work of attn_decode.hip with a workgroup of NW waves per (work
// item, split, kv head), every wave at every NW-th page of the split.
//
// What bounds it: the pages' bytes.  One wave per (work item, split, kv head) with a page on its way only while nothing
// else was done read 166 MB of pages that no cache holds (64 sequences of 300 - 900 tokens, 32 heads over 8) in 38.8 us,
// 4.3 TB/s.  Here
//   * K and V come in 1 KB pieces of neighbouring rows (keys as the product wants them, 64 bytes of 16 rows to an
//     access: 4 us more) and go through LDS; a page's registers are free once it is staged, and the next page is in
//     flight during all of the turn;
//   * as many waves share a split as the chip has room for;
//   * kv heads lie side by side in the grid, as in a page;
//   * a work item's two tiles of columns take a page together;
//   * pages go past the caches where the step's are more than those hold (launch_attn_decode_rows).
// Measured: these sequences 38.8 -> 32.8 us (two splits, two waves each; four waves, of which only half fit at once, 35), one
// sequence of 611 tokens 15.2 -> 9.0 us, 64 sequences of 450 - 900 whose first 13 pages are the same ones 56.0 -> 42.1 a pass
// of qkv product and attention (47.0 through the caches).  Extends in captured steps, 32 heads over 8, contexts of 600, in
// the general kernel and here (the two tiles of an item one after another: in brackets): four of eight rows and twelve
// single ones 20.1 -> 16.9 us (20.2), 56 of eight rows and eight single ones 48.9 -> 46.3 (68.5), one of 30 rows 14.1 -> 14.2
// (15.3), 16 rows of 2,000 tokens 16.3 -> 12.8 (15.4); with one tile an item, where eight rows to a sequence are captured,
// 0.94 to 1.05 of its time.
//
// The 16 columns of the products are (query, head) pairs of one kv head; S^T = K Q^T, O^T = V^T P^T with the weights in
// bf16; running maximum and sum per column.  The waves' results meet in LDS, the splits' as in attn_decode_core.h:
// partials in memory, merged by the last workgroup or by the caller.
#include <algorithm>

#include "attn_decode_core.h"

namespace rfq {

namespace {
constexpr int kRowS = kD + 8;                      // shorts of a staged row
constexpr int kWaveS = 2 * kPage * kRowS;          // of a wave: V, K; its results take the place of V

template <bool STREAM>
__device__ __forceinline__ s16x8 row_piece(const bf16_t* p) { return ld16<STREAM>(p); }
__device__ __forceinline__ float max_groups(float v) {      // over lanes 16 apart
  auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
  r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float sum_groups(float v) {
  auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = __uint_as_float(r[0]) + __uint_as_float(r[1]);
  r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
// Lanes read here what others of their wave wrote to LDS, whose accesses the hardware keeps in order: for the compiler.
__device__ __forceinline__ void wave_order() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}
typedef const __attribute__((address_space(4))) int32_t const_i32;
__device__ __forceinline__ int same(const int32_t* p, int64_t i) { return ((const_i32*)(uintptr_t)p)[i]; }
}  // namespace

struct DecodeRows {
  const bf16_t *q, *k_cache, *v_cache;
  int64_t q_stride, out_stride;
  const int32_t *block_tables, *q_start, *q_len, *kv_len, *work_seq, *work_ct;
  int32_t* tickets;
  bf16_t* out;
  float *part_o, *part_ml;
  int bt_stride, Hq, Hkv, splits;
  float scale_log2;
};

// The 16 N columns of a work item from c0 on, `cols` of them there: a page is read and staged once for all of them.
// One wave takes its pages with the arithmetic of the persistent decode layer (decode_persist.hip): the same bits.
template <int NW, int N, bool STREAM>
__device__ __forceinline__ void rows_columns(const DecodeRows& a, unsigned char* smem, int seq, int ql, int kvl, int q0,
                                             int split, int kvh, int c0, int cols) {
  const int tid = threadIdx.x, lane = tid & 63, c = lane & 15, g = lane >> 4;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int G = a.Hq / a.Hkv, S = a.splits;
  const_i32* bt = (const_i32*)(uintptr_t)(a.block_tables + (int64_t)seq * a.bt_stride);
  // pages split, split + S, ..: np of them; a wave takes the wid-th, wid + NW-th ..
  const int np = ((kvl + kPage - 1) / kPage - split + S - 1) / S;
  auto number = [&](int j) { return bt[min(split + max(min(j, np - 1), 0) * S, a.bt_stride - 1)]; };

  short* const Vt = reinterpret_cast<short*>(smem) + wid * kWaveS;
  short* const Kt = Vt + kPage * kRowS;
  float* const ml = reinterpret_cast<float*>(smem + (size_t)NW * kWaveS * 2);       // [NW][16 N] maxima, [NW][16 N] sums

  bool valid[N];
  int lim[N];                                       // keys [0, lim) are visible
  s16x8 qf[N][4];
#pragma unroll
  for (int t = 0; t < N; ++t) {
    const int cc = 16 * t + c;
    valid[t] = cc < cols;
    const int qi = valid[t] ? (c0 + cc) / G : 0, h = kvh * G + (valid[t] ? (c0 + cc) % G : 0);
    lim[t] = kvl - ql + qi + 1;
    const bf16_t* qp = a.q + (int64_t)(q0 + qi) * a.q_stride + (int64_t)h * kD + 8 * g;
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) qf[t][ks] = *reinterpret_cast<const s16x8*>(qp + 32 * ks);
  }
  s16x8 kr[8], vr[8];                               // 4 rows of 256 bytes to a load
  auto fetch = [&](int32_t page) {
    const int64_t at = ((int64_t)page * a.Hkv + kvh) * (kPage * kD) + lane * 8;
#pragma unroll
    for (int i = 0; i < 8; ++i) kr[i] = row_piece<STREAM>(a.k_cache + at + i * 512);
#pragma unroll
    for (int i = 0; i < 8; ++i) vr[i] = row_piece<STREAM>(a.v_cache + at + i * 512);
  };
  int32_t page = number(wid);
  if (np > 0) fetch(page);
  page = number(wid + NW);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int t = 0; t < N; ++t)
#pragma unroll
    for (int ks = 0; ks < 4; ++ks)
      if (!valid[t]) qf[t][ks] = (s16x8){0, 0, 0, 0, 0, 0, 0, 0};
  f32x4 o[N][8];
  float mrun[N], lrun[N];                           // lrun: the sum of this lane's keys
#pragma unroll
  for (int t = 0; t < N; ++t) {
    mrun[t] = -INFINITY;
    lrun[t] = 0.f;
#pragma unroll
    for (int m = 0; m < 8; ++m) o[t][m] = (f32x4){0.f, 0.f, 0.f, 0.f};
  }

  for (int j = wid; j < np; j += NW) {
    const int kt = (split + j * S) * kPage;
    if (kt + kPage > kvl) {                         // rows past the end may hold anything
#pragma unroll
      for (int i = 0; i < 8; ++i)
        if (kt + 4 * i + g >= kvl) vr[i] = (s16x8){0, 0, 0, 0, 0, 0, 0, 0};
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) *reinterpret_cast<s16x8*>(Kt + (4 * i + g) * kRowS + c * 8) = kr[i];
#pragma unroll
    for (int i = 0; i < 8; ++i) *reinterpret_cast<s16x8*>(Vt + (4 * i + g) * kRowS + c * 8) = vr[i];
    __builtin_amdgcn_sched_barrier(0);
    if (j + NW < np) {                              // the registers are free
      fetch(page);
      page = number(j + 2 * NW);
    }
    wave_order();
    f32x4 s[N][2];
#pragma unroll
    for (int t = 0; t < N; ++t) s[t][0] = s[t][1] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ks = 0; ks < 4; ++ks)
#pragma unroll
      for (int mt = 0; mt < 2; ++mt) {
        const s16x8 k = *reinterpret_cast<const s16x8*>(Kt + (16 * mt + c) * kRowS + 8 * g + 32 * ks);
#pragma unroll
        for (int t = 0; t < N; ++t)
          s[t][mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(k), as_bf16x8(qf[t][ks]), s[t][mt], 0, 0, 0);
      }
    __builtin_amdgcn_sched_barrier(0);
    s16x8 pb[N];
#pragma unroll
    for (int t = 0; t < N; ++t) {
      float p[8], mx = -INFINITY;                   // keys 16 mt + 4 g + i of column c
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        p[i] = kt + 16 * (i >> 2) + 4 * g + (i & 3) < lim[t] ? s[t][i >> 2][i & 3] * a.scale_log2 : -INFINITY;
        mx = fmaxf(mx, p[i]);
      }
      mx = max_groups(mx);
      // moved at once: the largest weight is then one, without a rounding (error of the results 2.1e-3, where it moves
      // only past 2^8 2.3e-3)
      const float mn = mx > mrun[t] ? mx : mrun[t];
      const float alpha = mrun[t] == mn ? 1.f : fast_exp2(mrun[t] - mn);
      if (__builtin_amdgcn_ballot_w64(alpha != 1.f) != 0ull) {
#pragma unroll
        for (int m = 0; m < 8; ++m) o[t][m] *= alpha;
      }
      mrun[t] = mn;
      const float mu = mn == -INFINITY ? 0.f : mn;  // nothing visible so far
      float sum = 0.f;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        p[i] = fast_exp2(p[i] - mu);
        sum += p[i];
      }
      lrun[t] = lrun[t] * alpha + sum;
      pb[t] = pack8(p);
    }
    const short* v0 = Vt + (4 * g + (c >> 2)) * kRowS + 4 * (c & 3);
#pragma unroll
    for (int m = 0; m < 8; ++m) {
      const s16x4 a0 = ds_read_tr16(v0 + 16 * m), a1 = ds_read_tr16(v0 + 16 * kRowS + 16 * m);
      const s16x8 v = {a0[0], a0[1], a0[2], a0[3], a1[0], a1[1], a1[2], a1[3]};
#pragma unroll
      for (int t = 0; t < N; ++t)
        o[t][m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(v), as_bf16x8(pb[t]), o[t][m], 0, 0, 0);
      if (m % 4 == 3) __builtin_amdgcn_sched_barrier(0);
    }
    wave_order();
  }

  // ---- the waves' results meet: [16 N][kD + 4] each, in the place of its page
  static_assert(16 * N * (kD + 4) * 4 <= kWaveS * 2, "");
  float* const res = reinterpret_cast<float*>(Vt);
#pragma unroll
  for (int t = 0; t < N; ++t) {
    const float l = sum_groups(lrun[t]);
    if (!valid[t]) continue;
#pragma unroll
    for (int m = 0; m < 8; ++m) *reinterpret_cast<f32x4*>(res + (16 * t + c) * (kD + 4) + 16 * m + 4 * g) = o[t][m];
    if (g == 0) {
      ml[wid * (16 * N) + 16 * t + c] = mrun[t];
      ml[(NW + wid) * (16 * N) + 16 * t + c] = l;
    }
  }
  __syncthreads();
  for (int y = tid; y < cols * (kD / 4); y += 64 * NW) {
    const int cc = y / (kD / 4), d = (y % (kD / 4)) * 4;
    const int64_t row = q0 + (c0 + cc) / G;
    const int hh = kvh * G + (c0 + cc) % G;
    float top = -INFINITY, l = 0.f;
#pragma unroll
    for (int u = 0; u < NW; ++u) top = fmaxf(top, ml[u * (16 * N) + cc]);
    f32x4 v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int u = 0; u < NW; ++u) {
      const float mu = ml[u * (16 * N) + cc], f = mu == -INFINITY ? 0.f : fast_exp2(mu - top);
      l += f * ml[(NW + u) * (16 * N) + cc];
      const f32x4 x = *reinterpret_cast<const f32x4*>(reinterpret_cast<const float*>(reinterpret_cast<const short*>(smem) + u * kWaveS) + cc * (kD + 4) + d);
      v += f * x;
    }
    if (S == 1) {
      const float inv = l > 0.f ? 1.f / l : 0.f;
      *reinterpret_cast<uint2*>(a.out + row * a.out_stride + (int64_t)hh * kD + d) =
          make_uint2(pack_bf16x2(v[0] * inv, v[1] * inv), pack_bf16x2(v[2] * inv, v[3] * inv));
    } else {
      // partials past this XCD's cache: whoever merges reads them there
      const int64_t pi = (row * a.Hq + hh) * S + split;
      gu64* to = (gu64*)(a.part_o + pi * kD + d);
      __hip_atomic_store(to, pack_f2(v[0], v[1]), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      __hip_atomic_store(to + 1, pack_f2(v[2], v[3]), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (d == 0) __hip_atomic_store((gu64*)(a.part_ml + pi * 2), pack_f2(top, l), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
  }
}

// NT: tiles of 16 columns to a work item
template <int NW, int NT, bool STREAM>
__global__ __launch_bounds__(64 * NW, 2) void attn_decode_rows_kernel(const DecodeRows a) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int tid = threadIdx.x;
  const int kvh = blockIdx.x % a.Hkv, split = blockIdx.x / a.Hkv % a.splits, w = blockIdx.x / (a.Hkv * a.splits);
  const int seq = same(a.work_seq, w);
  if (seq < 0) return;                              // padding work item (captured buckets)
  const int ql = same(a.q_len, seq), kvl = same(a.kv_len, seq), q0 = same(a.q_start, seq), c0 = same(a.work_ct, w) * (16 * NT);
  const int G = a.Hq / a.Hkv, S = a.splits, cols = min(16 * NT, ql * G - c0);
  if (cols <= 0) return;
  if (NT == 2 && cols > 16) rows_columns<NW, NT, STREAM>(a, smem, seq, ql, kvl, q0, split, kvh, c0, cols);
  else rows_columns<NW, 1, STREAM>(a, smem, seq, ql, kvl, q0, split, kvh, c0, cols);
  if (S == 1 || a.tickets == nullptr) return;

  // The last workgroup of the work item and kv head merges the splits: every thread's partials have left
  // before the ticket is taken, and it leaves the ticket at zero.
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  int32_t* const last = reinterpret_cast<int32_t*>(smem);
  __syncthreads();                                  // and the LDS is read
  if (tid == 0) {
    gu32* tk = (gu32*)(a.tickets + (int64_t)w * a.Hkv + kvh);
    const unsigned prev = __hip_atomic_fetch_add(tk, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    *last = prev == (unsigned)S - 1;
    if (prev == (unsigned)S - 1) __hip_atomic_store(tk, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  __syncthreads();
  if (*last == 0) return;
  for (int y = tid; y < cols * (kD / 4); y += 64 * NW) {
    const int cc = y / (kD / 4), d = (y % (kD / 4)) * 4;
    const int64_t row = q0 + (c0 + cc) / G;
    const int hh = kvh * G + (c0 + cc) % G;
    const int64_t base = (row * a.Hq + hh) * S;
    unsigned long long mls[16], x0[16], x1[16];
#pragma unroll
    for (int sp = 0; sp < 16; ++sp) {               // all on their way at once
      mls[sp] = x0[sp] = x1[sp] = 0;
      if (sp >= S) continue;
      mls[sp] = __hip_atomic_load((const gu64*)(a.part_ml + (base + sp) * 2), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      const gu64* from = (const gu64*)(a.part_o + (base + sp) * kD + d);
      x0[sp] = __hip_atomic_load(from, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      x1[sp] = __hip_atomic_load(from + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    auto lo = [](unsigned long long x) { return __uint_as_float((unsigned)x); };
    auto hi = [](unsigned long long x) { return __uint_as_float((unsigned)(x >> 32)); };
    float top = -INFINITY;
#pragma unroll
    for (int sp = 0; sp < 16; ++sp)
      if (sp < S) top = fmaxf(top, lo(mls[sp]));
    f32x4 v = {0.f, 0.f, 0.f, 0.f};
    float den[16];                                  // added up in twos, as lanes do it elsewhere
#pragma unroll
    for (int sp = 0; sp < 16; ++sp) {
      const float f = sp >= S || lo(mls[sp]) == -INFINITY ? 0.f : fast_exp2(lo(mls[sp]) - top);
      den[sp] = f * hi(mls[sp]);
      v += f * (f32x4){lo(x0[sp]), hi(x0[sp]), lo(x1[sp]), hi(x1[sp])};
    }
#pragma unroll
    for (int n = 1; n < 16; n *= 2)
#pragma unroll
      for (int sp = 0; sp < 16; sp += 2 * n) den[sp] += den[sp + n];
    const float l = den[0], inv = l > 0.f ? 1.f / l : 0.f;
    *reinterpret_cast<uint2*>(a.out + row * a.out_stride + (int64_t)hh * kD + d) =
        make_uint2(pack_bf16x2(v[0] * inv, v[1] * inv), pack_bf16x2(v[2] * inv, v[3] * inv));
  }
}

// ------------------------------------------------------------------ launcher
template <int NW, int NT, bool STREAM>
static void launch_rows_one(const DecodeRows& a, int64_t wgs, hipStream_t s) {
  constexpr size_t lds = (size_t)NW * kWaveS * 2 + 2 * NW * 16 * NT * sizeof(float);
  static_assert(lds <= 160 * 1024, "LDS of a CU");
  static bool attr = false;
  if (!attr) {          // dynamic LDS above 64 KB has to be allowed per kernel, once
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&attn_decode_rows_kernel<NW, NT, STREAM>),
                              hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
    attr = true;
  }
  attn_decode_rows_kernel<NW, NT, STREAM><<<dim3((unsigned)wgs), dim3(64 * NW), lds, s>>>(a);
}
template <int NW>
static void launch_rows_waves(const DecodeRows& a, int64_t wgs, int tiles, bool stream, hipStream_t s) {
  if (tiles == 2) {
    if (stream) launch_rows_one<NW, 2, true>(a, wgs, s);
    else launch_rows_one<NW, 2, false>(a, wgs, s);
  } else {
    if (stream) launch_rows_one<NW, 1, true>(a, wgs, s);
    else launch_rows_one<NW, 1, false>(a, wgs, s);
  }
}

void launch_attn_decode_rows(const bf16_t* q, int64_t q_stride, const bf16_t* k_cache, const bf16_t* v_cache,
                             const int32_t* block_tables, int bt_stride, const int32_t* seq_q_start, const int32_t* seq_q_len,
                             const int32_t* seq_kv_len, int seqs, const int32_t* work_seq, const int32_t* work_ct, int W, int rows,
                             bf16_t* out, int64_t out_stride, float* part_o, float* part_ml, int Hq, int Hkv, float scale_log2,
                             int num_splits, int tiles_per_item, int32_t* tickets, bool past, hipStream_t s) {
  const DecodeRows a{q, k_cache, v_cache, q_stride, out_stride, block_tables, seq_q_start, seq_q_len, seq_kv_len, work_seq,
                     work_ct, tickets, out, part_o, part_ml, bt_stride, Hq, Hkv, num_splits, scale_log2};
  // As many waves to a workgroup as its LDS leaves room for with all workgroups on the chip at once: 8.5 KB of a CU's 160
  // for a wave's keys, as much for its values.  Work items of a captured step's list that none of its sequences can need
  // are padding and leave at once.  Past the caches where the caller asks for it (`past`), and where the tables have room
  // for more than 96 MB, as in mix_keep_row.hip.  A captured step's have, whatever its sequences hold.  32 heads over 8, 600
  // tokens each, pages that no cache holds, through the caches and past them: 4 sequences 10.7 / 11.0 us, 8 12.8 / 12.4, 16
  // 16.1 / 14.8, 64 31.6 / 31.8; with the first 13 pages in common 10.0 / 10.3, 10.6 / 11.3, 12.0 / 12.4, 20.0 / 20.1.  Few
  // long ones gain: 4 of 2,000 tokens 14.7 / 13.9, 8 of 4,000 31.8 / 29.7, one of 32,000 70.4 / 58.2.
  const int64_t wgs = (int64_t)W * Hkv * num_splits;
  const int64_t items = std::min<int64_t>(W, seqs + (int64_t)rows * (Hq / Hkv) / (16 * tiles_per_item));
  const int64_t live = items * Hkv * num_splits;
  const bool stream = past || (int64_t)W * Hkv * bt_stride * (kPage * kD * 4) > (96 << 20);
  if (rows <= 4) return launch_rows_waves<1>(a, wgs, tiles_per_item, stream, s);   // steps that the persistent layer takes in a captured graph
  if (live <= 256) return launch_rows_waves<8>(a, wgs, tiles_per_item, stream, s);
  if (live <= 512) return launch_rows_waves<4>(a, wgs, tiles_per_item, stream, s);
  launch_rows_waves<2>(a, wgs, tiles_per_item, stream, s);
}

}  // namespace rfq
