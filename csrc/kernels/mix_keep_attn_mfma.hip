// attn_keep_window on MFMA tiles, prompt rows (bf16 pages of 32 tokens, key width a multiple of 32,
// value width a multiple of 32).  Semantics of mix_keep_attn.hip: sliding window with kept first
// tokens; softmax, softmax with a sink, or unnormalised sigmoid weights; optional output gate
// (a column per head, or gate_w = vdim: one per output, rows 8-byte aligned);
// the values may be the leading entries of the key rows themselves (latent attention).
// Decode rows have a kernel of their own (mix_keep_split.hip).
//
// One workgroup per (work item, HPW heads of one key/value head); a work item is (sequence, block of
// 32 queries).  Its 2 HPW waves are (16 queries) x (head): a wave keeps the running maximum and sum of
// its 16 query columns and the weighted values O^T [vdim x 16] in registers.  A key tile is one page,
// staged in LDS for all heads of the workgroup, the next page while this one is multiplied; one barrier
// per page.  Pages between the kept first tokens and the window are never read.
//
//   S^T[key, query] = K[key, :] . Q[query, :]   v_mfma_f32_16x16x32_bf16, A = key rows from LDS,
//                     B = the queries in registers as bf16 hi (+ lo for keys of up to 320
//                     entries: they arrive in fp32 and are not rounded a second time), up to 192
//                     entries already times the scale and log2 e
//   cap, mask, weights per query column in fp32, base 2
//   O^T[dv, query] += V^T[dv, keys] . P^T[keys, query]   A = two transposed reads of V
//                     (ds_read_tr16_b64), B = the weights straight from the score registers as bf16
//                     hi + lo parts (two MFMAs), so the weights keep fp32's precision
//
// What bounds it: the vector instructions between the products, and their latency.  Pages without an
// edge inside skip the masks, the maximum moves only when a score passes it by 2^11 (so the
// accumulators are rarely rescaled), rows meet by lane swaps instead of LDS, one barrier a page, and a
// sequence's last blocks, which see the most keys, start first.  Measured with the append before it,
// without -> with these: prompts of 2,048 and 600 tokens (32 heads over 8 of 128, softcap) 234 -> 223 us,
// five ragged prompts with sigmoid weights and a window of 1,024 125 -> 87 us, one prompt of 2,048 with
// 64 heads and a window 268 -> 174 us.  What is left of the first is the longest block's chain of 64
// pages.  32 x 32 tiles, a wave per 32 queries, took 217 and 116 us there and lost 20 % on prompts of a
// few hundred tokens; two waves sharing such a wave's pages 251 and 119.
#include <algorithm>

#include "common.h"
#include "mix_common.h"

namespace rfqmix {

using rfq::as_bf16x8;
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

template <int DK, int DV, bool SHARED>
constexpr int keep_page_shorts() {
  return WBS * (32 * DK + 8) + (SHARED ? 0 : WBS * (16 * DV + 8));
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
};

// the same over lanes 16 away
__device__ __forceinline__ float other_row_max(float x) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float both_rows_sum(float x) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// lane (col, grp) holds value channels 16 m + 4 grp .. + 3 of its query: 8-byte stores
template <int DV, int MODE>
__device__ __forceinline__ void store_rows(const KeepArgs& a, f32x4 (&o)[DV], float lrun, int64_t t, int hh, int grp,
                                           bool qlive) {
  constexpr int vdim = 16 * DV;
  const float l = both_halves_sum(both_rows_sum(lrun));
  if (!qlive) return;
  const bf16_t* gate = static_cast<const bf16_t*>(a.gate);
  float mul = MODE >= 2 ? a.out_mult : (l > 0.f ? a.out_mult / l : 0.f);
  if (gate != nullptr && a.gate_w == 1) mul /= 1.0f + __expf(-ldf(gate + t * a.gate_stride + hh));
  // a gate column per output: four neighbouring logits, 8-byte reads
  const bf16_t* grow = gate != nullptr && a.gate_w > 1 ? gate + t * a.gate_stride + (int64_t)hh * vdim + grp * 4 : nullptr;
  bf16_t* orow = static_cast<bf16_t*>(a.out) + t * a.out_stride + (int64_t)hh * vdim + grp * 4;
#pragma unroll
  for (int m = 0; m < DV; ++m) {
    float y[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) y[i] = o[m][i] * mul;
    if (grow != nullptr) {
      const uint2 gu = *reinterpret_cast<const uint2*>(grow + m * 16);
      y[0] /= 1.0f + __expf(-__uint_as_float(gu.x << 16));
      y[1] /= 1.0f + __expf(-__uint_as_float(gu.x & 0xffff0000u));
      y[2] /= 1.0f + __expf(-__uint_as_float(gu.y << 16));
      y[3] /= 1.0f + __expf(-__uint_as_float(gu.y & 0xffff0000u));
    }
    *reinterpret_cast<uint2*>(orow + m * 16) = make_uint2(rfq::pack_bf16x2(y[0], y[1]), rfq::pack_bf16x2(y[2], y[3]));
  }
}

// DK = E / 32, DV = vdim / 16, HPW heads per workgroup, SHARED: values = leading entries of the
// key rows, MODE: 0 softmax, 1 softmax of capped scores, 2 sigmoid, 3 sigmoid of capped scores.
// Two heads a workgroup: three waves a SIMD, which the compiler left to itself spends on 180 registers for
// two (16 chunks of 230 rows after 416, 12 heads over 2 of 128, softcap: 92 -> 70 us a pass).
template <int DK, int DV, int HPW, bool SHARED, int MODE>
__global__ __launch_bounds__(128 * HPW, HPW == 2 ? 3 : 1) void attn_keep_mfma_kernel(const KeepArgs a) {
  constexpr int E = 32 * DK, vdim = 16 * DV, NT = 128 * HPW;
  constexpr int KRS = E + 8;                       // shorts per key row in LDS (+ 16 bytes)
  constexpr int VRS = SHARED ? KRS : vdim + 8;     // shorts per value row
  constexpr int PGS = keep_page_shorts<DK, DV, SHARED>();
  const int item = gridDim.x - 1 - blockIdx.x;     // a sequence's later blocks see the most keys: they start first
  const int s = a.work_seq[item];
  if (s < 0) return;
  const int ql = a.q_len[s];
  const int i0 = a.work_qblk[item] * WQB;
  if (i0 >= ql) return;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col = lane & 15, grp = lane >> 4;
  const int g = ((int)blockIdx.y * HPW) / (a.H / a.G);
  const int hh = (int)blockIdx.y * HPW + (wid >> 1);
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  short* const pages = reinterpret_cast<short*>(smem);       // two of them

  const int nq = min(WQB, ql - i0);
  const int p0 = a.kv_len[s] - ql + i0, plast = p0 + nq - 1;
  const int window = a.window, keep_first = a.keep_first;
  const int jwin = window > 0 ? max(0, p0 - window + 1) : 0;
  const int kf = window > 0 ? min(keep_first, jwin) : 0;     // kept keys before the window
  const int row = (wid & 1) * 16 + col, pi = p0 + row;       // this lane's query
  const bool qlive = row < nq;
  const int64_t t = a.q_start[s] + i0 + (qlive ? row : 0);
  typedef const __attribute__((address_space(4))) int32_t const_i32;
  const_i32* bt = (const_i32*)(uintptr_t)(a.bt + (int64_t)s * a.maxb);

  // scores arrive as exponents of 2: s log2 e; 2 s log2 e / cap; -s log2 e (sigmoid, no cap)
  const float qmul = a.scale * (MODE % 2 == 1 ? 2.f * kLog2e / a.softcap : MODE == 2 ? -kLog2e : kLog2e);
  const float cap2 = MODE % 2 == 1 ? a.softcap * kLog2e : 0.f;
  s16x8 qhi[DK], qlo[DK];
  {
    const float* qp = a.q + (t * a.H + hh) * E + grp * 8;
#pragma unroll
    for (int ks = 0; ks < DK; ++ks) {
      const float4 x = *reinterpret_cast<const float4*>(qp + ks * 32);
      const float4 y = *reinterpret_cast<const float4*>(qp + ks * 32 + 4);
      const float f[8] = {x.x * qmul, x.y * qmul, x.z * qmul, x.w * qmul, y.x * qmul, y.y * qmul, y.z * qmul, y.w * qmul};
      split_bf16w(f, qhi[ks], qlo[ks]);
    }
  }
  f32x4 o[DV];
#pragma unroll
  for (int m = 0; m < DV; ++m) o[m] = (f32x4){0.f, 0.f, 0.f, 0.f};
  const float hb = a.head_bias != nullptr ? a.head_bias[hh] * kLog2e : 0.f;
  const bool sink = MODE < 2 && a.head_bias != nullptr;
  // the sink is one more entry of the row: it starts the maximum, and one lane's part of the sum
  float mrun = sink ? hb : kNegInfW, lrun = sink && grp == 0 ? 1.f : 0.f;

  // ---- staging
  constexpr int NKV = (WBS * E / 8 + NT - 1) / NT;
  constexpr int NVV = SHARED ? 1 : (WBS * vdim / 8 + NT - 1) / NT;
  s16x8 kreg[NKV], vreg[NVV];
  auto fetch = [&](int page) {
    const int64_t at = ((int64_t)page * a.G + g) * WBS;      // the page's first slot
    const bf16_t* kb = static_cast<const bf16_t*>(a.k_cache) + at * E;
#pragma unroll
    for (int i = 0; i < NKV; ++i) {
      const int x = tid + i * NT;
      if (x < WBS * E / 8) kreg[i] = reinterpret_cast<const s16x8*>(kb)[x];
    }
    if constexpr (!SHARED) {
      const bf16_t* vb = static_cast<const bf16_t*>(a.v_cache) + at * a.vrs;
#pragma unroll
      for (int i = 0; i < NVV; ++i) {
        const int x = tid + i * NT;
        if (x < WBS * vdim / 8) {
          const int jj = x / (vdim / 8), c = x - jj * (vdim / 8);
          vreg[i] = *reinterpret_cast<const s16x8*>(vb + jj * a.vrs + c * 8);
        }
      }
    }
  };
  // Rows past the sequence's end were never written and may hold anything: zeros.
  auto stage = [&](int jb, int buf) {
    short* Ks = pages + buf * PGS;
    short* Vs = SHARED ? Ks : Ks + WBS * KRS;
    const bool tail = jb + WBS - 1 > plast;
#pragma unroll
    for (int i = 0; i < NKV; ++i) {
      const int x = tid + i * NT;
      if (x < WBS * E / 8) {
        const int jj = x / (E / 8), c = x - jj * (E / 8);
        s16x8 v = kreg[i];
        if (SHARED && tail && jb + jj > plast) v = (s16x8){0, 0, 0, 0, 0, 0, 0, 0};
        *reinterpret_cast<s16x8*>(Ks + jj * KRS + c * 8) = v;
      }
    }
    if constexpr (!SHARED) {
#pragma unroll
      for (int i = 0; i < NVV; ++i) {
        const int x = tid + i * NT;
        if (x < WBS * vdim / 8) {
          const int jj = x / (vdim / 8), c = x - jj * (vdim / 8);
          s16x8 v = vreg[i];
          if (tail && jb + jj > plast) v = (s16x8){0, 0, 0, 0, 0, 0, 0, 0};
          *reinterpret_cast<s16x8*>(Vs + jj * VRS + c * 8) = v;
        }
      }
    }
  };
  const int kat = col * KRS + grp * 8;
  // transposed reads: a 16-lane group takes 4 key rows x 16 value columns, lane `col` receives its
  // column (keys 4 grp .. 4 grp + 3 of each 16-key half)
  const int vat = (4 * grp + (col >> 2)) * VRS + 4 * (col & 3);

  // pages [0 .. pg_keep] hold the kept first tokens, pages [pg_win .. pg_last] the window
  const int pg_last = plast / WBS;
  const int pg_keep = kf > 0 ? (kf - 1) / WBS : -1;
  const int pg_win = jwin / WBS;
  auto next_page = [&](int pg) { return (pg == pg_keep && pg_win > pg) ? pg_win : pg + 1; };
  int pg = kf > 0 ? 0 : pg_win, buf = 0;
  fetch(bt[pg]);
  stage(pg * WBS, 0);
  int pn = next_page(pg);
  if (pn <= pg_last) fetch(bt[pn]);
  __syncthreads();
  while (pg <= pg_last) {
    const int jb = pg * WBS;
    const short* Ks = pages + buf * PGS;
    const short* Vs = SHARED ? Ks : Ks + WBS * KRS;
    f32x4 sc[2][2];                                          // two chains per half page
#pragma unroll
    for (int kt = 0; kt < 2; ++kt) {
      sc[kt][0] = sc[kt][1] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < DK; ++ks) {
        const s16x8 k = *reinterpret_cast<const s16x8*>(Ks + kat + kt * 16 * KRS + ks * 32);
        sc[kt][0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(k), as_bf16x8(qhi[ks]), sc[kt][0], 0, 0, 0);
        sc[kt][1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(k), as_bf16x8(qlo[ks]), sc[kt][1], 0, 0, 0);
      }
    }
    float p[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      float x = sc[i >> 2][0][i & 3] + sc[i >> 2][1][i & 3];
      if constexpr (MODE % 2 == 1) x = cap2 - 2.f * cap2 * __builtin_amdgcn_rcpf(__builtin_amdgcn_exp2f(x) + 1.f);
      if constexpr (MODE >= 2) x = __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f((MODE == 3 ? -x : x) - hb));
      p[i] = x;
    }
    if (!(jb + WBS - 1 <= p0 && (window <= 0 || plast - jb < window || jb + WBS <= keep_first))) {
#pragma unroll
      for (int i = 0; i < 8; ++i) {                          // an edge inside the page
        const int j = jb + (i >> 2) * 16 + grp * 4 + (i & 3);
        const bool ok = j <= pi && (window <= 0 || pi - j < window || j < keep_first);
        p[i] = ok ? p[i] : MODE >= 2 ? 0.f : kNegInfW;
      }
    }
    if constexpr (MODE < 2) {
      float mx = fmaxf(fmaxf(fmaxf(p[0], p[1]), fmaxf(p[2], p[3])), fmaxf(fmaxf(p[4], p[5]), fmaxf(p[6], p[7])));
      mx = other_half_max(other_row_max(mx));
      const bool moves = mx > mrun + kDeferW;                // also for the first keys: mrun = -inf
      if (__builtin_amdgcn_ballot_w64(moves) != 0ull) {
        const float mn = moves ? mx : mrun;
        const float alpha = moves ? __builtin_amdgcn_exp2f(mrun - mn) : 1.f;
        mrun = mn;
        lrun *= alpha;
#pragma unroll
        for (int m = 0; m < DV; ++m) o[m] *= alpha;
      }
      const float mu = mrun == kNegInfW ? 0.f : mrun;        // no visible key so far: every weight 0
      float l0 = 0.f, l1 = 0.f;
#pragma unroll
      for (int i = 0; i < 8; i += 2) {
        p[i] = __builtin_amdgcn_exp2f(p[i] - mu);
        p[i + 1] = __builtin_amdgcn_exp2f(p[i + 1] - mu);
        l0 += p[i];
        l1 += p[i + 1];
      }
      lrun += l0 + l1;
    }
    s16x8 phi, plo;
    split_bf16w(p, phi, plo);
    constexpr int MG = DV % 4 == 0 ? 4 : 2;                  // value blocks taken together
#pragma unroll
    for (int m = 0; m < DV; m += MG) {
      s16x8 v[MG];
#pragma unroll
      for (int u = 0; u < MG; ++u) {
        const s16x4 a0 = rfq::ds_read_tr16(Vs + vat + 16 * (m + u));
        const s16x4 a1 = rfq::ds_read_tr16(Vs + vat + 16 * VRS + 16 * (m + u));
        v[u] = (s16x8){a0[0], a0[1], a0[2], a0[3], a1[0], a1[1], a1[2], a1[3]};
      }
#pragma unroll
      for (int u = 0; u < MG; ++u)
        o[m + u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(v[u]), as_bf16x8(phi), o[m + u], 0, 0, 0);
#pragma unroll
      for (int u = 0; u < MG; ++u)
        o[m + u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(v[u]), as_bf16x8(plo), o[m + u], 0, 0, 0);
    }
    pg = pn;
    if (pg <= pg_last) {
      stage(pg * WBS, buf ^ 1);          // it has been on its way since the last page
      pn = next_page(pg);
      if (pn <= pg_last) fetch(bt[pn]);
    }
    __syncthreads();
    buf ^= 1;
  }
  store_rows<DV, MODE>(a, o, lrun, t, hh, grp, qlive);
}

// Wide latents: keys of 320 or 576 entries whose first 256 or 512 are the values.  32 queries' results
// (256 registers at 512 values) and the queries themselves (144) leave no room for the rest, so a wave
// has 16 queries on 16x16x32 tiles, two waves a head, and the page's LDS reads are what bounds it (K
// rows 36 x 1 KB, V 64 x 512 B a wave and page: 4,350 clocks for eight waves against 3,200 of MFMA).
// One prompt of 2,048 over 576 (32 heads) took 904 us a pass on the kernel above, 420 here; four of
// them with 64 heads 3,249 and 1,402.  Pages come by LDS-DMA, the next one during this one; their rows lie unpadded, 16-byte pieces
// permuted inside each 128 bytes by wide_swizzle(row).
// DEC: decode rows.  A wave's columns are 16 heads of one row, so that a workgroup reads a page once for up to
// 128 heads; the pages come one after another, which pays once every CU has a workgroup (launch_split_waves).
// 256 sequences of 300 tokens with 64 heads of 576 entries 44 us, 32 of 500 with four rows each 50; split over
// waves 116 and 129.
// Sixteen rows of one piece (a K read) and four neighbouring rows of a pair of pieces beside the next
// four (a transposed V read) then lie on different banks: the row's parity picks a half of them, bits
// 1 and 2 the pair, bit 3 the order inside it.
__device__ __forceinline__ int wide_swizzle(int r) { return ((r >> 1) & 1) << 2 | ((r >> 2) & 1) << 1 | ((r >> 3) & 1); }

template <int DK, int DV, int HPW, int MODE, bool DEC>
__global__ __launch_bounds__(128 * HPW, DEC && HPW == 1 ? 1 : 2) void attn_keep_wide_kernel(const KeepArgs a) {
  constexpr int E = 32 * DK, vdim = 16 * DV, NWV = 2 * HPW, NP = WBS * E / 512, ND = (NP + NWV - 1) / NWV;
  constexpr bool QLO = DK <= 10;
  static_assert(E % 64 == 0 && DV % 4 == 0, "whole 128-byte lines");
  const int item = gridDim.x - 1 - blockIdx.x;     // a sequence's later blocks see the most keys: they start first
  const int s = DEC ? item : a.work_seq[item];
  if (s < 0) return;
  const int ql = a.q_len[s];
  const int i0 = DEC ? 0 : a.work_qblk[item] * WQB;
  if (i0 >= ql) return;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col = lane & 15, grp = lane >> 4;
  constexpr int HW = DEC ? 16 * NWV : HPW;                    // heads of a workgroup
  const int rep = a.H / a.G, per = (rep + HW - 1) / HW;       // workgroups of a key head, the last partly idle
  const int g = (int)blockIdx.y / per, h0 = ((int)blockIdx.y - g * per) * HW;
  const int hd = DEC ? h0 + wid * 16 + col : h0 + (wid >> 1);
  const bool idle = DEC && h0 + wid * 16 >= rep;             // a wave that only copies pages
  const int hh = g * rep + min(hd, rep - 1);                 // past the last head: it once more, not stored
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  short* const pages = reinterpret_cast<short*>(smem);       // two of them

  for (int r = DEC ? (int)blockIdx.z : 0; r < (DEC ? ql : 1); r += DEC ? (int)gridDim.z : 1) {
  const int nq = DEC ? 1 : min(WQB, ql - i0);
  const int p0 = a.kv_len[s] - ql + (DEC ? r : i0), plast = p0 + nq - 1;
  const int window = a.window, keep_first = a.keep_first;
  const int jwin = window > 0 ? max(0, p0 - window + 1) : 0;
  const int kf = window > 0 ? min(keep_first, jwin) : 0;
  const int row = DEC ? 0 : (wid & 1) * 16 + col, pi = p0 + row;       // this lane's query
  const bool qlive = row < nq && hd < rep;
  const int64_t t = a.q_start[s] + (DEC ? r : i0) + (qlive ? row : 0);
  typedef const __attribute__((address_space(4))) int32_t const_i32;
  const_i32* bt = (const_i32*)(uintptr_t)(a.bt + (int64_t)s * a.maxb);

  const float qmul = __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(
      a.scale * (MODE % 2 == 1 ? 2.f * kLog2e / a.softcap : MODE == 2 ? -kLog2e : kLog2e))));
  const float cap2 = MODE % 2 == 1 ? a.softcap * kLog2e : 0.f;
  s16x8 qhi[DK], qlo[QLO ? DK : 1];
  {
    const float* qp = a.q + (t * a.H + hh) * E + grp * 8;
#pragma unroll
    for (int ks = 0; ks < DK; ++ks) {
      const float4 x = *reinterpret_cast<const float4*>(qp + ks * 32);
      const float4 y = *reinterpret_cast<const float4*>(qp + ks * 32 + 4);
      const float f[8] = {x.x, x.y, x.z, x.w, y.x, y.y, y.z, y.w};   // as they are: bf16 values stay exact
      if constexpr (QLO) split_bf16w(f, qhi[ks], qlo[ks]);
      else qhi[ks] = rfq::pack8(f);
    }
  }
  f32x4 o[DV];
#pragma unroll
  for (int m = 0; m < DV; ++m) o[m] = (f32x4){0.f, 0.f, 0.f, 0.f};
  const float hb = a.head_bias != nullptr ? a.head_bias[hh] * kLog2e : 0.f;
  const bool sink = MODE < 2 && a.head_bias != nullptr;
  float mrun = sink ? hb : kNegInfW, lrun = sink && grp == 0 ? 1.f : 0.f;      // sums: a quarter per lane

  uint32_t src[ND];                                          // this lane's source pieces, bytes from the page's first
#pragma unroll
  for (int i = 0; i < ND; ++i) {
    const int p = (wid + i * NWV) * 64 + lane, r = p / (E / 8), c = p - r * (E / 8);
    src[i] = (r * E + ((c & ~7) | ((c & 7) ^ wide_swizzle(r))) * 8) * 2;
  }
  auto fetch = [&](int page, int buf) {
    const char* kb = static_cast<const char*>(a.k_cache) + ((int64_t)page * a.G + g) * WBS * E * 2;
#pragma unroll
    for (int i = 0; i < ND; ++i) {
      const int piece = wid + i * NWV;
      uint32_t at = src[i];
      asm("" : "+v"(at));      // widened here: hoisted out of the loop the offsets are pairs of registers, spilled
      if ((i + 1) * NWV <= NP || piece < NP)
        rfq::glds16(reinterpret_cast<const bf16_t*>(kb + at),
                    reinterpret_cast<bf16_t*>(pages + buf * WBS * E + piece * 512));
    }
  };
  // The page has landed for everyone, and everyone is done with the one before it, whose place the next
  // takes; rows past the sequence's end were never written: zeros.
  auto landed = [&](int jb, int buf) {
    __builtin_amdgcn_s_waitcnt(0x0F70);                      // vmcnt(0)
    __syncthreads();
    if (jb + WBS - 1 > plast) {
      for (int x = max(0, plast + 1 - jb) * (E / 8) + tid; x < WBS * (E / 8); x += 64 * NWV)
        *reinterpret_cast<s16x8*>(pages + buf * WBS * E + x * 8) = (s16x8){0, 0, 0, 0, 0, 0, 0, 0};
      __syncthreads();
    }
    if (DEC && jb < jwin && jb + WBS > kf) {                 // out of the row's sight: may hold infinities
      const int end = min(jwin - jb, WBS) * (E / 8);
      for (int x = max(0, kf - jb) * (E / 8) + tid; x < end; x += 64 * NWV)
        *reinterpret_cast<s16x8*>(pages + buf * WBS * E + x * 8) = (s16x8){0, 0, 0, 0, 0, 0, 0, 0};
      __syncthreads();
    }
  };
  // keys: row col (+ 16), entries 32 ks + 8 grp ..; values, transposed: rows 4 grp + col / 4 (+ 16),
  // channels 16 m + 4 (col % 4) ..
  const int ksw = wide_swizzle(col), vrow = 4 * grp + (col >> 2), vsw = wide_swizzle(vrow);
  int kat[2], vat[4];
#pragma unroll
  for (int i = 0; i < 2; ++i) kat[i] = col * E + ((4 * i + grp) ^ ksw) * 8;
#pragma unroll
  for (int i = 0; i < 4; ++i) vat[i] = vrow * E + ((2 * i + ((col >> 1) & 1)) ^ vsw) * 8 + (col & 1) * 4;

  const int pg_last = plast / WBS;
  const int pg_keep = kf > 0 ? (kf - 1) / WBS : -1;
  const int pg_win = jwin / WBS;
  auto next_page = [&](int pg) { return (pg == pg_keep && pg_win > pg) ? pg_win : pg + 1; };
  s16x8 phi, plo;
  auto weigh = [&](const short* P) {                         // O += V^T P^T
#pragma unroll
    for (int m = 0; m < DV; m += 4) {
      s16x8 v[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const short* vp = P + vat[u] + (m >> 2) * 64;
        const s16x4 a0 = rfq::ds_read_tr16(vp), a1 = rfq::ds_read_tr16(vp + 16 * E);
        v[u] = (s16x8){a0[0], a0[1], a0[2], a0[3], a1[0], a1[1], a1[2], a1[3]};
      }
#pragma unroll
      for (int u = 0; u < 4; ++u)
        o[m + u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(v[u]), as_bf16x8(phi), o[m + u], 0, 0, 0);
#pragma unroll
      for (int u = 0; u < 4; ++u)
        o[m + u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(v[u]), as_bf16x8(plo), o[m + u], 0, 0, 0);
    }
  };
  int pg = kf > 0 ? 0 : pg_win, buf = 0;
  fetch(bt[pg], 0);
  int ahead = bt[min(next_page(pg), pg_last)];                 // the next page's number, read a page early
  while (pg <= pg_last) {
    const int jb = pg * WBS, pn = next_page(pg);
    landed(jb, buf);
    if (pn <= pg_last) fetch(ahead, buf ^ 1);
    ahead = bt[min(next_page(pn), pg_last)];
    if (idle) {
      pg = pn;
      buf ^= 1;
      continue;
    }
    const short* P = pages + buf * WBS * E;
    f32x4 sc[2][2];                                          // two chains per half page
#pragma unroll
    for (int kt = 0; kt < 2; ++kt) {
      sc[kt][0] = sc[kt][1] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < DK; ++ks) {
        const s16x8 k = *reinterpret_cast<const s16x8*>(P + kat[ks & 1] + kt * 16 * E + (ks >> 1) * 64);
        f32x4& acc = sc[kt][ks & 1];
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(k), as_bf16x8(qhi[ks]), acc, 0, 0, 0);
        if constexpr (QLO) acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(k), as_bf16x8(qlo[ks]), acc, 0, 0, 0);
      }
    }
    float p[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      float x = (sc[i >> 2][0][i & 3] + sc[i >> 2][1][i & 3]) * qmul;
      if constexpr (MODE % 2 == 1) x = cap2 - 2.f * cap2 * __builtin_amdgcn_rcpf(__builtin_amdgcn_exp2f(x) + 1.f);
      if constexpr (MODE >= 2) x = __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f((MODE == 3 ? -x : x) - hb));
      p[i] = x;
    }
    if (!(jb + WBS - 1 <= p0 && (window <= 0 || plast - jb < window || jb + WBS <= keep_first))) {
#pragma unroll
      for (int i = 0; i < 8; ++i) {                          // an edge inside the page
        const int j = jb + (i >> 2) * 16 + grp * 4 + (i & 3);
        const bool ok = j <= pi && (window <= 0 || pi - j < window || j < keep_first);
        p[i] = ok ? p[i] : MODE >= 2 ? 0.f : kNegInfW;
      }
    }
    if constexpr (MODE < 2) {
      float mx = fmaxf(fmaxf(fmaxf(p[0], p[1]), fmaxf(p[2], p[3])), fmaxf(fmaxf(p[4], p[5]), fmaxf(p[6], p[7])));
      mx = other_half_max(other_row_max(mx));
      const bool moves = mx > mrun + kDeferW;                // also for the first keys: mrun = -inf
      if (__builtin_amdgcn_ballot_w64(moves) != 0ull) {
        const float mn = moves ? mx : mrun;
        const float alpha = moves ? __builtin_amdgcn_exp2f(mrun - mn) : 1.f;
        mrun = mn;
        lrun *= alpha;
#pragma unroll
        for (int m = 0; m < DV; ++m) o[m] *= alpha;
      }
      const float mu = mrun == kNegInfW ? 0.f : mrun;        // no visible key so far: every weight 0
      float l0 = 0.f, l1 = 0.f;
#pragma unroll
      for (int i = 0; i < 8; i += 2) {
        p[i] = __builtin_amdgcn_exp2f(p[i] - mu);
        p[i + 1] = __builtin_amdgcn_exp2f(p[i + 1] - mu);
        l0 += p[i];
        l1 += p[i + 1];
      }
      lrun += l0 + l1;
    }
    split_bf16w(p, phi, plo);
    weigh(P);
    pg = pn;
    buf ^= 1;
  }
  store_rows<DV, MODE>(a, o, lrun, t, hh, grp, qlive);
  if constexpr (DEC) __syncthreads();                        // the next row's pages take this one's places
  }
}

// ------------------------------------------------------------------ launcher
namespace {
bool plain_sizes(int DK, int DV) { return DK >= 1 && DK <= 4 && (DV == 2 || DV == 4 || DV == 8); }
bool shared_sizes(int DK, int DV) {
  return (DK == 3 && DV == 4) || (DK == 4 && (DV == 4 || DV == 6)) || (DK == 5 && DV == 8) ||
         (DK == 6 && DV == 8) || (DK == 10 && DV == 16) || (DK == 18 && DV == 32);
}
}  // namespace

bool keep_mfma_ok(int E, int vdim, int BS, bool shared) {
  if (BS != WBS || E % 32 != 0 || vdim % 16 != 0) return false;
  return shared ? shared_sizes(E / 32, vdim / 16) : plain_sizes(E / 32, vdim / 16);
}

template <int DK, int DV, int HPW, bool SHARED, int MODE>
static void launch_keep_mfma_one(const KeepArgs& a) {
  constexpr bool WIDE = SHARED && DK >= 10;
  constexpr size_t lds = (size_t)2 * (WIDE ? WBS * 32 * DK : keep_page_shorts<DK, DV, SHARED>()) * sizeof(short);
  static_assert(lds <= 160 * 1024, "LDS of a CU");
  static bool attr = false;
  auto run = [&](auto kernel, int threads) {
    if (!attr) {
      (void)hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                                160 * 1024);
      attr = true;
    }
    const int rep = a.H / a.G;
    hipLaunchKernelGGL(kernel, dim3(a.W, a.G * ((rep + HPW - 1) / HPW)), dim3(threads), lds, a.s, a);
  };
  if constexpr (WIDE) run(&attn_keep_wide_kernel<DK, DV, HPW, MODE, false>, 128 * HPW);
  else run(&attn_keep_mfma_kernel<DK, DV, HPW, SHARED, MODE>, 128 * HPW);
}

template <int DK, int DV, int HPW, bool SHARED>
static void launch_keep_mfma_mode(const KeepArgs& a) {
  const bool cap = a.softcap > 0.f;
  if (a.sigmoid && cap) launch_keep_mfma_one<DK, DV, HPW, SHARED, 3>(a);
  else if (a.sigmoid) launch_keep_mfma_one<DK, DV, HPW, SHARED, 2>(a);
  else if (cap) launch_keep_mfma_one<DK, DV, HPW, SHARED, 1>(a);
  else launch_keep_mfma_one<DK, DV, HPW, SHARED, 0>(a);
}

template <int DK, int DV, bool SHARED>
static void launch_keep_mfma_heads(const KeepArgs& a) {
  const int rep = a.H / a.G;
  // Odd groups of wide keys take four heads together too, the last workgroup's spare waves idle: one head is
  // two waves, and the pages' LDS lets a CU hold two workgroups.  576 entries with 3 heads, sixteen chunks
  // of 230 rows after 416: 120 us a pass with a head a workgroup, 101 so; four prompts of 2,048: 434, 238.
  constexpr bool WIDE = SHARED && DK >= 10;
  if (rep % 4 == 0 || (WIDE && rep % 2 == 1 && rep > 1)) launch_keep_mfma_mode<DK, DV, 4, SHARED>(a);
  else if (rep % 2 == 0) launch_keep_mfma_mode<DK, DV, 2, SHARED>(a);
  else launch_keep_mfma_mode<DK, DV, 1, SHARED>(a);
}

template <int DK, int DV, int HPW, int MODE>
static void launch_keep_rows_one(const KeepArgs& a, int NA, int rows) {
  constexpr size_t lds = (size_t)2 * WBS * 32 * DK * sizeof(short);
  static bool attr = false;
  if (!attr) {
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&attn_keep_wide_kernel<DK, DV, HPW, MODE, true>),
                              hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
    attr = true;
  }
  const int per = (a.H / a.G + 32 * HPW - 1) / (32 * HPW);
  hipLaunchKernelGGL((attn_keep_wide_kernel<DK, DV, HPW, MODE, true>), dim3(NA, a.G * per, rows), dim3(128 * HPW), lds,
                     a.s, a);
}

template <int DK, int DV, int HPW>
static void launch_keep_rows_mode(const KeepArgs& a, int NA, int rows) {
  const bool cap = a.softcap > 0.f;
  if (a.sigmoid && cap) launch_keep_rows_one<DK, DV, HPW, 3>(a, NA, rows);
  else if (a.sigmoid) launch_keep_rows_one<DK, DV, HPW, 2>(a, NA, rows);
  else if (cap) launch_keep_rows_one<DK, DV, HPW, 1>(a, NA, rows);
  else launch_keep_rows_one<DK, DV, HPW, 0>(a, NA, rows);
}

void launch_attn_keep_wide_rows(const float* q, const void* k_cache, int64_t vrs, const int32_t* bt, int maxb,
                                const int32_t* q_start, const int32_t* q_len, const int32_t* kv_len, int T, int NA,
                                const float* head_bias, const void* gate, int64_t gate_stride, int gate_w, void* out,
                                int64_t out_stride, float scale, int window, int keep_first, bool sigmoid, int H, int G,
                                int E, float softcap, float out_mult, hipStream_t s) {
  const KeepArgs a{q, k_cache, k_cache, vrs, bt, maxb, q_start, q_len, kv_len, nullptr, nullptr,
                   0, head_bias, gate, gate_stride, gate_w, out, out_stride, scale, window, keep_first,
                   sigmoid, H, G, softcap, out_mult, s};
  // Rows side by side: as many as the sequences have on the average, or four, the others follow.  Heads: as
  // few a workgroup as leave no more workgroups than fit the chip, two to a CU.
  const int rep = H / G, rows = std::min(std::max((T + NA - 1) / NA, 4), T);
  auto wgs = [&](int heads) { return (int64_t)T * G * ((rep + heads - 1) / heads); };
#define ROWS_GO(dk, dv)                                                                        \
  do {                                                                                         \
    if (rep <= 32 || wgs(32) <= 512) launch_keep_rows_mode<dk, dv, 1>(a, NA, rows);            \
    else if (rep <= 64 || wgs(64) <= 512) launch_keep_rows_mode<dk, dv, 2>(a, NA, rows);       \
    else launch_keep_rows_mode<dk, dv, 4>(a, NA, rows);                                        \
  } while (0)
  if (E == 576) ROWS_GO(18, 32);
  else ROWS_GO(10, 16);
#undef ROWS_GO
}

bool launch_attn_keep_mfma(const float* q, const void* k_cache, const void* v_cache, int64_t vrs,
                           const int32_t* bt, int maxb, const int32_t* q_start,
                           const int32_t* q_len, const int32_t* kv_len, const int32_t* work_seq,
                           const int32_t* work_qblk, int W, const float* head_bias,
                           const void* gate, int64_t gate_stride, int gate_w, void* out,
                           int64_t out_stride, float scale, int window, int keep_first, bool sigmoid, int H, int G,
                           int E, int vdim, int BS, bool shared, float softcap, float out_mult,
                           hipStream_t s) {
  if (!keep_mfma_ok(E, vdim, BS, shared)) return false;
  if (W == 0) return true;
  const KeepArgs a{q, k_cache, v_cache, vrs, bt, maxb, q_start, q_len, kv_len, work_seq, work_qblk,
                   W, head_bias, gate, gate_stride, gate_w, out, out_stride, scale, window, keep_first,
                   sigmoid, H, G, softcap, out_mult, s};
  const int DK = E / 32, DV = vdim / 16;
  if (shared) {
    if (DK == 3) launch_keep_mfma_heads<3, 4, true>(a);
    else if (DK == 4 && DV == 4) launch_keep_mfma_heads<4, 4, true>(a);
    else if (DK == 4) launch_keep_mfma_heads<4, 6, true>(a);
    else if (DK == 5) launch_keep_mfma_heads<5, 8, true>(a);
    else if (DK == 6) launch_keep_mfma_heads<6, 8, true>(a);
    else if (DK == 10) launch_keep_mfma_heads<10, 16, true>(a);
    else launch_keep_mfma_heads<18, 32, true>(a);
    return true;
  }
#define KEEP_DV(DKK)                                                    \
  do {                                                                  \
    if (DV == 2) launch_keep_mfma_heads<DKK, 2, false>(a);              \
    else if (DV == 4) launch_keep_mfma_heads<DKK, 4, false>(a);         \
    else launch_keep_mfma_heads<DKK, 8, false>(a);                      \
  } while (0)
  if (DK == 1) KEEP_DV(1);
  else if (DK == 2) KEEP_DV(2);
  else if (DK == 3) KEEP_DV(3);
  else KEEP_DV(4);
#undef KEEP_DV
  return true;
}

}  // namespace rfqmix
