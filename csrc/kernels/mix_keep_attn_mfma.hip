// attn_keep_window on MFMA tiles, prompt rows (bf16 pages of 32 tokens, key width a multiple of 32,
// value width a multiple of 32).  Semantics of mix_keep_attn.hip: sliding window with kept first
// tokens; softmax, softmax with a sink, or unnormalised sigmoid weights; optional output gate
// (a column per head, or gate_w = vdim: one per output, rows 8-byte aligned);
// the values may be the leading entries of the key rows themselves (latent attention).
// Prompt rows of 576-wide latents with groups of four heads: mix_keep_latent.hip.
// Decode rows have kernels of their own: mix_keep_split.hip, mix_keep_streams.hip (wide latents, pages shared by several
// workgroups), and here those of wide latents with many heads at a time (attn_keep_wide_kernel, DEC).
//
// One workgroup per (work item, HPW heads of one key/value head); a work item is (sequence, block of 32 queries).
// A wave has the 32 queries of a head: it keeps the running maximum and sum of its query columns and the weighted
// values O^T [vdim x 32] in registers.  A key tile is one page, staged in LDS for all heads of the workgroup, the
// next ones while this one is multiplied; one barrier per page.  Pages between the kept first tokens and the window
// are never read.
//
//   S^T[key, query] = K[key, :] . Q[query, :]   v_mfma_f32_32x32x16_bf16, A = key rows from LDS, B = the queries in
//                     registers as bf16 hi + lo (they arrive in fp32 and are not rounded a second time), already
//                     times the scale and log2 e
//   cap, mask, weights per query column in fp32, base 2
//   O^T[dv, query] += V^T[dv, keys] . P^T[keys, query]   A = two transposed reads of V (ds_read_tr16_b64), B = the
//                     weights straight from the score registers as bf16 hi + lo parts (two MFMAs), so the weights
//                     keep fp32's precision
//
// What bounds it: the vector instructions between the products (five and one and a half transcendental ones to an
// MFMA) and how well they hide behind them.  A SIMD issues one in four clocks beside an MFMA of 32, one wave alone in
// six to seven; so the order is fixed piece by piece (sched_barrier): the products of the next page's scores stand
// beside this page's weights, those of this page's values beside the next page's caps and maximum, one product to
// every four or five others, operands from LDS two products ahead, page copies as LDS-DMA that nothing waits for but
// the barrier.  The maximum is looked at lane by lane and moves only when a score passes it by 2^11, pages without an
// edge inside skip the masks.  A block's workgroups lie side by side and blocks with the most keys start first, in
// front of the others on their SIMD (s_setprio): the longest block's chain of pages is the end of a short step.
// Groups of one or two heads a workgroup and short rows keep 16 queries a wave where the chip is not full
// (small_groups).
// Measured, the attention alone, against 16 x 16 tiles with a wave per 16 queries, compiler's order and heads one
// after the other: prompts of 2,048 and 600 tokens (32 heads over 8 of 128, softcap) 194 -> 90 us, five ragged
// prompts with sigmoid weights and a window of 1,024 72 -> 51 us, one prompt of 2,048 over 192-wide latents (32
// heads) 177 -> 96 us, sixteen chunks of 230 rows after 416 over two 192-wide latents of one head each 40 -> 27 us; a
// workgroup alone takes 0.86 us a page, a full chip 1.1 us a page and CU.  Two pages to a barrier, two score chains, or
// operands four products ahead changed nothing.
#include <algorithm>
#include <type_traits>

#include "common.h"
#include "mix_common.h"
#include "mix_keep_mfma.h"

namespace rfqmix {

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

template <int DK, int DV, bool SHARED>
constexpr int keep_page_shorts() {
  return WBS * (32 * DK + 8) + (SHARED ? 0 : WBS * (16 * DV + 8));
}

// DK = E / 32, DV = vdim / 16, HPW heads per workgroup, SHARED: values = leading entries of the key rows, MODE: 0
// softmax, 1 softmax of capped scores, 2 sigmoid, 3 sigmoid of capped scores.
//
// Groups of one or two heads, and short rows, where the chip is not full (small_groups): a wave has 16 queries of a
// head on 16 x 16 tiles, so that a head's 32 queries are two waves side by side, with half the weights to make each;
// pages come through registers into padded rows.  The tiles of 32 queries below leave half of the SIMDs idle there, and
// sigmoid weights, two transcendental instructions each and no maximum to wait for, are their time (eight prompts of
// 200, 12 heads over 2 of 128, sigmoid: 15 us against 17 there).  Two heads a workgroup: three waves a SIMD, which the
// compiler left to itself spends on 180 registers for two.
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

// A row's 16-byte pieces are permuted inside it, and rows of 256 bytes lie 16 bytes apart after every four, so
// that the pieces that one LDS access takes together (K: a piece of 16 neighbouring rows; V, transposed: 64
// bytes of four neighbouring rows) lie on different banks.
template <int E>
__device__ __forceinline__ int page_swizzle(int r) {
  if constexpr (E == 128) return (r & 3) << 2;
  if constexpr (E != 128 && E % 64 == 0) return ((r >> 1) & 1) << 2 | ((r >> 2) & 3);
  return (r >> 2) & 3;
}
template <int E>
constexpr int page_row(int r) { return r * E + (E == 128 ? (r >> 2) * 8 : 0); }     // shorts before row r
template <int DK, int DV, bool SHARED>
constexpr int tile_lds_shorts() { return SHARED ? 3 * page_row<32 * DK>(WBS) : 2 * (page_row<32 * DK>(WBS) + page_row<16 * DV>(WBS)); }

template <int DK, int DV, int HPW, bool SHARED, int MODE>
__global__ __launch_bounds__(64 * HPW, 2) void attn_keep_tile_kernel(const KeepArgs a) {
  constexpr int E = 32 * DK, vdim = 16 * DV, KS = 2 * DK, VM = DV / 2, NT = 64 * HPW;
  constexpr int VR = SHARED ? E : vdim;                      // shorts per row of the values' image
  constexpr int KP = page_row<E>(WBS), VP = page_row<VR>(WBS);
  const int groups = a.H / HPW;
  const int at = gridDim.x - 1 - blockIdx.x;       // a sequence's later blocks see the most keys: they start first
  const int item = at / groups;
  int hg = at - item * groups;
  if (a.turned && (hg += item % groups) >= groups) hg -= groups;
  const int s = a.work_seq[item];
  if (s < 0) return;
  const int ql = a.q_len[s];
  const int i0 = a.work_qblk[item] * WQB;
  if (i0 >= ql) return;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col = lane & 31, half = lane >> 5;
  const int hh = hg * HPW + wid, g = hg * HPW / (a.H / a.G);
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const uint32_t lds0 = lds_byte(smem);
  short* const kpages = reinterpret_cast<short*>(smem);
  short* const vpages = SHARED ? kpages : kpages + 2 * KP;

  const int nq = min(WQB, ql - i0);
  const int p0 = a.kv_len[s] - ql + i0, plast = p0 + nq - 1;
  const int window = a.window, keep_first = a.keep_first;
  const int jwin = window > 0 ? max(0, p0 - window + 1) : 0;
  const int kf = window > 0 ? min(keep_first, jwin) : 0;     // kept keys before the window
  const int pi = p0 + col;                                   // this lane's query
  const bool qlive = col < nq;
  const int64_t t = a.q_start[s] + i0 + (qlive ? col : 0);
  typedef const __attribute__((address_space(4))) int32_t const_i32;
  const_i32* bt = (const_i32*)(uintptr_t)(a.bt + (int64_t)s * a.maxb);

  // pages [0, n_keep) hold the kept first tokens, pages [pg_win, pg_last] the window
  const int pg_last = plast / WBS, pg_win = jwin / WBS;
  const int n_keep = min((kf + WBS - 1) / WBS, pg_win), skip = pg_win - n_keep, turns = pg_last + 1 - skip;
  // Long chains in front of the short ones that share their SIMD.  Over fourteen mixes of prompts, three head counts and
  // three sizes it is worth half a percent: up to 11 % where long and short prompts or odd numbers of blocks meet, and
  // 3 - 8 % lost on prompts of one length and on 192-wide rows.
  if (turns >= 32) __builtin_amdgcn_s_setprio(3);
  else if (turns >= 20) __builtin_amdgcn_s_setprio(2);
  else if (turns >= 10) __builtin_amdgcn_s_setprio(1);
  auto page_at = [&](int i) { return i < n_keep ? i : i + skip; };
  auto number = [&](int i) { return bt[page_at(min(i, turns - 1))]; };

  // ---- staging: LDS-DMA, 64 pieces of 16 bytes a time, permuted at the source
  constexpr int NPK = WBS * E / 512, NPV = SHARED ? 0 : WBS * vdim / 512;
  constexpr int NK = (NPK + HPW - 1) / HPW, NV = (NPV + HPW - 1) / HPW;
  // rows 16 apart are permuted alike: a wave whose pieces lie so needs the offsets of half of them
  constexpr int UK = NPK % (2 * HPW) == 0 ? NK / 2 : NK, UV = NPV % (2 * HPW) == 0 ? NV / 2 : NV;
  uint32_t ksrc[UK], vsrc[UV > 0 ? UV : 1];
#pragma unroll
  for (int i = 0; i < UK; ++i) {
    const int x = (wid + i * HPW) * 64 + lane, r = x / (E / 8), c = x - r * (E / 8);
    ksrc[i] = (r * E + (c ^ page_swizzle<E>(r)) * 8) * 2;
  }
#pragma unroll
  for (int i = 0; i < UV; ++i) {
    const int x = (wid + i * HPW) * 64 + lane, r = x / (vdim / 8), c = x - r * (vdim / 8);
    vsrc[i] = (r * (int)a.vrs + (c ^ page_swizzle<vdim>(r)) * 8) * 2;
  }
  auto fetch_k = [&](int page, int buf) {
    const char* kb = static_cast<const char*>(a.k_cache) + ((int64_t)page * a.G + g) * WBS * E * 2;
#pragma unroll
    for (int i = 0; i < NK; ++i) {
      const int piece = wid + i * HPW;
      if ((i + 1) * HPW <= NPK || piece < NPK)
        lds_copy16(kb + i / UK * (WBS * E), ksrc[i % UK], lds0 + 2 * (buf * KP + piece * (E == 128 ? 520 : 512)));
    }
  };
  auto fetch_v = [&](int page, int buf) {
    if constexpr (!SHARED) {
      const char* vb = static_cast<const char*>(a.v_cache) + ((int64_t)page * a.G + g) * WBS * a.vrs * 2;
#pragma unroll
      for (int i = 0; i < NV; ++i) {
        const int piece = wid + i * HPW;
        if ((i + 1) * HPW <= NPV || piece < NPV)
          lds_copy16(vb + i / UV * (WBS * a.vrs), vsrc[i % UV], lds0 + 2 * (2 * KP + buf * VP + piece * (vdim == 128 ? 520 : 512)));
      }
    }
  };
  int32_t n0 = number(0), n1 = number(1), n2 = number(2);    // numbers of the pages of this turn, the next two
  fetch_k(n0, 0);
  fetch_v(n0, 0);
  if (turns > 1) fetch_k(n1, 1);

  // scores arrive as exponents of 2: s log2 e; 2 s log2 e / cap; -s log2 e (sigmoid, no cap)
  const float qmul = a.scale * (MODE % 2 == 1 ? 2.f * kLog2e / a.softcap : MODE == 2 ? -kLog2e : kLog2e);
  const float cap2 = MODE % 2 == 1 ? a.softcap * kLog2e : 0.f;
  s16x8 qhi[KS], qlo[KS];
  {
    const float* qp = a.q + (t * a.H + hh) * E + half * 8;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const float4 x = *reinterpret_cast<const float4*>(qp + ks * 16);
      const float4 y = *reinterpret_cast<const float4*>(qp + ks * 16 + 4);
      const float f[8] = {x.x * qmul, x.y * qmul, x.z * qmul, x.w * qmul, y.x * qmul, y.y * qmul, y.z * qmul, y.w * qmul};
      split_bf16w(f, qhi[ks], qlo[ks]);
    }
  }
  f32x16 o[VM];
#pragma unroll
  for (int m = 0; m < VM; ++m)
#pragma unroll
    for (int i = 0; i < 16; ++i) o[m][i] = 0.f;
  const float hb = a.head_bias != nullptr ? a.head_bias[hh] * kLog2e : 0.f;
  const bool sink = MODE < 2 && a.head_bias != nullptr;
  // the sink is one more entry of the row: it starts the maximum, and one lane's part of the sum
  float mrun = sink ? hb : kNegInfW, lrun = sink && half == 0 ? 1.f : 0.f;

  // keys: row col, entries 16 ks + 8 half ..; values, transposed: rows 16 t + 8 j + 4 half + lane % 16 / 4,
  // channels 32 m + 16 (lane / 16 % 2) + 4 (lane % 4) ..
  constexpr int KA = E % 64 == 0 ? 4 : 2, KI = E == 128 ? 2 : 1;       // KI neighbouring pieces at a fixed distance
  constexpr int VA = VR == 128 ? 4 : VR % 64 == 0 ? 2 : 1, VJ = VR == 128 ? 1 : 2;
  int kat[KA], vat[VJ][VA];
#pragma unroll
  for (int i = 0; i < KA; ++i) kat[i] = page_row<E>(col) + ((2 * KI * i + half) ^ page_swizzle<E>(col)) * 8;
#pragma unroll
  for (int j = 0; j < VJ; ++j)
#pragma unroll
    for (int i = 0; i < VA; ++i) {
      const int r = 8 * j + 4 * half + ((lane & 15) >> 2);
      vat[j][i] = page_row<VR>(r) + ((4 * i + 2 * ((lane >> 4) & 1) + ((lane & 3) >> 1)) ^ page_swizzle<VR>(r)) * 8 + (lane & 1) * 4;
    }

  auto key = [&](const short* Ks, int ks) {
    return *reinterpret_cast<const s16x8*>(Ks + kat[ks / KI % KA] + (ks % KI) * 16 + (ks / (KI * KA)) * KI * KA * 16);
  };
  auto value = [&](const short* Vs, int c) {                 // 16 keys (c / VM) x 32 channels (c % VM)
    const int u = c / VM, m = c % VM;
    const short* vp = Vs + (m / VA) * VA * 32 + vat[0][m % VA] + page_row<VR>(16 * u);
    const short* vq = Vs + (m / VA) * VA * 32 + vat[VJ - 1][m % VA] + page_row<VR>(16 * u + (VJ == 1 ? 8 : 0));
    const s16x4 a0 = rfq::ds_read_tr16(vp), a1 = rfq::ds_read_tr16(vq);
    return (s16x8){a0[0], a0[1], a0[2], a0[3], a1[0], a1[1], a1[2], a1[3]};
  };
  float p[16], top = kNegInfW;
  // What a score becomes before the maximum is known.  Capped: cap2 - 2 cap2 / (2^x + 1), here the quotient,
  // which falls where the score rises; sigmoid: the weight itself.
  auto prepare = [&](int i, float x) {
    if constexpr (MODE % 2 == 1) x = __builtin_amdgcn_rcpf(__builtin_amdgcn_exp2f(x) + 1.f);
    if constexpr (MODE == 3) x = 2.f * cap2 * x - cap2;
    if constexpr (MODE >= 2) x = __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(x - hb));
    p[i] = x;
    if constexpr (MODE < 2) top = i == 0 ? x : MODE == 1 ? fminf(top, x) : fmaxf(top, x);
  };
  auto mask = [&](int jb) {                                  // a page with an edge inside
    if (jb + WBS - 1 <= p0 && (window <= 0 || plast - jb < window || jb + WBS <= keep_first)) return;
    const int at = jb + half * 4, hi = pi - at, lo = window > 0 ? hi - window : -WBS, kept = keep_first - at;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int j = (i >> 2) * 8 + (i & 3);
      const bool ok = (j <= hi) & ((j > lo) | (j < kept));
      const float x = ok ? p[i] : MODE >= 2 ? 0.f : MODE == 1 ? -kNegInfW : kNegInfW;
      p[i] = x;
      if constexpr (MODE < 2) top = i == 0 ? x : MODE == 1 ? fminf(top, x) : fmaxf(top, x);
    }
  };
  auto passes = [&]() { return MODE == 1 ? cap2 - 2.f * cap2 * top : top; };   // this lane's largest score

  auto landed = [] {
    __builtin_amdgcn_s_waitcnt(0x0F70);                      // vmcnt(0)
    __syncthreads();
  };
  // One turn: the weighted values of page i, whose scores p has, and the scores of page i + 1.  The order is
  // kept piece by piece: products of the next page's scores beside the weights of this one, products of this
  // page's values beside the next page's caps and maximum.
  auto turn = [&](int i, auto next_c) {
    constexpr bool NEXT = next_c;                            // there is a next page
    const short* Kn = kpages + (SHARED ? (i + 1) % 3 : (i + 1) & 1) * KP;
    const short* Vs = vpages + (SHARED ? i % 3 : i & 1) * VP;
    // operands are read that many pieces ahead
    constexpr int AK = DK > 4 ? 1 : 2, AV = AK;
    s16x8 kc[AK], vc[AV];
    if constexpr (NEXT) {
#pragma unroll
      for (int x = 0; x < AK; ++x) kc[x] = key(Kn, x);
    }
    const float mu = mrun == kNegInfW ? 0.f : mrun;          // no visible key so far: every weight 0
    const float top0 = cap2 - mu;
    u32x4 phi[2], plo[2];
    // the weights of keys 2 e and 2 e + 1, in two steps
    auto weigh = [&](int e) {
      if constexpr (MODE < 2) {
        p[2 * e] = __builtin_amdgcn_exp2f(MODE == 1 ? top0 - 2.f * cap2 * p[2 * e] : p[2 * e] - mu);
        p[2 * e + 1] = __builtin_amdgcn_exp2f(MODE == 1 ? top0 - 2.f * cap2 * p[2 * e + 1] : p[2 * e + 1] - mu);
      }
    };
    auto parts = [&](int e) {
      const float x = p[2 * e], y = p[2 * e + 1];
      if constexpr (MODE < 2) lrun += x + y;
      const uint32_t h = rfq::pack_bf16x2(x, y);
      phi[e >> 2][e & 3] = h;
      plo[e >> 2][e & 3] = rfq::pack_bf16x2(x - __uint_as_float(h << 16), y - __uint_as_float(h & 0xffff0000u));
    };
    auto add = [&](const s16x8& v, int c, const u32x4& w) {
      o[c % VM] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(as_bf16x8(v), __builtin_bit_cast(rfq::bf16x8, w), o[c % VM], 0, 0, 0);
    };
    f32x16 sn;
    constexpr int C = 2 * VM;
    if constexpr (NEXT) {
#pragma unroll
      for (int e = 0; e < 16; ++e) sn[e] = 0.f;
      each<KS>([&](auto step) {
        constexpr int ks = step, e0 = 8 * ks / KS, e1 = 8 * (ks + 1) / KS;
        const s16x8 k = kc[ks % AK];
        if constexpr (ks + AK < KS) kc[ks % AK] = key(Kn, ks + AK);
        if constexpr (ks + AV >= KS) vc[ks + AV - KS] = value(Vs, ks + AV - KS);
        sn = __builtin_amdgcn_mfma_f32_32x32x16_bf16(as_bf16x8(k), as_bf16x8(qhi[ks]), sn, 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
        each<e1 - e0>([&](auto e) { weigh(e0 + e); });
        __builtin_amdgcn_sched_barrier(0);
        sn = __builtin_amdgcn_mfma_f32_32x32x16_bf16(as_bf16x8(k), as_bf16x8(qlo[ks]), sn, 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
        each<e1 - e0>([&](auto e) { parts(e0 + e); });
        __builtin_amdgcn_sched_barrier(0);
      });
    } else {
#pragma unroll
      for (int x = 0; x < AV; ++x) vc[x] = value(Vs, x);
#pragma unroll
      for (int e = 0; e < 8; ++e) weigh(e);
#pragma unroll
      for (int e = 0; e < 8; ++e) parts(e);
    }
    // two products a piece of values, the second beside the next piece's first; from the third product on the
    // next page's scores are there
    s16x8 before;
    constexpr int Q = VM > 1 ? 4 * VM - 2 : 1;
    auto some = [&](auto nc) {
      if constexpr (NEXT) {
        if constexpr (nc >= 0) {
          constexpr int e0 = 16 * nc / Q, e1 = 16 * (nc + 1) / Q;
          each<e1 - e0>([&](auto e) { prepare(e0 + e, sn[e0 + e]); });
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    };
    each<C>([&](auto step) {
      constexpr int c = step;
      const s16x8 v = vc[c % AV];
      if constexpr (c + AV < C) vc[c % AV] = value(Vs, c + AV);
      if constexpr (VM == 1 && c > 0) {
        add(before, c - 1, plo[(c - 1) / VM]);
        some(std::integral_constant<int, 2 * c - 3>{});
      }
      add(v, c, phi[c / VM]);
      some(std::integral_constant<int, 2 * c - 2>{});
      if constexpr (VM > 1 && c > 0) {
        add(before, c - 1, plo[(c - 1) / VM]);
        some(std::integral_constant<int, 2 * c - 1>{});
      }
      before = v;
    });
    add(before, C - 1, plo[1]);
    __builtin_amdgcn_sched_barrier(0);
  };

  // K of page i + 1 and V of page i have landed for everyone, and everyone is done with K of page i and V of
  // page i - 1, whose places the next ones take.
  auto next = [&](int i) {
    landed();
    if (i + 2 < turns) fetch_k(n2, SHARED ? (i + 2) % 3 : i & 1);
    fetch_v(n1, (i + 1) & 1);
    n1 = n2;
    n2 = number(i + 3);
  };
  // rows past the sequence's end were never written: zeros
  auto last = [&]() {
    landed();
    const int jb = page_at(turns - 1) * WBS;
    if (jb + WBS - 1 > plast) {
      short* Vs = vpages + (SHARED ? (turns - 1) % 3 : (turns - 1) & 1) * VP;
      for (int x = max(0, plast + 1 - jb) * (VR / 8) + tid; x < WBS * (VR / 8); x += NT)
        *reinterpret_cast<s16x8*>(Vs + page_row<VR>(x / (VR / 8)) + x % (VR / 8) * 8) = (s16x8){0, 0, 0, 0, 0, 0, 0, 0};
      __syncthreads();
    }
  };
  landed();
  {
    f32x16 sc;
#pragma unroll
    for (int e = 0; e < 16; ++e) sc[e] = 0.f;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const s16x8 k = key(kpages, ks);
      sc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(as_bf16x8(k), as_bf16x8(qhi[ks]), sc, 0, 0, 0);
      sc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(as_bf16x8(k), as_bf16x8(qlo[ks]), sc, 0, 0, 0);
    }
#pragma unroll
    for (int e = 0; e < 16; ++e) prepare(e, sc[e]);
    mask(page_at(0) * WBS);
  }
  int i = 0;
  while (true) {
    if constexpr (MODE < 2) {                                // the maximum moves; also for the first keys: mrun = -inf
      const float mx = other_half_max(passes());
      const bool moves = mx > mrun + kDeferW;
      const float mn = moves ? mx : mrun;
      const float alpha = moves ? __builtin_amdgcn_exp2f(mrun - mn) : 1.f;
      mrun = mn;
      lrun *= alpha;
#pragma unroll
      for (int m = 0; m < VM; ++m) o[m] *= alpha;
    }
    bool stays = true;
    while (stays && i + 1 < turns) {
      next(i);
      turn(i, std::true_type{});
      ++i;
      mask(page_at(i) * WBS);
      if constexpr (MODE < 2) stays = __builtin_amdgcn_ballot_w64(passes() > mrun + kDeferW) == 0ull;
    }
    if (stays) break;
  }
  last();
  turn(i, std::false_type{});
  store_tiles32<VM>(a, o, row_factor<MODE>(a, both_halves_sum(lrun), t, hh), t, hh, vdim, 0, half, qlive);
}

// Wide latents: keys of 320 entries whose first 256 are the values; of 576 and 512 in groups of two heads or of one
// (groups of four and odd ones: mix_keep_latent.hip).  32 queries' results (256 registers at 512 values) and the queries
// themselves (144) leave no room for the rest, so a wave has 16 queries on 16x16x32 tiles, two waves a head: a page's
// LDS reads are K rows 36 x 1 KB, V 64 x 512 B a wave at 576.  A block's heads lie side by side: one after the other the
// last heads' long blocks started at seven eighths of the time.  Pages come by LDS-DMA, the next one during this one;
// their rows lie unpadded, 16-byte pieces permuted inside each 128 bytes by wide_swizzle(row).  576 entries in groups
// of two, 16 heads over 8, two prompts of 2,048: 237 us; a workgroup of four heads, half of them idle, took 358.
// DEC: decode rows.  A wave's columns are 16 heads of one row, so that a workgroup reads a page once for up to
// 128 heads; the pages come one after another, which pays once every CU has a workgroup (launch_split_waves).
// 256 sequences of 300 tokens with 64 heads of 576 entries 44 us, 32 of 500 with four rows each 50; split over
// waves 116 and 129.
template <int DK, int DV, int HPW, int MODE, bool DEC>
__global__ __launch_bounds__(128 * HPW, DEC && HPW == 1 ? 1 : 2) void attn_keep_wide_kernel(const KeepArgs a) {
  constexpr int E = 32 * DK, vdim = 16 * DV, NWV = 2 * HPW, NP = WBS * E / 512, ND = (NP + NWV - 1) / NWV;
  constexpr bool QLO = DK <= 10;
  static_assert(E % 64 == 0 && DV % 4 == 0, "whole 128-byte lines");
  // prompts: a block's workgroups lie side by side, a sequence's later blocks, which see the most keys, start first
  constexpr int HW = DEC ? 16 * NWV : HPW;                    // heads of a workgroup
  const int rep = a.H / a.G, per = (rep + HW - 1) / HW;       // workgroups of a key head, the last partly idle
  const int at = gridDim.x - 1 - blockIdx.x, item = DEC ? at : at / (a.G * per), hg = DEC ? (int)blockIdx.y : at - item * a.G * per;
  const int s = DEC ? item : a.work_seq[item];
  if (s < 0) return;
  const int ql = a.q_len[s];
  const int i0 = DEC ? 0 : a.work_qblk[item] * WQB;
  if (i0 >= ql) return;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col = lane & 15, grp = lane >> 4;
  const int g = hg / per, h0 = (hg - g * per) * HW;
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
  const uint32_t lds0 = lds_byte(smem);
  auto fetch = [&](int page, int buf) {
    const char* kb = static_cast<const char*>(a.k_cache) + ((int64_t)page * a.G + g) * WBS * E * 2;
#pragma unroll
    for (int i = 0; i < ND; ++i) {
      const int piece = wid + i * NWV;
      uint32_t at = src[i];
      asm("" : "+v"(at));      // widened here: hoisted out of the loop the offsets are pairs of registers, spilled
      if ((i + 1) * NWV <= NP || piece < NP)
        lds_copy16(kb, at, lds0 + 2 * (buf * WBS * E + piece * 512));
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
  constexpr size_t lds = (size_t)(WIDE ? 2 * WBS * 32 * DK : tile_lds_shorts<DK, DV, SHARED>()) * sizeof(short);
  static_assert(lds <= 160 * 1024, "LDS of a CU");
  static bool attr = false;
  auto run = [&](auto kernel, int threads) {
    if (!attr) {
      (void)hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                                160 * 1024);
      attr = true;
    }
    const int rep = a.H / a.G;
    const int groups = a.G * ((rep + HPW - 1) / HPW), most = std::max(1, (1 << 22) / groups);   // threads in 32 bits
    // Heads side by side put a head group's blocks on one XCD where there are eight of them: each reads only its key
    // heads' pages (32 heads over 8 of 128, sigmoid: 400 tokens 29.4 us a pass with the append, 32.1 with the groups
    // turned by one from block to block), but its L2 sees an eighth of every row's columns, which costs the kernel
    // that writes the next rows up to 4 us while queries and results just fill the L2s (780 tokens 46.5 against 42.9,
    // 900 50.8 and 47.2; 64 heads, 500 tokens 40.8 and 38.8).  From 24 MB of queries on neither matters, with softmax
    // weights they are even, and under eight pages the blocks' common pages count for more (16 prompts of 64 30.2, 31.5).
    const int64_t queries = (int64_t)a.W * WQB * a.H * 32 * DK * sizeof(float);
    for (int w = 0; w < a.W; w += most) {
      KeepArgs part = a;
      part.turned = MODE >= 2 && a.maxb >= 8 && queries > (8 << 20) && queries <= (24 << 20);
      part.work_seq += w;
      part.work_qblk += w;
      hipLaunchKernelGGL(kernel, dim3((unsigned)std::min(most, a.W - w) * groups), dim3(threads), lds, a.s, part);
    }
  };
  if constexpr (DK == 18 && HPW == 4) return launch_attn_keep_latent(a);
  else if constexpr (WIDE) run(&attn_keep_wide_kernel<DK, DV, HPW, MODE, false>, 128 * HPW);
  else run(&attn_keep_tile_kernel<DK, DV, HPW, SHARED, MODE>, 64 * HPW);
}

// Steps whose 32 queries of a head are better two waves, by the heads of a workgroup and its number `wgs`.
// One or two heads: rows of up to three pages, where the way to the first page is the time (one prompt of 33 tokens,
// two heads a group: 0.91 - 0.97 of the other kernel's time; of one head a group only sigmoid weights of latents, 0.88 -
// 0.97), and sigmoid weights of two heads up to 1,024 workgroups, four waves to a CU of the other kernel (1 - 32 prompts
// of 33 - 1,200 tokens: 0.75 - 1.0 of its time, where it has fewer than 512; from 1,024 on the other is as fast or takes
// down to 0.6 of this one's).
// Four heads are eight waves here, a workgroup to a CU: where that is one round, sigmoid weights over up to four pages,
// over up to eight if most CUs have one, and any weights over two (passes with the append, 16 heads over 4 of 128: 8
// prompts of 64 17.9 us against 19.3, 32 of them 28.2 and 31.0, softcap 34.3 and 35.7; 32 over 8, 4 of 200: 29.7 and
// 32.0, 8 of 128 29.4 and 31.7; longer prompts 0 - 6 % the other way round).
template <int HPW, bool SHARED, int MODE>
static bool small_groups(const KeepArgs& a) {
  const int64_t wgs = (int64_t)a.W * (a.H / HPW);
  if (a.W > (1 << 22)) return false;               // a grid's threads in 32 bits; the other kernel's launches are cut
  if constexpr (HPW == 1) return SHARED && MODE >= 2 && a.maxb <= 3;
  if constexpr (HPW == 2) return a.maxb <= 3 || (MODE >= 2 && wgs < 1024);
  return wgs <= 256 && ((MODE >= 2 && a.maxb <= 4) || (wgs > 192 && a.maxb <= (MODE >= 2 ? 8 : 2)));
}

template <int DK, int DV, int HPW, bool SHARED, int MODE>
static void launch_keep_small_one(const KeepArgs& a) {
  constexpr size_t lds = (size_t)2 * keep_page_shorts<DK, DV, SHARED>() * sizeof(short);
  static_assert(lds <= 64 * 1024, "LDS without an allowance");
  hipLaunchKernelGGL((attn_keep_mfma_kernel<DK, DV, HPW, SHARED, MODE>), dim3(a.W, a.H / HPW), dim3(128 * HPW), lds, a.s, a);
}

template <int DK, int DV, int HPW, bool SHARED, int MODE>
static void launch_keep_mfma_any(const KeepArgs& a) {
  if constexpr (!(SHARED && DK >= 10) && (HPW > 1 || (SHARED && MODE >= 2)))
    if (small_groups<HPW, SHARED, MODE>(a)) return launch_keep_small_one<DK, DV, HPW, SHARED, MODE>(a);
  launch_keep_mfma_one<DK, DV, HPW, SHARED, MODE>(a);
}

template <int DK, int DV, int HPW, bool SHARED>
static void launch_keep_mfma_mode(const KeepArgs& a) {
  const bool cap = a.softcap > 0.f;
  if (a.sigmoid && cap) launch_keep_mfma_any<DK, DV, HPW, SHARED, 3>(a);
  else if (a.sigmoid) launch_keep_mfma_any<DK, DV, HPW, SHARED, 2>(a);
  else if (cap) launch_keep_mfma_any<DK, DV, HPW, SHARED, 1>(a);
  else launch_keep_mfma_any<DK, DV, HPW, SHARED, 0>(a);
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
