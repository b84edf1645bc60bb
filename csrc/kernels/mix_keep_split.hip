// attn_keep_window for decode rows on MFMA tiles, a sequence's pages split over the waves of a
// workgroup (bf16 pages of 32 tokens; semantics of mix_keep_attn.hip).
//
// What bounds it: the pages' bytes.  A workgroup per (sequence, key/value head) that walked the pages
// one after the other took, with fp32 FMAs, 162 us for 64 sequences of 300 - 900 tokens with 32 heads
// over 8 key/value heads of 128 (166 MB: 1.0 TB/s) and 96 us for one such sequence, whose eight
// workgroups had nothing beside them; for 64 sequences of a 576-wide latent with 32 heads, on MFMA
// tiles, 121 us.  Here every wave takes every NW-th piece: its key rows go from memory straight into
// MFMA operands, its value rows through the wave's own piece of LDS (read back transposed), the next
// rows are in flight meanwhile, and no wave waits for another until the partial results (running
// maximum, sum, weighted values) meet in LDS at the end.  Measured: 37 us (4.5 TB/s; 44 where no cache holds the pages),
// 15 us and 54 us.  (Groups of up to eight heads with keys and values of 64 or 128, no more rows than sequences, do not
// come here: mix_keep_row.hip.  Nor do steps of the 576-wide latent with more than 16 heads, no more rows than sequences
// and more than 13 pages to see while CUs are free: a row's pages are split over workgroups as well, mix_keep_streams.hip.)
//
// The 16 MFMA columns are (row, head) pairs of one key/value head, so the rows of a short extend and
// the heads of a group share one pass.
//   S^T[key, column] = K . Q^T, the fp32 queries as sums of bf16; O^T = V^T . P^T, the weights likewise
// Groups of fewer than 16 heads take three parts of each, all of fp32's bits; wider ones two parts of the
// weights, and of the queries two for keys of up to 320 entries, one above.
//
// SHARED (latent attention): a page's rows are keys and, their leading entries, values: staged once
// in LDS, read as they lie for S and transposed for O.
#include <algorithm>
#include <type_traits>

#include "common.h"
#include "mix_common.h"
#include "mix_keep_split.h"

namespace rfqmix {

namespace {
// keys per turn: a page, or half of one where queries and results of a wide latent fill the registers
template <int DK, bool SHARED>
constexpr int turn_keys() { return SHARED && DK >= 10 ? 16 : PG; }
// and there the queries stay in LDS and two turns' rows are in flight
template <int DK, bool SHARED>
constexpr int turns_ahead() { return SHARED && DK >= 10 ? 2 : 1; }
template <int DK, int DV, bool SHARED>
constexpr int stage_row() { return SHARED ? 32 * DK + 8 : 16 * DV + 8; }      // shorts per staged row
// bf16 parts of a query entry
template <int DK, bool EXACT>
constexpr int query_parts() { return EXACT ? 3 : DK <= 10 ? 2 : 1; }
// the partial results meet in as many passes: beside three parts of a wide latent's queries one is too large
template <int DV, int NW, bool EXACT>
constexpr int merge_passes() { return EXACT && DV > 16 ? 2 : 1; }
// a wave's LDS: its staged page, later a pass of its 16 x vdim partial results (4 floats between rows)
template <int DK, int DV, bool SHARED, int NW, bool EXACT>
constexpr int wave_lds() {
  return std::max(turn_keys<DK, SHARED>() * stage_row<DK, DV, SHARED>() * 2,
                  16 * (16 * DV / merge_passes<DV, NW, EXACT>() + 4) * 4);
}
}  // namespace

void launch_attn_keep_wide_rows(const float*, const void*, int64_t, const int32_t*, int, const int32_t*, const int32_t*,
                                const int32_t*, int, int, const float*, const void*, int64_t, int, void*, int64_t, float,
                                int, int, bool, int, int, int, float, float, hipStream_t);   // mix_keep_attn_mfma.hip

// EXACT (groups of fewer than 16 heads): queries, weights and their functions in full fp32.
template <int DK, int DV, bool SHARED, int NW, bool EXACT>
__global__ __launch_bounds__(64 * NW, SHARED && DK >= 10 ? 1 : 2) void attn_keep_split_kernel(const KeepSplitArgs a) {
  constexpr int E = 32 * DK, vdim = 16 * DV, SR = stage_row<DK, DV, SHARED>();
  constexpr int KS = turn_keys<DK, SHARED>(), KT = KS / 16, AHEAD = turns_ahead<DK, SHARED>();
  constexpr bool QLDS = AHEAD == 2;
  constexpr int QR = E + 8;                              // shorts per query row in LDS
  constexpr int MG = DV % 4 == 0 ? 4 : 2;                // value blocks taken together
  constexpr int QP = query_parts<DK, EXACT>(), PP = EXACT ? 3 : 2;   // parts of a query entry, of a weight
  constexpr int WL = wave_lds<DK, DV, SHARED, NW, EXACT>(), MP = merge_passes<DV, NW, EXACT>(), VP = vdim / MP;
  const int s = blockIdx.x, g = blockIdx.y;
  const int ql = a.q_len[s], kvl = a.kv_len[s];
  const int rep = a.H / a.G;
  const int tiles = (ql * rep + 15) / 16;
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col = lane & 15, grp = lane >> 4;
  // page numbers by scalar loads: a vector load would be waited for behind the rows in flight
  typedef const __attribute__((address_space(4))) int32_t const_i32;
  const_i32* bt = (const_i32*)(uintptr_t)(a.bt + (int64_t)s * a.maxb);
  const int64_t t_first = a.q_start[s];

  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  short* St = reinterpret_cast<short*>(smem + (size_t)w * WL);
  float* part = reinterpret_cast<float*>(St);            // [16][VP + 4]
  float* ml = reinterpret_cast<float*>(smem + (size_t)NW * WL);   // [NW][16] m, [NW][16] l
  short* Qs = reinterpret_cast<short*>(ml + 2 * NW * 16);       // QLDS: [QP][16][QR]

  for (int ct = blockIdx.z; ct < tiles; ct += gridDim.z) {
    const int c = ct * 16 + col;                         // this lane's (row, head)
    const bool live = c < ql * rep;
    const int row = live ? c / rep : ql - 1, hh = g * rep + (live ? c - row * rep : 0);
    const int pi = kvl - ql + row;
    const int r_first = ct * 16 / rep, r_last = min(ql - 1, (ct * 16 + 15) / rep);
    const int p_first = kvl - ql + r_first, p_last = kvl - ql + r_last;
    const int jwin = a.window > 0 ? max(0, p_first - a.window + 1) : 0;
    const int kf = a.window > 0 ? min(a.keep_first, jwin) : 0;
    // pieces [0, n_keep) of KS keys hold the kept first tokens, [k_win, k_last] the window
    const int k_last = p_last / KS, k_win = jwin / KS;
    const int n_keep = min((kf + KS - 1) / KS, k_win);
    const int n_turns = n_keep + k_last - k_win + 1;
    auto keys_at = [&](int i) { return (i < n_keep ? i : k_win + i - n_keep) * KS; };

    s16x8 qr[QLDS ? 1 : DK][QP];
    if constexpr (QLDS) {
      for (int x = tid; x < 16 * (E / 8); x += 64 * NW) {
        const int cc = x / (E / 8), e = (x - cc * (E / 8)) * 8, cx = min(ct * 16 + cc, ql * rep - 1), r = cx / rep;
        const float* qp = a.q + ((t_first + r) * a.H + g * rep + cx - r * rep) * E + e;
        const float4 u = *reinterpret_cast<const float4*>(qp), v = *reinterpret_cast<const float4*>(qp + 4);
        const float f[8] = {u.x, u.y, u.z, u.w, v.x, v.y, v.z, v.w};
        s16x8 p[QP];
        split_parts<EXACT>(f, p);
#pragma unroll
        for (int n = 0; n < QP; ++n) *reinterpret_cast<s16x8*>(Qs + (16 * n + cc) * QR + e) = p[n];
      }
      __syncthreads();
    } else {
      // an operand's eight entries: keys straight from memory take 16 neighbouring entries in two
      // steps, so that a row's line is read whole by two loads; staged keys take eight
      const float* qp = a.q + ((t_first + row) * a.H + hh) * E;
#pragma unroll
      for (int ks = 0; ks < DK; ++ks) {
        const int at = SHARED || DK % 2 != 0 ? ks * 32 + grp * 8 : (ks >> 1) * 64 + grp * 16 + (ks & 1) * 8;
        float f[8];
        const float4 x = *reinterpret_cast<const float4*>(qp + at);
        const float4 y = *reinterpret_cast<const float4*>(qp + at + 4);
        f[0] = x.x; f[1] = x.y; f[2] = x.z; f[3] = x.w; f[4] = y.x; f[5] = y.y; f[6] = y.z; f[7] = y.w;
        split_parts<EXACT>(f, qr[ks]);
      }
    }
    f32x4 o[DV];
#pragma unroll
    for (int m = 0; m < DV; ++m) o[m] = (f32x4){0.f, 0.f, 0.f, 0.f};
    const float hb = a.head_bias != nullptr ? a.head_bias[hh] : 0.f;
    float mrun = kNegInfS, lrun = 0.f;

    constexpr int NS = KS * (SHARED ? E : vdim) / 8 / 64;   // 16-byte pieces of staged rows per lane
    // A lane's pieces lie at fixed distances where a row is whole 128-byte lines: eight lanes to a line,
    // eight rows to a load
    constexpr int WD = SHARED ? E : vdim, LN = WD / 64;
    constexpr bool LINES = WD % 64 == 0;
    auto piece_row = [&](int x) { return LINES ? x / (LN > 0 ? LN : 1) * 8 + (lane >> 3) : (lane + 64 * x) / (WD / 8); };
    auto piece_at = [&](int x) {
      return LINES ? x % (LN > 0 ? LN : 1) * 64 + (lane & 7) * 8 : (lane + 64 * x) % (WD / 8) * 8;
    };
    s16x8 sreg[AHEAD][NS], kreg[SHARED ? 1 : KT][SHARED ? 1 : DK];
    auto fetch = [&](int jb, int32_t page, auto set) {
      const int64_t at = ((int64_t)page * a.G + g) * PG + jb % PG;            // the first key's slot
      const bf16_t* kp = a.k_cache + at * E;
      if constexpr (SHARED) {
#pragma unroll
        for (int i = 0; i < NS; ++i)
          sreg[set][i] = *reinterpret_cast<const s16x8*>(kp + piece_row(i) * E + piece_at(i));
      } else {
        const bf16_t* vp = a.v_cache + at * a.vrs;
#pragma unroll
        for (int kt = 0; kt < KT; ++kt)
#pragma unroll
          for (int ks = 0; ks < DK; ++ks) {
            const int e0 = DK % 2 != 0 ? ks * 32 + grp * 8 : (ks >> 1) * 64 + grp * 16 + (ks & 1) * 8;
            kreg[kt][ks] = *reinterpret_cast<const s16x8*>(kp + (kt * 16 + col) * E + e0);
          }
#pragma unroll
        for (int i = 0; i < NS; ++i) {
          sreg[set][i] = *reinterpret_cast<const s16x8*>(vp + piece_row(i) * a.vrs + piece_at(i));
        }
      }
    };
    // a turn's rows are read AHEAD turns ahead, its page number one more; past the last turn the last
    // one's again (a load in every turn: the wave then knows how many are behind the one it waits for)
    constexpr std::integral_constant<int, 0> even{};
    constexpr std::integral_constant<int, AHEAD - 1> odd{};
    auto page_of = [&](int i) { return bt[keys_at(min(i, n_turns - 1)) / PG]; };
    auto first_key = [&](int i) { return keys_at(min(i, n_turns - 1)); };
    fetch(first_key(w), page_of(w), even);
    if constexpr (AHEAD == 2) fetch(first_key(w + NW), page_of(w + NW), odd);
    int32_t page = page_of(w + AHEAD * NW);
    auto turn = [&](int i, auto set) {
      const int jb = keys_at(i);
      // rows past the sequence's end may hold anything, rows before the window infinities: zeros
      if (jb + KS - 1 > p_last || (jb < jwin && jb + KS > kf)) {
#pragma unroll
        for (int x = 0; x < NS; ++x) {
          const int j = jb + piece_row(x);
          if (j > p_last || (j < jwin && j >= kf)) sreg[set][x] = (s16x8){0, 0, 0, 0, 0, 0, 0, 0};
        }
      }
#pragma unroll
      for (int x = 0; x < NS; ++x) *reinterpret_cast<s16x8*>(St + piece_row(x) * SR + piece_at(x)) = sreg[set][x];
      wave_lds_order();
      f32x4 sc[KT], sd[KT];
#pragma unroll
      for (int kt = 0; kt < KT; ++kt) {
        sc[kt] = sd[kt] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ks = 0; ks < DK; ++ks) {
          s16x8 kfr;
          if constexpr (SHARED) kfr = *reinterpret_cast<const s16x8*>(St + (kt * 16 + col) * SR + grp * 8 + ks * 32);
          else kfr = kreg[kt][ks];
          f32x4& acc = ks % 2 == 0 ? sc[kt] : sd[kt];      // two chains
#pragma unroll
          for (int n = 0; n < QP; ++n) {
            s16x8 q;
            if constexpr (QLDS) q = *reinterpret_cast<const s16x8*>(Qs + (16 * n + col) * QR + grp * 8 + ks * 32);
            else q = qr[ks][n];
            acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(kfr), as_bf16x8(q), acc, 0, 0, 0);
          }
        }
      }
      fetch(first_key(i + AHEAD * NW), page, set);           // in flight during the rest of this turn
      page = page_of(i + (AHEAD + 1) * NW);
#pragma unroll
      for (int kt = 0; kt < KT; ++kt) sc[kt] = (sc[kt] + sd[kt]) * a.scale;
      if (a.softcap > 0.f) {
        // wide groups: c tanh(s / c) = c - 2 c / (exp(2 s / c) + 1), off by some 2^-23 of c
        const float two_c = 2.f * a.softcap, inv1 = 1.f / a.softcap, inv = 2.f * inv1;
#pragma unroll
        for (int kt = 0; kt < KT; ++kt)
#pragma unroll
          for (int e = 0; e < 4; ++e)
            sc[kt][e] = EXACT ? a.softcap * tanh_of(sc[kt][e] * inv1)
                              : a.softcap - two_c * __builtin_amdgcn_rcpf(__expf(sc[kt][e] * inv) + 1.f);
      }
      float pv[4 * KT];
      float mx = kNegInfS;
#pragma unroll
      for (int kt = 0; kt < KT; ++kt)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int j = jb + kt * 16 + grp * 4 + e;
          const bool ok = live && j <= pi && (a.window <= 0 || pi - j < a.window || j < a.keep_first);
          if (a.sigmoid) {
            pv[kt * 4 + e] = ok ? 1.0f / (1.0f + exp_of<EXACT>(-(sc[kt][e] + hb))) : 0.f;
          } else {
            sc[kt][e] = ok ? sc[kt][e] : kNegInfS;
            mx = fmaxf(mx, sc[kt][e]);
          }
        }
      float alpha = 1.f;
      if (!a.sigmoid) {
        mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
        mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
        const float mn = mx > mrun + kDefer ? mx : mrun;   // also true for the first keys: mrun = -inf
        float sum = 0.f;
#pragma unroll
        for (int kt = 0; kt < KT; ++kt)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float p = sc[kt][e] == kNegInfS ? 0.f : exp_of<EXACT>(sc[kt][e] - mn);
            pv[kt * 4 + e] = p;
            sum += p;
          }
        sum += __shfl_xor(sum, 16, 64);
        sum += __shfl_xor(sum, 32, 64);
        alpha = mrun == kNegInfS ? 0.f : exp_of<EXACT>(mrun - mn);
        lrun = lrun * alpha + sum;
        mrun = mn;
      }
      if (__builtin_amdgcn_ballot_w64(alpha != 1.f) != 0ull) {
#pragma unroll
        for (int m = 0; m < DV; ++m) o[m] *= alpha;
      }
      const short* v0 = St + (4 * grp + (col >> 2)) * SR + 4 * (col & 3);
      if constexpr (KT == 2) {
        s16x8 pp[PP];
        split_parts<false>(pv, pp);
#pragma unroll
        for (int m = 0; m < DV; m += MG) {                 // a value block's products MG - 1 others apart
          s16x8 v[MG];
#pragma unroll
          for (int u = 0; u < MG; ++u) {
            const s16x4 a0 = rfq::ds_read_tr16(v0 + 16 * (m + u));
            const s16x4 a1 = rfq::ds_read_tr16(v0 + 16 * SR + 16 * (m + u));
            v[u] = (s16x8){a0[0], a0[1], a0[2], a0[3], a1[0], a1[1], a1[2], a1[3]};
          }
#pragma unroll
          for (int n = 0; n < PP; ++n)
#pragma unroll
            for (int u = 0; u < MG; ++u)
              o[m + u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(v[u]), as_bf16x8(pp[n]), o[m + u], 0, 0, 0);
        }
      } else {
        s16x4 pp[PP];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          float r = pv[e];
#pragma unroll
          for (int n = 0; n < PP; ++n) {
            pp[n][e] = (short)rfq::f2bf(r);
            r -= rfq::bf2f_s(pp[n][e]);
          }
        }
#pragma unroll
        for (int m = 0; m < DV; m += MG) {
          s16x4 v[MG];
#pragma unroll
          for (int u = 0; u < MG; ++u) v[u] = rfq::ds_read_tr16(v0 + 16 * (m + u));
#pragma unroll
          for (int n = 0; n < PP; ++n)
#pragma unroll
            for (int u = 0; u < MG; ++u)
              o[m + u] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(v[u], pp[n], o[m + u], 0, 0, 0);
        }
      }
      wave_lds_order();                                    // the next turn's rows, or the partial results, take their place
    };
    if constexpr (AHEAD == 2) {
      int i = w;
      for (; i + NW < n_turns; i += 2 * NW) {
        turn(i, even);
        turn(i + NW, odd);
      }
      if (i < n_turns) turn(i, even);
    } else {
      for (int i = w; i < n_turns; i += NW) turn(i, even);
    }
    // ---- the waves' parts meet: [16 columns][VP] each, beside their maxima and sums
#pragma unroll
    for (int mp = 0; mp < MP; ++mp) {
      if (mp > 0) __syncthreads();
#pragma unroll
      for (int m = 0; m < DV / MP; ++m)
        *reinterpret_cast<f32x4*>(part + col * (VP + 4) + 16 * m + 4 * grp) = o[mp * (DV / MP) + m];
      if (grp == 0) {
        // scores that are no numbers leave the maximum at -inf, which marks a wave without visible keys
        ml[w * 16 + col] = lrun != 0.f && mrun == kNegInfS ? 0.f : mrun;
        ml[(NW + w) * 16 + col] = lrun;
      }
      __syncthreads();
      for (int x = tid; x < 16 * (VP / 4); x += 64 * NW) {
        const int cc = x / (VP / 4), dp = (x - cc * (VP / 4)) * 4, dv = mp * VP + dp, cx = ct * 16 + cc;
        if (cx >= ql * rep) break;
        const int r = cx / rep, hx = g * rep + cx - r * rep;
        const int64_t t = t_first + r;
        float mul = a.out_mult, top = kNegInfS;
        if (!a.sigmoid) {
          const bool sink = a.head_bias != nullptr;
          const float hs = sink ? a.head_bias[hx] : kNegInfS;
          top = hs;
#pragma unroll
          for (int u = 0; u < NW; ++u) top = fmaxf(top, ml[u * 16 + cc]);
          float l = sink ? exp_of<EXACT>(hs - top) : 0.f;
#pragma unroll
          for (int u = 0; u < NW; ++u) {
            const float mu = ml[u * 16 + cc];
            l += mu == kNegInfS ? 0.f : ml[(NW + u) * 16 + cc] * exp_of<EXACT>(mu - top);
          }
          mul = l > 0.f ? a.out_mult / l : 0.f;
        }
        float y[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int u = 0; u < NW; ++u) {
          const float mu = ml[u * 16 + cc];
          if (!a.sigmoid && mu == kNegInfS) continue;        // a wave without visible keys
          const float f = a.sigmoid ? 1.f : exp_of<EXACT>(mu - top);
          const float4 p = *reinterpret_cast<const float4*>(
              smem + (size_t)u * WL + (size_t)(cc * (VP + 4) + dp) * 4);
          y[0] += f * p.x; y[1] += f * p.y; y[2] += f * p.z; y[3] += f * p.w;
        }
        if (a.gate != nullptr && a.gate_w == 1) mul /= 1.0f + exp_of<EXACT>(-ldf(a.gate + t * a.gate_stride + hx));
        bf16_t b[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          float v = y[e] * mul;
          if (a.gate != nullptr && a.gate_w > 1)
            v /= 1.0f + exp_of<EXACT>(-ldf(a.gate + t * a.gate_stride + (int64_t)hx * vdim + dv + e));
          stf(&b[e], v);
        }
        *reinterpret_cast<uint2*>(a.out + t * a.out_stride + (int64_t)hx * vdim + dv) =
            make_uint2((uint32_t)b[0] | ((uint32_t)b[1] << 16), (uint32_t)b[2] | ((uint32_t)b[3] << 16));
      }
    }
    __syncthreads();                                       // the next column tile reuses the LDS
  }
}

// ------------------------------------------------------------------ launcher
template <int DK, int DV, bool SHARED, int NW, bool EXACT>
static void launch_split_one(const KeepSplitArgs& a, int NA, int z, hipStream_t s) {
  constexpr size_t lds = (size_t)NW * wave_lds<DK, DV, SHARED, NW, EXACT>() + 2 * NW * 16 * sizeof(float) +
                         (turns_ahead<DK, SHARED>() == 2 ? query_parts<DK, EXACT>() * 16 * (32 * DK + 8) * 2 : 0);
  static_assert(lds <= 160 * 1024, "LDS of a CU");
  static bool attr = false;
  if (!attr) {          // dynamic LDS above 64 KB has to be allowed per kernel, once
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&attn_keep_split_kernel<DK, DV, SHARED, NW, EXACT>),
                              hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
    attr = true;
  }
  hipLaunchKernelGGL((attn_keep_split_kernel<DK, DV, SHARED, NW, EXACT>), dim3(NA, a.G, z),
                     dim3(64 * NW), lds, s, a);
}

// Eight waves to a workgroup where sequences and heads alone leave CUs idle: a wave's chain of pages is the
// time then.  The wide latent's staged page leaves room for four, one workgroup to a CU; once there are more
// workgroups than CUs the prompts' kernel takes its rows, which reads a page once for all heads, not for every
// 16 of them (64 heads of 576: 128 sequences of 600 tokens 78 us split, 54 there; 64 of them 40 and 53; where rows may
// see more than 13 to 20 pages, steps of no more rows than sequences have gone to keep_streams' workgroups before).  Many
// workgroups of large groups in plain sizes: two waves, or one, whose partial results need no merge (512 sequences of
// 100 tokens, 32 heads over 2 of 128: 23 us with four waves, 20 with one; of 1,000: 100 and 99).
// Column tiles side by side: as many as the sequences have on the average, more where CUs would idle (one
// sequence of 600 tokens with 33 rows, 64 heads: 1,130 us with four side by side, 38 with all).
template <int DK, int DV, bool SHARED, bool EXACT>
static void launch_split_waves(const KeepSplitArgs& a, int T, int NA, int tiles, hipStream_t s) {
  const int64_t work = (int64_t)a.G * (((int64_t)T * (a.H / a.G) + 15) / 16), wgs = (int64_t)NA * a.G;
  const int z = (int)std::min<int64_t>(std::min(tiles, 65535), std::max((work + wgs - 1) / wgs, 256 / wgs));
  if constexpr (SHARED && DK >= 10) {
    if constexpr (!EXACT) {
      if (work > 256)
        return launch_attn_keep_wide_rows(a.q, a.k_cache, a.vrs, a.bt, a.maxb, a.q_start, a.q_len, a.kv_len, T, NA,
                                          a.head_bias, a.gate, a.gate_stride, a.gate_w, a.out, a.out_stride, a.scale,
                                          a.window, a.keep_first, a.sigmoid != 0, a.H, a.G, 32 * DK, a.softcap,
                                          a.out_mult, s);
    }
  } else {
    if (wgs < 256) return launch_split_one<DK, DV, SHARED, 8, EXACT>(a, NA, z, s);
    if constexpr (!EXACT) {
      if (work >= 1024) return launch_split_one<DK, DV, SHARED, 1, EXACT>(a, NA, z, s);
      if (work >= 512) return launch_split_one<DK, DV, SHARED, 2, EXACT>(a, NA, z, s);
    }
  }
  launch_split_one<DK, DV, SHARED, 4, EXACT>(a, NA, z, s);
}

// The sizes are those of keep_mfma_ok, which the caller has asked.
void launch_attn_keep_split(const float* q, const void* k_cache, const void* v_cache, int64_t vrs, const int32_t* bt,
                            int maxb, const int32_t* q_start, const int32_t* q_len, const int32_t* kv_len, int T,
                            int NA, int short_rows, const float* head_bias, const void* gate, int64_t gate_stride, int gate_w,
                            void* out, int64_t out_stride, float scale, int window, int keep_first, bool sigmoid,
                            int H, int G, int E, int vdim, bool shared, float softcap, float out_mult, hipStream_t s) {
  if (NA == 0 || T == 0) return;
  const KeepSplitArgs a{q, (const bf16_t*)k_cache, (const bf16_t*)v_cache, vrs, bt, maxb, q_start, q_len, kv_len,
                        head_bias, (const bf16_t*)gate, gate_stride, gate_w, (bf16_t*)out, out_stride,
                        scale, softcap, out_mult, window, keep_first, (int)sigmoid, H, G};
  if (keep_row_ok(T, NA, H, G, E, vdim, shared)) return launch_attn_keep_row(a, T, NA, E, s);
  const int DK = E / 32, DV = vdim / 16;
  const bool exact = H / G < 16;
  const int tiles = (int)(((int64_t)std::min(short_rows, T) * (H / G) + 15) / 16);   // at most, of a sequence
#define SPLIT_GO(dk, dv, sh)                                                         \
  return exact ? launch_split_waves<dk, dv, sh, true>(a, T, NA, tiles, s)          \
               : launch_split_waves<dk, dv, sh, false>(a, T, NA, tiles, s)
  if (shared) {
    if (DK == 3) SPLIT_GO(3, 4, true);
    if (DK == 4 && DV == 4) SPLIT_GO(4, 4, true);
    if (DK == 4) SPLIT_GO(4, 6, true);
    if (DK == 5) SPLIT_GO(5, 8, true);
    if (DK == 6) SPLIT_GO(6, 8, true);
    if (DK == 10) SPLIT_GO(10, 16, true);
    SPLIT_GO(18, 32, true);
  }
#define SPLIT_DV(dk)                       \
  do {                                     \
    if (DV == 2) SPLIT_GO(dk, 2, false);   \
    if (DV == 4) SPLIT_GO(dk, 4, false);   \
    SPLIT_GO(dk, 8, false);                \
  } while (0)
  if (DK == 1) SPLIT_DV(1);
  if (DK == 2) SPLIT_DV(2);
  if (DK == 3) SPLIT_DV(3);
  SPLIT_DV(4);
#undef SPLIT_DV
#undef SPLIT_GO
}

}  // namespace rfqmix
