// attn_keep_window for decode rows of groups of up to eight heads (bf16 pages of 32 tokens, keys and values of 64 or
// 128 entries in pages of their own; semantics of mix_keep_attn.hip): a workgroup per (row, key/value head), every
// wave takes every NW-th page, as in mix_keep_split.hip, whose sixteen MFMA columns a group of four would leave to
// three quarters empty.
//
// Where there are no more rows than sequences, a sequence may still have several: in a captured step rows of an extend
// stand where other sequences are padding.  So a row has workgroups of its own, and neighbouring rows share one only where
// its columns hold the heads of both.  32 heads over 8 of 128, as many rows as sequences, one after another in a sequence's
// workgroup and now: 12 rows of a sequence of 600 tokens and four sequences of one in a step of 16, 128 -> 14.2 us (29 by
// mix_keep_split.hip); twice eight rows of 1,900 tokens 183 -> 24 (31); 32 rows of 1,500 tokens and 32 sequences of 300
// 650 -> 27 (304).  Sixteen rows of as many sequences take 14.5 either way.
//
// Here the columns are (part, head): a head's query is the exact sum of three bf16 (all of fp32's bits), and its parts
// are columns of one product instead of three products of one column.  Up to four heads fit with all parts, up to
// eight with the first two, the third part in a product of its own.  The sums over parts are scores, of which every
// lane of a head's four (two) takes a quarter (a half): cap, mask and weight are made once for a key and head, not
// for sixteen columns.  The weights' three parts go back into columns through LDS, and the weighted values' parts are
// added up once, behind the last page.
//   S^T[key, (part, head)] = K . Q^T      O^T[channel, (part, head)] = V^T . P^T
//
// What bounds it: the pages' bytes once they are many, before that a wave's chain of pages.  With all products and
// functions of sixteen columns, 48 products and some 450 vector instructions a page, 64 sequences of 300 - 900 tokens (32
// heads over 8 of 128, softcap) took 29 us without any page but the first; so 20 us.  A wave stages a page in LDS at once,
// and the next one is in flight during all of its work.  Rows of pages come in 1 KB pieces of neighbouring rows: read as
// the product wants keys, 32 bytes of 16 rows to an access, 160 MB of pages took 36 us with nothing else to do, and 28 - 30
// so.  Two pages ahead spill.
// Measured with pages that no cache holds: these 64 sequences (160 MB) 44 -> 31 us (5.2 TB/s), one sequence of 611 tokens,
// eight workgroups, 13.6 -> 11.8 us; whole passes: groups of eight heads 63.7 -> 48.3, a window with sigmoid weights 45.8 ->
// 35.9, eight sequences of up to 1,900 35.4 -> 29.1.
#include <algorithm>
#include <type_traits>

#include "common.h"
#include "mix_common.h"
#include "mix_keep_split.h"
#include "mix_split.h"

namespace rfqmix {

namespace {
// the lane 4 away in the other half of eight
__device__ __forceinline__ float lane_xor4(float v) {
  const int up = __builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x104, 0xf, 0x5, false);       // 4 lanes on: banks 0, 2
  return __int_as_float(__builtin_amdgcn_update_dpp(up, __float_as_int(v), 0x114, 0xf, 0xa, false));   // 4 lanes back
}
__device__ __forceinline__ float lane_ror(float v, std::integral_constant<int, 4>) {
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x124, 0xf, 0xf, true));
}
__device__ __forceinline__ float lane_ror(float v, std::integral_constant<int, 8>) {
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x128, 0xf, 0xf, true));
}
constexpr std::integral_constant<int, 4> k4{};
constexpr std::integral_constant<int, 8> k8{};

// over the lanes that hold the keys of a head
template <int HC, typename F>
__device__ __forceinline__ float head_all(float v, F f) {
  if constexpr (HC == 4) v = f(v, lane_ror(v, k4));
  v = f(v, lane_ror(v, k8));
  auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = f(__uint_as_float(r[0]), __uint_as_float(r[1]));
  r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return f(__uint_as_float(r[0]), __uint_as_float(r[1]));
}

template <bool STREAM>
__device__ __forceinline__ s16x8 rows16(const bf16_t* p) {
  if constexpr (STREAM) return __builtin_nontemporal_load(reinterpret_cast<const s16x8*>(p));
  else return *reinterpret_cast<const s16x8*>(p);
}

// shorts: a wave's staged values, keys and weights; its partial results take the values' place
template <int DK, int DV, int HC>
struct RowLds {
  static constexpr int VR = 16 * DV + 8, KR = 32 * DK + 8;
  static constexpr int K = PG * VR, P = K + PG * KR, ALL = P + 4 * HC * 32;
};
}  // namespace

// E = 32 DK, vdim = 16 DV, HC heads to a tile of columns, NW waves; STREAM: pages past the caches.  rep: heads a group;
// side4: rows whose heads the columns hold, one of more than four.
template <int DK, int DV, int HC, int NW, bool STREAM>
__global__ __launch_bounds__(64 * NW, 2) void attn_keep_row_kernel(const KeepSplitArgs a, int NA, int rep, int side4) {
  constexpr int E = 32 * DK, vdim = 16 * DV, NL = 16 / HC, QP = HC == 4 ? 1 : 2, NE = 8 / NL;
  typedef RowLds<DK, DV, HC> L;
  typedef const __attribute__((address_space(4))) int32_t const_i32;
  const int side = HC == 4 ? side4 : 1;
  // a row's heads lie side by side, as their pages do
  const int64_t t = blockIdx.x / a.G;
  const int g = blockIdx.x - (int)t * a.G;
  const int tid = threadIdx.x, lane = tid & 63, col = lane & 15, grp = lane >> 4;
  // most steps have a row a sequence: then row t is sequence t's, whose numbers are on their way at once
  int s = min((int)t, NA - 1);
  auto of = [&](const int32_t* x) { return ((const_i32*)(uintptr_t)x)[s]; };
  int from = of(a.q_start), ql = of(a.q_len), kvl = of(a.kv_len);
  asm volatile("" : "+s"(from), "+s"(ql), "+s"(kvl));      // all three before the branch, not one after another
  if (__builtin_expect((from > t) | (from + ql <= t), 0)) {
    s = -1;
    for (int b = 0; b < NA && s < 0; b += 64) {
      const int x = b + lane, xf = x < NA ? a.q_start[x] : 0, xn = x < NA ? a.q_len[x] : 0;
      const uint64_t m = __builtin_amdgcn_ballot_w64(xf <= t && t < xf + xn);
      if (m != 0) s = b + __builtin_ctzll(m);
    }
    if (s < 0) return;                                     // a row of a captured step beyond those of its sequences
    from = of(a.q_start);
    ql = of(a.q_len);
    kvl = of(a.kv_len);
  }
  const_i32* bt = (const_i32*)(uintptr_t)(a.bt + (int64_t)s * a.maxb);
  const int r0 = (int)t - from;
  if (r0 > 0 && r0 % side != 0) return;                    // with the row above
  const int rows = min(side, ql - r0), all = rows * rep;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int hc = col & (HC - 1), part = col / HC;
  const bool odd = HC == 4 ? (part & 1) != 0 : part != 0, high = part >= 2;     // which keys of a page the lane takes

  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  short* const Vt = reinterpret_cast<short*>(smem) + w * L::ALL;
  short* const Kt = Vt + L::K;
  short* const Pt = Vt + L::P;                             // [4 parts, the last zeros][HC][4 grp][8 keys]
  float* const ml = reinterpret_cast<float*>(smem + (size_t)NW * L::ALL * 2);   // [NW][HC] maxima, [NW][HC] sums

  for (int x = lane; x < HC * 16; x += 64) *reinterpret_cast<uint32_t*>(Pt + 3 * HC * 32 + 2 * x) = 0;
  const bool live = hc < all;
  const int row = live && side > 1 ? hc / rep : 0, hh = g * rep + (live ? hc - row * rep : 0);     // this lane's (row, head)
  const int p_first = kvl - ql + r0, p_last = p_first + rows - 1, pi = p_first + row;
  const int jwin = a.window > 0 ? max(0, p_first - a.window + 1) : 0;
  const int kf = a.window > 0 ? min(a.keep_first, jwin) : 0;
  // pages [0, n_keep) hold the kept first tokens, [k_win, k_last] the window
  const int k_last = p_last / PG, k_win = jwin / PG;
  const int n_keep = min((kf + PG - 1) / PG, k_win);
  const int n_turns = n_keep + k_last - k_win + 1;
  auto page_at = [&](int i) { return i < n_keep ? i : k_win + i - n_keep; };
  auto number = [&](int i) { return bt[page_at(min(i, n_turns - 1))]; };

  // 16-byte pieces of a page per lane: 1 KB of neighbouring rows to a load
  constexpr int NV = PG * vdim / 512, NK = PG * E / 512, VP = vdim / 8, KP = E / 8;
  static_assert(64 % VP == 0 && 64 % KP == 0);
  s16x8 vreg[NV], kreg[NK];
  auto fetch = [&](int32_t page) {
    const int64_t at = ((int64_t)page * a.G + g) * PG;   // the first key's slot
    const bf16_t* kp = a.k_cache + at * E + lane * 8;
    const bf16_t* vp = a.v_cache + at * a.vrs + (lane / VP) * a.vrs + lane % VP * 8;
#pragma unroll
    for (int i = 0; i < NK; ++i) kreg[i] = rows16<STREAM>(kp + i * 512);
#pragma unroll
    for (int i = 0; i < NV; ++i) vreg[i] = rows16<STREAM>(vp + i * (64 / VP) * a.vrs);
  };
  float4 qf[DK][2];
  {
    const float* qp = a.q + ((t + row) * a.H + hh) * E + grp * 8;
#pragma unroll
    for (int ks = 0; ks < DK; ++ks) {
      qf[ks][0] = ld4(qp + ks * 32);
      qf[ks][1] = ld4(qp + ks * 32 + 4);
    }
  }
  const float hb = a.head_bias != nullptr ? a.head_bias[hh] : 0.f;
  int32_t page = number(w);
  fetch(page);                                           // on its way before the queries are waited for
  page = number(w + NW);
  __builtin_amdgcn_sched_barrier(0);
  s16x8 q[DK][QP];
#pragma unroll
  for (int ks = 0; ks < DK; ++ks) {
    const float4 x = qf[ks][0], y = qf[ks][1];
    const float f[8] = {x.x, x.y, x.z, x.w, y.x, y.y, y.z, y.w};
    s16x8 p[3];
    split_parts<true>(f, p);
    const s16x8 zero = {0, 0, 0, 0, 0, 0, 0, 0};
    if constexpr (HC == 4) {
      q[ks][0] = part == 0 ? p[0] : part == 1 ? p[1] : part == 2 ? p[2] : zero;
    } else {
      q[ks][0] = part == 0 ? p[0] : p[1];
      q[ks][QP - 1] = part == 0 ? p[2] : zero;
    }
  }
  f32x4 o[DV];
#pragma unroll
  for (int m = 0; m < DV; ++m) o[m] = (f32x4){0.f, 0.f, 0.f, 0.f};
  float mrun = kNegInfS, lrun = 0.f;                     // of the head; of this lane's keys

  for (int i = w; i < n_turns; i += NW) {
    const int jb = page_at(i) * PG;
    // rows past the sequence's end may hold anything, rows before the window infinities: zeros
    if (jb + PG - 1 > p_last || (jb < jwin && jb + PG > kf)) {
#pragma unroll
      for (int x = 0; x < NV; ++x) {
        const int j = jb + x * (64 / VP) + lane / VP;
        if (j > p_last || (j < jwin && j >= kf)) vreg[x] = (s16x8){0, 0, 0, 0, 0, 0, 0, 0};
      }
    }
#pragma unroll
    for (int x = 0; x < NK; ++x) *reinterpret_cast<s16x8*>(Kt + (x * (64 / KP) + lane / KP) * L::KR + lane % KP * 8) = kreg[x];
#pragma unroll
    for (int x = 0; x < NV; ++x) *reinterpret_cast<s16x8*>(Vt + (x * (64 / VP) + lane / VP) * L::VR + lane % VP * 8) = vreg[x];
    __builtin_amdgcn_sched_barrier(0);
    if (i + NW < n_turns) {                              // the registers are free: in flight during all of this turn
      fetch(page);
      page = number(i + 2 * NW);
    }
    wave_lds_order();
    f32x4 sc[2];
#pragma unroll
    for (int kt = 0; kt < 2; ++kt) sc[kt] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ks = 0; ks < DK; ++ks)
#pragma unroll
      for (int kt = 0; kt < 2; ++kt) {
        const s16x8 k = *reinterpret_cast<const s16x8*>(Kt + (kt * 16 + col) * L::KR + grp * 8 + ks * 32);
#pragma unroll
        for (int n = 0; n < QP; ++n)
          sc[kt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(k), as_bf16x8(q[ks][n]), sc[kt], 0, 0, 0);
      }
    __builtin_amdgcn_sched_barrier(0);
    // the parts' sums: a lane keeps one tile's keys, and of four lanes a half of them
    float x[NE];
    {
      float y[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float give = odd ? sc[0][e] : sc[1][e], keep = odd ? sc[1][e] : sc[0][e];
        y[e] = keep + (HC == 4 ? lane_xor4(give) : lane_ror(give, k8));
      }
      if constexpr (HC == 4) {
#pragma unroll
        for (int e = 0; e < 2; ++e) {
          const float give = high ? y[e] : y[2 + e], keep = high ? y[2 + e] : y[e];
          x[e] = keep + lane_ror(give, k8);
        }
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) x[e] = y[e];
      }
    }
    const int j0 = jb + (odd ? 16 : 0) + 4 * grp + (HC == 4 && high ? 2 : 0);     // key of x[0]
    float mx = kNegInfS;
#pragma unroll
    for (int e = 0; e < NE; ++e) {
      x[e] *= a.scale;
      if (a.softcap > 0.f) x[e] = a.softcap * tanh_of(x[e] * (1.f / a.softcap));
      const int j = j0 + e;
      const bool ok = live && j <= pi && (a.window <= 0 || pi - j < a.window || j < a.keep_first);
      if (a.sigmoid) {
        x[e] = ok ? sigmoid_c(x[e] + hb) : 0.f;
      } else {
        x[e] = ok ? x[e] : kNegInfS;
        mx = fmaxf(mx, x[e]);
      }
    }
    if (!a.sigmoid) {
      mx = head_all<HC>(mx, [](float p, float r) { return fmaxf(p, r); });
      const float mn = mx > mrun + kDefer ? mx : mrun;   // also true for the first keys: mrun = -inf
      const float alpha = mrun == kNegInfS ? 0.f : exp_c(mrun - mn);
      if (__builtin_amdgcn_ballot_w64(alpha != 1.f) != 0ull) {
        lrun *= alpha;
#pragma unroll
        for (int m = 0; m < DV; ++m) o[m] *= alpha;
      }
      mrun = mn;
#pragma unroll
      for (int e = 0; e < NE; ++e) {
        x[e] = x[e] == kNegInfS ? 0.f : exp_c(x[e] - mn);
        lrun += x[e];
      }
    }
    // the weights' parts into their columns: keys 16 kt + 4 grp + e of a head side by side
    short* const put = Pt + hc * 32 + grp * 8 + (odd ? 4 : 0) + (HC == 4 && high ? 2 : 0);
    const Split2 p0 = split3(x[0], x[1]);
    if constexpr (HC == 4) {
      *reinterpret_cast<uint32_t*>(put) = p0.h;
      *reinterpret_cast<uint32_t*>(put + HC * 32) = p0.m;
      *reinterpret_cast<uint32_t*>(put + 2 * HC * 32) = p0.l;
    } else {
      const Split2 p1 = split3(x[NE - 2], x[NE - 1]);
      *reinterpret_cast<uint2*>(put) = make_uint2(p0.h, p1.h);
      *reinterpret_cast<uint2*>(put + HC * 32) = make_uint2(p0.m, p1.m);
      *reinterpret_cast<uint2*>(put + 2 * HC * 32) = make_uint2(p0.l, p1.l);
    }
    wave_lds_order();
    s16x8 p[QP];
    p[0] = *reinterpret_cast<const s16x8*>(Pt + part * HC * 32 + hc * 32 + grp * 8);
    if constexpr (HC == 8) p[QP - 1] = *reinterpret_cast<const s16x8*>(Pt + (part + 2) * HC * 32 + hc * 32 + grp * 8);
    const short* v0 = Vt + (4 * grp + (col >> 2)) * L::VR + 4 * (col & 3);
#pragma unroll
    for (int m = 0; m < DV; ++m) {
      const s16x4 a0 = rfq::ds_read_tr16(v0 + 16 * m), a1 = rfq::ds_read_tr16(v0 + 16 * L::VR + 16 * m);
      const s16x8 v = {a0[0], a0[1], a0[2], a0[3], a1[0], a1[1], a1[2], a1[3]};
#pragma unroll
      for (int n = 0; n < QP; ++n)
        o[m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(v), as_bf16x8(p[n]), o[m], 0, 0, 0);
      if (m % 4 == 3) __builtin_amdgcn_sched_barrier(0);   // not all of a page's operands at once: registers
    }
    wave_lds_order();                                    // the next turn's rows, or the partial results, take their place
  }
  // ---- the parts of a column, then the waves' results meet: [HC][vdim] each, beside their maxima and sums
  lrun = head_all<HC>(lrun, [](float p, float r) { return p + r; });
  float* const res = reinterpret_cast<float*>(Vt);       // [HC][vdim + 4]
#pragma unroll
  for (int m = 0; m < DV; ++m) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      if constexpr (HC == 4) o[m][e] += lane_ror(o[m][e], k4);
      o[m][e] += lane_ror(o[m][e], k8);
    }
    if (part == 0) *reinterpret_cast<f32x4*>(res + hc * (vdim + 4) + 16 * m + 4 * grp) = o[m];
  }
  if (part == 0 && grp == 0) {
    // scores that are no numbers leave the maximum at -inf, which marks a wave without visible keys
    ml[w * HC + hc] = lrun != 0.f && mrun == kNegInfS ? 0.f : mrun;
    ml[(NW + w) * HC + hc] = lrun;
  }
  __syncthreads();
  for (int y = tid; y < HC * (vdim / 4); y += 64 * NW) {
    const int cc = y / (vdim / 4), dv = (y - cc * (vdim / 4)) * 4;
    if (cc >= all) break;
    const int r = cc / rep, hx = g * rep + cc - r * rep;
    float mul = a.out_mult, top = kNegInfS;
    if (!a.sigmoid) {
      const bool sink = a.head_bias != nullptr;
      const float hs = sink ? a.head_bias[hx] : kNegInfS;
      top = hs;
#pragma unroll
      for (int u = 0; u < NW; ++u) top = fmaxf(top, ml[u * HC + cc]);
      float l = sink ? exp_c(hs - top) : 0.f;
#pragma unroll
      for (int u = 0; u < NW; ++u) {
        const float mu = ml[u * HC + cc];
        l += mu == kNegInfS ? 0.f : ml[(NW + u) * HC + cc] * exp_c(mu - top);
      }
      mul = l > 0.f ? a.out_mult / l : 0.f;
    }
    float v[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int u = 0; u < NW; ++u) {
      const float mu = ml[u * HC + cc];
      if (!a.sigmoid && mu == kNegInfS) continue;        // a wave without visible keys
      const float f = a.sigmoid ? 1.f : exp_c(mu - top);
      const float4 p = ld4(reinterpret_cast<const float*>(reinterpret_cast<const short*>(smem) + u * L::ALL) + cc * (vdim + 4) + dv);
      v[0] += f * p.x; v[1] += f * p.y; v[2] += f * p.z; v[3] += f * p.w;
    }
    if (a.gate != nullptr && a.gate_w == 1) mul *= sigmoid_c(ldf(a.gate + (t + r) * a.gate_stride + hx));
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      v[e] *= mul;
      if (a.gate != nullptr && a.gate_w > 1)
        v[e] *= sigmoid_c(ldf(a.gate + (t + r) * a.gate_stride + (int64_t)hx * vdim + dv + e));
    }
    *reinterpret_cast<uint2*>(a.out + (t + r) * a.out_stride + (int64_t)hx * vdim + dv) =
        make_uint2(rfq::pack_bf16x2(v[0], v[1]), rfq::pack_bf16x2(v[2], v[3]));
  }
}

// ------------------------------------------------------------------ launcher
bool keep_row_ok(int T, int NA, int H, int G, int E, int vdim, bool shared) {
  return !shared && T <= NA && H / G <= 8 && ((E == 64 && vdim == 64) || (E == 128 && vdim == 128));
}

template <int DK, int DV, int HC, int NW, bool STREAM>
static void launch_row_one(const KeepSplitArgs& a, int T, int NA, hipStream_t s) {
  constexpr size_t lds = (size_t)NW * RowLds<DK, DV, HC>::ALL * 2 + 2 * NW * HC * sizeof(float);
  static_assert(lds <= 160 * 1024, "LDS of a CU");
  static bool attr = false;
  if (!attr) {          // dynamic LDS above 64 KB has to be allowed per kernel, once
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&attn_keep_row_kernel<DK, DV, HC, NW, STREAM>),
                              hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
    attr = true;
  }
  hipLaunchKernelGGL((attn_keep_row_kernel<DK, DV, HC, NW, STREAM>), dim3((unsigned)T * a.G), dim3(64 * NW), lds, s, a, NA,
                     a.H / a.G, std::max(HC / (a.H / a.G), 1));
}
// Eight waves to a workgroup where rows and heads alone leave CUs idle: a wave's chain of pages is the time then.
// Pages past the caches where what the tables have room for is more than 96 MB: the last-level cache, 256 MB, then holds
// nothing of them by the time they are read again.  32 heads over 8 of 128, 300 - 900 tokens, through the caches and past
// them: 8 sequences (of up to 1,900) 29.2 / 32.0 us, 24 24.7 / 25.7, 32 29.3 / 28.3, 48 42.2 / 37.2, 64 50.0 / 42.1.  A
// captured step's tables are as wide as the longest context, whatever its sequences hold.  600 tokens each, pages that no
// cache holds: 4 sequences 11.9 / 13.3 us, 8 14.1 / 13.7, 16 15.2 / 14.3, 64 29.9 / 30.0; with the first 13 pages in common
// 11.7 / 13.0, 12.1 / 13.1, 13.5 / 13.3, 20.6 / 20.0.  Few long ones gain: 4 of 2,000 tokens 28.1 / 27.5, 15 of 2,000 32.5 /
// 30.5, one of 32,000 290 / 282.
template <int DK, int DV, int HC>
static void launch_row_waves(const KeepSplitArgs& a, int T, int NA, hipStream_t s) {
  const int64_t wgs = (int64_t)T * a.G;
  const bool stream = wgs * a.maxb * (PG * (32 * DK + 16 * DV) * 2) > (96 << 20);
  if (wgs < 256) {
    if (stream) launch_row_one<DK, DV, HC, 8, true>(a, T, NA, s);
    else launch_row_one<DK, DV, HC, 8, false>(a, T, NA, s);
  } else {
    if (stream) launch_row_one<DK, DV, HC, 4, true>(a, T, NA, s);
    else launch_row_one<DK, DV, HC, 4, false>(a, T, NA, s);
  }
}

void launch_attn_keep_row(const KeepSplitArgs& a, int T, int NA, int E, hipStream_t s) {
  const bool four = a.H / a.G <= 4;
  if (E == 64) {
    if (four) launch_row_waves<2, 4, 4>(a, T, NA, s);
    else launch_row_waves<2, 4, 8>(a, T, NA, s);
  } else {
    if (four) launch_row_waves<4, 8, 4>(a, T, NA, s);
    else launch_row_waves<4, 8, 8>(a, T, NA, s);
  }
}

}  // namespace rfqmix
