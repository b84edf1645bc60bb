// attn_keep_window, decode rows of 576-wide latents whose first 512 entries are the values (bf16 pages of 32 tokens), more
// than 16 heads a key head, few sequences: a row's pages are shared by up to S workgroups, whose results meet in
// attn_keep_streams_merge_kernel by way of `part` ([T, S, H] of 512 weighted values each, then as many pairs of maximum, in
// base 2, and sum; -inf: no key).  Semantics of mix_keep_attn.hip.
//
// A workgroup takes its pages one after another for 32 heads (64: HT), every page with all of its eight waves:
//   scores    S^T[key, head] = K . Q^T on 16 x 16 tiles: a wave has 16 keys, 16 heads and 320 or 256 of the entries, the
//             queries as bf16 in registers; the two parts meet in LDS
//   weights   every wave for its 16 heads, cap, mask, maximum and sum in fp32
//   values    O^T[channel, head] += V^T . P^T: a wave has 16 heads and 128 channels, the weights as bf16 hi + lo parts
// The scores of page k + 1 stand beside the values of page k, before them in the half of the waves and behind them in the
// others (1 - 3 % of the time), so that one barrier a page does.  Four pages lie in LDS: two in use, two on their way
// (LDS-DMA, counted waits).  Results stay where they are, a channel has one wave.
//
// What bounds it: for few rows the way to the first page (3.3 us for the step's numbers, a chain of three loads, 2.7 for
// queries and page), 1.25 us a page (its LDS accesses, of 200 KB) and 2 us for the results; for many the pages' bytes, the
// queries of every share and the shares' results.  With a page a pair of waves, four pages at a time and none on its way
// meanwhile, and a meeting of the four in LDS: 576 entries, 32 heads, attention and merge alone, one sequence of 2,000 tokens
// 25.8 -> 17.4 us, four of 4,000 28.5 -> 23.6, 16 of 2,000 32.8 -> 24.0, 64 of 600 30.6 -> 25.2, of 300 - 900 30.2 -> 27.4, of
// 2,000 46.2 -> 40; one of 600 under a wide table 19.0 -> 14.0.  64 heads, 16 of 2,000 31.8 -> 28, 64 of 300 - 900 37.1 -> 35.8.
// Changed nothing: page numbers read beside the row's own numbers.
#include <algorithm>

#include "mix_keep_mfma.h"

namespace rfqmix {

constexpr int kLatE = 576, kLatV = 512;
constexpr int kLatPage = WBS * kLatE * 2;        // bytes
constexpr int stream_pages(int tiles) { return tiles == 1 ? 4 : 3; }        // in LDS
constexpr int kSharePages = 2;                   // pages of a workgroup, at least
constexpr int kWholePages = 8;                   // rows of so many and fewer are a workgroup's, of two tiles of heads

// What a row of the step sees: pages [0, n_keep) of its sequence s (-1: none, a row of a captured step beyond those of
// its sequences) hold the kept first tokens, `skip` pages follow that are not read, then those of the window up to the
// row's own.
struct RowPages {
  int s, pi, jwin, kf, n_keep, skip, pages;                   // pi: query, jwin: window's first key, kf: kept keys before it
};
// Most steps have a row a sequence: then row t is sequence t's, whose numbers are on their way at once.
__device__ __forceinline__ RowPages row_pages(const KeepArgs& a, int NA, int t) {
  RowPages r;
  const int i = min(t, NA - 1);
  int from = a.q_start[i], n = a.q_len[i], kv = a.kv_len[i];
  r.s = i;
  if (from > t || from + n <= t) {
    r.s = -1;
    for (int b = 0; b < NA && r.s < 0; b += 64) {
      const int x = b + (threadIdx.x & 63), xf = x < NA ? a.q_start[x] : 0, xn = x < NA ? a.q_len[x] : 0;
      const uint64_t m = __builtin_amdgcn_ballot_w64(xf <= t && t < xf + xn);
      if (m != 0) r.s = b + __builtin_ctzll(m);
    }
    if (r.s < 0) return r;
    from = a.q_start[r.s];
    n = a.q_len[r.s];
    kv = a.kv_len[r.s];
  }
  r.pi = kv - n + t - from;
  r.jwin = a.window > 0 ? max(0, r.pi - a.window + 1) : 0;
  r.kf = a.window > 0 ? min(a.keep_first, r.jwin) : 0;
  const int pg_win = r.jwin / WBS;
  r.n_keep = min((r.kf + WBS - 1) / WBS, pg_win);
  r.skip = pg_win - r.n_keep;
  r.pages = r.pi / WBS + 1 - r.skip;
  return r;
}
// What a row's weighted values of head h are multiplied by, given the maximum and sum of all its keys: the sink's part
// of the sum, a gate per head.
template <int MODE>
__device__ __forceinline__ float whole(const KeepArgs& a, int64_t t, int h, float top, float sum) {
  float f = 1.f, l = sum;
  if constexpr (MODE < 2) {
    const float sink = a.head_bias != nullptr ? a.head_bias[h] * kLog2e : kNegInfW, m = fmaxf(top, sink);
    f = top == kNegInfW ? 0.f : __builtin_amdgcn_exp2f(top - m);
    l = (top == kNegInfW ? 0.f : f * sum) + (sink == kNegInfW ? 0.f : __builtin_amdgcn_exp2f(sink - m));
  }
  float mul = MODE >= 2 ? a.out_mult : (l > 0.f ? a.out_mult / l : 0.f);
  if (a.gate != nullptr && a.gate_w == 1)
    mul /= 1.0f + __expf(-ldf(static_cast<const bf16_t*>(a.gate) + t * a.gate_stride + h));
  return f * mul;
}
// Four neighbouring outputs of head h, through a gate per output
template <int vdim>
__device__ __forceinline__ void store_gated(const KeepArgs& a, float (&y)[4], int64_t t, int h, int dv) {
  if (a.gate != nullptr && a.gate_w > 1) {
    const float4 x = ld4(static_cast<const bf16_t*>(a.gate) + t * a.gate_stride + (int64_t)h * vdim + dv);
    y[0] /= 1.0f + __expf(-x.x);
    y[1] /= 1.0f + __expf(-x.y);
    y[2] /= 1.0f + __expf(-x.z);
    y[3] /= 1.0f + __expf(-x.w);
  }
  *reinterpret_cast<uint2*>(static_cast<bf16_t*>(a.out) + t * a.out_stride + (int64_t)h * vdim + dv) =
      make_uint2(rfq::pack_bf16x2(y[0], y[1]), rfq::pack_bf16x2(y[2], y[3]));
}
// How many of S workgroups have a part in the row: no more than have two pages, the first in any case
template <int HT>
__device__ __forceinline__ int row_shares(const RowPages& r, int S) {
  if (HT == 2 && r.pages <= kWholePages) return 1;
  return min(S, max(1, (r.pages + kSharePages - 1) / kSharePages));
}

// HT: tiles of 16 heads a wave, for groups of up to 32 HT heads a workgroup
template <int HT, int MODE>
__global__ __launch_bounds__(512, 2) void attn_keep_streams_kernel(const KeepArgs a, float* part, int T, int NA) {
  constexpr int E = kLatE, vdim = kLatV, KS = E / 32, K0 = 10, NP = kLatPage / 1024, NB = stream_pages(HT);
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int hf = w & 1, kt = (w >> 1) & 1, part_e = w >> 2, cq = w >> 1;   // heads, keys, entries; channels
  const int64_t t = blockIdx.x;
  const int S = gridDim.z, z = blockIdx.z;
  const int col = lane & 15, grp = lane >> 4;
  const int rep = a.H / a.G, per = (rep + 32 * HT - 1) / (32 * HT);
  const int g = (int)blockIdx.y / per, h0 = ((int)blockIdx.y - g * per) * (32 * HT) + hf * (16 * HT);
  const bool idle = h0 >= rep;                                // a wave that only copies pages
  int hh[HT];                                                 // past the last head: it once more, not stored
#pragma unroll
  for (int h = 0; h < HT; ++h) hh[h] = g * rep + min(h0 + h * 16 + col, rep - 1);
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const short* const pages_at = reinterpret_cast<const short*>(smem);
  float4* const meet = reinterpret_cast<float4*>(smem + NB * kLatPage);      // [2][HT][wave][lane] scores of part of the entries

  // the queries, shared by the waves: a wave packs every fourth piece of 32 entries of its heads.  They are asked for first.
  constexpr int NQ = (KS + 3) / 4;
  float4 qx[HT][NQ], qy[HT][NQ];
#pragma unroll
  for (int h = 0; h < HT; ++h) {
    const float* qp = a.q + (t * a.H + hh[h]) * E + grp * 8;
#pragma unroll
    for (int x = 0; x < NQ; ++x) {
      const int ks = min(x * 4 + cq, KS - 1);
      qx[h][x] = *reinterpret_cast<const float4*>(qp + ks * 32);
      qy[h][x] = *reinterpret_cast<const float4*>(qp + ks * 32 + 4);
    }
  }
  const RowPages row = row_pages(a, NA, (int)t);
  if (row.s < 0) return;
  const int shares = row_shares<HT>(row, S);
  if (z >= shares) return;                                    // no page for this workgroup
  const int from = z * row.pages / shares, n = (z + 1) * row.pages / shares - from;
  typedef const __attribute__((address_space(4))) int32_t const_i32;
  const_i32* bt = (const_i32*)(uintptr_t)(a.bt + (int64_t)row.s * a.maxb);
  auto block_of = [&](int k) { return from + k < row.n_keep ? from + k : from + k + row.skip; };
  auto number = [&](int k) { return bt[block_of(min(k, n - 1))]; };
  int32_t ahead[NB];
#pragma unroll
  for (int k = 0; k < NB; ++k) ahead[k] = number(k);

  const uint32_t lds0 = lds_byte(smem);
  uint32_t src[(NP + 7) / 8];                                 // bytes from a page's first, of this wave's pieces
#pragma unroll
  for (int x = 0; x < (NP + 7) / 8; ++x) {
    const int p = (w + 8 * x) * 64 + lane, rw = p / (E / 8), c = p - rw * (E / 8);
    src[x] = (uint32_t)(rw * E + ((c & ~7) | ((c & 7) ^ wide_swizzle(rw))) * 8) * 2;
  }
  auto copy = [&](int32_t page, int k) {
    const char* kb = static_cast<const char*>(a.k_cache) + ((int64_t)page * a.G + g) * kLatPage;
    const uint32_t to = lds0 + k % NB * kLatPage + w * 1024;
#pragma unroll
    for (int x = 0; x < NP / 8; ++x) lds_copy16(kb, src[x], to + x * 8192);
    if (w < NP % 8) lds_copy16(kb, src[NP / 8], to + NP / 8 * 8192);
  };
  // this wave's copies but those of the last `pages` ones have landed
  static_assert(NP / 8 == 4 && NP % 8 == 4, "the waits below count five or four copies a page");
  auto wait = [&](int pages) {
    if (pages <= 0) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    else if (pages == 1) {
      if (w < 4) asm volatile("s_waitcnt vmcnt(5)" ::: "memory");
      else asm volatile("s_waitcnt vmcnt(4)" ::: "memory");
    } else {
      if (w < 4) asm volatile("s_waitcnt vmcnt(10)" ::: "memory");
      else asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
    }
  };
  // everyone's LDS accesses before are done; copies may be on their way
  auto sync = [] {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };

  // where the last HT pages of the ring will be: [tile][piece] KB
  static_assert(2 * KS * 1024 == kLatPage, "");
  unsigned char* const qs = smem + (NB - HT) * kLatPage;
#pragma unroll
  for (int h = 0; h < HT; ++h)
#pragma unroll
    for (int x = 0; x < NQ; ++x) {
      const float4 u = qx[h][x], v = qy[h][x];
      const float f[8] = {u.x, u.y, u.z, u.w, v.x, v.y, v.z, v.w};
      *reinterpret_cast<s16x8*>(qs + ((hf * HT + h) * KS + min(x * 4 + cq, KS - 1)) * 1024 + lane * 16) = rfq::pack8(f);
    }
  asm volatile("" ::: "memory");                              // the queries are here: nothing but copies is on its way
#pragma unroll
  for (int k = 0; k < NB - HT; ++k)
    if (k < n) copy(ahead[k], k);
  sync();
  s16x8 q[HT][K0];
#pragma unroll
  for (int h = 0; h < HT; ++h)
#pragma unroll
    for (int x = 0; x < K0; ++x)
      q[h][x] = *reinterpret_cast<const s16x8*>(qs + ((hf * HT + h) * KS + min(part_e * K0 + x, KS - 1)) * 1024 + lane * 16);
  const float qmul = __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(
      a.scale * (MODE % 2 == 1 ? 2.f * kLog2e / a.softcap : MODE == 2 ? -kLog2e : kLog2e))));
  const float cap2 = MODE % 2 == 1 ? a.softcap * kLog2e : 0.f;
  float hb[HT];
#pragma unroll
  for (int h = 0; h < HT; ++h) hb[h] = MODE >= 2 && a.head_bias != nullptr ? a.head_bias[hh[h]] * kLog2e : 0.f;

  const int ksw = wide_swizzle(col), vrow = 4 * grp + (col >> 2), vsw = wide_swizzle(vrow);
  const int k_even = (kt * 16 + col) * E + part_e * (K0 * 32) + (grp ^ ksw) * 8;
  const int k_odd = (kt * 16 + col) * E + part_e * (K0 * 32) + ((4 + grp) ^ ksw) * 8;
  int vat[4];
#pragma unroll
  for (int u = 0; u < 4; ++u) vat[u] = vrow * E + ((2 * u + ((col >> 1) & 1)) ^ vsw) * 8 + (col & 1) * 4 + cq * 128;
  auto first_key = [&](int k) { return block_of(k) * WBS; };
  auto is_edge = [&](int jb) { return jb + WBS - 1 > row.pi || (jb < row.jwin && jb + WBS > row.kf); };
  // rows past the query were never written, rows out of its sight may hold infinities: zeros
  auto clear = [&](int k) {
    const int jb = first_key(k);
    if (!is_edge(jb)) return;
    short* const P = reinterpret_cast<short*>(smem) + k % NB * (kLatPage / 2);
    for (int x = tid; x < WBS * (E / 8); x += 512) {
      const int j = jb + x / (E / 8);
      if (j > row.pi || (j < row.jwin && j >= row.kf)) *reinterpret_cast<s16x8*>(P + x * 8) = (s16x8){0, 0, 0, 0, 0, 0, 0, 0};
    }
    sync();
  };
  auto scores = [&](int k) {
    const short* const P = pages_at + k % NB * (kLatPage / 2);
    f32x4 sc[HT][2];
#pragma unroll
    for (int h = 0; h < HT; ++h) sc[h][0] = sc[h][1] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int x = 0; x < K0; ++x)
      if (x < KS - K0 || part_e == 0) {
        const s16x8 kv = *reinterpret_cast<const s16x8*>(P + (x % 2 == 0 ? k_even : k_odd) + (x >> 1) * 64);
#pragma unroll
        for (int h = 0; h < HT; ++h)
          sc[h][x & 1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(kv), as_bf16x8(q[h][x]), sc[h][x & 1], 0, 0, 0);
      }
#pragma unroll
    for (int h = 0; h < HT; ++h) {
      const f32x4 s = sc[h][0] + sc[h][1];
      meet[((k & 1) * HT + h) * 512 + tid] = make_float4(s[0], s[1], s[2], s[3]);
    }
  };
  constexpr int DV = vdim / 16 / 4;
  f32x4 o[HT][DV];
#pragma unroll
  for (int h = 0; h < HT; ++h)
#pragma unroll
    for (int m = 0; m < DV; ++m) o[h][m] = (f32x4){0.f, 0.f, 0.f, 0.f};
  float mrun[HT], lrun[HT];
#pragma unroll
  for (int h = 0; h < HT; ++h) {
    mrun[h] = kNegInfW;
    lrun[h] = 0.f;
  }

  wait(min(n, NB - HT) - 1);
  sync();                                                     // and everyone has its queries
#pragma unroll
  for (int k = NB - HT; k < NB; ++k)
    if (k < n) copy(ahead[k], k);
  int32_t next = number(NB);
  clear(0);
  if (!idle) scores(0);
  for (int k = 0; k < n; ++k) {
    wait((k == 0 ? min(n, NB) : min(n, k + NB - 1)) - (k + 2));       // page k + 1
    sync();                                                   // scores of page k; nobody needs page k - 1
    if (k > 0 && k + NB - 1 < n) {
      copy(next, k + NB - 1);
      next = number(k + NB);
    }
    if (k + 1 < n) clear(k + 1);
    if (idle) continue;
    // waves w and w + 4 share a SIMD: one has scores to make while the other has weights and values
    if (k + 1 < n && part_e == 0) scores(k + 1);
    const int jb = first_key(k);
    const bool edge = is_edge(jb);
    s16x8 phi[HT], plo[HT];
#pragma unroll
    for (int h = 0; h < HT; ++h) {
      const float4* const part_s = meet + ((k & 1) * HT + h) * 512 + lane;
      float p[8];
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const float4 x = part_s[(hf + 2 * u) * 64], y = part_s[(hf + 2 * u + 4) * 64];
        p[4 * u] = x.x + y.x;
        p[4 * u + 1] = x.y + y.y;
        p[4 * u + 2] = x.z + y.z;
        p[4 * u + 3] = x.w + y.w;
      }
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        float x = p[e] * qmul;
        if constexpr (MODE % 2 == 1) x = cap2 - 2.f * cap2 * __builtin_amdgcn_rcpf(__builtin_amdgcn_exp2f(x) + 1.f);
        if constexpr (MODE >= 2) x = __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f((MODE == 3 ? -x : x) - hb[h]));
        p[e] = x;
      }
      if (edge) {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const int j = jb + (e >> 2) * 16 + grp * 4 + (e & 3);
          const bool ok = (j <= row.pi) & ((j >= row.jwin) | (j < row.kf));
          p[e] = ok ? p[e] : MODE >= 2 ? 0.f : kNegInfW;
        }
      }
      if constexpr (MODE < 2) {
        float mx = fmaxf(fmaxf(fmaxf(p[0], p[1]), fmaxf(p[2], p[3])), fmaxf(fmaxf(p[4], p[5]), fmaxf(p[6], p[7])));
        mx = other_half_max(other_row_max(mx));
        const bool moves = mx > mrun[h] + kDeferW;            // also for the first keys: mrun = -inf
        if (__builtin_amdgcn_ballot_w64(moves) != 0ull) {
          const float mn = moves ? mx : mrun[h];
          const float alpha = moves ? __builtin_amdgcn_exp2f(mrun[h] - mn) : 1.f;
          mrun[h] = mn;
          lrun[h] *= alpha;
#pragma unroll
          for (int m = 0; m < DV; ++m) o[h][m] *= alpha;
        }
        const float mu = mrun[h] == kNegInfW ? 0.f : mrun[h];         // no visible key so far: every weight 0
        float l0 = 0.f, l1 = 0.f;
#pragma unroll
        for (int e = 0; e < 8; e += 2) {
          p[e] = __builtin_amdgcn_exp2f(p[e] - mu);
          p[e + 1] = __builtin_amdgcn_exp2f(p[e + 1] - mu);
          l0 += p[e];
          l1 += p[e + 1];
        }
        lrun[h] += l0 + l1;
      }
      split_bf16w(p, phi[h], plo[h]);
    }
    const short* const P = pages_at + k % NB * (kLatPage / 2);
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
      for (int h = 0; h < HT; ++h) {
#pragma unroll
        for (int u = 0; u < 4; ++u)
          o[h][m + u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(v[u]), as_bf16x8(phi[h]), o[h][m + u], 0, 0, 0);
#pragma unroll
        for (int u = 0; u < 4; ++u)
          o[h][m + u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(v[u]), as_bf16x8(plo[h]), o[h][m + u], 0, 0, 0);
      }
    }
    if (k + 1 < n && part_e == 1) scores(k + 1);
  }
  const int dv = cq * 128 + 4 * grp;
#pragma unroll
  for (int h = 0; h < HT; ++h) {
    const float l = both_halves_sum(both_rows_sum(lrun[h]));
    if (h0 + h * 16 + col >= rep) continue;
    // scores that are no numbers leave the maximum at -inf, which marks a share without visible keys
    const float mx = MODE >= 2 || (l != 0.f && mrun[h] == kNegInfW) ? 0.f : mrun[h];
    if (shares == 1) {                                        // nobody to meet
      const float f = whole<MODE>(a, t, hh[h], mx, l);
#pragma unroll
      for (int m = 0; m < DV; ++m) {
        float y[4] = {o[h][m][0] * f, o[h][m][1] * f, o[h][m][2] * f, o[h][m][3] * f};
        store_gated<vdim>(a, y, t, hh[h], dv + 16 * m);
      }
      continue;
    }
    const int64_t at = (t * S + z) * a.H + hh[h];
#pragma unroll
    for (int m = 0; m < DV; ++m) *reinterpret_cast<f32x4*>(part + at * vdim + dv + 16 * m) = o[h][m];
    if (cq == 0 && grp == 0) *reinterpret_cast<float2*>(part + (int64_t)T * S * a.H * vdim + 2 * at) = make_float2(mx, l);
  }
}

// One wave per row and head: the workgroups' parts, the sink, the gate.
template <int HT, int MODE>
__global__ __launch_bounds__(64) void attn_keep_streams_merge_kernel(const KeepArgs a, const float* part, int T, int S,
                                                                      int NA) {
  constexpr int vdim = kLatV, NC = vdim / 256, AHEAD = 4;     // pieces of four channels a lane; shares on their way at once
  const int64_t t = blockIdx.x;
  const int hx = blockIdx.y, lane = threadIdx.x;
  const RowPages row = row_pages(a, NA, (int)t);
  if (row.s < 0) return;
  const int shares = row_shares<HT>(row, S);
  if (shares == 1) return;                                    // its workgroup has stored the row itself
  const float2* ml = reinterpret_cast<const float2*>(part + (int64_t)T * S * a.H * vdim);
  const int64_t at = t * S * a.H + hx;
  const float2 m = ml[at + (int64_t)min(lane, shares - 1) * a.H];           // a lane's share
  const float4* from = reinterpret_cast<const float4*>(part + at * vdim) + lane;
  const float top = wave_max(m.x);
  const float f = m.x == kNegInfW ? 0.f : MODE >= 2 ? 1.f : __builtin_amdgcn_exp2f(m.x - top);   // 0: without visible keys
  const float l = wave_sum(lane < shares && f != 0.f ? f * m.y : 0.f);
  float y[NC][4];
#pragma unroll
  for (int n = 0; n < NC; ++n) y[n][0] = y[n][1] = y[n][2] = y[n][3] = 0.f;
  for (int z0 = 0; z0 < shares; z0 += AHEAD) {
    float4 v[AHEAD][NC];
#pragma unroll
    for (int u = 0; u < AHEAD; ++u)
#pragma unroll
      for (int n = 0; n < NC; ++n) v[u][n] = from[((int64_t)min(z0 + u, shares - 1) * a.H * vdim + 256 * n) / 4];
#pragma unroll
    for (int u = 0; u < AHEAD; ++u) {
      const float fz = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(f), min(z0 + u, shares - 1)));
      if (z0 + u >= shares || fz == 0.f) continue;
#pragma unroll
      for (int n = 0; n < NC; ++n) {
        y[n][0] += fz * v[u][n].x; y[n][1] += fz * v[u][n].y; y[n][2] += fz * v[u][n].z; y[n][3] += fz * v[u][n].w;
      }
    }
  }
  const float mul = whole<MODE>(a, t, hx, top, l);
#pragma unroll
  for (int n = 0; n < NC; ++n) {
#pragma unroll
    for (int e = 0; e < 4; ++e) y[n][e] *= mul;
    store_gated<vdim>(a, y[n], t, hx, 256 * n + 4 * lane);
  }
}

// ------------------------------------------------------------------ launcher
// How many workgroups share a row's pages, 0 where the streams are not the way: more than the 16 heads of one wave,
// room for two workgroups or more a row, and pages that a row may see, by its table and window, which repay the scratch and
// the second launch: they cost a layer's pass that the host bounds 4 us (32 heads, one or eight sequences of 300 tokens 35 us
// split over waves, 40 in streams; of 400 40 both, of 450 42.5 and 39.5, of 600 47 and 39.5; 64 sequences of 300 39 both, of
// 400 44 and 39.7, of 600 51 and 39.6; with 64 heads and so two workgroups a row 48 and 54 up to 500 tokens, 53 and 54 of 600).
// Captured steps have wide tables over any number of pages: there a row of one page takes 15 us split, twelve in streams.
// 64 heads together, half as many reads of a page for three pages in LDS instead of four and 5 us more on the way to the
// first: where 32 leave no two workgroups a row (100 sequences of 900 tokens with 64 heads 82 us by the prompts' kernel, 53;
// 128 of 600 58, 45), or just two and the rows are long (64 of 2,000 60 us with 32 heads, 55.5 with 64; of 600 30 and 34; a
// captured step's table says nothing about that).  Short rows of captured steps cost more so than by the prompts' kernel: 128
// sequences with 64 heads of 20 tokens 17.9 for 12.5, of 100 24.7 for 20.8, of 200 31 for 29, of 300 38 for 37.  Rows of up to
// eight pages shared by two workgroups, whose parts then meet, took 29 and 35 of 100 and 200.
// Of up to NA rows a sequence may have several: each has workgroups of its own, as in a captured step rows of an extend
// stand where other sequences are padding (one sequence of 600 tokens with 16 rows, 16 of one and 15 without: 143 us
// split over waves, 269 with an extend's rows one after another, 23 side by side).
namespace {
struct Streams {
  int S, tiles;                                    // workgroups a row, of 32 heads times tiles each
};
Streams streams_of(int T, int NA, int H, int G, int maxb, int window, int keep_first) {
  const int rep = H / G;
  // pages that a row can see: of its table, of the window and of the kept first tokens
  const int64_t seen = ((int64_t)window + WBS - 2) / WBS + 1 + ((int64_t)keep_first + WBS - 1) / WBS;
  const int64_t most = window > 0 ? std::min<int64_t>(maxb, seen) : maxb;
  auto shares = [&](int heads) {
    const int64_t wgs = std::max<int64_t>((int64_t)NA * G * ((rep + heads - 1) / heads), 1);
    return (int)std::min(256 / wgs, std::min<int64_t>((most + kSharePages - 1) / kSharePages, 16));
  };
  const int narrow = shares(32), wide = shares(64);
  if (most <= (narrow >= 4 ? 13 : 20) || T > NA) return {0, 1};
  if (rep > 32 && wide >= 2 && (narrow < 2 || (narrow == 2 && most > 48 && most < 128))) return {wide, 2};
  return {narrow >= 2 ? narrow : 0, 1};
}
}  // namespace
int keep_streams(int T, int NA, int H, int G, int E, int vdim, bool shared, int maxb, int window, int keep_first) {
  if (!shared || E != kLatE || vdim != kLatV || H / G <= 16 || NA <= 0 || H > 65535) return 0;
  return streams_of(T, NA, H, G, maxb, window, keep_first).S;
}
int64_t keep_streams_floats(int T, int S, int H, int vdim) { return (int64_t)T * S * H * (vdim + 2); }

template <int HT, int MODE>
static void launch_streams_tiles(const KeepArgs& a, int T, int NA, int S, float* part) {
  constexpr size_t lds = stream_pages(HT) * kLatPage + 2 * HT * 512 * sizeof(float4);
  static_assert(lds <= 160 * 1024, "LDS of a CU");
  static bool attr = false;
  if (!attr) {
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&attn_keep_streams_kernel<HT, MODE>),
                              hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
    attr = true;
  }
  hipLaunchKernelGGL((attn_keep_streams_kernel<HT, MODE>), dim3(T, a.G * ((a.H / a.G + 32 * HT - 1) / (32 * HT)), S), dim3(512), lds, a.s, a,
                     part, T, NA);
  hipLaunchKernelGGL((attn_keep_streams_merge_kernel<HT, MODE>), dim3(T, a.H), dim3(64), 0, a.s, a, part, T, S, NA);
}
template <int MODE>
static void launch_streams_one(const KeepArgs& a, int T, int NA, int S, float* part) {
  if (streams_of(T, NA, a.H, a.G, a.maxb, a.window, a.keep_first).tiles == 2) launch_streams_tiles<2, MODE>(a, T, NA, S, part);
  else launch_streams_tiles<1, MODE>(a, T, NA, S, part);
}

void launch_attn_keep_streams(const float* q, const void* k_cache, int64_t vrs, const int32_t* bt, int maxb,
                              const int32_t* q_start, const int32_t* q_len, const int32_t* kv_len, int T, int NA, int S,
                              const float* head_bias, const void* gate, int64_t gate_stride, int gate_w, void* out,
                              int64_t out_stride, float scale, int window, int keep_first, bool sigmoid, int H, int G,
                              float softcap, float out_mult, float* part, hipStream_t s) {
  const KeepArgs a{q, k_cache, k_cache, vrs, bt, maxb, q_start, q_len, kv_len, nullptr, nullptr,
                   0, head_bias, gate, gate_stride, gate_w, out, out_stride, scale, window, keep_first,
                   sigmoid, H, G, softcap, out_mult, s};
  const bool cap = softcap > 0.f;
  if (sigmoid && cap) launch_streams_one<3>(a, T, NA, S, part);
  else if (sigmoid) launch_streams_one<2>(a, T, NA, S, part);
  else if (cap) launch_streams_one<1>(a, T, NA, S, part);
  else launch_streams_one<0>(a, T, NA, S, part);
}

}  // namespace rfqmix
