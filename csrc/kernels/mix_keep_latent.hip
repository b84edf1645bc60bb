// attn_keep_window, prompt rows of 576-wide latents whose first 512 entries are the values (bf16 pages of 32 tokens),
// four heads a workgroup.  Semantics of mix_keep_attn_mfma.hip.
//
// One workgroup per (work item, four heads of a key head), two waves a head and its 32 queries, one on each half of a
// SIMD's registers: 32 queries' values (256 registers) and the queries (144) do not fit one wave's 256 together.
//
//   scores    S^T[key, query] = K . Q^T on 32 x 32 tiles, the queries as bf16 in registers; cap, mask, maximum and
//             weights; the weights to LDS as bf16 hi + lo parts (fp32's precision), with the factor by which the
//             maximum's move scales what was there; the last three of sixteen tiles of values
//   values    the other thirteen tiles of O^T[channel, query] += V^T . P^T, a page behind; the copies of pages
//
// One barrier a page, three pages in LDS: scores of page i, values of page i - 1, page i + 1 on its way (LDS-DMA, its
// pieces issued between the products).  Rows of 1,152 bytes lie unpadded, 16-byte pieces permuted by wide_swizzle:
// reads of 32 rows, plain and transposed, are without bank conflicts.
//
// What bounds it: the products' power.  A page of a wave pair is 100 products (36 of scores, 2 x 32 of values, hi and
// lo), 3,200 clocks of a SIMD, of which a turn takes 3,900; at that rate the chip lowers its clock to 1.25 - 1.5 GHz,
// 1.37 PFLOP/s of these products, as much as a large bf16 product reaches.  Without its LDS reads a turn would be 6 %
// shorter, without the lo parts 22 %.  Beside it 870 MB of queries and results where a step has 8,192 rows of 32 heads.
// A page a workgroup takes 2.4 us; on 16 x 16 tiles, 16 queries a wave and every wave with all of a page, twice the LDS
// reads, it took 3.0.  Queries come by LDS-DMA in whole lines, results leave by way of LDS: as the tiles have them, 32
// bytes and 8 bytes of 32 rows to an access, these took 15 and 10 us a workgroup.  Attention alone, call after call, 32
// heads: four prompts of 2,048 854 -> 725 us (772 and more where it is traced behind a pass's large products), one 213 -> 181,
// one of 77 24.2 -> 13.5, eight chunks of 96 - 740 rows after 416 227 -> 181; 187 steps of 1 to 8,192 rows, 3 to 64 heads, all
// kinds of weights and windows 1.02 - 2.1 times as fast.
// Four tiles of values beside the scores take 2.8 us a page; with two the other wave's fourteen spill.
#include <algorithm>
#include <type_traits>

#include "mix_keep_mfma.h"

namespace rfqmix {

constexpr int kScoreTiles = 3;          // tiles of 32 value channels that a wave of scores has room for beside its queries

// A thread's number that what was derived from it before does not come back with: it would stay in registers over the
// loops, of which these kernels have none to spare.
__device__ __forceinline__ int fresh(int tid) {
  asm volatile("" : "+v"(tid));
  return tid;
}

// N tiles of 32 value channels (lane (col, half): channels 8 b + 4 half .. + 3 of query col) from channel c0 on, times
// mul and a gate per output, by way of `stage` (2 KB a tile): stores of 64 bytes a row, 16 rows to an access.  As the
// tiles lie, 8 bytes of 32 rows, they took 10 us a workgroup.
template <int N>
__device__ __forceinline__ void store_staged(const KeepArgs& a, const f32x16 (&o)[N], float mul, int t0, int nq, int hh,
                                             int c0, short* stage, int lane) {
  const int col = lane & 31, half = lane >> 5, vdim = 512;
  const bf16_t* gate = static_cast<const bf16_t*>(a.gate);
  const bool gated = gate != nullptr && a.gate_w > 1;
  gate += gated ? (int64_t)(t0 + min(col, nq - 1)) * a.gate_stride + (int64_t)hh * vdim + c0 + half * 4 : 0;
  auto put = [&](auto gated_c) {
#pragma unroll
    for (int m = 0; m < N; ++m)
#pragma unroll
      for (int b = 0; b < 4; ++b) {
        float y[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) y[i] = o[m][4 * b + i] * mul;
        if constexpr (gated_c) {                                           // four neighbouring logits, 8-byte reads
          const uint2 gu = *reinterpret_cast<const uint2*>(gate + m * 32 + b * 8);
          y[0] /= 1.0f + __expf(-__uint_as_float(gu.x << 16));
          y[1] /= 1.0f + __expf(-__uint_as_float(gu.x & 0xffff0000u));
          y[2] /= 1.0f + __expf(-__uint_as_float(gu.y << 16));
          y[3] /= 1.0f + __expf(-__uint_as_float(gu.y & 0xffff0000u));
        }
        *reinterpret_cast<uint2*>(stage + m * 1024 + col * 32 + (b ^ ((col >> 2) & 3)) * 8 + half * 4) =
            make_uint2(rfq::pack_bf16x2(y[0], y[1]), rfq::pack_bf16x2(y[2], y[3]));
      }
  };
  if (gated) put(std::true_type{});
  else put(std::false_type{});
  typedef uint32_t u32x4_8 __attribute__((ext_vector_type(4), aligned(8)));        // rows may be 8-byte aligned
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int row = 16 * h + (lane >> 2);
    if (row >= nq) continue;
    bf16_t* out = static_cast<bf16_t*>(a.out) + (int64_t)(t0 + row) * a.out_stride + (int64_t)hh * vdim + c0 + (lane & 3) * 8;
    const short* from = stage + row * 32 + ((lane & 3) ^ ((row >> 2) & 3)) * 8;
#pragma unroll
    for (int m = 0; m < N; ++m)
      *reinterpret_cast<u32x4_8*>(out + m * 32) = *reinterpret_cast<const u32x4*>(from + m * 1024);
  }
}

template <int MODE>
__global__ __launch_bounds__(512, 2) void attn_keep_roles_kernel(const KeepArgs a) {
  constexpr int E = 576, vdim = 512, KS = E / 16, VM = vdim / 32, VS = kScoreTiles, VP = VM - VS, HPW = 4;
  constexpr int PG = WBS * E;                       // shorts of a page
  const int rep = a.H / a.G, per = (rep + HPW - 1) / HPW;
  const int at = gridDim.x - 1 - blockIdx.x, item = at / (a.G * per), hg = at - item * a.G * per;
  const int s = a.work_seq[item];
  if (s < 0) return;
  const int ql = a.q_len[s];
  const int i0 = a.work_qblk[item] * WQB;
  if (i0 >= ql) return;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const bool scores = wid < HPW;                   // waves w and w + 4 share a SIMD
  const int w = wid & 3, col = lane & 31, half = lane >> 5;
  const int g = hg / per, hd = (hg - g * per) * HPW + w, hh = g * rep + min(hd, rep - 1);
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  short* const pages = reinterpret_cast<short*>(smem);                       // three of them
  u32x4* const weights = reinterpret_cast<u32x4*>(smem + 3 * PG * 2);        // two pages': [4][4][64]
  float* const factors = reinterpret_cast<float*>(smem + 3 * PG * 2 + 32768);   // [2][4][32]

  const int nq = min(WQB, ql - i0);
  const int p0 = a.kv_len[s] - ql + i0, plast = p0 + nq - 1;
  const int window = a.window, keep_first = a.keep_first;
  const int jwin = window > 0 ? max(0, p0 - window + 1) : 0;
  const int kf = window > 0 ? min(keep_first, jwin) : 0;     // kept keys before the window
  const int t0 = a.q_start[s] + i0;
  typedef const __attribute__((address_space(4))) int32_t const_i32;
  const_i32* bt = (const_i32*)(uintptr_t)(a.bt + (int64_t)s * a.maxb);

  // pages [0, n_keep) hold the kept first tokens, pages [pg_win, pg_last] the window
  const int pg_last = plast / WBS, pg_win = jwin / WBS;
  const int n_keep = min((kf + WBS - 1) / WBS, pg_win), skip = pg_win - n_keep, turns = pg_last + 1 - skip;
  auto page_at = [&](int i) { return i < n_keep ? i : i + skip; };
  auto number = [&](int i) { return bt[page_at(min(i, turns - 1))]; };

  const uint32_t lds0 = lds_byte(smem);
  // A quarter of a page is eight rows or nine pieces of 64 x 16 bytes; piece i has row i from lane 8 i on and row i - 1
  // below.  Source and image differ in the permutation alone, of which the quarter adds 2 to odd ones.
  const uint32_t lane16 = (uint32_t)(lane ^ ((w & 1) << 1)) * 16;
  auto copy = [&](int page, int buf, auto piece) {
    constexpr int i = piece;
    const char* kb = static_cast<const char*>(a.k_cache) + (((int64_t)page * a.G + g) * PG + w * (PG / 4) + i * 512) * 2;
    const uint32_t upper = i < 8 ? wide_swizzle(i) * 16 : 0, lower = i > 0 ? wide_swizzle(i - 1) * 16 : 0;
    lds_copy16(kb, lane16 ^ (lane < 8 * i ? lower : upper), lds0 + 2 * (buf * PG + w * (PG / 4) + i * 512));
  };
  // everyone's copies have landed, everyone is done with what the next ones overwrite
  auto landed = [] {
    __builtin_amdgcn_s_waitcnt(0x0F70);                      // vmcnt(0)
    __syncthreads();
  };
  // rows past the sequence's end were never written: zeros
  auto tail = [&](int i) {
    const int jb = page_at(i) * WBS;
    if (i == turns - 1 && jb + WBS - 1 > plast) {
      for (int x = max(0, plast + 1 - jb) * (E / 8) + fresh(threadIdx.x); x < WBS * (E / 8); x += 512)
        *reinterpret_cast<s16x8*>(pages + i % 3 * PG + x * 8) = (s16x8){0, 0, 0, 0, 0, 0, 0, 0};
      __syncthreads();
    }
  };
  // values, transposed: rows 16 u + 8 j + 4 half + lane % 16 / 4, channels 32 m + 16 (lane / 16 % 2) + 4 (lane % 4) ..
  int vat[2][2];
#pragma unroll
  for (int j = 0; j < 2; ++j)
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int r = 8 * j + 4 * half + ((lane & 15) >> 2);
      vat[j][i] = r * E + ((4 * i + 2 * ((lane >> 4) & 1) + ((lane & 3) >> 1)) ^ wide_swizzle(r)) * 8 + (lane & 1) * 4;
    }
  auto value = [&](const short* P, int u, int m) {           // 16 keys x 32 channels
    const short* vp = P + (m >> 1) * 64 + u * 16 * E;
    const s16x4 a0 = rfq::ds_read_tr16(vp + vat[0][m & 1]), a1 = rfq::ds_read_tr16(vp + vat[1][m & 1]);
    return (s16x8){a0[0], a0[1], a0[2], a0[3], a1[0], a1[1], a1[2], a1[3]};
  };
  auto add = [](f32x16& o, const s16x8& v, const u32x4& p) {
    o = __builtin_amdgcn_mfma_f32_32x32x16_bf16(as_bf16x8(v), __builtin_bit_cast(rfq::bf16x8, p), o, 0, 0, 0);
  };
  const float hb = a.head_bias != nullptr ? a.head_bias[hh] * kLog2e : 0.f;

  if (scores) {
    const float qmul = a.scale * (MODE % 2 == 1 ? 2.f * kLog2e / a.softcap : MODE == 2 ? -kLog2e : kLog2e);
    const float cap2 = MODE % 2 == 1 ? a.softcap * kLog2e : 0.f;
    // The queries come through LDS, where the pages after the first will be, 64 entries of 32 rows a time, three
    // times on the way, up to eight rows all at once.  Read as the products want them, 32 bytes of 32 rows to an
    // access, they took 15 us.
    s16x8 q[KS];
    {
      constexpr int NCH = E / 64;
      const int base = 2 * PG + w * 3 * 8192;
      uint32_t src[8];                                       // four rows a piece; 16-byte parts permuted by the row
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const int r = 4 * i + (lane >> 4);
        src[i] = (uint32_t)(min(r, nq - 1) - min(4 * i, nq - 1)) * (uint32_t)(a.H * E * 4) + ((lane & 15) ^ (r & 15)) * 16;
      }
      auto bring = [&](int ch, int to, auto pieces) {
        each<pieces>([&](auto i) {
          lds_copy16(a.q + ((int64_t)(t0 + min(4 * i, nq - 1)) * a.H + hh) * E + ch * 64, src[i], lds0 + base + to + i * 1024);
        });
      };
      auto take = [&](int ch, int at, int r, auto next) {
        const float* rows = reinterpret_cast<const float*>(smem + base + at) + r * 64;
        float4 f[8];
#pragma unroll
        for (int x = 0; x < 8; ++x) f[x] = ld4(rows + ((4 * (x >> 1) + 2 * half + (x & 1)) ^ (r & 15)) * 4);
        next();
#pragma unroll
        for (int x = 0; x < 4; ++x) q[4 * ch + x] = rfq::pack8(&f[2 * x].x);     // as they are: bf16 values stay exact
        __builtin_amdgcn_sched_barrier(0);
      };
      constexpr std::integral_constant<int, 2> two{};
      constexpr std::integral_constant<int, 8> eight{};
      if (nq <= 8) {
        each<NCH>([&](auto ch) { bring(ch, ch * 2048, two); });
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        each<NCH>([&](auto ch) { take(ch, ch * 2048, col & 7, [] {}); });
      } else {
        each<3>([&](auto ch) { bring(ch, ch * 8192, eight); });
        each<NCH>([&](auto chunk) {
          constexpr int ch = chunk;
          if constexpr (ch + 2 < NCH) asm volatile("s_waitcnt vmcnt(16)" ::: "memory");
          else if constexpr (ch + 1 < NCH) asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
          else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
          take(ch, ch % 3 * 8192, col, [&] {
            if constexpr (ch + 3 < NCH) {
              asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
              bring(ch + 3, ch % 3 * 8192, eight);
            }
          });
        });
      }
    }
    f32x16 o[VS];
#pragma unroll
    for (int m = 0; m < VS; ++m)
#pragma unroll
      for (int e = 0; e < 16; ++e) o[m][e] = 0.f;
    const bool sink = MODE < 2 && a.head_bias != nullptr;
    float mrun = sink ? hb : kNegInfW, lrun = sink && half == 0 ? 1.f : 0.f;
    int kat[4];                                              // keys: row col, entries 16 ks + 8 half ..
#pragma unroll
    for (int i = 0; i < 4; ++i) kat[i] = col * E + ((2 * i + half) ^ wide_swizzle(col)) * 8;

    for (int i = 0; i < turns; ++i) {
      landed();
      tail(i);
      const short* P = pages + i % 3 * PG;
      const int jb = page_at(i) * WBS;
      constexpr int AK = 4;                                  // operands are read that many products ahead
      auto key = [&](int ks) { return *reinterpret_cast<const s16x8*>(P + kat[ks & 3] + (ks >> 2) * 64); };
      s16x8 kc[AK];
#pragma unroll
      for (int x = 0; x < AK; ++x) kc[x] = key(x);
      f32x16 sc;
#pragma unroll
      for (int e = 0; e < 16; ++e) sc[e] = 0.f;
      each<KS>([&](auto step) {
        constexpr int ks = step;
        sc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(as_bf16x8(kc[ks % AK]), as_bf16x8(q[ks]), sc, 0, 0, 0);
        if constexpr (ks + AK < KS) kc[ks % AK] = key(ks + AK);
        __builtin_amdgcn_sched_barrier(0);
      });
      float p[16];
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        float x = sc[e] * qmul;
        if constexpr (MODE % 2 == 1) x = cap2 - 2.f * cap2 * __builtin_amdgcn_rcpf(__builtin_amdgcn_exp2f(x) + 1.f);
        if constexpr (MODE >= 2) x = __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f((MODE == 3 ? -x : x) - hb));
        p[e] = x;
      }
      if (!(jb + WBS - 1 <= p0 && (window <= 0 || plast - jb < window || jb + WBS <= keep_first))) {
        const int at = jb + half * 4, hi = p0 + col - at, lo = window > 0 ? hi - window : -WBS, kept = keep_first - at;
#pragma unroll
        for (int e = 0; e < 16; ++e) {                       // an edge inside the page
          const int j = (e >> 2) * 8 + (e & 3);
          const bool ok = (j <= hi) & ((j > lo) | (j < kept));
          p[e] = ok ? p[e] : MODE >= 2 ? 0.f : kNegInfW;
        }
      }
      if constexpr (MODE < 2) {
        float mx = p[0];
#pragma unroll
        for (int e = 1; e < 16; ++e) mx = fmaxf(mx, p[e]);
        mx = other_half_max(mx);
        const bool moves = mx > mrun + kDeferW;              // also for the first keys: mrun = -inf
        float alpha = 1.f;
        if (__builtin_amdgcn_ballot_w64(moves) != 0ull) {
          const float mn = moves ? mx : mrun;
          alpha = moves ? __builtin_amdgcn_exp2f(mrun - mn) : 1.f;
          mrun = mn;
          lrun *= alpha;
#pragma unroll
          for (int m = 0; m < VS; ++m) o[m] *= alpha;
        }
        if (half == 0) factors[((i & 1) * HPW + w) * 32 + col] = alpha;
        const float mu = mrun == kNegInfW ? 0.f : mrun;      // no visible key so far: every weight 0
        float l0 = 0.f, l1 = 0.f;
#pragma unroll
        for (int e = 0; e < 16; e += 2) {
          p[e] = __builtin_amdgcn_exp2f(p[e] - mu);
          p[e + 1] = __builtin_amdgcn_exp2f(p[e + 1] - mu);
          l0 += p[e];
          l1 += p[e + 1];
        }
        lrun += l0 + l1;
      }
      u32x4 phi[2], plo[2];
      u32x4* const wp = weights + ((i & 1) * HPW + w) * 256 + lane;
#pragma unroll
      for (int u = 0; u < 2; ++u) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float x = p[8 * u + 2 * e], y = p[8 * u + 2 * e + 1];
          const uint32_t h = rfq::pack_bf16x2(x, y);
          phi[u][e] = h;
          plo[u][e] = rfq::pack_bf16x2(x - __uint_as_float(h << 16), y - __uint_as_float(h & 0xffff0000u));
        }
        wp[u * 128] = phi[u];
        wp[u * 128 + 64] = plo[u];
      }
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int m = 0; m < VS; ++m) {
          const s16x8 v = value(P, u, VP + m);
          add(o[m], v, phi[u]);
          add(o[m], v, plo[u]);
        }
    }
    landed();                                                // the other waves' last page
    const int ln = fresh(threadIdx.x) & 63, cl = ln & 31;
    const int64_t t = t0 + (cl < nq ? cl : 0);
    const float mul = row_factor<MODE>(a, both_halves_sum(lrun), t, hh);
    landed();                                                // factors of the last page have been read
    if (ln < 32) factors[w * 32 + cl] = mul;
    __syncthreads();
    if (hd >= rep) return;
    store_staged<VS>(a, o, mul, t0, nq, hh, 32 * VP, pages + (4 * VP + w * VS) * 1024, ln);
  } else {
    f32x16 o[VP];
#pragma unroll
    for (int m = 0; m < VP; ++m)
#pragma unroll
      for (int e = 0; e < 16; ++e) o[m][e] = 0.f;
    int32_t ahead = number(0);
    each<9>([&](auto piece) { copy(ahead, 0, piece); });
    ahead = number(1);
    landed();
    tail(0);
    each<9>([&](auto piece) { copy(ahead, 1, piece); });
    ahead = number(2);
    for (int i = 1; i <= turns; ++i) {
      landed();
      if (i < turns) tail(i);
      const short* P = pages + (i - 1) % 3 * PG;
      const u32x4* const wp = weights + (((i - 1) & 1) * HPW + w) * 256 + lane;
      if constexpr (MODE < 2) {
        const float alpha = factors[(((i - 1) & 1) * HPW + w) * 32 + col];
        if (__builtin_amdgcn_ballot_w64(alpha != 1.f) != 0ull) {
#pragma unroll
          for (int m = 0; m < VP; ++m) o[m] *= alpha;
        }
      }
      constexpr int AV = 3, C = 2 * VP;
      u32x4 phi = wp[0], plo = wp[64], hi1, lo1;
      s16x8 vc[AV];
#pragma unroll
      for (int x = 0; x < AV; ++x) vc[x] = value(P, x / VP, x % VP);
      each<C>([&](auto step) {
        constexpr int c = step;
        if constexpr (c == VP) {
          phi = hi1;
          plo = lo1;
        }
        const s16x8 v = vc[c % AV];
        add(o[c % VP], v, phi);
        add(o[c % VP], v, plo);
        if constexpr (c + AV < C) vc[c % AV] = value(P, (c + AV) / VP, (c + AV) % VP);
        if constexpr (c >= 2 && c % 2 == 0 && c < 20) {
          copy(ahead, (i + 1) % 3, std::integral_constant<int, c / 2 - 1>{});
        }
        if constexpr (c == VP - 4) {
          hi1 = wp[128];
          lo1 = wp[192];
        }
        __builtin_amdgcn_sched_barrier(0);
      });
      ahead = number(i + 2);
    }
    landed();
    __syncthreads();
    if (hd >= rep) return;
    const int ln = fresh(threadIdx.x) & 63, cl = ln & 31;
    store_staged<VP>(a, o, factors[w * 32 + cl], t0, nq, hh, 0, pages + w * VP * 1024, ln);
  }
}

// ------------------------------------------------------------------ launcher
template <int MODE>
static void launch_latent_mode(const KeepArgs& a) {
  constexpr int lds = 3 * WBS * 576 * 2 + 32768 + 1024;
  static bool attr = false;
  if (!attr) {
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&attn_keep_roles_kernel<MODE>),
                              hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
    attr = true;
  }
  const int groups = a.G * ((a.H / a.G + 3) / 4), most = std::max(1, (1 << 22) / groups);   // threads in 32 bits
  for (int w = 0; w < a.W; w += most) {
    KeepArgs part = a;
    part.work_seq += w;
    part.work_qblk += w;
    hipLaunchKernelGGL(attn_keep_roles_kernel<MODE>, dim3((unsigned)std::min(most, a.W - w) * groups), dim3(512), lds, a.s, part);
  }
}

void launch_attn_keep_latent(const KeepArgs& a) {
  const bool cap = a.softcap > 0.f;
  if (a.sigmoid && cap) launch_latent_mode<3>(a);
  else if (a.sigmoid) launch_latent_mode<2>(a);
  else if (cap) launch_latent_mode<1>(a);
  else launch_latent_mode<0>(a);
}

}  // namespace rfqmix
