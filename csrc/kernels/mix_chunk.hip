// Linear recurrences with a decay per key channel (wkv, gated linear attention, gated delta rule:
// mix_wkv.hip and mix_linrec.hip have their definitions) in chunks of 16 tokens on fp32 MFMA tiles.
//
// With D_t = diag(a_t), inside a chunk that starts from the state S,
//
//   o_t = Qd_t S + sum_{s<=t} A[t,s] u_s          Qd_t = q_t a_1 .. a_t
//   S  <- a_1 .. a_16 S + sum_s Kd_s u_s          Kd_s = k_s a_{s+1} .. a_16
//   A[t,s] = sum_c q_t[c] k_s[c] (a_{s+1} .. a_t)[c]
//
// (wkv reads before it writes: its products of q end at a_{t-1}, and A[t,t] = sum_c q u k.)  Without
// the delta rule u_s = v_s.  With it U = T (beta (V - Kk S)), Kk_t = k_t a_1 .. a_t, T the inverse
// of the unit lower triangle I + beta A_kk, A_kk[t,s] = sum_c k_t k_s a_{s+1} .. a_t for s < t.
// All decay products are running products of the decays themselves: no logarithm, no quotient, so
// nothing overflows and nothing cancels however strong the decay.  Pairs of different four-token
// blocks factor at the block's edge: (a_{block} .. a_t) from the reader's side, (a_{s+1} ..) from
// the writer's, both at most 1; pairs inside a block multiply their decays directly.
//
// What bounds it: the chain over a run's chunks, and inside a chunk the instructions of the waves
// that share a SIMD.  Token by token the chain was 0.2 - 2.6 us a token (LDS round trips, 64 x 64
// FMAs on one or four waves); here a chunk's chain is 36 (wkv, gla) or 56 (delta) MFMAs of 16x16x4
// per wave, 1.6 - 2.3 us.  One workgroup per (run, head, 64 value channels): four consumer waves hold
// 64 x 16 of the state in accumulators, which are MFMA operands as they lie (a lane holds channels
// 16 i + 4 grp + r of its column: exactly the K slices that step (i, r) of Qd S takes); the other
// waves work ahead: decays and their products for chunk c + 3, A for chunk c + 2, T for chunk c + 1,
// wkv's norm and gate for chunk c - 1; one barrier per chunk.  A state operand never leaves the
// registers, an fp32 operand is never narrowed.  Measured, two runs of 2,048 tokens in bf16: wkv with
// 64 heads of 64 x 64 5,353 -> 203 us; delta rule with 32 heads of 64 x 128 741 (decays and scan) ->
// 301 us; gla in fp32, five ragged runs of up to 1,031, 32 heads, 447 -> 121 us.
//
// Without the delta rule a run's chain is cut where workgroups leave CUs idle (chunk_seg_rows): chunk_segment_kernel
// makes what every segment's rows leave of a state of zeros and the products of its decays, all segments at once, and a
// segment's workgroup begins from the state of before the run carried through those in front of it.  wkv, two runs of
// 2,048 with 64 heads: 204 -> 26 + 118 us.  What bounds the first kernel: exponentials (22 instructions a decay, 38 of gla)
// and the way to its first rows and out, 10 us of a workgroup.
#include <algorithm>
#include <type_traits>

#include "common.h"
#include "mix_common.h"
#include "mix_chunk.h"

namespace rfqmix {

using rfq::f32x4;

namespace {
constexpr int CT = 16;                  // tokens per chunk
constexpr int NC = kChunkDim;           // key channels (those past dim are zeros)
constexpr int RS = NC + 4;              // floats per token row in LDS
constexpr int TS = CT + 4;              // floats per row of a 16 x 16 tile, of Kd^T

// four consumers, four waves for the decays, four for A (and T), wkv: four for norm and gate
constexpr int chunk_threads(int mode) { return mode == kChunkWkv ? 1024 : 768; }

__device__ __forceinline__ float ror_add(float v) {   // sum over the 16 lanes of a row
  v += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x128, 0xf, 0xf, true));
  v += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x124, 0xf, 0xf, true));
  v += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x122, 0xf, 0xf, true));
  v += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x121, 0xf, 0xf, true));
  return v;
}
// What a chunk's producers leave in LDS.
template <int MODE>
struct ChunkLds {
  static constexpr bool DELTA = MODE == kChunkDelta;
  float qd[4][CT * RS];                 // four chunks in flight between producers and consumers
  float kk[DELTA ? 4 : 1][DELTA ? CT * RS : 4];
  float kd[4][NC * TS];                 // Kd^T
  float dec[4][NC];
  float beta[4][CT];
  float aq[4][CT * TS];
  float ak[2][DELTA ? CT * TS : 4];
  float tt[2][DELTA ? CT * TS : 4];
  float q[2][CT * RS], k[2][CT * RS], a[2][CT * RS];      // operands of A: raw,
  float ql[2][CT * RS], kl[2][CT * RS];                   // times the block's products up to / after
  float kb[2][DELTA ? CT * RS : 4];
  float blk[2][4 * NC];                 // product of a block's decays
  float o[2][MODE == kChunkWkv ? CT * RS : 4];
};

__device__ __forceinline__ float4 mul4(float4 x, float4 y) {
  return make_float4(x.x * y.x, x.y * y.y, x.z * y.z, x.w * y.w);
}
__device__ __forceinline__ float dot4(float4 x, float4 y) {
  return x.x * y.x + x.y * y.y + x.z * y.z + x.w * y.w;
}
__device__ __forceinline__ float silu_c(float x) {
  return x * __builtin_amdgcn_rcpf(1.f + exp_c(x < -87.f ? 87.f : -x));
}

// An operand in flight across a turn of the loop: its bits as loaded.  `arrived` converts it where it
// stands: left to the compiler, the conversion moves to the end of the turn that loaded it, or past
// the next load into the same register, and either way the wave waits there for memory.
template <typename T>
__device__ __forceinline__ T load_at(const T* base, uint32_t bytes) {
  return *reinterpret_cast<const T*>(reinterpret_cast<const char*>(base) + bytes);
}
__device__ __forceinline__ float arrived(float bits) {
  float f;
  asm volatile("v_mov_b32 %0, %1" : "=v"(f) : "v"(bits));
  return f;
}
__device__ __forceinline__ float arrived(bf16_t bits) {
  float f;
  asm volatile("v_lshlrev_b32 %0, 16, %1" : "=v"(f) : "v"(bits));
  return f;
}
}  // namespace

namespace {
__device__ __forceinline__ bool finite4(const f32x4& x) {      // no infinity, no NaN among them
  return fabsf((fabsf(x[0]) + fabsf(x[1])) + (fabsf(x[2]) + fabsf(x[3]))) < __builtin_huge_valf();
}

// o[t] += sum_{s<=t} m[t][s] x[s] with the pairs s > t left out instead of multiplied by zero: a
// token's infinity or NaN stays out of the tokens before it.  (Also taken, with the same result,
// where the sum of four finite values overflows.)
__device__ __forceinline__ void lower_product(const float* m, const f32x4& x, int col, int grp, f32x4& o) {
#pragma unroll 1
  for (int b = 0; b < 4; ++b) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int s = 4 * b + e;
      const float xs = __shfl(x[e], 16 * b + col, 64);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float y = o[r] + m[(4 * grp + r) * TS + s] * xs;
        o[r] = s <= 4 * grp + r ? y : o[r];
      }
    }
  }
}
}  // namespace

// A run's segment `seg` (the slot-th of the step): rows [t0, t0 + n) of the run from row run0 on.
struct ChunkSegment {
  int run0, t0, n, seg, slot;
  bool last;
};
__device__ __forceinline__ ChunkSegment whole_run(const ChunkArgs& a, int t0) {
  return {t0, t0, a.row_fwd[t0] + 1, 0, 0, true};
}
// The slot-th segment of the step's runs in their order, every wave for itself; n = 0: there are fewer.
__device__ __forceinline__ ChunkSegment find_segment(const ChunkArgs& a, int slot, int lane) {
  int left = slot;
  for (int base = 0; base < a.runs; base += 64) {
    const int r = base + lane < a.runs ? a.run_rows[base + lane] : -1;
    const int n = r >= 0 && a.row_back[r] == 0 ? a.row_fwd[r] + 1 : 0;
    const int mine = (n + a.seg_rows - 1) / a.seg_rows;
    int upto = mine;                                       // segments of the runs up to this lane's
#pragma unroll
    for (int o = 1; o < 64; o *= 2) {
      const int x = __shfl_up(upto, o, 64);
      if (lane >= o) upto += x;
    }
    const uint64_t m = __builtin_amdgcn_ballot_w64(left < upto);
    if (m != 0) {
      const int at = __builtin_ctzll(m);
      const int seg = left - __builtin_amdgcn_readlane(upto - mine, at), rows = __builtin_amdgcn_readlane(n, at);
      const int run0 = __builtin_amdgcn_readlane(r, at), from = seg * a.seg_rows;
      return {run0, run0 + from, min(rows - from, a.seg_rows), seg, slot, from + a.seg_rows >= rows};
    }
    left -= __builtin_amdgcn_readlane(upto, 63);
  }
  return {0, 0, 0, 0, 0, false};
}

// 64 value channels, from z64 on, of head h of a run or of a segment of one.
template <typename TI, typename TG, int MODE>
__device__ __forceinline__ void chunk_run(const ChunkArgs& a, const ChunkSegment& sg, const int h, const int z64, const int tid) {
  constexpr bool WKV = MODE == kChunkWkv, DELTA = MODE == kChunkDelta;
  const int lane = tid & 63, col = lane & 15, grp = lane >> 4;
  const int t0 = sg.t0, n = sg.n, nc = (n + CT - 1) / CT;
  const int code = a.row_state[sg.run0];
  const int H = a.H, dim = a.dim, vdim = a.vdim;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int role = wave >> 2, w = wave & 3;               // 0 consumers, 1 decays, 2 A and T, 3 wkv's norm and gate

  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  ChunkLds<MODE>& L = *reinterpret_cast<ChunkLds<MODE>*>(smem);
  for (int x = tid; x < 4 * CT * TS; x += chunk_threads(MODE)) (&L.aq[0][0])[x] = 0.f;    // pairs s > t stay zero
  if constexpr (DELTA)
    for (int x = tid; x < 2 * CT * TS; x += chunk_threads(MODE)) {
      (&L.ak[0][0])[x] = 0.f;
      (&L.tt[0][0])[x] = 0.f;
    }

  // Row offsets inside a chunk in bytes (the launcher bounds 16 rows by 2^31); a chunk's first row
  // is a wave-uniform pointer.  Rows past the run's end are read as its last row and left out later.
  auto offsets = [&](uint32_t (&o)[4], int64_t stride, int first, int esz, int c) {
#pragma unroll
    for (int i = 0; i < 4; ++i) o[i] = (uint32_t)min(first + i, n - 1 - c * CT) * (uint32_t)(stride * esz);
  };
  // ---- consumers: 16 value channels, S[16 i + 4 grp + r][column]
  const int vcol = z64 + 16 * w + col;
  const bool vlive = vcol < vdim;
  const bool from_state = code >= 0 && a.pos[sg.run0] > 0;
  const int64_t hsz = (int64_t)dim * vdim;
  f32x4 st[4];
  TI vreg[4];
  uint32_t vo[4];
  const TI* vb = static_cast<const TI*>(a.v) + t0 * a.vs + (int64_t)h * vdim;
  auto fetch_v = [&](int c) {
    if (c * CT + CT > n) offsets(vo, a.vs, 4 * grp, sizeof(TI), c);   // the last, partial chunk
    const TI* base = vb + (int64_t)c * CT * a.vs;
#pragma unroll
    for (int r = 0; r < 4; ++r) vreg[r] = load_at(base, vo[r] + (uint32_t)(min(vcol, vdim - 1) * sizeof(TI)));
  };
  // ---- producers: a lane has four tokens of one key channel
  const int ch = 16 * w + col, chl = min(ch, dim - 1);
  const bool klive = ch < dim;
  const int hq = h / a.rep;
  typedef typename std::conditional<WKV, TI, float>::type TZ;
  TI rq[4], rk[4];
  TZ rz[4];
  TG rb{};
  TI rg[4] = {};                                          // wkv: four channels' gates of one token
  uint32_t qo[4], ko[4], zo[4];
  const TI* qb = static_cast<const TI*>(a.q) + t0 * a.qs + (int64_t)hq * dim;
  const TI* kb = static_cast<const TI*>(a.k) + t0 * a.ks + (int64_t)hq * dim;
  const TZ* zb = static_cast<const TZ*>(a.z) + t0 * a.zs + (int64_t)h * dim;
  const TG* bb = DELTA ? static_cast<const TG*>(a.beta) + t0 * a.bs + h : nullptr;
  const TI* gb = WKV ? static_cast<const TI*>(a.gate) + t0 * a.gs + (int64_t)h * vdim : nullptr;
  auto fetch = [&](int c) {
    if (c * CT + CT > n) {
      offsets(qo, a.qs, 4 * grp, sizeof(TI), c);
      offsets(ko, a.ks, 4 * grp, sizeof(TI), c);
      offsets(zo, a.zs, 4 * grp, sizeof(TZ), c);
    }
    const TI *q = qb + (int64_t)c * CT * a.qs, *k = kb + (int64_t)c * CT * a.ks;
    const TZ* z = zb + (int64_t)c * CT * a.zs;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      rq[i] = load_at(q, qo[i] + (uint32_t)(chl * sizeof(TI)));
      rk[i] = load_at(k, ko[i] + (uint32_t)(chl * sizeof(TI)));
      rz[i] = load_at(z, zo[i] + (uint32_t)(chl * sizeof(TZ)));
    }
    if constexpr (DELTA) rb = load_at(bb + (int64_t)min(c * CT + col, n - 1) * a.bs, 0);
  };
  float4 nw = {}, bonus = {};
  float zbias = 0.f, rate = 0.f;

  if (role == 0) {
    offsets(vo, a.vs, 4 * grp, sizeof(TI), 0);
    const float* rd = a.state + (((int64_t)(code & 1) * a.slots + (code >> 1)) * H + h) * hsz;
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int c = 16 * i + 4 * grp + r;
        st[i][r] = (from_state && vlive && c < dim) ? rd[(int64_t)c * vdim + vcol] : 0.f;
      }
    fetch_v(0);
    if constexpr (!DELTA) {
      const int64_t slots = a.runs + a.T / max(a.seg_rows, 1);
      for (int j = sg.slot - sg.seg; j < sg.slot; ++j) {     // the run's segments before this one
        const float* left = a.seg + ((int64_t)j * H + h) * hsz + vcol;
        const float* kept = a.seg + slots * H * hsz + ((int64_t)j * H + h) * dim;
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int c = 16 * i + 4 * grp + r;
            st[i][r] = fmaf(kept[c], st[i][r], left[(int64_t)c * vdim]);
          }
      }
    }
  } else if (role == 1) {
    offsets(qo, a.qs, 4 * grp, sizeof(TI), 0);
    offsets(ko, a.ks, 4 * grp, sizeof(TI), 0);
    offsets(zo, a.zs, 4 * grp, sizeof(TZ), 0);
    fetch(0);
    zbias = a.zbias[h * dim + chl];
    if constexpr (!WKV) rate = a.rate[h];
  } else if constexpr (WKV) {
    const float *np = a.norm_w + h * NC + 4 * col, *up = a.u + h * NC + 4 * col;
    nw = make_float4(np[0], np[1], np[2], np[3]);
    bonus = make_float4(up[0], up[1], up[2], up[3]);
  }
  __syncthreads();

  // The kinds of wave run loops of their own with the same number of barriers.
  const int turns = nc + (WKV ? 1 : 0);                   // and three turns ahead of them
  if (role == 0) {
    for (int i = 0; i < 3; ++i) __syncthreads();
    // The operands of the next chunk are there a turn ahead: they are read into registers behind the
    // products that use the present ones.
    float4 qa[4], ka[DELTA ? 4 : 1], kh[4], dc[4], aa;
    auto queries = [&](int b) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        qa[i] = ld4(&L.qd[b][col * RS + 16 * i + 4 * grp]);
        if constexpr (DELTA) ka[i] = ld4(&L.kk[b][col * RS + 16 * i + 4 * grp]);
      }
    };
    auto keys = [&](int b) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        kh[i] = ld4(&L.kd[b][(16 * i + col) * TS + 4 * grp]);
        dc[i] = ld4(&L.dec[b][16 * i + 4 * grp]);
      }
      aa = ld4(&L.aq[b][col * TS + 4 * grp]);
    };
    queries(0);
    keys(0);
    for (int it = 0; it < nc; ++it) {
      const int b = it & 3;
      float v[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) v[r] = arrived(vreg[r]);
      fetch_v(min(it + 1, nc - 1));
      if (!vlive || it * CT + CT > n) {
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] = vlive && it * CT + 4 * grp + r < n ? v[r] : 0.f;
      }
      f32x4 o = (f32x4){0.f, 0.f, 0.f, 0.f}, u;
      if constexpr (DELTA) {
        const float4 bt = ld4(&L.beta[b][4 * grp]), ta = ld4(&L.tt[it & 1][col * TS + 4 * grp]);
        f32x4 y = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          y = __builtin_amdgcn_mfma_f32_16x16x4f32(ka[i].x, st[i][0], y, 0, 0, 0);
          o = __builtin_amdgcn_mfma_f32_16x16x4f32(qa[i].x, st[i][0], o, 0, 0, 0);
          y = __builtin_amdgcn_mfma_f32_16x16x4f32(ka[i].y, st[i][1], y, 0, 0, 0);
          o = __builtin_amdgcn_mfma_f32_16x16x4f32(qa[i].y, st[i][1], o, 0, 0, 0);
          y = __builtin_amdgcn_mfma_f32_16x16x4f32(ka[i].z, st[i][2], y, 0, 0, 0);
          o = __builtin_amdgcn_mfma_f32_16x16x4f32(qa[i].z, st[i][2], o, 0, 0, 0);
          y = __builtin_amdgcn_mfma_f32_16x16x4f32(ka[i].w, st[i][3], y, 0, 0, 0);
          o = __builtin_amdgcn_mfma_f32_16x16x4f32(qa[i].w, st[i][3], o, 0, 0, 0);
        }
        const f32x4 x = {bt.x * (v[0] - y[0]), bt.y * (v[1] - y[1]), bt.z * (v[2] - y[2]), bt.w * (v[3] - y[3])};
        u = (f32x4){0.f, 0.f, 0.f, 0.f};
        if (__builtin_amdgcn_ballot_w64(!finite4(x)) == 0ull) {
          u = __builtin_amdgcn_mfma_f32_16x16x4f32(ta.x, x[0], u, 0, 0, 0);
          u = __builtin_amdgcn_mfma_f32_16x16x4f32(ta.y, x[1], u, 0, 0, 0);
          u = __builtin_amdgcn_mfma_f32_16x16x4f32(ta.z, x[2], u, 0, 0, 0);
          u = __builtin_amdgcn_mfma_f32_16x16x4f32(ta.w, x[3], u, 0, 0, 0);
        } else {
          lower_product(L.tt[it & 1], x, col, grp, u);
        }
      } else {
        f32x4 o2 = (f32x4){0.f, 0.f, 0.f, 0.f};           // two independent chains
#pragma unroll
        for (int i = 0; i < 4; i += 2) {
          o = __builtin_amdgcn_mfma_f32_16x16x4f32(qa[i].x, st[i][0], o, 0, 0, 0);
          o2 = __builtin_amdgcn_mfma_f32_16x16x4f32(qa[i + 1].x, st[i + 1][0], o2, 0, 0, 0);
          o = __builtin_amdgcn_mfma_f32_16x16x4f32(qa[i].y, st[i][1], o, 0, 0, 0);
          o2 = __builtin_amdgcn_mfma_f32_16x16x4f32(qa[i + 1].y, st[i + 1][1], o2, 0, 0, 0);
          o = __builtin_amdgcn_mfma_f32_16x16x4f32(qa[i].z, st[i][2], o, 0, 0, 0);
          o2 = __builtin_amdgcn_mfma_f32_16x16x4f32(qa[i + 1].z, st[i + 1][2], o2, 0, 0, 0);
          o = __builtin_amdgcn_mfma_f32_16x16x4f32(qa[i].w, st[i][3], o, 0, 0, 0);
          o2 = __builtin_amdgcn_mfma_f32_16x16x4f32(qa[i + 1].w, st[i + 1][3], o2, 0, 0, 0);
        }
        o += o2;
        u = (f32x4){v[0], v[1], v[2], v[3]};
      }
      queries((it + 1) & 3);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        st[i][0] *= dc[i].x;
        st[i][1] *= dc[i].y;
        st[i][2] *= dc[i].z;
        st[i][3] *= dc[i].w;
      }
#define CHUNK_STATE(r, f)                                                           \
do {                                                                              \
  st[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(kh[0].f, u[r], st[0], 0, 0, 0);    \
  st[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(kh[1].f, u[r], st[1], 0, 0, 0);    \
  st[2] = __builtin_amdgcn_mfma_f32_16x16x4f32(kh[2].f, u[r], st[2], 0, 0, 0);    \
  st[3] = __builtin_amdgcn_mfma_f32_16x16x4f32(kh[3].f, u[r], st[3], 0, 0, 0);    \
} while (0)
      if (__builtin_amdgcn_ballot_w64(!finite4(u)) != 0ull) {
        lower_product(L.aq[b], u, col, grp, o);
      } else {
        o = __builtin_amdgcn_mfma_f32_16x16x4f32(aa.x, u[0], o, 0, 0, 0);
        o = __builtin_amdgcn_mfma_f32_16x16x4f32(aa.y, u[1], o, 0, 0, 0);
        o = __builtin_amdgcn_mfma_f32_16x16x4f32(aa.z, u[2], o, 0, 0, 0);
        o = __builtin_amdgcn_mfma_f32_16x16x4f32(aa.w, u[3], o, 0, 0, 0);
      }
      CHUNK_STATE(0, x);
      CHUNK_STATE(1, y);
      CHUNK_STATE(2, z);
      CHUNK_STATE(3, w);
#undef CHUNK_STATE
      keys((it + 1) & 3);
      if constexpr (WKV) {
#pragma unroll
        for (int r = 0; r < 4; ++r) L.o[it & 1][(4 * grp + r) * RS + 16 * w + col] = o[r];
      } else {
        float* rw = a.raw + ((int64_t)(t0 + it * CT + 4 * grp) * H + h) * vdim + vcol;
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (vlive && it * CT + 4 * grp + r < n) rw[(int64_t)r * H * vdim] = o[r] * a.q_scale;
      }
      __syncthreads();
    }
    if constexpr (WKV) __syncthreads();
  } else if (role == 1) {
    for (int it = -3; it < turns; ++it) {
      float q[4], k[4], d[4], bt = 0.f;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        q[i] = arrived(rq[i]);
        k[i] = arrived(rk[i]);
        d[i] = arrived(rz[i]) + zbias;
      }
      if constexpr (DELTA) bt = arrived(rb);
      fetch(min(it + 4, nc - 1));
      if (const int c = it + 3; c < nc) {                 // decays and their products of chunk c
        const int b = c & 3, e = c & 1;
#pragma unroll
        for (int i = 0; i < 4; ++i) d[i] = WKV ? exp_c(-exp_c(d[i] > 80.f ? 80.f : d[i])) : exp_c(-rate * softplus_c(a.zsign * d[i]));
        if constexpr (DELTA)
          if (w == 0 && grp == 0) L.beta[b][col] = c * CT + col < n ? sigmoid_c(bt) : 0.f;
        if (dim < NC || c * CT + CT > n) {
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const bool ok = klive && c * CT + 4 * grp + i < n;
            q[i] = ok ? q[i] : 0.f;
            k[i] = ok ? k[i] : 0.f;
            d[i] = ok ? d[i] : 1.f;
          }
        }
        float up[4], after[4];                            // products inside the block: up to t, after t
        up[0] = d[0];
        up[1] = up[0] * d[1];
        up[2] = up[1] * d[2];
        up[3] = up[2] * d[3];
        after[3] = 1.f;
        after[2] = d[3];
        after[1] = d[2] * after[2];
        after[0] = d[1] * after[1];
        // the products of the blocks grp ^ 1, grp ^ 2, grp ^ 3 from the lanes that hold them
        const float b1 = __shfl_xor(up[3], 16, 64), b2 = __shfl_xor(up[3], 32, 64), b3 = __shfl_xor(b1, 32, 64);
        const float b23 = b2 * b3;
        const float pre = ((grp & 1) ? b1 : 1.f) * ((grp & 2) ? b23 : 1.f);
        const float post = ((grp & 1) ? 1.f : b1) * ((grp & 2) ? 1.f : b23);
        if (grp == 0) L.dec[b][ch] = up[3] * post;
        L.blk[e][grp * NC + ch] = up[3];
        float4 kd;
        float* kdp = reinterpret_cast<float*>(&kd);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int at = (4 * grp + i) * RS + ch;
          const float ql = WKV ? (i == 0 ? q[0] : q[i] * up[i - 1]) : q[i] * up[i];
          const float kl = k[i] * after[i];
          L.qd[b][at] = ql * pre;
          kdp[i] = kl * post;
          L.q[e][at] = q[i];
          L.k[e][at] = k[i];
          L.a[e][at] = d[i];
          L.ql[e][at] = ql;
          L.kl[e][at] = kl;
          if constexpr (DELTA) {
            const float kb = k[i] * up[i];
            L.kb[e][at] = kb;
            L.kk[b][at] = kb * pre;
          }
        }
        *reinterpret_cast<float4*>(&L.kd[b][ch * TS + 4 * grp]) = kd;
      }
      __syncthreads();
    }
  } else if (role == 2) {
    for (int it = -3; it < turns; ++it) {
      if constexpr (DELTA) {
        const int c = it + 1;
        if (w == 3 && c >= 0 && c < nc && lane < CT) {    // T: column `lane` by forward substitution
          const float* m = L.ak[c & 1];
          const float* bt = L.beta[c & 3];
          float x[CT];
#pragma unroll
          for (int t = 0; t < CT; ++t) {
            float p[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int s4 = 0; s4 < (t + 3) / 4; ++s4) {
              const float4 r = ld4(m + t * TS + 4 * s4);
              if (4 * s4 < t) p[0] += r.x * x[4 * s4];
              if (4 * s4 + 1 < t) p[1] += r.y * x[4 * s4 + 1];
              if (4 * s4 + 2 < t) p[2] += r.z * x[4 * s4 + 2];
              if (4 * s4 + 3 < t) p[3] += r.w * x[4 * s4 + 3];
            }
            x[t] = (t == lane ? 1.f : 0.f) - bt[t] * ((p[0] + p[1]) + (p[2] + p[3]));
            L.tt[c & 1][t * TS + lane] = x[t];
          }
        }
      }
      if (const int c = it + 2; c >= 0 && c < nc) {
        // A of chunk c.  Pairs of blocks `far` apart: one 16 x 16 product of the readers' rows with
        // the writers' rows times the blocks between them, of which those pairs are kept.  The delta
        // rule's keys as readers take the same columns: beside q's rows where they fit (rows 0..7 q,
        // 8..15 k of the last two blocks), else in a product of their own.
        const int b = c & 1;
        auto product = [&](auto far_c, auto rows_c) {     // rows: 0 q, 1 k, 2 both
          constexpr int far = far_c, rows = rows_c;
          const float* src = rows == 1 || (rows == 2 && col >= 8) ? L.kb[DELTA ? b : 0] : L.ql[b];
          const int tr = rows == 2 ? 8 + (col & 7) : col;
          float4 q[4], k[4], g[4], g2[4];
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int at = 16 * i + 4 * grp;
            q[i] = ld4(src + tr * RS + at);
            k[i] = ld4(&L.kl[b][col * RS + at]);
            if constexpr (far > 1) g[i] = ld4(&L.blk[b][min((col >> 2) + 1, 3) * NC + at]);
            if constexpr (far > 2) g2[i] = ld4(&L.blk[b][min((col >> 2) + 2, 3) * NC + at]);
          }
          f32x4 x = (f32x4){0.f, 0.f, 0.f, 0.f}, y = x;
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            if constexpr (far > 1) k[i] = mul4(k[i], g[i]);
            if constexpr (far > 2) k[i] = mul4(k[i], g2[i]);
            x = __builtin_amdgcn_mfma_f32_16x16x4f32(q[i].x, k[i].x, x, 0, 0, 0);
            y = __builtin_amdgcn_mfma_f32_16x16x4f32(q[i].y, k[i].y, y, 0, 0, 0);
            x = __builtin_amdgcn_mfma_f32_16x16x4f32(q[i].z, k[i].z, x, 0, 0, 0);
            y = __builtin_amdgcn_mfma_f32_16x16x4f32(q[i].w, k[i].w, y, 0, 0, 0);
          }
          x += y;
          const int tb = rows == 2 ? 2 + (grp & 1) : grp;  // this lane's block of rows, its column's block
          float* to = rows == 1 || (rows == 2 && grp >= 2) ? L.ak[DELTA ? b : 0] : L.aq[c & 3];
          if (tb - (col >> 2) == far) {
#pragma unroll
            for (int r = 0; r < 4; ++r) to[(4 * tb + r) * TS + col] = x[r];
          }
        };
        constexpr std::integral_constant<int, 0> i0{};
        constexpr std::integral_constant<int, 1> i1{};
        constexpr std::integral_constant<int, 2> i2{};
        constexpr std::integral_constant<int, 3> i3{};
        if constexpr (DELTA) {
          if (w == 0) product(i1, i0);
          else if (w == 1) product(i1, i1);
          else if (w == 2) { product(i2, i2); product(i3, i2); }
        } else {
          if (w == 0) product(i1, i0);
          else if (w == 1) product(i2, i0);
          else if (w == 2) product(i3, i0);
        }
        if (w == (DELTA ? 0 : 3)) {
          // pairs inside a block: sixteen lanes per block, four key channels each
          float4 q[4], k[4], d[4];
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int at = (4 * grp + i) * RS + 4 * col;
            q[i] = ld4(&L.q[b][at]);
            k[i] = ld4(&L.k[b][at]);
            d[i] = ld4(&L.a[b][at]);
          }
          float acc[10], ack[6];                          // (0,0) (1,0) (1,1) (2,0) .. (3,3); without s = t
          if constexpr (WKV) {
            acc[1] = dot4(q[1], k[0]);
            acc[4] = dot4(q[2], k[1]);
            acc[8] = dot4(q[3], k[2]);
            const float4 e1 = mul4(d[1], k[0]);
            acc[3] = dot4(q[2], e1);
            acc[7] = dot4(q[3], mul4(d[2], k[1]));
            acc[6] = dot4(q[3], mul4(d[2], e1));
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[i * (i + 3) / 2] = dot4(mul4(q[i], bonus), k[i]);
          } else {
            const float4 e10 = mul4(d[1], k[0]), e21 = mul4(d[2], k[1]), e32 = mul4(d[3], k[2]);
            const float4 e20 = mul4(d[2], e10), e31 = mul4(d[3], e21), e30 = mul4(d[3], e20);
            acc[1] = dot4(q[1], e10);
            acc[3] = dot4(q[2], e20);
            acc[4] = dot4(q[2], e21);
            acc[6] = dot4(q[3], e30);
            acc[7] = dot4(q[3], e31);
            acc[8] = dot4(q[3], e32);
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[i * (i + 3) / 2] = dot4(q[i], k[i]);
            if constexpr (DELTA) {
              ack[0] = dot4(k[1], e10);
              ack[1] = dot4(k[2], e20);
              ack[2] = dot4(k[2], e21);
              ack[3] = dot4(k[3], e30);
              ack[4] = dot4(k[3], e31);
              ack[5] = dot4(k[3], e32);
            }
          }
          float* ao = &L.aq[c & 3][4 * grp * TS + 4 * grp];
#pragma unroll
          for (int i = 0; i < 10; ++i) acc[i] = ror_add(acc[i]);
          if (col == 0) {
            ao[0] = acc[0];
            *reinterpret_cast<float2*>(ao + TS) = make_float2(acc[1], acc[2]);
            *reinterpret_cast<float2*>(ao + 2 * TS) = make_float2(acc[3], acc[4]);
            ao[2 * TS + 2] = acc[5];
            *reinterpret_cast<float4*>(ao + 3 * TS) = make_float4(acc[6], acc[7], acc[8], acc[9]);
          }
          if constexpr (DELTA) {
            float* ko4 = &L.ak[b][4 * grp * TS + 4 * grp];
#pragma unroll
            for (int i = 0; i < 6; ++i) ack[i] = ror_add(ack[i]);
            if (col == 0) {
              ko4[TS] = ack[0];
              *reinterpret_cast<float2*>(ko4 + 2 * TS) = make_float2(ack[1], ack[2]);
              *reinterpret_cast<float2*>(ko4 + 3 * TS) = make_float2(ack[3], ack[4]);
              ko4[3 * TS + 2] = ack[5];
            }
          }
        }
      }
      __syncthreads();
    }
  } else if constexpr (WKV) {
    for (int it = -3; it < turns; ++it) {
      float g[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) g[e] = arrived(rg[e]);
      const int tn = min(max(it, 0) * CT + 4 * w + grp, n - 1);  // the gates of chunk it, for the next turn
      const TI* gr = gb + tn * a.gs + 4 * col;
#pragma unroll
      for (int e = 0; e < 4; ++e) rg[e] = load_at(gr + e, 0);
      if (it >= 1) {                                    // norm and gate of chunk it - 1
        const int tl = 4 * w + grp, t = (it - 1) * CT + tl;
        const float4 o4 = ld4(&L.o[(it - 1) & 1][tl * RS + 4 * col]);
        const float inv = 1.0f / sqrtf(ror_add(dot4(o4, o4)) / (float)NC + a.eps);
        const float y[4] = {o4.x * nw.x, o4.y * nw.y, o4.z * nw.z, o4.w * nw.w};
        TI* op = static_cast<TI*>(a.out) + ((int64_t)(t0 + t) * H + h) * NC + 4 * col;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float z = y[e] * inv * silu_c(g[e]);
          if (t < n) stf(op + e, z);
        }
      }
      __syncthreads();
    }
  }

  if (role == 0 && code >= 0 && vlive && sg.last) {
    float* wr = a.state + (((int64_t)(1 - (code & 1)) * a.slots + (code >> 1)) * H + h) * hsz;
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int c = 16 * i + 4 * grp + r;
        if (c < dim) wr[(int64_t)c * vdim + vcol] = st[i][r];
      }
  }
}

// A workgroup per entry of the list, head and 64 value channels.
template <typename TI, typename TG, int MODE>
__global__ __launch_bounds__(chunk_threads(MODE)) void chunk_recurrence_kernel(const ChunkArgs a) {
  const int t0 = a.run_rows[blockIdx.x];
  if (t0 >= 0 && a.row_back[t0] == 0) chunk_run<TI, TG, MODE>(a, whole_run(a, t0), blockIdx.y, blockIdx.z * 64, threadIdx.x);
}

// Two and four neighbouring entries in flight, and their values where they are needed (see `arrived`).
__device__ __forceinline__ void raw4(const float* base, uint32_t bytes, uint4& x) { x = load_at(reinterpret_cast<const uint4*>(base), bytes); }
__device__ __forceinline__ void raw4(const bf16_t* base, uint32_t bytes, uint2& x) { x = load_at(reinterpret_cast<const uint2*>(base), bytes); }
__device__ __forceinline__ void raw2(const float* base, uint32_t bytes, uint2& x) { x = load_at(reinterpret_cast<const uint2*>(base), bytes); }
__device__ __forceinline__ void raw2(const bf16_t* base, uint32_t bytes, uint32_t& x) { x = load_at(reinterpret_cast<const uint32_t*>(base), bytes); }
__device__ __forceinline__ void arrived2(uint2 x, float* f) {
  asm volatile("" : "+v"(x.x), "+v"(x.y));
  f[0] = __uint_as_float(x.x);
  f[1] = __uint_as_float(x.y);
}
__device__ __forceinline__ void arrived2(uint32_t x, float* f) {
  asm volatile("" : "+v"(x));
  f[0] = __uint_as_float(x << 16);
  f[1] = __uint_as_float(x & 0xffff0000u);
}
__device__ __forceinline__ void arrived4(uint4 x, float* f) {
  asm volatile("" : "+v"(x.x), "+v"(x.y), "+v"(x.z), "+v"(x.w));
  f[0] = __uint_as_float(x.x);
  f[1] = __uint_as_float(x.y);
  f[2] = __uint_as_float(x.z);
  f[3] = __uint_as_float(x.w);
}
__device__ __forceinline__ void arrived4(uint2 x, float* f) {
  asm volatile("" : "+v"(x.x), "+v"(x.y));
  f[0] = __uint_as_float(x.x << 16);
  f[1] = __uint_as_float(x.x & 0xffff0000u);
  f[2] = __uint_as_float(x.y << 16);
  f[3] = __uint_as_float(x.y & 0xffff0000u);
}

// What a segment's rows leave of a state of zeros, and the products of its decays: for every segment but a run's last,
// one workgroup per segment, head, 32 key and 64 value channels.  A wave has an eighth (a sixteenth) of the rows and goes through them
// from the last chunk to the first, the keys times all decays behind them: nothing is rescaled, and the lane that makes
// such a product (four tokens of two key channels) has it as the MFMA operand.  No LDS but to add the waves' parts up.
constexpr int kSegKeys = 32;
template <typename TI, int MODE, int kSegWaves>
__global__ __launch_bounds__(64 * kSegWaves, 4) void chunk_segment_kernel(const ChunkArgs a) {
  constexpr bool WKV = MODE == kChunkWkv;
  typedef typename std::conditional<WKV, TI, float>::type TZ;
  typedef typename std::conditional<sizeof(TI) == 2, uint2, uint4>::type RV;
  typedef typename std::conditional<sizeof(TI) == 2, uint32_t, uint2>::type RK;
  typedef typename std::conditional<sizeof(TZ) == 2, uint32_t, uint2>::type RZ;
  const int tid = threadIdx.x, lane = tid & 63, col = lane & 15, grp = lane >> 4;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const ChunkSegment sg = find_segment(a, blockIdx.z, lane);
  if (sg.n == 0 || sg.last) return;
  __shared__ __attribute__((aligned(16))) float sums[kSegWaves / 2][kSegKeys * NC];
  const int h = blockIdx.x, z64 = (blockIdx.y >> 1) * 64, c0 = (blockIdx.y & 1) * kSegKeys, H = a.H, vdim = a.vdim, hq = h / a.rep;
  const int rows = a.seg_rows / kSegWaves;
  // the wave's last chunk; a lane's tokens by their offsets in bytes
  const int64_t at = sg.t0 + (w + 1) * rows - CT;
  const TI* kb = static_cast<const TI*>(a.k) + at * a.ks + (int64_t)hq * NC + c0;
  const TI* vb = static_cast<const TI*>(a.v) + at * a.vs + (int64_t)h * vdim + z64;
  const TZ* zb = static_cast<const TZ*>(a.z) + at * a.zs + (int64_t)h * NC + c0;
  uint32_t ko[4], vo[4], zo[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    ko[i] = (uint32_t)((4 * grp + i) * a.ks + 2 * col) * (uint32_t)sizeof(TI);
    vo[i] = (uint32_t)((4 * grp + i) * a.vs + 4 * col) * (uint32_t)sizeof(TI);
    zo[i] = (uint32_t)((4 * grp + i) * a.zs + 2 * col) * (uint32_t)sizeof(TZ);
  }
  RK kr[4];
  RV vr[4];
  RZ zr[4];
  auto fetch = [&]() {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      raw2(zb, zo[i], zr[i]);
      raw2(kb, ko[i], kr[i]);
      raw4(vb, vo[i], vr[i]);
    }
    kb -= CT * a.ks;
    vb -= CT * a.vs;
    zb -= CT * a.zs;
  };
  fetch();
  const float bias[2] = {a.zbias[h * NC + c0 + 2 * col], a.zbias[h * NC + c0 + 2 * col + 1]};
  const float rate = WKV ? 0.f : a.rate[h];
  f32x4 st[2][4];                                            // [key channel % 2][value channel % 4]
#pragma unroll
  for (int x = 0; x < 2; ++x)
#pragma unroll
    for (int y = 0; y < 4; ++y) st[x][y] = (f32x4){0.f, 0.f, 0.f, 0.f};
  float behind[2] = {1.f, 1.f};                              // products of the decays behind the chunk
  for (int c = rows / CT; c > 0; --c) {
    float k[4][2], d[4][2], v[4][4];                         // [token][channel % 2 or 4]
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      arrived2(zr[i], d[i]);
      arrived2(kr[i], k[i]);
      arrived4(vr[i], v[i]);
    }
    if (c > 1) fetch();
#pragma unroll
    for (int x = 0; x < 2; ++x) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float z = d[i][x] + bias[x];
        d[i][x] = WKV ? exp_c(-exp_c(z > 80.f ? 80.f : z)) : exp_c(-rate * softplus_c(a.zsign * z));
      }
      const float a2 = d[3][x], a1 = d[2][x] * a2, a0 = d[1][x] * a1, up = d[0][x] * a0;
      const float b1 = __shfl_xor(up, 16, 64), b2 = __shfl_xor(up, 32, 64), b3 = __shfl_xor(b1, 32, 64);
      const float b23 = b2 * b3;
      const float post = ((grp & 1) ? 1.f : b1) * ((grp & 2) ? 1.f : b23) * behind[x];
      behind[x] *= (up * b1) * b23;
      k[0][x] *= a0 * post;
      k[1][x] *= a1 * post;
      k[2][x] *= a2 * post;
      k[3][x] *= post;
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int y = 0; y < 4; ++y) st[x][y] = __builtin_amdgcn_mfma_f32_16x16x4f32(k[i][x], v[i][y], st[x][y], 0, 0, 0);
    }
  }
  // a wave's part times the decays of those behind it
  float* decays = &sums[0][0];
  if (grp == 0) *reinterpret_cast<float2*>(decays + w * kSegKeys + 2 * col) = make_float2(behind[0], behind[1]);
  __syncthreads();
  if (blockIdx.y < 2 && tid < kSegKeys) {
    float f = decays[tid];
#pragma unroll
    for (int u = 1; u < kSegWaves; ++u) f *= decays[u * kSegKeys + tid];
    a.seg[(a.runs + a.T / a.seg_rows) * (int64_t)(H * NC) * vdim + ((int64_t)sg.slot * H + h) * NC + c0 + tid] = f;
  }
  float4 f[2];                                               // of channels 8 grp ..
  f[0] = f[1] = make_float4(1.f, 1.f, 1.f, 1.f);
  for (int u = w + 1; u < kSegWaves; ++u)
#pragma unroll
    for (int r = 0; r < 2; ++r) f[r] = mul4(f[r], ld4(decays + u * kSegKeys + 8 * grp + 4 * r));
#pragma unroll
  for (int r = 0; r < 2; ++r)
#pragma unroll
    for (int y = 0; y < 4; ++y) {
      st[0][y][2 * r] *= f[r].x;
      st[1][y][2 * r] *= f[r].y;
      st[0][y][2 * r + 1] *= f[r].z;
      st[1][y][2 * r + 1] *= f[r].w;
    }
  constexpr int half = kSegWaves / 2;
  auto place = [&](int x, int r) { return &sums[w & (half - 1)][(2 * (4 * grp + r) + x) * NC + 4 * col]; };
#pragma unroll
  for (int part = 0; part < 2; ++part) {                     // the later half's parts to the earlier half's, those out
    __syncthreads();
    if ((w >= half) == (part == 0)) {
#pragma unroll
      for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int r = 0; r < 4; ++r) st4(place(x, r), make_float4(st[x][0][r], st[x][1][r], st[x][2][r], st[x][3][r]));
    }
    __syncthreads();
    if (part == 0 && w < half) {
#pragma unroll
      for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float4 o = ld4(place(x, r));
          st[x][0][r] += o.x;
          st[x][1][r] += o.y;
          st[x][2][r] += o.z;
          st[x][3][r] += o.w;
        }
    }
  }
  float* out = a.seg + (((int64_t)sg.slot * H + h) * NC + c0) * vdim + z64;
#pragma unroll
  for (int i = 0; i < kSegKeys * NC / (128 * kSegWaves); ++i) {
    const int e = (i * 64 * kSegWaves + tid) * 2;
    float2 y = make_float2(0.f, 0.f);
#pragma unroll
    for (int u = 0; u < half; u += 2) {
      const float2 p = *reinterpret_cast<const float2*>(&sums[u][e]), q = *reinterpret_cast<const float2*>(&sums[u + 1][e]);
      y.x += p.x + q.x;
      y.y += p.y + q.y;
    }
    *reinterpret_cast<float2*>(out + (int64_t)(e / NC) * vdim + e % NC) = y;
  }
}

// A workgroup per segment, head and 64 value channels, behind chunk_segment_kernel.
template <typename TI, typename TG, int MODE>
__global__ __launch_bounds__(chunk_threads(MODE)) void chunk_recurrence_segments_kernel(const ChunkArgs a) {
  const ChunkSegment sg = find_segment(a, blockIdx.z, threadIdx.x & 63);
  if (sg.n > 0) chunk_run<TI, TG, MODE>(a, sg, blockIdx.x, blockIdx.y * 64, threadIdx.x);
}

// Workgroups, one to a CU at most, that share the runs of min_run rows or more, which every wave counts for
// itself: one for every run that the step has room for costs 16 us where there is none (64 runs of 16, wkv).
template <typename TI, typename TG, int MODE>
__global__ __launch_bounds__(chunk_threads(MODE)) void chunk_recurrence_share_kernel(const ChunkArgs a) {
  const int lane = threadIdx.x & 63, cols = (a.vdim + 63) >> 6, per = a.H * cols;
#pragma unroll 1
  for (int item = blockIdx.x;; item += gridDim.x) {
    int left = item / per, t0 = -1;
    const int part = item - left * per, z = part / a.H;
    for (int base = 0; base < a.runs; base += 64) {
      const int r = base + lane < a.runs ? a.run_rows[base + lane] : -1;
      const bool fits = r >= 0 && a.row_back[r] == 0 && a.row_fwd[r] + 1 >= a.min_run;
      uint64_t m = __builtin_amdgcn_ballot_w64(fits);
      const int c = __builtin_popcountll(m);
      if (left < c) {
        for (; left > 0; --left) m &= m - 1;
        t0 = __builtin_amdgcn_readfirstlane(__shfl(r, __builtin_ctzll(m), 64));
        break;
      }
      left -= c;
    }
    if (t0 < 0) return;
    // The last barrier of a run lies behind every wave's last read of LDS: the next run's first writes need no
    // other.
    // thread and arguments are taken anew for every run: what the compiler derives from them would stay in
    // registers over the loop, 55 of them spilled
    typedef const __attribute__((address_space(4))) ChunkArgs const_args;
    const_args* p = (const_args*)__builtin_amdgcn_kernarg_segment_ptr();
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid), "+s"(p));
    chunk_run<TI, TG, MODE>(*(const ChunkArgs*)p, whole_run(*(const ChunkArgs*)p, t0), part - z * a.H, z * 64, tid);
  }
}

// ------------------------------------------------------------------ launcher
// A workgroup costs some 8 us before its first chunk is out and 1.6 - 2.3 us a chunk, one to a CU; the
// token-by-token kernels some 6 us and 0.2 (64 runs) - 2.6 us a token, many to a CU.  Times below are of whole
// steps, 32 heads of 64 x 128 (wkv: 64 of 64 x 64), chunks against tokens.
// Two workgroups to a CU or fewer: everything in chunks from 8 rows a run on (one run of 8: gla 14 us against 25,
// delta 14 against 28, wkv 8 against 24).
// More: a step's runs, decode rows beside prompts as a rule, are shared by their length (64 decode rows beside
// a prompt of 200: gla 59 us, wkv 52, tokens alone 123 and 515), from 24 rows where the step has room for no
// more than 2,048 workgroups of such runs, delta rule 512 (16 runs of 24: gla 47 against 74, wkv 40 against 73,
// delta 55 against 46).  Beyond that the CUs' rounds add up: from 48 for wkv (64 runs of 41: 180 against 162, of
// 64: 210 against 247), 40 for gla (205 against 201, of 64: 235 against 345), 24 with up to 64 value channels
// (64 runs of 24: 83 against 98), 80 for the delta rule (64 runs of 64: 282 against 249, of 96: 358 against 387).
int chunk_min_run(int mode, int T, const ChunkArgs& a) {
  constexpr int kNever = INT32_MAX;
  if (a.run_rows == nullptr || a.dim > NC || (mode == kChunkWkv && (a.dim != NC || a.vdim != NC))) return kNever;
  for (int64_t st : {a.qs, a.ks, a.vs, a.zs})             // a chunk's rows in 32-bit byte offsets
    if (st < 0 || st >= (1ll << 24)) return kNever;
  const int64_t per = (int64_t)a.H * ((a.vdim + 63) / 64);
  if (a.runs * per <= 512 && T >= 8 * a.runs) return 1;
  const int few = 24, many = mode == kChunkWkv ? 48 : mode == kChunkDelta ? 80 : a.vdim > 64 ? 40 : 24;
  const int from = std::min(a.runs, T / few) * per <= (mode == kChunkDelta ? 512 : 2048) ? few : many;
  return T - a.runs + 1 >= from ? from : kNever;          // no run can be longer than that
}

// Segments instead of whole runs where they leave fewer or shorter rounds of one workgroup a CU, by the times of
// the kernels below (us): a workgroup's start and end and its chunks, as many rounds as workgroups ask for; the same of
// chunk_segment_kernel, whose workgroups of eight waves stand two to a CU.  Runs are taken as equally long, the
// case that gains least.  Two runs of 2,048 tokens in bf16, whole -> in segments: wkv, 64 heads 204 -> 145 us, 32
// heads 194 -> 89; gla, 16 heads of 128 218 -> 112; one run of 2,048, 64 heads, 190 -> 81.  The delta rule's decays are
// matrices: its runs stay whole.
int chunk_seg_rows(int mode, bool in_f32, int T, const ChunkArgs& a) {
  if (mode == kChunkDelta || chunk_min_run(mode, T, a) != 1 || a.dim != NC || a.vdim % 64 != 0) return 0;
  const uintptr_t wide = in_f32 ? 16 : 8, zwide = mode == kChunkWkv && !in_f32 ? 4 : 8;     // loads of four, of two
  for (const void* p : {a.k, a.v})
    if (reinterpret_cast<uintptr_t>(p) % wide != 0) return 0;
  if (reinterpret_cast<uintptr_t>(a.z) % zwide != 0) return 0;
  for (int64_t st : {a.ks, a.vs, a.zs})
    if (st % 4 != 0) return 0;
  const int64_t per = (int64_t)a.H * (a.vdim / 64);
  const int c = (T + CT * a.runs - 1) / (CT * a.runs);    // chunks of a run
  const double turn = mode == kChunkWkv ? 1.65 : 1.85;
  auto rounds = [](int64_t wgs, int at_once) { return (double)((wgs + at_once - 1) / at_once); };
  double best = 0.9 * rounds(a.runs * per, 256) * (6 + turn * c) - 5;
  int rows = 0;
  for (int s = 2; s <= 16; ++s) {
    int cs = ((c + s - 1) / s + 7) / 8 * 8;               // chunks of a segment
    if (cs >= 64) cs = (cs + 15) / 16 * 16;
    const int64_t n = (c + cs - 1) / cs, w1 = a.runs * (n - 1) * per * (NC / kSegKeys);
    const double t = 6 + (cs >= 64 ? rounds(w1, 256) * (8 + 3.3 * cs / 16) : rounds(w1, 512) * (6 + 2.0 * cs / 8)) +
                     rounds(a.runs * n * per, 256) * (6 + turn * cs);
    if (n > 1 && t < best) {
      best = t;
      rows = cs * CT;
    }
  }
  return rows;
}
int64_t chunk_seg_floats(int T, const ChunkArgs& a) {
  return (a.runs + (int64_t)T / a.seg_rows) * a.H * a.dim * (a.vdim + 1);
}

template <typename TI, typename TG, int MODE>
static void launch_chunk_one(int T, const ChunkArgs& a, hipStream_t s) {
  static bool attr = false;
  if (!attr) {          // dynamic LDS above 64 KB has to be allowed per kernel, once
    for (auto* k : {&chunk_recurrence_kernel<TI, TG, MODE>, &chunk_recurrence_share_kernel<TI, TG, MODE>})
      (void)hipFuncSetAttribute(reinterpret_cast<const void*>(k), hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
    attr = true;
  }
  static_assert(sizeof(ChunkLds<MODE>) <= 160 * 1024, "LDS of a CU");
  const int cols = (a.vdim + 63) / 64;
  if constexpr (MODE != kChunkDelta)
    if (a.seg != nullptr) {
      static bool seg_attr = false;
      if (!seg_attr) {
        (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&chunk_recurrence_segments_kernel<TI, TG, MODE>),
                                  hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
        seg_attr = true;
      }
      const dim3 grid(a.H, cols, a.runs + T / a.seg_rows);
      const dim3 parts(a.H, cols * (NC / kSegKeys), grid.z);
      if (a.seg_rows >= 64 * CT) hipLaunchKernelGGL((chunk_segment_kernel<TI, MODE, 16>), parts, dim3(1024), 0, s, a);
      else hipLaunchKernelGGL((chunk_segment_kernel<TI, MODE, 8>), parts, dim3(512), 0, s, a);
      hipLaunchKernelGGL((chunk_recurrence_segments_kernel<TI, TG, MODE>), grid, dim3(chunk_threads(MODE)),
                         sizeof(ChunkLds<MODE>), s, a);
      return;
    }
  if (a.min_run <= 1)
    hipLaunchKernelGGL((chunk_recurrence_kernel<TI, TG, MODE>), dim3(a.runs, a.H, cols), dim3(chunk_threads(MODE)),
                       sizeof(ChunkLds<MODE>), s, a);
  else                        // no more long runs than rows allow
    hipLaunchKernelGGL((chunk_recurrence_share_kernel<TI, TG, MODE>),
                       dim3((unsigned)std::min<int64_t>((int64_t)std::min(a.runs, T / a.min_run) * a.H * cols, 256)),
                       dim3(chunk_threads(MODE)), sizeof(ChunkLds<MODE>), s, a);
}

void launch_chunk(int mode, bool in_f32, bool act_f32, int T, const ChunkArgs& a, hipStream_t s) {
  if (a.runs == 0) return;
  if (mode == kChunkWkv) {
    if (in_f32) launch_chunk_one<float, float, kChunkWkv>(T, a, s);
    else launch_chunk_one<bf16_t, bf16_t, kChunkWkv>(T, a, s);
  } else if (mode == kChunkGla) {
    if (in_f32) launch_chunk_one<float, float, kChunkGla>(T, a, s);
    else launch_chunk_one<bf16_t, float, kChunkGla>(T, a, s);
  } else if (in_f32) {
    if (act_f32) launch_chunk_one<float, float, kChunkDelta>(T, a, s);
    else launch_chunk_one<float, bf16_t, kChunkDelta>(T, a, s);
  } else {
    if (act_f32) launch_chunk_one<bf16_t, float, kChunkDelta>(T, a, s);
    else launch_chunk_one<bf16_t, bf16_t, kChunkDelta>(T, a, s);
  }
}

}  // namespace rfqmix
