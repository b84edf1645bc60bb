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
// What bounds it: the vector instructions of the waves that share a SIMD, 60 - 70 % of its cycles, and their order inside
// a chunk.  (fp32 MFMA 16x16x4 hold a SIMD's vector unit for their 32 clocks, other waves' instructions as well: with the
// state's products in it the decay waves stood for as long as they took, 2.3 us a chunk of the delta rule.)  The state's
// products, 48 of 56 a wave, therefore go to the matrix cores in bf16: an fp32 operand is the exact sum of three bf16, six
// products of them leave out at most 2^-24 of each (split3).  Operands at the ends of bf16's range have ways of their own
// (kUp, kSplitLeast, odd_split), which cost 1 us of wkv's 100.  Those inside a chunk stay in fp32 MFMA: pairs of blocks on
// tiles of 4x4x1, whose sixteen side by side take 64 channels of one pair in 32 clocks (16x16x4, which made all pairs of a
// distance and sixteen more each in 512: 4 - 5 % more a pass).  Errors against 64 bits: state of the delta rule 6.3e-8 for
// 6.4e-8 in fp32 products, outputs of gla in fp32 5.7e-7 and of wkv 2.0e-7, the same.
// One workgroup per (run, head, 64 or 128 value channels): four consumer waves hold 64 x 16 of the state, or twice that, in
// accumulators, which are MFMA operands as they lie (a lane holds channels 16 i + 4 grp + r of its column); the other
// waves work ahead: decays, their products and parts for chunk c + 3, A for chunk c + 2, T for chunk c + 1, wkv's norm
// and gate for chunk c - 1; one barrier per chunk.  The state never leaves the registers.  A chunk takes 2.1 us with 64
// channels (delta; gla 1.65, wkv 1.45) and 2.7 with 128 (gla 2.0), for which the other waves' work is done once.
// Measured, two runs of 2,048 tokens in bf16, all kernels of the recurrence: delta rule with 32 heads of 64 x 128 301 ->
// 171 us, wkv with 64 heads of 64 x 64 203 -> 128; gla in fp32, five ragged runs of up to 1,031, 32 heads, 121 -> 82.
//
// A run's chain is cut where workgroups leave CUs idle (chunk_seg_cap, segment_rows).  Without the delta rule
// chunk_segment_kernel makes what every segment's rows leave of a state of zeros and the products of its decays, all
// segments at once, and a segment's workgroup begins from the state of before the run carried through those in front of
// it.  What bounds the first kernel: exponentials (22 instructions a decay, 38 of gla) and the way to its first rows and
// out, 10 us of a workgroup.  The delta rule's first kernel makes matrices of 64 x 64 in place of the products
// (chunk_delta_first_kernel).  One run of 4,096, whole runs in fp32 products before, all kernels of a layer's pass: delta, 32
// heads, 668 -> 295 us, gla in fp32 449 -> 182, wkv, 64 heads, 425 -> 182.
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "common.h"
#include "mix_common.h"
#include "mix_chunk.h"
#include "mix_split.h"

namespace rfqmix {

using rfq::f32x4;

namespace {
constexpr int CT = kChunkRows;          // tokens per chunk
constexpr int NC = kChunkDim;           // key channels (those past dim are zeros)
constexpr int RS = NC + 4;              // floats per token row in LDS
constexpr int TS = CT + 4;              // floats per row of a 16 x 16 tile
constexpr int PS = NC + 8;              // bf16 per token row of a part of Qd or Kk, per channel row of Kd^T's parts
constexpr float kTurnMost = 1.001f;     // see chunk_delta_later_kernel
// Operands of products of parts that bf16's range would cut (kSplitLeast).  Qd and Kk, which decays make as small as they
// please, are split times kUp, and products with them come out that much larger.  Kd, u and the state are sums of their own
// along 16 or 64 entries: where all of these are too small, the products are in fp32, of Kd's parts split times kUpKd.
constexpr float kUp = 0x1p32f, kDown = 0x1p-32f, kUpKd = 0x1p64f, kDownKd = 0x1p-64f;
// What a column of the state all of whose entries are below kSplitLeast cannot make with four rows of Qd (each entry
// below kSplitMost).
constexpr float kReadLeast = 0x1p-28f;
constexpr uint32_t kOddLarge = 1, kOddSmall = 2;

// four consumers, four waves for the decays, four for A (and T), wkv: four for norm and gate
constexpr int chunk_threads(int mode) { return mode == kChunkWkv ? 1024 : 768; }

__device__ __forceinline__ float ror_add(float v) {   // sum over the 16 lanes of a row
  v += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x128, 0xf, 0xf, true));
  v += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x124, 0xf, 0xf, true));
  v += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x122, 0xf, 0xf, true));
  v += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x121, 0xf, 0xf, true));
  return v;
}
// Sixteen tiles of 4x4 added up: lane 16 i + j (and those 4, 8, 12 further) gets entry (i, j).
__device__ __forceinline__ float tiles_sum(const f32x4& x) {
  auto swap32 = [](float p, float q) {                    // lanes below 32: p's two halves, above: q's
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(p), __float_as_uint(q), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
  };
  const float e = swap32(x[0], x[2]), o = swap32(x[1], x[3]);
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(e), __float_as_uint(o), false, false);
  float v = __uint_as_float(r[0]) + __uint_as_float(r[1]);
  v += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x128, 0xf, 0xf, true));
  v += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x124, 0xf, 0xf, true));
  return v;
}
// What a chunk's producers leave in LDS.
template <int MODE>
struct ChunkLds {
  static constexpr bool DELTA = MODE == kChunkDelta;
  // What is written in small pieces comes first: its places are constants of LDS instructions, up to 64 KB.
  float aq[4][CT * TS];
  float ak[2][DELTA ? CT * TS : 4];
  float tt[2][DELTA ? CT * TS : 4];
  float dec[4][NC];
  float beta[4][CT];
  uint32_t odd[4][4];                   // of each wave: operands that are split otherwise (kOddLarge: odd_split, without
                                        // kUp; kOddSmall: Kd times kUpKd)
  float blk[2][4 * NC];                 // product of a block's decays
  float ql[2][CT * RS], kl[2][CT * RS];                   // operands of A: times the block's products up to / after,
  float kb[2][DELTA ? CT * RS : 4];
  float q[2][CT * RS], k[2][CT * RS], a[2][CT * RS];      // raw
  // four chunks in flight between producers and consumers; parts as split3 makes them
  uint16_t qd[4][3][CT * PS];           // [part][token][operand_at(channel)]
  uint16_t kk[DELTA ? 4 : 1][3][DELTA ? CT * PS : 8];
  uint16_t kd[4][NC * PS];              // Kd^T: [channel][four tokens: two parts of four, first and third again]
  float o[2][MODE == kChunkWkv ? CT * RS : 4];
};

// split3 cut instead of rounded: for values that are added up in fp32 (kSplitMost); infinities and NaN are h alone.
__device__ __forceinline__ Split2 odd_split(float a, float b) {
  uint32_t p[3][2];
  float f[2] = {a, b};
#pragma unroll
  for (int e = 0; e < 2; ++e) {
    const uint32_t all = __float_as_uint(f[e]);
    const bool whole = (all & 0x7f800000u) != 0x7f800000u;
    p[0][e] = all >> 16 | (!whole && (all & 0xffffu) != 0 ? 1u : 0u);       // a NaN stays one
    const float r = f[e] - __uint_as_float(all & 0xffff0000u);
    p[1][e] = whole ? __float_as_uint(r) >> 16 : 0;
    p[2][e] = whole ? __float_as_uint(r - __uint_as_float(__float_as_uint(r) & 0xffff0000u)) >> 16 : 0;
  }
  return {p[0][0] | p[0][1] << 16, p[1][0] | p[1][1] << 16, p[2][0] | p[2][1] << 16};
}
// Where a row of an operand's parts holds channel c: a lane's eight of a 16x16x32 product are channels 4 grp + r of two
// neighbouring tiles of sixteen, as the accumulators of the state hold them.
__device__ __forceinline__ int operand_at(int c) { return (c & 32) | (c & 12) << 1 | (c & 16) >> 2 | (c & 3); }
__device__ __forceinline__ uint4 ld8(const uint16_t* p) { return *reinterpret_cast<const uint4*>(p); }
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
  return (fabsf(x[0]) + fabsf(x[1])) + (fabsf(x[2]) + fabsf(x[3])) < __builtin_huge_valf();
}

// Whether the sixteen lanes' columns that a wave's lanes 16 grp + col hold in fours are too small for products of parts.
__device__ __forceinline__ bool small_column(float most) {
  most = fmaxf(most, __shfl_xor(most, 16, 64));
  most = fmaxf(most, __shfl_xor(most, 32, 64));
  return most > 0.f && most < kSplitLeast;
}
// lo <= x < hi, of numbers that are not negative
__device__ __forceinline__ bool within(float x, float lo, float hi) {
  return __float_as_uint(x) - __float_as_uint(lo) < __float_as_uint(hi) - __float_as_uint(lo);
}
__device__ __forceinline__ float sum_of_sizes(const f32x4& x) { return (fabsf(x[0]) + fabsf(x[1])) + (fabsf(x[2]) + fabsf(x[3])); }
__device__ __forceinline__ float largest(const f32x4& x) {
  return fmaxf(fmaxf(fabsf(x[0]), fabsf(x[1])), fmaxf(fabsf(x[2]), fabsf(x[3])));
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
  int rows;                             // of the step's segments but a run's last
};
__device__ __forceinline__ ChunkSegment whole_run(const ChunkArgs& a, int t0) {
  return {t0, t0, a.row_fwd[t0] + 1, 0, 0, true, 0};
}

// How long the step's segments are: only the device knows its runs (64 at most).  Lane l tries the longest run in l + 1
// equal parts (of whole chunks, a.unit rows where the first kernel shares a segment over its waves); of those that make no
// more than a.cap segments (workgroups of one of the delta rule's kernels) the one takes over that the times below (us, as
// measured) say is done first.  The same for every wave of both kernels.  Where only one of them is launched runs stay
// whole: entries without a run leave a.cap room that nobody may take then.
template <int MODE, int NV>
__device__ __forceinline__ int segment_rows(const ChunkArgs& a, int n, int lane) {
  constexpr bool DELTA = MODE == kChunkDelta;
  int longest = n;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) longest = max(longest, __shfl_xor(longest, o, 64));
  const int rows = (int)((uint32_t)(longest + lane) / (uint32_t)(lane + 1) + a.unit - 1) / a.unit * a.unit;
  int all = 0, cut = 0, runs = 0, most = 0;                  // segments, runs of more than one, runs, segments of one
  for (int r = 0; r < a.runs; ++r) {
    const int m = __builtin_amdgcn_readlane(n, r);
    const int parts = rows > 0 ? (int)((uint32_t)(m + rows - 1) / (uint32_t)rows) : 0;
    all += parts;
    cut += parts > 1;
    most = max(most, parts);
    runs += m > 0;
  }
  auto rounds = [&](int segments) { return (float)((segments * a.per + 255) / 256); };
  const float c = (float)((min(rows, longest) + CT - 1) / CT);
  float t;
  if constexpr (DELTA)
    t = rounds(all - cut) * (9.f + 2.7f * c) +
        (all > runs ? 3.f + rounds(all - runs) * (11.f + 2.8f * c) + 3.f * (most - 2) : 0.f);
  else
    t = rounds(all) * (6.f + (MODE == kChunkWkv ? 1.45f : NV == 1 ? 1.65f : 2.f) * c) +
        (all > runs ? 10.f + 0.25f * c + 0.8f * most : 0.f);
  const bool may = lane == 0 || (chunk_may_cut(a) && (DELTA ? all - cut : all) <= a.cap);
  uint32_t best = may ? (__float_as_uint(t) & ~63u) | (uint32_t)lane : ~0u;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) best = min(best, (uint32_t)__shfl_xor((int)best, o, 64));
  return __builtin_amdgcn_readlane(rows, (int)(best & 63u));
}
// The item-th segment of the step's runs in their order that the kernel has work for, every wave for itself; n = 0: there
// are fewer.  Items without a gap: where workgroups that leave at once lie between others, those of one remainder are
// left for the same few CUs, which then take two rounds (240 on 256 CUs: 72 us for 36).
enum SegmentKind { kAllSegments, kFirstSegments, kLaterSegments };   // all; a run's only one or all but its last; but its first
template <int MODE, int NV, int KIND>
__device__ __forceinline__ ChunkSegment find_segment(const ChunkArgs& a, int item, int lane) {
  const int r = lane < a.runs ? a.run_rows[lane] : -1;
  const int n = r >= 0 && a.row_back[r] == 0 ? a.row_fwd[r] + 1 : 0;
  const int size = segment_rows<MODE, NV>(a, n, lane);
  if (size == 0) return {0, 0, 0, 0, 0, false, 0};
  const int parts = (n + size - 1) / size;
  const int mine = parts - (KIND == kLaterSegments ? parts > 0 : KIND == kFirstSegments ? parts > 1 : 0);
  int upto = mine;                                         // items of the runs up to this lane's
#pragma unroll
  for (int o = 1; o < 64; o *= 2) {
    const int x = __shfl_up(upto, o, 64);
    if (lane >= o) upto += x;
  }
  const uint64_t m = __builtin_amdgcn_ballot_w64(item < upto);
  if (m == 0) return {0, 0, 0, 0, 0, false, 0};
  const uint64_t single = __builtin_amdgcn_ballot_w64(parts == 1);
  const int at = __builtin_ctzll(m);
  const int before = __builtin_amdgcn_readlane(upto - mine, at), rows = __builtin_amdgcn_readlane(n, at);
  const int seg = item - before + (KIND == kLaterSegments ? 1 : 0);
  // the slot is the item of all or of the first segments
  const int slot = KIND == kLaterSegments ? before + __builtin_popcountll(single & ((1ull << at) - 1)) + seg : item;
  const int run0 = __builtin_amdgcn_readlane(r, at), from = seg * size;
  return {run0, run0 + from, min(rows - from, size), seg, slot, from + size >= rows, size};
}

// Scratch of the delta rule's segments: what a segment leaves of a state of zeros (a run's first one: the state itself),
// [slots, H, dim, vdim]; what it makes of a state, [slots, H, NC, NC]; whether that is bounded, [slots, H, 4].
struct DeltaSeg {
  float *left, *turn, *wild;
};
__device__ __forceinline__ DeltaSeg delta_seg(const ChunkArgs& a, int slot, int h) {
  const int64_t n = (int64_t)a.cap * a.H, at = (int64_t)slot * a.H + h, hsz = (int64_t)NC * a.vdim;
  return {a.seg + at * hsz, a.seg + n * hsz + at * NC * NC, a.seg + n * (hsz + NC * NC) + at * 4};
}

// 64 NV value channels, from zv on, of head h of a run or of a segment of one.  TURN: beside what the rows leave of a
// state of zeros, what they make of any: the state's own columns are 64 more, which begin as the unit matrix and take no
// values; there are no read-outs.
template <typename TI, typename TG, int MODE, int NV = 1, bool TURN = false>
__device__ __forceinline__ void chunk_run(const ChunkArgs& a, const ChunkSegment& sg, const int h, const int zv, const int tid) {
  constexpr bool WKV = MODE == kChunkWkv, DELTA = MODE == kChunkDelta;
  constexpr int NT = NV + (TURN ? 1 : 0);                 // tiles of 16 columns a consumer wave holds
  constexpr bool BF16U = !DELTA && sizeof(TI) == 2;       // u, the values, is of one part
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

  // Offsets inside a chunk in bytes (the launcher bounds 16 rows by 2^31), of a lane's four rows and its column; a chunk's
  // first row is a wave-uniform pointer, which goes on from chunk to chunk: a product for every turn's address costs the
  // wave more than the load.  Rows past the run's end are read as its last row and left out later.
  auto offsets = [&](uint32_t (&o)[4], int64_t stride, int column, int esz, int c) {
#pragma unroll
    for (int i = 0; i < 4; ++i) o[i] = (uint32_t)min(4 * grp + i, n - 1 - c * CT) * (uint32_t)(stride * esz) + (uint32_t)(column * esz);
  };
  // ---- consumers: tiles of 16 value channels, S[16 i + 4 grp + r][column]
  const int vcol = zv + 16 * NV * w + col;                // of the first tile
  auto vlive = [&](int j) { return vcol + 16 * j < vdim; };
  const bool from_state = code >= 0 && a.pos[sg.run0] > 0;
  const int64_t hsz = (int64_t)dim * vdim;
  f32x4 st[NT][4];
  TI vreg[NV][4];
  uint32_t vo[4];
  const TI* vb = static_cast<const TI*>(a.v) + t0 * a.vs + (int64_t)h * vdim;     // of the chunk in flight
  int cf = 0;
  auto next_v = [&]() {                                   // behind the last chunk: that again
    if (cf + 1 < nc) {
      ++cf;
      vb += CT * a.vs;
      if (cf * CT + CT > n) offsets(vo, a.vs, min(vcol, vdim - 1), sizeof(TI), cf);   // the last, partial chunk
    }
  };
  auto fetch_v = [&]() {
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int j = 0; j < NV; ++j)
        vreg[j][r] = load_at(vb, vo[r] + (uint32_t)((min(vcol + 16 * j, vdim - 1) - min(vcol, vdim - 1)) * sizeof(TI)));
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
  auto next = [&]() {                                     // behind the last chunk: that again
    if (cf + 1 < nc) {
      ++cf;
      qb += CT * a.qs;
      kb += CT * a.ks;
      zb += CT * a.zs;
      if (cf * CT + CT > n) {
        offsets(qo, a.qs, chl, sizeof(TI), cf);
        offsets(ko, a.ks, chl, sizeof(TI), cf);
        offsets(zo, a.zs, chl, sizeof(TZ), cf);
      }
    }
  };
  auto fetch = [&]() {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if constexpr (!TURN) rq[i] = load_at(qb, qo[i]);
      rk[i] = load_at(kb, ko[i]);
      rz[i] = load_at(zb, zo[i]);
    }
    if constexpr (DELTA) rb = load_at(bb + (int64_t)min(cf * CT + col, n - 1) * a.bs, 0);
  };
  float4 nw = {}, bonus = {};
  float zbias = 0.f, rate = 0.f;
  const float least = grp == 3 ? kSplitLeast : 0.f;       // of a lane's keys

  if (role == 0) {
    offsets(vo, a.vs, min(vcol, vdim - 1), sizeof(TI), 0);
    const float* rd = a.state + (((int64_t)(code & 1) * a.slots + (code >> 1)) * H + h) * hsz;
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int c = 16 * i + 4 * grp + r;
          if constexpr (TURN) st[j][i][r] = j == NV && c == 16 * w + col ? 1.f : 0.f;
          else st[j][i][r] = (from_state && vlive(j) && c < dim) ? rd[(int64_t)c * vdim + vcol + 16 * j] : 0.f;
        }
    fetch_v();
    if constexpr (DELTA && !TURN) {
      if (sg.seg > 0) {
        // from the state behind the run's first segment through the others before this one
        const uint32_t lo = (uint32_t)(4 * grp * vdim + vcol) * 4, to = (uint32_t)(col * NC + 4 * grp) * 4;
        const float* left = delta_seg(a, sg.slot - sg.seg, h).left;
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int r = 0; r < 4; ++r)
#pragma unroll
            for (int j = 0; j < NT; ++j) st[j][i][r] = load_at(left + (16 * i + r) * vdim, lo + 64 * j);
#pragma unroll 1
        for (int s = sg.slot - sg.seg + 1; s < sg.slot; ++s) {
          const DeltaSeg d = delta_seg(a, s, h);
          f32x4 sum[NT][4];
#pragma unroll
          for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int r = 0; r < 4; ++r)
#pragma unroll
              for (int j = 0; j < NT; ++j) sum[j][i][r] = load_at(d.left + (16 * i + r) * vdim, lo + 64 * j);
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            float4 m[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) m[i] = load_at(reinterpret_cast<const float4*>(d.turn + 16 * i * NC + 16 * e), to);
#define CHUNK_TURN(r, f)                                                                                \
  do {                                                                                                  \
    _Pragma("unroll") for (int j = 0; j < NT; ++j)                                                      \
      _Pragma("unroll") for (int i = 0; i < 4; ++i)                                                     \
        sum[j][i] = __builtin_amdgcn_mfma_f32_16x16x4f32(m[i].f, st[j][e][r], sum[j][i], 0, 0, 0);      \
  } while (0)
            CHUNK_TURN(0, x);
            CHUNK_TURN(1, y);
            CHUNK_TURN(2, z);
            CHUNK_TURN(3, w);
#undef CHUNK_TURN
          }
#pragma unroll
          for (int j = 0; j < NT; ++j)
#pragma unroll
            for (int i = 0; i < 4; ++i) st[j][i] = sum[j][i];
        }
      }
    }
    if constexpr (!DELTA) {
      const uint32_t lo = (uint32_t)(4 * grp * vdim + vcol) * 4;
#pragma unroll 1
      for (int s = sg.slot - sg.seg; s < sg.slot; ++s) {     // through the run's segments before this one
        const float* left = a.seg + ((int64_t)s * H + h) * hsz;
        const float* kept = a.seg + (int64_t)a.cap * H * hsz + ((int64_t)s * H + h) * dim + 4 * grp;
        float x[NT][4][4];
        float4 f[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          f[i] = ld4(kept + 16 * i);
#pragma unroll
          for (int r = 0; r < 4; ++r)
#pragma unroll
            for (int j = 0; j < NT; ++j) x[j][i][r] = load_at(left + (16 * i + r) * vdim, lo + 64 * j);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int j = 0; j < NT; ++j) {
            st[j][i][0] = fmaf(f[i].x, st[j][i][0], x[j][i][0]);
            st[j][i][1] = fmaf(f[i].y, st[j][i][1], x[j][i][1]);
            st[j][i][2] = fmaf(f[i].z, st[j][i][2], x[j][i][2]);
            st[j][i][3] = fmaf(f[i].w, st[j][i][3], x[j][i][3]);
          }
      }
    }
  } else if (role == 1) {
    offsets(qo, a.qs, chl, sizeof(TI), 0);
    offsets(ko, a.ks, chl, sizeof(TI), 0);
    offsets(zo, a.zs, chl, sizeof(TZ), 0);
    fetch();
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
    // The next chunk's values are waited for before this chunk's read-outs are stored: a wait at the top of the turn
    // would be one for the stores, which are counted with the loads and in order.
    float v[NV][4];
    auto values = [&](int c) {
#pragma unroll
      for (int j = 0; j < NV; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) v[j][r] = arrived(vreg[j][r]);
      if (!vlive(NV - 1) || c * CT + CT > n) {
#pragma unroll
        for (int j = 0; j < NV; ++j)
#pragma unroll
          for (int r = 0; r < 4; ++r) v[j][r] = vlive(j) && c * CT + 4 * grp + r < n ? v[j][r] : 0.f;
      }
    };
    values(0);
    float* rw = WKV || TURN ? nullptr : a.raw + ((int64_t)t0 * H + h) * vdim;
    const uint32_t ro = (uint32_t)(4 * grp * H * vdim + vcol);
    for (int it = 0; it < nc; ++it) {
      const int b = it & 3;
      next_v();
      fetch_v();
      f32x4 o[NT], u[NT], y[NT];
      const uint16_t *qp = &L.qd[b][0][col * PS + 8 * grp], *kp = &L.kk[DELTA ? b : 0][0][col * PS + 8 * grp];
      const uint16_t* sp = &L.kd[b][col * PS + 16 * grp];
#pragma unroll
      for (int j = 0; j < NT; ++j) o[j] = y[j] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        uint4 qa[3], ka[3];
#pragma unroll
        for (int p = 0; p < 3; ++p) {
          if constexpr (DELTA) ka[p] = ld8(kp + p * CT * PS + 32 * e);
          if constexpr (!TURN) qa[p] = ld8(qp + p * CT * PS + 32 * e);
        }
#pragma unroll
        for (int j = 0; j < NT; ++j) {
          const f32x4 &s0 = st[j][2 * e], &s1 = st[j][2 * e + 1];
          const Split2 x0 = split3(s0[0], s0[1]), x1 = split3(s0[2], s0[3]), x2 = split3(s1[0], s1[1]), x3 = split3(s1[2], s1[3]);
          const uint4 h = make_uint4(x0.h, x1.h, x2.h, x3.h), m = make_uint4(x0.m, x1.m, x2.m, x3.m),
                      l = make_uint4(x0.l, x1.l, x2.l, x3.l);
          auto product = [&](const uint4 (&a)[3], f32x4& to) {
            to = mma32(a[2], h, to);
            to = mma32(a[0], l, to);
            to = mma32(a[1], m, to);
            to = mma32(a[1], h, to);
            to = mma32(a[0], m, to);
            to = mma32(a[0], h, to);
          };
          if constexpr (DELTA) product(ka, y[j]);
          if constexpr (!TURN) product(qa, o[j]);
        }
      }
      __builtin_amdgcn_sched_barrier(0);                  // operands of later products wait: registers
      const uint4 oddw = *reinterpret_cast<const uint4*>(L.odd[b]);
      const bool flagged = (oddw.x | oddw.y | oddw.z | oddw.w) != 0;
      // Infinities, NaN, and values too large or too small for products of parts: in fp32 products
      bool plain = !flagged;
#pragma unroll
      for (int j = 0; j < NT; ++j) {
        plain &= j < NV ? within(sum_of_sizes(TURN ? y[j] : o[j]), kReadLeast, __builtin_huge_valf()) : finite4(y[j]);
        if constexpr (DELTA && !TURN) plain &= finite4(y[j]);
      }
      bool odd = false;
      if (__builtin_amdgcn_ballot_w64(!plain) != 0ull) {
        bool bad = flagged;
#pragma unroll
        for (int j = 0; j < NT; ++j) {
          float most = 0.f;                               // a turn's columns may be as small as they are: they began as one
#pragma unroll
          for (int i = 0; i < 4; ++i) most = j < NV ? fmaxf(most, largest(st[j][i])) : 0.f;
          bad |= !finite4(o[j]) | !finite4(y[j]) | small_column(most);
        }
        odd = __builtin_amdgcn_ballot_w64(bad) != 0ull;
      }
      if (odd) {
#pragma unroll
        for (int j = 0; j < NT; ++j) o[j] = y[j] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float down = L.odd[b][i] == kOddLarge ? 1.f : kDown;
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int at = 32 * (i >> 1) + 4 * (i & 1) + r;
            auto whole = [&](const uint16_t* p) { return ((ldf(p + at) + ldf(p + at + CT * PS)) + ldf(p + at + 2 * CT * PS)) * down; };
#pragma unroll
            for (int j = 0; j < NT; ++j) {
              if constexpr (DELTA) y[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(whole(kp), st[j][i][r], y[j], 0, 0, 0);
              if constexpr (!TURN) o[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(whole(qp), st[j][i][r], o[j], 0, 0, 0);
            }
          }
        }
      }
      const float down = odd ? 1.f : kDown;
      f32x4 own[NT];                                      // read-outs of the chunk's own tokens
#pragma unroll
      for (int j = 0; j < NT; ++j) own[j] = (f32x4){0.f, 0.f, 0.f, 0.f};
      if constexpr (DELTA) {
        const float4 bt = ld4(&L.beta[b][4 * grp]), ta = ld4(&L.tt[it & 1][col * TS + 4 * grp]);
        f32x4 x[NT];
        bool whole = true;
#pragma unroll
        for (int j = 0; j < NT; ++j) {
          const f32x4 val = j < NV ? (f32x4){v[j % NV][0], v[j % NV][1], v[j % NV][2], v[j % NV][3]} : (f32x4){0.f, 0.f, 0.f, 0.f};
          x[j] = (f32x4){bt.x * fmaf(-down, y[j][0], val[0]), bt.y * fmaf(-down, y[j][1], val[1]),
                         bt.z * fmaf(-down, y[j][2], val[2]), bt.w * fmaf(-down, y[j][3], val[3])};
          u[j] = (f32x4){0.f, 0.f, 0.f, 0.f};
          whole = whole && finite4(x[j]);
        }
        if (__builtin_amdgcn_ballot_w64(!whole) == 0ull) {
#pragma unroll
          for (int j = 0; j < NT; ++j) u[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(ta.x, x[j][0], u[j], 0, 0, 0);
#pragma unroll
          for (int j = 0; j < NT; ++j) u[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(ta.y, x[j][1], u[j], 0, 0, 0);
#pragma unroll
          for (int j = 0; j < NT; ++j) u[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(ta.z, x[j][2], u[j], 0, 0, 0);
#pragma unroll
          for (int j = 0; j < NT; ++j) u[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(ta.w, x[j][3], u[j], 0, 0, 0);
        } else {
#pragma unroll
          for (int j = 0; j < NT; ++j) lower_product(L.tt[it & 1], x[j], col, grp, u[j]);
        }
      } else {
#pragma unroll
        for (int j = 0; j < NT; ++j) u[j] = (f32x4){v[j][0], v[j][1], v[j][2], v[j][3]};
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float4 dc = ld4(&L.dec[b][16 * i + 4 * grp]);
#pragma unroll
        for (int j = 0; j < NT; ++j) {
          st[j][i][0] *= dc.x;
          st[j][i][1] *= dc.y;
          st[j][i][2] *= dc.z;
          st[j][i][3] *= dc.w;
        }
      }
      bool fits = !odd;                                   // for products of parts
#pragma unroll
      for (int j = 0; j < NT; ++j)
        fits &= j < NV && !BF16U ? within(sum_of_sizes(u[j]), kSplitLeast, kSplitMost) : sum_of_sizes(u[j]) < kSplitMost;
      auto bad = [&]() {
        bool any = odd;
#pragma unroll
        for (int j = 0; j < NT; ++j) any |= !(sum_of_sizes(u[j]) < kSplitMost) | small_column(j < NV && !BF16U ? largest(u[j]) : 0.f);
        return __builtin_amdgcn_ballot_w64(any) != 0ull;
      };
      if (__builtin_amdgcn_ballot_w64(!fits) != 0ull && bad()) {
#pragma unroll
        for (int j = 0; j < NT; ++j) {
          if constexpr (!TURN) lower_product(L.aq[b], u[j], col, grp, own[j]);
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const float down = L.odd[b][i] == kOddSmall ? kDownKd : 1.f;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              const uint16_t* p = sp + 16 * i * PS + r;
              const float k = ((ldf(p) + ldf(p + 4)) + ldf(p + 12)) * down;
              st[j][i] = __builtin_amdgcn_mfma_f32_16x16x4f32(k, u[j][r], st[j][i], 0, 0, 0);
            }
          }
        }
      } else {
        if constexpr (!TURN) {
          const float4 aa = ld4(&L.aq[b][col * TS + 4 * grp]);
#pragma unroll
          for (int j = 0; j < NT; ++j) own[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(aa.x, u[j][0], own[j], 0, 0, 0);
#pragma unroll
          for (int j = 0; j < NT; ++j) own[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(aa.y, u[j][1], own[j], 0, 0, 0);
#pragma unroll
          for (int j = 0; j < NT; ++j) own[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(aa.z, u[j][2], own[j], 0, 0, 0);
#pragma unroll
          for (int j = 0; j < NT; ++j) own[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(aa.w, u[j][3], own[j], 0, 0, 0);
        }
        // a lane's eight are two parts of four tokens: (l h + h l), (h m + m m), (h h + m h)
        uint4 kh[4][2];
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int p = 0; p < 2; ++p) kh[i][p] = ld8(sp + 16 * i * PS + 8 * p);
#pragma unroll
        for (int j = 0; j < NT; ++j) {
          Split2 p{}, q{};
          if constexpr (BF16U) {
            p.h = rfq::pack_bf16x2(u[j][0], u[j][1]);
            q.h = rfq::pack_bf16x2(u[j][2], u[j][3]);
          } else {
            p = split3(u[j][0], u[j][1]);
            q = split3(u[j][2], u[j][3]);
          }
          const uint4 lh = make_uint4(p.l, q.l, p.h, q.h), mm = make_uint4(p.m, q.m, p.m, q.m), hh = make_uint4(p.h, q.h, p.h, q.h);
#pragma unroll
          for (int i = 0; i < 4; ++i) st[j][i] = mma32(kh[i][1], lh, st[j][i]);
          if constexpr (!BF16U)
#pragma unroll
            for (int i = 0; i < 4; ++i) st[j][i] = mma32(kh[i][0], mm, st[j][i]);
#pragma unroll
          for (int i = 0; i < 4; ++i) st[j][i] = mma32(kh[i][0], hh, st[j][i]);
        }
      }
      if constexpr (!TURN)
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
          for (int r = 0; r < 4; ++r) o[j][r] = fmaf(o[j][r], down, own[j][r]);
      values(min(it + 1, nc - 1));
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (WKV) {
#pragma unroll
        for (int r = 0; r < 4; ++r) L.o[it & 1][(4 * grp + r) * RS + 16 * w + col] = o[0][r];
      } else if constexpr (!TURN) {
        float* row = rw;                                  // of the chunk's first row, then the next
        const bool all = it * CT + CT <= n && zv + 64 * NV <= vdim;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
#pragma unroll
          for (int j = 0; j < NT; ++j)
            if (all || (vlive(j) && it * CT + 4 * grp + r < n)) row[ro + 16 * j] = o[j][r] * a.q_scale;
          row += H * vdim;
        }
        rw += (int64_t)CT * H * vdim;
      }
      __syncthreads();
    }
    if constexpr (WKV) __syncthreads();
  } else if (role == 1) {
    for (int it = -3; it < turns; ++it) {
      float q[4], k[4], d[4], bt = 0.f;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        q[i] = 0.f;
        if constexpr (!TURN) q[i] = arrived(rq[i]);
        k[i] = arrived(rk[i]);
        d[i] = arrived(rz[i]) + zbias;
      }
      if constexpr (DELTA) bt = arrived(rb);
      next();
      fetch();
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
        float qd[4], kk[4], kd[4], sizes = 0.f, most = 0.f;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int at = (4 * grp + i) * RS + ch;
          const float ql = WKV ? (i == 0 ? q[0] : q[i] * up[i - 1]) : q[i] * up[i];
          const float kl = k[i] * after[i];
          kd[i] = kl * post;
          qd[i] = ql * pre;
          kk[i] = 0.f;
          sizes += fabsf(kd[i]);
          most += fabsf(qd[i]);
          if constexpr (!TURN) {
            L.q[e][at] = q[i];
            L.ql[e][at] = ql;
          }
          L.k[e][at] = k[i];
          L.a[e][at] = d[i];
          L.kl[e][at] = kl;
          if constexpr (DELTA) {
            const float kb = k[i] * up[i];
            L.kb[e][at] = kb;
            kk[i] = kb * pre;
            most += fabsf(kk[i]);
          }
        }
        // as a rule the last four tokens say that a channel's keys are not too small
        uint32_t odd = 0;
        const float all = fmaf(most, kUp, sizes);
        if (__builtin_amdgcn_ballot_w64(!((all < kSplitMost) & (sizes >= least))) != 0ull) {
          if (__builtin_amdgcn_ballot_w64(!(all < kSplitMost)) != 0ull) {
            odd = kOddLarge;
          } else if (__builtin_amdgcn_ballot_w64(small_column(sizes)) != 0ull) {
            odd = kOddSmall;
#pragma unroll
            for (int i = 0; i < 4; ++i) kd[i] *= kUpKd;
          }
        }
        if (lane == 0) L.odd[b][w] = odd;
        auto put = [&](auto split, float up) {
          const Split2 p = split(kd[0], kd[1]), q = split(kd[2], kd[3]);
          uint4* to = reinterpret_cast<uint4*>(&L.kd[b][ch * PS + 16 * grp]);
          to[0] = make_uint4(p.h, q.h, p.m, q.m);
          to[1] = make_uint4(p.h, q.h, p.l, q.l);
          const int at = 4 * grp * PS + operand_at(ch);
#pragma unroll
          for (int i = 0; i < 4; i += 2) {
            auto rows = [&](uint16_t (&part)[3][CT * PS], const Split2& x) {
              const uint32_t f[3] = {x.h, x.m, x.l};
#pragma unroll
              for (int y = 0; y < 3; ++y) {
                part[y][at + i * PS] = (uint16_t)f[y];
                part[y][at + (i + 1) * PS] = (uint16_t)(f[y] >> 16);
              }
            };
            if constexpr (!TURN) rows(L.qd[b], split(qd[i] * up, qd[i + 1] * up));
            if constexpr (DELTA) rows(L.kk[b], split(kk[i] * up, kk[i + 1] * up));
          }
        };
        if (odd == kOddLarge) put([](float x, float y) { return odd_split(x, y); }, 1.f);
        else put([](float x, float y) { return split3(x, y); }, kUp);
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
        // A of chunk c.  A pair of blocks: the readers' rows with the writers' rows times the blocks between them, on tiles
        // of 4x4x1, of which sixteen side by side take four key channels each.
        const int b = c & 1, at = lane & ~3;
        auto pair = [&](auto tb_c, auto sb_c) {
          constexpr int tb = tb_c, sb = sb_c;
          float4 k = ld4(&L.kl[b][(4 * sb + (lane & 3)) * RS + at]);
          if constexpr (tb > sb + 1) k = mul4(k, ld4(&L.blk[b][(sb + 1) * NC + at]));
          if constexpr (tb > sb + 2) k = mul4(k, ld4(&L.blk[b][(sb + 2) * NC + at]));
          auto product = [&](const float* rows, float* to) {
            const float4 q = ld4(rows + (4 * tb + (lane & 3)) * RS + at);
            f32x4 x = (f32x4){0.f, 0.f, 0.f, 0.f};
            x = __builtin_amdgcn_mfma_f32_4x4x1f32(q.x, k.x, x, 0, 0, 0);
            x = __builtin_amdgcn_mfma_f32_4x4x1f32(q.y, k.y, x, 0, 0, 0);
            x = __builtin_amdgcn_mfma_f32_4x4x1f32(q.z, k.z, x, 0, 0, 0);
            x = __builtin_amdgcn_mfma_f32_4x4x1f32(q.w, k.w, x, 0, 0, 0);
            const float y = tiles_sum(x);
            if ((lane & 12) == 0) to[(4 * tb + grp) * TS + 4 * sb + (lane & 3)] = y;
          };
          if constexpr (!TURN) product(L.ql[b], L.aq[c & 3]);
          if constexpr (DELTA) product(L.kb[b], L.ak[b]);
        };
        constexpr std::integral_constant<int, 0> i0{};
        constexpr std::integral_constant<int, 1> i1{};
        constexpr std::integral_constant<int, 2> i2{};
        constexpr std::integral_constant<int, 3> i3{};
        if constexpr (DELTA) {
          if (w == 1) { pair(i1, i0); pair(i2, i1); pair(i3, i0); }
          else if (w == 2) { pair(i3, i2); pair(i2, i0); pair(i3, i1); }
        } else {
          if (w == 0) { pair(i1, i0); pair(i2, i0); }
          else if (w == 1) { pair(i2, i1); pair(i3, i1); }
          else if (w == 2) { pair(i3, i2); pair(i3, i0); }
        }
        if (w == (DELTA ? 0 : 3)) {
          // pairs inside a block: sixteen lanes per block, four key channels each
          float4 q[4], k[4], d[4];
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int at = (4 * grp + i) * RS + 4 * col;
            if constexpr (!TURN) q[i] = ld4(&L.q[b][at]);
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
            if constexpr (!TURN) {
              acc[1] = dot4(q[1], e10);
              acc[3] = dot4(q[2], e20);
              acc[4] = dot4(q[2], e21);
              acc[6] = dot4(q[3], e30);
              acc[7] = dot4(q[3], e31);
              acc[8] = dot4(q[3], e32);
#pragma unroll
              for (int i = 0; i < 4; ++i) acc[i * (i + 3) / 2] = dot4(q[i], k[i]);
            }
            if constexpr (DELTA) {
              ack[0] = dot4(k[1], e10);
              ack[1] = dot4(k[2], e20);
              ack[2] = dot4(k[2], e21);
              ack[3] = dot4(k[3], e30);
              ack[4] = dot4(k[3], e31);
              ack[5] = dot4(k[3], e32);
            }
          }
          if constexpr (!TURN) {
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

  if constexpr (DELTA) {
    // what the later kernel reads: never written by it, whose workgroups begin and end at any time
    if (role == 0 && !sg.last && (TURN || sg.seg == 0)) { // a segment: dim is NC and all channels are there
      const DeltaSeg d = delta_seg(a, sg.slot, h);
#pragma unroll
      for (int j = 0; j < NV; ++j)
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int r = 0; r < 4; ++r) d.left[(16 * i + 4 * grp + r) * vdim + vcol + 16 * j] = st[j][i][r];
      if constexpr (TURN)
        if (zv == 0) {
          bool ok = true;
#pragma unroll
          for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              d.turn[(16 * i + 4 * grp + r) * NC + 16 * w + col] = st[NV][i][r];
              ok = ok && fabsf(st[NV][i][r]) <= kTurnMost;
            }
          const uint64_t all = __builtin_amdgcn_ballot_w64(ok);
          if (lane == 0) d.wild[w] = all == ~0ull ? 0.f : 1.f;
        }
    }
  }
  if (role == 0 && code >= 0 && sg.last) {
    float* wr = a.state + (((int64_t)(1 - (code & 1)) * a.slots + (code >> 1)) * H + h) * hsz;
#pragma unroll
    for (int j = 0; j < NV; ++j)
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int c = 16 * i + 4 * grp + r;
          if (c < dim && vlive(j)) wr[(int64_t)c * vdim + vcol + 16 * j] = st[j][i][r];
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
// one workgroup per segment, head, 32 key and 64 value channels.  A wave has an eighth (a sixteenth) of the rows and goes
// through them from the last chunk to the first, the keys times all decays behind them: nothing is rescaled, and the lane
// that makes such a product (four tokens of two key channels) has it as the MFMA operand.  No LDS but to add the waves' parts.
constexpr int kSegKeys = 32;
template <typename TI, int MODE, int NV, int kSegWaves>
__global__ __launch_bounds__(64 * kSegWaves, 4) void chunk_segment_kernel(const ChunkArgs a) {
  constexpr bool WKV = MODE == kChunkWkv;
  typedef typename std::conditional<WKV, TI, float>::type TZ;
  typedef typename std::conditional<sizeof(TI) == 2, uint2, uint4>::type RV;
  typedef typename std::conditional<sizeof(TI) == 2, uint32_t, uint2>::type RK;
  typedef typename std::conditional<sizeof(TZ) == 2, uint32_t, uint2>::type RZ;
  const int tid = threadIdx.x, lane = tid & 63, col = lane & 15, grp = lane >> 4;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const ChunkSegment sg = find_segment<MODE, NV, kAllSegments>(a, blockIdx.z, lane);
  if (sg.n == 0 || sg.last) return;
  __shared__ __attribute__((aligned(16))) float sums[kSegWaves / 2][kSegKeys * NC];
  const int h = blockIdx.x, z64 = (blockIdx.y >> 1) * 64, c0 = (blockIdx.y & 1) * kSegKeys, H = a.H, vdim = a.vdim, hq = h / a.rep;
  const int rows = sg.rows / kSegWaves;
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
    a.seg[a.cap * (int64_t)(H * NC) * vdim + ((int64_t)sg.slot * H + h) * NC + c0 + tid] = f;
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

// A workgroup per segment, head and 64 NV value channels, behind chunk_segment_kernel.
template <typename TI, typename TG, int MODE, int NV>
__global__ __launch_bounds__(chunk_threads(MODE)) void chunk_recurrence_segments_kernel(const ChunkArgs a) {
  const ChunkSegment sg = find_segment<MODE, NV, kAllSegments>(a, blockIdx.z, threadIdx.x & 63);
  if (sg.n > 0) chunk_run<TI, TG, MODE, NV>(a, sg, blockIdx.x, blockIdx.y * 64 * NV, threadIdx.x);
}

// The delta rule's segments.  Before: a run's first segment to its end, read-outs and all, and of the others but a run's
// last what their rows leave of a state of zeros and the 64 x 64 turn that they make of any, by the same chunks with 64
// more columns.  After it the later segments, from the state that the turns carry to them.  A workgroup per segment,
// head and 128 value channels: the producers' work, which 64 channels cost as much, is done half as often.
// Two runs of 2,048 with 32 heads: 301 -> 82 + 89 us.  Error of the state against 64 bits as with whole runs (6.3e-8 to
// 6.5e-8).  Unit keys and betas of at most 1 turn a state no larger.  Where an entry passes that (other keys, whose turns may
// grow or overflow though the state does not), the rest of the run is gone through in sequence, by the workgroups of its
// second segment and of its third (there is one: turns are of segments between others), 64 channels each, which take 2.1 us
// a chunk for 128 channels' 2.7: two runs of 2,048 with 32 heads 284 us a call, one of 4,096 491 (as whole runs in fp32
// products 319 and 596, in one go of 128 channels 352 and 638); four of 600 with 16 heads 106, 103 as whole runs.
template <typename TI, typename TG>
__global__ __launch_bounds__(chunk_threads(kChunkDelta)) void chunk_delta_first_kernel(const ChunkArgs a) {
  const ChunkSegment sg = find_segment<kChunkDelta, 2, kFirstSegments>(a, blockIdx.z, threadIdx.x & 63);
  if (sg.n == 0) return;
  if (sg.seg == 0) chunk_run<TI, TG, kChunkDelta, 2>(a, sg, blockIdx.x, blockIdx.y * 128, threadIdx.x);
  else chunk_run<TI, TG, kChunkDelta, 2, true>(a, sg, blockIdx.x, blockIdx.y * 128, threadIdx.x);
}
template <typename TI, typename TG>
__global__ __launch_bounds__(chunk_threads(kChunkDelta)) void chunk_delta_later_kernel(const ChunkArgs a) {
  const int lane = threadIdx.x & 63, h = blockIdx.x;
  ChunkSegment sg = find_segment<kChunkDelta, 2, kLaterSegments>(a, blockIdx.z, lane);
  if (sg.n == 0) return;
  const int rows = a.row_fwd[sg.run0] + 1, turns = (rows + sg.rows - 1) / sg.rows - 2;
  const float* wild = delta_seg(a, sg.slot - sg.seg + 1, h).wild;        // of the run's second segment
  uint64_t any = 0;
  for (int x = lane; x < 4 * turns; x += 64) any |= wild[(int64_t)(x >> 2) * a.H * 4 + (x & 3)] != 0.f;
  if (__builtin_amdgcn_ballot_w64(any != 0) == 0ull) {
    chunk_run<TI, TG, kChunkDelta, 2>(a, sg, h, blockIdx.y * 128, threadIdx.x);
  } else if (sg.seg <= 2) {
    const int part = sg.seg - 1;
    sg.slot -= part;
    sg.seg = 1;
    sg.t0 = sg.run0 + sg.rows;
    sg.n = rows - sg.rows;
    sg.last = true;
    chunk_run<TI, TG, kChunkDelta>(a, sg, h, blockIdx.y * 128 + 64 * part, threadIdx.x);
  }
}

// Workgroups, one to a CU at most, that share the runs of min_run rows or more, which every wave counts for
// itself: one for every run that the step has room for costs 16 us where there is none (64 runs of 16, wkv).  Where those
// runs are more than one round, a workgroup takes 128 value channels at a time, 1.25 of the time for twice the work.
template <typename TI, typename TG, int MODE>
__global__ __launch_bounds__(chunk_threads(MODE)) void chunk_recurrence_share_kernel(const ChunkArgs a) {
  const int lane = threadIdx.x & 63;
  auto fits = [&](int base, int& r) {
    r = base + lane < a.runs ? a.run_rows[base + lane] : -1;
    return __builtin_amdgcn_ballot_w64(r >= 0 && a.row_back[r] == 0 && a.row_fwd[r] + 1 >= a.min_run);
  };
  int width = 64, r;
  if constexpr (MODE != kChunkWkv)
    if (a.vdim > 64) {
      int all = 0;
      for (int base = 0; base < a.runs; base += 64) all += __builtin_popcountll(fits(base, r));
      if ((int64_t)all * a.H * ((a.vdim + 63) / 64) > gridDim.x) width = 128;
    }
  const int per = a.H * ((a.vdim + width - 1) / width);
#pragma unroll 1
  for (int item = blockIdx.x;; item += gridDim.x) {
    int left = item / per, t0 = -1;
    const int part = item - left * per, z = part / a.H;
    for (int base = 0; base < a.runs; base += 64) {
      uint64_t m = fits(base, r);
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
    if (MODE == kChunkWkv || width == 64)
      chunk_run<TI, TG, MODE>(*(const ChunkArgs*)p, whole_run(*(const ChunkArgs*)p, t0), part - z * a.H, z * 64, tid);
    else if constexpr (MODE != kChunkWkv)
      chunk_run<TI, TG, MODE, 2>(*(const ChunkArgs*)p, whole_run(*(const ChunkArgs*)p, t0), part - z * a.H, z * 128, tid);
  }
}

// ------------------------------------------------------------------ launcher
// A workgroup costs some 8 us before its first chunk is out and 1.45 - 2.1 us a chunk (1.6 - 2.3 with the state's products
// in fp32, which the times below are of: the lines are on the safe side), one to a CU; the token-by-token kernels some 6 us
// and 0.2 (64 runs) - 2.6 us a token, many to a CU.  Times of whole steps, 32 heads of 64 x 128 (wkv: 64 of 64 x 64), chunks
// against tokens.
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

// Segments instead of whole runs, which the kernels place where that is faster (segment_rows; only they know the runs):
// from steps on whose runs, taken as equally long, gain a tenth by it by the same times (a first kernel that finds nothing
// to cut costs 5 - 10 us: gla, 16 heads, 8 runs of 128, 32 us for 45), and in all steps whose whole runs are more than
// one round of workgroups of 64 value channels, for workgroups of 128 are no more than one then (gla, 32 heads, 8 runs of
// 512: 156 -> 110).  Room is for as many segments as the chip has CUs; for twice the runs where these fill it alone, from 40
// chunks a run on.  183 steps of 72 to 4,096 tokens, 16 to 64 heads, against whole runs of 64 channels in fp32 products:
// 1.34 times as fast on the average, 5.8 at the most, six of them (72 or 128 tokens a run) 1 - 2 % slower.
int chunk_seg_cap(int mode, bool in_f32, int T, ChunkArgs& a) {
  if (chunk_min_run(mode, T, a) != 1 || a.dim != NC || a.runs > 64) return 0;
  const int wide = a.vdim % 128 == 0 ? 2 : 1;             // 64 value channels to a workgroup
  if (mode == kChunkDelta) {
    if (wide == 1) return 0;
  } else {
    if (a.vdim % 64 != 0) return 0;
    const uintptr_t v4 = in_f32 ? 16 : 8, z2 = mode == kChunkWkv && !in_f32 ? 4 : 8;     // loads of four, of two
    for (const void* p : {a.k, a.v})
      if (reinterpret_cast<uintptr_t>(p) % v4 != 0) return 0;
    if (reinterpret_cast<uintptr_t>(a.z) % z2 != 0) return 0;
    for (int64_t st : {a.ks, a.vs, a.zs})
      if (st % 4 != 0) return 0;
  }
  const int64_t narrow = (int64_t)a.H * (a.vdim / 64);
  a.per = (int)(narrow / wide);
  const int room = std::max(256 / a.per, a.runs), parts = room / a.runs;
  // sixteen waves to a segment of chunk_segment_kernel where it is that long, else eight
  a.unit = mode == kChunkDelta ? CT : CT * (T / std::min(room, 2 * a.runs) >= 64 * CT && T / room >= 48 * CT ? 16 : 8);
  const double c = (double)T / (CT * a.runs);             // chunks of a run
  if (room == a.runs) return wide == 1 ? 0 : c >= 40 ? 2 * room : a.runs * narrow > 256 ? room : 0;
  if (a.runs * narrow <= 256) {
    const double turn = mode == kChunkDelta ? 2.1 : mode == kChunkWkv ? 1.45 : 1.65;
    double cut = 1e9;
    for (int n = 2; n <= std::min(parts + (mode == kChunkDelta), 64); ++n)
      cut = std::min(cut, mode == kChunkDelta ? 20 + 5.5 * std::ceil(c / n) + 3 * (n - 2)
                                              : 18 + (0.25 + (wide == 1 ? turn : 2.)) * std::max(std::ceil(c / n), 8.) + 0.8 * n);
    if (cut > 0.9 * (6 + turn * c)) return 0;
  }
  return room;
}
int64_t chunk_seg_floats(int mode, const ChunkArgs& a) {
  return (int64_t)a.cap * a.H * (mode == kChunkDelta ? NC * a.vdim + NC * NC + 4 : a.dim * (a.vdim + 1));
}

// Dynamic LDS above 64 KB has to be allowed per kernel, once.
template <auto kernel>
static void allow_lds() {
  static bool done = false;
  if (!done) (void)hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
  done = true;
}

template <typename TI, typename TG, int MODE, int NV>
static void launch_chunk_segments(const ChunkArgs& a, hipStream_t s) {
  constexpr int lds = sizeof(ChunkLds<MODE>);
  const dim3 grid(a.H, a.vdim / (64 * NV), a.cap), wg(chunk_threads(MODE));
  if constexpr (MODE == kChunkDelta) {
    allow_lds<&chunk_delta_first_kernel<TI, TG>>();
    allow_lds<&chunk_delta_later_kernel<TI, TG>>();
    hipLaunchKernelGGL((chunk_delta_first_kernel<TI, TG>), grid, wg, lds, s, a);
    if (chunk_may_cut(a)) hipLaunchKernelGGL((chunk_delta_later_kernel<TI, TG>), grid, wg, lds, s, a);
  } else {
    allow_lds<&chunk_recurrence_segments_kernel<TI, TG, MODE, NV>>();
    const dim3 parts(a.H, a.vdim / 64 * (NC / kSegKeys), a.cap);
    if (chunk_may_cut(a) && a.unit > 8 * CT) hipLaunchKernelGGL((chunk_segment_kernel<TI, MODE, NV, 16>), parts, dim3(1024), 0, s, a);
    else if (chunk_may_cut(a)) hipLaunchKernelGGL((chunk_segment_kernel<TI, MODE, NV, 8>), parts, dim3(512), 0, s, a);
    hipLaunchKernelGGL((chunk_recurrence_segments_kernel<TI, TG, MODE, NV>), grid, wg, lds, s, a);
  }
}

template <typename TI, typename TG, int MODE>
static void launch_chunk_one(int T, const ChunkArgs& a, hipStream_t s) {
  constexpr int lds = sizeof(ChunkLds<MODE>);
  static_assert(lds <= 160 * 1024, "LDS of a CU");
  const int cols = (a.vdim + 63) / 64;
  const dim3 wg(chunk_threads(MODE));
  if (a.seg != nullptr) {
    if constexpr (MODE != kChunkWkv)
      if (a.vdim % 128 == 0) return launch_chunk_segments<TI, TG, MODE, 2>(a, s);
    if constexpr (MODE != kChunkDelta) launch_chunk_segments<TI, TG, MODE, 1>(a, s);
  } else if (a.min_run <= 1) {
    allow_lds<&chunk_recurrence_kernel<TI, TG, MODE>>();
    hipLaunchKernelGGL((chunk_recurrence_kernel<TI, TG, MODE>), dim3(a.runs, a.H, cols), wg, lds, s, a);
  } else {                    // no more long runs than rows allow
    allow_lds<&chunk_recurrence_share_kernel<TI, TG, MODE>>();
    hipLaunchKernelGGL((chunk_recurrence_share_kernel<TI, TG, MODE>),
                       dim3((unsigned)std::min<int64_t>((int64_t)std::min(a.runs, T / a.min_run) * a.H * cols, 256)), wg,
                       lds, s, a);
  }
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
