// The linear recurrences of mix_linrec.hip and mix_wkv.hip where runs are short, decode rows above all: token by token,
// a head's state once through the registers of a workgroup.  Keys of 32, 64 or 128 channels (wkv: 64), value channels in
// fours.
//
// What bounds it: the state's bytes, read from one half of the pool and written to the other.  So they go in 16-byte
// pieces, eight lanes to a line of 128 bytes and 1 KB to an access, and all of a lane's pieces are on their way before it
// waits for the first.  A wave has 32 value channels and all key channels: lane (kg, vl) holds S[8 i + kg][4 vl .. 4 vl + 3],
// so that sums over keys stay inside the wave (three steps between lanes), and the workgroups of a sequence's heads lie
// side by side in memory and in the grid.  64 registers a lane: 64 sequences of 32 heads of 64 x 128 are all on the chip at
// once.  Writes go past the caches, reads do not (all through them 31.6 us a pass of gla, neither 28.3, so 25.4).
// Measured with states that no cache holds, 64 decode rows, against a value channel a thread with 4-byte accesses:
// delta rule, 32 heads of 64 x 128 (134 MB), 36.1 -> 22.2 us (6.0 TB/s; a copy of that size reaches 5.9), a pass of gla of
// these sizes 36.1 -> 25.4, of wkv, 64 heads of 64 x 64, 35.6 -> 28.5.  One to eight sequences: the same, launches.
#include <algorithm>
#include <type_traits>

#include "mix_common.h"
#include "mix_chunk.h"
#include "mix_linrec.h"

namespace rfqmix {

namespace {
typedef float f4 __attribute__((ext_vector_type(4)));

// Sum over the eight lanes 8 kg + vl of a value lane; every one of them receives it.
__device__ __forceinline__ float keys_sum(float v) {
  v += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x128, 0xf, 0xf, true));      // 8 lanes on, in a row of 16
  auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = __uint_as_float(r[0]) + __uint_as_float(r[1]);
  r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
__device__ __forceinline__ f4 keys_sum(const f4& v) { return (f4){keys_sum(v[0]), keys_sum(v[1]), keys_sum(v[2]), keys_sum(v[3])}; }

// Global memory, and what a whole wave reads alike, by scalar loads.
template <typename T>
using glob = const __attribute__((address_space(1))) T;
template <typename T>
__device__ __forceinline__ glob<T>* global_at(const void* base, int64_t elements) {
  return (glob<T>*)(uintptr_t)(static_cast<const T*>(base) + elements);
}
// entry i of lane's own behind a base that is the wave's: an offset of 32 bits in bytes
template <typename T>
__device__ __forceinline__ T lane_at(glob<T>* base, uint32_t i) {
  return *(glob<T>*)((glob<char>*)base + i * (uint32_t)sizeof(T));
}
template <typename T>
__device__ __forceinline__ T same(const T* p, int64_t i) {
  return ((const __attribute__((address_space(4))) T*)(uintptr_t)p)[i];
}
// Four values as loaded: converted where they are used, so that nothing waits for them before.
__device__ __forceinline__ float up(float x) { return x; }
__device__ __forceinline__ float up(bf16_t x) { return __uint_as_float((uint32_t)x << 16); }
template <typename T>
struct Four {
  typedef T bits __attribute__((ext_vector_type(4)));
  bits b;
  __device__ __forceinline__ f4 get() const {
    if constexpr (sizeof(T) == 4) return b;
    else return (f4){up(b[0]), up(b[1]), up(b[2]), up(b[3])};
  }
};
}  // namespace

// KR key channels a lane (8 KR in all); MODE as for the chunks.
template <typename TI, typename TG, int KR, int MODE>
__global__ __launch_bounds__(512, MODE == kChunkWkv ? 7 : KR <= 8 ? 8 : 4) void state_rows_kernel(const StateRows a) {
  constexpr bool WKV = MODE == kChunkWkv, DELTA = MODE == kChunkDelta;
  constexpr int dim = 8 * KR, RS = KR + 4;                // floats of a key group in LDS: groups on different banks
  const int run = blockIdx.z * 65535 + blockIdx.y, h = blockIdx.x;
  if (run >= a.runs) return;
  const int t0 = a.run_rows != nullptr ? same(a.run_rows, run) : run;
  if (t0 < 0) return;
  const int back = same(a.row_back, t0), n = same(a.row_fwd, t0) + 1, code = same(a.row_state, t0), pos = same(a.pos, t0);
  if (back != 0 || n >= a.below) return;                  // not a run's first row; a run of the chunked kernel
  const int tid = threadIdx.x, lane = tid & 63, kg = lane >> 3, H = a.H, vdim = a.vdim;
  // what a thread's number says, made anew where it is used: registers
  auto fresh = [] {
    int t = threadIdx.x;
    asm volatile("" : "+v"(t));
    return t;
  };
  const float zsign = a.zsign, eps = a.eps, q_scale = a.q_scale;
  const bool sigmoid = a.gate_sigmoid != 0;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const bool live = wave * 32 + (lane & 7) * 4 < vdim;
  // four value channels; the one that the lane writes; its bytes of the state
  auto four_of = [&](int t) { return (uint32_t)min(wave * 32 + (t & 7) * 4, vdim - 4); };
  auto one_of = [&](int t) { return four_of(t) + (t >> 3 & 3); };
  auto state_of = [&](int t) { return ((t >> 3 & 7) * vdim + four_of(t)) * 4; };
  const uint32_t kc = min(tid, dim - 1);

  __shared__ __attribute__((aligned(16))) float ops[WKV ? 4 : 3][8 * RS];   // decay, k, q, wkv: q u k of key channel 8 i + kg at [kg][i]
  __shared__ float part[8];

  typedef typename std::conditional<WKV, TI, float>::type TZ;
  TI rq, rk;
  TZ rz;
  TG rg, rb{};
  Four<TI> rv;
  const int hk = h / a.rep * dim;
  auto fetch = [&](int row) {                             // a token's operands
    asm volatile("" : "+s"(row));                         // addresses are made anew from token to token: registers
    const int64_t t = row;
    const int me = fresh();
    const uint32_t kc = min(me, dim - 1);
    rq = lane_at(global_at<TI>(a.q, t * a.qs + hk), kc);
    rk = lane_at(global_at<TI>(a.k, t * a.ks + hk), kc);
    rz = lane_at(global_at<TZ>(a.z, t * a.zs + h * dim), kc);
    rv.b = lane_at((glob<typename Four<TI>::bits>*)global_at<TI>(a.v, t * a.vs + h * vdim), four_of(me) / 4);
    rg = lane_at(global_at<TG>(a.gate, t * a.gs + h * vdim), one_of(me));
    if constexpr (DELTA) rb = global_at<TG>(a.beta, t * a.bs + h)[0];
  };
  fetch(t0);
  const float zbias = lane_at(global_at<float>(a.zbias, h * dim), kc), rate = WKV ? 0.f : same(a.rate, h);
  const float nw = lane_at(global_at<float>(a.norm_w, WKV ? h * vdim : 0), one_of(tid));
  float bonus = 0.f;
  if constexpr (WKV) bonus = lane_at(global_at<float>(a.u, h * dim), kc);

  const int64_t hsz = (int64_t)dim * vdim;
  const uint32_t step = 8 * vdim, at = state_of(tid);
  f4 st[KR];
  if (code >= 0 && pos > 0) {
    auto rd = global_at<float>(a.state, (((int64_t)(code & 1) * a.slots + (code >> 1)) * H + h) * hsz);
#pragma unroll
    for (int i = 0; i < KR; ++i) st[i] = *(glob<f4>*)((glob<char>*)(rd + i * step) + at);
  } else {
#pragma unroll
    for (int i = 0; i < KR; ++i) st[i] = (f4){0.f, 0.f, 0.f, 0.f};
  }

#pragma unroll 1
  for (int row = t0;;) {
    if (tid < dim) {
      const int me = fresh(), put = (me & 7) * RS + (me >> 3);
      float d = up(rz) + zbias;
      if constexpr (WKV) d = exp_c(-exp_c(d > 80.f ? 80.f : d));
      else d = exp_c(-rate * softplus_c(zsign * d));
      ops[0][put] = d;
      ops[1][put] = up(rk);
      ops[2][put] = up(rq);
      if constexpr (WKV) ops[3][put] = up(rq) * up(rk) * bonus;
    }
    const f4 v = rv.get();
    const TG g = rg;
    const float beta = DELTA ? sigmoid_c(up(rb)) : 1.f;
    __syncthreads();
    auto operand = [&](int which, int x) { return *reinterpret_cast<const f4*>(&ops[which][kg * RS + x]); };
    f4 u = v, o = {0.f, 0.f, 0.f, 0.f};
    float own = 0.f;                                      // wkv: what the token reads of itself
    if constexpr (DELTA) {
      f4 sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int x = 0; x < KR; x += 4) {
        const f4 d = operand(0, x), k = operand(1, x);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          st[x + e] *= d[e];
          sum += st[x + e] * k[e];
        }
        __builtin_amdgcn_sched_barrier(0);                // four channels' operands at a time: registers
      }
      u = beta * (v - keys_sum(sum));
    }
#pragma unroll
    for (int x = 0; x < KR; x += 4) {
      const f4 k = operand(1, x), q = operand(2, x);
      f4 d, bonus4;
      if constexpr (!DELTA) d = operand(0, x);
      if constexpr (WKV) bonus4 = operand(3, x);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if constexpr (WKV) {
          o += q[e] * st[x + e];
          own += bonus4[e];
          st[x + e] = d[e] * st[x + e] + k[e] * v;
        } else {
          if constexpr (DELTA) st[x + e] += k[e] * u;
          else st[x + e] = d[e] * st[x + e] + k[e] * u;
          o += st[x + e] * q[e];
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    o = keys_sum(o);
    if constexpr (WKV) o += keys_sum(own) * v;
    else o *= q_scale;
    float ss = live ? (o[0] * o[0] + o[1] * o[1]) + (o[2] * o[2] + o[3] * o[3]) : 0.f;
    ss = group_sum(ss, 8);
    if (lane == 0) part[wave] = ss;
    __syncthreads();
    if (kg < 4 && live) {
      ss = part[0];
#pragma unroll 1
      for (int w = 1; w < (int)(blockDim.x >> 6); ++w) ss += part[w];
      const float even = kg & 2 ? o[2] : o[0], odd = kg & 2 ? o[3] : o[1], x = kg & 1 ? odd : even, y = up(g);
      const float act = (sigmoid ? 1.0f : y) / (1.0f + expf(-y));
      TG out;
      stf(&out, x / sqrtf(ss / (float)vdim + eps) * nw * act);
      ((__attribute__((address_space(1))) TG*)(uintptr_t)(static_cast<TG*>(a.out) + (int64_t)row * a.os + h * vdim))[one_of(fresh())] = out;
    }
    if (++row == t0 + n) break;
    __syncthreads();                                      // LDS is read before the next token's
    fetch(row);
  }
  if (code >= 0 && live) {
    const uint32_t at = state_of(fresh());
    auto wr = (__attribute__((address_space(1))) float*)(uintptr_t)(
        a.state + (((int64_t)(1 - (code & 1)) * a.slots + (code >> 1)) * H + h) * hsz);
#pragma unroll
    for (int i = 0; i < KR; ++i) __builtin_nontemporal_store(st[i], (__attribute__((address_space(1))) f4*)((__attribute__((address_space(1))) char*)(wr + i * step) + at));
  }
}

// ------------------------------------------------------------------ launcher
// Steps with a run entry for every row: decode rows, and captured steps with extends of up to 32 rows, whose other entries
// are missing (-1).  The next row's operands are not on their way while a row is made (registers), and a longer run still
// takes half the time that a value channel a thread takes with them on their way, one run of 32 rows, 32 heads of 64 x 128:
// delta rule 99 -> 51 us, gla 99 -> 41, wkv (64 heads of 64 x 64) 83 -> 39; one of eight rows and 24 of one 36 -> 20, 36 -> 18,
// 30 -> 18; other sizes 0.4 - 0.7 of the time.
bool state_rows_ok(int mode, bool in_f32, int T, const StateRows& a) {
  if (T > 1 && (a.run_rows == nullptr || a.runs < T)) return false;
  if (mode == kChunkWkv ? a.dim != 64 : a.dim != 32 && a.dim != 64 && a.dim != 128) return false;
  return a.vdim % 4 == 0 && a.vdim <= 256 && reinterpret_cast<uintptr_t>(a.state) % 16 == 0 &&
         reinterpret_cast<uintptr_t>(a.v) % (in_f32 ? 16 : 8) == 0 && a.vs % 4 == 0;
}

template <typename TI, typename TG, int KR, int MODE>
static void launch_state_rows_one(const StateRows& a, hipStream_t s) {
  const int waves = std::max((a.vdim + 31) / 32, (a.dim + 63) / 64);
  hipLaunchKernelGGL((state_rows_kernel<TI, TG, KR, MODE>), dim3(a.H, std::min(a.runs, 65535), (a.runs + 65534) / 65535),
                     dim3(64 * waves), 0, s, a);
}
template <typename TI, typename TG>
static void launch_state_rows_types(int mode, const StateRows& a, hipStream_t s) {
  if (mode == kChunkGla) {
    if (a.dim == 32) launch_state_rows_one<TI, TG, 4, kChunkGla>(a, s);
    else if (a.dim == 64) launch_state_rows_one<TI, TG, 8, kChunkGla>(a, s);
    else launch_state_rows_one<TI, TG, 16, kChunkGla>(a, s);
  } else if (mode == kChunkDelta) {
    if (a.dim == 32) launch_state_rows_one<TI, TG, 4, kChunkDelta>(a, s);
    else if (a.dim == 64) launch_state_rows_one<TI, TG, 8, kChunkDelta>(a, s);
    else launch_state_rows_one<TI, TG, 16, kChunkDelta>(a, s);
  } else if constexpr (sizeof(TI) == sizeof(TG)) {
    launch_state_rows_one<TI, TG, 8, kChunkWkv>(a, s);
  }
}

void launch_state_rows(int mode, bool in_f32, bool act_f32, const StateRows& a, hipStream_t s) {
  if (in_f32 && act_f32) launch_state_rows_types<float, float>(mode, a, s);
  else if (in_f32) launch_state_rows_types<float, bf16_t>(mode, a, s);
  else if (!act_f32) launch_state_rows_types<bf16_t, bf16_t>(mode, a, s);
  else launch_state_rows_types<bf16_t, float>(mode, a, s);
}

}  // namespace rfqmix
