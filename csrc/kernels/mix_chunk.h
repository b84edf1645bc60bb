// Arguments of the chunked linear recurrences (mix_chunk.hip), shared by their launchers.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace rfqmix {

constexpr int kChunkDim = 64;          // most key channels
constexpr int kChunkRows = 16;         // tokens of a chunk
enum ChunkMode { kChunkWkv = 0, kChunkGla = 1, kChunkDelta = 2 };

struct ChunkArgs {
  const void *q, *k, *v;            // rows of H / rep heads of dim (q, k), H heads of vdim (v)
  int64_t qs, ks, vs;
  const void* z;                    // decay logits [T, H dim]: fp32, wkv: of q's type
  int64_t zs;
  const float *rate, *zbias;        // [H] (not wkv), [H dim]
  float zsign;
  const void* beta;                 // [T, H] logits (delta rule)
  int64_t bs;
  const float* u;                   // [H, dim] bonus (wkv)
  const void* gate;                 // wkv only: [T, H vdim] and norm_w [H vdim]; the others leave
  int64_t gs;                       // norm and gate to the caller's kernel
  const float* norm_w;
  float eps, q_scale;
  float* raw;                       // [T, H vdim] read-outs (not wkv)
  void* out;                        // [T, H vdim] contiguous (wkv)
  float* state;                     // [2 slots, H, dim, vdim]
  const int32_t *row_state, *row_back, *row_fwd, *pos, *run_rows;
  int runs, H, rep, dim, vdim, slots;
  int min_run;                      // shorter runs are left alone
  int cap = 0, per = 0, unit = 0;   // segments of runs that the step is shared in at most (0: whole runs), workgroups of
                                    // each, and what divides their rows
  float* seg = nullptr;             // scratch of cap segments: [cap, H, dim, vdim] what a segment's rows leave of a state of
                                    // zeros, then [cap, H, dim] products of its decays (delta rule: see delta_seg)
};

// How a step of T rows is shared: runs of at least this many rows go to the chunked kernel, the
// others to the token-by-token one (1: all in chunks, INT32_MAX: none).
int chunk_min_run(int mode, int T, const ChunkArgs& a);
// Segments that the step's runs are shared in at most where they are, else 0 (sets a.per and a.unit), and the scratch floats
// of a.cap.
int chunk_seg_cap(int mode, bool in_f32, int T, ChunkArgs& a);
int64_t chunk_seg_floats(int mode, const ChunkArgs& a);
// Whether the kernels may cut a run: the device's choice of segments and the launches that it needs go by this alone.
__host__ __device__ inline bool chunk_may_cut(const ChunkArgs& a) { return a.cap > a.runs; }
// in_f32: q, k, v (and wkv's z, gate, out) are fp32, else bf16; act_f32: beta's type.
// T: rows of the step.
void launch_chunk(int mode, bool in_f32, bool act_f32, int T, const ChunkArgs& a, hipStream_t s);

}  // namespace rfqmix
