// Arguments of the gated linear recurrence's launcher (mix_linrec.hip), shared with the
// bindings.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <functional>

namespace rfqmix {

struct LinrecArgs {
  const void *q, *k, *v;            // [T, Hq, dim] x2, [T, H, vdim]; row strides below
  int64_t qs, ks, vs;
  const float* z;                   // decay logits [T, H dim]
  int64_t zs;
  const float *rate, *zbias;        // [H], [H dim]
  float zsign;
  const void* beta;                 // [T, H] logits (delta rule) or null
  int64_t bs;
  const void* gate;                 // [T, H vdim]
  int64_t gs;
  int gate_sigmoid;
  const float* norm_w;              // [vdim]
  float eps, q_scale;
  float* raw;                       // [T, H vdim] fp32 scratch or null: read-outs before norm and gate
  float* state;                     // [2 slots, H, dim, vdim]
  const int32_t *row_state, *row_back, *row_fwd, *pos, *run_rows;
  int runs;
  void* out;                        // [T, H vdim], row stride os
  int64_t os;
  int T, H, rep, dim, vdim, slots;
  int below = INT32_MAX;            // the token-by-token kernel leaves longer runs to the chunked one
};

// Runs of fewer than `below` rows, token by token with the state in registers (mix_state_rows.hip).
struct StateRows {
  const void *q, *k, *v, *z, *beta, *gate;             // as in LinrecArgs; wkv: r, k, v and z of one type
  int64_t qs, ks, vs, zs, bs, gs;
  const float *rate, *zbias, *u, *norm_w;              // u: wkv's bonus; norm_w [vdim], wkv: [H vdim]
  float* state;
  const int32_t *row_state, *row_back, *row_fwd, *pos, *run_rows;
  int runs;                                            // without run_rows: rows of the step
  void* out;
  int64_t os;
  int H, rep, dim, vdim, slots, below, gate_sigmoid;
  float zsign, eps, q_scale;
};
bool state_rows_ok(int mode, bool in_f32, int T, const StateRows& a);      // mode: ChunkMode; T rows in the step
void launch_state_rows(int mode, bool in_f32, bool act_f32, const StateRows& a, hipStream_t s);

bool linrec_ok(int dim, int vdim);
// scratch(n): n floats that stay until the launches are queued
void launch_gated_linrec(bool in_f32, bool act_f32, bool delta, const LinrecArgs& a,
                         const std::function<float*(int64_t)>& scratch, hipStream_t s);

}  // namespace rfqmix
