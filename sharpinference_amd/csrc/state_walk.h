// Matrix-valued recurrent states with one scalar decay per (token, head): what the token-by-token walk
// (state_walk.hip) and the chunk form of long entries (state_chunk.hip) share.  The recurrences and the
// layout of a state are described in state_walk.hip.
#pragma once
#include "common.h"

enum : int { WALK_EXP_GATES = 0, WALK_STATE_SPACE = 1, WALK_FIXED_DECAY = 2 };
constexpr int kWalkCols = 8;       // value columns of a slice
constexpr float kWalkFloor = 1e-6f;

// floats of a slice: S, then (exponential gates) n and 8 floats that begin with m
static inline __host__ __device__ int walk_slice_floats(int dkp, int mode) {
  return (dkp / 8) * 64 + (mode == WALK_EXP_GATES ? dkp + 8 : 0);
}

__device__ __forceinline__ float softplus_f32(float x) { return fmaxf(x, 0.f) + log1pf(expf(-fabsf(x))); }
__device__ __forceinline__ float log_sigmoid_f32(float x) { return fminf(x, 0.f) - log1pf(expf(-fabsf(x))); }

struct WalkArgs {
  const void* proj; int stride, q_off, k_off, v_off, heads_per_group;
  const float* gates; int gate_stride; const float *p0, *p1, *p2;
  float cap, q_scale; float* state; const int *state_slots, *cu_tokens; float* out;
  int n_entries, nh, dk, dv;
  const int *segs, *ent_segs; int n_segs, n_scratch, n_long; float *seg_local, *seg_start, *seg_decay;
  const int* positions; const float* inv_freq; int rot_dim; float k_scale;      // WALK_FIXED_DECAY
};

// The segments' first and last pass in chunk form (state_chunk.hip), for the sizes state_chunk_takes names; entries
// of fewer than kChunkFrom tokens are left out and walked (a.n_long: the leading segments of all others).
constexpr int kChunkFrom = 32;
constexpr int kSeg = 128;          // tokens of a segment at most (the lists are cut to it: a chunk's LDS holds no more)
bool state_chunk_takes(const WalkArgs& a, int dtype);
int state_chunk_local(const WalkArgs& a, int dtype, int mode, hipStream_t stream);
int state_chunk_final(const WalkArgs& a, int dtype, int mode, hipStream_t stream);
