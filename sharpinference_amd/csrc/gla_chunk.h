// The segments of gated linear attention as matrix products (gla_chunk.hip), for the launcher of the segmented walk.
#pragma once
#include "common.h"

struct GlaChunkArgs {
  const void* proj;
  int stride, q_off, k_off, v_off;
  const float* alpha;
  float q_scale;
  float* state;
  const int* state_slots;
  float* out;
  int nh;
  const int* segs;
  float *seg_state, *seg_decay;
};

// whether the kernels are compiled for these sizes and the operands lie on the borders of their 16-byte accesses
bool gla_chunk_takes(int dtype, int stride, int q_off, int k_off, int v_off, const GlaChunkArgs& a, int dk, int dv);
// final: the outputs and the entries' new states; else the segments' local states and decays
void gla_chunk_launch(int dtype, const GlaChunkArgs& a, int dk, int dv, int n_segs, bool final, hipStream_t stream);
