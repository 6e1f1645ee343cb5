// Matrix products of many rows through a ring of operand steps in LDS: see gemm_bf16_ring.hip.
#pragma once
#include "common.h"

// The tiles the kernel is compiled for, rows x weight rows; _HALVES: two groups of waves take half of k each.
enum RingTile { RING_128x128 = 0, RING_128x128_HALVES, RING_256x128, RING_256x192, RING_256x256, RING_TILES };
// How a product of these sizes runs: its tile (or -1: not with this kernel) and in how many parts of K (1: in one go; more: bare sums
// [part][M][N] for a finishing kernel, plain products only).  What a plain product writes says what parts cost it (see cost_us).
enum RingOutput { RING_F32 = 0, RING_GATED = 1, RING_BF16 = 2 };
struct RingPlan {
  int tile, parts;
  double us = 0.;      // the estimate it was chosen by
};
RingPlan gemm_ring_plan(int M, int N, int K, int layout, RingOutput output);
// The sums of a plain bfloat16 product left apart: its plan if that has parts, the two halves of k of a plan that adds them up itself;
// one part where neither.
RingPlan gemm_ring_bare_plan(int M, int N, int K, int layout);
// The activations lie in blocks of 16 rows x 32 columns (bh_blocked_index).  c_dtype BH_F32 (accumulate allowed) or BH_BF16 (no
// accumulate); activation 1 = gated, bfloat16 output only; form: what stands on its gate, or that a plain product squares its bfloat16
// output behind a ReLU; c_blocked: the output of either in blocks of 16 rows.
int gemm_ring_launch(const void* a, const void* w, void* c, int c_dtype, int accumulate, int M, int N, int K, int activation, int tile,
                     int c_blocked, GateForm form, hipStream_t stream);
int gemm_ring_launch_parts(const void* a, const void* w, float* sums, int M, int N, int K, const RingPlan& plan, hipStream_t stream);
