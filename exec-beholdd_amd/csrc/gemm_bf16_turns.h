// Matrix products of many rows in which two groups of waves take turns: see gemm_bf16_turns.hip.
#pragma once
#include "common.h"

// Tiles of 256 rows x 32 `blocks` weight rows (8 or 6).  The activations lie in blocks of 16 rows x 32 columns (bh_blocked_index), in a
// buffer of whole tiles of 256 rows.  mode 0: bfloat16; 1: float32, added to what is there if `accumulate`, or with `parts` of K the
// bare sums [part][M][N]; 2: gated (the gate as `form` says), N bfloat16 outputs; 3: bfloat16, squared behind a ReLU.  c_blocked (mode 2
// and 3): the output in blocks of 16 rows.
bool gemm_turns_can(int M, int N, int K, int mode, int blocks, int parts);
int gemm_turns_launch(const void* a, const void* w, void* c, int mode, int accumulate, int M, int N, int K, int blocks, int parts,
                      int c_blocked, GateForm form, hipStream_t stream);
