// Products of up to 32 rows from packed weights and activations in blocks: see gemm_bf16_few.hip.
#pragma once
#include "common.h"

// An RMSNorm between two products can ride on them (struct RidingNorm):
//   behind: the product that completes the float32 residual h also writes bfloat16(h[m][n] * g[n]) (the
//           norm's output but for the row factor) and, per workgroup, the sum of h[m][n]^2 over its
//           columns (those it owns in the kernels for few rows, 64 in the finishing kernel, a tile's width in whole tiles);
//   ahead:  the product that consumes the norm's output takes those unscaled rows as its activations and
//           multiplies its result by 1 / sqrt(sum of the partial sums / K + eps) of the row.
// The row factor commutes with the product, so the result is the norm's up to the rounding of the
// activations; the partial sums are added in a fixed order.  The kernels for few rows and whole tiles (with or
// without the finishing kernel) do this; the tiled kernel for every shape does not.
struct RidingNorm {
  const float* ahead_ss;   // [M][ahead_blocks] partial sums of squares for the rows of `a`, or null
  int ahead_blocks;
  float ahead_eps;
  const void* behind_weight;  // [N] norm weight for the rows this product completes, or null
  int behind_weight_f32;      // its element type: float32, else bfloat16
  uint16_t* behind_rows;      // [M][N] bfloat16 out
  float* behind_ss;           // [M][bh_gemm_bf16_norm_blocks()] out
};

// Rows per block (bh_rows_index in layout.h; 0: rows one after the other) of a product's bfloat16 matrices: its activations,
// its output (a gated one's, which the next product reads) and the rows it prepares for a norm behind it.
struct RowBlocks {
  int a, c, behind;
};

// How many weight rows (gated: pairs of them) a workgroup owns for N outputs, a multiple of 16.
int gemm_few_rows(int N, int K, bool gated);
// Whether the kernel is the better one for a product of up to 32 rows (N % 16 == 0, K % 64 == 0, W in the tiles layout): else the
// kernel of gemm_bf16.hip that asks for its chunks in bursts, with 16 weight rows a workgroup.
bool gemm_few_takes(int M, int N, int K, bool gated);
int gemm_few_launch(const void* a, const void* w, void* c, bool f32, int accumulate, int M, int N, int K, int gated, const RidingNorm& norm,
                    const RowBlocks& blocks, GateForm form, hipStream_t stream);
