// bfloat16 products of up to 32 rows from packed weights (tiles layout of gemm_bf16.hip) and activations in blocks of 8 or 16 rows:
// C[M, N] (+)= A[M, K] * W[N, K]^T, plain or gated, with the RMSNorm before and after it riding on it (gemm_bf16_few.h).
//
// Bound by reading W once, and for small W by the chain of a launch: 1.7 us of the launch itself, a trip to memory, the sum over the
// waves.  A workgroup owns `span` rows of W (gated: as many pairs); its eight waves take the 64-wide chunks of k in turn and feed
// v_mfma_f32_16x16x32_bf16 with W as the row operand and the activations as the column operand; the waves' tiles are summed through
// LDS in a fixed order.
//
// The chunks go through DEPTH sets of registers, each asked for again as soon as it is multiplied, so that a wave has loads in flight
// all the time and its last chunks are no trips of their own (asked for in bursts of four, and one by one where fewer were left, 3,072
// gated outputs of k of 1,024 took 6.0 us a launch instead of 4.8).  Two sets, four where only a part of a block's rows is loaded:
// more of them bring nothing for few workgroups and cost the others their second and third workgroup on a compute unit (gated
// 12,288 x 4,096 at 8 rows 32.1 us with two, 34.4 with four).  A chunk's activations are asked for before its weights: they come from the
// L2 and are there when the weights are (4,096 x 2,048 5.2 -> 5.0 us).
//
// Which rows (gemm_few_rows), us at 8 / 16 rows:
//   16, the block of the layout.
//   8 where blocks of 16 leave half of the compute units idle and k is 1,536 or more (2,048 x 6,144 8.2 / 9.9 -> 7.2 / 8.5, 1,024 x
//   3,072 5.2 / 5.9 -> 5.0 / 5.3; 1,024 x 1,024 3.5 -> 3.7: there the launch is the time).  At 17 to 32 rows too, where the blocks of
//   16 went in bursts (32 rows: 2,048 x 2,048 5.2 -> 5.1, 1,024 x 3,072 6.9 -> 6.2, 2,048 x 6,144 11.3 -> 10.8, 512 x 12,288 18.4 ->
//   17.6, 2,048 x 12,288 21.0 -> 20.0; the least is 512 x 2,048 with 4.7 -> 4.75).  Both halves of a block are whole cache lines.
//   20 or 24 where the blocks of 16 are more than the compute units and fewer than twice as many: otherwise some compute units carry
//   two blocks, the others one, and the product takes as long as one of twice the compute units' blocks.
#include "gemm_bf16_few.h"

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));

#define MFMA16(a, b, c) __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0)

// every lane's value of the lane eight further on in its group of 16 (lanes 8 to 15: nothing that matters)
__device__ inline u32x4_t from_lane_plus_8(u32x4_t v) {
  u32x4_t out;
#pragma unroll
  for (int word = 0; word < 4; ++word)
    out[word] = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v[word], 0x108 /* row_shl:8 */, 0xf, 0xf, true);
  return out;
}

#define FEW_WAVES 8
// MB: blocks of 16 activation rows, which lie in blocks of XB rows.  NB: blocks of W that a span touches; MASKED: it is not the whole of
// one.  SHORT: no wave has more than DEPTH chunks.  GATED: 1, or 2 with a clamped gate (gate_mul).
template <int MB, typename TC, int XB, int NB, int GATED, bool MASKED, int DEPTH, bool SHORT>
__global__ __launch_bounds__(FEW_WAVES * 64) void gemm_few_kernel(const uint16_t* __restrict__ a, const uint16_t* __restrict__ w,
                                                                  TC* __restrict__ c, int M, int N, int K, int accumulate, int span,
                                                                  RidingNorm norm, RowBlocks blocks, GateForm form) {
  constexpr int WAVES = FEW_WAVES, T = NB * (GATED ? 2 : 1);
  __shared__ float partial[WAVES][T][MB][256];
  __shared__ float row_factor[MB * 16];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), lane = threadIdx.x % 64;
  const int i = lane % 16, g = lane / 16;
  const int full = K / 64, left = (full - wave + WAVES - 1) / WAVES;   // 64-wide chunks of k, and how many of them are this wave's
  // workgroups go to the XCDs in turn: the ones of an XCD own a run of neighbouring spans
  const int owner = gridDim.x % 8 == 0 ? (int)(blockIdx.x % 8) * (int)(gridDim.x / 8) + (int)(blockIdx.x / 8) : (int)blockIdx.x;
  const int first_row = owner * span, first_tile = first_row / 16;
  int lo[NB], hi[NB];   // the rows of each block that this workgroup owns: lo <= row < hi (none: hi <= lo)
  const uint16_t* wp[T];
#pragma unroll
  for (int t = 0; t < NB; ++t) {
    const int tile_row = (first_tile + t) * 16;
    lo[t] = MASKED ? max(first_row, tile_row) - tile_row : 0;
    hi[t] = MASKED ? min(min(first_row + span, N), tile_row + 16) - tile_row : 16;
    const int tile = NB == 1 ? first_tile : min(first_tile + t, N / 16 - 1);   // (a block beyond the matrix is never loaded; its address stays inside)
    wp[t] = w + (size_t)tile * full * 1024;
    if (GATED) wp[NB + t] = w + (size_t)(tile + N / 16) * full * 1024;
  }
  // A lane without a row of its own in a block loads nothing; or, where all of a wave's chunks are asked for at once, what the lane of the
  // nearest owned row does, which brings no line more and goes nowhere: each load under a branch of its own costs more there (2,048 x
  // 2,048 at 8 / 16 / 32 rows 4.1 / 4.4 / 5.3 us, 3.8 / 4.1 / 5.1 so).  In turn it is the other way round (2,048 x 12,288 at 32 rows
  // 20.0 us, 20.7 so).
  constexpr bool SWITCHED = MASKED && !SHORT;
  bool mine[NB];
  int place[NB];
#pragma unroll
  for (int t = 0; t < NB; ++t) {
    mine[t] = i >= lo[t] && i < hi[t];
    place[t] = 8 * (MASKED && SHORT ? 16 * g + max(min(i, hi[t] - 1), lo[t]) : lane);
  }
  // A lane's two pieces of a chunk are the pieces 2 g and 2 g + 1 of its two 32-wide steps (bh_rows_index): 16 lanes read 256
  // neighbouring bytes; of blocks of 8 rows 128, and lanes 8 to 15 take the second piece of rows 0 to 7, which lies right behind the
  // first ones, so that one load brings both and a lane move hands the second to the lane of its row.
  constexpr int x_half = XB ? XB * 8 : 8, x_chunk = XB ? 64 * XB : 64;
  const uint16_t* xp[MB];
#pragma unroll
  for (int b = 0; b < MB; ++b) {
    if constexpr (XB) xp[b] = a + (size_t)(b * 16 / XB) * (K / 32) * (32 * XB) + (g / 2) * (32 * XB) + ((2 * g) % 4 * XB + i) * 8;
    else xp[b] = a + (size_t)min(b * 16 + i, M - 1) * K + g * 16;
  }

  f32x4_t acc[T][MB];
#pragma unroll
  for (int t = 0; t < T; ++t)
#pragma unroll
    for (int b = 0; b < MB; ++b) acc[t][b] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  u32x4_t wv[DEPTH][T][2], xv[DEPTH][MB][2];
  const u32x4_t zero = {0u, 0u, 0u, 0u};
  auto ask = [&](int u, int n) {   // the wave's n-th chunk
    const int at = wave + n * WAVES;
#pragma unroll
    for (int b = 0; b < MB; ++b) {
      const uint16_t* p = xp[b] + (size_t)at * x_chunk;
      xv[u][b][0] = *reinterpret_cast<const u32x4_t*>(p);
      if (XB != 8) xv[u][b][1] = *reinterpret_cast<const u32x4_t*>(p + x_half);
    }
#pragma unroll
    for (int t = 0; t < T; ++t) {
      if (NB > 1 && SHORT && hi[t % NB] <= lo[t % NB]) continue;   // the same for the whole workgroup
      const uint16_t* p = wp[t] + (size_t)at * 1024;
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const u32x4_t* from = reinterpret_cast<const u32x4_t*>(p + h * 512 + place[t % NB]);
        wv[u][t][h] = (!SWITCHED || mine[t % NB]) ? __builtin_nontemporal_load(from) : zero;
      }
    }
  };
  auto multiply = [&](int u) {
#pragma unroll
    for (int b = 0; b < MB; ++b) {
      if (XB == 8) xv[u][b][1] = from_lane_plus_8(xv[u][b][0]);
#pragma unroll
      for (int t = 0; t < T; ++t) {
        if (NB > 1 && hi[t % NB] <= lo[t % NB]) continue;   // the same for the whole workgroup
        acc[t][b] = MFMA16(wv[u][t][0], xv[u][b][0], acc[t][b]);
        acc[t][b] = MFMA16(wv[u][t][1], xv[u][b][1], acc[t][b]);
      }
    }
  };

  // The norm ahead: 32 threads per row, each with every 32nd partial sum, of which the first 256 of a row are asked for before they
  // are needed.
  constexpr int ROWS_PER_PASS = WAVES * 2, PASSES = (MB * 16 + ROWS_PER_PASS - 1) / ROWS_PER_PASS;
  const int part = threadIdx.x % 32;
  float early[PASSES][8];
  // What a float32 output holds before this product adds to it, and the weight of the norm behind: a thread knows the elements that it
  // will write (the residual was written on other XCDs: it comes from beyond this one's L2).
  constexpr int OUT_PASSES = (MB * 256 + WAVES * 64 - 1) / (WAVES * 64);
  constexpr bool OUT_EARLY = !GATED && sizeof(TC) == 4;
  float before[OUT_PASSES][NB], behind_gain[OUT_PASSES][NB];
  auto ask_beside = [&]() {
    if (OUT_EARLY) {
#pragma unroll
      for (int pass = 0; pass < OUT_PASSES; ++pass)
#pragma unroll
        for (int t = 0; t < NB; ++t) {
          const int e = threadIdx.x + pass * WAVES * 64;
          const int m = e / 256 * 16 + (e % 256) / 16, column = e % 16, n = (first_tile + t) * 16 + column;
          const bool valid = e < MB * 256 && m < M && column >= lo[t] && column < hi[t];
          before[pass][t] = (valid && accumulate) ? reinterpret_cast<const float*>(c)[(size_t)m * N + n] : 0.f;
          behind_gain[pass][t] = 0.f;
          if (valid && norm.behind_weight)
            behind_gain[pass][t] = norm.behind_weight_f32 ? reinterpret_cast<const float*>(norm.behind_weight)[n]
                                                          : bf16_bits_to_f32(reinterpret_cast<const uint16_t*>(norm.behind_weight)[n]);
        }
    }
  };

  auto find_factor = [&]() {
  if (norm.ahead_ss) {
#pragma unroll
    for (int pass = 0; pass < PASSES; ++pass) {
      const int r = pass * ROWS_PER_PASS + threadIdx.x / 32;
      float ss = 0.f;
#pragma unroll
      for (int u = 0; u < 8; ++u) ss += early[pass][u];
      if (r < M)
        for (int block = part + 256; block < norm.ahead_blocks; block += 32) ss += norm.ahead_ss[(size_t)r * norm.ahead_blocks + block];
#pragma unroll
      for (int off = 16; off > 0; off >>= 1) ss += __shfl_xor(ss, off, 64);
      if (part == 0 && r < MB * 16) row_factor[r] = (r < M) ? 1.0f / sqrtf(ss / (float)K + norm.ahead_eps) : 0.f;
    }
  }
  };
  auto ask_norm = [&]() {
    if (norm.ahead_ss) {
#pragma unroll
      for (int pass = 0; pass < PASSES; ++pass) {
        const int r = pass * ROWS_PER_PASS + threadIdx.x / 32;
#pragma unroll
        for (int u = 0; u < 8; ++u) {
          const int block = part + 32 * u;
          early[pass][u] = (r < M && block < norm.ahead_blocks) ? norm.ahead_ss[(size_t)r * norm.ahead_blocks + block] : 0.f;
        }
      }
    }
  };
  if constexpr (SHORT) {   // everything at once
#pragma unroll
    for (int u = 0; u < DEPTH; ++u)
      if (u < left) ask(u, u);
    ask_norm();
    ask_beside();
#pragma unroll
    for (int u = 0; u < DEPTH; ++u)
      if (u < left) multiply(u);
    find_factor();
  } else {                 // (every wave has DEPTH chunks or more)
    ask_norm();
#pragma unroll
    for (int u = 0; u < DEPTH; ++u) ask(u, u);
    ask_beside();
    find_factor();         // while the first chunks are on their way
    int n = 0;
    for (; n + 2 * DEPTH <= left; n += DEPTH)
#pragma unroll
      for (int u = 0; u < DEPTH; ++u) {
        multiply(u);
        ask(u, n + DEPTH + u);
      }
#pragma unroll
    for (int u = 0; u < DEPTH; ++u) {
      multiply(u);
      if (n + DEPTH + u < left) ask(u, n + DEPTH + u);
    }
#pragma unroll
    for (int u = 0; u < DEPTH; ++u)
      if (n + DEPTH + u < left) multiply(u);
  }

  // D: lane holds column (activation row) i and rows (W rows) 4g..4g+3 of each block; lay it out as [m][n]
#pragma unroll
  for (int t = 0; t < T; ++t)
#pragma unroll
    for (int b = 0; b < MB; ++b)
      *reinterpret_cast<f32x4_t*>(&partial[wave][t][b][i * 16 + 4 * g]) = acc[t][b];
  __syncthreads();
#pragma unroll
  for (int pass = 0; pass < OUT_PASSES; ++pass) {
    const int e = threadIdx.x + pass * WAVES * 64;
    if (e >= MB * 256) break;   // whole waves enter or stay out
    const int b = e / 256, m = b * 16 + (e % 256) / 16, column = e % 16;
    float sq = 0.f;   // of what this workgroup adds to row m of the residual (norm.behind_weight)
#pragma unroll
    for (int t = 0; t < NB; ++t) {
      const int n = (first_tile + t) * 16 + column;
      const bool valid = m < M && column >= lo[t] && column < hi[t];
      float sum[GATED ? 2 : 1];
#pragma unroll
      for (int k = 0; k < (GATED ? 2 : 1); ++k) {
        sum[k] = 0.f;
#pragma unroll
        for (int v = 0; v < WAVES; ++v) sum[k] += partial[v][k * NB + t][b][e % 256];
        if (norm.ahead_ss) sum[k] *= row_factor[m];
      }
      if (!valid) continue;
      if constexpr (GATED) {
        c[bh_rows_index(blocks.c, m, n, N)] = from_f32<TC>(gate_mul<GATED == 2>(sum[0], sum[GATED ? 1 : 0], form));
      } else if constexpr (OUT_EARLY) {
        const float value = accumulate ? before[pass][t] + sum[0] : sum[0];
        c[(size_t)m * N + n] = value;
        if (norm.behind_weight) {
          sq += value * value;
          norm.behind_rows[bh_rows_index(blocks.behind, m, n, N)] = f32_to_bf16_bits(value * behind_gain[pass][t]);
        }
      } else if (form.squared) {
        c[bh_rows_index(blocks.c, m, n, N)] = from_f32<TC>(relu_squared(sum[0]));
      } else {
        const size_t at = (size_t)m * N + n;
        c[at] = from_f32<TC>(accumulate ? sum[0] + to_f32(c[at]) : sum[0]);
      }
    }
    if (OUT_EARLY && norm.behind_weight) {
      sq += __shfl_xor(sq, 8, 64);   // the 16 columns of a row sit in 16 neighbouring lanes
      sq += __shfl_xor(sq, 4, 64);
      sq += __shfl_xor(sq, 2, 64);
      sq += __shfl_xor(sq, 1, 64);
      if (column == 0 && m < M) norm.behind_ss[(size_t)m * gridDim.x + blockIdx.x] = sq;
    }
  }
}

int gemm_few_rows(int N, int K, bool gated) {
  if (gated) return 16;
  const int tiles = N / 16, units = bh_compute_units();
  if (2 * tiles <= units && K >= 1536) return 8;
  if (tiles > units && tiles < 2 * units)
    for (int rows = 20; rows <= 24; rows += 4)   // (28 rows can lie in three blocks: 7168 x 5120 at 8 rows 14.6 -> 17.1 us)
      if (N % rows == 0 && N / rows <= units) return rows;
  return 16;
}

// The bursts of four chunks are left: many workgroups a compute unit, where what counts is the bytes asked for at once (us, bursts / here:
// 32,768 x 4,096 at 16 rows 46.2 / 46.6, gated 17,408 x 5,120 59.9 / 60.6), and long k at 17 to 32 rows, whose chunks are two loads of W
// and four of the activations (4,096 x 12,288 at 32 rows 24.3 / 26.4; 4,096 x 2,048 7.3 / 6.3).
bool gemm_few_takes(int M, int N, int K, bool gated) {
  if (gemm_few_rows(N, K, gated) != 16) return true;
  const bool many = N / 16 > 4 * bh_compute_units();
  if (gated) return !many || M > 16;
  return !many && (M <= 16 || K <= 2048);
}

template <int MB, typename TC, int XB, int NB, int GATED, bool MASKED, int DEPTH>
static void launch_depth(const void* a, const void* w, void* c, int accumulate, int M, int N, int K, int span, const RidingNorm& norm,
                         const RowBlocks& blocks, GateForm form, hipStream_t stream) {
#define BH_FEW(SHORT)                                                                                                      \
  gemm_few_kernel<MB, TC, XB, NB, GATED, MASKED, DEPTH, SHORT><<<N / span, FEW_WAVES * 64, 0, stream>>>(                   \
      (const uint16_t*)a, (const uint16_t*)w, (TC*)c, M, N, K, accumulate, span, norm, blocks, form)
  if (K / 64 <= DEPTH * FEW_WAVES) BH_FEW(true);
  else BH_FEW(false);
#undef BH_FEW
}

template <int MB, typename TC, int XB>
static void launch_rows(const void* a, const void* w, void* c, int accumulate, int M, int N, int K, int gated, const RidingNorm& norm,
                        const RowBlocks& blocks, GateForm form, hipStream_t stream) {
  const int span = gemm_few_rows(N, K, gated);
#define BH_FEW(...) launch_depth<MB, TC, XB, __VA_ARGS__>(a, w, c, accumulate, M, N, K, span, norm, blocks, form, stream)
  if constexpr (sizeof(TC) == 2) {
    if (gated == GATED_CLAMPED) {
      BH_FEW(1, 2, false, 2);
      return;
    }
  }
  if (gated) BH_FEW(1, 1, false, 2);
  else if (span == 16) BH_FEW(1, 0, false, 2);
  else if (span == 8) BH_FEW(1, 0, true, 4);
  else BH_FEW(2, 0, true, MB == 1 && sizeof(TC) == 4 ? 4 : 2);
#undef BH_FEW
}

int gemm_few_launch(const void* a, const void* w, void* c, bool f32, int accumulate, int M, int N, int K, int gated, const RidingNorm& norm,
                    const RowBlocks& blocks, GateForm form, hipStream_t stream) {
#define BH_FEW_ARGS a, w, c, accumulate, M, N, K, gated, norm, blocks, form, stream
  if (blocks.a == 0 && M <= 16) {
    if (f32) launch_rows<1, float, 0>(BH_FEW_ARGS);
    else launch_rows<1, bf16_t, 0>(BH_FEW_ARGS);
  } else if (blocks.a == 0) {
    if (f32) launch_rows<2, float, 0>(BH_FEW_ARGS);
    else launch_rows<2, bf16_t, 0>(BH_FEW_ARGS);
  } else if (blocks.a == 8) {
    if (f32) launch_rows<1, float, 8>(BH_FEW_ARGS);
    else launch_rows<1, bf16_t, 8>(BH_FEW_ARGS);
  } else if (M <= 16) {
    if (f32) launch_rows<1, float, 16>(BH_FEW_ARGS);
    else launch_rows<1, bf16_t, 16>(BH_FEW_ARGS);
  } else {
    if (f32) launch_rows<2, float, 16>(BH_FEW_ARGS);
    else launch_rows<2, bf16_t, 16>(BH_FEW_ARGS);
  }
#undef BH_FEW_ARGS
  return bh_check_launch("gemm_few");
}
