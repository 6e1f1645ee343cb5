// A sequence of many rows that a recurrence walks in chunks side by side: what the later chunks' rows owe the state their chunk
// started from, which is linear in that state, is added once the chunks' states are joined.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <type_traits>

// out[row][head] += S_in(the row's chunk)^T (the row's carried query), for the rows of every chunk but a sequence's first.  states
// [n_seqs][chunk_count][H][dim][vdim]: the state every chunk started from; queries [rows][H][dim]; out [rows][H * vdim]; all float32.
int bh_chunk_carry(const float* states, const float* queries, int chunk_rows, int chunk_count, const int32_t* seq_start, float* out, int n_seqs,
                   int H, int dim, int vdim, hipStream_t stream);

// x of the lane whose number differs in the bits of a group of 2, 4, 8 or 16 neighbours, added: all lanes of the group end with the sum
template <int SL>
__device__ inline float slices_sum(float x) {
  auto moved = [](float v, auto ctrl) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), decltype(ctrl)::value, 0xf, 0xf, false));
  };
  if constexpr (SL >= 2) x += moved(x, std::integral_constant<int, 0xB1>());      // neighbours swapped
  if constexpr (SL >= 4) x += moved(x, std::integral_constant<int, 0x4E>());      // pairs swapped
  if constexpr (SL >= 8) x += moved(x, std::integral_constant<int, 0x141>());     // halves of a row of 16 lanes mirrored
  if constexpr (SL >= 16) x += moved(x, std::integral_constant<int, 0x140>());    // rows mirrored
  return x;
}
