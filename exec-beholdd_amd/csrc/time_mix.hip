// What stands ahead of a wkv recurrence's products:
//   token_shift   from the rows h of a step, several mixes of every row with the row before it, out_s = h + (h' - h) * mu_s; h' is the
//                 row before in the row's sequence, or, for a sequence's first row of the step, what the sequence's slot keeps (zeros
//                 when a sequence starts), where the sequence's last row of the step is left for the next one
//   tanh_rows     out = tanh(x), float32 rows into the activation type
// The mixes are made in float32 from h as the activations hold it, and rounded once.
#include "attention_bf16.h"
#include "common.h"

#define TS_MOST 8        // mixes of a row

struct ShiftOuts {
  void* to[TS_MOST];
};

__device__ inline void ts_load8(float (&x)[8], const float* p) {
#pragma unroll
  for (int i = 0; i < 8; i += 4) {
    const float4 v = *reinterpret_cast<const float4*>(p + i);
    x[i] = v.x, x[i + 1] = v.y, x[i + 2] = v.z, x[i + 3] = v.w;
  }
}
__device__ inline void ts_load8(float (&x)[8], const bf16_t* p) {
  const u32x4_t v = *reinterpret_cast<const u32x4_t*>(p);
#pragma unroll
  for (int i = 0; i < 8; ++i) x[i] = bf16_bits_to_f32((uint16_t)(v[i / 2] >> (16 * (i % 2))));
}
__device__ inline void ts_store8(float* p, const float (&x)[8]) {
#pragma unroll
  for (int i = 0; i < 8; i += 4) *reinterpret_cast<float4*>(p + i) = float4{x[i], x[i + 1], x[i + 2], x[i + 3]};
}
__device__ inline void ts_store8(bf16_t* p, const float (&x)[8]) {
  u32x4_t v;
#pragma unroll
  for (int i = 0; i < 4; ++i) v[i] = pack_bf16(x[2 * i], x[2 * i + 1]);
  *reinterpret_cast<u32x4_t*>(p) = v;
}

// A thread takes eight neighbouring columns (16 bytes of them lie together in rows and in blocks alike) of one row at a time.  Where the
// mixes lie in blocks of rows, a wave's lanes are the 16-byte pieces of a block in their order, so that its stores (and its loads, where h
// lies in such blocks too) cover contiguous memory; otherwise they are neighbouring columns of a row.  Many rows: `turns` of them a thread.
// The thread of a sequence's first row reads what the slot keeps of these columns and then
// writes what it shall keep, to the row seq_to names (the same one or another).
template <typename T>
__global__ __launch_bounds__(256) void token_shift_kernel(const T* __restrict__ h, int h_block_rows, const float* __restrict__ mu, int mixes,
                                                          float* __restrict__ state, long slot_stride, const int32_t* __restrict__ row_seq,
                                                          const int32_t* __restrict__ seq_start, const int32_t* __restrict__ seq_slot, const int32_t* __restrict__ seq_to, ShiftOuts outs,
                                                          int out_block_rows, int n_rows, int width, int turns, int pieces) {
  const int piece = blockIdx.x * 256 + threadIdx.x;      // within a group of `apart` rows
  if (piece >= pieces) return;
  const int apart = out_block_rows ? out_block_rows : 1;
  const int column = out_block_rows ? piece / (4 * apart) * 32 + piece / apart % 4 * 8 : piece * 8, row_in = piece % apart;
  for (int turn = 0; turn < turns; ++turn) {
    const int row = (blockIdx.y * turns + turn) * apart + row_in;
    if (row >= n_rows) return;
    const int seq = row_seq[row], opens = seq_start[seq];
    float now[8], before[8];
    ts_load8(now, h + bh_rows_index(h_block_rows, row, column, width));
    if (opens == row) {
      const float* kept = state + (size_t)seq_slot[seq] * slot_stride + column;
      float* keeps = state + (size_t)seq_to[seq] * slot_stride + column;
      float last[8];
      ts_load8(last, h + bh_rows_index(h_block_rows, seq_start[seq + 1] - 1, column, width));
#pragma unroll
      for (int e = 0; e < 8; ++e) before[e] = kept[e];
#pragma unroll
      for (int e = 0; e < 8; ++e) keeps[e] = last[e];
    } else {
      ts_load8(before, h + bh_rows_index(h_block_rows, row - 1, column, width));
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) before[e] -= now[e];
    for (int s = 0; s < mixes; ++s) {
      float m[8], y[8];
      ts_load8(m, mu + (size_t)s * width + column);
#pragma unroll
      for (int e = 0; e < 8; ++e) y[e] = fmaf(before[e], m[e], now[e]);
      ts_store8((T*)outs.to[s] + bh_rows_index(out_block_rows, row, column, width), y);
    }
  }
}

// Any width, a thread an element.
template <typename T>
__global__ __launch_bounds__(256) void token_shift_plain_kernel(const T* __restrict__ h, const float* __restrict__ mu, int mixes,
                                                                float* __restrict__ state, long slot_stride, const int32_t* __restrict__ row_seq,
                                                                const int32_t* __restrict__ seq_start, const int32_t* __restrict__ seq_slot, const int32_t* __restrict__ seq_to,
                                                                ShiftOuts outs, int n_rows, int width) {
  const int column = blockIdx.x * 256 + threadIdx.x, row = blockIdx.y;
  if (column >= width) return;
  const int seq = row_seq[row];
  const float now = to_f32(h[(size_t)row * width + column]);
  float before;
  if (seq_start[seq] == row) {
    before = state[(size_t)seq_slot[seq] * slot_stride + column];
    state[(size_t)seq_to[seq] * slot_stride + column] = to_f32(h[(size_t)(seq_start[seq + 1] - 1) * width + column]);
  } else {
    before = to_f32(h[(size_t)(row - 1) * width + column]);
  }
  for (int s = 0; s < mixes; ++s)
    ((T*)outs.to[s])[(size_t)row * width + column] = from_f32<T>(fmaf(before - now, mu[(size_t)s * width + column], now));
}

// h [n_rows][width] (dtype; rows or blocks); mu f32 [mixes][width]; state: `width` floats a slot from state + slot * slot_stride; outs: `mixes`
// matrices like h.
extern "C" int bh_token_shift(const void* h, int dtype, int h_block_rows, const float* mu, int mixes, float* state, long slot_stride,
                              const int32_t* row_seq, const int32_t* seq_start, const int32_t* seq_slot, const int32_t* seq_to, void* const* outs, int out_block_rows,
                              int n_rows, int width, hipStream_t stream) {
  BH_REQUIRE(n_rows > 0 && width > 0, "token_shift: sizes must be positive");
  BH_REQUIRE(mixes >= 1 && mixes <= TS_MOST, "token_shift: 1 to %d mixes, not %d", TS_MOST, mixes);
  BH_REQUIRE(slot_stride >= width, "token_shift: a slot keeps a row of %d", width);
  const int blocks[2] = {h_block_rows, out_block_rows};
  for (int b : blocks)
    BH_REQUIRE(b == 0 || ((b == 8 || b == 16) && width % 32 == 0 && dtype == BH_BF16), "token_shift: rows in blocks of %d of width %d", b, width);
  ShiftOuts to = {};
  for (int s = 0; s < mixes; ++s) {
    BH_REQUIRE(outs[s] != nullptr, "token_shift: a matrix for every mix");
    to.to[s] = outs[s];
  }
  if (width % 8 == 0) {
    const int apart = out_block_rows ? out_block_rows : 1, pieces = width / 8 * apart, groups = (n_rows + apart - 1) / apart;
    const int turns = groups * (pieces / 256 + 1) > 32 * bh_compute_units() ? 4 : 1;
    const dim3 grid((pieces + 255) / 256, (groups + turns - 1) / turns);
    BH_REQUIRE(grid.y <= 65535, "token_shift: too many rows");
    if (dtype == BH_F32)
      token_shift_kernel<float><<<grid, 256, 0, stream>>>((const float*)h, h_block_rows, mu, mixes, state, slot_stride, row_seq, seq_start, seq_slot, seq_to, to,
                                                          out_block_rows, n_rows, width, turns, pieces);
    else if (dtype == BH_BF16)
      token_shift_kernel<bf16_t><<<grid, 256, 0, stream>>>((const bf16_t*)h, h_block_rows, mu, mixes, state, slot_stride, row_seq, seq_start, seq_slot, seq_to,
                                                           to, out_block_rows, n_rows, width, turns, pieces);
    else return bh_fail("token_shift: unknown dtype %d", dtype);
    return bh_check_launch("token_shift");
  }
  BH_REQUIRE(n_rows <= 65535, "token_shift: %d rows of a width that is no multiple of 8", n_rows);
  const dim3 grid((width + 255) / 256, n_rows);
  if (dtype == BH_F32)
    token_shift_plain_kernel<float><<<grid, 256, 0, stream>>>((const float*)h, mu, mixes, state, slot_stride, row_seq, seq_start, seq_slot, seq_to, to, n_rows,
                                                              width);
  else if (dtype == BH_BF16)
    token_shift_plain_kernel<bf16_t><<<grid, 256, 0, stream>>>((const bf16_t*)h, mu, mixes, state, slot_stride, row_seq, seq_start, seq_slot, seq_to, to, n_rows,
                                                               width);
  else return bh_fail("token_shift: unknown dtype %d", dtype);
  return bh_check_launch("token_shift");
}

template <typename T>
__global__ __launch_bounds__(256) void tanh_rows_kernel(const float* __restrict__ x, int row_stride, T* __restrict__ out, int width, size_t n,
                                                        int out_block_rows) {
  const size_t e = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (e >= n) return;
  const int row = (int)(e / width), column = (int)(e % width);
  out[bh_rows_index(out_block_rows, row, column, width)] = from_f32<T>(tanhf(x[(size_t)row * row_stride + column]));
}

// x [n_rows][row_stride] float32, of whose rows the first `width` numbers are taken; out [n_rows][width] (dtype; rows or blocks of rows).
extern "C" int bh_tanh_rows(const float* x, int row_stride, void* out, int dtype, int n_rows, int width, int out_block_rows, hipStream_t stream) {
  BH_REQUIRE(n_rows > 0 && width > 0 && width <= row_stride, "tanh_rows: rows of %d hold the %d numbers that are taken", row_stride, width);
  BH_REQUIRE(out_block_rows == 0 || ((out_block_rows == 8 || out_block_rows == 16) && width % 32 == 0 && dtype == BH_BF16),
             "tanh_rows: rows in blocks of %d of width %d are not written", out_block_rows, width);
  const size_t n = (size_t)n_rows * width, blocks = (n + 255) / 256;
  BH_REQUIRE(blocks <= 2147483647u, "tanh_rows: too many elements");
  if (dtype == BH_F32) tanh_rows_kernel<float><<<(unsigned)blocks, 256, 0, stream>>>(x, row_stride, (float*)out, width, n, out_block_rows);
  else if (dtype == BH_BF16) tanh_rows_kernel<bf16_t><<<(unsigned)blocks, 256, 0, stream>>>(x, row_stride, (bf16_t*)out, width, n, out_block_rows);
  else return bh_fail("tanh_rows: unknown dtype %d", dtype);
  return bh_check_launch("tanh_rows");
}
