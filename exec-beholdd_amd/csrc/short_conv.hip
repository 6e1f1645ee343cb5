// A short causal convolution over time on every channel of a slice of a projected matrix, continued from step to
// step through a state that holds the last taps - 1 inputs of each sequence:
//   y[t][c] = sum_j w[c][j] * u[t - taps + 1 + j][c]  (+ bias[c])  (then silu),   zeros before a sequence starts.
//   short_conv        the rows of a step; inputs that lie before the step come from the state.  With seq_to the thread of a sequence's
//                     last row leaves the state after the step in these rows, which no sequence of the step reads
//   short_conv_state  the state after the step, otherwise (run it after every reader of the old state), left in the rows seq_to, which
//                     may be those it is read from
// State of one sequence: [taps - 1][channels] float32, the oldest input first, at `state + slot * slot_stride`.
// Sums are float32; the result is float32.
#include "short_conv.h"

template <typename T>
__global__ __launch_bounds__(256) void short_conv_kernel(const T* __restrict__ u, int row_stride, int first,
                                                         const float* __restrict__ w, const float* __restrict__ bias,
                                                         float* __restrict__ state, long slot_stride,
                                                         const int32_t* __restrict__ row_seq, const int32_t* __restrict__ seq_start,
                                                         const int32_t* __restrict__ seq_slot, const int32_t* __restrict__ seq_to,
                                                         float* __restrict__ out, int n_rows, int channels, int taps, int silu) {
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= channels) return;
  float wc[SC_MAX_TAPS];
#pragma unroll
  for (int j = 0; j < SC_MAX_TAPS; ++j) wc[j] = j < taps ? w[(size_t)c * taps + j] : 0.f;
  const float b = bias ? bias[c] : 0.f;
  for (int row = blockIdx.y; row < n_rows; row += gridDim.y) {
    const int seq = row_seq[row];
    const int t = row - seq_start[seq];      // the row's place among its sequence's rows of this step
    const float* old = state + (size_t)seq_slot[seq] * slot_stride;
    float acc = b;
#pragma unroll
    for (int j = 0; j < SC_MAX_TAPS; ++j) {
      if (j >= taps) break;
      const int back = taps - 1 - j;         // how many rows before this one
      float v;
      if (back <= t) v = to_f32(u[(size_t)(row - back) * row_stride + first + c]);
      else v = old[(size_t)(taps - 1 + t - back) * channels + c];
      acc = fmaf(wc[j], v, acc);
    }
    if (silu) acc = acc / (1.0f + expf(-acc));
    out[(size_t)row * channels + c] = acc;
    if (seq_to && row + 1 == seq_start[seq + 1])
      sc_leave_inputs(u, row_stride, first + c, row - t, t + 1, taps, old, state + (size_t)seq_to[seq] * slot_stride, channels, c);
  }
}

// The same for steps of many rows: a thread walks SC_ROWS consecutive rows of its channel with the last TAPS inputs in
// registers, so that every input is loaded once (where a sequence starts inside the stretch, the window is filled anew
// from that sequence's state).
#define SC_ROWS 32

template <typename T, int TAPS>
__global__ __launch_bounds__(256) void short_conv_walk_kernel(const T* __restrict__ u, int row_stride, int first,
                                                              const float* __restrict__ w, const float* __restrict__ bias,
                                                              float* __restrict__ state, long slot_stride,
                                                              const int32_t* __restrict__ row_seq, const int32_t* __restrict__ seq_start,
                                                              const int32_t* __restrict__ seq_slot, const int32_t* __restrict__ seq_to,
                                                              float* __restrict__ out, int n_rows, int channels, int silu) {
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= channels) return;
  float wc[TAPS], win[TAPS];
#pragma unroll
  for (int j = 0; j < TAPS; ++j) wc[j] = w[(size_t)c * TAPS + j];
  const float b = bias ? bias[c] : 0.f;
  const int r0 = blockIdx.y * SC_ROWS, r1 = r0 + SC_ROWS < n_rows ? r0 + SC_ROWS : n_rows;
  int seq = -1;
  for (int row = r0; row < r1; ++row) {
    const int here = row_seq[row];
    if (here != seq) {      // the first row of the stretch, or of a sequence: the inputs before it
      seq = here;
      const int t = row - seq_start[seq];
      const float* old = state + (size_t)seq_slot[seq] * slot_stride;
#pragma unroll
      for (int j = 0; j < TAPS - 1; ++j) {
        const int back = TAPS - 1 - j;
        win[j] = back <= t ? to_f32(u[(size_t)(row - back) * row_stride + first + c]) : old[(size_t)(TAPS - 1 + t - back) * channels + c];
      }
    } else {
#pragma unroll
      for (int j = 0; j < TAPS - 1; ++j) win[j] = win[j + 1];
    }
    win[TAPS - 1] = to_f32(u[(size_t)row * row_stride + first + c]);
    float acc = b;
#pragma unroll
    for (int j = 0; j < TAPS; ++j) acc = fmaf(wc[j], win[j], acc);
    if (silu) acc = acc / (1.0f + expf(-acc));
    out[(size_t)row * channels + c] = acc;
    if (seq_to && row + 1 == seq_start[seq + 1]) {      // the window's later inputs are what the next step starts with
      float* to = state + (size_t)seq_to[seq] * slot_stride;
#pragma unroll
      for (int j = 1; j < TAPS; ++j) to[(size_t)(j - 1) * channels + c] = win[j];
    }
  }
}

// The same in pieces of four channels: a thread asks for all inputs of its stretch of SC_FAR rows together and waits for them once, where the
// walk above has a load a row and its wait.  A stretch in which a sequence starts is walked row by row.  Bound by its bytes (the inputs once,
// 3 in 19 of them twice, float32 outputs) and, with few waves a compute unit, the way to memory.  2,100 rows of 6,144 and of 3,072 channels, on average 32.9 -> 23.8 us; 1,024 rows of 6,144
// 21.5 / 16.5; at the fewest, 128 rows of 512 channels 11.9 / 10.6, of 6,144 12.8 / 11.3 (512 to 6,144 channels, bfloat16 and float32, one and eight
// sequences: 0.92 of the walk's time at worst).
#define SC_FAR 16

template <typename T>
struct FourOf {      // four channels' inputs as they come
  float4 raw;
  __device__ void load(const T* from) { raw = load_four(from); }
  __device__ float4 values() const { return raw; }
};
template <>
struct FourOf<bf16_t> {
  uint2 raw;
  __device__ void load(const bf16_t* from) { raw = *reinterpret_cast<const uint2*>(from); }
  __device__ float4 values() const {
    return make_float4(bf16_bits_to_f32((uint16_t)(raw.x & 0xffffu)), bf16_bits_to_f32((uint16_t)(raw.x >> 16)),
                       bf16_bits_to_f32((uint16_t)(raw.y & 0xffffu)), bf16_bits_to_f32((uint16_t)(raw.y >> 16)));
  }
};

template <typename T, int TAPS>
__global__ __launch_bounds__(256) void short_conv_pieces_kernel(const T* __restrict__ u, int row_stride, int first,
                                                                const float* __restrict__ w, const float* __restrict__ bias,
                                                                float* __restrict__ state, long slot_stride,
                                                                const int32_t* __restrict__ row_seq, const int32_t* __restrict__ seq_start,
                                                                const int32_t* __restrict__ seq_slot, const int32_t* __restrict__ seq_to,
                                                                float* __restrict__ out, int n_rows, int channels, int silu) {
  const int c = 4 * (blockIdx.x * blockDim.x + threadIdx.x);
  if (c >= channels) return;
  const int r0 = blockIdx.y * SC_FAR, r1 = r0 + SC_FAR < n_rows ? r0 + SC_FAR : n_rows;
  const T* column = u + first + c;
  FourOf<T> ahead[SC_FAR];
#pragma unroll
  for (int i = 0; i < SC_FAR; ++i) ahead[i].load(column + (size_t)(r0 + i < r1 ? r0 + i : r1 - 1) * row_stride);
  float wc[4][TAPS], b[4], win[4][TAPS];
#pragma unroll
  for (int v = 0; v < 4; ++v) {
    b[v] = bias ? bias[c + v] : 0.f;
#pragma unroll
    for (int j = 0; j < TAPS; ++j) wc[v][j] = w[(size_t)(c + v) * TAPS + j];
  }
  int seq = row_seq[r0], seq_stop = seq_start[seq + 1];
  auto enter = [&](int row) {      // the inputs before a sequence's row
    const int t = row - seq_start[seq];
    const float* old = state + (size_t)seq_slot[seq] * slot_stride;
#pragma unroll
    for (int j = 0; j < TAPS - 1; ++j) {
      const int back = TAPS - 1 - j;
      const float4 x = back <= t ? load_four(column + (size_t)(row - back) * row_stride) : make_float4(0.f, 0.f, 0.f, 0.f);
      win[0][j] = x.x, win[1][j] = x.y, win[2][j] = x.z, win[3][j] = x.w;
      if (back > t) {
#pragma unroll
        for (int v = 0; v < 4; ++v) win[v][j] = old[(size_t)(TAPS - 1 + t - back) * channels + c + v];
      }
    }
  };
  enter(r0);
#pragma unroll
  for (int i = 0; i < SC_FAR; ++i) {
    const int row = r0 + i;
    if (row >= r1) break;
    if (row >= seq_stop) {
      seq = row_seq[row], seq_stop = seq_start[seq + 1];
      enter(row);
    }
    const float4 x = ahead[i].values();
    win[0][TAPS - 1] = x.x, win[1][TAPS - 1] = x.y, win[2][TAPS - 1] = x.z, win[3][TAPS - 1] = x.w;
    float y[4];
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      float acc = b[v];
#pragma unroll
      for (int j = 0; j < TAPS; ++j) acc = fmaf(wc[v][j], win[v][j], acc);
      y[v] = silu ? acc / (1.0f + expf(-acc)) : acc;
    }
    store_four(out + (size_t)row * channels + c, y[0], y[1], y[2], y[3]);
    if (seq_to && row + 1 == seq_stop) {      // the window's later inputs are what the next step starts with
      float* to = state + (size_t)seq_to[seq] * slot_stride;
#pragma unroll
      for (int v = 0; v < 4; ++v)
#pragma unroll
        for (int j = 1; j < TAPS; ++j) to[(size_t)(j - 1) * channels + c + v] = win[v][j];
    }
#pragma unroll
    for (int v = 0; v < 4; ++v)
#pragma unroll
      for (int j = 0; j < TAPS - 1; ++j) win[v][j] = win[v][j + 1];
  }
}

// seq_to [n_seqs]: the rows of the state to leave what the next step starts with in, none of which this step reads; or null: short_conv_state
// does it.
extern "C" int bh_short_conv(const void* u, int dtype, int row_stride, int first, const float* w, const float* bias,
                             float* state, long slot_stride, const int32_t* row_seq, const int32_t* seq_start,
                             const int32_t* seq_slot, const int32_t* seq_to, float* out, int n_rows, int channels, int taps, int silu,
                             hipStream_t stream) {
  BH_REQUIRE(n_rows > 0 && channels > 0, "short_conv: sizes must be positive");
  BH_REQUIRE(taps >= 1 && taps <= SC_MAX_TAPS, "short_conv: 1 to %d taps, got %d", SC_MAX_TAPS, taps);
  BH_REQUIRE(first >= 0 && first + channels <= row_stride, "short_conv: channels %d..%d lie outside a row of %d", first,
             first + channels, row_stride);
  BH_REQUIRE(taps == 1 || state != nullptr, "short_conv: more than one tap needs a state");
  if (n_rows >= 4 * SC_ROWS && taps >= 2 && taps <= 4 && (dtype == BH_F32 || dtype == BH_BF16)) {
    const size_t piece = 4 * (dtype == BH_F32 ? sizeof(float) : 2);
    if (channels % 4 == 0 && first % 4 == 0 && row_stride % 4 == 0 && (uintptr_t)u % piece == 0 && (uintptr_t)out % 16 == 0 &&
        n_rows <= 65535 * SC_FAR) {
      const int pieces = channels / 4, threads = (int)bh_piece_threads(pieces);
      dim3 stretches((pieces + threads - 1) / threads, (n_rows + SC_FAR - 1) / SC_FAR);
#define BH_SP(T, TAPS)                                                                                                              \
  short_conv_pieces_kernel<T, TAPS><<<stretches, threads, 0, stream>>>((const T*)u, row_stride, first, w, bias, state, slot_stride, row_seq, \
                                                                       seq_start, seq_slot, seq_to, out, n_rows, channels, silu)
      if (dtype == BH_F32) {
        if (taps == 2) BH_SP(float, 2);
        else if (taps == 3) BH_SP(float, 3);
        else BH_SP(float, 4);
      } else {
        if (taps == 2) BH_SP(bf16_t, 2);
        else if (taps == 3) BH_SP(bf16_t, 3);
        else BH_SP(bf16_t, 4);
      }
#undef BH_SP
      return bh_check_launch("short_conv");
    }
    dim3 walk((channels + 255) / 256, (n_rows + SC_ROWS - 1) / SC_ROWS);
#define BH_SW(T, TAPS)                                                                                                              \
  short_conv_walk_kernel<T, TAPS><<<walk, 256, 0, stream>>>((const T*)u, row_stride, first, w, bias, state, slot_stride, row_seq, seq_start, \
                                                            seq_slot, seq_to, out, n_rows, channels, silu)
    if (dtype == BH_F32) {
      if (taps == 2) BH_SW(float, 2);
      else if (taps == 3) BH_SW(float, 3);
      else BH_SW(float, 4);
    } else {
      if (taps == 2) BH_SW(bf16_t, 2);
      else if (taps == 3) BH_SW(bf16_t, 3);
      else BH_SW(bf16_t, 4);
    }
#undef BH_SW
    return bh_check_launch("short_conv");
  }
  dim3 grid((channels + 255) / 256, n_rows < 4096 ? n_rows : 4096);
  if (dtype == BH_F32)
    short_conv_kernel<float><<<grid, 256, 0, stream>>>((const float*)u, row_stride, first, w, bias, state, slot_stride, row_seq,
                                                       seq_start, seq_slot, seq_to, out, n_rows, channels, taps, silu);
  else if (dtype == BH_BF16)
    short_conv_kernel<bf16_t><<<grid, 256, 0, stream>>>((const bf16_t*)u, row_stride, first, w, bias, state, slot_stride, row_seq,
                                                        seq_start, seq_slot, seq_to, out, n_rows, channels, taps, silu);
  else
    return bh_fail("short_conv: unknown dtype %d", dtype);
  return bh_check_launch("short_conv");
}

// One thread a (sequence, channel): it reads what the new state takes from the old one before it writes.
template <typename T>
__global__ __launch_bounds__(256) void short_conv_state_kernel(const T* __restrict__ u, int row_stride, int first,
                                                               float* __restrict__ state, long slot_stride,
                                                               const int32_t* __restrict__ seq_start,
                                                               const int32_t* __restrict__ seq_slot, const int32_t* __restrict__ seq_to, int channels, int taps) {
  const int c = blockIdx.x * blockDim.x + threadIdx.x, seq = blockIdx.y;
  if (c >= channels) return;
  const int start = seq_start[seq], n_new = seq_start[seq + 1] - start;
  sc_leave_inputs(u, row_stride, first + c, start, n_new, taps, state + (size_t)seq_slot[seq] * slot_stride, state + (size_t)seq_to[seq] * slot_stride,
                  channels, c);
}

extern "C" int bh_short_conv_state(const void* u, int dtype, int row_stride, int first, float* state, long slot_stride,
                                   const int32_t* seq_start, const int32_t* seq_slot, const int32_t* seq_to, int n_seqs, int channels, int taps,
                                   hipStream_t stream) {
  BH_REQUIRE(n_seqs > 0 && channels > 0, "short_conv_state: sizes must be positive");
  BH_REQUIRE(taps >= 1 && taps <= SC_MAX_TAPS, "short_conv_state: 1 to %d taps, got %d", SC_MAX_TAPS, taps);
  BH_REQUIRE(first >= 0 && first + channels <= row_stride, "short_conv_state: channels lie outside a row");
  if (taps == 1) return 0;
  dim3 grid((channels + 255) / 256, n_seqs);
  if (dtype == BH_F32)
    short_conv_state_kernel<float><<<grid, 256, 0, stream>>>((const float*)u, row_stride, first, state, slot_stride, seq_start,
                                                             seq_slot, seq_to, channels, taps);
  else if (dtype == BH_BF16)
    short_conv_state_kernel<bf16_t><<<grid, 256, 0, stream>>>((const bf16_t*)u, row_stride, first, state, slot_stride, seq_start,
                                                              seq_slot, seq_to, channels, taps);
  else
    return bh_fail("short_conv_state: unknown dtype %d", dtype);
  return bh_check_launch("short_conv_state");
}
