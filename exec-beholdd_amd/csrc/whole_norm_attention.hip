// What stands around the paged attention kernels for an attention whose queries and keys are normed over the whole
// projection (all heads of a row together), turned in neighbouring pairs on the first dimensions of each head, and
// whose heads are gated before the output projection:
//   whole_norm_rope_write   per row of [q | k | v] (float32): q <- rms(q over all its channels) * wq, k likewise;
//                           dimensions 2i and 2i+1 (i < turned/2) of every head of q and k turned by
//                           position * freq[i]; q into a matrix of heads of `pad` dimensions, k and v into the cache
//                           pages of (sequence, position) as heads of `pad` (zeros beyond dim and vdim), so that keys of
//                           one size and values of another go through kernels that know one head size
//   conv_norm_rope_write    the same from the projected rows, the short convolution made on the way
//   gate_heads              out[row][h][i] = attended[row][h][i] * sigmoid(gate[row][h][i]) for i < vdim; the gate may be one
//                           number a head (gate[row][h]) or absent (the heads' first vdim elements are put side by side)
// Statistics, angles, cosines and sines are float32; the angle is the float32 product position * freq[i].
#include "short_conv.h"

template <typename T>
__global__ __launch_bounds__(256) void whole_norm_rope_write_kernel(
    const float* __restrict__ qkv, const float* __restrict__ wq, const float* __restrict__ wk, float eps,
    const float* __restrict__ freq, int turned, const int32_t* __restrict__ positions, const int32_t* __restrict__ row_seq,
    T* __restrict__ q_out, T* __restrict__ k_pages, T* __restrict__ v_pages, const int32_t* __restrict__ page_table,
    int table_stride, int H, int G, int dim, int vdim, int pad, int kv_order, int write) {
  extern __shared__ float turns[];      // the cosines, then the sines, of the row's turned pairs: one of each a pair and row
  __shared__ float scratch[8];
  const int row = blockIdx.x;
  const int q_width = H * dim, k_width = G * dim, v_width = G * vdim;
  const float* q = qkv + (size_t)row * (q_width + k_width + v_width);
  const float* k = q + q_width;
  const float* v = k + k_width;
  const int pos = positions[row];
  float* cosines = turns;
  float* sines = turns + turned / 2;
  for (int i = threadIdx.x; i < turned / 2; i += blockDim.x) {
    const float angle = (float)pos * freq[i];
    cosines[i] = cosf(angle);
    sines[i] = sinf(angle);
  }
  float ss_q = 0.f, ss_k = 0.f;
  for (int e = threadIdx.x; e < q_width + k_width; e += blockDim.x) {
    const float x = q[e];
    if (e < q_width) ss_q += x * x;
    else ss_k += x * x;
  }
  const float inv_q = 1.0f / sqrtf(block_sum(ss_q, scratch) / (float)q_width + eps);
  const float inv_k = 1.0f / sqrtf(block_sum(ss_k, scratch) / (float)k_width + eps);
  // a thread takes a pair of neighbouring dimensions: both of a turned pair come from the same two loads
  const int half = pad / 2;
  for (int e = threadIdx.x; e < H * half; e += blockDim.x) {
    const int head = e / half, i = 2 * (e % half);
    float y0 = 0.f, y1 = 0.f;
    if (i < dim) {
      const int at = head * dim + i;
      y0 = q[at] * inv_q * wq[at];
      if (i + 1 < dim) y1 = q[at + 1] * inv_q * wq[at + 1];
      if (i < turned) {
        const float c = cosines[i >> 1], s = sines[i >> 1], u = y0, w = y1;
        y0 = u * c - w * s;
        y1 = w * c + u * s;
      }
    }
    T* out = q_out + (size_t)row * H * pad + head * pad + i;
    out[0] = from_f32<T>(y0);
    out[1] = from_f32<T>(y1);
  }
  if (!write) return;
  const int page = page_table[(size_t)row_seq[row] * table_stride + pos / BH_PAGE], token = pos % BH_PAGE;
  for (int e = threadIdx.x; e < G * half; e += blockDim.x) {
    const int head = e / half, i = 2 * (e % half);
    float y0 = 0.f, y1 = 0.f;
    if (i < dim) {
      const int at = head * dim + i;
      y0 = k[at] * inv_k * wk[at];
      if (i + 1 < dim) y1 = k[at + 1] * inv_k * wk[at + 1];
      if (i < turned) {
        const float c = cosines[i >> 1], s = sines[i >> 1], u = y0, w = y1;
        y0 = u * c - w * s;
        y1 = w * c + u * s;
      }
    }
    T* keys = k_pages + ((size_t)page * G + head) * BH_PAGE * pad;
    T* values = v_pages + ((size_t)page * G + head) * BH_PAGE * pad;
    keys[bh_key_index(kv_order, token, i, pad)] = from_f32<T>(y0);
    keys[bh_key_index(kv_order, token, i + 1, pad)] = from_f32<T>(y1);
    values[bh_value_index(kv_order, token, i, pad)] = from_f32<T>(i < vdim ? v[head * vdim + i] : 0.f);
    values[bh_value_index(kv_order, token, i + 1, pad)] = from_f32<T>(i + 1 < vdim ? v[head * vdim + i + 1] : 0.f);
  }
}

// The same for steps of many rows, in pieces of four dimensions that a thread keeps between the statistics and the turn: PER pieces of q and k a
// thread, all asked for at once with those of v, where the kernel above reads q and k twice, an element at a time.  Bound by its bytes and two
// barriers a row.  2,048 rows of 16 heads of 128 on 4 20.7 -> 15.1 us, of 32 on 8 35.1 -> 26.7, 8,192 of these 152 -> 93.
template <typename T, int PER>
__global__ __launch_bounds__(256) void whole_norm_rope_write_pieces_kernel(
    const float* __restrict__ qkv, const float* __restrict__ wq, const float* __restrict__ wk, float eps,
    const float* __restrict__ freq, int turned, const int32_t* __restrict__ positions, const int32_t* __restrict__ row_seq,
    T* __restrict__ q_out, T* __restrict__ k_pages, T* __restrict__ v_pages, const int32_t* __restrict__ page_table,
    int table_stride, int H, int G, int dim, int vdim, int pad, int kv_order, int write, int n_rows) {
  extern __shared__ float turns[];
  __shared__ float scratch[8];
  const int row = bh_row_of_block<true>();      // 16 neighbours to an XCD: rows meet in the cache's lines
  if (row >= n_rows) return;
  const int q_width = H * dim, k_width = G * dim, v_width = G * vdim, pieces = pad / 4;      // (of a head)
  const float* x = qkv + (size_t)row * (q_width + k_width + v_width);
  const int pos = positions[row];
  int page = 0;
  if (write) page = page_table[(size_t)row_seq[row] * table_stride + pos / BH_PAGE];
  float* cosines = turns;
  float* sines = turns + turned / 2;
  const int units = (H + G) * pieces;
  const float4 zero = make_float4(0.f, 0.f, 0.f, 0.f);
  float4 held[PER];
  float ss_q = 0.f, ss_k = 0.f;
#pragma unroll
  for (int u = 0; u < PER; ++u) {
    const int e = threadIdx.x + blockDim.x * u, head = e / pieces, i = e % pieces * 4;
    held[u] = e < units && i < dim ? load_four(x + head * dim + i) : zero;      // (the heads of k stand behind those of q)
  }
  for (int i = threadIdx.x; i < turned / 2; i += blockDim.x) {
    const float angle = (float)pos * freq[i];
    cosines[i] = cosf(angle);
    sines[i] = sinf(angle);
  }
#pragma unroll
  for (int u = 0; u < PER; ++u) {
    const float4 y = held[u];
    const float squares = y.x * y.x + y.y * y.y + y.z * y.z + y.w * y.w;
    if (threadIdx.x + blockDim.x * u < H * pieces) ss_q += squares;
    else ss_k += squares;
  }
  const float inv_q = 1.0f / sqrtf(block_sum(ss_q, scratch) / (float)q_width + eps);
  const float inv_k = 1.0f / sqrtf(block_sum(ss_k, scratch) / (float)k_width + eps);
#pragma unroll
  for (int u = 0; u < PER; ++u) {
    const int e = threadIdx.x + blockDim.x * u, head = e / pieces, i = e % pieces * 4;
    if (e >= units) break;
    const bool is_key = head >= H;
    float4 y = zero;
    if (i < dim) {
      const float inv = is_key ? inv_k : inv_q;
      const float4 w = load_four(is_key ? wk + (head - H) * dim + i : wq + head * dim + i);
      y = make_float4(held[u].x * inv * w.x, held[u].y * inv * w.y, held[u].z * inv * w.z, held[u].w * inv * w.w);
      if (i < turned) {
        const float c = cosines[i >> 1], s = sines[i >> 1], a = y.x, b = y.y;
        y.x = a * c - b * s;
        y.y = b * c + a * s;
      }
      if (i + 2 < turned) {
        const float c = cosines[(i >> 1) + 1], s = sines[(i >> 1) + 1], a = y.z, b = y.w;
        y.z = a * c - b * s;
        y.w = b * c + a * s;
      }
    }
    if (!is_key) store_four(q_out + ((size_t)row * H + head) * pad + i, y.x, y.y, y.z, y.w);
    else if (write) store_four(k_pages + ((size_t)page * G + head - H) * BH_PAGE * pad + bh_key_index(kv_order, pos % BH_PAGE, i, pad), y.x, y.y, y.z, y.w);
  }
  if (!write) return;
  for (int e = threadIdx.x; e < G * pieces; e += blockDim.x) {
    const int head = e / pieces, i = e % pieces * 4;
    const float4 y = i < vdim ? load_four(x + q_width + k_width + head * vdim + i) : zero;
    T* values = v_pages + ((size_t)page * G + head) * BH_PAGE * pad;
    const float four[4] = {y.x, y.y, y.z, y.w};
#pragma unroll
    for (int j = 0; j < 4; ++j) values[bh_value_index(kv_order, pos % BH_PAGE, i + j, pad)] = from_f32<T>(four[j]);
  }
}

extern "C" int bh_whole_norm_rope_write(const float* qkv, const float* wq, const float* wk, float eps, const float* freq,
                                        int turned, const int32_t* positions, const int32_t* row_seq, void* q_out, int dtype,
                                        void* k_pages, void* v_pages, const int32_t* page_table, int table_stride, int n_rows,
                                        int H, int G, int dim, int vdim, int pad, int kv_order, int write, hipStream_t stream) {
  BH_REQUIRE(n_rows > 0 && H > 0 && G > 0 && dim > 0 && vdim > 0, "whole_norm_rope_write: sizes must be positive");
  BH_REQUIRE(pad >= dim && pad >= vdim, "whole_norm_rope_write: heads of %d do not hold keys of %d and values of %d", pad, dim, vdim);
  BH_REQUIRE(turned >= 0 && turned % 2 == 0 && turned <= dim && dim % 2 == 0 || turned == 0,
             "whole_norm_rope_write: %d turned dimensions of %d", turned, dim);
  BH_REQUIRE(turned == 0 || freq != nullptr, "whole_norm_rope_write: a rotation needs its frequencies");
  BH_REQUIRE(kv_order == BH_KV_ROWS || (kv_order == BH_KV_PIECES && pad % 32 == 0),
             "whole_norm_rope_write: cache order %d does not exist for head size %d", kv_order, pad);
  BH_REQUIRE(pad % 2 == 0, "whole_norm_rope_write: heads of an even size, got %d", pad);
  const size_t lds = (size_t)(turned > 0 ? turned : 1) * sizeof(float);
  // Rows for every compute unit, whole pieces of four, and no more of them than the threads hold.
  const int pieces = (H + G) * (pad / 4);
  if (n_rows >= bh_compute_units() && bh_rows_spread(n_rows, 16) && dim % 4 == 0 && vdim % 4 == 0 && pad % 4 == 0 && pieces <= 8 * 256 && (dtype == BH_F32 || dtype == BH_BF16) &&
      ((uintptr_t)qkv | (uintptr_t)wq | (uintptr_t)wk | (uintptr_t)q_out | (uintptr_t)k_pages) % 16 == 0) {
    const int threads = (int)bh_piece_threads(pieces), each = (pieces + threads - 1) / threads;
#define BH_WNP(T, PER)                                                                                                          \
  whole_norm_rope_write_pieces_kernel<T, PER><<<bh_rows_grid(n_rows, 16), threads, lds, stream>>>(qkv, wq, wk, eps, freq, turned, positions, row_seq, (T*)q_out, (T*)k_pages, \
                                                                           (T*)v_pages, page_table, table_stride, H, G, dim, vdim, pad, kv_order, write, n_rows)
#define BH_WNP_OF(T)               \
  if (each <= 1) BH_WNP(T, 1);     \
  else if (each <= 2) BH_WNP(T, 2); \
  else if (each <= 4) BH_WNP(T, 4); \
  else BH_WNP(T, 8)
    if (dtype == BH_F32) {
      BH_WNP_OF(float);
    } else {
      BH_WNP_OF(bf16_t);
    }
#undef BH_WNP_OF
#undef BH_WNP
    return bh_check_launch("whole_norm_rope_write");
  }
  if (dtype == BH_F32)
    whole_norm_rope_write_kernel<float><<<n_rows, 256, lds, stream>>>(qkv, wq, wk, eps, freq, turned, positions, row_seq, (float*)q_out,
                                                                  (float*)k_pages, (float*)v_pages, page_table, table_stride, H, G,
                                                                  dim, vdim, pad, kv_order, write);
  else if (dtype == BH_BF16)
    whole_norm_rope_write_kernel<bf16_t><<<n_rows, 256, lds, stream>>>(qkv, wq, wk, eps, freq, turned, positions, row_seq,
                                                                   (bf16_t*)q_out, (bf16_t*)k_pages, (bf16_t*)v_pages, page_table,
                                                                   table_stride, H, G, dim, vdim, pad, kv_order, write);
  else
    return bh_fail("whole_norm_rope_write: unknown dtype %d", dtype);
  return bh_check_launch("whole_norm_rope_write");
}

// The same from the projected rows themselves: the short convolution over time (csrc/short_conv.hip has its definition and
// its state) is made on the way, a row's convolved channels stand in LDS as float32 and are never written to memory.
// proj [n_rows][row_stride]: a row holds, from `first`, q, k and v; w_conv [q + k + v channels][taps] (taps 0: no convolution).
// TAPS: four, whose loads are all asked for before the first is used, of a whole thread's channels where these are up to four, or 0: any
// number, a trip to memory a tap (us, so / asked for together, 24 heads of 128 and 8 of keys and values: one row 11.7 / 9.7, 16 rows 12.0 / 10.1, a prompt of
// 127 13.4 / 10.6; 64 and 8, 127 rows 21.6 / 14.8; 4 of 64 and 2, 16 rows 6.7 / 6.0).  seq_to: as in short_conv.hip.
template <typename T, int TAPS>
__global__ __launch_bounds__(1024) void conv_norm_rope_write_kernel(
    const T* __restrict__ proj, int row_stride, int first, const float* __restrict__ w_conv, int taps, float* __restrict__ state,
    long slot_stride, const int32_t* __restrict__ seq_start, const int32_t* __restrict__ seq_slot, const int32_t* __restrict__ seq_to,
    const float* __restrict__ wq,
    const float* __restrict__ wk, float eps, const float* __restrict__ freq, int turned, const int32_t* __restrict__ positions,
    const int32_t* __restrict__ row_seq, T* __restrict__ q_out, T* __restrict__ k_pages, T* __restrict__ v_pages,
    const int32_t* __restrict__ page_table, int table_stride, int H, int G, int dim, int vdim, int pad, int kv_order, int write) {
  extern __shared__ float conv[];      // [q | k | v] of this row, then the cosines and sines of the row's turned pairs
  __shared__ float scratch[16];
  const int row = blockIdx.x;
  const int q_width = H * dim, k_width = G * dim, v_width = G * vdim, channels = q_width + k_width + v_width;
  float* cosines = conv + channels;
  float* sines = cosines + turned / 2;
  const int seq = row_seq[row], pos = positions[row];
  const int t = row - seq_start[seq];
  const float* old = state ? state + (size_t)seq_slot[seq] * slot_stride : nullptr;
  for (int i = threadIdx.x; i < turned / 2; i += blockDim.x) {
    const float angle = (float)pos * freq[i];
    cosines[i] = cosf(angle);
    sines[i] = sinf(angle);
  }
  float ss_q = 0.f, ss_k = 0.f;
  const bool leaves = seq_to && row + 1 == seq_start[seq + 1];
  float* left = leaves ? state + (size_t)seq_to[seq] * slot_stride : nullptr;
  auto put = [&](int c, float acc) {
    conv[c] = acc;
    if (c < q_width) ss_q += acc * acc;
    else if (c < q_width + k_width) ss_k += acc * acc;
  };
  if constexpr (TAPS > 0) {
    constexpr int TOGETHER = 4;      // channels a thread
    for (int c0 = threadIdx.x; c0 < channels; c0 += TOGETHER * blockDim.x) {
      // (a row's input and an old one are both asked for, wherever they lie, and the one that counts is taken: no load waits for a branch)
      T now[TOGETHER][TAPS];
      float before[TOGETHER][TAPS], w[TOGETHER][TAPS], u[TOGETHER][TAPS];
#pragma unroll
      for (int i = 0; i < TOGETHER; ++i) {
        const int c = min(c0 + i * (int)blockDim.x, channels - 1);
#pragma unroll
        for (int j = 0; j < TAPS; ++j) {
          const int back = TAPS - 1 - j;
          w[i][j] = w_conv[(size_t)c * TAPS + j];
          now[i][j] = proj[(size_t)(row - min(back, t)) * row_stride + first + c];
          before[i][j] = 0.f;
        }
      }
      if (t < TAPS - 1) {
#pragma unroll
        for (int i = 0; i < TOGETHER; ++i)
#pragma unroll
          for (int j = 0; j < TAPS - 1; ++j) before[i][j] = old[(size_t)min(t + j, TAPS - 2) * channels + min(c0 + i * (int)blockDim.x, channels - 1)];
      }
#pragma unroll
      for (int i = 0; i < TOGETHER; ++i) {
        const int c = c0 + i * (int)blockDim.x;
        if (c >= channels) break;
        float acc = 0.f;
#pragma unroll
        for (int j = 0; j < TAPS; ++j) {
          u[i][j] = TAPS - 1 - j <= t ? to_f32(now[i][j]) : before[i][j];
          acc = fmaf(w[i][j], u[i][j], acc);
        }
        put(c, acc);
        if (leaves) {
#pragma unroll
          for (int j = 1; j < TAPS; ++j) left[(size_t)(j - 1) * channels + c] = u[i][j];
        }
      }
    }
  } else {
    for (int c = threadIdx.x; c < channels; c += blockDim.x) {
      float acc;
      if (taps <= 1) {
        acc = to_f32(proj[(size_t)row * row_stride + first + c]) * (taps ? w_conv[c] : 1.f);
      } else {
        acc = 0.f;
        for (int j = 0; j < taps; ++j) {
          const int back = taps - 1 - j;
          const float u = back <= t ? to_f32(proj[(size_t)(row - back) * row_stride + first + c])
                                    : old[(size_t)(taps - 1 + t - back) * channels + c];
          acc = fmaf(w_conv[(size_t)c * taps + j], u, acc);
        }
      }
      put(c, acc);
      if (leaves) sc_leave_inputs(proj, row_stride, first + c, row - t, t + 1, taps, old, left, channels, c);
    }
  }
  const float inv_q = 1.0f / sqrtf(block_sum(ss_q, scratch) / (float)q_width + eps);
  const float inv_k = 1.0f / sqrtf(block_sum(ss_k, scratch) / (float)k_width + eps);
  const float* q = conv;
  const float* k = conv + q_width;
  const float* v = k + k_width;
  for (int e = threadIdx.x; e < H * pad; e += blockDim.x) {
    const int head = e / pad, i = e % pad;
    float y = 0.f;
    if (i < dim) {
      const int at = head * dim + i;
      y = q[at] * inv_q * wq[at];
      if (i < turned) {
        const int mate = at ^ 1;
        const float other = q[mate] * inv_q * wq[mate];
        const float c = cosines[i >> 1], s = sines[i >> 1];
        y = (i & 1) ? y * c + other * s : y * c - other * s;
      }
    }
    q_out[(size_t)row * H * pad + e] = from_f32<T>(y);
  }
  if (!write) return;
  const int page = page_table[(size_t)seq * table_stride + pos / BH_PAGE], token = pos % BH_PAGE;
  for (int e = threadIdx.x; e < G * pad; e += blockDim.x) {
    const int head = e / pad, i = e % pad;
    float y = 0.f;
    if (i < dim) {
      const int at = head * dim + i;
      y = k[at] * inv_k * wk[at];
      if (i < turned) {
        const int mate = at ^ 1;
        const float other = k[mate] * inv_k * wk[mate];
        const float c = cosines[i >> 1], s = sines[i >> 1];
        y = (i & 1) ? y * c + other * s : y * c - other * s;
      }
    }
    T* keys = k_pages + ((size_t)page * G + head) * BH_PAGE * pad;
    T* values = v_pages + ((size_t)page * G + head) * BH_PAGE * pad;
    keys[bh_key_index(kv_order, token, i, pad)] = from_f32<T>(y);
    values[bh_value_index(kv_order, token, i, pad)] = from_f32<T>(i < vdim ? v[head * vdim + i] : 0.f);
  }
}

extern "C" int bh_conv_norm_rope_write(const void* proj, int dtype, int row_stride, int first, const float* w_conv, int taps,
                                       float* state, long slot_stride, const int32_t* seq_start, const int32_t* seq_slot,
                                       const int32_t* seq_to, const float* wq, const float* wk, float eps, const float* freq, int turned,
                                       const int32_t* positions, const int32_t* row_seq, void* q_out, void* k_pages, void* v_pages,
                                       const int32_t* page_table, int table_stride, int n_rows, int H, int G, int dim, int vdim, int pad,
                                       int kv_order, int write, hipStream_t stream) {
  BH_REQUIRE(n_rows > 0 && H > 0 && G > 0 && dim > 0 && vdim > 0, "conv_norm_rope_write: sizes must be positive");
  BH_REQUIRE(pad >= dim && pad >= vdim, "conv_norm_rope_write: heads of %d do not hold keys of %d and values of %d", pad, dim, vdim);
  BH_REQUIRE(turned == 0 || (turned % 2 == 0 && turned <= dim && dim % 2 == 0 && freq != nullptr),
             "conv_norm_rope_write: %d turned dimensions of %d", turned, dim);
  BH_REQUIRE(taps >= 0 && taps <= 16 && (taps <= 1 || state != nullptr) && (taps == 0 || w_conv != nullptr),
             "conv_norm_rope_write: %d taps need their weights and, beyond one, a state", taps);
  const int channels = (H + G) * dim + G * vdim;
  BH_REQUIRE(first >= 0 && first + channels <= row_stride, "conv_norm_rope_write: q, k and v lie outside a row of %d", row_stride);
  BH_REQUIRE(kv_order == BH_KV_ROWS || (kv_order == BH_KV_PIECES && pad % 32 == 0),
             "conv_norm_rope_write: cache order %d does not exist for head size %d", kv_order, pad);
  const size_t lds = (size_t)(channels + turned) * sizeof(float);
  BH_REQUIRE(lds <= 128 * 1024, "conv_norm_rope_write: %d channels do not fit the local memory", channels);
  const int threads = n_rows < 2 * bh_compute_units() && channels >= 2048 ? 1024 : 256;      // few rows: more of the chip a row
#define BH_CW(T, TAPS)                                                                                                             \
  do {                                                                                                                             \
    bh_allow_lds<conv_norm_rope_write_kernel<T, TAPS>>(lds);                                                                       \
    conv_norm_rope_write_kernel<T, TAPS><<<n_rows, threads, lds, stream>>>((const T*)proj, row_stride, first, w_conv, taps, state, slot_stride,  \
                                                                 seq_start, seq_slot, seq_to, wq, wk, eps, freq, turned, positions, row_seq, \
                                                                 (T*)q_out, (T*)k_pages, (T*)v_pages, page_table, table_stride, H, G, \
                                                                 dim, vdim, pad, kv_order, write);                                  \
  } while (0)
  if (dtype == BH_F32 && taps == 4) BH_CW(float, 4);
  else if (dtype == BH_F32) BH_CW(float, 0);
  else if (dtype == BH_BF16 && taps == 4) BH_CW(bf16_t, 4);
  else if (dtype == BH_BF16) BH_CW(bf16_t, 0);
  else return bh_fail("conv_norm_rope_write: unknown dtype %d", dtype);
#undef BH_CW
  return bh_check_launch("conv_norm_rope_write");
}

template <typename T>
__global__ __launch_bounds__(256) void gate_heads_kernel(const T* __restrict__ attended, int pad, const T* __restrict__ gate,
                                                         int gate_stride, int gate_first, T* __restrict__ out, int n_rows, int H,
                                                         int vdim, int out_block_rows, int gate_per_head) {
  const int width = H * vdim;
  const size_t n = (size_t)n_rows * width;
  for (size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x; e < n; e += (size_t)gridDim.x * blockDim.x) {
    const int r = (int)(e / width), c = (int)(e % width), head = c / vdim, i = c % vdim;
    const float a = to_f32(attended[((size_t)r * H + head) * pad + i]);
    if (gate == nullptr) {      // no gate: the heads' first vdim elements, side by side
      out[bh_rows_index(out_block_rows, r, c, width)] = from_f32<T>(a);
      continue;
    }
    const float g = to_f32(gate[(size_t)r * gate_stride + gate_first + (gate_per_head ? head : c)]);
    out[bh_rows_index(out_block_rows, r, c, width)] = from_f32<T>(a / (1.0f + expf(-g)));
  }
}

// The same in pieces of 16 bytes (4 or 8 neighbouring elements of a head, which lie together in rows and in blocks alike).
template <typename T>
__global__ __launch_bounds__(256) void gate_heads_pieces_kernel(const T* __restrict__ attended, int pad, const T* __restrict__ gate,
                                                                int gate_stride, int gate_first, T* __restrict__ out, int n_rows, int H,
                                                                int vdim, int out_block_rows, int gate_per_head) {
  constexpr int N = 16 / sizeof(T);
  const int width = H * vdim, row = bh_row_of_block(out_block_rows), c = N * (blockIdx.y * blockDim.x + threadIdx.x);
  if (row >= n_rows || c >= width) return;
  const int head = c / vdim, i = c % vdim;
  union Piece {
    uint4 raw;
    T v[N];
  } piece, gates;
  piece.raw = *reinterpret_cast<const uint4*>(attended + ((size_t)row * H + head) * pad + i);
  if (gate) {
    const T* own = gate + (size_t)row * gate_stride + gate_first;
    if (gate_per_head) {
#pragma unroll
      for (int e = 0; e < N; ++e) gates.v[e] = own[head];
    } else {
      gates.raw = *reinterpret_cast<const uint4*>(own + c);
    }
#pragma unroll
    for (int e = 0; e < N; ++e) piece.v[e] = from_f32<T>(to_f32(piece.v[e]) / (1.0f + expf(-to_f32(gates.v[e]))));
  }
  *reinterpret_cast<uint4*>(out + bh_rows_index(out_block_rows, row, c, width)) = piece.raw;
}

extern "C" int bh_gate_heads(const void* attended, int dtype, int pad, const void* gate, int gate_stride, int gate_first,
                             void* out, int n_rows, int H, int vdim, int out_block_rows, int gate_per_head, hipStream_t stream) {
  BH_REQUIRE(n_rows > 0 && H > 0 && vdim > 0 && pad >= vdim, "gate_heads: sizes do not fit");
  BH_REQUIRE(gate == nullptr || (gate_first >= 0 && gate_first + (gate_per_head ? H : H * vdim) <= gate_stride),
             "gate_heads: the gate lies outside its row");
  BH_REQUIRE(out_block_rows == 0 || ((out_block_rows == 8 || out_block_rows == 16) && (H * vdim) % 32 == 0 && dtype == BH_BF16),
             "gate_heads: rows in blocks of %d of width %d are not written", out_block_rows, H * vdim);
  const int piece = dtype == BH_F32 ? 4 : 8;
  const bool gates_on16 = gate == nullptr || gate_per_head || ((uintptr_t)gate % 16 == 0 && gate_stride % piece == 0 && gate_first % piece == 0);
  if ((dtype == BH_F32 || bh_pieces_pay((long)n_rows * H * vdim)) && vdim % piece == 0 && pad % piece == 0 && gates_on16 && (((uintptr_t)attended | (uintptr_t)out) % 16) == 0 && (long)H * vdim <= 4L * 256 * 65535 &&
      (dtype == BH_F32 || dtype == BH_BF16)) {
    const dim3 grid(bh_rows_grid(n_rows, out_block_rows), (H * vdim / piece + 255) / 256), block(bh_piece_threads(H * vdim / piece));
    if (dtype == BH_F32)
      gate_heads_pieces_kernel<float><<<grid, block, 0, stream>>>((const float*)attended, pad, (const float*)gate, gate_stride, gate_first, (float*)out,
                                                               n_rows, H, vdim, out_block_rows, gate_per_head);
    else
      gate_heads_pieces_kernel<bf16_t><<<grid, block, 0, stream>>>((const bf16_t*)attended, pad, (const bf16_t*)gate, gate_stride, gate_first,
                                                                (bf16_t*)out, n_rows, H, vdim, out_block_rows, gate_per_head);
    return bh_check_launch("gate_heads");
  }
  const size_t n = (size_t)n_rows * H * vdim;
  const int blocks = (int)((n + 255) / 256 < 8192 ? (n + 255) / 256 : 8192);
  if (dtype == BH_F32)
    gate_heads_kernel<float><<<blocks, 256, 0, stream>>>((const float*)attended, pad, (const float*)gate, gate_stride, gate_first,
                                                       (float*)out, n_rows, H, vdim, out_block_rows, gate_per_head);
  else if (dtype == BH_BF16)
    gate_heads_kernel<bf16_t><<<blocks, 256, 0, stream>>>((const bf16_t*)attended, pad, (const bf16_t*)gate, gate_stride, gate_first,
                                                        (bf16_t*)out, n_rows, H, vdim, out_block_rows, gate_per_head);
  else
    return bh_fail("gate_heads: unknown dtype %d", dtype);
  return bh_check_launch("gate_heads");
}
