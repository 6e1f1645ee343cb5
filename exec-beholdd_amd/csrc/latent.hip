// Attention over a cached latent: every position keeps one normed vector c [rank] and one rotated key part
// [rot_dim] that all heads share.  A head's score is q_c . (U_k c) + q_r . k_r = (U_k^T q_c) . c + q_r . k_r, and its
// output U_v (sum_j p_j c_j): with the queries carried into the latent's space the attention is the paged
// attention kernels' own case of ONE key/value head of size rank + rot_dim shared by all query heads, whose
// key is [c | k_r] and whose value is [c | 0].  This file holds what stands around that call:
//   latent_write    norm of c, rotation of k_r, and both into the cache pages of (sequence, position)
//   heads_linear    a small matrix per head: y[row, h, :] = W_h x[row, h, :] (queries into the latent's space,
//                   attended latents into the heads' values)
//   rotate_heads    rotation of a slice of every head of a row into a slice of another matrix's heads
// The angle of pair i at position p is the float32 product p * freq[i]; cosine and sine are taken of that float32.
#include "common.h"

// ---- the cached row: c = rms(x[:rank]) * w, k_r = rotate(x[rank:]) --------------------------------------------
template <typename T>
__global__ __launch_bounds__(256) void latent_write_kernel(
    const T* __restrict__ down, int row_stride, int offset, const float* __restrict__ w, float eps,
    const float* __restrict__ freq, int turned, const int32_t* __restrict__ positions, const int32_t* __restrict__ row_seq,
    T* __restrict__ k_pages, T* __restrict__ v_pages, const int32_t* __restrict__ page_table, int table_stride, int rank,
    int rot_dim, int kv_order, int write, T* __restrict__ query, long q_row, int q_head, int q_first, int src_head, int src_first,
    int H, const T* __restrict__ q_src, long q_src_row, int neighbours, float magnitude) {
  __shared__ float scratch[16];
  const int row = blockIdx.x;
  const T* x = down + (size_t)row * row_stride + offset;
  const int pos = positions[row], hd = rank + rot_dim;
  const int half = turned / 2;
  if (query != nullptr) {      // the heads' rotated query parts, from the same projected row or from a matrix of their own
    for (int e = threadIdx.x; e < H * rot_dim; e += blockDim.x) {
      const int head = e / rot_dim, i = e % rot_dim;
      const T* from = q_src + (size_t)row * q_src_row + (size_t)head * src_head + src_first;
      float y;
      if (i < turned) {
        // the pair's first and second dimension: i and i + half, or the neighbours 2 pair and 2 pair + 1
        const int pair = neighbours ? i / 2 : (i < half ? i : i - half);
        const bool is_first = neighbours ? (i % 2 == 0) : (i < half);
        const float angle = (float)pos * freq[pair];
        const float c = cosf(angle) * magnitude, s = sinf(angle) * magnitude;
        const float u = to_f32(from[neighbours ? 2 * pair : pair]), v = to_f32(from[neighbours ? 2 * pair + 1 : pair + half]);
        y = is_first ? u * c - v * s : v * c + u * s;
      } else {
        y = to_f32(from[i]);
      }
      query[(size_t)row * q_row + (size_t)head * q_head + q_first + i] = from_f32<T>(y);
    }
  }
  if (!write) return;
  const int page = page_table[(size_t)row_seq[row] * table_stride + pos / BH_PAGE], token = pos % BH_PAGE;
  T* keys = k_pages + (size_t)page * BH_PAGE * hd;
  T* values = v_pages + (size_t)page * BH_PAGE * hd;
  float ss = 0.f;
  for (int i = threadIdx.x; i < rank; i += blockDim.x) {
    const float v = to_f32(x[i]);
    ss += v * v;
  }
  ss = block_sum(ss, scratch);
  const float inv = 1.0f / sqrtf(ss / (float)rank + eps);
  for (int i = threadIdx.x; i < rank; i += blockDim.x) {
    const T c = from_f32<T>(to_f32(x[i]) * inv * (w ? w[i] : 1.f));
    keys[bh_key_index(kv_order, token, i, hd)] = c;
    values[bh_value_index(kv_order, token, i, hd)] = c;
  }
  for (int i = threadIdx.x; i < rot_dim; i += blockDim.x) {
    float y;
    if (i < turned) {
      const int pair = neighbours ? i / 2 : (i < half ? i : i - half);
      const bool is_first = neighbours ? (i % 2 == 0) : (i < half);
      const float angle = (float)pos * freq[pair];
      const float c = cosf(angle) * magnitude, s = sinf(angle) * magnitude;
      const float u = to_f32(x[rank + (neighbours ? 2 * pair : pair)]), v = to_f32(x[rank + (neighbours ? 2 * pair + 1 : pair + half)]);
      y = is_first ? u * c - v * s : v * c + u * s;
    } else {
      y = to_f32(x[rank + i]);
    }
    keys[bh_key_index(kv_order, token, rank + i, hd)] = from_f32<T>(y);
    values[bh_value_index(kv_order, token, rank + i, hd)] = from_f32<T>(0.f);
  }
}

// down [n_rows][row_stride]: a row holds, from `offset`, rank latent elements and rot_dim key elements.
// Pages as the attention kernels take them for one kv head of size rank + rot_dim (written when `write` is set).
// With `query`, the same launch rotates the rot_dim elements at src_first of each of the H heads (src_head apart) of the
// same row into query[row][head * q_head + q_first ..]: the heads' rotated query parts, beside the key's.  With `q_src`
// (rows of q_src_row elements) the heads' parts are read from that matrix instead of `down`.  `neighbours`: a pair is
// dimensions 2i and 2i + 1 instead of i and i + turned/2; `magnitude` multiplies every cosine and sine.
extern "C" int bh_latent_write(const void* down, int dtype, int row_stride, int offset, const float* w, float eps,
                               const float* freq, int turned, const int32_t* positions, const int32_t* row_seq,
                               void* k_pages, void* v_pages, const int32_t* page_table, int table_stride, int n_rows,
                               int rank, int rot_dim, int kv_order, int write, void* query, long q_row, int q_head, int q_first,
                               int src_head, int src_first, int H, const void* q_src, long q_src_row, int neighbours,
                               float magnitude, hipStream_t stream) {
  BH_REQUIRE(write || query != nullptr, "latent_write: nothing to do");
  if (q_src == nullptr) {
    q_src = down;
    q_src_row = row_stride;
  }
  BH_REQUIRE(query == nullptr || (H > 0 && q_first >= 0 && src_first >= 0 && q_first + rot_dim <= q_head && src_first + rot_dim <= src_head &&
                                  (long)H * q_head <= q_row && (long)H * src_head <= q_src_row),
             "latent_write: the heads' rotated slices do not lie inside their rows");
  BH_REQUIRE(n_rows > 0 && rank > 0 && rot_dim >= 0, "latent_write: sizes must be positive (the rotated part may be absent)");
  BH_REQUIRE(turned >= 0 && turned % 2 == 0 && turned <= rot_dim, "latent_write: %d turned dimensions of %d", turned, rot_dim);
  BH_REQUIRE(turned == 0 || freq != nullptr, "latent_write: a rotation needs its frequencies");
  BH_REQUIRE(offset >= 0 && offset + rank + rot_dim <= row_stride, "latent_write: the latent does not lie inside a row of %d", row_stride);
  BH_REQUIRE(kv_order == BH_KV_ROWS || (kv_order == BH_KV_PIECES && (rank + rot_dim) % 32 == 0),
             "latent_write: cache order %d does not exist for head size %d", kv_order, rank + rot_dim);
#define BH_LW(T)                                                                                                      \
  latent_write_kernel<T><<<dim3(n_rows), dim3(256), 0, stream>>>((const T*)down, row_stride, offset, w, eps, freq, turned, \
                                                                 positions, row_seq, (T*)k_pages, (T*)v_pages, page_table, \
                                                                 table_stride, rank, rot_dim, kv_order, write, (T*)query, q_row, q_head, \
                                                                 q_first, src_head, src_first, H, (const T*)q_src, q_src_row, \
                                                                 neighbours, magnitude)
  if (dtype == BH_F32) BH_LW(float);
  else if (dtype == BH_BF16) BH_LW(bf16_t);
  else return bh_fail("latent_write: unknown dtype %d", dtype);
#undef BH_LW
  return bh_check_launch("latent_write");
}

// ---- a small matrix per head ---------------------------------------------------------------------------------
// y[row][h][o] = sum_i w[h][i][o] * x[row][h][i] for o < n_out, i < n_in; x and y are slices of the heads of wider rows
// (row stride, head stride and first element given for each); w [H][n_in][n_out], the output index running fastest,
// so that the lanes of a wave read neighbouring weights.  Float32 sums; a workgroup takes HL_ROWS rows of one head
// and up to 256 outputs, the rows' inputs going through LDS once.  y's rows lie one after the other, or, for the
// product that reads them next, in blocks of rows (bh_rows_index; y_row is then the matrix's width).
#define HL_ROWS 16

template <typename T>
__global__ __launch_bounds__(256) void heads_linear_kernel(const T* __restrict__ x, long x_row, int x_head, int x_first,
                                                           const T* __restrict__ w, T* __restrict__ y, long y_row, int y_head,
                                                           int y_first, int n_rows, int n_in, int n_out, int y_block_rows) {
  extern __shared__ __align__(16) float xs[];      // [n_in][HL_ROWS]: the rows' values of one input side by side
  const int row0 = blockIdx.x * HL_ROWS, head = blockIdx.y, o = blockIdx.z * 256 + threadIdx.x;
  const int rows = n_rows - row0 < HL_ROWS ? n_rows - row0 : HL_ROWS;
  for (int e = threadIdx.x; e < HL_ROWS * n_in; e += 256) {
    const int r = e / n_in, i = e % n_in;      // neighbouring threads read neighbouring inputs of a row
    xs[i * HL_ROWS + r] = r < rows ? to_f32(x[(size_t)(row0 + r) * x_row + (size_t)head * x_head + x_first + i]) : 0.f;
  }
  __syncthreads();
  if (o >= n_out) return;
  const T* wh = w + (size_t)head * n_in * n_out + o;
  float acc[HL_ROWS] = {};
  for (int i = 0; i < n_in; ++i) {
    const float wv = to_f32(wh[(size_t)i * n_out]);
#pragma unroll
    for (int r = 0; r < HL_ROWS; r += 4) {      // four rows a read of LDS, the same address for every lane
      const float4 x4 = *reinterpret_cast<const float4*>(xs + i * HL_ROWS + r);
      acc[r] = fmaf(x4.x, wv, acc[r]);
      acc[r + 1] = fmaf(x4.y, wv, acc[r + 1]);
      acc[r + 2] = fmaf(x4.z, wv, acc[r + 2]);
      acc[r + 3] = fmaf(x4.w, wv, acc[r + 3]);
    }
  }
#pragma unroll
  for (int r = 0; r < HL_ROWS; ++r)
    if (r < rows) y[bh_rows_index(y_block_rows, row0 + r, head * y_head + y_first + o, (int)y_row)] = from_f32<T>(acc[r]);
}

// The same for a step of at most HL_ROWS rows (decoding): a workgroup takes 64 outputs of one head and its four waves
// a quarter of the inputs each, so that a head's weights are streamed by several workgroups and no thread walks all the
// inputs alone; the quarters' sums are added through LDS in a fixed order.
template <typename T>
__global__ __launch_bounds__(256) void heads_linear_few_kernel(const T* __restrict__ x, long x_row, int x_head, int x_first,
                                                               const T* __restrict__ w, T* __restrict__ y, long y_row, int y_head,
                                                               int y_first, int n_rows, int n_in, int n_out, int y_block_rows) {
  extern __shared__ __align__(16) float xs[];      // [n_in][HL_ROWS]
  __shared__ float parts[3][64][HL_ROWS + 1];
  const int head = blockIdx.y, lane = threadIdx.x % 64, quarter = threadIdx.x / 64, o = blockIdx.z * 64 + lane;
  for (int e = threadIdx.x; e < HL_ROWS * n_in; e += 256) {
    const int r = e / n_in, i = e % n_in;
    xs[i * HL_ROWS + r] = r < n_rows ? to_f32(x[(size_t)r * x_row + (size_t)head * x_head + x_first + i]) : 0.f;
  }
  __syncthreads();
  const int each = (n_in + 3) / 4, from = quarter * each, to = from + each < n_in ? from + each : n_in;
  const T* wh = w + (size_t)head * n_in * n_out + (o < n_out ? o : n_out - 1);
  float acc[HL_ROWS] = {};
  for (int i = from; i < to; ++i) {
    const float wv = to_f32(wh[(size_t)i * n_out]);
#pragma unroll
    for (int r = 0; r < HL_ROWS; r += 4) {
      const float4 x4 = *reinterpret_cast<const float4*>(xs + i * HL_ROWS + r);
      acc[r] = fmaf(x4.x, wv, acc[r]);
      acc[r + 1] = fmaf(x4.y, wv, acc[r + 1]);
      acc[r + 2] = fmaf(x4.z, wv, acc[r + 2]);
      acc[r + 3] = fmaf(x4.w, wv, acc[r + 3]);
    }
  }
  if (quarter > 0) {
#pragma unroll
    for (int r = 0; r < HL_ROWS; ++r) parts[quarter - 1][lane][r] = acc[r];
  }
  __syncthreads();
  if (quarter > 0 || o >= n_out) return;
#pragma unroll
  for (int r = 0; r < HL_ROWS; ++r) {
    if (r >= n_rows) continue;
    const float total = ((acc[r] + parts[0][lane][r]) + parts[1][lane][r]) + parts[2][lane][r];
    y[bh_rows_index(y_block_rows, r, head * y_head + y_first + o, (int)y_row)] = from_f32<T>(total);
  }
}

// The same on the matrix cores, for bfloat16 with n_in a multiple of 32 and n_out of 16: v_mfma_f32_16x16x32_bf16 with the outputs as rows
// and 16 rows of the step as columns.  A wave keeps its OT tiles of 16 outputs of one head in registers (the weights' index that the
// matrix instruction wants together lies n_out apart: eight 2-byte loads an operand, once) and walks over tiles of rows, whose inputs
// are 16-byte loads.  Products are exact and sums 32-bit, as in the kernels above.
// Bound by the rows' way in and out.  Measured, 128 -> 192 and 192 -> 128 a head: a prompt of 2,048 rows of 16 heads 14 us where the kernel for every
// size takes 51; a decode step of 16 rows of 32 heads 4.5 us where the kernel for few rows takes 27.  So every bfloat16 call that this
// one can take, of any number of rows, takes it.
typedef __bf16 hl_bf16x8_t __attribute__((ext_vector_type(8)));
typedef float hl_f32x4_t __attribute__((ext_vector_type(4)));
typedef uint16_t hl_u16x8_t __attribute__((ext_vector_type(8)));

template <int KS, int OT>
__global__ __launch_bounds__(256) void heads_linear_tiles_kernel(const uint16_t* __restrict__ x, long x_row, int x_head, int x_first,
                                                                 const uint16_t* __restrict__ w, bf16_t* __restrict__ y, long y_row, int y_head,
                                                                 int y_first, int n_rows, int n_out, int y_block_rows, int tiles_each) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, j = lane & 15, g = lane >> 4;
  const int head = blockIdx.y, o0 = 16 * OT * (4 * blockIdx.z + wave);
  if (o0 >= n_out) return;      // a wave without outputs
  hl_u16x8_t wv[OT][KS];
  const uint16_t* from = w + (size_t)head * (32 * KS) * n_out + (size_t)(8 * g) * n_out + j;
#pragma unroll
  for (int t = 0; t < OT; ++t) {
    const int o = min(o0 + 16 * t, n_out - 16);      // a tile beyond the last output repeats the last one and is not stored
#pragma unroll
    for (int k = 0; k < KS; ++k)
#pragma unroll
      for (int e = 0; e < 8; ++e) wv[t][k][e] = from[(size_t)(32 * k + e) * n_out + o];
  }
  const int first = blockIdx.x * tiles_each, last = min(first + tiles_each, (n_rows + 15) / 16);
  for (int tile = first; tile < last; ++tile) {
    const int row = 16 * tile + j;
    const uint16_t* in = x + (size_t)min(row, n_rows - 1) * x_row + (size_t)head * x_head + x_first + 8 * g;
    uint4 xv[KS];
#pragma unroll
    for (int k = 0; k < KS; ++k) xv[k] = *reinterpret_cast<const uint4*>(in + 32 * k);
    hl_f32x4_t acc[OT] = {};
#pragma unroll
    for (int k = 0; k < KS; ++k)
#pragma unroll
      for (int t = 0; t < OT; ++t)
        acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(hl_bf16x8_t, wv[t][k]), __builtin_bit_cast(hl_bf16x8_t, xv[k]), acc[t], 0, 0, 0);
    if (row >= n_rows) continue;
#pragma unroll
    for (int t = 0; t < OT; ++t)
      if (o0 + 16 * t < n_out)
        store_four(y + bh_rows_index(y_block_rows, row, head * y_head + y_first + o0 + 16 * t + 4 * g, (int)y_row), acc[t][0], acc[t][1], acc[t][2], acc[t][3]);
  }
}

template <int KS>
static void heads_linear_tiles(const uint16_t* x, long x_row, int x_head, int x_first, const uint16_t* w, bf16_t* y, long y_row, int y_head,
                               int y_first, int n_rows, int H, int n_out, int y_block_rows, hipStream_t stream) {
  // Few rows: a tile of outputs a wave, as many waves as there are.  Many: up to four tiles a wave, so that a row's inputs are read by
  // few waves, and eight tiles of rows, or fewer where that leaves compute units without two workgroups.
  const int out_tiles = n_out / 16, row_tiles = (n_rows + 15) / 16;
  constexpr int MOST = KS >= 7 ? 2 : KS >= 5 ? 3 : 4;      // what the registers hold
  const int ot = row_tiles == 1 ? 1 : (out_tiles + 3) / 4 < MOST ? (out_tiles + 3) / 4 : MOST;
  const int z = (out_tiles + 4 * ot - 1) / (4 * ot);
  int each = 8;
  while (each > 1 && (long)((row_tiles + each - 1) / each) * H * z < 2L * bh_compute_units()) each /= 2;
  const dim3 grid((row_tiles + each - 1) / each, H, z);
#define BH_HT(OT) \
  heads_linear_tiles_kernel<KS, OT><<<grid, 256, 0, stream>>>(x, x_row, x_head, x_first, w, y, y_row, y_head, y_first, n_rows, n_out, y_block_rows, each)
  if (ot == 1) BH_HT(1);
  else if (ot == 2) BH_HT(2);
  else if (ot == 3) BH_HT((MOST < 3 ? MOST : 3));
  else BH_HT(MOST);
#undef BH_HT
}

extern "C" int bh_heads_linear(const void* x, long x_row, int x_head, int x_first, const void* w, void* y, long y_row,
                               int y_head, int y_first, int dtype, int n_rows, int H, int n_in, int n_out, int y_block_rows,
                               hipStream_t stream) {
  BH_REQUIRE(y_block_rows == 0 || ((y_block_rows == 8 || y_block_rows == 16) && dtype == BH_BF16 && y_row % 32 == 0 && y_row < (1L << 31)),
             "heads_linear: an output in blocks of %d rows needs bfloat16 and rows of a multiple of 32 elements (got %ld)",
             y_block_rows, y_row);
  BH_REQUIRE(n_rows > 0 && H > 0 && n_in > 0 && n_out > 0, "heads_linear: sizes must be positive");
  BH_REQUIRE(H <= 65535 && (n_out + 255) / 256 <= 65535, "heads_linear: too many heads or outputs");
  BH_REQUIRE(x_first >= 0 && y_first >= 0 && x_first + n_in <= x_head && y_first + n_out <= y_head &&
                 (long)H * x_head <= x_row && (long)H * y_head <= y_row,
             "heads_linear: the heads' slices do not lie inside their rows");
  if (dtype == BH_BF16 && n_in % 32 == 0 && n_in <= 256 && n_out % 16 == 0 && (x_row | x_head | x_first) % 8 == 0 &&
      (y_row | y_head | y_first) % 4 == 0 && (uintptr_t)x % 16 == 0 && (uintptr_t)y % 8 == 0) {
#define BH_HLT(KS) \
  heads_linear_tiles<KS>((const uint16_t*)x, x_row, x_head, x_first, (const uint16_t*)w, (bf16_t*)y, y_row, y_head, y_first, n_rows, H, n_out, y_block_rows, stream)
    switch (n_in / 32) {
      case 1: BH_HLT(1); break;
      case 2: BH_HLT(2); break;
      case 3: BH_HLT(3); break;
      case 4: BH_HLT(4); break;
      case 5: BH_HLT(5); break;
      case 6: BH_HLT(6); break;
      case 7: BH_HLT(7); break;
      default: BH_HLT(8); break;
    }
#undef BH_HLT
    return bh_check_launch("heads_linear");
  }
  const size_t smem = (size_t)HL_ROWS * n_in * sizeof(float);
  BH_REQUIRE(smem <= 64 * 1024, "heads_linear: %d inputs a head are above the limit of %d", n_in, 64 * 1024 / 4 / HL_ROWS);
  if (n_rows <= HL_ROWS && smem + sizeof(float) * 3 * 64 * (HL_ROWS + 1) <= 64 * 1024) {      // (its partial sums need LDS too)
    dim3 few(1, H, (n_out + 63) / 64);
#define BH_HL_FEW(T)                                                                                                      \
  heads_linear_few_kernel<T><<<few, dim3(256), smem, stream>>>((const T*)x, x_row, x_head, x_first, (const T*)w, (T*)y, y_row, \
                                                               y_head, y_first, n_rows, n_in, n_out, y_block_rows)
    if (dtype == BH_F32) BH_HL_FEW(float);
    else if (dtype == BH_BF16) BH_HL_FEW(bf16_t);
    else return bh_fail("heads_linear: unknown dtype %d", dtype);
#undef BH_HL_FEW
    return bh_check_launch("heads_linear_few");
  }
  dim3 grid((n_rows + HL_ROWS - 1) / HL_ROWS, H, (n_out + 255) / 256), block(256);
#define BH_HL(T)                                                                                                         \
  heads_linear_kernel<T><<<grid, block, smem, stream>>>((const T*)x, x_row, x_head, x_first, (const T*)w, (T*)y, y_row, y_head, \
                                                        y_first, n_rows, n_in, n_out, y_block_rows)
  if (dtype == BH_F32) BH_HL(float);
  else if (dtype == BH_BF16) BH_HL(bf16_t);
  else return bh_fail("heads_linear: unknown dtype %d", dtype);
#undef BH_HL
  return bh_check_launch("heads_linear");
}

// ---- rotation of a slice of every head ------------------------------------------------------------------------
// y[row][h][y_first + i] = rotated x[row][h][x_first + i] for i < width: the first `turned` of them in pairs
// (i, i + turned/2) by the angle position[row] * freq[i], the rest as they are.
template <typename T>
__global__ void rotate_heads_kernel(const T* __restrict__ x, long x_row, int x_head, int x_first, T* __restrict__ y,
                                    long y_row, int y_head, int y_first, const float* __restrict__ freq, int turned,
                                    const int32_t* __restrict__ positions, int H, int width) {
  const int row = blockIdx.x;
  const float pos = (float)positions[row];
  const int half = turned / 2;
  for (int e = threadIdx.x; e < H * width; e += blockDim.x) {
    const int head = e / width, i = e % width;
    const T* from = x + (size_t)row * x_row + (size_t)head * x_head + x_first;
    float v;
    if (i < turned) {
      const int pair = i < half ? i : i - half;
      const float angle = pos * freq[pair];
      const float c = cosf(angle), s = sinf(angle);
      const float a = to_f32(from[pair]), b = to_f32(from[pair + half]);
      v = i < half ? a * c - b * s : b * c + a * s;
    } else {
      v = to_f32(from[i]);
    }
    y[(size_t)row * y_row + (size_t)head * y_head + y_first + i] = from_f32<T>(v);
  }
}

extern "C" int bh_rotate_heads(const void* x, long x_row, int x_head, int x_first, void* y, long y_row, int y_head,
                               int y_first, int dtype, const float* freq, int turned, const int32_t* positions, int n_rows,
                               int H, int width, hipStream_t stream) {
  BH_REQUIRE(n_rows > 0 && H > 0 && width > 0, "rotate_heads: sizes must be positive");
  BH_REQUIRE(turned >= 0 && turned % 2 == 0 && turned <= width, "rotate_heads: %d turned dimensions of %d", turned, width);
  BH_REQUIRE(turned == 0 || freq != nullptr, "rotate_heads: a rotation needs its frequencies");
  BH_REQUIRE(x_first >= 0 && y_first >= 0 && x_first + width <= x_head && y_first + width <= y_head &&
                 (long)H * x_head <= x_row && (long)H * y_head <= y_row,
             "rotate_heads: the heads' slices do not lie inside their rows");
#define BH_RH(T)                                                                                                          \
  rotate_heads_kernel<T><<<dim3(n_rows), dim3(256), 0, stream>>>((const T*)x, x_row, x_head, x_first, (T*)y, y_row, y_head, \
                                                                 y_first, freq, turned, positions, H, width)
  if (dtype == BH_F32) BH_RH(float);
  else if (dtype == BH_BF16) BH_RH(bf16_t);
  else return bh_fail("rotate_heads: unknown dtype %d", dtype);
#undef BH_RH
  return bh_check_launch("rotate_heads");
}
