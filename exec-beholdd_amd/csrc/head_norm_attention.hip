// What stands ahead of the paged attention kernels for an attention whose projections carry biases, whose queries and
// keys are normed head by head with one weight for all heads, and whose rotation turns the first dimensions of a head,
// dimension i with dimension i + turned/2:
//   head_norm_rope_write   per row of the stacked projection [q | k | v] (from column `first` of a wider row):
//                          x <- x + bias;  every head of q and k: x / sqrt(mean(x^2 over the head's dim) + eps) * w  (w [dim],
//                          the same for all heads; without w no norm);  dimensions i and i + turned/2 (i < turned/2) of every
//                          head of q and k turned by position * freq[i];  q into a matrix of heads of `pad` dimensions, k and v
//                          into the cache pages of (sequence, position) as heads of `pad` (zeros beyond dim and vdim), so that
//                          keys of one size and values of another go through kernels that know one head size.
//                          `unit_norm`: that norm without weights (a turn keeps a head's length, so it does not matter which of
//                          the two comes first).  `values_are_keys`: the row holds no v, a head's value is its key as it stands
//                          there, ahead of norm and turn; one wave then writes both.
// Sums, statistics, angles, cosines and sines are float32; the angle is the float32 product position * freq[i].
#include "common.h"

#define HN_WAVES 4

// A workgroup a row and a stretch of `per_group` heads (the heads of q, then those of k, then those of v, numbered through), a
// wave a head at a time.  The head stands in the wave's own stretch of LDS between the statistic and the rotation, which
// needs a dimension's mate.  Few rows: a stretch is one head a wave, so that a decode step's heads run side by side.
template <typename T>
__global__ __launch_bounds__(HN_WAVES * BH_WAVE) void head_norm_rope_write_kernel(
    const T* __restrict__ proj, int row_stride, int first, const float* __restrict__ bias, const float* __restrict__ wq,
    const float* __restrict__ wk, float eps, const float* __restrict__ freq, int turned, const int32_t* __restrict__ positions,
    const int32_t* __restrict__ row_seq, T* __restrict__ q_out, T* __restrict__ k_pages, T* __restrict__ v_pages,
    const int32_t* __restrict__ page_table, int table_stride, int H, int G, int dim, int vdim, int pad, int kv_order, int write,
    int per_group, int neighbours, float magnitude, int unit_norm, int values_are_keys) {
  extern __shared__ float lds[];      // the cosines and sines of the row's turned pairs, then a head of `dim` floats a wave
  const int row = blockIdx.x, wave = threadIdx.x / BH_WAVE, lane = threadIdx.x % BH_WAVE;
  const int half = turned / 2;
  float* cosines = lds;
  float* sines = lds + half;
  float* mine = lds + turned + wave * dim;
  const int pos = positions[row];
  for (int i = threadIdx.x; i < half; i += blockDim.x) {
    const float angle = (float)pos * freq[i];
    cosines[i] = cosf(angle) * magnitude;
    sines[i] = sinf(angle) * magnitude;
  }
  __syncthreads();
  const T* x = proj + (size_t)row * row_stride + first;
  const int q_width = H * dim, k_width = G * dim;
  int page = 0;
  const int token = pos % BH_PAGE;
  if (write) page = page_table[(size_t)row_seq[row] * table_stride + pos / BH_PAGE];
  const int heads = write ? (values_are_keys ? H + G : H + 2 * G) : H;
  const int stretch_end = ((int)blockIdx.y + 1) * per_group < heads ? ((int)blockIdx.y + 1) * per_group : heads;
  for (int unit = blockIdx.y * per_group + wave; unit < stretch_end; unit += HN_WAVES) {
    if (unit >= H + G) {      // a head of values: the bias, and zeros beyond vdim
      const int head = unit - H - G, at = q_width + k_width + head * vdim;
      T* values = v_pages + ((size_t)page * G + head) * BH_PAGE * pad;
      for (int i = lane; i < pad; i += BH_WAVE) {
        const float v = i < vdim ? to_f32(x[at + i]) + (bias ? bias[at + i] : 0.f) : 0.f;
        values[bh_value_index(kv_order, token, i, pad)] = from_f32<T>(v);
      }
      continue;
    }
    const bool is_key = unit >= H;
    const int head = is_key ? unit - H : unit, at = (is_key ? q_width : 0) + head * dim;
    const float* w = is_key ? wk : wq;
    float ss = 0.f;
    for (int i = lane; i < dim; i += BH_WAVE) {
      const float v = to_f32(x[at + i]) + (bias ? bias[at + i] : 0.f);
      mine[i] = v;
      ss += v * v;
    }
    ss = wave_sum(ss);
    const float inv = w || unit_norm ? 1.0f / sqrtf(ss / (float)dim + eps) : 1.0f;
    // (a wave's lanes run together: what the lanes wrote above is there for all of them below)
    __builtin_amdgcn_wave_barrier();
    T* keys = is_key ? k_pages + ((size_t)page * G + head) * BH_PAGE * pad : nullptr;
    T* queries = q_out + ((size_t)row * H + head) * pad;
    if (is_key && values_are_keys) {
      T* values = v_pages + ((size_t)page * G + head) * BH_PAGE * pad;
      for (int i = lane; i < pad; i += BH_WAVE) values[bh_value_index(kv_order, token, i, pad)] = from_f32<T>(i < dim ? mine[i] : 0.f);
    }
    for (int i = lane; i < pad; i += BH_WAVE) {
      float y = 0.f;
      if (i < dim) {
        y = mine[i] * inv * (w ? w[i] : 1.f);
        if (i < turned) {
          // the pair's mate: i + half and i - half, or the neighbour (2 pair, 2 pair + 1)
          const int pair = neighbours ? i / 2 : (i < half ? i : i - half);
          const bool is_first = neighbours ? (i % 2 == 0) : (i < half);
          const int mate = neighbours ? (i ^ 1) : (i < half ? i + half : i - half);
          const float other = mine[mate] * inv * (w ? w[mate] : 1.f);
          const float c = cosines[pair], s = sines[pair];
          y = is_first ? y * c - other * s : y * c + other * s;
        }
      }
      if (is_key) keys[bh_key_index(kv_order, token, i, pad)] = from_f32<T>(y);
      else queries[i] = from_f32<T>(y);
    }
    __builtin_amdgcn_wave_barrier();
  }
}

// The same for steps of many rows, in pieces of four dimensions: the lanes of a head (pad / 4 of them, neighbours) keep it in registers, add its
// squares up by exchanges and ask the mate of a half-split turn for its piece; a thread asks for the pieces of HEADS heads at once.  The
// kernel above goes through one head a wave after the other, an element a lane.  Bound by its bytes and, a third of it, the values,
// whose tokens lie two bytes apart.  32 heads of 128 on 8, 64 dimensions turned: 2,048 rows 42.3 -> 29.6 us, 8,192 rows 144 -> 98.
template <typename T, int HEADS>
__global__ __launch_bounds__(HN_WAVES * BH_WAVE) void head_norm_rope_write_pieces_kernel(
    const T* __restrict__ proj, int row_stride, int first, const float* __restrict__ bias, const float* __restrict__ wq,
    const float* __restrict__ wk, float eps, const float* __restrict__ freq, int turned, const int32_t* __restrict__ positions,
    const int32_t* __restrict__ row_seq, T* __restrict__ q_out, T* __restrict__ k_pages, T* __restrict__ v_pages,
    const int32_t* __restrict__ page_table, int table_stride, int H, int G, int dim, int vdim, int pad, int kv_order, int write,
    int neighbours, float magnitude, int unit_norm, int values_are_keys, int n_rows) {
  extern __shared__ float lds[];      // the cosines and sines of the row's turned pairs
  const int row = bh_row_of_block<true>();      // 16 neighbours to an XCD: rows meet in the cache's lines
  if (row >= n_rows) return;
  const int half = turned / 2, lanes = pad / 4, lane = threadIdx.x % BH_WAVE, at_once = blockDim.x / lanes;
  const int i = threadIdx.x % lanes * 4, place = threadIdx.x / lanes, unit0 = blockIdx.y * HEADS * at_once + place;
  float* cosines = lds;
  float* sines = lds + half;
  const int pos = positions[row], token = pos % BH_PAGE;
  int page = 0;
  if (write) page = page_table[(size_t)row_seq[row] * table_stride + pos / BH_PAGE];
  const T* x = proj + (size_t)row * row_stride + first;
  const int q_width = H * dim, k_width = G * dim, heads = write ? (values_are_keys ? H + G : H + 2 * G) : H;
  const float4 zero = make_float4(0.f, 0.f, 0.f, 0.f);
  float4 held[HEADS];
#pragma unroll
  for (int u = 0; u < HEADS; ++u) {
    const int unit = unit0 + u * at_once;
    const bool is_value = unit >= H + G;
    const int at = is_value ? q_width + k_width + (unit - H - G) * vdim + i : unit * dim + i;      // (the heads of k stand behind those of q)
    held[u] = zero;
    if (unit < heads && i < (is_value ? vdim : dim)) {
      held[u] = load_four(x + at);
      if (bias) {
        const float4 b = load_four(bias + at);
        held[u].x += b.x, held[u].y += b.y, held[u].z += b.z, held[u].w += b.w;
      }
    }
  }
  for (int j = threadIdx.x; j < half; j += blockDim.x) {
    const float angle = (float)pos * freq[j];
    cosines[j] = cosf(angle) * magnitude;
    sines[j] = sinf(angle) * magnitude;
  }
  __syncthreads();
  const bool turns = i < turned;
  const int pair = neighbours ? i / 2 : (i < half ? i : i - half);      // the angles: of two pairs of neighbours, or of four halves' pairs
  float c[4] = {1.f, 1.f, 1.f, 1.f}, s[4] = {0.f, 0.f, 0.f, 0.f};
  if (turns) {
#pragma unroll
    for (int j = 0; j < 4; ++j) c[j] = cosines[neighbours ? pair + j / 2 : pair + j], s[j] = sines[neighbours ? pair + j / 2 : pair + j];
  }
  const int mate_lane = neighbours || !turns ? lane : i < half ? lane + half / 4 : lane - half / 4;
#pragma unroll
  for (int u = 0; u < HEADS; ++u) {
    const int unit = unit0 + u * at_once;
    const bool is_value = unit >= H + G, is_key = unit >= H && !is_value;
    float ss = held[u].x * held[u].x + held[u].y * held[u].y + held[u].z * held[u].z + held[u].w * held[u].w;
    for (int off = lanes / 2; off > 0; off >>= 1) ss += __shfl_xor(ss, off, BH_WAVE);
    const float* w = is_key ? wk : wq;
    const float inv = w || unit_norm ? 1.0f / sqrtf(ss / (float)dim + eps) : 1.0f;
    float y[4] = {0.f, 0.f, 0.f, 0.f};      // beyond dim, whatever the norm's factor is
    if (i < dim) y[0] = held[u].x * inv, y[1] = held[u].y * inv, y[2] = held[u].z * inv, y[3] = held[u].w * inv;
    if (w && i < dim) {
      const float4 scale = load_four(w + i);
      y[0] *= scale.x, y[1] *= scale.y, y[2] *= scale.z, y[3] *= scale.w;
    }
    float mate[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) mate[j] = neighbours ? y[j ^ 1] : __shfl(y[j], mate_lane, BH_WAVE);
    if (unit >= heads) continue;      // (a head's lanes together, behind their exchanges)
    if (is_value || (is_key && values_are_keys)) {
      T* values = v_pages + ((size_t)page * G + (is_value ? unit - H - G : unit - H)) * BH_PAGE * pad;
      const float four[4] = {held[u].x, held[u].y, held[u].z, held[u].w};
#pragma unroll
      for (int j = 0; j < 4; ++j) values[bh_value_index(kv_order, token, i + j, pad)] = from_f32<T>(four[j]);
      if (is_value) continue;
    }
    if (turns) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const bool is_first = neighbours ? j % 2 == 0 : i < half;
        y[j] = is_first ? y[j] * c[j] - mate[j] * s[j] : y[j] * c[j] + mate[j] * s[j];
      }
    }
    if (is_key) store_four(k_pages + ((size_t)page * G + unit - H) * BH_PAGE * pad + bh_key_index(kv_order, token, i, pad), y[0], y[1], y[2], y[3]);
    else store_four(q_out + ((size_t)row * H + unit) * pad + i, y[0], y[1], y[2], y[3]);
  }
}

// proj [n_rows][row_stride]: a row holds, from `first`, H heads of q and G heads of k of `dim` and G heads of v of `vdim`;
// bias f32 over those channels, or null; wq, wk f32 [dim], both or neither.  Pages as the attention kernels take them for G
// kv heads of size `pad` (written when `write` is set); q_out [n_rows][H * pad].  `neighbours`: a turned pair is
// dimensions 2i and 2i + 1 instead of i and i + turned/2; `magnitude` multiplies every cosine and sine.
extern "C" int bh_head_norm_rope_write(const void* proj, int dtype, int row_stride, int first, const float* bias, const float* wq,
                                       const float* wk, float eps, const float* freq, int turned, const int32_t* positions,
                                       const int32_t* row_seq, void* q_out, void* k_pages, void* v_pages, const int32_t* page_table,
                                       int table_stride, int n_rows, int H, int G, int dim, int vdim, int pad, int kv_order, int write,
                                       int neighbours, float magnitude, int unit_norm, int values_are_keys, hipStream_t stream) {
  BH_REQUIRE(n_rows > 0 && H > 0 && G > 0 && dim > 0 && vdim > 0, "head_norm_rope_write: sizes must be positive");
  BH_REQUIRE(pad >= dim && pad >= vdim, "head_norm_rope_write: heads of %d do not hold keys of %d and values of %d", pad, dim, vdim);
  BH_REQUIRE(turned >= 0 && turned % 2 == 0 && turned <= dim, "head_norm_rope_write: %d turned dimensions of %d", turned, dim);
  BH_REQUIRE(turned == 0 || freq != nullptr, "head_norm_rope_write: a rotation needs its frequencies");
  BH_REQUIRE((wq == nullptr) == (wk == nullptr), "head_norm_rope_write: give both norm weights or neither");
  BH_REQUIRE(!unit_norm || wq == nullptr, "head_norm_rope_write: a norm without weights has none");
  BH_REQUIRE(!values_are_keys || vdim == dim, "head_norm_rope_write: values that are keys of %d have that size, not %d", dim, vdim);
  // (without `write` a row may hold queries alone)
  BH_REQUIRE(first >= 0 && first + H * dim + (write ? G * dim + (values_are_keys ? 0 : G * vdim) : 0) <= row_stride, "head_norm_rope_write: q, k and v lie outside a row of %d", row_stride);
  BH_REQUIRE(kv_order == BH_KV_ROWS || (kv_order == BH_KV_PIECES && pad % 32 == 0),
             "head_norm_rope_write: cache order %d does not exist for head size %d", kv_order, pad);
  const size_t lds = (size_t)(turned + HN_WAVES * dim) * sizeof(float);
  BH_REQUIRE(lds <= 48 * 1024, "head_norm_rope_write: heads of %d dimensions do not fit the local memory", dim);
  const int heads = write ? (values_are_keys ? H + G : H + 2 * G) : H;
  // Rows for every compute unit, heads that fill a wave or many rows, whole pieces of four in both halves of a turn, heads of a power of two up to a wave's
  // lanes.  An element / four a thread, us, all dimensions turned, bfloat16: 16 heads of 128 on 4 256 rows 6.8 / 5.5, 4,096 rows 46 / 27; 4 of 64 on
  // 2 256 rows 4.6 / 4.8, 4,096 rows 15.2 / 8.5; 2 of 32 on 1, half a wave, 4,096 rows 10.4 / 6.6, but 256 rows 4.3 / 4.8, 1,024 rows 5.1 / 5.2.
  const size_t piece = 4 * (dtype == BH_F32 ? sizeof(float) : 2);
  if (n_rows >= bh_compute_units() && bh_rows_spread(n_rows, 16) && (heads * (pad / 4) >= BH_WAVE || n_rows > 4 * bh_compute_units()) && (pad == 32 || pad == 64 || pad == 128 || pad == 256) && dim % 4 == 0 && vdim % 4 == 0 && turned % (neighbours ? 4 : 8) == 0 &&
      first % 4 == 0 && row_stride % 4 == 0 && ((uintptr_t)proj | (uintptr_t)q_out | (uintptr_t)k_pages) % piece == 0 &&
      ((uintptr_t)bias | (uintptr_t)wq | (uintptr_t)wk) % 16 == 0 && (dtype == BH_F32 || dtype == BH_BF16)) {
    // As many heads a thread as leave no more than eight waves a row, and no waves without a head; rows that do not fill the chip: one.
    const int lanes = heads * (pad / 4), most = HN_WAVES * BH_WAVE;
    const int each = lanes <= most || n_rows < 4 * bh_compute_units() ? 1 : lanes <= 2 * most ? 2 : 4;
    const int threads = std::min(most, ((lanes + each - 1) / each + BH_WAVE - 1) / BH_WAVE * BH_WAVE), at_once = each * (threads / (pad / 4));
    const dim3 stretches(bh_rows_grid(n_rows, 16), (heads + at_once - 1) / at_once);
    BH_REQUIRE(stretches.y <= 65535, "head_norm_rope_write: too many heads");
#define BH_HNP(T, HEADS)                                                                                                           \
  head_norm_rope_write_pieces_kernel<T, HEADS><<<stretches, threads, turned * sizeof(float), stream>>>(                            \
      (const T*)proj, row_stride, first, bias, wq, wk, eps, freq, turned, positions, row_seq, (T*)q_out, (T*)k_pages, (T*)v_pages, page_table, \
      table_stride, H, G, dim, vdim, pad, kv_order, write, neighbours, magnitude, unit_norm, values_are_keys, n_rows)
    if (dtype == BH_F32) {
      if (each == 1) BH_HNP(float, 1);
      else if (each == 2) BH_HNP(float, 2);
      else BH_HNP(float, 4);
    } else {
      if (each == 1) BH_HNP(bf16_t, 1);
      else if (each == 2) BH_HNP(bf16_t, 2);
      else BH_HNP(bf16_t, 4);
    }
#undef BH_HNP
    return bh_check_launch("head_norm_rope_write");
  }
  const int per_group = n_rows >= 4 * bh_compute_units() ? 4 * HN_WAVES : HN_WAVES;      // many rows fill the chip by themselves
  const dim3 grid(n_rows, (heads + per_group - 1) / per_group);
  BH_REQUIRE(grid.y <= 65535, "head_norm_rope_write: too many heads");
#define BH_HN(T)                                                                                                                  \
  head_norm_rope_write_kernel<T><<<grid, HN_WAVES * BH_WAVE, lds, stream>>>((const T*)proj, row_stride, first, bias, wq, wk, eps, freq, \
                                                                           turned, positions, row_seq, (T*)q_out, (T*)k_pages,    \
                                                                           (T*)v_pages, page_table, table_stride, H, G, dim, vdim, \
                                                                           pad, kv_order, write, per_group, neighbours, magnitude, unit_norm, values_are_keys)
  if (dtype == BH_F32) BH_HN(float);
  else if (dtype == BH_BF16) BH_HN(bf16_t);
  else return bh_fail("head_norm_rope_write: unknown dtype %d", dtype);
#undef BH_HN
  return bh_check_launch("head_norm_rope_write");
}
