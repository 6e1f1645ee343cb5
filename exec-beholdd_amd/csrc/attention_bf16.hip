// bfloat16 attention over the paged cache on the gfx950 matrix cores: the kernel for few columns per
// sequence (decode, short steps) and the entry point, which hands steps with many columns per sequence
// to the prefill kernel (attention_prefill_bf16.hip).
//
// A *column* is one (row, query head) pair.  A workgroup takes 16 columns that share a sequence
// and a kv head (consecutive rows x the heads of one group) and a range of that sequence's cache
// pages; its four waves take the pages of the range in turn.  For each page of 64 keys a wave
// computes, with v_mfma_f32_16x16x32_bf16,
//     S^T[key, column] = K[key, :] . Q[column, :]        (keys as rows: K is loaded straight from
//                                                          the cache in operand layout)
//     running maximum / sum per column in float32 (online softmax, exponent base 2)
//     O^T[d, column] += V^T[d, key] . P^T[key, column]   (the cache keeps V transposed inside a
//                                                          page, so this operand is a straight load too)
// The rows of an S^T tile are assigned to keys so that every lane ends up with the keys its P^T
// operand needs: tile t, row i <-> key 32*(t/2) + 4*(t%2) + 8*(i/4) + i%4.  Lane (column j, group g)
// then holds keys 8g..8g+7 (tiles 0, 1) and 32+8g..32+8g+7 (tiles 2, 3): the k-slices of the two
// P.V products of a page, whose V^T operands are 16 contiguous bytes per lane and 64 contiguous
// bytes per row and instruction.  The same holds for K along head_dim.
// The waves' results are merged through LDS.  When the keys of a sequence are split over several
// workgroups (decode: few columns, long caches) each writes an unnormalised partial result and
// its (maximum, sum) to scratch memory and a second kernel combines them.  (Letting the last
// workgroup combine, behind a device-wide fence and an arrival counter, was measured: the fences
// write back the L2 of every workgroup's XCD and cost several times what the second launch costs.)
//
// head_dim must be a multiple of 32, at most 256.  Masking is by position: column j sees keys
// lo_j .. pos_j.  Rows of a page beyond the last written key are never multiplied in: their
// probabilities are zero and their V values are zeroed before use.
#include "attention_bf16.h"
#include <type_traits>

// A decode step can hand the kernel the fused projection rows themselves (struct FusedQkv) instead of
// finished queries and a cache that already holds the new keys: every workgroup then norms and rotates
// its own queries (a fifth wave for the four with the pages, or, in the lean form, each wave for itself), and one
// wave of the sequence's last split norms and rotates the new key, attends to it with one product of it and the
// queries and to the new value in plain float32, and writes both into the cache for the steps to come.  The keys
// that come from the cache end one position earlier.  This takes the place of the launch of the
// norm/rotation/cache-write kernel.
//
// The rows' heads come in one of two forms.  Whole heads turned in split halves by tables over positions (FUSED 1: HeadPrep);
// or the first `turned` dimensions in neighbouring pairs by cosines and sines of the step's rows (FUSED 2: PairPrep), with the
// norm's weights optional, in rows of any stride whose values may be the projected keys themselves.
struct FusedQkv {
  const uint16_t* qkv;      // one row per sequence: H heads of q from column 0; null: queries and cache are ready
  int row_stride;           // elements from one row to the next
  int k_first, v_first;     // where a row's keys and its values begin (the same column: a value is its raw key)
  int turned;               // FUSED 2: how many of a head's first dimensions turn
  int unit_norm;            // FUSED 2: without weights the heads are still brought to unit root mean square
  const void* q_weight;     // per-head RMSNorm weights [head_dim], or null for no norm
  const void* k_weight;
  int weight_f32;           // their element type: float32, else bfloat16
  float eps;
  const float* cos_table;   // [positions][head_dim / 2]: rotation over the whole head (FUSED 2: [rows][turned / 2]), or null for none
  const float* sin_table;
  int write_kv;             // 0: the cache entry belongs to another layer, which has written the new key already
  uint16_t* k_pages;        // the cache again, to write into
  uint16_t* v_pages;
};

// What a lane needs to norm and rotate its share of a head (elements 32 s + 8 g + e; the other three g share
// the head): asked for early (`ask`), used late (`apply`), so that the loads of the first cache page can be
// under way in between.
template <int NS>
struct HeadPrep {
  static constexpr int HD = 32 * NS, HS = NS / 2;
  u32x4_t weight_raw[NS][2];   // bfloat16 weights fill the first of each pair, float32 both
  float cos_v[HS > 0 ? HS : 1][8], sin_v[HS > 0 ? HS : 1][8];

  __device__ inline void ask(const void* weight, int weight_f32, const float* cos_table, const float* sin_table,
                             int pos, int g) {
    if (weight != nullptr) {
#pragma unroll
      for (int s = 0; s < NS; ++s) {
        const int i = 32 * s + 8 * g;
        if (weight_f32) {
          weight_raw[s][0] = *reinterpret_cast<const u32x4_t*>(reinterpret_cast<const float*>(weight) + i);
          weight_raw[s][1] = *reinterpret_cast<const u32x4_t*>(reinterpret_cast<const float*>(weight) + i + 4);
        } else {
          weight_raw[s][0] = load16(reinterpret_cast<const uint16_t*>(weight) + i);
        }
      }
    }
    if (cos_table != nullptr) {
#pragma unroll
      for (int s = 0; s < HS; ++s)
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const int i = 32 * s + 8 * g + e;
          cos_v[s][e] = cos_table[(size_t)pos * (HD / 2) + i];
          sin_v[s][e] = sin_table[(size_t)pos * (HD / 2) + i];
        }
    }
  }

  __device__ inline void take_angles(const HeadPrep& other) {
#pragma unroll
    for (int s = 0; s < HS; ++s)
#pragma unroll
      for (int e = 0; e < 8; ++e) cos_v[s][e] = other.cos_v[s][e], sin_v[s][e] = other.sin_v[s][e];
  }

  // RMSNorm over the head, then split-half rotation: the partner of element i < HD / 2 is i + HD / 2, in the
  // same lane, HS slices on.
  __device__ inline void apply(float (&x)[NS][8], bool with_weight, int weight_f32, float eps, bool with_rotation) const {
    if (with_weight) {
      float ss = 0.f;
#pragma unroll
      for (int s = 0; s < NS; ++s)
#pragma unroll
        for (int e = 0; e < 8; ++e) ss += x[s][e] * x[s][e];
      ss += __shfl_xor(ss, 16, 64);
      ss += __shfl_xor(ss, 32, 64);
      const float inv = 1.0f / sqrtf(ss / (float)HD + eps);
#pragma unroll
      for (int s = 0; s < NS; ++s)
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const float w = weight_f32 ? __uint_as_float(weight_raw[s][e / 4][e % 4])
                                     : bf16_bits_to_f32((uint16_t)(weight_raw[s][0][e / 2] >> (16 * (e % 2))));
          x[s][e] = x[s][e] * inv * w;
        }
    }
    if (with_rotation) {
#pragma unroll
      for (int s = 0; s < HS; ++s)
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const float lo = x[s][e], hi = x[s + HS][e];
          x[s][e] = lo * cos_v[s][e] - hi * sin_v[s][e];
          x[s + HS][e] = lo * sin_v[s][e] + hi * cos_v[s][e];
        }
    }
  }
};

// The same for FUSED 2: a turned pair is dimensions 2i and 2i + 1, both in one lane; `row` is the row of the cosines and sines.
template <int NS>
struct PairPrep {
  static constexpr int HD = 32 * NS;
  u32x4_t weight_raw[NS][2];
  float cos_v[NS][4], sin_v[NS][4];

  __device__ inline void ask(const void* weight, int weight_f32) {
    if (weight != nullptr) {
#pragma unroll
      for (int s = 0; s < NS; ++s) {
        const int i = 32 * s + 8 * ((threadIdx.x % 64) / 16);
        if (weight_f32) {
          weight_raw[s][0] = *reinterpret_cast<const u32x4_t*>(reinterpret_cast<const float*>(weight) + i);
          weight_raw[s][1] = *reinterpret_cast<const u32x4_t*>(reinterpret_cast<const float*>(weight) + i + 4);
        } else {
          weight_raw[s][0] = load16(reinterpret_cast<const uint16_t*>(weight) + i);
        }
      }
    }
  }
  __device__ inline void ask_angles(const float* cos_rows, const float* sin_rows, int turned, int row, int g) {
    const int half = turned / 2;
#pragma unroll
    for (int s = 0; s < NS; ++s)
#pragma unroll
      for (int p = 0; p < 4; ++p) {
        const int pair = 16 * s + 4 * g + p;
        cos_v[s][p] = pair < half ? cos_rows[(size_t)row * half + pair] : 1.f;
        sin_v[s][p] = pair < half ? sin_rows[(size_t)row * half + pair] : 0.f;
      }
  }
  __device__ inline void take_angles(const PairPrep& other) {
#pragma unroll
    for (int s = 0; s < NS; ++s)
#pragma unroll
      for (int p = 0; p < 4; ++p) cos_v[s][p] = other.cos_v[s][p], sin_v[s][p] = other.sin_v[s][p];
  }
  __device__ inline void apply(float (&x)[NS][8], bool with_norm, bool with_weight, int weight_f32, float eps, bool with_rotation) const {
    if (with_norm) {
      float ss = 0.f;
#pragma unroll
      for (int s = 0; s < NS; ++s)
#pragma unroll
        for (int e = 0; e < 8; ++e) ss += x[s][e] * x[s][e];
      ss += __shfl_xor(ss, 16, 64);
      ss += __shfl_xor(ss, 32, 64);
      const float inv = 1.0f / sqrtf(ss / (float)HD + eps);
#pragma unroll
      for (int s = 0; s < NS; ++s)
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          float w = 1.f;
          if (with_weight)
            w = weight_f32 ? __uint_as_float(weight_raw[s][e / 4][e % 4])
                           : bf16_bits_to_f32((uint16_t)(weight_raw[s][0][e / 2] >> (16 * (e % 2))));
          x[s][e] = x[s][e] * inv * w;
        }
    }
    if (with_rotation) {
#pragma unroll
      for (int s = 0; s < NS; ++s)
#pragma unroll
        for (int p = 0; p < 4; ++p) {
          const float a = x[s][2 * p], b = x[s][2 * p + 1];
          x[s][2 * p] = a * cos_v[s][p] - b * sin_v[s][p];
          x[s][2 * p + 1] = b * cos_v[s][p] + a * sin_v[s][p];
        }
    }
  }
};

template <int NS>
__device__ inline void widen_head(float (&x)[NS][8], const u32x4_t (&raw)[NS]) {
#pragma unroll
  for (int s = 0; s < NS; ++s)
#pragma unroll
    for (int e = 0; e < 8; ++e) x[s][e] = bf16_bits_to_f32((uint16_t)(raw[s][e / 2] >> (16 * (e % 2))));
}

template <int NS>
__device__ inline void pack_head(u32x4_t (&out)[NS], const float (&x)[NS][8]) {
#pragma unroll
  for (int s = 0; s < NS; ++s)
#pragma unroll
    for (int word = 0; word < 4; ++word) out[s][word] = pack_bf16(x[s][2 * word], x[s][2 * word + 1]);
}

// NS = head_dim / 32.
// STREAM = one workgroup per (sequence, kv head, split): each cache byte is read once, past the caches.
// FUSED = the step is a decode step and `fused.qkv` is given, in form 1 or 2 (struct FusedQkv).
// LEAN (with FUSED) = the queries are normed and rotated before the first page is asked for, and the new key's
// numbers are asked for after the last page: nothing of that overlaps with the pages any more, but four waves do with what they
// have, so that two workgroups fit a compute unit (a fifth wave a workgroup would be a third one on some SIMDs, whose
// registers are two waves').  For launches of more workgroups than compute units, where the second workgroup is worth more
// than the overlap; and for heads of more than 128, which went to scratch memory with all of it in registers (16 sequences of
// 1,000 to 2,000 keys, 16 heads on 8, the launch and its combining: of 256 119.8 -> 38.0 us, of 192 41.6 -> 29.8).
// FORMED = scores are more than a scaled product (struct ScoreForm): they are made in full, and exponentials taken of them as they
// are (scale_log2 is then log2(e)).  Otherwise a column's factor is in scale_log2 (ScoreForm::scaled_only).
// A workgroup of a FUSED step that is not LEAN has a fifth wave (heads of up to 128, whose pages leave two waves a SIMD their registers):
// it norms and rotates the queries for all of them, while the others ask for their first pages and nothing else, and then takes the new
// key, beside the pages.  (Every wave its own queries under its first page's loads, and the new key by the first wave behind its pages:
// 4 sequences of 1,000 keys, 16 heads on 4 11.5 us with the combining, 9.4 now, in a chain of such launches, of which more is the
// combining's and the merge's.  The lean form in its place: 5 to 9 % of the launch slower where a page is all, within 5 % either way at up
// to 24 pages a workgroup.)
__host__ __device__ constexpr bool fifth_wave(int ns, int fused, bool lean) { return fused && !lean && ns <= 4; }
template <int NS, bool STREAM, int FUSED, bool LEAN = false, int FORMED = 0>
__global__ __launch_bounds__((fifth_wave(NS, FUSED, LEAN) ? 320 : 256), (LEAN && NS <= 4 ? 2 : 1)) void attention_mfma_kernel(
    const uint16_t* __restrict__ q, uint16_t* __restrict__ out, float* __restrict__ part_o,
    float* __restrict__ part_ml, const uint16_t* __restrict__ k_pages, const uint16_t* __restrict__ v_pages,
    const int32_t* __restrict__ page_table, int table_stride, const int32_t* __restrict__ positions,
    const int32_t* __restrict__ seq_start, int H, int KVH, int window, int n_splits,
    int pages_per_split, int tile_groups, FusedQkv fused, int out_block_rows, HeadEnd finish, ScoreForm form) {
  constexpr int HD = 32 * NS, WAVES = fifth_wave(NS, FUSED, LEAN) ? 5 : 4;
  __shared__ u32x4_t sm_q[WAVES == 5 ? NS : 1][64];
  __shared__ float sm_m[WAVES][16];
  __shared__ float sm_l[WAVES][16];
  __shared__ __attribute__((aligned(16))) float sm_o[WAVES][16][HD + 4];      // rows of 16-byte pieces, 4 banks apart

  const int tile = blockIdx.x % tile_groups, unit = blockIdx.x / tile_groups;
  const int kvh = unit % KVH, z = unit / KVH;
  const int seq = z / n_splits, split = z % n_splits;
  const int G = H / KVH;
  // FUSED is a decode step: sequence s has the one row s, and nobody waits for `seq_start` to say so
  const int row0 = FUSED ? seq : seq_start[seq];
  const int n_cols = FUSED ? G : (seq_start[seq + 1] - row0) * G;
  if (tile * 16 >= n_cols) return;
  // The number of this wave's first page, if no window cuts the front off, is asked for beside the row's position
  // instead of after it: one trip to memory less before the first key is on its way.
  const int32_t* table = page_table + (size_t)seq * table_stride;
  const int first_guess = split * pages_per_split + (int)(threadIdx.x / 64);
  const int page_guess = first_guess < table_stride ? table[first_guess] : 0;

  // (a scalar: the fifth wave's way parts from the others', with a barrier on both)
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), lane = threadIdx.x % 64;
  const int j = lane % 16, g = lane / 16;
  const int wanted = tile * 16 + j;
  const int c = wanted < n_cols ? wanted : n_cols - 1;
  const int row = row0 + c / G, head = kvh * G + c % G;
  const int pos_row = positions[row];                   // the row's own position
  const bool new_key_apart = FUSED && fused.write_kv;   // the key at pos_row is not in the cache yet
  const int pos = new_key_apart ? pos_row - 1 : pos_row;   // the last key the row takes from the cache (-1: none)
  const int lo = bh_first_visible(pos_row, window);
  // what this lane's column makes of its products (FORMED), and of its scores or else its products into powers of two
  const float scale_log2 = FORMED ? BH_LOG2E : query_scale(form, pos_row) * BH_LOG2E;
  const float col_scale = FORMED ? query_scale(form, pos_row) : 0.f, cap_rate = FORMED == 2 ? 2.0f * BH_LOG2E / form.cap : 0.f;
  const float slope = FORMED && form.slopes ? form.slopes[head] : 0.f;
  bf16x8_t q_vec[NS];
  // FUSED: the raw rows and what norms and rotates them.
  u32x4_t q_raw[NS], k_raw[NS];
  uint16_t new_value[2 * NS];   // dim 16 dt + j of the new value, as the cache takes it
  u32x2_t value_raw[2 * NS];    // dims 16 dt + 4 g .. + 3 of it, as the lane's sums do
  std::conditional_t<FUSED == 2, PairPrep<NS>, HeadPrep<NS>> q_prep, k_prep;
  const bool new_key_here = FUSED && fused.write_kv && split == n_splits - 1, takes_new_key = new_key_here && wave == (WAVES == 5 ? 4 : 0);
  auto ask_new_key = [&]() {   // one row per sequence: every lane's row is this row
    const uint16_t* qkv_row = fused.qkv + (size_t)row * fused.row_stride;
#pragma unroll
    for (int s = 0; s < NS; ++s) k_raw[s] = load16(qkv_row + fused.k_first + kvh * HD + 32 * s + 8 * g);
#pragma unroll
    for (int dt = 0; dt < 2 * NS; ++dt) {
      new_value[dt] = qkv_row[fused.v_first + kvh * HD + 16 * dt + j];
      value_raw[dt] = *reinterpret_cast<const u32x2_t*>(qkv_row + fused.v_first + kvh * HD + 16 * dt + 4 * g);
    }
    // the rotation's numbers are q's, or (LEAN: q's are gone by then) asked for again
    if constexpr (FUSED == 2) {
      k_prep.ask(fused.k_weight, fused.weight_f32);
      if (LEAN && fused.cos_table) k_prep.ask_angles(fused.cos_table, fused.sin_table, fused.turned, row, g);
    } else {
      k_prep.ask(fused.k_weight, fused.weight_f32, LEAN ? fused.cos_table : nullptr, LEAN ? fused.sin_table : nullptr, pos_row, g);
    }
  };
  auto ask_q = [&]() {
    const uint16_t* qkv_row = fused.qkv + (size_t)row * fused.row_stride;
#pragma unroll
    for (int s = 0; s < NS; ++s) q_raw[s] = load16(qkv_row + (size_t)head * HD + 32 * s + 8 * g);
    if constexpr (FUSED == 2) {
      q_prep.ask(fused.q_weight, fused.weight_f32);
      if (fused.cos_table) q_prep.ask_angles(fused.cos_table, fused.sin_table, fused.turned, row, g);
    } else {
      q_prep.ask(fused.q_weight, fused.weight_f32, fused.cos_table, fused.sin_table, pos_row, g);
    }
  };
  if constexpr (FUSED) {
    if (WAVES == 4) ask_q();
  } else {
    const uint16_t* qp = q + ((size_t)row * H + head) * HD + 8 * g;
#pragma unroll
    for (int s = 0; s < NS; ++s) q_vec[s] = as_bf16x8(load16(qp + 32 * s));
  }
  auto finish_q = [&]() {
    float x[NS][8];
    widen_head<NS>(x, q_raw);
    if constexpr (FUSED == 2)
      q_prep.apply(x, fused.unit_norm || fused.q_weight != nullptr, fused.q_weight != nullptr, fused.weight_f32, fused.eps, fused.cos_table != nullptr);
    else
      q_prep.apply(x, fused.q_weight != nullptr, fused.weight_f32, fused.eps, fused.cos_table != nullptr);
    u32x4_t packed[NS];
    pack_head<NS>(packed, x);
#pragma unroll
    for (int s = 0; s < NS; ++s) q_vec[s] = as_bf16x8(packed[s]);
  };
  if (FUSED && LEAN) finish_q();
  const int pos_max = wave_max_int(pos), pos_min = wave_min_int(pos);
  const int lo_min = wave_min_int(lo), lo_max = wave_max_int(lo);

  const int begin = lo_min / BH_PAGE + split * pages_per_split;
  const int last = pos_max >= 0 ? pos_max / BH_PAGE : -1;
  const int end = (begin + pages_per_split < last + 1) ? begin + pages_per_split : last + 1;

  f32x4_t o[2 * NS];
  float run_max = -INFINITY, run_sum = 0.f;  // run_sum: this lane's share of the column's sum
#pragma unroll
  for (int dt = 0; dt < 2 * NS; ++dt) o[dt] = f32x4_t{0.f, 0.f, 0.f, 0.f};

  // One page of keys and values in operand order against the 16 columns: lane (j, g) holds keys
  // 64 p + 8 g + 32 (t / 2) + 4 (t % 2) + r.  A column sees keys lo .. pos; the bounds over the
  // wave say whether anything has to be masked at all.
  auto attend = [&](const u32x4_t (&k_vec)[4][NS], u32x4_t (&v_vec)[2 * NS][2], int p) {
    const int key0 = p * BH_PAGE + 8 * g;
    const bool mask_needed = (p * BH_PAGE + BH_PAGE - 1 > pos_min) || (p * BH_PAGE < lo_max);
    f32x4_t st[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < NS; ++s)
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(k_vec[t][s]), q_vec[s], acc, 0, 0, 0);
      st[t] = acc;
    }
    if constexpr (FORMED) {
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float off = slope * (float)(key0 + 32 * (t / 2) + 4 * (t % 2) + r - pos_row);
          const float s = st[t][r] * col_scale;
          st[t][r] = (FORMED == 2 ? capped_score(s, form.cap, cap_rate) : s) + off;
        }
    }
    // Online softmax with few instructions: the maximum is taken over the raw scores, the scale
    // enters through one fused multiply-add per score, and the exponentials are bare v_exp_f32
    // (arguments <= 0; results below the normal range may flush to zero).
    if (mask_needed) {
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int key = key0 + 32 * (t / 2) + 4 * (t % 2) + r;
          if (key > pos || key < lo) st[t][r] = -INFINITY;
        }
    }
    float local_max = fmaxf(fmaxf(st[0][0], st[0][1]), fmaxf(st[0][2], st[0][3]));
#pragma unroll
    for (int t = 1; t < 4; ++t)
      local_max = fmaxf(local_max, fmaxf(fmaxf(st[t][0], st[t][1]), fmaxf(st[t][2], st[t][3])));
    local_max = fmaxf(local_max, __shfl_xor(local_max, 16, 64));
    local_max = fmaxf(local_max, __shfl_xor(local_max, 32, 64));
    const float new_max = fmaxf(run_max, local_max);              // raw (unscaled) scores
    const float shift = (new_max == -INFINITY) ? 0.f : -new_max * scale_log2;
    // exactly 1 while the maximum stands still, 0 when nothing was seen before
    const float alpha = (run_max == new_max) ? 1.0f : __builtin_amdgcn_exp2f((run_max - new_max) * scale_log2);
    float page_sum = 0.f;
    u32x4_t p_vec[2];
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int half = 0; half < 2; ++half) {
        const int t = 2 * u + half;
        const float e0 = __builtin_amdgcn_exp2f(fmaf(st[t][0], scale_log2, shift));
        const float e1 = __builtin_amdgcn_exp2f(fmaf(st[t][1], scale_log2, shift));
        const float e2 = __builtin_amdgcn_exp2f(fmaf(st[t][2], scale_log2, shift));
        const float e3 = __builtin_amdgcn_exp2f(fmaf(st[t][3], scale_log2, shift));
        page_sum += (e0 + e1) + (e2 + e3);
        p_vec[u][2 * half] = pack_bf16(e0, e1);
        p_vec[u][2 * half + 1] = pack_bf16(e2, e3);
      }
    run_sum = run_sum * alpha + page_sum;
    run_max = new_max;
    if (p * BH_PAGE + BH_PAGE - 1 > pos_max) {  // the page's tail was never written: zero it
      const int valid = pos_max + 1 - key0;
#pragma unroll
      for (int dt = 0; dt < 2 * NS; ++dt) {
        v_vec[dt][0] = keep_first(v_vec[dt][0], valid);
        v_vec[dt][1] = keep_first(v_vec[dt][1], valid - 32);
      }
    }
    if (__any(alpha != 1.0f)) {   // after the first pages the maximum seldom moves
#pragma unroll
      for (int dt = 0; dt < 2 * NS; ++dt) o[dt] = o[dt] * alpha;
    }
#pragma unroll
    for (int dt = 0; dt < 2 * NS; ++dt) {
      f32x4_t acc = o[dt];
      acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(v_vec[dt][0]), as_bf16x8(p_vec[0]), acc, 0, 0, 0);
      acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(v_vec[dt][1]), as_bf16x8(p_vec[1]), acc, 0, 0, 0);
      o[dt] = acc;
    }
  };

  // The new key and value of this (sequence, kv head): normed and rotated here, attended to, and written into the cache.  The key stands
  // in all 16 rows of the product's operand, so that every lane has its column's score; the value is added in plain arithmetic.
  auto take_new_key = [&]() {
    float x[NS][8];
    widen_head<NS>(x, k_raw);
    if (!LEAN) k_prep.take_angles(q_prep);
    if constexpr (FUSED == 2)
      k_prep.apply(x, fused.unit_norm || fused.k_weight != nullptr, fused.k_weight != nullptr, fused.weight_f32, fused.eps, fused.cos_table != nullptr);
    else
      k_prep.apply(x, fused.k_weight != nullptr, fused.weight_f32, fused.eps, fused.cos_table != nullptr);
    u32x4_t new_key[NS];
    pack_head<NS>(new_key, x);
    f32x4_t product = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < NS; ++s) product = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(new_key[s]), q_vec[s], product, 0, 0, 0);
    float score = product[0];
    if constexpr (FORMED) {
      score *= col_scale;
      if (FORMED == 2) score = capped_score(score, form.cap, cap_rate);
    }
    const float new_max = fmaxf(run_max, score);
    const float shift = (new_max == -INFINITY) ? 0.f : -new_max * scale_log2;
    const float alpha = (run_max == new_max) ? 1.0f : __builtin_amdgcn_exp2f((run_max - new_max) * scale_log2);
    const float p = __builtin_amdgcn_exp2f(fmaf(score, scale_log2, shift));
    run_sum = run_sum * alpha + (g == 0 ? p : 0.f);      // once for the column
    run_max = new_max;
#pragma unroll
    for (int dt = 0; dt < 2 * NS; ++dt)
#pragma unroll
      for (int r = 0; r < 4; ++r) o[dt][r] = fmaf(p, bf16_bits_to_f32((uint16_t)(value_raw[dt][r / 2] >> (16 * (r % 2)))), o[dt][r] * alpha);
    const int token = pos_row % BH_PAGE;
    const int token_t = 2 * (token / 32) + (token / 4) % 2, token_j = 4 * ((token / 8) % 4) + token % 4;
    const int page = table[pos_row / BH_PAGE];
    uint16_t* kb = fused.k_pages + ((size_t)page * KVH + kvh) * BH_PAGE * HD;
    uint16_t* vb = fused.v_pages + ((size_t)page * KVH + kvh) * HD * BH_PAGE;
    if (j == 0) {
#pragma unroll
      for (int s = 0; s < NS; ++s)
        *reinterpret_cast<u32x4_t*>(kb + ((token_t * NS + s) * 64 + 16 * g + token_j) * 8) = new_key[s];
    }
    if (g == 0) {
#pragma unroll
      for (int dt = 0; dt < 2 * NS; ++dt) vb[bh_value_index(BH_KV_PIECES, token, 16 * dt + j, HD)] = new_value[dt];
    }
  };

  // a page's number is asked for one page early
  int page_ahead = (begin + wave < end) ? (begin + wave == first_guess ? page_guess : table[begin + wave]) : 0;
  u32x4_t k_vec[4][NS], v_vec[2 * NS][2];
  auto ask_page = [&](int p) {
    const int page = page_ahead;
    if (p + 4 < end) page_ahead = table[p + 4];
    const uint16_t* kb = k_pages + ((size_t)page * KVH + kvh) * BH_PAGE * HD;
    const uint16_t* vb = v_pages + ((size_t)page * KVH + kvh) * HD * BH_PAGE;
    // the cache lies in pieces (BH_KV_PIECES): every load instruction covers 1 KB of contiguous memory
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int s = 0; s < NS; ++s) k_vec[t][s] = load16_cache<STREAM>(kb + ((t * NS + s) * 64 + lane) * 8);
#pragma unroll
    for (int dt = 0; dt < 2 * NS; ++dt) {
      v_vec[dt][0] = load16_cache<STREAM>(vb + ((dt * 2) * 64 + lane) * 8);
      v_vec[dt][1] = load16_cache<STREAM>(vb + ((dt * 2 + 1) * 64 + lane) * 8);
    }
  };
  // What the fifth wave hands over.  The barrier waits for LDS only: the first page stays on its way.  (One asm that may touch memory: the
  // builtins are said to touch none, so that nothing would hold the stores of sm_q above and its loads below on their sides of them.)
  auto meet = [&]() {
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  };
  if (WAVES == 5 && wave == 4) {
    ask_q();
    if (new_key_here) ask_new_key();
    finish_q();
#pragma unroll
    for (int s = 0; s < NS; ++s) sm_q[s][lane] = __builtin_bit_cast(u32x4_t, q_vec[s]);
    meet();
  } else {
    int p = begin + wave;
    if (WAVES == 5) {
      if (p < end) ask_page(p);
      meet();
#pragma unroll
      for (int s = 0; s < NS; ++s) q_vec[s] = as_bf16x8(sm_q[s][lane]);
    }
    for (bool asked = WAVES == 5; p < end; p += 4, asked = false) {
      if (!asked) ask_page(p);
      attend(k_vec, v_vec, p);
    }
  }

  if (takes_new_key) {
    if (WAVES == 4) ask_new_key();
    take_new_key();
  }

  // merge the waves: lane (j, g) holds O^T[16dt + 4g + r, j]
  {
    float lane_sum = run_sum;
    lane_sum += __shfl_xor(lane_sum, 16, 64);
    lane_sum += __shfl_xor(lane_sum, 32, 64);
    if (g == 0) {
      sm_m[wave][j] = run_max * scale_log2;   // in units of the base-2 exponent, as the merges use it
      sm_l[wave][j] = lane_sum;
    }
#pragma unroll
    for (int dt = 0; dt < 2 * NS; ++dt) *reinterpret_cast<f32x4_t*>(&sm_o[wave][j][16 * dt + 4 * g]) = o[dt];
    __syncthreads();
    if (WAVES == 5 && wave == 4) return;
    // 16 threads a column, each with neighbouring dimensions of it; or, of finished results of at most four columns, 64, each with a pair
    // (few query heads a kv head left most threads idle: 16 sequences of 200 keys, 8 heads on 4 9.6 us, 9.3 so)
    constexpr int EACH = HD / 16;
    const bool few = n_splits == 1 && n_cols - tile * 16 <= 4;
    const int col = few ? threadIdx.x / 64 : threadIdx.x / 16, place = few ? threadIdx.x % 64 : threadIdx.x % 16, cc = tile * 16 + col;
    if (cc >= n_cols) return;
    float top = fmaxf(fmaxf(sm_m[0][col], sm_m[1][col]), fmaxf(sm_m[2][col], sm_m[3][col]));
    if (WAVES == 5) top = fmaxf(top, sm_m[WAVES - 1][col]);
    const float safe_top = (top == -INFINITY) ? 0.f : top;
    const int out_row = row0 + cc / G, out_head = kvh * G + cc % G;
    const size_t column = (size_t)out_row * H + out_head;
    float gate = 1.f;
    auto finish_sum = [&](float sum) {      // a sink: one more term exp(sinks[head]) in the softmax's sum (`top` is in powers of two)
      gate = head_gate<bf16_t>(finish, out_row, out_head);
      return finish.sinks ? sum + exp2f(finish.sinks[out_head] * 1.4426950408889634f - safe_top) : sum;
    };
    // out_block_rows: the output [rows][H * HD] lies in blocks of that many rows (bh_rows_index); two neighbours from an even dimension on
    // are neighbours there too.  Their word need not stand on four bytes.
    auto write = [&](int d, float first, float second, float sum) {
      uint16_t* to = out + bh_rows_index(out_block_rows, out_row, out_head * HD + d, H * HD);
      const uint32_t word = (uint32_t)f32_to_bf16_bits(first * gate / sum) | ((uint32_t)f32_to_bf16_bits(second * gate / sum) << 16);
      __builtin_memcpy(to, &word, sizeof word);
    };
    if (!few) {
      const int d0 = place * EACH;
      float sum = 0.f, value[EACH];
#pragma unroll
      for (int d = 0; d < EACH; ++d) value[d] = 0.f;
#pragma unroll
      for (int v = 0; v < WAVES; ++v) {
        if (v == 4 && !new_key_here) break;
        const float f = exp2f(sm_m[v][col] - safe_top);
        sum += sm_l[v][col] * f;
#pragma unroll
        for (int d = 0; d < EACH; d += 2) {
          const float2 pair = *reinterpret_cast<const float2*>(&sm_o[v][col][d0 + d]);
          value[d] += pair.x * f;
          value[d + 1] += pair.y * f;
        }
      }
      if (n_splits == 1) {
        sum = finish_sum(sum);
#pragma unroll
        for (int d = 0; d < EACH; d += 2) write(d0 + d, value[d], value[d + 1], sum);
      } else {
        float* to = part_o + (column * n_splits + split) * HD + d0;
#pragma unroll
        for (int d = 0; d < EACH; d += 2) *reinterpret_cast<float2*>(to + d) = make_float2(value[d], value[d + 1]);
        if (d0 == 0) {
          part_ml[(column * n_splits + split) * 2] = top;
          part_ml[(column * n_splits + split) * 2 + 1] = sum;
        }
      }
    } else {
      float sum = 0.f, weight[WAVES];
#pragma unroll
      for (int v = 0; v < WAVES; ++v) {
        weight[v] = v == 4 && !new_key_here ? 0.f : exp2f(sm_m[v][col] - safe_top);
        sum += sm_l[v][col] * weight[v];
      }
      sum = finish_sum(sum);
#pragma unroll
      for (int d = 2 * place; d < HD; d += 128) {
        float2 value = make_float2(0.f, 0.f);
#pragma unroll
        for (int v = 0; v < WAVES; ++v) {
          if (v == 4 && !new_key_here) break;
          const float2 pair = *reinterpret_cast<const float2*>(&sm_o[v][col][d]);
          value.x += pair.x * weight[v];
          value.y += pair.y * weight[v];
        }
        write(d, value.x, value.y, sum);
      }
    }
  }
}

// One block per column, a group of 64 or 128 threads (a dimension each; heads of more take the others in turn) for every eight splits.
// Nothing here may wait for one split's numbers before asking for the next one's, nor for the maxima before asking for the outputs: a
// thread asks for all eight at once and makes their weights itself, from numbers that are the same for its wave.  The groups are merged
// through LDS.  The sums run over the splits in their order.  (One group for all, by eights, and the maxima and sums over the lanes of a
// wave, took 4.8 us in traces of decode steps of one sequence with eight splits and of eight sequences with four; 3.8 to 4.7 now, and 4.7
// to 4.8.)
#define COMBINE_SPLITS 8      // a group's; four where there are no more in all
template <int SPLITS>
__global__ __launch_bounds__(1024) void attention_combine_kernel(const float* __restrict__ part_o, const float* __restrict__ part_ml,
                                                                 uint16_t* __restrict__ out, int n_splits, int HD, int H, int out_block_rows,
                                                                 HeadEnd finish, int dims) {
  __shared__ float sm_value[COMBINE_SPLITS][256], sm_top[COMBINE_SPLITS], sm_sum[COMBINE_SPLITS];
  const int row = blockIdx.x / H, head = blockIdx.x % H, groups = (n_splits + SPLITS - 1) / SPLITS;
  const int group = __builtin_amdgcn_readfirstlane(threadIdx.x / dims), dim = threadIdx.x % dims, first = group * SPLITS;
  const size_t column = blockIdx.x;
  const float* ml = part_ml + column * n_splits * 2;
  const float* outputs = part_o + column * n_splits * HD;
  float part[SPLITS], weight[SPLITS], share[SPLITS];
#pragma unroll
  for (int u = 0; u < SPLITS; ++u) {
    const int s = min(first + u, n_splits - 1);
    part[u] = dim < HD ? outputs[s * HD + dim] : 0.f;
    weight[u] = ml[2 * s];
    share[u] = ml[2 * s + 1];
  }
  const float gate = head_gate<bf16_t>(finish, row, head);
  float top = weight[0];
#pragma unroll
  for (int u = 1; u < SPLITS; ++u) top = fmaxf(top, weight[u]);
  const float safe_top = top == -INFINITY ? 0.f : top;
  float sum = 0.f;
#pragma unroll
  for (int u = 0; u < SPLITS; ++u) {
    // (arguments <= 0; results below the normal range may be 0)
    weight[u] = first + u < n_splits ? __builtin_amdgcn_exp2f(weight[u] - safe_top) : 0.f;
    sum += share[u] * weight[u];
  }
  auto value_at = [&](int d) {
    float value = 0.f;
#pragma unroll
    for (int u = 0; u < SPLITS; ++u) value += (d == dim ? part[u] : outputs[min(first + u, n_splits - 1) * HD + d]) * weight[u];
    return value;
  };
  auto write = [&](int d, float value, float total, float highest) {
    // a sink: one more term exp(sinks[head]) in the softmax's sum
    if (finish.sinks) total += exp2f(finish.sinks[head] * 1.4426950408889634f - highest);
    out[bh_rows_index(out_block_rows, row, head * HD + d, H * HD)] = f32_to_bf16_bits(value * (gate / total));
  };
  if (groups == 1) {
    for (int d = dim; d < HD; d += dims) write(d, value_at(d), sum, safe_top);
    return;
  }
  for (int d = dim; d < HD; d += dims) sm_value[group][d] = value_at(d);
  if (dim == 0) sm_top[group] = top, sm_sum[group] = sum;
  __syncthreads();
  if (group != 0) return;
  for (int k = 1; k < groups; ++k) top = fmaxf(top, sm_top[k]);
  const float highest = top == -INFINITY ? 0.f : top;
  float total = 0.f;
  for (int k = 0; k < groups; ++k) total += sm_sum[k] * __builtin_amdgcn_exp2f(sm_top[k] - highest);
  for (int d = dim; d < HD; d += dims) {
    float value = 0.f;
    for (int k = 0; k < groups; ++k) value += sm_value[k][d] * __builtin_amdgcn_exp2f(sm_top[k] - highest);
    write(d, value, total, highest);
  }
}

// The order of a cache page's elements that the kernels of this library expect for a cache of the
// given element type and head size: the writer, the attention for any size and this file's agree on it.
extern "C" int bh_kv_order(int dtype, int hd) {
  return (dtype == BH_BF16 && hd % 32 == 0 && hd >= 32 && hd <= 256) ? BH_KV_PIECES : BH_KV_ROWS;
}

// How many ways the keys are split for a given launch; the caller sizes the scratch from it.
extern "C" int bh_attention_bf16_splits(int n_seqs, int max_rows_per_seq, int H, int KVH, int max_position) {
  if (n_seqs <= 0 || max_rows_per_seq <= 0 || H <= 0 || KVH <= 0 || H % KVH) return 1;
  const int G = H / KVH;
  const long tiles = (long)((max_rows_per_seq * G + 15) / 16) * KVH * n_seqs;
  const int pages = max_position / BH_PAGE + 1;
  // Every wave of a workgroup at least one page.  The workgroups run in rounds of one per compute unit (256 on an
  // MI355X), so what a launch costs is its rounds times a workgroup's pages (and about four pages' worth of start and
  // merge): the split count with the least of that, the smaller one among equals.  One workgroup per compute unit or
  // just beyond, as it was before, made 288 to 384 workgroups of 9 to 14 and of 17 to 24 sequences: two rounds of
  // nearly whole-sized workgroups (decode steps of the Qwen3-8B shape at context 8,192, 8 layers: 6 sequences 1.18 ->
  // 1.11 ms, 10 1.48 -> 1.40, 12 1.63 -> 1.48, 20 2.18 -> 2.02, 24 2.23 -> 2.19; 8, 16 and 32 sequences as before).
  const int units = bh_compute_units();
  if (pages < 8) return 1;
  long want = 1, least = -1;
  if (tiles > units) {
    // More workgroups than compute units: two of the lean kernel's share a compute unit.  Just above one per compute
    // unit (and just above two) the few compute units that carry one more hold the launch up, and three (two) splits
    // spread the pages evenly; from about 1.4 per compute unit on the whole workgroups are as fast or faster
    // (Qwen3-8B shape, context 8,192, 8 layers, ms per step with 1 / 2 / 3 / 4 / 6 splits: 33 sequences 3.04 / 2.80 / 2.72 /
    // 2.69 / 2.66, 40: 3.20 / 2.92 / 2.89 / 2.90 / 2.91, 48: 3.27 / 3.35 / 3.25 / 3.25 / 3.25, 56: 3.66 / 3.75 / 3.75 / 3.69 /
    // 3.73, 72: 4.55 / 4.43 / 4.43 / 4.52 / 4.54).
    const double each_unit = (double)tiles / units;
    want = each_unit < 1.4 ? 3 : (each_unit > 2.0 && each_unit < 2.4) ? 2 : 1;
    if (want > pages / 4) want = pages / 4;
  } else {
    for (long splits = 1; splits <= pages / 4 && splits <= 64; ++splits) {
      const long rounds = (tiles * splits + units - 1) / units, each = (pages + splits - 1) / splits;
      const long cost = rounds * (each + 4);
      if (least < 0 || cost < least) least = cost, want = splits;
    }
  }
  const int per = (int)((pages + want - 1) / want);
  return (pages + per - 1) / per;
}

// Whether the prefill kernel runs a step: from 1,024 tiles of columns (over kv heads and sequences) on, and, where no cache is longer
// than the seven pages up to which keys are never split, prompts of few pages and those whose tiles fill the
// chip: its four waves share a page that goes through LDS once, where a workgroup of this file's kernel has four waves on as many pages
// for 16 columns and a merge behind them.  us here / there: three prompts of 253 rows in all, 40 heads of 128 on 8 16.8 / 6.7, 128 rows of
// 32 on 8 8.2 / 6.4, 16 rows of 32 on 8 7.6 / 5.4; of seven pages 96 tiles 8.3 / 8.9, 160 11.3 / 10.6, 512 24.9 / 11.3.  (A step of up to
// eight rows has its output read in blocks of eight, which the prefill kernel does not write.)
#define PREFILL_FROM_TILES 1024
static bool prefill_wins(int n_seqs, int max_rows_per_seq, int H, int KVH, int max_position) {
  const long columns = (long)max_rows_per_seq * (H / KVH), tiles = (columns + 15) / 16 * KVH * n_seqs;
  const int pages = max_position / BH_PAGE + 1;
  if (tiles >= PREFILL_FROM_TILES) return true;
  return max_rows_per_seq > 8 && columns >= 16 && pages < 8 && (pages <= 4 || tiles >= bh_compute_units());
}
// Whether a step of these sizes goes to the kernel for many columns per sequence, which writes its output in rows
// or in blocks of 16 rows x 32 columns (bh_blocked_index); the other steps' kernels write blocks of 8 or 16 rows.
extern "C" int bh_attention_bf16_writes_blocked(int n_seqs, int max_rows_per_seq, int H, int KVH, int max_position) {
  if (n_seqs <= 0 || max_rows_per_seq <= 0 || H <= 0 || KVH <= 0 || H % KVH) return 0;
  return bh_attention_bf16_splits(n_seqs, max_rows_per_seq, H, KVH, max_position) == 1 && prefill_wins(n_seqs, max_rows_per_seq, H, KVH, max_position) ? 1 : 0;
}

static int attention_bf16_run(const void* q, void* out, void* part_o, void* part_ml, const void* k_pages,
                              const void* v_pages, const int32_t* page_table, int table_stride,
                              const int32_t* positions, const int32_t* seq_start, int n_seqs, int n_rows,
                              int max_rows_per_seq, int H, int KVH, int hd, const ScoreForm& form, int window,
                              int max_position, int n_splits, const FusedQkv& fused, bool pairs, int out_blocked,
                              const HeadEnd& finish, hipStream_t stream) {
  if (const char* fault = bh_score_form_fault(form)) return bh_fail("attention_bf16: %s", fault);
  BH_REQUIRE(n_seqs > 0 && n_rows > 0 && max_rows_per_seq > 0, "attention_bf16: empty batch");
  BH_REQUIRE(H > 0 && KVH > 0 && H % KVH == 0, "attention_bf16: %d query heads do not group evenly into %d kv heads", H, KVH);
  BH_REQUIRE(hd % 32 == 0 && hd >= 32 && hd <= 256, "attention_bf16: head size %d is not a multiple of 32 up to 256", hd);
  BH_REQUIRE(max_position >= 0, "attention_bf16: positions must not be negative");
  BH_REQUIRE(n_splits >= 1 && (n_splits == 1 || (part_o && part_ml)), "attention_bf16: split keys need scratch memory");
  BH_REQUIRE(n_splits <= COMBINE_SPLITS * COMBINE_SPLITS, "attention_bf16: keys in %d splits, at most %d are combined", n_splits, COMBINE_SPLITS * COMBINE_SPLITS);
  const int G = H / KVH;
  const int tiles = (max_rows_per_seq * G + 15) / 16;
  const int pages = max_position / BH_PAGE + 1;
  const int per = (pages + n_splits - 1) / n_splits;
  const int formed = bh_formed(form);
  BH_REQUIRE((long)tiles * KVH * n_seqs * n_splits < (1L << 31), "attention_bf16: too many workgroups");
  const bool is_fused = fused.qkv != nullptr;
  BH_REQUIRE(!is_fused || (tiles == 1 && max_rows_per_seq == 1 && n_rows == n_seqs),
             "attention_bf16: the fused projection rows are taken in decode steps of at most 16 heads per kv head only");
  if (!is_fused && n_splits == 1 && (uintptr_t)out % 8 == 0 && prefill_wins(n_seqs, max_rows_per_seq, H, KVH, max_position)) {   // it writes 8 bytes at a time
    // Where this file's kernel would else run, which takes a page's probabilities against its own maximum, the largest are ones there too
    // (no slack): they are exact in bfloat16.  Its error against 64 bits is 0.95 to 1.01 of that kernel's, on average 0.99 (9 to 448
    // rows, scores spread by 0.3 to 10; with a slack of 8 up to 1.07; with the sum over unrounded probabilities up to 1.12), and
    // the time the same (448 rows, 32 heads of 128 on 8 11.5 / 11.6 us).
    const bool many_tiles = (long)tiles * KVH * n_seqs >= PREFILL_FROM_TILES;
    BH_REQUIRE(out_blocked == 0 || out_blocked == 16, "attention_bf16: a step of many columns writes rows or blocks of 16 rows, not of %d", out_blocked);
    bh_attention_prefill_launch(q, out, k_pages, v_pages, page_table, table_stride, positions, seq_start, n_seqs,
                                tiles, H, KVH, hd, form, window, out_blocked == 16, many_tiles ? 8.0f : 0.0f, finish, stream);
    return bh_check_launch("attention_prefill_bf16");
  }
  BH_REQUIRE(out_blocked == 0 || ((out_blocked == 8 || out_blocked == 16) && (H * hd) % 32 == 0),
             "attention_bf16: the output's rows lie in blocks of 8 or 16, or one after the other (0), not %d", out_blocked);
  const int tile_groups = tiles, z_count = n_seqs * n_splits;
  // More workgroups than compute units: two of them per unit.  And long runs of pages, whose workgroups the fifth wave does not make faster
  // (32 sequences of 5,000 keys, 79 pages a workgroup, 32 heads on 8 106.4 us before there was one, 108.9 with it, 106.7 lean, 8 heads on
  // 8 101.6 / 106.4 / 102.8; at 31 and 40 pages within 2 % either way, at 16 and fewer up to 9 % for it where one page is all).
  const bool lean = (long)tiles * KVH * z_count > bh_compute_units() || per > 24;
  dim3 grid(tile_groups * KVH * z_count);
#define BH_ATT_ONE(NS, STREAM, FUSED, ...)                                                                      \
  attention_mfma_kernel<NS, STREAM, FUSED, __VA_ARGS__><<<grid, is_fused && !lean && NS <= 4 ? 320 : 256, 0, stream>>>(        \
      (const uint16_t*)q, (uint16_t*)out, (float*)part_o, (float*)part_ml, (const uint16_t*)k_pages,            \
      (const uint16_t*)v_pages, page_table, table_stride, positions, seq_start, H, KVH, window,                 \
      n_splits, per, tile_groups, fused, out_blocked, finish, form)
#define BH_ATT_FORM(NS, STREAM, FUSED, LEAN)                                  \
  do {                                                                        \
    if (formed == 2) BH_ATT_ONE(NS, STREAM, FUSED, LEAN, 2);                  \
    else if (formed) BH_ATT_ONE(NS, STREAM, FUSED, LEAN, 1);                  \
    else BH_ATT_ONE(NS, STREAM, FUSED, LEAN, 0);                              \
  } while (0)
#define BH_ATT(NS)                                                                          \
  do {                                                                                      \
    if (pairs && lean) BH_ATT_FORM(NS, true, 2, true);                                      \
    else if (pairs) BH_ATT_FORM(NS, true, 2, (NS > 4));                                     \
    else if (is_fused && lean) BH_ATT_ONE(NS, true, 1, true, 0);                            \
    else if (is_fused) BH_ATT_ONE(NS, true, 1, (NS > 4), 0);                                \
    else if (tile_groups == 1) BH_ATT_FORM(NS, true, 0, false);                             \
    else BH_ATT_FORM(NS, false, 0, false);                                                  \
  } while (0)
  switch (hd / 32) {
    case 1: BH_ATT(1); break;
    case 2: BH_ATT(2); break;
    case 3: BH_ATT(3); break;
    case 4: BH_ATT(4); break;
    case 5: BH_ATT(5); break;
    case 6: BH_ATT(6); break;
    case 7: BH_ATT(7); break;
    default: BH_ATT(8); break;
  }
#undef BH_ATT
#undef BH_ATT_FORM
#undef BH_ATT_ONE
  if (int status = bh_check_launch("attention_mfma")) return status;
  if (n_splits > 1) {
    const int dims = hd >= 128 ? 128 : 64, groups = (n_splits + COMBINE_SPLITS - 1) / COMBINE_SPLITS;
#define BH_COMBINE(SPLITS)                                                                                                                  \
  attention_combine_kernel<SPLITS><<<n_rows * H, dims * groups, 0, stream>>>((const float*)part_o, (const float*)part_ml, (uint16_t*)out, \
                                                                             n_splits, hd, H, out_blocked, finish, dims)
    if (n_splits <= 4) BH_COMBINE(4);
    else BH_COMBINE(COMBINE_SPLITS);
#undef BH_COMBINE
    return bh_check_launch("attention_combine");
  }
  return 0;
}

extern "C" int bh_attention_bf16(const void* q, void* out, void* part_o, void* part_ml, const void* k_pages,
                                 const void* v_pages, const int32_t* page_table, int table_stride,
                                 const int32_t* positions, const int32_t* seq_start, int n_seqs, int n_rows,
                                 int max_rows_per_seq, int H, int KVH, int hd, float scale, int window,
                                 int max_position, int n_splits, int out_blocked, const float* sinks, const void* gates,
                                 int gate_stride, float cap, const float* slopes, float temp_coef, int temp_every,
                                 float out_scale, hipStream_t stream) {
  BH_REQUIRE(gates == nullptr || gate_stride >= H, "attention_bf16: a gate a head (%d) lies outside a row of %d", H, gate_stride);
  const FusedQkv none = {};
  return attention_bf16_run(q, out, part_o, part_ml, k_pages, v_pages, page_table, table_stride, positions,
                            seq_start, n_seqs, n_rows, max_rows_per_seq, H, KVH, hd, ScoreForm{scale, cap, slopes, temp_coef, temp_every},
                            window, max_position, n_splits, none, false, out_blocked, HeadEnd{sinks, gates, gate_stride, out_scale}, stream);
}

// A decode step (one row per sequence) straight from the fused projection rows [q heads | k heads | v heads]:
// per-head RMSNorm of q and k (weights may be null), rotation over the whole head at the row's position
// (tables may be null), the new key and value into the cache (unless write_kv is 0: the entry is another
// layer's), and attention over the cache and the new key.  See struct FusedQkv.  Row s is sequence s's: `seq_start`
// can only say so (0, 1, ..., n_seqs) and is not read.
extern "C" int bh_attention_decode_fused(const void* qkv, void* out, void* part_o, void* part_ml, void* k_pages,
                                         void* v_pages, const int32_t* page_table, int table_stride,
                                         const int32_t* positions, const int32_t* seq_start, int n_seqs, int H,
                                         int KVH, int hd, float scale, int window, int max_position, int n_splits,
                                         const void* q_weight, const void* k_weight, int w_dtype, float eps,
                                         const float* cos_table, const float* sin_table, int table_positions,
                                         int rot, int write_kv, int out_block_rows, hipStream_t stream) {
  BH_REQUIRE(qkv != nullptr, "attention_decode_fused: the projection rows are required");
  BH_REQUIRE((q_weight == nullptr) == (k_weight == nullptr), "attention_decode_fused: give both norm weights or neither");
  BH_REQUIRE(q_weight == nullptr || w_dtype == BH_F32 || w_dtype == BH_BF16, "attention_decode_fused: unknown weight dtype %d", w_dtype);
  BH_REQUIRE((cos_table == nullptr) == (sin_table == nullptr), "attention_decode_fused: cos and sin tables come together");
  BH_REQUIRE(cos_table == nullptr || (rot == hd && hd % 64 == 0),
             "attention_decode_fused: the rotation must span the whole head (%d of %d) and the head be a multiple of 64", rot, hd);
  BH_REQUIRE(cos_table == nullptr || max_position < table_positions,
             "attention_decode_fused: position %d is outside the rotation table of %d positions", max_position, table_positions);
  const FusedQkv fused = {(const uint16_t*)qkv, (H + 2 * KVH) * hd, H * hd, (H + KVH) * hd, hd, 0, q_weight, k_weight,
                          w_dtype == BH_F32, eps, cos_table, sin_table, write_kv, (uint16_t*)k_pages, (uint16_t*)v_pages};
  return attention_bf16_run(nullptr, out, part_o, part_ml, k_pages, v_pages, page_table, table_stride, positions,
                            seq_start, n_seqs, n_seqs, 1, H, KVH, hd, ScoreForm{scale, 0.f, nullptr, 0.f, 0}, window, max_position, n_splits,
                            fused, false, out_block_rows, HeadEnd{}, stream);
}

// The same for rows whose heads turn in neighbouring pairs: from column `first` of rows of row_stride elements H heads of q, then
// KVH of k and (unless values_are_keys) KVH of v; norm weights float32 [hd], both or neither, or (unit_norm) a norm without;
// cos_rows and sin_rows [n_seqs][turned / 2] for the rows' positions; sinks, gates and out_scale as in struct HeadEnd, cap to temp_every
// as in struct ScoreForm.
extern "C" int bh_attention_decode_pairs(const void* rows, int row_stride, int first, void* out, void* part_o, void* part_ml,
                                         void* k_pages, void* v_pages, const int32_t* page_table, int table_stride,
                                         const int32_t* positions, const int32_t* seq_start, int n_seqs, int H, int KVH, int hd,
                                         float scale, int window, int max_position, int n_splits, const float* q_weight,
                                         const float* k_weight, int unit_norm, float eps, const float* cos_rows,
                                         const float* sin_rows, int turned, int values_are_keys, int write_kv, int out_block_rows,
                                         const float* sinks, const void* gates, int gate_stride, float cap, const float* slopes,
                                         float temp_coef, int temp_every, float out_scale, hipStream_t stream) {
  BH_REQUIRE(rows != nullptr && H > 0 && KVH > 0 && hd > 0, "attention_decode_pairs: the projection rows are required");
  const int k_first = H * hd, v_first = values_are_keys ? k_first : (H + KVH) * hd;
  // (without write_kv the new key and value are not read: a row may hold queries alone)
  BH_REQUIRE(first >= 0 && first % 8 == 0 && row_stride % 8 == 0 && ((uintptr_t)rows) % 16 == 0 &&
                 first + (write_kv ? v_first + KVH * hd : k_first) <= row_stride,
             "attention_decode_pairs: q, k and v from column %d lie outside a row of %d, or not on 16 bytes", first, row_stride);
  BH_REQUIRE((q_weight == nullptr) == (k_weight == nullptr) && !(unit_norm && q_weight), "attention_decode_pairs: both norm weights, or neither");
  BH_REQUIRE((cos_rows == nullptr) == (sin_rows == nullptr) && (cos_rows == nullptr || (turned > 0 && turned % 2 == 0 && turned <= hd)),
             "attention_decode_pairs: %d turned dimensions of %d and their cosines and sines", turned, hd);
  BH_REQUIRE(gates == nullptr || gate_stride >= H, "attention_decode_pairs: a gate a head (%d) lies outside a row of %d", H, gate_stride);
  const FusedQkv fused = {(const uint16_t*)rows + first, row_stride, k_first, v_first, turned, unit_norm, q_weight, k_weight,
                          1, eps, cos_rows, sin_rows, write_kv, (uint16_t*)k_pages, (uint16_t*)v_pages};
  return attention_bf16_run(nullptr, out, part_o, part_ml, k_pages, v_pages, page_table, table_stride, positions, seq_start,
                            n_seqs, n_seqs, 1, H, KVH, hd, ScoreForm{scale, cap, slopes, temp_coef, temp_every}, window, max_position, n_splits,
                            fused, true, out_block_rows, HeadEnd{sinks, gates, gate_stride, out_scale}, stream);
}

// cos_rows, sin_rows [n_rows][pairs]: cosine and sine (times `magnitude`) of the float32 angle position * freq[pair], once a step for
// all the layers that turn by these frequencies.
__global__ __launch_bounds__(256) void row_angles_kernel(const int32_t* __restrict__ positions, const float* __restrict__ freq,
                                                         float magnitude, float* __restrict__ cos_rows, float* __restrict__ sin_rows,
                                                         int n_rows, int pairs) {
  const size_t n = (size_t)n_rows * pairs;
  for (size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x; e < n; e += (size_t)gridDim.x * blockDim.x) {
    const float angle = (float)positions[e / pairs] * freq[e % pairs];
    cos_rows[e] = cosf(angle) * magnitude;
    sin_rows[e] = sinf(angle) * magnitude;
  }
}

extern "C" int bh_row_angles(const int32_t* positions, const float* freq, float magnitude, float* cos_rows, float* sin_rows, int n_rows,
                             int pairs, hipStream_t stream) {
  BH_REQUIRE(n_rows > 0 && pairs > 0, "row_angles: sizes must be positive");
  const size_t blocks = ((size_t)n_rows * pairs + 255) / 256;
  row_angles_kernel<<<(int)(blocks < 4096 ? blocks : 4096), 256, 0, stream>>>(positions, freq, magnitude, cos_rows, sin_rows, n_rows, pairs);
  return bh_check_launch("row_angles");
}
