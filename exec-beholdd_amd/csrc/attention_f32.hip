// Attention over the paged cache for float32 engines, head sizes of 32 to 256 in steps of 32.  Plain 32-bit multiply-adds; the
// same scores, masks, sinks and gates as attention_generic (generic.hip), which takes every other size.
//
// A workgroup takes one query head of one row, or of NR neighbouring rows where they belong to one sequence (prompts), and its
// waves (one, where the pages are few) take the visible pages in turn.  Keys lie [token][dim]: eight lanes share a key, 16 bytes each, so that a wave's load
// covers eight keys' whole 128-byte lines; their shares are added crosswise, which leaves lane l with the score of one key of the
// page.  Values lie [dim][token]: 16 lanes share a dimension, so that a load is 1 KB of contiguous memory, and every lane keeps
// its own sums over its four tokens of each page; they are added over the lanes once, behind the last page.  The waves' softmax
// sums are merged through LDS.
// Bound by the pages' way from memory or the L2 (a page of a head of 128 is 64 KB): NR rows share it.
// Measured (8 heads of 128 on 4): a decode step of 4 rows at 40 to 300 keys with its norms, rotation and cache write 7.0 us in a chain of
// such launches, 8.5 in two of them and 10.4 before eight waves took half pages (PARTS); the attention alone 54 with a thread a key
// (generic.hip: every lane its own line), 20 before a page's keys and values were asked for together; four prompts of 695 rows in all, up to 256 each,
// 41 us in waves of their own (30 in tiles of columns, see there), 94 in workgroups of four waves on four rows, 120 there.
#include "common.h"
#include <algorithm>
#include <cmath>

typedef float floatx4 __attribute__((ext_vector_type(4)));

namespace {

// A decode step's fused projection rows [q heads | k heads | v heads] in the place of finished queries and of a cache that holds the
// new keys already: see attend_rows.
struct F32Fused {
  const float* qkv;
  const float *q_weight, *k_weight;     // per-head RMSNorm weights [head size], or null for no norm
  float eps;
  const float *cos_table, *sin_table;   // [positions][head size / 2]: rotation over the whole head in split halves, or null for none
  int write_kv;                         // 0: the cache entry belongs to another layer, which has written the new key already
  float *k_pages, *v_pages;             // the cache again, to write into
};

struct F32Attention {
  const float* q;
  float* out;
  const float *k_pages, *v_pages;
  const int32_t* page_table;
  int table_stride;
  const int32_t *row_seq, *positions;
  int H, KVH;
  ScoreForm form;
  int window;
  HeadEnd finish;
  F32Fused fused;
};

__device__ inline floatx4 load4(const float* p) { return *reinterpret_cast<const floatx4*>(p); }

// LDS of a workgroup: a page's probabilities a wave and row, and the waves' results
template <int P, int NR, int WAVES>
struct Lds {
  float probs[WAVES][NR][BH_PAGE];
  float most[WAVES][NR], sum[WAVES][NR];
  float o[WAVES][NR][32 * P];
  float new_score;      // of a decode step's new key
};

// A head as a wave's lanes hold it (elements 32 p + 4 dq + e; the eight lanes of other keys hold the same): RMSNorm, then split-half
// rotation.  The partner of element i < HD / 2 is i + HD / 2, in the same lane, P / 2 slices on.
template <int P>
struct HeadTurn {
  floatx4 weight[P], cos_v[P > 1 ? P / 2 : 1], sin_v[P > 1 ? P / 2 : 1];

  __device__ void ask_weight(const float* of, int dq) {
    if (of)
#pragma unroll
      for (int p = 0; p < P; ++p) weight[p] = load4(of + 32 * p + 4 * dq);
  }
  __device__ void ask_angles(const F32Fused& f, int pos, int dq) {
    if (f.cos_table)
#pragma unroll
      for (int p = 0; p < P / 2; ++p) {
        cos_v[p] = load4(f.cos_table + (size_t)pos * (16 * P) + 32 * p + 4 * dq);
        sin_v[p] = load4(f.sin_table + (size_t)pos * (16 * P) + 32 * p + 4 * dq);
      }
  }
  __device__ void apply(floatx4 (&x)[P], const F32Fused& f, const HeadTurn& angles) const {
    if (f.q_weight) {
      float ss = 0.f;
#pragma unroll
      for (int p = 0; p < P; ++p)
#pragma unroll
        for (int e = 0; e < 4; ++e) ss += x[p][e] * x[p][e];
#pragma unroll
      for (int off = 4; off > 0; off >>= 1) ss += __shfl_xor(ss, off, BH_WAVE);
      const float inv = 1.0f / sqrtf(ss / (float)(32 * P) + f.eps);
#pragma unroll
      for (int p = 0; p < P; ++p)
#pragma unroll
        for (int e = 0; e < 4; ++e) x[p][e] = x[p][e] * inv * weight[p][e];
    }
    if (f.cos_table) {
#pragma unroll
      for (int p = 0; p < P / 2; ++p)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float lo = x[p][e], hi = x[p + P / 2][e], c = angles.cos_v[p][e], s = angles.sin_v[p][e];
          x[p][e] = lo * c - hi * s;
          x[p + P / 2][e] = lo * s + hi * c;
        }
    }
  }
};

// Rows row0 .. row0 + NR - 1, all of the sequence of row0.
// FUSED: a decode step (row s is sequence s's) from its projection rows, in place of the norm, rotation and cache write in a launch of
// their own: every wave norms and rotates its query while its first page is on its way, whose number it asks for beside the position;
// the last wave, which has the fewest pages, makes the new key and its score first.  In the merge that score and the new value are one
// wave more.  The first head of a group writes both into the cache, whose keys are read to one position earlier.
// PARTS: a wave takes a page's tokens in so many parts, a part at a time: of two parts a head of 96 or 128 fits the registers of eight waves
// with all of a part's loads ahead, of whole pages those of four (decode steps with norms, rotation and cache write, us, whole pages and four
// waves / half pages and eight: one row of 300 keys 9.1 / 7.0, 8 rows of 400 keys and 16 heads 10.0 / 7.9, 4 rows of 800 14.5 / 11.4).
template <int P, int NR, int WAVES, bool FUSED = false, int PARTS = 1>
__device__ void attend_rows(const F32Attention& t, Lds<P, NR, WAVES>& lds, int row0, int head) {
  static_assert(!FUSED || NR == 1, "a decode step's rows are each of their own sequence");
  static_assert(PARTS == 1 || PARTS == 2, "the sums over lanes are written for these");
  constexpr int TOKENS = BH_PAGE / PARTS, GROUPS = TOKENS / 8;      // of a part, and its keys by eights
  constexpr int TQ = TOKENS / 4, DL = 64 / TQ, ND = 32 * P / DL;    // lanes that share a dimension's values, dimensions a load, loads
  constexpr int HD = 32 * P;
  constexpr bool AHEAD = NR == 1 && P <= 4;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int kl = lane >> 3, dq = lane & 7;    // keys: the lane's key among eight, its 16 bytes of each 32 dimensions
  const int dl = lane / TQ, tq = lane % TQ;   // values: the lane's dimension of a load's, its four tokens
  const int kv_head = head / (t.H / t.KVH);
  const int32_t* table = t.page_table + (size_t)(FUSED ? row0 : t.row_seq[row0]) * t.table_stride;
  const float slope = t.form.slopes ? t.form.slopes[head] : 0.f;

  const int page_guess = FUSED && wave / PARTS < t.table_stride ? table[wave / PARTS] : 0;      // the wave's first page if no window cuts the front off
  const bool new_key_apart = FUSED && t.fused.write_kv, takes_new_key = new_key_apart && wave == WAVES - 1;
  // pos: a row's own position; last: that of the last key it takes from the cache (-1: none)
  int pos[NR], last[NR], first[NR], from = 0x7fffffff, upto = -1, new_page = 0;
  float scale[NR];
  floatx4 q[NR][P], new_key[FUSED ? P : 1];
  HeadTurn<P> q_turn, k_turn;
#pragma unroll
  for (int r = 0; r < NR; ++r) {
    pos[r] = t.positions[row0 + r];
    if constexpr (FUSED) {
      const float* row = t.fused.qkv + (size_t)row0 * (t.H + 2 * t.KVH) * HD;
#pragma unroll
      for (int p = 0; p < P; ++p) q[0][p] = load4(row + head * HD + 32 * p + 4 * dq);
      q_turn.ask_weight(t.fused.q_weight, dq);
      if (takes_new_key) {
#pragma unroll
        for (int p = 0; p < P; ++p) new_key[p] = load4(row + (t.H + kv_head) * HD + 32 * p + 4 * dq);
        k_turn.ask_weight(t.fused.k_weight, dq);
      }
      q_turn.ask_angles(t.fused, pos[0], dq);
      if (new_key_apart) new_page = table[pos[0] / BH_PAGE];
    }
    last[r] = new_key_apart ? pos[r] - 1 : pos[r];
    first[r] = bh_first_visible(pos[r], t.window);
    scale[r] = query_scale(t.form, pos[r]);
    from = min(from, first[r]);
    upto = max(upto, last[r]);
    if constexpr (!FUSED) {
#pragma unroll
      for (int p = 0; p < P; ++p) q[r][p] = load4(t.q + ((size_t)(row0 + r) * t.H + head) * HD + 32 * p + 4 * dq);
    }
  }
  const int last_part = upto >= 0 ? upto / TOKENS : -1;
  bool ready = !FUSED;      // the query is what the scores are made with
  auto finish_q = [&]() {
    if constexpr (FUSED) {
      if (ready) return;
      ready = true;
      q_turn.apply(q[0], t.fused, q_turn);
    }
  };
  if constexpr (FUSED) {
    if (takes_new_key) {      // before this wave's pages, if it has any: beside them there are not the registers
      finish_q();
      k_turn.apply(new_key, t.fused, q_turn);
      float dot = 0.f;
#pragma unroll
      for (int p = 0; p < P; ++p)
#pragma unroll
        for (int e = 0; e < 4; ++e) dot = fmaf(q[0][p][e], new_key[p][e], dot);
#pragma unroll
      for (int off = 4; off > 0; off >>= 1) dot += __shfl_xor(dot, off, BH_WAVE);
      if (lane == 0) lds.new_score = dot * scale[0];
      if (head % (t.H / t.KVH) == 0 && kl == 0) {
        float* to = t.fused.k_pages + (((size_t)new_page * t.KVH + kv_head) * BH_PAGE + pos[0] % BH_PAGE) * HD + 4 * dq;
#pragma unroll
        for (int p = 0; p < P; ++p) *reinterpret_cast<floatx4*>(to + 32 * p) = new_key[p];
      }
    }
  }

  // Heads of 256: with the query's weights and angles carried into the loop there are not the registers to ask for much of a page at a time (8
  // heads on 2, 4 rows of 300 keys 31.6 us, 13.8 so, 15.6 in two launches).  Heads of 160 to 224 have them, and lose: 4 rows of 100 keys of 160 7.9 / 16.7.
  if constexpr (FUSED && P >= 8) finish_q();

  float most[NR], sum[NR], acc[NR][ND];
#pragma unroll
  for (int r = 0; r < NR; ++r) {
    most[r] = -INFINITY;
    sum[r] = 0.f;
#pragma unroll
    for (int d = 0; d < ND; ++d) acc[r][d] = 0.f;
  }
  for (int part = from / TOKENS + wave; part <= last_part; part += WAVES) {
    const int page = part / PARTS, token0 = part % PARTS * TOKENS, at0 = part * TOKENS;      // its tokens in the page, and in the sequence
    const size_t block = ((size_t)(FUSED && part == wave ? page_guess : table[page]) * t.KVH + kv_head) * BH_PAGE * HD;
    const float* keys = t.k_pages + block + (token0 + kl) * HD + 4 * dq;
    const float* values = t.v_pages + block + dl * BH_PAGE + token0 + 4 * tq;
    float s[NR][GROUPS];
    floatx4 ahead[AHEAD ? ND : 1];
    if constexpr (AHEAD) {
      // one row and a page or two a wave: the page's way from memory is the time, so all of it is asked for at once
      floatx4 k[GROUPS][P];
#pragma unroll
      for (int g = 0; g < GROUPS; ++g)
#pragma unroll
        for (int p = 0; p < P; ++p) k[g][p] = load4(keys + 8 * g * HD + 32 * p);
#pragma unroll
      for (int d = 0; d < ND; ++d) ahead[d] = load4(values + DL * d * BH_PAGE);
      __builtin_amdgcn_sched_barrier(0);
      finish_q();
#pragma unroll
      for (int g = 0; g < GROUPS; ++g) {
        float dot = 0.f;
#pragma unroll
        for (int p = 0; p < P; ++p)
#pragma unroll
          for (int e = 0; e < 4; ++e) dot = fmaf(q[0][p][e], k[g][p][e], dot);
        s[0][g] = dot;
      }
    } else {
      finish_q();
#pragma unroll
      for (int g = 0; g < GROUPS; ++g) {
        floatx4 k[P];
#pragma unroll
        for (int p = 0; p < P; ++p) k[p] = load4(keys + 8 * g * HD + 32 * p);
#pragma unroll
        for (int r = 0; r < NR; ++r) {
          float dot = 0.f;
#pragma unroll
          for (int p = 0; p < P; ++p)
#pragma unroll
            for (int e = 0; e < 4; ++e) dot = fmaf(q[r][p][e], k[p][e], dot);
          s[r][g] = dot;
        }
      }
    }
    const int token = PARTS == 1 ? 8 * dq + kl : 8 * (dq >> 1) + kl, at = at0 + token;
    float alpha[NR];
    floatx4 w[NR];
#pragma unroll
    for (int r = 0; r < NR; ++r) {
#pragma unroll
      for (int half = GROUPS / 2; half > 0; half >>= 1) {
        const bool upper = dq & (half * PARTS);
#pragma unroll
        for (int g = 0; g < half; ++g)
          s[r][g] = (upper ? s[r][g + half] : s[r][g]) + __shfl_xor(upper ? s[r][g] : s[r][g + half], half * PARTS, BH_WAVE);
      }
      if (PARTS == 2) s[r][0] += __shfl_xor(s[r][0], 1, BH_WAVE);      // (two lanes then have the same key)
      float score = s[r][0] * scale[r];
      if (t.form.cap > 0.f) score = t.form.cap * tanhf(score / t.form.cap);
      score -= slope * (float)(pos[r] - at);
      const bool seen = at >= first[r] && at <= last[r];
      score = seen ? score : -INFINITY;
      const float now = fmaxf(most[r], wave_max(score));
      const float p = score == -INFINITY ? 0.f : expf(score - now);      // also where a seen key's score is: a page of those has now -inf
      alpha[r] = most[r] == -INFINITY ? 0.f : expf(most[r] - now);
      sum[r] = sum[r] * alpha[r] + (PARTS == 2 && (dq & 1) ? 0.f : p);
      most[r] = now;
      lds.probs[wave][r][token] = p;
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");   // a wave's own LDS writes and reads, in order
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
    for (int r = 0; r < NR; ++r) {
      w[r] = load4(&lds.probs[wave][r][4 * tq]);
#pragma unroll
      for (int d = 0; d < ND; ++d) acc[r][d] *= alpha[r];
    }
    // a key that a row does not see may hold anything (behind a sequence's end, or a later row's): it must not reach that row's
    // sums, not even times zero
    bool whole = true;
#pragma unroll
    for (int r = 0; r < NR; ++r) whole = whole && first[r] <= at0 && last[r] >= at0 + TOKENS - 1;
    if (whole) {
#pragma unroll
      for (int d = 0; d < ND; ++d) {
        const floatx4 v = AHEAD ? ahead[AHEAD ? d : 0] : load4(values + DL * d * BH_PAGE);
#pragma unroll
        for (int r = 0; r < NR; ++r)
#pragma unroll
          for (int e = 0; e < 4; ++e) acc[r][d] = fmaf(w[r][e], v[e], acc[r][d]);
      }
    } else {
#pragma unroll
      for (int d = 0; d < ND; ++d) {
        const floatx4 v = AHEAD ? ahead[AHEAD ? d : 0] : load4(values + DL * d * BH_PAGE);
#pragma unroll
        for (int r = 0; r < NR; ++r)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int j = at0 + 4 * tq + e;
            acc[r][d] = fmaf(w[r][e], j >= first[r] && j <= last[r] ? v[e] : 0.f, acc[r][d]);
          }
      }
    }
    __builtin_amdgcn_wave_barrier();
  }

  // over the lanes of a dimension: three halvings (two, of the eight lanes of half a page) leave lane tq with P dimensions' sums over half
  // of the lanes, then its neighbour's
#pragma unroll
  for (int r = 0; r < NR; ++r) {
#pragma unroll
    for (int step = 0; step < (PARTS == 1 ? 3 : 2); ++step) {
      const int half = ND / 2 >> step, bit = TQ / 2 >> step;
      const bool upper = tq & bit;
#pragma unroll
      for (int d = 0; d < half; ++d)
        acc[r][d] = (upper ? acc[r][d + half] : acc[r][d]) + __shfl_xor(upper ? acc[r][d] : acc[r][d + half], bit, BH_WAVE);
    }
#pragma unroll
    for (int d = 0; d < P; ++d) {
      const float whole = acc[r][d] + __shfl_xor(acc[r][d], 1, BH_WAVE);
      if ((tq & 1) == 0) lds.o[wave][r][DL * ((tq >> 1) * P + d) + dl] = whole;
    }
    const float all = wave_sum(sum[r]);
    if (lane == 0) {
      lds.most[wave][r] = most[r];
      lds.sum[wave][r] = all;
    }
  }
  constexpr int EACH = (NR * HD + 64 * WAVES - 1) / (64 * WAVES);      // elements that a thread merges
  float new_value[EACH];
  if constexpr (FUSED) {
#pragma unroll
    for (int u = 0; u < EACH; ++u) {
      const int e = tid + u * 64 * WAVES;
      new_value[u] = e < HD ? t.fused.qkv[((size_t)row0 * (t.H + 2 * t.KVH) + t.H + t.KVH + kv_head) * HD + e] : 0.f;
    }
  }
  __syncthreads();
  const float new_score = new_key_apart ? lds.new_score : -INFINITY;
#pragma unroll
  for (int u = 0; u < EACH; ++u) {
    const int e = tid + u * 64 * WAVES, r = e / HD, d = e % HD;
    if (e >= NR * HD) break;
    float top = lds.most[0][r];
#pragma unroll
    for (int s = 1; s < WAVES; ++s) top = fmaxf(top, lds.most[s][r]);
    float total = 0.f, all = 0.f;
    if constexpr (FUSED) {
      if (new_key_apart) {
        top = fmaxf(top, new_score);
        all = new_score == -INFINITY ? 0.f : expf(new_score - top);
        total = new_value[u] * all;
      }
    }
#pragma unroll
    for (int s = 0; s < WAVES; ++s) {
      const float share = lds.most[s][r] == -INFINITY ? 0.f : expf(lds.most[s][r] - top);
      all += lds.sum[s][r] * share;
      total += lds.o[s][r][d] * share;
    }
    // a sink: one more term exp(sinks[head]) in the softmax's sum, with no key and no value
    if (t.finish.sinks) all += expf(t.finish.sinks[head] - top);
    const int row = row0 + r;
    t.out[((size_t)row * t.H + head) * HD + d] = total / all * head_gate<float>(t.finish, row, head);
  }
  if constexpr (FUSED) {
    if (new_key_apart && head % (t.H / t.KVH) == 0) {
      const size_t block = ((size_t)new_page * t.KVH + kv_head) * BH_PAGE * HD;
      const int token = pos[0] % BH_PAGE;
#pragma unroll
      for (int u = 0; u < EACH; ++u) {
        const int e = tid + u * 64 * WAVES;
        if (e < HD) t.fused.v_pages[block + (size_t)e * BH_PAGE + token] = new_value[u];
      }
    }
  }
}

constexpr int parts_of(int slices, int waves) { return slices >= 3 && (waves == 8 || waves == 2) ? 2 : 1; }

template <int P, int NR, int WAVES>
__global__ __launch_bounds__(64 * WAVES) void attention_f32_kernel(F32Attention t, int n_rows) {
  __shared__ __attribute__((aligned(16))) Lds<P, NR, WAVES> lds;
  const int row0 = blockIdx.x * NR, head = blockIdx.y;
  if constexpr (NR == 1) {
    attend_rows<P, 1, WAVES, false, parts_of(P, WAVES)>(t, lds, row0, head);
  } else {
    bool together = row0 + NR <= n_rows;
    for (int r = 1; together && r < NR; ++r) together = t.row_seq[row0 + r] == t.row_seq[row0];
    if (together) {
      attend_rows<P, NR, WAVES>(t, lds, row0, head);
      return;
    }
    for (int r = 0; r < NR && row0 + r < n_rows; ++r) {     // the end of one sequence and the start of another, or of the step
      attend_rows<P, 1, WAVES>(t, reinterpret_cast<Lds<P, 1, WAVES>&>(lds), row0 + r, head);
      __syncthreads();
    }
  }
}

template <int P, int WAVES>
__global__ __launch_bounds__(64 * WAVES) void attention_f32_fused_kernel(F32Attention t) {
  __shared__ __attribute__((aligned(16))) Lds<P, 1, WAVES> lds;
  attend_rows<P, 1, WAVES, true, parts_of(P, WAVES)>(t, lds, blockIdx.x, blockIdx.y);
}

// ---- prompts -------------------------------------------------------------------------------------------
// Sixteen columns, (row, query head) pairs of one kv head in order, a workgroup, on the float32 matrix instructions (every product a
// 32-bit fused multiply-add): a page's keys and values are read once for all of them.  Each of its four waves takes 16 of a page's
// tokens, so that short prompts keep all four busy, and loads the next page's keys while it works on this one's.  With
// v_mfma_f32_16x16x4_f32, whose operands are an element of 16 rows and four k a lane,
//     S^T[key, column] = K[key, :] . Q[column, :]        O^T[d, column] += V^T[d, key] . P^T[key, column]
// lane (i = lane % 16, g = lane / 16) loads 16 bytes of row i of an operand at 16 s + 4 g and gives its four elements to four
// instructions in turn, which take k in that order on both sides.  A lane then holds the scores of column i and keys 4 g .. 4 g + 3
// of the 16: the P^T operands of the second product as they are.  The columns may belong to several sequences, which are walked
// one after another with the others' columns masked.  A page's sums are made apart and then added, as the walk above adds blocks.
// Bound by a wave's chain of a page: its loads, 64 (heads of 128) matrix instructions of 32 clocks, and the softmax between them.
// Measured: four prompts of 744 rows in all, 8 heads of 128 on 4: 30 us, 102 in waves of a row each, which read 8 times as much;
// error against 64 bits 1.14e-7 there (1.20e-7 in the waves), 1.33e-7 for 1,000 rows of 8 heads of 256 (1.48e-7).
template <int P>
__global__ __launch_bounds__(256, P <= 4 ? 2 : 1) void attention_f32_tiles_kernel(F32Attention t, int n_rows) {
  constexpr int HD = 32 * P, CHUNKS = 2 * P, STRIDE = HD + 4, WAVES = 4;
  __shared__ float o[WAVES][16][STRIDE];
  __shared__ float tops[WAVES][16], sums[WAVES][16];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, i = lane & 15, g = lane >> 4;
  const int group = t.H / t.KVH, kv_head = blockIdx.y;
  const long column = 16L * blockIdx.x + i;
  const int row = (int)(column / group), head = kv_head * group + (int)(column % group);
  const bool exists = row < n_rows;
  const int seq = exists ? t.row_seq[row] : -1, pos = exists ? t.positions[row] : -1;
  const int first = bh_first_visible(pos < 0 ? 0 : pos, t.window);
  const float scale = query_scale(t.form, pos < 0 ? 0 : pos), slope = t.form.slopes && exists ? t.form.slopes[head] : 0.f;
  floatx4 q[CHUNKS];
#pragma unroll
  for (int s = 0; s < CHUNKS; ++s)
    q[s] = exists ? load4(t.q + ((size_t)row * t.H + head) * HD + 16 * s + 4 * g) : floatx4{0.f, 0.f, 0.f, 0.f};

  float most = -INFINITY, sum = 0.f;
  floatx4 acc[CHUNKS];
#pragma unroll
  for (int d = 0; d < CHUNKS; ++d) acc[d] = floatx4{0.f, 0.f, 0.f, 0.f};
  unsigned long long left = __ballot(exists);      // the lanes whose columns are still to be walked
  while (left) {
    const int seq_now = __builtin_amdgcn_readfirstlane(__shfl(seq, __ffsll(left) - 1, BH_WAVE));
    const bool mine = exists && seq == seq_now;
    left &= ~__ballot(mine);
    int from = mine ? first : 0x7fffffff, upto = mine ? pos : -1;
#pragma unroll
    for (int off = 8; off > 0; off >>= 1) {
      from = min(from, __shfl_xor(from, off, BH_WAVE));
      upto = max(upto, __shfl_xor(upto, off, BH_WAVE));
    }
    from = __builtin_amdgcn_readfirstlane(from);
    upto = __builtin_amdgcn_readfirstlane(upto);
    const int32_t* table = t.page_table + (size_t)seq_now * t.table_stride;
    // the wave's pages: those in which some column sees one of its 16 tokens
    const int tokens = 16 * wave;
    int page = (from - tokens - 15 + BH_PAGE - 1) / BH_PAGE;
    if (from < tokens + 15) page = 0;
    const int last = upto < tokens ? -1 : (upto - tokens) / BH_PAGE;
    floatx4 k[CHUNKS];
    auto load_keys = [&](int of) {
      const float* keys = t.k_pages + (((size_t)table[of] * t.KVH + kv_head) * BH_PAGE + tokens + i) * HD + 4 * g;
#pragma unroll
      for (int s = 0; s < CHUNKS; ++s) k[s] = load4(keys + 16 * s);
    };
    if (page <= last) load_keys(page);
    for (; page <= last; ++page) {
      const size_t block = ((size_t)table[page] * t.KVH + kv_head) * BH_PAGE * HD;
      const float* values = t.v_pages + block + i * BH_PAGE + tokens + 4 * g;
      floatx4 v[CHUNKS];
#pragma unroll
      for (int d = 0; d < CHUNKS; ++d) v[d] = load4(values + 16 * d * BH_PAGE);
      // eight chains of half of k, then eight of the other half: no chain is longer than those of the walk above
      floatx4 p = {0.f, 0.f, 0.f, 0.f};
      constexpr int MIDDLE = (P + 1) / 2 * 2;
#pragma unroll
      for (int from_s = 0; from_s < CHUNKS; from_s += MIDDLE) {
        floatx4 chain[8] = {};
#pragma unroll
        for (int s = from_s; s < from_s + MIDDLE && s < CHUNKS; s += 2)
#pragma unroll
          for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int h = 0; h < 2; ++h)
              chain[2 * e + h] = __builtin_amdgcn_mfma_f32_16x16x4f32(k[s + h][e], q[s + h][e], chain[2 * e + h], 0, 0, 0);
        p += ((chain[0] + chain[1]) + (chain[2] + chain[3])) + ((chain[4] + chain[5]) + (chain[6] + chain[7]));
      }
      if (page < last) load_keys(page + 1);
      float top = -INFINITY;
      bool whole = mine;
      const int at = page * BH_PAGE + tokens + 4 * g;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        float score = p[e] * scale;
        if (t.form.cap > 0.f) score = t.form.cap * tanhf(score / t.form.cap);
        score -= slope * (float)(pos - at - e);
        const bool seen = mine && at + e >= first && at + e <= pos;
        whole = whole && seen;
        p[e] = seen ? score : -INFINITY;
        top = fmaxf(top, p[e]);
      }
      top = fmaxf(top, __shfl_xor(top, 16, BH_WAVE));
      top = fmaxf(top, __shfl_xor(top, 32, BH_WAVE));
      const float now = fmaxf(most, top);
      const float alpha = most == -INFINITY ? 0.f : expf(most - now);
#pragma unroll
      for (int e = 0; e < 4; ++e) p[e] = p[e] == -INFINITY ? 0.f : expf(p[e] - now);
      sum = sum * alpha + ((p[0] + p[1]) + (p[2] + p[3]));
      most = now;
      // A key that a column does not see may hold anything (behind a sequence's end, or a later row's): it must not reach that
      // column's sums, not even times zero.  Where a column does not see all of the tokens, numbers that are not finite are set aside
      // and then given to those who see them, one by one.
      bool odd_ones = false;
      if (!__all(whole)) {
#pragma unroll
        for (int d = 0; d < CHUNKS; ++d)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const bool finite = fabsf(v[d][e]) < INFINITY;
            odd_ones = odd_ones || !finite;
            v[d][e] = finite ? v[d][e] : 0.f;
          }
      }
#pragma unroll
      for (int d = 0; d < CHUNKS; d += 2) {
        floatx4 part[2][2] = {};
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
          for (int h = 0; h < 2; ++h) part[h][e & 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(v[d + h][e], p[e], part[h][e & 1], 0, 0, 0);
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int e = 0; e < 4; ++e) acc[d + h][e] = fmaf(acc[d + h][e], alpha, part[h][0][e] + part[h][1][e]);
      }
      if (__any(odd_ones)) {
        for (int token = 0; token < 16; ++token) {
          const int e = token & 3, place = page * BH_PAGE + tokens + token;
          const float w = __shfl(e == 0 ? p[0] : e == 1 ? p[1] : e == 2 ? p[2] : p[3], i + 16 * (token >> 2), BH_WAVE);
          if (mine && place >= first && place <= pos) {
#pragma unroll
            for (int d = 0; d < CHUNKS; ++d)
#pragma unroll
              for (int r = 0; r < 4; ++r) {
                const float one = t.v_pages[block + (size_t)(16 * d + 4 * g + r) * BH_PAGE + tokens + token];
                if (!(fabsf(one) < INFINITY)) acc[d][r] = fmaf(w, one, acc[d][r]);
              }
          }
        }
      }
    }
  }

  sum += __shfl_xor(sum, 16, BH_WAVE);
  sum += __shfl_xor(sum, 32, BH_WAVE);
#pragma unroll
  for (int d = 0; d < CHUNKS; ++d) *reinterpret_cast<floatx4*>(&o[wave][i][16 * d + 4 * g]) = acc[d];
  if (g == 0) {
    tops[wave][i] = most;
    sums[wave][i] = sum;
  }
  __syncthreads();
  for (int e = threadIdx.x; e < 16 * HD; e += 64 * WAVES) {
    const int c = e / HD, d = e % HD;
    const long of = 16L * blockIdx.x + c;
    const int to_row = (int)(of / group), to_head = kv_head * group + (int)(of % group);
    if (to_row >= n_rows) break;      // so are all that follow
    float top = tops[0][c];
#pragma unroll
    for (int s = 1; s < WAVES; ++s) top = fmaxf(top, tops[s][c]);
    float total = 0.f, all = 0.f;
#pragma unroll
    for (int s = 0; s < WAVES; ++s) {
      const float share = tops[s][c] == -INFINITY ? 0.f : expf(tops[s][c] - top);
      all += sums[s][c] * share;
      total += o[s][c][d] * share;
    }
    if (t.finish.sinks) all += expf(t.finish.sinks[to_head] - top);
    t.out[((size_t)to_row * t.H + to_head) * HD + d] = total / all * head_gate<float>(t.finish, to_row, to_head);
  }
}

// Whether a step of prompts goes in tiles.  A tile walks its sequences one after another, a page of a sequence after the other, where
// the walk above has every row's pages in waves of their own: rows of several sequences that look far back, one behind the other in a
// tile, are a chain of all their pages (a prompt of 512 rows beside 14 rows behind 1,000 keys, 8 heads of 128 on 4: 138 us, 406 in
// tiles).  So both times are estimated, each from its longest chain of pages and from all its pages together (us a page of the chain; ns
// a compute unit and page of a tile, ns a row, head and page of the walk, whose four waves share a row's pages, so that 1.5 more are
// waited for on average; they add as squares do).  Fitted to 304 steps of 1 to 13 sequences, prompts alone, behind up to 3,000 keys and
// beside decoding rows behind up to 4,000, of 16 head counts and sizes, to 13 % (tiles) and 17 % (walk): with 15 % asked of the tiles
// the choice takes 0.2 % longer than the better one on average, and one step of the 304 was 9 % slower than walked.
// `start` and `past`: the step's sequences as the host knows them, or null: then the average is all there is to go by.
bool tiles_pay(int n_rows, int n_seqs, int H, int KVH, int hd, int span, const int32_t* start, const int32_t* past) {
  if (n_rows < 32 * n_seqs || (long)n_rows * H <= 8L * bh_compute_units() || KVH > 65535) return false;
  if (!start || !past) return true;
  constexpr double TILE_PAGE[8] = {0.8, 1.6, 2.4, 2.9, 5.4, 6.5, 6.8, 7.8}, WALK_PAGE[8] = {0.43, 0.75, 2.44, 3.49, 3.13, 6.6, 8.88, 5.6};
  const int group = H / KVH, seen = span ? (span > 0 ? span : -span) / BH_PAGE + 2 : 0x7fffffff;      // pages that a window or chunk touches
  double row_pages = 0., tile_pages = 0.;
  long chain = 0, tile = -1, walked = 0, most = 0;      // tile: the one that the sequences so far end in; walked: the pages it walks for them
  for (int s = 0; s < n_seqs; ++s) {
    const int rows = start[s + 1] - start[s];
    if (rows <= 0) continue;
    const int pages = std::min((past[s] + rows - 1) / BH_PAGE + 1, seen);
    const double average = 0.5 * (std::min(past[s] / BH_PAGE + 1, seen) + pages);
    const long first = (long)start[s] * group / 16, last = ((long)start[s + 1] * group - 1) / 16;
    row_pages += rows * (average + 1.5);
    tile_pages += (double)(last - first + 1) * average;
    walked = (first == tile ? walked : 0) + pages;
    chain = std::max(chain, walked);
    most = std::max(most, (long)pages);
    if (last != first) walked = pages;
    tile = last;
  }
  const int size = hd / 32 - 1;
  const double in_tiles = 6.0 + std::hypot(chain * (0.67 + 0.018 * hd), tile_pages * KVH * TILE_PAGE[size] / bh_compute_units());
  const double by_rows = 18.0 + std::hypot((0.25 * most + 1.0) * 0.049 * hd, 1e-3 * row_pages * H * WALK_PAGE[size]);
  return 1.15 * in_tiles <= by_rows;
}

constexpr int many_waves(int slices) { return slices <= 4 ? 8 : 4; }
// Rows that see one page have work for one wave, or for two where the eight waves of longer rows take half pages: the parts and the order
// in which their sums are added are then the same, so that a row's result does not hang on how many pages its step may see (a captured
// step is launched for more than its rows hold; idle waves add zeros).
constexpr int one_page_waves(int slices) { return parts_of(slices, many_waves(slices)); }

// A decode step from its projection rows: as many waves a row and head as `launch` gives it.  In two launches / one, us, 8 rows of 100 keys,
// 16 heads of 128 on 8 7.3 / 5.9, 4 rows of 300 keys, 4 heads of 64 on 2 7.5 / 5.6.
template <int P>
void launch_fused(const F32Attention& t, int n_rows, int most_pages, hipStream_t stream) {
  const long units = bh_compute_units(), each = (long)n_rows * t.H;
  const dim3 grid(n_rows, t.H);
  if (most_pages <= 1 && each < 2 * units) attention_f32_fused_kernel<P, one_page_waves(P)><<<grid, 64 * one_page_waves(P), 0, stream>>>(t);
  else if (most_pages <= 1 || (most_pages <= 4 && each >= 4 * units)) attention_f32_fused_kernel<P, 1><<<grid, 64, 0, stream>>>(t);
  else if (each < 2 * units) attention_f32_fused_kernel<P, many_waves(P)><<<grid, 64 * many_waves(P), 0, stream>>>(t);
  else attention_f32_fused_kernel<P, 4><<<grid, 256, 0, stream>>>(t);
}

template <int P>
void launch(const F32Attention& t, int n_rows, int n_seqs, int most_pages, bool tiled, hipStream_t stream) {
  constexpr int NR = P <= 4 ? 4 : P <= 7 ? 2 : 1;      // what the registers hold without spilling
  const bool prompts = n_rows >= 8 * n_seqs;
  // Columns in tiles where (rows, heads) are more than the waves of two a SIMD, so that a wave a row would come in rounds, and the step
  // is prompts.  As below / in tiles, us: 300, 186, 200 and 58 rows of 8 heads of 128 on 4 102 / 30, on 16 heads 198 / 40, 16 prompts of
  // 40 rows of 16 heads 52 / 23, one of 256 40 / 18, of 2,048 of 8 heads 724 / 216, of 1,000 of 8 heads of 256 on 1 400 / 129; but
  // 4 prompts of 64 of 8 heads of 256 17 / 19, and one of 33 of 16 heads 6.8 / 10.2.
  if (tiled) {
    const long tiles = ((long)n_rows * (t.H / t.KVH) + 15) / 16;
    attention_f32_tiles_kernel<P><<<dim3((unsigned)tiles, t.KVH), 256, 0, stream>>>(t, n_rows);
    return;
  }
  // Rows that see one page have work for one wave a row and head, and rows that see a few have it where they and the heads fill the
  // chip: waves of their own leave no wave without a page.  Four waves on four rows / a wave a row, us, 16 heads of 128 on 8: one
  // prompt of 33 rows 15.9 / 6.8, 16 of 40 172 / 52, one of 256 61 / 40; 8 heads of 256 on 2: 4 prompts of 64 47 / 17, but 30 rows
  // behind 100 cached keys (240 workgroups) 8.5 / 12.3.
  if (most_pages <= 1 || (most_pages <= 4 && (long)n_rows * t.H >= (prompts ? 2L : 4L) * bh_compute_units())) {
    constexpr int FEW = P <= 4 ? 1 : NR;
    if (prompts) attention_f32_kernel<P, FEW, 1><<<dim3((n_rows + FEW - 1) / FEW, t.H), 64, 0, stream>>>(t, n_rows);
    else if ((long)n_rows * t.H < 2 * bh_compute_units())
      attention_f32_kernel<P, 1, one_page_waves(P)><<<dim3(n_rows, t.H), 64 * one_page_waves(P), 0, stream>>>(t, n_rows);
    else attention_f32_kernel<P, 1, 1><<<dim3(n_rows, t.H), 64, 0, stream>>>(t, n_rows);
    return;
  }
  // Prompts: rows of one sequence share the pages' reads.  Else a row a workgroup, of eight waves where the rows and heads alone
  // leave compute units idle and the registers allow it: as many pages are then on their way together.
  constexpr int MANY = many_waves(P);
  if (prompts) attention_f32_kernel<P, NR, 4><<<dim3((n_rows + NR - 1) / NR, t.H), 256, 0, stream>>>(t, n_rows);
  else if ((long)n_rows * t.H < 2 * bh_compute_units())
    attention_f32_kernel<P, 1, MANY><<<dim3(n_rows, t.H), 64 * MANY, 0, stream>>>(t, n_rows);
  else attention_f32_kernel<P, 1, 4><<<dim3(n_rows, t.H), 256, 0, stream>>>(t, n_rows);
}

}  // namespace

// Whether these sizes and addresses go here.
extern "C" int bh_attention_f32_takes(int H, int KVH, int hd, int kv_order) {
  return hd % 32 == 0 && hd >= 32 && hd <= 256 && KVH > 0 && H % KVH == 0 && H <= 65535 && kv_order == BH_KV_ROWS ? 1 : 0;
}
// Whether a step's rows go in tiles of columns: start [n_seqs + 1] and past [n_seqs] on the host, or null.
extern "C" int bh_attention_f32_tiles(int n_rows, int n_seqs, int H, int KVH, int hd, int window, const int32_t* start, const int32_t* past) {
  return n_rows > 0 && n_seqs > 0 && bh_attention_f32_takes(H, KVH, hd, BH_KV_ROWS) && tiles_pay(n_rows, n_seqs, H, KVH, hd, window, start, past) ? 1 : 0;
}
// `n_seqs`: the rows of the page table.  `most_pages`: how many pages a row sees at most, as far as the caller knows.  `host_start`
// [n_seqs + 1] and `host_past` [n_seqs]: where each sequence's rows begin and what its cache held before them, in host memory, or null.
extern "C" int bh_attention_f32(const float* q, float* out, const float* k_pages, const float* v_pages, const int32_t* page_table,
                                int table_stride, int n_seqs, int most_pages, const int32_t* host_start, const int32_t* host_past,
                                const int32_t* row_seq, const int32_t* positions, int n_rows, int H, int KVH, int hd, float scale, int window, int kv_order, const float* sinks, const void* gates,
                                int gate_stride, float cap, const float* slopes, float temp_coef, int temp_every, float out_scale,
                                hipStream_t stream) {
  BH_REQUIRE(n_rows > 0 && H > 0 && KVH > 0 && hd > 0 && n_seqs > 0, "attention: sizes must be positive");
  BH_REQUIRE(bh_attention_f32_takes(H, KVH, hd, kv_order), "attention: %d heads of %d on %d are not for the float32 kernel", H, hd, KVH);
  BH_REQUIRE((((uintptr_t)q | (uintptr_t)k_pages | (uintptr_t)v_pages) % 16) == 0, "attention: q, keys and values must be 16-byte aligned");
  BH_REQUIRE(gates == nullptr || gate_stride >= H, "attention: a gate a head (%d) lies outside a row of %d", H, gate_stride);
  const ScoreForm form = {scale, cap, slopes, temp_coef, temp_every};
  if (const char* fault = bh_score_form_fault(form)) return bh_fail("attention: %s", fault);
  const F32Attention t = {q, out, k_pages, v_pages, page_table, table_stride, row_seq, positions, H, KVH, form, window,
                          {sinks, gates, gate_stride, out_scale}, {}};
  const bool tiled = tiles_pay(n_rows, n_seqs, H, KVH, hd, window, host_start, host_past);
  switch (hd / 32) {
    case 1: launch<1>(t, n_rows, n_seqs, most_pages, tiled, stream); break;
    case 2: launch<2>(t, n_rows, n_seqs, most_pages, tiled, stream); break;
    case 3: launch<3>(t, n_rows, n_seqs, most_pages, tiled, stream); break;
    case 4: launch<4>(t, n_rows, n_seqs, most_pages, tiled, stream); break;
    case 5: launch<5>(t, n_rows, n_seqs, most_pages, tiled, stream); break;
    case 6: launch<6>(t, n_rows, n_seqs, most_pages, tiled, stream); break;
    case 7: launch<7>(t, n_rows, n_seqs, most_pages, tiled, stream); break;
    default: launch<8>(t, n_rows, n_seqs, most_pages, tiled, stream); break;
  }
  return bh_check_launch("attention_f32");
}

// A decode step (row s is sequence s's) from its fused projection rows [q heads | k heads | v heads]: per-head RMSNorm of q and k (weights
// may be null), rotation over the whole head at the row's position (tables may be null), the new key and value into the cache (unless
// write_kv is 0: the entry is another layer's), and attention over the cache and the new key.  `most_pages` as above.
extern "C" int bh_attention_f32_decode_fused(const float* qkv, float* out, float* k_pages, float* v_pages, const int32_t* page_table,
                                             int table_stride, const int32_t* positions, int n_rows, int H, int KVH, int hd, float scale,
                                             int window, int max_position, int most_pages, const float* q_weight, const float* k_weight, float eps,
                                             const float* cos_table, const float* sin_table, int table_positions, int rot, int write_kv,
                                             hipStream_t stream) {
  BH_REQUIRE(n_rows > 0 && H > 0 && KVH > 0 && hd > 0 && max_position >= 0, "attention_decode_fused: sizes must be positive");
  BH_REQUIRE(bh_attention_f32_takes(H, KVH, hd, BH_KV_ROWS), "attention_decode_fused: %d heads of %d on %d are not for the float32 kernel", H, hd, KVH);
  BH_REQUIRE((((uintptr_t)qkv | (uintptr_t)k_pages | (uintptr_t)v_pages | (uintptr_t)q_weight | (uintptr_t)k_weight | (uintptr_t)cos_table |
               (uintptr_t)sin_table) % 16) == 0, "attention_decode_fused: rows, cache, weights and tables must be 16-byte aligned");
  BH_REQUIRE((q_weight == nullptr) == (k_weight == nullptr), "attention_decode_fused: give both norm weights or neither");
  BH_REQUIRE((cos_table == nullptr) == (sin_table == nullptr), "attention_decode_fused: cos and sin tables come together");
  BH_REQUIRE(cos_table == nullptr || (rot == hd && hd % 64 == 0),
             "attention_decode_fused: the rotation must span the whole head (%d of %d) and the head be a multiple of 64", rot, hd);
  BH_REQUIRE(cos_table == nullptr || max_position < table_positions,
             "attention_decode_fused: position %d is outside the rotation table of %d positions", max_position, table_positions);
  const F32Attention t = {nullptr, out, k_pages, v_pages, page_table, table_stride, nullptr, positions, H, KVH,
                          ScoreForm{scale, 0.f, nullptr, 0.f, 0}, window, HeadEnd{},
                          {qkv, q_weight, k_weight, eps, cos_table, sin_table, write_kv, k_pages, v_pages}};
  switch (hd / 32) {
    case 1: launch_fused<1>(t, n_rows, most_pages, stream); break;
    case 2: launch_fused<2>(t, n_rows, most_pages, stream); break;
    case 3: launch_fused<3>(t, n_rows, most_pages, stream); break;
    case 4: launch_fused<4>(t, n_rows, most_pages, stream); break;
    case 5: launch_fused<5>(t, n_rows, most_pages, stream); break;
    case 6: launch_fused<6>(t, n_rows, most_pages, stream); break;
    case 7: launch_fused<7>(t, n_rows, most_pages, stream); break;
    default: launch_fused<8>(t, n_rows, most_pages, stream); break;
  }
  return bh_check_launch("attention_f32_decode_fused");
}
