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
// Measured (8 heads of 128 on 4): a decode step of 4 rows at 40 to 300 keys 8.2 us, 54 with a thread a key (generic.hip: every
// lane its own line), 20 before a page's keys and values were asked for together; four prompts of 695 rows in all, up to 256 each,
// 41 us in waves of their own, 94 in workgroups of four waves on four rows, 120 there.
#include "common.h"

typedef float floatx4 __attribute__((ext_vector_type(4)));

namespace {

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
};

__device__ inline floatx4 load4(const float* p) { return *reinterpret_cast<const floatx4*>(p); }

// LDS of a workgroup: a page's probabilities a wave and row, and the waves' results
template <int P, int NR, int WAVES>
struct Lds {
  float probs[WAVES][NR][BH_PAGE];
  float most[WAVES][NR], sum[WAVES][NR];
  float o[WAVES][NR][32 * P];
};

// Rows row0 .. row0 + NR - 1, all of the sequence of row0.
template <int P, int NR, int WAVES>
__device__ void attend_rows(const F32Attention& t, Lds<P, NR, WAVES>& lds, int row0, int head) {
  constexpr int HD = 32 * P;
  constexpr bool AHEAD = NR == 1 && P <= 4;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int kl = lane >> 3, dq = lane & 7;    // keys: the lane's key among eight, its 16 bytes of each 32 dimensions
  const int dl = lane >> 4, tq = lane & 15;   // values: the lane's dimension among four, its four tokens
  const int kv_head = head / (t.H / t.KVH);
  const int32_t* table = t.page_table + (size_t)t.row_seq[row0] * t.table_stride;
  const float slope = t.form.slopes ? t.form.slopes[head] : 0.f;

  int pos[NR], first[NR], from = 0x7fffffff, upto = 0;
  float scale[NR];
  floatx4 q[NR][P];
#pragma unroll
  for (int r = 0; r < NR; ++r) {
    pos[r] = t.positions[row0 + r];
    first[r] = bh_first_visible(pos[r], t.window);
    scale[r] = query_scale(t.form, pos[r]);
    from = min(from, first[r]);
    upto = max(upto, pos[r]);
#pragma unroll
    for (int p = 0; p < P; ++p) q[r][p] = load4(t.q + ((size_t)(row0 + r) * t.H + head) * HD + 32 * p + 4 * dq);
  }

  float most[NR], sum[NR], acc[NR][8 * P];
#pragma unroll
  for (int r = 0; r < NR; ++r) {
    most[r] = -INFINITY;
    sum[r] = 0.f;
#pragma unroll
    for (int d = 0; d < 8 * P; ++d) acc[r][d] = 0.f;
  }
  for (int page = from / BH_PAGE + wave; page <= upto / BH_PAGE; page += WAVES) {
    const size_t block = ((size_t)table[page] * t.KVH + kv_head) * BH_PAGE * HD;
    const float* keys = t.k_pages + block + kl * HD + 4 * dq;
    const float* values = t.v_pages + block + dl * BH_PAGE + 4 * tq;
    float s[NR][8];
    floatx4 ahead[AHEAD ? 8 * P : 1];
    if constexpr (AHEAD) {
      // one row and a page or two a wave: the page's way from memory is the time, so all of it is asked for at once
      floatx4 k[8][P];
#pragma unroll
      for (int g = 0; g < 8; ++g)
#pragma unroll
        for (int p = 0; p < P; ++p) k[g][p] = load4(keys + 8 * g * HD + 32 * p);
#pragma unroll
      for (int d = 0; d < 8 * P; ++d) ahead[d] = load4(values + 4 * d * BH_PAGE);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int g = 0; g < 8; ++g) {
        float dot = 0.f;
#pragma unroll
        for (int p = 0; p < P; ++p)
#pragma unroll
          for (int e = 0; e < 4; ++e) dot = fmaf(q[0][p][e], k[g][p][e], dot);
        s[0][g] = dot;
      }
    } else {
#pragma unroll
      for (int g = 0; g < 8; ++g) {
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
    const int token = 8 * dq + kl, at = page * BH_PAGE + token;
    float alpha[NR];
    floatx4 w[NR];
#pragma unroll
    for (int r = 0; r < NR; ++r) {
#pragma unroll
      for (int half = 4; half > 0; half >>= 1) {
        const bool upper = dq & half;
#pragma unroll
        for (int g = 0; g < half; ++g)
          s[r][g] = (upper ? s[r][g + half] : s[r][g]) + __shfl_xor(upper ? s[r][g] : s[r][g + half], half, BH_WAVE);
      }
      float score = s[r][0] * scale[r];
      if (t.form.cap > 0.f) score = t.form.cap * tanhf(score / t.form.cap);
      score -= slope * (float)(pos[r] - at);
      const bool seen = at >= first[r] && at <= pos[r];
      score = seen ? score : -INFINITY;
      const float now = fmaxf(most[r], wave_max(score));
      const float p = score == -INFINITY ? 0.f : expf(score - now);      // also where a seen key's score is: a page of those has now -inf
      alpha[r] = most[r] == -INFINITY ? 0.f : expf(most[r] - now);
      sum[r] = sum[r] * alpha[r] + p;
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
      for (int d = 0; d < 8 * P; ++d) acc[r][d] *= alpha[r];
    }
    // a key that a row does not see may hold anything (behind a sequence's end, or a later row's): it must not reach that row's
    // sums, not even times zero
    bool whole = true;
#pragma unroll
    for (int r = 0; r < NR; ++r) whole = whole && first[r] <= page * BH_PAGE && pos[r] >= page * BH_PAGE + BH_PAGE - 1;
    if (whole) {
#pragma unroll
      for (int d = 0; d < 8 * P; ++d) {
        const floatx4 v = AHEAD ? ahead[AHEAD ? d : 0] : load4(values + 4 * d * BH_PAGE);
#pragma unroll
        for (int r = 0; r < NR; ++r)
#pragma unroll
          for (int e = 0; e < 4; ++e) acc[r][d] = fmaf(w[r][e], v[e], acc[r][d]);
      }
    } else {
#pragma unroll
      for (int d = 0; d < 8 * P; ++d) {
        const floatx4 v = AHEAD ? ahead[AHEAD ? d : 0] : load4(values + 4 * d * BH_PAGE);
#pragma unroll
        for (int r = 0; r < NR; ++r)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int j = page * BH_PAGE + 4 * tq + e;
            acc[r][d] = fmaf(w[r][e], j >= first[r] && j <= pos[r] ? v[e] : 0.f, acc[r][d]);
          }
      }
    }
    __builtin_amdgcn_wave_barrier();
  }

  // over the 16 lanes of a dimension: three halvings leave lane tq with P dimensions' sums over eight lanes, then its neighbour's
#pragma unroll
  for (int r = 0; r < NR; ++r) {
#pragma unroll
    for (int step = 0; step < 3; ++step) {
      const int half = 4 * P >> step, bit = 8 >> step;
      const bool upper = tq & bit;
#pragma unroll
      for (int d = 0; d < half; ++d)
        acc[r][d] = (upper ? acc[r][d + half] : acc[r][d]) + __shfl_xor(upper ? acc[r][d] : acc[r][d + half], bit, BH_WAVE);
    }
#pragma unroll
    for (int d = 0; d < P; ++d) {
      const float whole = acc[r][d] + __shfl_xor(acc[r][d], 1, BH_WAVE);
      if ((tq & 1) == 0) lds.o[wave][r][4 * ((tq >> 1) * P + d) + dl] = whole;
    }
    const float all = wave_sum(sum[r]);
    if (lane == 0) {
      lds.most[wave][r] = most[r];
      lds.sum[wave][r] = all;
    }
  }
  __syncthreads();
  for (int e = tid; e < NR * HD; e += 64 * WAVES) {
    const int r = e / HD, d = e % HD;
    float top = lds.most[0][r];
#pragma unroll
    for (int s = 1; s < WAVES; ++s) top = fmaxf(top, lds.most[s][r]);
    float total = 0.f, all = 0.f;
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
}

template <int P, int NR, int WAVES>
__global__ __launch_bounds__(64 * WAVES) void attention_f32_kernel(F32Attention t, int n_rows) {
  __shared__ __attribute__((aligned(16))) Lds<P, NR, WAVES> lds;
  const int row0 = blockIdx.x * NR, head = blockIdx.y;
  if constexpr (NR == 1) {
    attend_rows<P, 1, WAVES>(t, lds, row0, head);
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

template <int P>
void launch(const F32Attention& t, int n_rows, int n_seqs, int most_pages, hipStream_t stream) {
  constexpr int NR = P <= 4 ? 4 : P <= 7 ? 2 : 1;      // what the registers hold without spilling
  const bool prompts = n_rows >= 8 * n_seqs;
  // Rows that see one page have work for one wave a row and head, and rows that see a few have it where they and the heads fill the
  // chip: waves of their own leave no wave without a page.  Four waves on four rows / a wave a row, us, 16 heads of 128 on 8: one
  // prompt of 33 rows 15.9 / 6.8, 16 of 40 172 / 52, one of 256 61 / 40; 8 heads of 256 on 2: 4 prompts of 64 47 / 17, but 30 rows
  // behind 100 cached keys (240 workgroups) 8.5 / 12.3.
  if (most_pages <= 1 || (most_pages <= 4 && (long)n_rows * t.H >= (prompts ? 2L : 4L) * bh_compute_units())) {
    constexpr int FEW = P <= 4 ? 1 : NR;
    if (prompts) attention_f32_kernel<P, FEW, 1><<<dim3((n_rows + FEW - 1) / FEW, t.H), 64, 0, stream>>>(t, n_rows);
    else attention_f32_kernel<P, 1, 1><<<dim3(n_rows, t.H), 64, 0, stream>>>(t, n_rows);
    return;
  }
  // Prompts: rows of one sequence share the pages' reads.  Else a row a workgroup, of eight waves where the rows and heads alone
  // leave compute units idle and the registers allow it: as many pages are then on their way together.
  constexpr int MANY = P <= 3 ? 8 : 4;
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
// `n_seqs`: the rows of the page table.  `most_pages`: how many pages a row sees at most, as far as the caller knows.
extern "C" int bh_attention_f32(const float* q, float* out, const float* k_pages, const float* v_pages, const int32_t* page_table,
                                int table_stride, int n_seqs, int most_pages, const int32_t* row_seq, const int32_t* positions,
                                int n_rows, int H, int KVH, int hd, float scale, int window, int kv_order, const float* sinks, const void* gates,
                                int gate_stride, float cap, const float* slopes, float temp_coef, int temp_every, float out_scale,
                                hipStream_t stream) {
  BH_REQUIRE(n_rows > 0 && H > 0 && KVH > 0 && hd > 0 && n_seqs > 0, "attention: sizes must be positive");
  BH_REQUIRE(bh_attention_f32_takes(H, KVH, hd, kv_order), "attention: %d heads of %d on %d are not for the float32 kernel", H, hd, KVH);
  BH_REQUIRE((((uintptr_t)q | (uintptr_t)k_pages | (uintptr_t)v_pages) % 16) == 0, "attention: q, keys and values must be 16-byte aligned");
  BH_REQUIRE(gates == nullptr || gate_stride >= H, "attention: a gate a head (%d) lies outside a row of %d", H, gate_stride);
  const ScoreForm form = {scale, cap, slopes, temp_coef, temp_every};
  if (const char* fault = bh_score_form_fault(form)) return bh_fail("attention: %s", fault);
  const F32Attention t = {q, out, k_pages, v_pages, page_table, table_stride, row_seq, positions, H, KVH, form, window,
                          {sinks, gates, gate_stride, out_scale}};
  switch (hd / 32) {
    case 1: launch<1>(t, n_rows, n_seqs, most_pages, stream); break;
    case 2: launch<2>(t, n_rows, n_seqs, most_pages, stream); break;
    case 3: launch<3>(t, n_rows, n_seqs, most_pages, stream); break;
    case 4: launch<4>(t, n_rows, n_seqs, most_pages, stream); break;
    case 5: launch<5>(t, n_rows, n_seqs, most_pages, stream); break;
    case 6: launch<6>(t, n_rows, n_seqs, most_pages, stream); break;
    case 7: launch<7>(t, n_rows, n_seqs, most_pages, stream); break;
    default: launch<8>(t, n_rows, n_seqs, most_pages, stream); break;
  }
  return bh_check_launch("attention_f32");
}
