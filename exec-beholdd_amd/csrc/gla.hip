// Recurrences over a matrix state per (sequence, head) whose rows decay each by a factor of its own that the token sets.  Two rules:
//   gated linear attention   S_t = diag(a_t) S_(t-1) + k_t v_t^T,   o_t = S_t^T q_t,   a_t = sigmoid(z_t + b)^(1/tau)
//   wkv (RWKV)               o_t = (S_(t-1) + diag(u) k_t v_t^T)^T r_t,   S_t = diag(a_t) S_(t-1) + k_t v_t^T,   a_t = exp(-exp(z_t + b)):
//                            what a token reads are the tokens before it, and itself through the bonus u
// (one a per key channel).
//   gla_scan, wkv_scan   walk a sequence's rows of the step in order from the state in row seq_slot and leave the state after the
//              last row in row seq_to (the same one, or one that no sequence of the step starts from); prompts, portions of prompts and decode steps are the same walk.
// S is [dim][vdim] float32.  Decays (through the logarithm of the sigmoid, so that 1/tau is a factor), bonus, state, both
// products and the read-out are float32; only q (r), k and v are read in the activations' type.
#include "chunks.h"
#include "common.h"

enum ScanRule { RULE_GLA = 0, RULE_WKV = 1 };
#define GLA_STAGE 16      // rows that go through LDS at a time

// A barrier between the waves of a workgroup that orders their LDS traffic only: a wave waits for its own LDS operations,
// not for the global loads it has in flight (__syncthreads waits for those too, which would end every read-ahead at the
// next barrier; here the next stage's loads stay on their way across the barriers of this stage).
__device__ inline void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

__device__ inline float log_sigmoid_f32(float x) { return fminf(x, 0.f) - log1pf(expf(-fabsf(x))); }

// A workgroup takes a (sequence, head, tile of VT value columns).  Thread (column, slice) keeps rows slice * R .. + R - 1 of its
// column of S in registers.  GLA_STAGE rows' decays, keys, queries (LDS rows of SL * R floats, zeros beyond dim) and the tile's
// values are staged at a time; a row's shares of o are added over a wave's slices by lane exchanges and over the waves through
// LDS, in a fixed order.  The next stage's numbers are asked for (into registers, GLA_AHEAD elements a thread and array; what a
// stage has beyond that is read when it is staged) before this stage's rows are walked, so that the walk hides their way from
// memory.
#define GLA_AHEAD 4
#define GLA_GROUP 4
#define GLA_KEPT 8        // key channels a thread keeps a product of decays for: heads of up to 2,048 key dimensions

// Long sequences in chunks of `rows` rows (0: whole sequences), `count` chunks for the longest; scratch memory for a chunk's last
// state [n_seqs][count][H][dim][vdim], its decays' product [n_seqs][count][H][dim] and a row's decayed query [rows][H][dim].
struct GlaChunks {
  int rows, count;
  float* states;
  float* decays;
  float* queries;
};

template <typename T, int R, int RULE>
__global__ __launch_bounds__(256, (R <= 16 ? 2 : 1)) void gla_scan_kernel(const T* __restrict__ q, const T* __restrict__ k, const T* __restrict__ v, int row_stride,
                                                       const float* __restrict__ z, int z_stride, const float* __restrict__ bias,
                                                       float inv_tau, const float* __restrict__ bonus, float q_scale,
                                                       float* __restrict__ state, long slot_stride,
                                                       const int32_t* __restrict__ seq_start, const int32_t* __restrict__ seq_slot, const int32_t* __restrict__ seq_to,
                                                       float* __restrict__ out, int H, int dim, int vdim, int VT, GlaChunks chunks) {
  extern __shared__ __align__(16) float lds[];
  constexpr int GROUP = RULE == RULE_WKV ? GLA_GROUP / 2 : GLA_GROUP;      // (the old state is read beside the new one: more registers a row)
  const int SL = 256 / VT, DP = SL * R;      // VT and R are powers of two, so are SL and DP: shifts and masks below
  const int dp_shift = __builtin_ctz(DP), vt_shift = __builtin_ctz(VT);
  float* a_s = lds;                          // [GLA_STAGE][DP]
  float* k_s = a_s + GLA_STAGE * DP;
  float* q_s = k_s + GLA_STAGE * DP;
  float* v_s = q_s + GLA_STAGE * DP;         // [GLA_STAGE][VT]
  float* part = v_s + GLA_STAGE * VT;        // [GLA_STAGE][PARTS][VT]: a wave's slices' shares added up (VT < 64), or a slice's own
  const int PARTS = VT >= BH_WAVE ? SL : 256 / BH_WAVE;
  // wkv: a token reads itself as (sum_d r_d u_d k_d) v, one number a row and head beside what it reads of the state
  __shared__ float own_s[RULE == RULE_WKV ? GLA_STAGE : 1];
  const int seq = blockIdx.x / chunks.count, chunk = blockIdx.x % chunks.count, head = blockIdx.y, v0 = blockIdx.z * VT;
  const int col = threadIdx.x & (VT - 1), slice = threadIdx.x >> vt_shift, d0 = slice * R;
  const bool has_column = v0 + col < vdim;
  // A sequence of more than chunks.rows rows is walked in chunks side by side: the first from the slot's state, the others
  // from nothing; a chunk leaves its last state, the product of its decays and, row by row, its queries times the decays up
  // to that row, from which gla_combine and chunk_carry make up what the later chunks' rows owe the state they started from.
  const int seq_first = seq_start[seq], seq_stop = seq_start[seq + 1];
  const int in_chunks = chunks.rows > 0 ? (seq_stop - seq_first + chunks.rows - 1) / chunks.rows : 1;      // chunks this sequence has
  const int start = seq_first + chunk * chunks.rows;
  const int stop = (chunks.rows > 0 && start + chunks.rows < seq_stop) ? start + chunks.rows : seq_stop;
  if (chunk > 0 && chunk >= in_chunks) return;      // a shorter sequence has fewer chunks
  const bool apart = in_chunks > 1;
  float* mine = apart ? chunks.states + ((size_t)(seq * chunks.count + chunk) * H + head) * dim * vdim + v0 + col
                      : state + (size_t)seq_to[seq] * slot_stride + (size_t)head * dim * vdim + v0 + col;
  const float* from = state + (size_t)seq_slot[seq] * slot_stride + (size_t)head * dim * vdim + v0 + col;
  float S[R];
#pragma unroll
  for (int r = 0; r < R; ++r) S[r] = (chunk == 0 && has_column && d0 + r < dim) ? from[(size_t)(d0 + r) * vdim] : 0.f;
  auto decay_of = [&](float x) { return RULE == RULE_WKV ? expf(-expf(x)) : expf(log_sigmoid_f32(x) * inv_tau); };
  float kept[GLA_KEPT];      // the decays' products so far, of key channels threadIdx.x, + 256, ... (first tile's workgroup only)
#pragma unroll
  for (int j = 0; j < GLA_KEPT; ++j) kept[j] = 1.0f;
  const bool keeps = apart && blockIdx.z == 0;
  const int width = H * vdim;
  float ahead_z[GLA_AHEAD], ahead_k[GLA_AHEAD], ahead_q[GLA_AHEAD], ahead_v[GLA_AHEAD];
  // a stage's element e of the decays, keys and queries is (row e / DP, key channel e % DP); of the values (row e / VT, column e % VT)
  auto ask = [&](int row0, int n) {
#pragma unroll
    for (int i = 0; i < GLA_AHEAD; ++i) {
      const int e = threadIdx.x + 256 * i, t = e >> dp_shift, d = e & (DP - 1);
      ahead_z[i] = ahead_k[i] = ahead_q[i] = ahead_v[i] = 0.f;
      if (e < n * DP && d < dim) {
        const size_t at = (size_t)(row0 + t) * row_stride + head * dim + d;
        ahead_z[i] = z[(size_t)(row0 + t) * z_stride + head * dim + d] + bias[head * dim + d];
        ahead_k[i] = to_f32(k[at]);
        ahead_q[i] = to_f32(q[at]);
      }
      const int tv = e >> vt_shift, c = e & (VT - 1);
      if (e < n * VT && v0 + c < vdim) ahead_v[i] = to_f32(v[(size_t)(row0 + tv) * row_stride + head * vdim + v0 + c]);
    }
  };
  if (start < stop) ask(start, stop - start < GLA_STAGE ? stop - start : GLA_STAGE);
  for (int row0 = start; row0 < stop; row0 += GLA_STAGE) {
    const int n = stop - row0 < GLA_STAGE ? stop - row0 : GLA_STAGE;
#pragma unroll
    for (int i = 0; i < GLA_AHEAD; ++i) {
      const int e = threadIdx.x + 256 * i;
      if (e < n * DP) {
        const bool real = (e & (DP - 1)) < dim;
        a_s[e] = real ? decay_of(ahead_z[i]) : 0.f;
        k_s[e] = ahead_k[i];
        q_s[e] = ahead_q[i] * q_scale;
      }
      if (e < n * VT) v_s[e] = ahead_v[i];
    }
    for (int e = threadIdx.x + 256 * GLA_AHEAD; e < n * DP; e += 256) {      // wide heads: what the registers did not hold
      const int t = e >> dp_shift, d = e & (DP - 1);
      float a = 0.f, kk = 0.f, qq = 0.f;
      if (d < dim) {
        const size_t at = (size_t)(row0 + t) * row_stride + head * dim + d;
        a = decay_of(z[(size_t)(row0 + t) * z_stride + head * dim + d] + bias[head * dim + d]);
        kk = to_f32(k[at]);
        qq = to_f32(q[at]) * q_scale;
      }
      a_s[e] = a;
      k_s[e] = kk;
      q_s[e] = qq;
    }
    lds_barrier();
    if (row0 + GLA_STAGE < stop) ask(row0 + GLA_STAGE, stop - row0 - GLA_STAGE < GLA_STAGE ? stop - row0 - GLA_STAGE : GLA_STAGE);
    if constexpr (RULE == RULE_WKV) {      // sixteen threads a row
      const int t = threadIdx.x / 16, at = threadIdx.x % 16;
      float own = 0.f;
      if (t < n)
#pragma unroll 1
        for (int d = at; d < dim; d += 16) own = fmaf(q_s[t * DP + d] * bonus[head * dim + d], k_s[t * DP + d], own);
#pragma unroll
      for (int off = 8; off > 0; off >>= 1) own += __shfl_xor(own, off, BH_WAVE);
      if (at == 0) own_s[t] = own;
    }
    if (keeps) {
#pragma unroll
      for (int j = 0; j < GLA_KEPT; ++j) {
        const int d = threadIdx.x + 256 * j;
        if (d >= dim) break;
        for (int t = 0; t < n; ++t) {
          const float before = kept[j];
          kept[j] *= a_s[t * DP + d];
          if (chunk > 0) chunks.queries[(size_t)(row0 + t) * H * dim + head * dim + d] = (RULE == RULE_WKV ? before : kept[j]) * q_s[t * DP + d];
        }
      }
    }
    // GLA_GROUP rows at a time: their operands are read from LDS with no store in between (the compiler may ask for all of
    // them at once), the slices of a wave add their shares up by lane exchanges, and one lane a column and wave stores them
#pragma unroll 1
    for (int t0 = 0; t0 < n; t0 += GROUP) {
      float acc[GROUP];
#pragma unroll
      for (int j = 0; j < GROUP; ++j) {
        const int t = t0 + j < n ? t0 + j : n - 1;      // a row beyond the last is walked on a copy of the state and dropped
        const float vv = v_s[t * VT + col];
        const float* a_row = a_s + t * DP + d0;
        const float* k_row = k_s + t * DP + d0;
        const float* q_row = q_s + t * DP + d0;
        const bool real = t0 + j < n;
        float sum = 0.f;
        if (R % 4 == 0) {
#pragma unroll
          for (int r = 0; r < R; r += 4) {
            const float4 a4 = *reinterpret_cast<const float4*>(a_row + r), k4 = *reinterpret_cast<const float4*>(k_row + r),
                         q4 = *reinterpret_cast<const float4*>(q_row + r);
            const float w0 = k4.x * vv, w1 = k4.y * vv, w2 = k4.z * vv, w3 = k4.w * vv;
            const float s0 = fmaf(a4.x, S[r], w0), s1 = fmaf(a4.y, S[r + 1], w1);
            const float s2 = fmaf(a4.z, S[r + 2], w2), s3 = fmaf(a4.w, S[r + 3], w3);
            sum = fmaf(RULE == RULE_WKV ? S[r] : s0, q4.x, sum);
            sum = fmaf(RULE == RULE_WKV ? S[r + 1] : s1, q4.y, sum);
            sum = fmaf(RULE == RULE_WKV ? S[r + 2] : s2, q4.z, sum);
            sum = fmaf(RULE == RULE_WKV ? S[r + 3] : s3, q4.w, sum);
            if (real) S[r] = s0, S[r + 1] = s1, S[r + 2] = s2, S[r + 3] = s3;
          }
        } else {
#pragma unroll
          for (int r = 0; r < R; ++r) {
            const float w0 = k_row[r] * vv;
            const float s0 = fmaf(a_row[r], S[r], w0);
            sum = fmaf(RULE == RULE_WKV ? S[r] : s0, q_row[r], sum);
            if (real) S[r] = s0;
          }
        }
        acc[j] = sum;
      }
      for (int off = VT; off < BH_WAVE; off <<= 1) {
#pragma unroll
        for (int j = 0; j < GROUP; ++j) acc[j] += __shfl_xor(acc[j], off, BH_WAVE);
      }
      if ((threadIdx.x % BH_WAVE) < VT || VT >= BH_WAVE) {
        const int share = VT >= BH_WAVE ? slice : threadIdx.x / BH_WAVE;
#pragma unroll
        for (int j = 0; j < GROUP; ++j)
          if (t0 + j < n) part[((t0 + j) * PARTS + share) * VT + col] = acc[j];
      }
    }
    lds_barrier();
    for (int e = threadIdx.x; e < n * VT; e += 256) {
      const int t = e >> vt_shift, c = e & (VT - 1);
      if (v0 + c >= vdim) continue;
      float total = 0.f;
      for (int s = 0; s < PARTS; ++s) total += part[(t * PARTS + s) * VT + c];
      if constexpr (RULE == RULE_WKV) total = fmaf(own_s[t], v_s[t * VT + c], total);
      out[(size_t)(row0 + t) * width + head * vdim + v0 + c] = total;
    }
    lds_barrier();      // the stage's LDS is written again
  }
#pragma unroll
  for (int r = 0; r < R; ++r)
    if (has_column && d0 + r < dim) mine[(size_t)(d0 + r) * vdim] = S[r];
  if (keeps) {
#pragma unroll
    for (int j = 0; j < GLA_KEPT; ++j) {
      const int d = threadIdx.x + 256 * j;
      if (d < dim) chunks.decays[((size_t)(seq * chunks.count + chunk) * H + head) * dim + d] = kept[j];
    }
  }
}

// The same walk for steps with many rows a sequence and rows of whole pieces of four: a thread keeps 16 elements of each of C columns, the SL
// threads of a column are neighbouring lanes (elements in turns of four: slice, slice + SL, ...) and add their shares by data-parallel
// moves.  What a row's decays, keys and queries cost in LDS reads, which bound the walk above, is shared by C columns, and no shares
// go through LDS.  The first tile's workgroup makes the carried queries, a thread a key channel.  Bound by the multiplications (three an
// element of the state and row, packed ones are not used) and, at one wave a SIMD, by a row's chain of them.  With the joining of the chunks, us:
// wkv, 64 heads of 64, 2,048 rows 273 -> 128; eight prompts of 512 rows, 32 heads 271 -> 126; gla, 8 heads of 128, 2,048 rows 109 -> 86,
// 16 heads of 256, 1,000 rows 1,275 -> 286.  Four columns a thread: 154, 165, 103, 334.
#define GC_R 16
template <typename T, int SL, int C, int WAVES, int RULE>
__global__ __launch_bounds__(WAVES * BH_WAVE) void gla_columns_kernel(const T* __restrict__ q, const T* __restrict__ k, const T* __restrict__ v, int row_stride,
                                                                      const float* __restrict__ z, int z_stride, const float* __restrict__ bias,
                                                                      float inv_tau, const float* __restrict__ bonus, float q_scale,
                                                                      float* __restrict__ state, long slot_stride, const int32_t* __restrict__ seq_start,
                                                                      const int32_t* __restrict__ seq_slot, const int32_t* __restrict__ seq_to,
                                                                      float* __restrict__ out, int H, int dim, int vdim, GlaChunks chunks) {
  constexpr int DP = GC_R * SL, PIECES = DP / 4, PER_WAVE = BH_WAVE / SL * C, COLS = WAVES * PER_WAVE, THREADS = WAVES * BH_WAVE;
  constexpr int EACH = GLA_STAGE * PIECES / THREADS, V_PIECES = GLA_STAGE * COLS / 4, V_EACH = (V_PIECES + THREADS - 1) / THREADS;
  constexpr int KEPT = (DP + THREADS - 1) / THREADS;
  static_assert(EACH * THREADS == GLA_STAGE * PIECES && THREADS % PIECES == 0, "a thread's pieces are of the same key channels");
  __shared__ float4 a_s[GLA_STAGE * PIECES], k_s[GLA_STAGE * PIECES], q_s[GLA_STAGE * PIECES];
  __shared__ float4 v_s[V_PIECES];
  __shared__ float own_s[GLA_STAGE];
  const int seq = blockIdx.x / chunks.count, chunk = blockIdx.x % chunks.count, head = blockIdx.y, v0 = blockIdx.z * COLS;
  const int seq_first = seq_start[seq], seq_stop = seq_start[seq + 1];
  const int in_chunks = chunks.rows > 0 ? (seq_stop - seq_first + chunks.rows - 1) / chunks.rows : 1;
  const int start = seq_first + chunk * chunks.rows;
  const int stop = (chunks.rows > 0 && start + chunks.rows < seq_stop) ? start + chunks.rows : seq_stop;
  if (chunk > 0 && chunk >= in_chunks) return;
  const bool apart = in_chunks > 1, keeps = apart && blockIdx.z == 0;
  const int lane = threadIdx.x % BH_WAVE, slice = lane % SL, local = threadIdx.x / BH_WAVE * PER_WAVE + lane / SL * C, column0 = v0 + local;
  const bool has_columns = column0 < vdim;      // (all C of them: vdim is a multiple)
  float* mine = apart ? chunks.states + ((size_t)(seq * chunks.count + chunk) * H + head) * dim * vdim
                      : state + (size_t)seq_to[seq] * slot_stride + (size_t)head * dim * vdim;
  const float* from = state + (size_t)seq_slot[seq] * slot_stride + (size_t)head * dim * vdim;
  float S[C][GC_R];
#pragma unroll
  for (int r = 0; r < GC_R; ++r) {
    const int d = 4 * (slice + SL * (r / 4)) + r % 4;
#pragma unroll
    for (int c = 0; c < C; ++c) S[c][r] = chunk == 0 && has_columns && d < dim ? from[(size_t)d * vdim + column0 + c] : 0.f;
  }
  auto decay_of = [&](float x) { return RULE == RULE_WKV ? expf(-expf(x)) : expf(log_sigmoid_f32(x) * inv_tau); };
  float kept[KEPT];
#pragma unroll
  for (int j = 0; j < KEPT; ++j) kept[j] = 1.0f;
  const float4 zero = make_float4(0.f, 0.f, 0.f, 0.f);
  const int my_d = threadIdx.x % PIECES * 4, my_t = threadIdx.x / PIECES;      // of a thread's pieces: key channels, and row of the first
  const bool real = my_d < dim;
  const float4 bias4 = real ? load_four(bias + head * dim + my_d) : zero;
  const float4 bonus4 = RULE == RULE_WKV && real ? load_four(bonus + head * dim + my_d) : zero;
  float4 z_ahead[EACH], k_ahead[EACH], q_ahead[EACH], v_ahead[V_EACH];
  auto ask = [&](int row0) {
#pragma unroll
    for (int i = 0; i < EACH; ++i) {
      const int row = row0 + my_t + i * (THREADS / PIECES);
      z_ahead[i] = k_ahead[i] = q_ahead[i] = zero;
      if (real && row < stop) {
        const size_t at = (size_t)row * row_stride + head * dim + my_d;
        z_ahead[i] = load_four(z + (size_t)row * z_stride + head * dim + my_d);
        k_ahead[i] = load_four(k + at);
        q_ahead[i] = load_four(q + at);
      }
    }
#pragma unroll
    for (int i = 0; i < V_EACH; ++i) {
      const int e = threadIdx.x + THREADS * i, row = row0 + e / (COLS / 4), c = v0 + e % (COLS / 4) * 4;
      v_ahead[i] = e < V_PIECES && row < stop && c < vdim ? load_four(v + (size_t)row * row_stride + head * vdim + c) : zero;
    }
  };
  ask(start);
  for (int row0 = start; row0 < stop; row0 += GLA_STAGE) {
    const int n = stop - row0 < GLA_STAGE ? stop - row0 : GLA_STAGE;
#pragma unroll
    for (int i = 0; i < EACH; ++i) {
      const float4 x = z_ahead[i], kk = k_ahead[i];
      float4 qq = q_ahead[i];
      qq.x *= q_scale, qq.y *= q_scale, qq.z *= q_scale, qq.w *= q_scale;
      const int e = threadIdx.x + THREADS * i;
      a_s[e] = real ? make_float4(decay_of(x.x + bias4.x), decay_of(x.y + bias4.y), decay_of(x.z + bias4.z), decay_of(x.w + bias4.w)) : zero;
      k_s[e] = kk;
      q_s[e] = qq;
      if constexpr (RULE == RULE_WKV) {
        float own = fmaf(qq.x * bonus4.x, kk.x, fmaf(qq.y * bonus4.y, kk.y, fmaf(qq.z * bonus4.z, kk.z, qq.w * bonus4.w * kk.w)));
#pragma unroll
        for (int off = PIECES / 2; off > 0; off >>= 1) own += __shfl_xor(own, off, BH_WAVE);
        if (my_d == 0) own_s[my_t + i * (THREADS / PIECES)] = own;
      }
    }
#pragma unroll
    for (int i = 0; i < V_EACH; ++i)
      if (threadIdx.x + THREADS * i < V_PIECES) v_s[threadIdx.x + THREADS * i] = v_ahead[i];
    lds_barrier();
    if (row0 + GLA_STAGE < stop) ask(row0 + GLA_STAGE);
    if (keeps) {
      const float* decays = reinterpret_cast<const float*>(a_s);
      const float* queries = reinterpret_cast<const float*>(q_s);
#pragma unroll
      for (int j = 0; j < KEPT; ++j) {
        const int d = threadIdx.x + THREADS * j;
        if (d >= dim) break;
        float a[GLA_STAGE], x[GLA_STAGE];
#pragma unroll
        for (int t = 0; t < GLA_STAGE; ++t) a[t] = decays[t * DP + d], x[t] = queries[t * DP + d];
#pragma unroll
        for (int t = 0; t < GLA_STAGE; ++t) {
          if (t >= n) break;
          const float before = kept[j];
          kept[j] *= a[t];
          if (chunk > 0) chunks.queries[((size_t)(row0 + t) * H + head) * dim + d] = (RULE == RULE_WKV ? before : kept[j]) * x[t];
        }
      }
    }
    float o_kept[C];
#pragma unroll
    for (int c = 0; c < C; ++c) o_kept[c] = 0.f;
    // a row's operands are asked for while the row before is walked
    struct Row {
      float4 a[GC_R / 4], k[GC_R / 4], q[GC_R / 4];
      float v[C], own;
    };
    auto fetch = [&](Row& row, int t) {
      t = t < GLA_STAGE ? t : GLA_STAGE - 1;
#pragma unroll
      for (int i = 0; i < GC_R / 4; ++i) {
        const int at = t * PIECES + slice + SL * i;
        row.a[i] = a_s[at], row.k[i] = k_s[at], row.q[i] = q_s[at];
      }
#pragma unroll
      for (int c = 0; c < C; ++c) row.v[c] = reinterpret_cast<const float*>(v_s)[t * COLS + local + c];
      row.own = RULE == RULE_WKV ? own_s[t] : 0.f;
    };
    auto walk = [&](const Row& row, int t) {
      float sum[C][2];
#pragma unroll
      for (int c = 0; c < C; ++c) sum[c][0] = sum[c][1] = 0.f;
#pragma unroll
      for (int i = 0; i < GC_R / 4; ++i) {
        const float a4[4] = {row.a[i].x, row.a[i].y, row.a[i].z, row.a[i].w}, k4[4] = {row.k[i].x, row.k[i].y, row.k[i].z, row.k[i].w};
        const float q4[4] = {row.q[i].x, row.q[i].y, row.q[i].z, row.q[i].w};
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
          for (int c = 0; c < C; ++c) {
            float& s = S[c][4 * i + r];
            if (RULE == RULE_WKV) sum[c][r & 1] = fmaf(s, q4[r], sum[c][r & 1]);
            s *= a4[r];
            s = fmaf(k4[r], row.v[c], s);
            if (RULE == RULE_GLA) sum[c][r & 1] = fmaf(s, q4[r], sum[c][r & 1]);
          }
      }
#pragma unroll
      for (int c = 0; c < C; ++c) {
        float o = slices_sum<SL>(sum[c][0] + sum[c][1]);
        if constexpr (RULE == RULE_WKV) o = fmaf(row.own, row.v[c], o);
        if (slice == (t & (SL - 1))) o_kept[c] = o;
      }
      // every SL rows (and behind the last) each lane of a column writes the row it kept
      if ((t & (SL - 1)) == SL - 1 || t == n - 1) {
        const int kept_row = (t & ~(SL - 1)) + slice;
        if (kept_row <= t && has_columns) {
#pragma unroll
          for (int c = 0; c < C; ++c) out[(size_t)(row0 + kept_row) * H * vdim + head * vdim + column0 + c] = o_kept[c];
        }
      }
    };
    Row even, odd;
    fetch(even, 0);
#pragma unroll 1
    for (int t = 0; t < n; t += 2) {
      fetch(odd, t + 1);
      walk(even, t);
      if (t + 1 >= n) break;
      fetch(even, t + 2);
      walk(odd, t + 1);
    }
    lds_barrier();      // the stage's LDS is written again
  }
#pragma unroll
  for (int r = 0; r < GC_R; ++r) {
    const int d = 4 * (slice + SL * (r / 4)) + r % 4;
#pragma unroll
    for (int c = 0; c < C; ++c)
      if (has_columns && d < dim) mine[(size_t)d * vdim + column0 + c] = S[c][r];
  }
  if (keeps) {
#pragma unroll
    for (int j = 0; j < KEPT; ++j) {
      const int d = threadIdx.x + THREADS * j;
      if (d < dim) chunks.decays[((size_t)(seq * chunks.count + chunk) * H + head) * dim + d] = kept[j];
    }
  }
}

// One thread a state element (sequence, head, key channel, value column): through the sequence's chunks in order,
// S_in(c + 1) = A(c) S_in(c) + S_loc(c), A(c) the chunk's product of decays; a chunk's place in `states` then holds the state
// it started from (for chunk_carry), and the state after the last chunk goes to the sequence's slot.
__global__ __launch_bounds__(256) void gla_combine_kernel(GlaChunks chunks, float* __restrict__ state, long slot_stride,
                                                          const int32_t* __restrict__ seq_start, const int32_t* __restrict__ seq_slot, const int32_t* __restrict__ seq_to, int H,
                                                          int dim, int vdim) {
  const int seq = blockIdx.y;
  const size_t per = (size_t)H * dim * vdim, e = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (e >= per) return;
  const int in_chunks = (seq_start[seq + 1] - seq_start[seq] + chunks.rows - 1) / chunks.rows;
  if (in_chunks <= 1) return;      // the walk itself wrote the slot
  const size_t channel = e / vdim;      // (head, key channel)
  float run = 0.f;
  for (int c = 0; c < in_chunks; ++c) {
    float* place = chunks.states + (size_t)(seq * chunks.count + c) * per + e;
    const float local = *place;
    *place = run;
    run = c == 0 ? local : fmaf(chunks.decays[(size_t)(seq * chunks.count + c) * H * dim + channel], run, local);
  }
  state[(size_t)seq_to[seq] * slot_stride + e] = run;
}

// out[row] += (carried query of the row) . S_in(the row's chunk), for the rows of every chunk but a sequence's first, on the float32
// matrix instructions: a workgroup takes a (sequence, chunk, head, 64 value columns, 64 rows), a wave 16 of the rows as v_mfma_f32_16x16x4_f32
// tiles.  64 key channels of the state's columns go through LDS at a time (rows of 68: the four rows that a wave reads at once lie in
// other banks); a lane takes its row's queries as 16-byte pieces, four neighbouring key channels at a time.
typedef float carry_f32x4_t __attribute__((ext_vector_type(4)));
#define CARRY_STRIDE 68
__global__ __launch_bounds__(256) void chunk_carry_kernel(const float* __restrict__ states, const float* __restrict__ queries, int chunk_rows,
                                                          int chunk_count, const int32_t* __restrict__ seq_start, float* __restrict__ out, int H,
                                                          int dim, int vdim, int v_tiles) {
  __shared__ float s_tile[64 * CARRY_STRIDE];
  const int seq = blockIdx.x / chunk_count, chunk = blockIdx.x % chunk_count, head = blockIdx.y, v0 = blockIdx.z % v_tiles * 64;
  if (chunk == 0) return;
  const int first = seq_start[seq] + chunk * chunk_rows, seq_stop = seq_start[seq + 1], row0 = first + blockIdx.z / v_tiles * 64;
  const int stop = first + chunk_rows < seq_stop ? first + chunk_rows : seq_stop;
  if (row0 >= stop) return;
  const int wave = threadIdx.x / BH_WAVE, lane = threadIdx.x % BH_WAVE, j = lane % 16, g = lane / 16;
  const float* began = states + ((size_t)(seq * chunk_count + chunk) * H + head) * dim * vdim;
  const int my_row = row0 + wave * 16 + j;
  const float* query = queries + ((size_t)(my_row < stop ? my_row : stop - 1) * H + head) * dim;
  const bool whole = dim % 4 == 0;
  carry_f32x4_t acc[4];
#pragma unroll
  for (int ct = 0; ct < 4; ++ct) acc[ct] = carry_f32x4_t{0.f, 0.f, 0.f, 0.f};
  for (int dd = 0; dd < dim; dd += 64) {
    float q[4][4];
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      const int d = dd + 16 * b + 4 * g;
      if (whole && d < dim) {
        const float4 x = *reinterpret_cast<const float4*>(query + d);
        q[b][0] = x.x, q[b][1] = x.y, q[b][2] = x.z, q[b][3] = x.w;
      } else {
#pragma unroll
        for (int s = 0; s < 4; ++s) q[b][s] = d + s < dim ? query[d + s] : 0.f;
      }
    }
    __syncthreads();      // the tile is written again
    for (int e = threadIdx.x; e < 64 * 64; e += 256) {
      const int a = e >> 6, b = e & 63;
      s_tile[a * CARRY_STRIDE + b] = (dd + a < dim && v0 + b < vdim) ? began[(size_t)(dd + a) * vdim + v0 + b] : 0.f;
    }
    __syncthreads();
#pragma unroll
    for (int b = 0; b < 4; ++b)
#pragma unroll
      for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int ct = 0; ct < 4; ++ct)
          acc[ct] = __builtin_amdgcn_mfma_f32_16x16x4f32(q[b][s], s_tile[(16 * b + 4 * g + s) * CARRY_STRIDE + 16 * ct + j], acc[ct], 0, 0, 0);
  }
#pragma unroll
  for (int ct = 0; ct < 4; ++ct)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int row = row0 + wave * 16 + 4 * g + r, column = v0 + 16 * ct + j;
      if (row < stop && column < vdim) out[(size_t)row * H * vdim + head * vdim + column] += acc[ct][r];
    }
}

int bh_chunk_carry(const float* states, const float* queries, int chunk_rows, int chunk_count, const int32_t* seq_start, float* out, int n_seqs,
                   int H, int dim, int vdim, hipStream_t stream) {
  const int v_tiles = (vdim + 63) / 64, row_tiles = (chunk_rows + 63) / 64;
  BH_REQUIRE((long)v_tiles * row_tiles <= 65535, "chunk_carry: chunks of %d rows and heads of %d values are too many tiles", chunk_rows, vdim);
  chunk_carry_kernel<<<dim3(n_seqs * chunk_count, H, v_tiles * row_tiles), 256, 0, stream>>>(states, queries, chunk_rows, chunk_count, seq_start, out,
                                                                                           H, dim, vdim, v_tiles);
  return bh_check_launch("chunk_carry");
}

// How many value columns a workgroup takes for a step of these sizes.  A stage costs a workgroup about as many instructions
// whatever its tile (the staging of decays, keys and queries is the same for every tile of a head), so narrow tiles multiply
// the work: they pay only while they bring idle compute units in, up to about one workgroup a unit; and never so narrow that
// a thread's slice of a state column exceeds 64 rows.
static int gla_tile(long walks, int H, int dim, int vdim) {
  int tile = 64;
  while (tile > 8 && (tile / 2 >= vdim || walks * H * ((vdim + tile - 1) / tile) < (long)bh_compute_units())) tile /= 2;
  while (tile > 8 && (dim + 256 / tile - 1) / (256 / tile) > 64) tile /= 2;
  return tile;
}

// Rows of a chunk for a step whose longest sequence brings max_rows rows: a walk over a sequence is a chain of stages that one
// workgroup runs at one wave a SIMD, so long sequences are cut until about four workgroups stand on every compute unit, in
// chunks of whole stages and no fewer than 64 rows; max_rows and more: the sequences are walked whole.
extern "C" int bh_gla_chunk_rows(int n_seqs, int max_rows, int H, int dim, int vdim) {
  if (max_rows < 128 || dim > 256 * GLA_KEPT) return max_rows;
  const long whole = (long)n_seqs * H * ((vdim + 63) / 64);
  long wanted = (4L * bh_compute_units() + whole - 1) / whole;
  if (wanted <= 1) return max_rows;
  if (wanted > max_rows / 64) wanted = max_rows / 64;
  int rows = (int)((max_rows + wanted - 1) / wanted);
  rows = (rows + GLA_STAGE - 1) / GLA_STAGE * GLA_STAGE;
  return rows >= max_rows ? max_rows : rows;
}

// Chunks of all sequences together, at most, over the steps of up to n_seqs sequences, n_rows rows and max_rows rows a sequence (0: no such
// step is cut): fewer sequences are cut into more chunks each.
extern "C" long bh_gla_most_chunks(int n_seqs, int n_rows, int max_rows, int H, int dim, int vdim) {
  if (dim > 256 * GLA_KEPT) return 0;
  const long enough = 4L * bh_compute_units(), tiles = (vdim + 63) / 64;
  long most = 0;
  for (long n = 1; n <= n_seqs && n * H * tiles < enough; ++n) {
    const long longest = n_rows - n + 1 < max_rows ? n_rows - n + 1 : max_rows;      // the other sequences bring a row each
    if (longest < 128) break;
    const long wanted = (enough + n * H * tiles - 1) / (n * H * tiles), pieces = longest / 64;
    most = n * (wanted < pieces ? wanted : pieces) > most ? n * (wanted < pieces ? wanted : pieces) : most;
  }
  return most;
}

// The chunks' states joined, and what the later chunks' rows owe them.
static int gla_join(const GlaChunks& chunks, float* state, long slot_stride, const int32_t* seq_start, const int32_t* seq_slot, const int32_t* seq_to,
                    float* out, int n_seqs, int H, int dim, int vdim, hipStream_t stream) {
  if (chunks.rows == 0) return 0;
  const size_t per = (size_t)H * dim * vdim;
  gla_combine_kernel<<<dim3((unsigned)((per + 255) / 256), n_seqs), 256, 0, stream>>>(chunks, state, slot_stride, seq_start, seq_slot, seq_to, H, dim, vdim);
  if (int status = bh_check_launch("gla_combine")) return status;
  return bh_chunk_carry(chunks.states, chunks.queries, chunks.rows, chunks.count, seq_start, out, n_seqs, H, dim, vdim, stream);
}

// Which steps share what is read between columns: long walks (a decode step is its state's way in and out) of which a compute unit has one at
// least; below that a row's chain of steps is the time, and that of 16 elements a thread is the longer one (wkv, 64 heads of 64, 2,048 rows, us,
// apart / in columns: 1,024 workgroups 273 / 128, 512 workgroups 266 / 195; one sequence of 100 rows, 64 heads, 64 workgroups 64 / 62; 32
// heads, 128 workgroups 293 / 306; gla, 8 heads of 128, 64 workgroups 321 / 314; 20 heads of 48, 333 rows, 100 workgroups 59 / 70).  At the line, 256
// workgroups, sequences of 64 / of 127 rows: wkv, 4 of 64 heads of 64 50.2 / 36.0 and 93.5 / 63.6, gla the same 40.4 / 39.6 and 77.0 / 71.4, 8 of 16 heads
// of 128 62.9 / 42.5 and 122.0 / 77.2; but gla, 8 of 64 heads of 64, 64 rows, 512 workgroups 50.1 / 52.0.
#define GC_ROWS 64
#define GC_C 2
static bool gla_columns_take(long walks, int max_rows, int H, int dim, int vdim) {
  return max_rows >= GC_ROWS && dim % 4 == 0 && dim > 32 && dim <= 256 && vdim % 4 == 0 && vdim > 32 &&
         walks * H * ((vdim + 63) / 64) >= (long)bh_compute_units();
}

// For tests: whether a step of operands on 16 bytes, in rows of whole pieces of four, is walked in columns.
extern "C" int bh_gla_in_columns(int n_seqs, int max_rows, int H, int dim, int vdim) {
  const int rows = bh_gla_chunk_rows(n_seqs, max_rows, H, dim, vdim);
  return gla_columns_take((long)n_seqs * ((max_rows + rows - 1) / rows), max_rows, H, dim, vdim);
}

template <int RULE, typename T>
static void gla_columns(const T* q, const T* k, const T* v, int row_stride, const float* z, int z_stride, const float* bias, float inv_tau,
                        const float* bonus, float q_scale, float* state, long slot_stride, const int32_t* seq_start, const int32_t* seq_slot,
                        const int32_t* seq_to, float* out, int n_seqs, int H, int dim, int vdim, const GlaChunks& chunks, hipStream_t stream) {
#define BH_GC(SL, WAVES)                                                                                                                \
  do {                                                                                                                                  \
    static_assert((WAVES) * (BH_WAVE / (SL)) * GC_C == 64, "a tile is 64 columns");                                                     \
    gla_columns_kernel<T, SL, GC_C, WAVES, RULE><<<dim3(n_seqs * chunks.count, H, (vdim + 63) / 64), (WAVES) * BH_WAVE, 0, stream>>>(   \
        q, k, v, row_stride, z, z_stride, bias, inv_tau, bonus, q_scale, state, slot_stride, seq_start, seq_slot, seq_to, out, H, dim, vdim, \
        chunks);                                                                                                                        \
  } while (0)
  if (dim <= 64) BH_GC(4, 2);
  else if (dim <= 128) BH_GC(8, 4);
  else BH_GC(16, 8);
#undef BH_GC
}

// What both rules' entry points share.  q, k [rows][row_stride] (dtype): H heads of `dim` from a row's start; v: H heads of vdim.
template <int RULE>
static int scan_run(const char* what, const void* q, const void* k, const void* v, int dtype, int row_stride, const float* z, int z_stride,
                    const float* bias, float inv_tau, const float* bonus, float q_scale, float* state, long slot_stride,
                    const int32_t* seq_start, const int32_t* seq_slot, const int32_t* seq_to, float* out, int n_seqs, int H, int dim, int vdim, int n_rows,
                    int max_rows, int chunk_rows, float* scratch, hipStream_t stream) {
  BH_REQUIRE(n_seqs > 0 && H > 0 && dim > 0 && vdim > 0, "%s: sizes must be positive", what);
  BH_REQUIRE(z_stride >= H * dim, "%s: the decays' rows hold %d numbers, %d are needed", what, z_stride, H * dim);
  BH_REQUIRE(slot_stride >= (long)H * dim * vdim, "%s: a slot's state is smaller than the heads' states", what);
  BH_REQUIRE(H <= 65535 && (vdim + 7) / 8 <= 65535, "%s: too many heads or value columns", what);
  BH_REQUIRE(max_rows > 0 && n_rows >= n_seqs && chunk_rows > 0, "%s: a step has rows, and chunks have rows", what);
  GlaChunks chunks = {0, 1, nullptr, nullptr, nullptr};
  if (chunk_rows < max_rows) {
    BH_REQUIRE(scratch != nullptr && chunk_rows % GLA_STAGE == 0 && dim <= 256 * GLA_KEPT, "%s: chunks need scratch memory and whole stages", what);
    chunks.rows = chunk_rows;
    chunks.count = (max_rows + chunk_rows - 1) / chunk_rows;
    chunks.states = scratch;
    chunks.decays = chunks.states + (size_t)n_seqs * chunks.count * H * dim * vdim;
    chunks.queries = chunks.decays + (size_t)n_seqs * chunks.count * H * dim;
  }
  BH_REQUIRE((long)n_seqs * chunks.count < (1L << 31), "%s: too many chunks", what);
  const size_t piece = 4 * (dtype == BH_F32 ? sizeof(float) : 2);
  const bool in_columns = gla_columns_take((long)n_seqs * chunks.count, max_rows, H, dim, vdim) && row_stride % 4 == 0 && z_stride % 4 == 0 &&
                          ((uintptr_t)q | (uintptr_t)k | (uintptr_t)v) % piece == 0 && ((uintptr_t)z | (uintptr_t)bias | (uintptr_t)bonus) % 16 == 0;
  if (in_columns) {
    if (dtype == BH_F32) gla_columns<RULE>((const float*)q, (const float*)k, (const float*)v, row_stride, z, z_stride, bias, inv_tau, bonus, q_scale, state,
                                           slot_stride, seq_start, seq_slot, seq_to, out, n_seqs, H, dim, vdim, chunks, stream);
    else if (dtype == BH_BF16) gla_columns<RULE>((const bf16_t*)q, (const bf16_t*)k, (const bf16_t*)v, row_stride, z, z_stride, bias, inv_tau, bonus, q_scale,
                                                 state, slot_stride, seq_start, seq_slot, seq_to, out, n_seqs, H, dim, vdim, chunks, stream);
    else return bh_fail("%s: unknown dtype %d", what, dtype);
    if (int status = bh_check_launch(what)) return status;
    return gla_join(chunks, state, slot_stride, seq_start, seq_slot, seq_to, out, n_seqs, H, dim, vdim, stream);
  }
  const int VT = gla_tile((long)n_seqs * chunks.count, H, dim, vdim), SL = 256 / VT;
  int R = 1;
  while (R * SL < dim) R *= 2;
  BH_REQUIRE(R <= 64, "%s: heads of %d key dimensions are above the limit of %d", what, dim, 64 * 32);
  const size_t lds = (size_t)GLA_STAGE * (3 * SL * R + VT + 256) * sizeof(float);
  BH_REQUIRE(lds <= 160 * 1024, "%s: heads of %d key dimensions do not fit the local memory", what, dim);
  const dim3 grid(n_seqs * chunks.count, H, (vdim + VT - 1) / VT);
#define BH_GLA(T, RR)                                                                                                        \
  do {                                                                                                                       \
    bh_allow_lds<gla_scan_kernel<T, RR, RULE>>(lds);                                                                         \
    gla_scan_kernel<T, RR, RULE><<<grid, 256, lds, stream>>>((const T*)q, (const T*)k, (const T*)v, row_stride, z, z_stride, bias, \
                                                             inv_tau, bonus, q_scale, state, slot_stride, seq_start, seq_slot, seq_to, out, \
                                                             H, dim, vdim, VT, chunks);                                      \
  } while (0)
#define BH_GLA_R(T)                  \
  switch (R) {                       \
    case 1: BH_GLA(T, 1); break;     \
    case 2: BH_GLA(T, 2); break;     \
    case 4: BH_GLA(T, 4); break;     \
    case 8: BH_GLA(T, 8); break;     \
    case 16: BH_GLA(T, 16); break;   \
    case 32: BH_GLA(T, 32); break;   \
    default: BH_GLA(T, 64); break;   \
  }
  if (dtype == BH_F32) BH_GLA_R(float)
  else if (dtype == BH_BF16) BH_GLA_R(bf16_t)
  else return bh_fail("%s: unknown dtype %d", what, dtype);
#undef BH_GLA_R
#undef BH_GLA
  if (int status = bh_check_launch(what)) return status;
  return gla_join(chunks, state, slot_stride, seq_start, seq_slot, seq_to, out, n_seqs, H, dim, vdim, stream);
}

// proj [rows][proj_stride] (dtype): a row holds H heads of q and of k (dim each) from q_off and k_off and H heads of v (vdim) from
// v_off.  z [rows][z_stride] float32: the decays' pre-activations, H x dim from column 0; bias [H * dim] float32.
// state [slots][slot_stride] float32, a slot's first H * dim * vdim floats being its heads' states; seq_start [n_seqs + 1],
// seq_slot [n_seqs]; out [rows][H * vdim] float32.  chunk_rows: bh_gla_chunk_rows' answer for the step (max_rows: its longest
// sequence's rows); where that is less than max_rows, scratch holds n_seqs * chunks * H * dim * (vdim + 1) + n_rows * H * dim floats.
extern "C" int bh_gla_scan(const void* proj, int dtype, int proj_stride, int q_off, int k_off, int v_off, const float* z, int z_stride,
                           const float* bias, float tau, float q_scale, float* state, long slot_stride, const int32_t* seq_start,
                           const int32_t* seq_slot, const int32_t* seq_to, float* out, int n_seqs, int H, int dim, int vdim, int n_rows, int max_rows,
                           int chunk_rows, float* scratch, hipStream_t stream) {
  BH_REQUIRE(tau > 0.f, "gla_scan: tau must be positive, got %f", (double)tau);
  BH_REQUIRE(q_off >= 0 && k_off >= 0 && v_off >= 0 && q_off + H * dim <= proj_stride && k_off + H * dim <= proj_stride &&
                 v_off + H * vdim <= proj_stride, "gla_scan: q, k or v lie outside a row of %d", proj_stride);
  const size_t element = dtype == BH_F32 ? 4 : 2;
  const char* rows = (const char*)proj;
  return scan_run<RULE_GLA>("gla_scan", rows + q_off * element, rows + k_off * element, rows + v_off * element, dtype, proj_stride, z, z_stride,
                            bias, 1.0f / tau, nullptr, q_scale, state, slot_stride, seq_start, seq_slot, seq_to, out, n_seqs, H, dim, vdim, n_rows,
                            max_rows, chunk_rows, scratch, stream);
}

// r, k [rows][row_stride] (dtype): H heads of `dim`; v: H heads of vdim; z, bias, state and the rest as above; bonus [H * dim] float32.
extern "C" int bh_wkv_scan(const void* r, const void* k, const void* v, int dtype, int row_stride, const float* z, int z_stride, const float* bias,
                           const float* bonus, float* state, long slot_stride, const int32_t* seq_start, const int32_t* seq_slot, const int32_t* seq_to, float* out,
                           int n_seqs, int H, int dim, int vdim, int n_rows, int max_rows, int chunk_rows, float* scratch, hipStream_t stream) {
  BH_REQUIRE(bonus != nullptr && H * dim <= row_stride && H * vdim <= row_stride, "wkv_scan: r, k or v lie outside a row of %d", row_stride);
  return scan_run<RULE_WKV>("wkv_scan", r, k, v, dtype, row_stride, z, z_stride, bias, 1.0f, bonus, 1.0f, state, slot_stride, seq_start, seq_slot, seq_to,
                            out, n_seqs, H, dim, vdim, n_rows, max_rows, chunk_rows, scratch, stream);
}
