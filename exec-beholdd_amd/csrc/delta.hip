// The gated delta rule, walked as a recurrence over a float32 matrix state S [dim][vdim] per (sequence, head):
//   q, k, v = silu(conv(.)) of the projected channels (a causal convolution over time on every channel, `taps` long);
//   q, k brought to unit length head by head, x / sqrt(sum x^2 + 1e-6), q then times dim^(-1/2);  H heads of v share G of q and k
//   beta = sigmoid(b),  g = exp(-exp(A_log) softplus(a + dt_bias))        one of each a head
//   S <- g S;   u = beta (v - S^T k);   S <- S + k u^T;   o = S^T q        (the read-out sees the token's own write)
//   delta_prep   convolution, activation, unit lengths, beta, g and k.q of every row
//   delta_scan   the recurrence over a sequence's rows of the step in order, from the state in row seq_slot, which it moves on into row
//                seq_to (the same one, or one that no sequence of the step starts from)
//   delta_step   all of it, the heads' norm and gate too, for a step of one row a sequence (a decode step), one launch
// A slot's state: H states [dim][vdim], then the last taps - 1 projected rows of (q | k | v), oldest first.  Everything is float32 but the
// projected rows, which come in the activation type.
#include "chunks.h"
#include "common.h"
#include <algorithm>
#include <cmath>

#define DR_UNIT_EPS 1e-6f
#define DR_MAX_TAPS 16
#define DR_BESIDE 4      // floats a row and head beside q, k and v: g, beta, k.q, one unused

__device__ inline float dr_softplus(float x) { return x > 20.f ? x : log1pf(expf(x)); }
__device__ inline float dr_silu(float x) { return x / (1.0f + expf(-x)); }

// What both kernels that begin with the projected rows know of them.
struct DeltaRows {
  int row_stride, first, b_first, a_first;      // columns: q, k, v from `first` on; the heads' b and a
  const float* conv;                            // [channels][taps]
  int taps;
  float* state;                                 // slots
  long slot_stride, conv_offset;                // a slot's conv inputs stand conv_offset floats into it
  const float* a_log;
  const float* dt_bias;
  int H, G, dim, vdim;
  __device__ inline int channels() const { return 2 * G * dim + H * vdim; }
};

// silu of the convolution on one channel; `row` is the t-th of its sequence's rows of this step
template <typename T>
__device__ inline float dr_convolved(const DeltaRows& in, const T* __restrict__ proj, const float* __restrict__ old, int row, int t, int c) {
  const float* w = in.conv + (size_t)c * in.taps;
  const int channels = in.channels();
  float acc = 0.f;
  for (int j = 0; j < in.taps; ++j) {
    const int back = in.taps - 1 - j;
    const float u = back <= t ? to_f32(proj[(size_t)(row - back) * in.row_stride + in.first + c]) : old[(size_t)(in.taps - 1 + t - back) * channels + c];
    acc = fmaf(w[j], u, acc);
  }
  return dr_silu(acc);
}

// ---- what the recurrence reads --------------------------------------------------------------------------------
// A workgroup a row and four units (grid.y), a wave a unit: G pairs of a query head and its key head, H heads of values, and one
// unit for the heads' g and beta.  A lane reads its own channels back between the sums and the scaling.
template <typename T>
__global__ __launch_bounds__(256) void delta_prep_kernel(const T* __restrict__ proj, DeltaRows in, const int32_t* __restrict__ row_seq,
                                                         const int32_t* __restrict__ seq_start, const int32_t* __restrict__ seq_slot,
                                                         float* __restrict__ qkv, float* __restrict__ beside) {
  const int row = blockIdx.x, unit = blockIdx.y * 4 + threadIdx.x / BH_WAVE, lane = threadIdx.x % BH_WAVE;
  const int seq = row_seq[row], t = row - seq_start[seq];
  const float* old = in.state + (size_t)seq_slot[seq] * in.slot_stride + in.conv_offset;
  float* mine = qkv + (size_t)row * in.channels();
  if (unit < in.G) {
    const int q0 = unit * in.dim, k0 = (in.G + unit) * in.dim;
    float qq = 0.f, kk = 0.f, qk = 0.f;
    for (int i = lane; i < in.dim; i += BH_WAVE) {
      const float q = dr_convolved(in, proj, old, row, t, q0 + i), k = dr_convolved(in, proj, old, row, t, k0 + i);
      mine[q0 + i] = q;
      mine[k0 + i] = k;
      qq += q * q;
      kk += k * k;
      qk += q * k;
    }
    const float q_scale = 1.0f / sqrtf(wave_sum(qq) + DR_UNIT_EPS) / sqrtf((float)in.dim), k_scale = 1.0f / sqrtf(wave_sum(kk) + DR_UNIT_EPS);
    qk = wave_sum(qk) * q_scale * k_scale;
    for (int i = lane; i < in.dim; i += BH_WAVE) {
      mine[q0 + i] *= q_scale;
      mine[k0 + i] *= k_scale;
    }
    const int per = in.H / in.G;
    for (int i = lane; i < per; i += BH_WAVE) beside[((size_t)row * in.H + unit * per + i) * DR_BESIDE + 2] = qk;
  } else if (unit < in.G + in.H) {
    const int v0 = 2 * in.G * in.dim + (unit - in.G) * in.vdim;
    for (int i = lane; i < in.vdim; i += BH_WAVE) mine[v0 + i] = dr_convolved(in, proj, old, row, t, v0 + i);
  } else if (unit == in.G + in.H) {
    const T* x = proj + (size_t)row * in.row_stride;
    for (int h = lane; h < in.H; h += BH_WAVE) {
      float* out = beside + ((size_t)row * in.H + h) * DR_BESIDE;
      out[0] = expf(-expf(in.a_log[h]) * dr_softplus(to_f32(x[in.a_first + h]) + in.dt_bias[h]));
      out[1] = 1.0f / (1.0f + expf(-to_f32(x[in.b_first + h])));
    }
  }
}

// The same for steps of many rows: a workgroup takes DP_ROWS rows and a unit, a pair of a query and a key head or a stretch of value channels;
// a thread walks down the rows of its channel with the last TAPS inputs in registers, so that every input is loaded once (where a
// sequence starts inside the stretch, the window is filled anew).  A pair's rows stand in LDS between the convolution and the scaling, a
// wave makes every fourth row's sums.  The gates have units of their own: a thread a (row, head).
#define DP_ROWS 32
#define DP_AHEAD 8
template <typename T, int TAPS>
__global__ __launch_bounds__(256) void delta_prep_walk_kernel(const T* __restrict__ proj, DeltaRows in, const int32_t* __restrict__ row_seq,
                                                              const int32_t* __restrict__ seq_start, const int32_t* __restrict__ seq_slot,
                                                              float* __restrict__ qkv, float* __restrict__ beside, int n_rows, int v_units) {
  extern __shared__ float pair[];      // [DP_ROWS][2 dim]
  const int row0 = blockIdx.x * DP_ROWS, stop = row0 + DP_ROWS < n_rows ? row0 + DP_ROWS : n_rows, unit = blockIdx.y;
  const int channels = in.channels(), dim = in.dim;
  if (unit >= in.G + v_units) {
    for (int e = threadIdx.x; e < (stop - row0) * in.H; e += 256) {
      const int row = row0 + e / in.H, h = e % in.H;
      const T* x = proj + (size_t)row * in.row_stride;
      float* to = beside + ((size_t)row * in.H + h) * DR_BESIDE;
      to[0] = expf(-expf(in.a_log[h]) * dr_softplus(to_f32(x[in.a_first + h]) + in.dt_bias[h]));
      to[1] = 1.0f / (1.0f + expf(-to_f32(x[in.b_first + h])));
    }
    return;
  }
  const bool keys = unit < in.G;
  const int width = keys ? 2 * dim : 256;
  for (int e = threadIdx.x; e < width; e += 256) {
    const int c = !keys ? 2 * in.G * dim + (unit - in.G) * 256 + e : (e < dim ? unit * dim + e : (in.G + unit) * dim + e - dim);
    if (c >= channels) continue;
    float w[TAPS], win[TAPS];
#pragma unroll
    for (int j = 0; j < TAPS; ++j) w[j] = in.conv[(size_t)c * TAPS + j];
    int seq = -1;
    float ahead[DP_AHEAD];      // the next rows' inputs, asked for together
    for (int row = row0; row < stop; ++row) {
      if ((row - row0) % DP_AHEAD == 0) {
#pragma unroll
        for (int i = 0; i < DP_AHEAD; ++i) ahead[i] = to_f32(proj[(size_t)(row + i < stop ? row + i : stop - 1) * in.row_stride + in.first + c]);
      }
      const int here = row_seq[row];
      if (here != seq) {      // the first row of the stretch, or of a sequence: the inputs before it
        seq = here;
        const int t = row - seq_start[seq];
        const float* old = in.state + (size_t)seq_slot[seq] * in.slot_stride + in.conv_offset;
#pragma unroll
        for (int j = 0; j < TAPS - 1; ++j) {
          const int back = TAPS - 1 - j;
          win[j] = back <= t ? to_f32(proj[(size_t)(row - back) * in.row_stride + in.first + c]) : old[(size_t)(TAPS - 1 + t - back) * channels + c];
        }
      } else {
#pragma unroll
        for (int j = 0; j < TAPS - 1; ++j) win[j] = win[j + 1];
      }
      win[TAPS - 1] = ahead[0];
#pragma unroll
      for (int i = 0; i + 1 < DP_AHEAD; ++i) ahead[i] = ahead[i + 1];
      float acc = 0.f;
#pragma unroll
      for (int j = 0; j < TAPS; ++j) acc = fmaf(w[j], win[j], acc);
      acc = dr_silu(acc);
      if (keys) pair[(row - row0) * width + e] = acc;
      else qkv[(size_t)row * channels + c] = acc;
    }
  }
  if (!keys) return;
  __syncthreads();
  const int lane = threadIdx.x % BH_WAVE, per = in.H / in.G;
  for (int row = row0 + threadIdx.x / BH_WAVE; row < stop; row += 4) {
    const float* mine = pair + (row - row0) * width;
    float qq = 0.f, kk = 0.f, qk = 0.f;
    for (int i = lane; i < dim; i += BH_WAVE) {
      const float q = mine[i], k = mine[dim + i];
      qq += q * q;
      kk += k * k;
      qk += q * k;
    }
    const float q_scale = 1.0f / sqrtf(wave_sum(qq) + DR_UNIT_EPS) / sqrtf((float)dim), k_scale = 1.0f / sqrtf(wave_sum(kk) + DR_UNIT_EPS);
    qk = wave_sum(qk) * q_scale * k_scale;
    float* to = qkv + (size_t)row * channels;
    for (int i = lane; i < dim; i += BH_WAVE) {
      to[unit * dim + i] = mine[i] * q_scale;
      to[(in.G + unit) * dim + i] = mine[dim + i] * k_scale;
    }
    for (int i = lane; i < per; i += BH_WAVE) beside[((size_t)row * in.H + unit * per + i) * DR_BESIDE + 2] = qk;
  }
}

static const char* delta_fault(const DeltaRows& in) {
  if (in.H <= 0 || in.G <= 0 || in.dim <= 0 || in.vdim <= 0) return "sizes must be positive";
  if (in.H % in.G) return "the heads of values do not fall evenly to the heads of queries and keys";
  if (in.taps < 1 || in.taps > DR_MAX_TAPS) return "a convolution has 1 to 16 taps";
  const long channels = 2L * in.G * in.dim + (long)in.H * in.vdim;
  if (in.first < 0 || in.first + channels > in.row_stride || in.b_first < 0 || in.b_first + in.H > in.row_stride || in.a_first < 0 ||
      in.a_first + in.H > in.row_stride)
    return "q, k, v, b or a lie outside their row";
  if (in.conv_offset < (long)in.H * in.dim * in.vdim || in.conv_offset + (in.taps - 1) * channels > in.slot_stride)
    return "a slot's state is smaller than the heads' states and the convolution's inputs";
  return nullptr;
}

// proj [n_rows][row_stride] (dtype); qkv f32 [n_rows][2 G dim + H vdim]; beside f32 [n_rows][H][4].
extern "C" int bh_delta_prep(const void* proj, int dtype, int row_stride, int first, int b_first, int a_first, const float* conv, int taps,
                             float* state, long slot_stride, long conv_offset, const float* a_log, const float* dt_bias,
                             const int32_t* row_seq, const int32_t* seq_start, const int32_t* seq_slot, float* qkv, float* beside, int n_rows,
                             int H, int G, int dim, int vdim, hipStream_t stream) {
  const DeltaRows in = {row_stride, first, b_first, a_first, conv, taps, state, slot_stride, conv_offset, a_log, dt_bias, H, G, dim, vdim};
  if (const char* fault = delta_fault(in)) return bh_fail("delta_prep: %s", fault);
  BH_REQUIRE(n_rows > 0, "delta_prep: a step has rows");
  const size_t lds = (size_t)DP_ROWS * 2 * dim * sizeof(float);
  if (n_rows >= 4 * DP_ROWS && taps <= 4 && lds <= 64 * 1024 && (dtype == BH_F32 || dtype == BH_BF16)) {
    const int v_units = (H * vdim + 255) / 256;
    const dim3 walk((n_rows + DP_ROWS - 1) / DP_ROWS, G + v_units + 1);
    BH_REQUIRE(walk.y <= 65535, "delta_prep: too many heads");
#define BH_DP(T, TAPS)                                                                                                            \
  do {                                                                                                                            \
    bh_allow_lds<delta_prep_walk_kernel<T, TAPS>>(lds);                                                                           \
    delta_prep_walk_kernel<T, TAPS><<<walk, 256, lds, stream>>>((const T*)proj, in, row_seq, seq_start, seq_slot, qkv, beside, n_rows, v_units); \
  } while (0)
#define BH_DP_TAPS(T)               \
  switch (taps) {                   \
    case 1: BH_DP(T, 1); break;     \
    case 2: BH_DP(T, 2); break;     \
    case 3: BH_DP(T, 3); break;     \
    default: BH_DP(T, 4); break;    \
  }
    if (dtype == BH_F32) BH_DP_TAPS(float)
    else BH_DP_TAPS(bf16_t)
#undef BH_DP_TAPS
#undef BH_DP
    return bh_check_launch("delta_prep");
  }
  const dim3 grid(n_rows, (G + H + 1 + 3) / 4);
  BH_REQUIRE(grid.y <= 65535, "delta_prep: too many heads");
  if (dtype == BH_F32) delta_prep_kernel<float><<<grid, 256, 0, stream>>>((const float*)proj, in, row_seq, seq_start, seq_slot, qkv, beside);
  else if (dtype == BH_BF16) delta_prep_kernel<bf16_t><<<grid, 256, 0, stream>>>((const bf16_t*)proj, in, row_seq, seq_start, seq_slot, qkv, beside);
  else return bh_fail("delta_prep: unknown dtype %d", dtype);
  return bh_check_launch("delta_prep");
}

// ---- the recurrence -------------------------------------------------------------------------------------------
// The columns of S go their ways apart: s <- g s + k u, u = beta (v - g s.k), o = g s.q + (k.q) u, all from one pass over the old s.
// A thread keeps R elements of each of C columns; the SL threads of a column are neighbouring lanes and hold its elements in turns of
// four (slice, slice + SL, ...), so that a row's k and q come from LDS as 16-byte pieces; their shares of s.k and s.q are added by
// data-parallel moves.  DR_STAGE rows go through LDS at a time, the next stage is asked for ahead and written to the other half.
//
// Long sequences are walked in chunks side by side.  A chunk but the first starts from nothing; since the rule is linear in the state
// it starts from, dim further columns without values, started from the unit vectors, give the chunk's move M (S_end = M S_in +
// S_local) and, read out, every row's carried query (its o owes S_in^T of it).  delta_combine joins the chunks' states in order and
// chunk_carry adds what the rows owe.
#define DR_STAGE 16
#define DR_WAVES 4

struct DeltaChunks {
  int rows, count;      // 0 rows: whole sequences
  float* states;        // [n_seqs][count][H][dim][vdim]
  float* moves;         // [n_seqs][count][H][dim][dim]
  float* queries;       // [n_rows][H][dim]
};

template <int R, int SL, int C>
__global__ __launch_bounds__(DR_WAVES * BH_WAVE) void delta_scan_kernel(const float* __restrict__ qkv, const float* __restrict__ beside,
                                                                        float* __restrict__ state, long slot_stride,
                                                                        const int32_t* __restrict__ seq_start,
                                                                        const int32_t* __restrict__ seq_slot, const int32_t* __restrict__ seq_to, float* __restrict__ out, int H, int G,
                                                                        int dim, int vdim, DeltaChunks chunks) {
  constexpr int DP = R * SL, PER_WAVE = BH_WAVE / SL * C, COLS = DR_WAVES * PER_WAVE;
  constexpr int KQ = DR_STAGE * DP / 4;                              // 16-byte pieces of a stage's keys (and of its queries)
  constexpr int KQ_EACH = (KQ + 255) / 256, V_EACH = (DR_STAGE * COLS + 255) / 256;
  __shared__ float4 k_s[2][KQ], q_s[2][KQ];
  __shared__ float v_s[2][DR_STAGE * COLS];
  __shared__ float4 gates[2][DR_STAGE];                              // g, beta, k.q
  const int seq = blockIdx.x / chunks.count, chunk = blockIdx.x % chunks.count, head = blockIdx.y, tile0 = blockIdx.z * COLS;
  const int seq_first = seq_start[seq], seq_stop = seq_start[seq + 1];
  const int in_chunks = chunks.rows > 0 ? (seq_stop - seq_first + chunks.rows - 1) / chunks.rows : 1;
  const int start = seq_first + chunk * chunks.rows;
  const int stop = (chunks.rows > 0 && start + chunks.rows < seq_stop) ? start + chunks.rows : seq_stop;
  if (chunk > 0 && chunk >= in_chunks) return;
  const bool apart = in_chunks > 1;
  const int n_columns = chunk > 0 ? vdim + dim : vdim;
  if (tile0 >= n_columns) return;
  const int lane = threadIdx.x % BH_WAVE, slice = lane % SL;
  const int local = threadIdx.x / BH_WAVE * PER_WAVE + lane / SL * C, column0 = tile0 + local;
  const int channels = 2 * G * dim + H * vdim, group = head / (H / G);
  const size_t head_state = (size_t)head * dim * vdim;
  const float* slot = state + (size_t)seq_slot[seq] * slot_stride + head_state;
  const size_t place = (size_t)(seq * chunks.count + chunk) * H + head;
  float* values_to = apart ? chunks.states + place * dim * vdim : state + (size_t)seq_to[seq] * slot_stride + head_state;
  float* moves_to = apart ? chunks.moves + place * dim * dim : nullptr;

  float S[C][R];
#pragma unroll
  for (int c = 0; c < C; ++c)
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int d = 4 * (slice + SL * (r / 4)) + r % 4, column = column0 + c;
      S[c][r] = 0.f;
      if (chunk == 0) {
        if (d < dim && column < vdim) S[c][r] = slot[(size_t)d * vdim + column];
      } else if (column == vdim + d) {
        S[c][r] = 1.f;
      }
    }

  float4 k_ahead[KQ_EACH], q_ahead[KQ_EACH], gates_ahead = {0.f, 0.f, 0.f, 0.f};
  float v_ahead[V_EACH];
  const bool whole = dim % 4 == 0 && vdim % 4 == 0;      // rows of 16-byte pieces
  auto piece = [&](const float* at, int d) -> float4 {
    float4 x = {0.f, 0.f, 0.f, 0.f};
    if (whole) {
      if (d < dim) x = *reinterpret_cast<const float4*>(at + d);
    } else {
      if (d < dim) x.x = at[d];
      if (d + 1 < dim) x.y = at[d + 1];
      if (d + 2 < dim) x.z = at[d + 2];
      if (d + 3 < dim) x.w = at[d + 3];
    }
    return x;
  };
  auto ask = [&](int row0) {
#pragma unroll
    for (int i = 0; i < KQ_EACH; ++i) {
      const int e = threadIdx.x + 256 * i, t = e / (DP / 4), d = e % (DP / 4) * 4;
      k_ahead[i] = q_ahead[i] = float4{0.f, 0.f, 0.f, 0.f};
      if (e < KQ && row0 + t < stop) {
        const float* x = qkv + (size_t)(row0 + t) * channels + group * dim;
        q_ahead[i] = piece(x, d);
        k_ahead[i] = piece(x + G * dim, d);
      }
    }
#pragma unroll
    for (int i = 0; i < V_EACH; ++i) {
      const int e = threadIdx.x + 256 * i, t = e / COLS, column = tile0 + e % COLS;
      v_ahead[i] = 0.f;
      if (e < DR_STAGE * COLS && row0 + t < stop && column < vdim) v_ahead[i] = qkv[(size_t)(row0 + t) * channels + 2 * G * dim + head * vdim + column];
    }
    if (threadIdx.x < DR_STAGE && row0 + (int)threadIdx.x < stop)
      gates_ahead = *reinterpret_cast<const float4*>(beside + ((size_t)(row0 + threadIdx.x) * H + head) * DR_BESIDE);
  };
  auto put = [&](int half) {
#pragma unroll
    for (int i = 0; i < KQ_EACH; ++i) {
      const int e = threadIdx.x + 256 * i;
      if (e < KQ) k_s[half][e] = k_ahead[i], q_s[half][e] = q_ahead[i];
    }
#pragma unroll
    for (int i = 0; i < V_EACH; ++i) {
      const int e = threadIdx.x + 256 * i;
      if (e < DR_STAGE * COLS) v_s[half][e] = v_ahead[i];
    }
    if (threadIdx.x < DR_STAGE) gates[half][threadIdx.x] = gates_ahead;
  };
  ask(start);
  put(0);
  __syncthreads();
  int half = 0;
  for (int row0 = start; row0 < stop; row0 += DR_STAGE, half ^= 1) {
    const bool more = row0 + DR_STAGE < stop;
    if (more) ask(row0 + DR_STAGE);
    const int n = stop - row0 < DR_STAGE ? stop - row0 : DR_STAGE;
    float o_kept[C];
#pragma unroll
    for (int c = 0; c < C; ++c) o_kept[c] = 0.f;
    for (int t = 0; t < n; ++t) {
      const float4 gate = gates[half][t];
      float4 k4[R / 4];
      float sk[C], sq[C], k_sum[C][2], q_sum[C][2];
#pragma unroll
      for (int c = 0; c < C; ++c) k_sum[c][0] = k_sum[c][1] = q_sum[c][0] = q_sum[c][1] = 0.f;
#pragma unroll
      for (int i = 0; i < R / 4; ++i) {
        k4[i] = k_s[half][t * (DP / 4) + slice + SL * i];
        const float4 q4 = q_s[half][t * (DP / 4) + slice + SL * i];
#pragma unroll
        for (int c = 0; c < C; ++c) {
          k_sum[c][0] = fmaf(S[c][4 * i], k4[i].x, k_sum[c][0]);
          k_sum[c][1] = fmaf(S[c][4 * i + 1], k4[i].y, k_sum[c][1]);
          k_sum[c][0] = fmaf(S[c][4 * i + 2], k4[i].z, k_sum[c][0]);
          k_sum[c][1] = fmaf(S[c][4 * i + 3], k4[i].w, k_sum[c][1]);
          q_sum[c][0] = fmaf(S[c][4 * i], q4.x, q_sum[c][0]);
          q_sum[c][1] = fmaf(S[c][4 * i + 1], q4.y, q_sum[c][1]);
          q_sum[c][0] = fmaf(S[c][4 * i + 2], q4.z, q_sum[c][0]);
          q_sum[c][1] = fmaf(S[c][4 * i + 3], q4.w, q_sum[c][1]);
        }
      }
#pragma unroll
      for (int c = 0; c < C; ++c) {
        sk[c] = slices_sum<SL>(k_sum[c][0] + k_sum[c][1]);
        sq[c] = slices_sum<SL>(q_sum[c][0] + q_sum[c][1]);
      }
#pragma unroll
      for (int c = 0; c < C; ++c) {
        const float u = gate.y * (v_s[half][t * COLS + local + c] - gate.x * sk[c]);
        const float o = fmaf(gate.z, u, gate.x * sq[c]);
        if (slice == (t & (SL - 1))) o_kept[c] = o;
#pragma unroll
        for (int i = 0; i < R / 4; ++i) {
          S[c][4 * i] = fmaf(k4[i].x, u, gate.x * S[c][4 * i]);
          S[c][4 * i + 1] = fmaf(k4[i].y, u, gate.x * S[c][4 * i + 1]);
          S[c][4 * i + 2] = fmaf(k4[i].z, u, gate.x * S[c][4 * i + 2]);
          S[c][4 * i + 3] = fmaf(k4[i].w, u, gate.x * S[c][4 * i + 3]);
        }
      }
      // every SL rows (and behind the last) each lane of a column writes the row it kept
      if ((t & (SL - 1)) == SL - 1 || t == n - 1) {
        const int kept = (t & ~(SL - 1)) + slice;
        if (kept <= t) {
#pragma unroll
          for (int c = 0; c < C; ++c) {
            const int column = column0 + c;
            if (column < vdim) out[(size_t)(row0 + kept) * H * vdim + head * vdim + column] = o_kept[c];
            else if (column < n_columns) chunks.queries[((size_t)(row0 + kept) * H + head) * dim + column - vdim] = o_kept[c];
          }
        }
      }
    }
    if (more) {
      put(half ^ 1);      // (everyone was done with that half at the last barrier)
      __syncthreads();
    }
  }
#pragma unroll
  for (int c = 0; c < C; ++c)
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int d = 4 * (slice + SL * (r / 4)) + r % 4, column = column0 + c;
      if (d >= dim) continue;
      if (column < vdim) values_to[(size_t)d * vdim + column] = S[c][r];
      else if (column < n_columns) moves_to[(size_t)d * dim + column - vdim] = S[c][r];
    }
}

// Through a sequence's chunks in order: S_in(c + 1) = M(c) S_in(c) + S_local(c); a chunk's place in `states` then holds the state it
// started from, and the state after the last chunk goes to the slot.  A workgroup a (sequence, head, 16 value columns): the running
// state's columns stand in LDS (rows of DC_STRIDE: the four rows that a wave reads at once lie in other banks), a wave makes every fourth
// 16 x 16 tile of the next one with v_mfma_f32_16x16x4_f32, M's pieces straight from memory, four neighbouring columns of a row a lane.
#define DC_COLS 16
#define DC_STRIDE 20
typedef float dr_f32x4_t __attribute__((ext_vector_type(4)));
__global__ __launch_bounds__(256) void delta_combine_kernel(DeltaChunks chunks, float* __restrict__ state, long slot_stride,
                                                            const int32_t* __restrict__ seq_start, const int32_t* __restrict__ seq_slot, const int32_t* __restrict__ seq_to, int H,
                                                            int dim, int vdim) {
  extern __shared__ float run[];           // [2][rows of 16-row tiles][DC_STRIDE]
  const int seq = blockIdx.x, head = blockIdx.y, v0 = blockIdx.z * DC_COLS;
  const int in_chunks = (seq_start[seq + 1] - seq_start[seq] + chunks.rows - 1) / chunks.rows;
  if (in_chunks <= 1) return;      // the walk itself wrote the slot
  const int wave = threadIdx.x / BH_WAVE, lane = threadIdx.x % BH_WAVE, j = lane % 16, g = lane / 16;
  const int tiles = (dim + 15) / 16, half = tiles * 16 * DC_STRIDE, column = v0 + j;
  const bool real = column < vdim, whole = dim % 4 == 0;
  for (int e = threadIdx.x; e < 2 * half; e += 256) run[e] = 0.f;
  __syncthreads();
  int now = 0;
  for (int c = 0; c < in_chunks; ++c) {
    const size_t place = (size_t)(seq * chunks.count + c) * H + head;
    float* states = chunks.states + place * dim * vdim + column;
    const float* moves = chunks.moves + place * dim * dim;
    const float* old = run + now * half;
    float* next = run + (now ^ 1) * half;
    for (int tile = wave; tile < tiles; tile += 4) {
      dr_f32x4_t acc;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int d = 16 * tile + 4 * g + r;
        acc[r] = real && d < dim ? states[(size_t)d * vdim] : 0.f;
      }
      if (c > 0) {
        const int my_row = 16 * tile + j;
        const float* m = moves + (size_t)(my_row < dim ? my_row : dim - 1) * dim;      // (rows beyond dim are never kept)
        for (int k0 = 0; k0 < tiles; k0 += 8) {
          float x[8][4];
#pragma unroll
          for (int b = 0; b < 8; ++b) {
            const int d = 16 * (k0 + b) + 4 * g;
            if (whole && d < dim) {
              const float4 piece = *reinterpret_cast<const float4*>(m + d);
              x[b][0] = piece.x, x[b][1] = piece.y, x[b][2] = piece.z, x[b][3] = piece.w;
            } else {
#pragma unroll
              for (int s = 0; s < 4; ++s) x[b][s] = d + s < dim ? m[d + s] : 0.f;
            }
          }
#pragma unroll
          for (int b = 0; b < 8; ++b) {
            if (k0 + b >= tiles) break;
#pragma unroll
            for (int s = 0; s < 4; ++s)
              acc = __builtin_amdgcn_mfma_f32_16x16x4f32(x[b][s], old[(16 * (k0 + b) + 4 * g + s) * DC_STRIDE + j], acc, 0, 0, 0);
          }
        }
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int d = 16 * tile + 4 * g + r;
        if (d < dim) {
          if (real) states[(size_t)d * vdim] = old[d * DC_STRIDE + j];
          next[d * DC_STRIDE + j] = acc[r];
        }
      }
    }
    __syncthreads();
    now ^= 1;
  }
  float* slot = state + (size_t)seq_to[seq] * slot_stride + (size_t)head * dim * vdim + column;
  for (int d = threadIdx.x / 16; d < dim; d += 16)
    if (real) slot[(size_t)d * vdim] = run[now * half + d * DC_STRIDE + j];
}

struct DeltaShape {
  int R, SL, C;
  int columns() const { return DR_WAVES * (BH_WAVE / SL) * C; }
};
static DeltaShape delta_shape(int dim) {
  if (dim <= 16) return {4, 4, 1};
  if (dim <= 32) return {8, 4, 1};
  if (dim <= 64) return {8, 8, 1};
  if (dim <= 128) return {16, 8, 1};
  if (dim <= 256) return {16, 16, 1};
  return {32, 16, 1};
}

// What a walk is estimated to take, for the number of chunks with the least of it.  A row of a workgroup's chain takes hypot(row, shared *
// workgroups) us where so many of them stand on a compute unit, of which `resident` fit it (their stages in LDS, their registers); more come in
// rounds.  A chunk but the first carries dim more columns.  The first's missing ones are felt where the number of chunks is odd: where
// it is even, workgroups dealt to the eight XCDs in turn leave it all to some of them.  Joining takes 2 us a chunk and 4 more at heads of
// 128 x 128, the launches behind the walk 16.
// Fitted to 223 steps of 1 to 128 heads of 16 to 256, 256 to 8,192 rows in 1 to 16 sequences, each at up to 17 numbers of chunks: what it
// chooses takes 1.004 times the best of these on average, 1.06 at most.  Six workgroups a compute unit wanted, whatever a row costs then, took 1.09;
// us, so / by the estimate: 32 heads of 128, 2,048 rows 383 / 343, 512 rows 148 / 126, 16 heads, 2,048 rows 250 / 219, 48 heads 502 / 446; 8 heads of
// 256 576 / 489; 16 heads of 64 125 / 102; 128 heads of 64 344 / 344; but 96 of 64, 8,192 rows 1,143 / 1,193, 8 of 256 1,983 / 2,106.
struct DeltaCost {
  double row, shared;
  int resident;
  long walks, tiles, later_tiles;
  double joining;

  DeltaCost(int n_seqs, int H, int dim, int vdim) {
    const int columns = delta_shape(dim).columns();
    if (dim <= 16) row = 0.2, shared = 0.054, resident = 8;
    else if (dim <= 32) row = 0.223, shared = 0.075, resident = 6;
    else if (dim <= 64) row = 0.2, shared = 0.083, resident = 6;
    else if (dim <= 128) row = 0.306, shared = 0.121, resident = 4;
    else row = 0.36, shared = 0.146, resident = 2;
    walks = (long)n_seqs * H, tiles = (vdim + columns - 1) / columns, later_tiles = (vdim + dim + columns - 1) / columns;
    joining = 2.0 + 3.9 * dim * dim / 16384.0;
  }
  double beside(long workgroups) const { return workgroups > 0 ? std::hypot(row, shared * (double)workgroups) : 0.0; }
  double a_row(int chunks) const {
    const long workgroups = walks * (chunks == 1 ? tiles : chunks % 2 == 0 ? chunks * later_tiles : tiles + (chunks - 1) * later_tiles);
    const long share = (workgroups + bh_compute_units() - 1) / bh_compute_units();
    return (double)(share / resident) * beside(resident) + beside(share % resident);
  }
  // (of odd numbers above three the workgroups are left on some compute units one more than the average says)
  static bool tried(int chunks) { return chunks <= 3 || chunks % 2 == 0; }
  double behind(int chunks) const { return 16.0 + joining * chunks; }
  // (the chunks' states of as many sequences are much memory for a last round's gain)
  bool fills() const { return walks * tiles >= 4L * bh_compute_units(); }
};
#define DELTA_MOST_CHUNKS 64
#define DELTA_CHUNK 64       // rows, at least

// Rows of a chunk for a step whose longest sequence brings max_rows rows (max_rows and more: sequences are walked whole).
extern "C" int bh_delta_chunk_rows(int n_seqs, int max_rows, int H, int dim, int vdim) {
  if (max_rows < 3 * DELTA_CHUNK || n_seqs <= 0 || H <= 0 || dim <= 0 || vdim <= 0 || dim > 256) return max_rows;
  const DeltaCost cost(n_seqs, H, dim, vdim);
  if (cost.fills()) return max_rows;
  int best = max_rows;
  double least = max_rows * cost.a_row(1);
  for (int wanted = 2; wanted <= max_rows / DELTA_CHUNK && wanted <= DELTA_MOST_CHUNKS; ++wanted) {
    if (!DeltaCost::tried(wanted)) continue;
    const int rows = ((max_rows + wanted - 1) / wanted + DR_STAGE - 1) / DR_STAGE * DR_STAGE, count = (max_rows + rows - 1) / rows;
    const double takes = rows * cost.a_row(count) + cost.behind(count);
    if (rows < max_rows && takes < least) best = rows, least = takes;
  }
  return best;
}

// Chunks of all sequences together, at most, over the steps of up to n_seqs sequences, n_rows rows and max_rows rows a sequence (0: no such
// step is cut).  Fewer sequences are cut into more chunks each, and a number of chunks may be the best one at any number of rows: it is
// left out where for the fewest and the most rows, and so, both costs being linear in them, for all between, fewer chunks cost less though their
// rows are rounded up to a stage.
extern "C" long bh_delta_most_chunks(int n_seqs, int n_rows, int max_rows, int H, int dim, int vdim) {
  if (H <= 0 || dim <= 0 || vdim <= 0 || dim > 256) return 0;
  long most = 0;
  for (int n = 1; n <= n_seqs; ++n) {
    const DeltaCost cost(n, H, dim, vdim);
    const int longest = n_rows - n + 1 < max_rows ? n_rows - n + 1 : max_rows;      // the other sequences bring a row each
    if (longest < 3 * DELTA_CHUNK || cost.fills()) break;
    double a_row[DELTA_MOST_CHUNKS + 1];
    const int pieces = longest / DELTA_CHUNK < DELTA_MOST_CHUNKS ? longest / DELTA_CHUNK : DELTA_MOST_CHUNKS;
    for (int chunks = 1; chunks <= pieces; ++chunks) a_row[chunks] = cost.a_row(chunks);
    const auto never = [&](int chunks) {
      const int ends[2] = {std::max(chunks, 3) * DELTA_CHUNK, longest};
      for (int fewer = 1; fewer < chunks; ++fewer) {
        bool less = DeltaCost::tried(fewer);
        for (int rows : ends) {
          const double takes = (double)rows / chunks * a_row[chunks] + cost.behind(chunks);
          less = less && (fewer == 1 ? rows * a_row[1] : ((double)rows / fewer + DR_STAGE) * a_row[fewer] + cost.behind(fewer)) < takes;
        }
        if (less) return true;
      }
      return false;
    };
    int chunks = pieces;
    while (chunks > 1 && never(chunks)) --chunks;
    if (chunks > 1) most = std::max(most, (long)n * chunks);
  }
  return most;
}

extern "C" int bh_delta_takes(int dim, int vdim) { return dim > 0 && dim <= 512 && vdim > 0; }

// qkv and beside as delta_prep leaves them; out [n_rows][H * vdim] float32.  chunk_rows: bh_delta_chunk_rows' answer for the step; where
// that is less than max_rows (the rows of the longest sequence), scratch holds n_seqs * chunks * H * dim * (vdim + dim) +
// n_rows * H * dim floats.
extern "C" int bh_delta_scan(const float* qkv, const float* beside, float* state, long slot_stride, const int32_t* seq_start,
                             const int32_t* seq_slot, const int32_t* seq_to, float* out, int n_seqs, int H, int G, int dim, int vdim, int n_rows, int max_rows,
                             int chunk_rows, float* scratch, hipStream_t stream) {
  BH_REQUIRE(n_seqs > 0 && H > 0 && G > 0 && dim > 0 && vdim > 0 && H % G == 0, "delta_scan: sizes must be positive, heads fall evenly to groups");
  BH_REQUIRE(bh_delta_takes(dim, vdim), "delta_scan: heads of %d key dimensions are above the limit of 512", dim);
  BH_REQUIRE(slot_stride >= (long)H * dim * vdim, "delta_scan: a slot's state is smaller than the heads' states");
  BH_REQUIRE(max_rows > 0 && n_rows >= n_seqs && chunk_rows > 0 && H <= 65535, "delta_scan: a step has rows, and chunks have rows");
  DeltaChunks chunks = {0, 1, nullptr, nullptr, nullptr};
  if (chunk_rows < max_rows) {
    BH_REQUIRE(scratch != nullptr && chunk_rows % DR_STAGE == 0, "delta_scan: chunks need scratch memory and whole stages");
    chunks.rows = chunk_rows;
    chunks.count = (max_rows + chunk_rows - 1) / chunk_rows;
    chunks.states = scratch;
    chunks.moves = chunks.states + (size_t)n_seqs * chunks.count * H * dim * vdim;
    chunks.queries = chunks.moves + (size_t)n_seqs * chunks.count * H * dim * dim;
  }
  const DeltaShape shape = delta_shape(dim);
  const int columns = shape.columns(), most = chunks.rows ? vdim + dim : vdim;
  BH_REQUIRE((long)n_seqs * chunks.count < (1L << 31) && (most + columns - 1) / columns <= 65535, "delta_scan: too many chunks or columns");
  const dim3 grid(n_seqs * chunks.count, H, (most + columns - 1) / columns);
#define BH_DR(R, SL, C)                                                                                                            \
  delta_scan_kernel<R, SL, C><<<grid, DR_WAVES * BH_WAVE, 0, stream>>>(qkv, beside, state, slot_stride, seq_start, seq_slot, seq_to, out, H, G, dim, \
                                                                       vdim, chunks)
  if (dim <= 16) BH_DR(4, 4, 1);
  else if (dim <= 32) BH_DR(8, 4, 1);
  else if (dim <= 64) BH_DR(8, 8, 1);
  else if (dim <= 128) BH_DR(16, 8, 1);
  else if (dim <= 256) BH_DR(16, 16, 1);
  else BH_DR(32, 16, 1);
#undef BH_DR
  if (int status = bh_check_launch("delta_scan")) return status;
  if (chunks.rows == 0) return 0;
  const size_t lds = (size_t)2 * ((dim + 15) / 16) * 16 * DC_STRIDE * sizeof(float);
  bh_allow_lds<delta_combine_kernel>(lds);
  delta_combine_kernel<<<dim3(n_seqs, H, (vdim + DC_COLS - 1) / DC_COLS), 256, lds, stream>>>(chunks, state, slot_stride, seq_start, seq_slot, seq_to, H,
                                                                                            dim, vdim);
  if (int status = bh_check_launch("delta_combine")) return status;
  return bh_chunk_carry(chunks.states, chunks.queries, chunks.rows, chunks.count, seq_start, out, n_seqs, H, dim, vdim, stream);
}

// ---- a decode step --------------------------------------------------------------------------------------------
// A workgroup a (sequence, group): it owns the group's channels of q and k and its heads' channels of v, so that it may move their kept
// inputs on.  Its 256-thread teams take the group's heads in turn.  A team's four waves are column tiles of 64 side by side, and
// slices of the state's rows where there are fewer than four tiles: thread (column, slice) keeps R rows of its column in registers, from
// loads that were asked for before the convolutions; the slices' shares of S^T k and S^T q meet in LDS.
template <typename T, int R, int TEAMS>
__global__ __launch_bounds__(256 * TEAMS) void delta_step_kernel(const T* __restrict__ proj, DeltaRows in, int g_first,
                                                                 const int32_t* __restrict__ seq_slot, const int32_t* __restrict__ seq_to, const float* __restrict__ norm, float eps,
                                                                 T* __restrict__ out, int out_block_rows, int tiles) {
  extern __shared__ __align__(16) float lds[];
  const int H = in.H, G = in.G, dim = in.dim, vdim = in.vdim, per = H / G;
  const int slices = 4 / tiles, dp = R * slices;      // rows of a column that the registers of its slices hold
  float* q_s = lds;                           // [dp], zeros beyond dim
  float* k_s = q_s + dp;
  float* v_s = k_s + dp;                      // [per][vdim]
  float* gates = v_s + per * vdim;            // [per][2]: g, beta
  float* sums = gates + 2 * per;              // q's and k's scale, k.q
  float* part = sums + 4;                     // [TEAMS][4][64][2]
  float* squares = part + TEAMS * 512;        // [TEAMS][4]
  const int seq = blockIdx.x, group = blockIdx.y, row = seq;
  // (a wave's team, tile and slice are the same in all its lanes: the addresses of a state's rows stay out of the vector registers)
  const int lane = threadIdx.x % BH_WAVE, team_wave = __builtin_amdgcn_readfirstlane(threadIdx.x / BH_WAVE), team = team_wave / 4, wave = team_wave % 4;
  const int column = (wave % tiles) * BH_WAVE + lane, slice = wave / tiles, d0 = slice * R;
  const float* slot = in.state + (size_t)seq_slot[seq] * in.slot_stride;
  float* left = in.state + (size_t)seq_to[seq] * in.slot_stride;
  float S[R];
  auto load = [&](int i) {      // the state of the group's head i
    const float* from = slot + (size_t)(group * per + (i < per ? i : 0)) * dim * vdim;
    const int at = column < vdim ? column : 0;
#pragma unroll
    for (int r = 0; r < R; ++r) {      // (rows beyond dim read the last one, times keys and queries of zero)
      const float* of_row = from + (size_t)(d0 + r < dim ? d0 + r : dim - 1) * vdim;
      S[r] = of_row[at];
    }
  };
  load(team);
  // the convolutions, and the inputs they leave for the next step
  const int channels = in.channels(), mine = 2 * dim + per * vdim, keep = in.taps - 1;
  const float* old = slot + in.conv_offset;
  float* inputs = left + in.conv_offset;
  const T* x = proj + (size_t)row * in.row_stride;
  for (int e = threadIdx.x; e < mine; e += 256 * TEAMS) {
    const int c = e < dim ? group * dim + e : (e < 2 * dim ? (G + group) * dim + e - dim : 2 * G * dim + group * per * vdim + e - 2 * dim);
    const float* w = in.conv + (size_t)c * in.taps;
    const float u = to_f32(x[in.first + c]);
    float acc = 0.f;
    for (int j = 0; j < keep; ++j) {
      const float before = old[(size_t)j * channels + c];
      acc = fmaf(w[j], before, acc);
      if (j > 0) inputs[(size_t)(j - 1) * channels + c] = before;
    }
    if (keep > 0) inputs[(size_t)(keep - 1) * channels + c] = u;
    acc = dr_silu(fmaf(w[keep], u, acc));
    if (e < dim) q_s[e] = acc;
    else if (e < 2 * dim) k_s[e - dim] = acc;
    else v_s[e - 2 * dim] = acc;
  }
  for (int e = dim + threadIdx.x; e < dp; e += 256 * TEAMS) q_s[e] = k_s[e] = 0.f;
  for (int i = threadIdx.x; i < per; i += 256 * TEAMS) {
    const int h = group * per + i;
    gates[2 * i] = expf(-expf(in.a_log[h]) * dr_softplus(to_f32(x[in.a_first + h]) + in.dt_bias[h]));
    gates[2 * i + 1] = 1.0f / (1.0f + expf(-to_f32(x[in.b_first + h])));
  }
  __syncthreads();
  if (threadIdx.x < BH_WAVE) {
    float qq = 0.f, kk = 0.f, qk = 0.f;
    for (int i = lane; i < dim; i += BH_WAVE) {
      const float q = q_s[i], k = k_s[i];
      qq += q * q;
      kk += k * k;
      qk += q * k;
    }
    const float q_scale = 1.0f / sqrtf(wave_sum(qq) + DR_UNIT_EPS) / sqrtf((float)dim), k_scale = 1.0f / sqrtf(wave_sum(kk) + DR_UNIT_EPS);
    qk = wave_sum(qk) * q_scale * k_scale;
    if (lane == 0) sums[0] = q_scale, sums[1] = k_scale, sums[2] = qk;
  }
  __syncthreads();
  const float q_scale = sums[0], k_scale = sums[1], kq = sums[2];
  for (int i0 = 0; i0 < per; i0 += TEAMS) {
    const int i = i0 + team, head = group * per + i;
    const bool works = i < per;
    if (i0 > 0) load(i);
    float sk = 0.f, sq = 0.f;
#pragma unroll
    for (int r = 0; r < R; r += 4) {
      const float4 k4 = *reinterpret_cast<const float4*>(k_s + d0 + r), q4 = *reinterpret_cast<const float4*>(q_s + d0 + r);
      sk = fmaf(S[r], k4.x, fmaf(S[r + 1], k4.y, fmaf(S[r + 2], k4.z, fmaf(S[r + 3], k4.w, sk))));
      sq = fmaf(S[r], q4.x, fmaf(S[r + 1], q4.y, fmaf(S[r + 2], q4.z, fmaf(S[r + 3], q4.w, sq))));
    }
    if (slices > 1) {
      float* shares = part + team * 512;
      __syncthreads();      // the last head's shares have been read
      shares[(wave * BH_WAVE + lane) * 2] = sk;
      shares[(wave * BH_WAVE + lane) * 2 + 1] = sq;
      __syncthreads();
      sk = sq = 0.f;
      for (int s = 0; s < slices; ++s) {
        const float* share = shares + ((wave % tiles + s * tiles) * BH_WAVE + lane) * 2;
        sk += share[0];
        sq += share[1];
      }
    }
    const float g = works ? gates[2 * i] : 0.f, beta = works ? gates[2 * i + 1] : 0.f;
    const bool real = works && column < vdim;
    sk *= k_scale;
    sq *= q_scale;
    const float u = real ? beta * (v_s[i * vdim + column] - g * sk) : 0.f, o = real ? fmaf(kq, u, g * sq) : 0.f;
    const float ku = k_scale * u;
    float* to = left + (size_t)head * dim * vdim;
    if (real) {
#pragma unroll
      for (int r = 0; r < R; ++r) {
        float* of_row = to + (size_t)(d0 + r) * vdim;
        if (d0 + r < dim) of_row[column] = fmaf(k_s[d0 + r], ku, g * S[r]);
      }
    }
    // the head's norm and gate
    const float ss = wave_sum(slice == 0 ? o * o : 0.f);
    __syncthreads();      // the last head's sums have been read
    if (lane == 0) squares[team * 4 + wave] = ss;
    __syncthreads();
    const float* parts = squares + team * 4;
    const float inv = 1.0f / sqrtf((parts[0] + parts[1] + parts[2] + parts[3]) / (float)vdim + eps);
    if (real && slice == 0) {
      const int at = head * vdim + column;
      out[bh_rows_index(out_block_rows, row, at, H * vdim)] = from_f32<T>(o * inv * norm[at] * dr_silu(to_f32(x[g_first + at])));
    }
  }
}

// Column tiles side by side for heads of vdim (0: delta_step does not take them), and rows of a column that a thread then keeps.
static int delta_step_tiles(int vdim) { return vdim <= 64 ? 1 : (vdim <= 128 ? 2 : (vdim <= 256 ? 4 : 0)); }
extern "C" int bh_delta_step_takes(int dim, int vdim) {
  const int tiles = delta_step_tiles(vdim);
  return dim > 0 && vdim > 0 && tiles > 0 && dim * tiles <= 4 * 128;
}

// One row a sequence: proj [n_seqs][row_stride] (dtype) as for delta_prep, g from g_first; norm f32 [H * vdim]; out [n_seqs][H * vdim] (dtype; rows or
// blocks of rows): the heads' read-outs over their root mean square, times norm, times silu(g).
extern "C" int bh_delta_step(const void* proj, int dtype, int row_stride, int first, int g_first, int b_first, int a_first, const float* conv, int taps,
                             float* state, long slot_stride, long conv_offset, const float* a_log, const float* dt_bias, const int32_t* seq_slot, const int32_t* seq_to,
                             const float* norm, float eps, void* out, int out_block_rows, int n_seqs, int H, int G, int dim, int vdim,
                             hipStream_t stream) {
  const DeltaRows in = {row_stride, first, b_first, a_first, conv, taps, state, slot_stride, conv_offset, a_log, dt_bias, H, G, dim, vdim};
  if (const char* fault = delta_fault(in)) return bh_fail("delta_step: %s", fault);
  BH_REQUIRE(n_seqs > 0 && G <= 65535 && g_first >= 0 && g_first + H * vdim <= row_stride, "delta_step: the gate lies outside its row");
  BH_REQUIRE(bh_delta_step_takes(dim, vdim), "delta_step: heads of %d x %d are not taken", dim, vdim);
  BH_REQUIRE(out_block_rows == 0 || ((out_block_rows == 8 || out_block_rows == 16) && (H * vdim) % 32 == 0 && dtype == BH_BF16),
             "delta_step: rows in blocks of %d of width %d are not written", out_block_rows, H * vdim);
  const int tiles = delta_step_tiles(vdim), slices = 4 / tiles, each = (dim + slices - 1) / slices;
  const int R = each <= 16 ? 16 : (each <= 32 ? 32 : (each <= 64 ? 64 : 128)), teams = H / G > 1 ? 2 : 1;
  const size_t lds = (size_t)(2 * R * slices + H / G * (vdim + 2) + 4 + teams * 516) * sizeof(float) + 16;
  BH_REQUIRE(lds <= 160 * 1024, "delta_step: %d heads of %d values to a group do not fit the local memory", H / G, vdim);
  const dim3 grid(n_seqs, G);
#define BH_DS_ONE(T, RR, TEAMS)                                                                                                      \
  do {                                                                                                                               \
    bh_allow_lds<delta_step_kernel<T, RR, TEAMS>>(lds);                                                                              \
    delta_step_kernel<T, RR, TEAMS><<<grid, 256 * TEAMS, lds, stream>>>((const T*)proj, in, g_first, seq_slot, seq_to, norm, eps, (T*)out,   \
                                                                        out_block_rows, tiles);                                      \
  } while (0)
#define BH_DS(T, RR)                          \
  do {                                        \
    if (teams == 2) BH_DS_ONE(T, RR, 2);      \
    else BH_DS_ONE(T, RR, 1);                 \
  } while (0)
#define BH_DS_R(T)                            \
  switch (R) {                                \
    case 16: BH_DS(T, 16); break;             \
    case 32: BH_DS(T, 32); break;             \
    case 64: BH_DS(T, 64); break;             \
    default: BH_DS(T, 128); break;            \
  }
  if (dtype == BH_F32) BH_DS_R(float)
  else if (dtype == BH_BF16) BH_DS_R(bf16_t)
  else return bh_fail("delta_step: unknown dtype %d", dtype);
#undef BH_DS_R
#undef BH_DS
#undef BH_DS_ONE
  return bh_check_launch("delta_step");
}
