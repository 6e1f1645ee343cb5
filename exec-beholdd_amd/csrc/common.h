// Shared definitions of the gfx950 kernel library: element types, conversions, wave and
// block reductions, error reporting.  Wavefronts are 64 lanes wide throughout.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "layout.h"

__device__ inline float to_f32(float x) { return x; }
__device__ inline float to_f32(bf16_t x) { return bf16_bits_to_f32(x.bits); }

template <typename T>
__device__ inline T from_f32(float x);
template <>
__device__ inline float from_f32<float>(float x) {
  return x;
}
template <>
__device__ inline bf16_t from_f32<bf16_t>(float x) {
  bf16_t r;
  r.bits = f32_to_bf16_bits(x);
  return r;
}

// ---- rows that are written in blocks of 16 ---------------------------------------------------------------
// A row puts 16 bytes into each 128-byte line of such a block; the line is whole when its eight rows are there.  Workgroups go to the
// eight XCDs in turn, each with an L2 of its own, so with a workgroup a row in order the eight parts of a line meet in no cache and
// go to memory as parts.  Kernels of a workgroup a row therefore take 16 neighbouring rows to an XCD: workgroup i's place on its XCD
// is i / 8.  The grid is made of whole rounds of 128 workgroups; those beyond the last row have nothing to do.
// Measured: rmsnorm of 8,160 rows of 4,096 70 -> 47 us, the squared ReLU of 2,048 x 6,144 23 -> 13, one stream's update and norm of
// 2,048 rows of 4,096 42 -> 24.
#define BH_ROWS_ROUND 128
inline bool bh_rows_spread(int n_rows, int block_rows) { return block_rows == 16 && n_rows >= BH_ROWS_ROUND; }
inline unsigned bh_rows_grid(int n_rows, int block_rows) {
  return bh_rows_spread(n_rows, block_rows) ? ((unsigned)n_rows + BH_ROWS_ROUND - 1) / BH_ROWS_ROUND * BH_ROWS_ROUND : (unsigned)n_rows;
}
// SPREAD: the grid is whole rounds.  The norms of few rows are compiled without any of it, which is 0.05 to 0.2 us of their 2.5 to 5.
template <bool SPREAD>
__device__ inline int bh_row_of_block() {
  if constexpr (!SPREAD) return blockIdx.x;
  const int place = blockIdx.x / 8;
  return (place / 16 * 8 + blockIdx.x % 8) * 16 + place % 16;
}
__device__ inline int bh_row_of_block(int block_rows) {
  return block_rows != 16 || gridDim.x % BH_ROWS_ROUND ? (int)blockIdx.x : bh_row_of_block<true>();
}
// KERNEL with its last template argument SPREAD as the rows want it; TO: the output's element type (only 2-byte ones lie in blocks).
#define BH_BY_ROWS(TO, n_rows, block_rows, threads, stream, ARGS, KERNEL, ...)                                         \
  do {                                                                                                                 \
    if constexpr (sizeof(TO) == 2) {                                                                                   \
      if (bh_rows_spread(n_rows, block_rows)) {                                                                        \
        KERNEL<__VA_ARGS__, true><<<bh_rows_grid(n_rows, block_rows), threads, 0, stream>>> ARGS;                      \
        break;                                                                                                         \
      }                                                                                                                \
    }                                                                                                                  \
    KERNEL<__VA_ARGS__, false><<<n_rows, threads, 0, stream>>> ARGS;                                                   \
  } while (0)

// ---- element-wise kernels in pieces of 16 bytes --------------------------------------------------------------
// A thread's 8 elements of bfloat16 are a chain of as many exponentials or stores: worth it from the size on at which an element a
// thread would keep the chip busy (1,536 threads a compute unit), not below it, where the chain is the time.  An element / a piece a
// thread, us: gated heads of 65 x 2,048 2.9 / 3.5, of 2,000 x 256 4.8 / 3.8 into blocks, clamped gate of 300 x 1,000 2.8 / 3.2, of
// 300 x 2,048 3.6 / 3.3, squared ReLU of 65 x 5,120 2.8 / 3.0, of 2,000 x 256 3.6 / 2.9 into blocks.  Four of float32 cost nothing.
int bh_compute_units();
inline bool bh_pieces_pay(long elements) { return elements >= 1536L * bh_compute_units(); }
// A row's pieces go to workgroups of up to four waves, of fewer where the row has no more (8,160 rows of 256, gelu 7.0 us with four).
inline unsigned bh_piece_threads(int pieces) { return pieces >= 256 ? 256u : ((unsigned)pieces + 63) / 64 * 64; }

// Four neighbouring elements in one store; `to` lies on the bytes of four of them.
__device__ inline void store_four(float* to, float a, float b, float c, float d) { *reinterpret_cast<float4*>(to) = make_float4(a, b, c, d); }
__device__ inline void store_four(bf16_t* to, float a, float b, float c, float d) {
  *reinterpret_cast<uint2*>(to) = make_uint2(f32_to_bf16_bits(a) | ((uint32_t)f32_to_bf16_bits(b) << 16),
                                             f32_to_bf16_bits(c) | ((uint32_t)f32_to_bf16_bits(d) << 16));
}

// The same as loads.
__device__ inline float4 load_four(const float* from) { return *reinterpret_cast<const float4*>(from); }
__device__ inline float4 load_four(const bf16_t* from) {
  const uint2 v = *reinterpret_cast<const uint2*>(from);
  return make_float4(bf16_bits_to_f32(v.x & 0xffff), bf16_bits_to_f32(v.x >> 16), bf16_bits_to_f32(v.y & 0xffff), bf16_bits_to_f32(v.y >> 16));
}

// Threads and pieces a thread of a row: a row on as many waves as have a piece each where the rows are few (their latency is the
// time), four pieces a thread where the rows fill the chip.
inline void bh_wide_row(int n_rows, int pieces, int* threads, int* per) {
  const int most = n_rows <= 64 ? 1024 : 256;
  *threads = pieces >= most ? most : (pieces + BH_WAVE - 1) / BH_WAVE * BH_WAVE;
  while ((pieces + *threads - 1) / *threads > 4 && *threads < 1024) *threads *= 2;
  *per = (pieces + *threads - 1) / *threads;
}

// ---- gated activations ----------------------------------------------------------------------
// act(gate) * up with act(g) = g / (1 + exp(-g (slope + cube g^2))): silu with slope 1 and cube 0, and with slope
// 2 sqrt(2/pi) and cube 2 sqrt(2/pi) 0.044715 the tanh form of GELU, since (1 + tanh(y)) / 2 = 1 / (1 + exp(-2y)).
// `squared`: no gate, but max(x, 0)^2 on a plain product's bfloat16 output.
struct GateForm {
  float slope, cube;
  bool squared = false;
};
#define GATED_CLAMPED 2      // what a launcher's `gated` says where the gate is a clamped one (1: any other)
enum BhGate { BH_GATE_SILU = 1, BH_GATE_GELU_TANH = 2 };
inline GateForm bh_gate_form(int gate) {
  return gate == BH_GATE_GELU_TANH ? GateForm{1.5957691216057308f, 1.5957691216057308f * 0.044715f} : GateForm{1.0f, 0.0f};
}
__device__ inline float relu_squared(float x) {
  const float v = fmaxf(x, 0.f);
  return v * v;
}
// CLAMPED: the gate is at most a limit, which stands in the place of `cube`, and up lies between its negative and itself and has one added
// (with the limit asked of `form` at each value, plain gated products of one row took 0.3 us more).
template <bool CLAMPED = false>
__device__ inline float gate_mul(float gate, float up, GateForm form) {
  if constexpr (CLAMPED) {
    gate = fminf(gate, form.cube);
    return gate / (1.0f + expf(-gate * form.slope)) * (fminf(fmaxf(up, -form.cube), form.cube) + 1.0f);
  }
  return gate / (1.0f + expf(-gate * fmaf(form.cube, gate * gate, form.slope))) * up;
}

// ---- what an attention kernel makes of the product of a query and a key --------------------------------
// s = scale t q.k, then cap tanh(s / cap) where there is a cap, then slopes[head] * (i - j) taken off, for a query at position i
// and a key at position j.  t = 1 + temp_coef ln(floor((i + 1) / temp_every) + 1) where temp_every is given: a query counts the more
// the later it stands.
struct ScoreForm {
  float scale;
  float cap;             // 0: none
  const float* slopes;   // [heads] or null
  float temp_coef;
  int temp_every;        // 0: none
  // Whether a score is its product times a positive factor of the query: then the largest product has the largest score, and the
  // matrix-core kernels take the factor into the exponential instead of making the scores (2,048 rows, 32 heads of 128 on 8, which
  // count the more the later they stand: 76 -> 53 us).  A factor that falls with the position may turn negative, and one of zero makes
  // NaN of it: keys that are not seen stand at minus infinity, and nothing was summed before the first.
  BH_BOTH bool scaled_only() const { return cap == 0.f && slopes == nullptr && scale > 0.f && (temp_every == 0 || temp_coef >= 0.f); }
};
// What the matrix-core kernels are compiled for: 0 scaled products only, 1 a factor and a distance's share, 2 a cap as well (asked of a number
// at each score, both ways were made: 2,048 rows, 32 heads of 128 on 8 with slopes 79 -> 60 us, with a cap 93 -> 70).
inline int bh_formed(const ScoreForm& form) { return form.scaled_only() ? 0 : form.cap > 0.f ? 2 : 1; }
__device__ inline float query_scale(const ScoreForm& form, int position) {
  if (form.temp_every == 0) return form.scale;
  return form.scale * (1.0f + form.temp_coef * logf((float)((position + 1) / form.temp_every) + 1.0f));
}
inline const char* bh_score_form_fault(const ScoreForm& form) {
  if (!(form.cap >= 0.f)) return "a cap on the scores is positive, or 0 for none";
  if (form.temp_every < 0) return "a temperature step is a positive count of positions, or 0 for none";
  return nullptr;
}

// ---- what an attention kernel does where a (row, head)'s sum is finished ---------------------------
struct HeadEnd {
  const float* sinks;   // [heads] or null: exp(sinks[head]) is one more term of the head's softmax sums, without key and value
  const void* gates;    // [rows][gate_stride] in the activations' type, or null: a finished head times sigmoid(gates[row][head])
  int gate_stride;
  float scale = 1.0f;   // a finished head times this
};
template <typename T>
__device__ inline float head_gate(const HeadEnd& end, int row, int head) {
  if (end.gates == nullptr) return end.scale;
  return end.scale / (1.0f + expf(-to_f32(reinterpret_cast<const T*>(end.gates)[(size_t)row * end.gate_stride + head])));
}

// ---- reductions -------------------------------------------------------------------------

__device__ inline float wave_sum(float v) {
#pragma unroll
  for (int off = BH_WAVE / 2; off > 0; off >>= 1) v += __shfl_xor(v, off, BH_WAVE);
  return v;
}

__device__ inline float wave_max(float v) {
#pragma unroll
  for (int off = BH_WAVE / 2; off > 0; off >>= 1) v = fmaxf(v, __shfl_xor(v, off, BH_WAVE));
  return v;
}

// Block-wide sum; `scratch` holds at least blockDim.x / 64 floats.  Every thread gets the result.
__device__ inline float block_sum(float v, float* scratch) {
  const int lane = threadIdx.x & (BH_WAVE - 1), wave = threadIdx.x / BH_WAVE;
  const int n_waves = (blockDim.x + BH_WAVE - 1) / BH_WAVE;
  v = wave_sum(v);
  __syncthreads();
  if (lane == 0) scratch[wave] = v;
  __syncthreads();
  float total = 0.f;
  for (int i = 0; i < n_waves; ++i) total += scratch[i];
  return total;
}

__device__ inline float block_max(float v, float* scratch) {
  const int lane = threadIdx.x & (BH_WAVE - 1), wave = threadIdx.x / BH_WAVE;
  const int n_waves = (blockDim.x + BH_WAVE - 1) / BH_WAVE;
  v = wave_max(v);
  __syncthreads();
  if (lane == 0) scratch[wave] = v;
  __syncthreads();
  float total = scratch[0];
  for (int i = 1; i < n_waves; ++i) total = fmaxf(total, scratch[i]);
  return total;
}

// ---- errors ------------------------------------------------------------------------------

// Every entry point returns 0 on success; otherwise bh_last_error() gives the reason.
int bh_fail(const char* format, ...);
int bh_check_launch(const char* what);
// The compute units of the GPU that is current when it is first asked (256 on an MI355X): what launch plans count
// workgroups against.  Where no GPU is visible (a byte plan made on another machine) it says 256.
int bh_compute_units();

// Lets KERNEL use `bytes` of dynamic LDS where that is more than the 48 KB a kernel may use unasked.  The runtime is told
// once per kernel and size (the first, eager run of a step): nothing is asked of it while a stream captures a graph.
template <auto KERNEL>
inline void bh_allow_lds(size_t bytes) {
  static size_t allowed = 48 * 1024;
  if (bytes > allowed) {
    (void)hipFuncSetAttribute((const void*)KERNEL, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
    allowed = bytes;
  }
}

#define BH_REQUIRE(cond, ...)                  \
  do {                                         \
    if (!(cond)) return bh_fail(__VA_ARGS__);  \
  } while (0)

// The cache of one layer as the kernels see it: pages of BH_PAGE tokens found through a
// per-sequence page table.  Keys lie [page][kv_head][token in page][head_dim]; values lie
// transposed, [page][kv_head][head_dim][token in page], so that a matrix-core operand of
// "head_dim rows x consecutive tokens" is a contiguous load.
