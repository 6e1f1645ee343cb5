// Matrix products of float32 operands on the float32 matrix instructions: C[M, N] (+)= A[M, K] W[N, K]^T, and for few rows the gated
// form out[M, F] = act(A W[:F]^T) * (A W[F:]^T).  Every product is a 32-bit fused multiply-add with a 32-bit sum, as in the plain FMA
// kernel (generic.hip); only the order of the sums differs, and it is blocked here as there.
//
// Three kernels.  Up to 32 rows (decode steps, short steps) a product is its weights, read once: `gemm_f32_few`, gated or not.  More rows are
// matrix-core work: `gemm_f32_ring` where K is a multiple of 32 and not short, else `gemm_f32_tiles`; gated products are followed by an activation of
// their own.
#include "common.h"
#include "gemm_f32.h"
#include <type_traits>

// s_waitcnt of gfx9 (vmcnt in bits 3:0 and 15:14, expcnt 6:4, lgkmcnt 11:8): all LDS reads are back, and at most `vm` of the wave's
// global loads are still on their way.  F32_MEET: every wave has waited; nothing may be moved across it by the compiler.
#define F32_WAIT(vm) __builtin_amdgcn_s_waitcnt(((vm) & 15) | (((vm) >> 4) << 14) | (7 << 4) | (0 << 8))
#define F32_MEET()                        \
  do {                                    \
    __builtin_amdgcn_sched_barrier(0);    \
    __builtin_amdgcn_s_barrier();         \
    __builtin_amdgcn_sched_barrier(0);    \
  } while (0)

typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef float floatx16 __attribute__((ext_vector_type(16)));

__device__ static inline floatx4 load4(const float* p) { return *reinterpret_cast<const floatx4*>(p); }

// ---- few rows ------------------------------------------------------------------------------------------
// v_mfma_f32_4x4x1_16B multiplies 16 independent 4 x 4 blocks: lane 4 b + i holds row i of block b of either operand.  A block is
// a slice of k here: lane 4 b + i loads 16 bytes of weight row i at k = k0 + 4 b, so that a wave's load covers four rows of 256
// contiguous bytes, the next four products take their four elements in turn, and the 16 blocks' sums (every 16th group of four k)
// are added at the end, then those of the workgroup's waves, which share K.  The activations are loaded the same way, from the L2.
// Bound by the weights' stream; against 64 bits the sum of K terms is one of K / (16 WAVES) and one of 16 WAVES.
// Measured at 4 rows: 1,024 x 3,072 in 6.5 us and 32,768 x 1,024 in 29 us (4.6 TB/s); the FMA tiles of generic.hip, whose
// workgroups of 64 weight rows do 16 times the products and number 16 there, took 150 to 290 us.
//   R: groups of four weight rows a wave, C: groups of four activation rows, WAVES: waves that share K.
// NORM: the activations are the rows of a float32 residual, and the product is that of their RMSNorm: every workgroup reads all of them
// anyway, multiplies what it loads by the norm's weight, sums its squares beside the products and multiplies what comes out by the row's
// 1 / sqrt(mean + eps).  That is a launch less in front of every such product (4 rows of 1,024: 4.7 us in a chain of decode steps, of which
// 0.2 come back in the product of 2,048 x 1,024 and 1.2 in the gated one of 3,072 x 1,024; 16 tokens for four prompts 10.05 -> 9.4 ms).
struct RowNorm {
  const float* weight;   // [K]
  float eps;
};
template <int R, int C, int WAVES, bool GATED, bool NORM>
__global__ __launch_bounds__(64 * WAVES) void gemm_f32_few_kernel(const float* __restrict__ a, const float* __restrict__ w,
                                                                  float* __restrict__ c, int M, int N, int K, int accumulate,
                                                                  GateForm form, RowNorm norm) {
  constexpr int GROUPS = GATED ? R / 2 : R;   // groups of outputs; GATED: the first half of the R groups are gates, the rest ups
  constexpr int U = C >= 4 ? 2 : 4;           // chunks of 64 k whose loads are in flight together
  __shared__ float sums[WAVES][R * C][16];
  __shared__ float squares[NORM ? WAVES : 1][4 * C];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, i = lane & 3, b = lane >> 2;
  const int n0 = blockIdx.x * 4 * GROUPS;
  const float* w_row[R];
  const float* a_row[C];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int n = min(n0 + 4 * (r % GROUPS) + i, N - 1);      // rows beyond the last one repeat it and are not written
    w_row[r] = w + (size_t)(GATED && r >= GROUPS ? N + n : n) * K + 4 * b;
  }
#pragma unroll
  for (int j = 0; j < C; ++j) a_row[j] = a + (size_t)min(4 * j + i, M - 1) * K + 4 * b;
  floatx4 acc[R][C] = {};
  float square[C] = {};
  auto multiply = [&](const floatx4 (&wv)[R], floatx4 (&av)[C], floatx4 gain) {
    if constexpr (NORM) {
#pragma unroll
      for (int j = 0; j < C; ++j) {
        float ss = 0.f;
#pragma unroll
        for (int t = 0; t < 4; ++t) ss = fmaf(av[j][t], av[j][t], ss), av[j][t] *= gain[t];
        square[j] += ss;
      }
    }
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int r = 0; r < R; ++r)
#pragma unroll
        for (int j = 0; j < C; ++j) acc[r][j] = __builtin_amdgcn_mfma_f32_4x4x1f32(wv[r][t], av[j][t], acc[r][j], 0, 0, 0);
  };
  int k0 = 64 * wave;
  for (; k0 + 64 * WAVES * (U - 1) + 64 <= K; k0 += 64 * WAVES * U) {
    floatx4 wv[U][R], av[U][C], gain[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
#pragma unroll
      for (int r = 0; r < R; ++r) wv[u][r] = load4(w_row[r] + k0 + 64 * WAVES * u);
#pragma unroll
      for (int j = 0; j < C; ++j) av[u][j] = load4(a_row[j] + k0 + 64 * WAVES * u);
      if constexpr (NORM) gain[u] = load4(norm.weight + 4 * b + k0 + 64 * WAVES * u);
    }
#pragma unroll
    for (int u = 0; u < U; ++u) multiply(wv[u], av[u], NORM ? gain[u] : floatx4{});
  }
  if (k0 < K) {      // what is left, all of it asked for at once as well
    const floatx4 zero = {0.f, 0.f, 0.f, 0.f};
    floatx4 wv[U][R], av[U][C], gain[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int k = k0 + 64 * WAVES * u;
      const bool inside = k + 4 * b < K;       // K is a multiple of 4
#pragma unroll
      for (int r = 0; r < R; ++r) wv[u][r] = inside ? load4(w_row[r] + k) : zero;
#pragma unroll
      for (int j = 0; j < C; ++j) av[u][j] = inside ? load4(a_row[j] + k) : zero;
      if constexpr (NORM) gain[u] = inside ? load4(norm.weight + 4 * b + k) : zero;
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (k0 + 64 * WAVES * u < K) multiply(wv[u], av[u], NORM ? gain[u] : floatx4{});
  }
  if constexpr (NORM) {
#pragma unroll
    for (int j = 0; j < C; ++j) {
#pragma unroll
      for (int off = 4; off < BH_WAVE; off <<= 1) square[j] += __shfl_xor(square[j], off, BH_WAVE);
      if (lane < 4) squares[wave][4 * j + lane] = square[j];
    }
  }
  // a lane's four numbers are rows 0..3 of its block's result, column i.  Over the blocks: halves of the lanes take half of the
  // rows each, twice, then the rest of the blocks are added, so that lane 32 h + 16 q + .. + i holds row 2 h + q, column i.
  const bool high = lane & 32, odd = lane & 16;
#pragma unroll
  for (int r = 0; r < R; ++r)
#pragma unroll
    for (int j = 0; j < C; ++j) {
      const floatx4 v = acc[r][j];
      const float x0 = (high ? v[2] : v[0]) + __shfl_xor(high ? v[0] : v[2], 32, BH_WAVE);
      const float x1 = (high ? v[3] : v[1]) + __shfl_xor(high ? v[1] : v[3], 32, BH_WAVE);
      float x = (odd ? x1 : x0) + __shfl_xor(odd ? x0 : x1, 16, BH_WAVE);
      x += __shfl_xor(x, 8, BH_WAVE);
      x += __shfl_xor(x, 4, BH_WAVE);
      if ((lane & 12) == 0) sums[wave][r * C + j][4 * (lane >> 4) + i] = x;
    }
  __syncthreads();
  for (int e = threadIdx.x; e < GROUPS * C * 16; e += 64 * WAVES) {
    const int row = e % (4 * GROUPS), m = e / (4 * GROUPS);   // neighbouring threads: neighbouring outputs of one activation row
    const int n = n0 + row;
    if (n >= N || m >= M) continue;
    const int place = 4 * (row % 4) + m % 4, at = (row / 4) * C + m / 4;
    float v = 0.f;
#pragma unroll
    for (int s = 0; s < WAVES; ++s) v += sums[s][at][place];
    float factor = 1.f;
    if constexpr (NORM) {
      float ss = 0.f;
#pragma unroll
      for (int s = 0; s < WAVES; ++s) ss += squares[s][m];
      factor = 1.0f / sqrtf(ss / (float)K + norm.eps);
      v *= factor;
    }
    if (GATED) {
      float up = 0.f;
#pragma unroll
      for (int s = 0; s < WAVES; ++s) up += sums[s][at + GROUPS * C][place];
      v = gate_mul(v, up * factor, form);
    }
    const size_t to = (size_t)m * N + n;
    c[to] = accumulate ? v + c[to] : v;
  }
}

// ---- many rows, K a multiple of 32 ---------------------------------------------------------------------
// A workgroup of four waves owns 32 WM x 32 WN outputs, a wave 32 x 32 of them for one of KG shares of k (WM WN KG = 4): the fewer the
// outputs, the more of the waves share k, so that few rows fill the chip too.  Slices of 32 k go from global memory straight to LDS
// (1 KB a load: eight whole rows of a slice) into a ring of R, R steps ahead; a step's operands are read from LDS into registers while
// the step before is multiplied.  The 16-byte piece c of row r of a slice lies at place c ^ (r % 8) of the row's eight, so that the
// eight rows that a read takes at a time lie in different banks.  A slice is summed on its own and then added, as below, the even and
// the odd ones apart: error against 64 bits of 744 rows of 6,144 x 1,024 1.31e-7 (below 1.48e-7), of 1,024 x 3,072 1.67e-7 on both.
// Bound by the matrix instructions (64 cycles an instruction, 16 a slice and wave), the last round of workgroups, and their start.
template <int WM, int WN, int KG, int R, bool ACCUMULATE>
__global__ __launch_bounds__(256, KG == 4 ? 1 : 2) void gemm_f32_ring_kernel(const float* __restrict__ a, const float* __restrict__ w,
                                                                             float* __restrict__ c, int M, int N, int K) {
  static_assert(WM * WN * KG == 4 && R >= 3, "four waves; a step's loads, the next one's and one more");
  constexpr int WAVES = WM * WN, A_PIECES = 4 * WM, PIECES = 4 * (WM + WN), EACH = PIECES / WAVES;
  // one array: before a read from one of several the compiler waits for all loads on their way to that one
  __shared__ __attribute__((aligned(16))) floatx4 ring[KG * R * PIECES * 64];      // [share][step in turn][8 rows of A, then of W][lane]
  const int lane = threadIdx.x & 63, wave_of_all = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wave = wave_of_all % WAVES, share = wave_of_all / WAVES, wm = wave / WN, wn = wave % WN;
  const int m0 = blockIdx.y * 32 * WM, n0 = blockIdx.x * 32 * WN, steps = K / 32 / KG;
  const float* from[EACH];
#pragma unroll
  for (int i = 0; i < EACH; ++i) {
    const int piece = wave * EACH + i, row = 8 * (piece < A_PIECES ? piece : piece - A_PIECES) + lane / 8;      // rows beyond the last one repeat it
    from[i] = (piece < A_PIECES ? a + (size_t)min(m0 + row, M - 1) * K : w + (size_t)min(n0 + row, N - 1) * K) + 32 * share +
              4 * ((lane & 7) ^ (lane / 8));
  }
  auto ask = [&](int i, int step, int place) {
    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(from[i] + (size_t)step * (32 * KG)),
                                     (__attribute__((address_space(3))) void*)&ring[((share * R + place) * PIECES + wave * EACH + i) * 64], 16, 0, 0);
  };
  const int half = lane >> 5, row = lane & 31;
  int at[4];      // the lane's pieces of its row, one for every 8 k
#pragma unroll
  for (int t = 0; t < 4; ++t) at[t] = (row / 8) * 64 + (row & 7) * 8 + ((2 * t + half) ^ (row & 7));
  for (int j = 0; j < R && j < steps; ++j) {
#pragma unroll
    for (int i = 0; i < EACH; ++i) ask(i, j, j);
  }
  F32_WAIT(0);
  F32_MEET();
  floatx4 av[2][4], wv[2][4];      // the operands of an even and of an odd step
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    av[0][t] = ring[(share * R * PIECES + 4 * wm) * 64 + at[t]];
    wv[0][t] = ring[(share * R * PIECES + A_PIECES + 4 * wn) * 64 + at[t]];
  }
  // the sums of even and of odd steps, added at the end; a step's own sum is added while the next step's is made
  floatx16 sum[2] = {}, part[2] = {};
  int place = 0;                         // of the step that is multiplied
  // Step j: its operands are in registers or on their way there, and every wave has waited for its reads of them before the barrier, so
  // step j + R may take their place.  STEADY: it does, and what step j + 1 needs was asked for before the loads of the R - 2 steps
  // behind it; otherwise (the last R steps) everything asked for is waited for.
  auto multiply = [&](int j, auto odd, auto steady) {
    constexpr int U = decltype(odd)::value;
    constexpr bool STEADY = decltype(steady)::value;
    if (STEADY) F32_WAIT(EACH * (R - 2));
    else F32_WAIT(0);
    F32_MEET();
    const int next = place == R - 1 ? 0 : place + 1, base = (share * R + next) * PIECES;
    if (!STEADY && j + R < steps) {
#pragma unroll
      for (int i = 0; i < EACH; ++i) ask(i, j + R, place);
    }
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      // (beyond the last step this reads what an earlier one has left there, and nobody uses it)
      av[1 - U][t] = ring[(base + 4 * wm) * 64 + at[t]];
      wv[1 - U][t] = ring[(base + A_PIECES + 4 * wn) * 64 + at[t]];
      if (STEADY) {
#pragma unroll
        for (int i = 0; i < EACH; ++i)
          if (i * 4 / EACH == t) ask(i, j + R, place);
      }
#pragma unroll
      for (int e = 0; e < 4; ++e)
        part[U] = __builtin_amdgcn_mfma_f32_32x32x2f32(av[U][t][e], wv[U][t][e], t + e == 0 ? floatx16{} : part[U], 0, 0, 0);
#pragma unroll
      for (int e = 0; e < 4; ++e) sum[1 - U][4 * t + e] += part[1 - U][4 * t + e];
      __builtin_amdgcn_sched_barrier(0);
    }
    place = next;
  };
  const std::integral_constant<int, 0> even;
  const std::integral_constant<int, 1> odd;
  int j = 0;
  for (; j + 1 + R < steps; j += 2) {
    multiply(j, even, std::true_type());
    multiply(j + 1, odd, std::true_type());
  }
  for (; j + 1 < steps; j += 2) {
    multiply(j, even, std::false_type());
    multiply(j + 1, odd, std::false_type());
  }
  if (j < steps) multiply(j, even, std::false_type());
  if (steps % 2) sum[0] += part[0];
  else sum[1] += part[1];
  floatx16 acc = sum[0] + sum[1];
  if constexpr (KG > 1) {      // the shares' sums, lane by lane
    F32_WAIT(0);
    F32_MEET();
    floatx16* sums = reinterpret_cast<floatx16*>(ring) + wave * 64 + lane;
    if (share > 0) sums[(share - 1) * WAVES * 64] = acc;
    __syncthreads();
    if (share > 0) return;
#pragma unroll
    for (int s = 0; s < KG - 1; ++s) acc += sums[s * WAVES * 64];
  }
  const int n = n0 + 32 * wn + row;
  if (n >= N) return;
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const int m = m0 + 32 * wm + 8 * (r >> 2) + 4 * half + (r & 3);
    if (m >= M) continue;
    const size_t to = (size_t)m * N + n;
    c[to] = ACCUMULATE ? acc[r] + c[to] : acc[r];
  }
}
#undef F32_WAIT
#undef F32_MEET

// ---- many rows, any K ----------------------------------------------------------------------------------
// Four waves own 64 B x 64 B outputs (B = 1 or 2), a wave B x B tiles of v_mfma_f32_32x32x2_f32; a workgroup is one such group, or
// KG of them that take the slices of k in turn (B = 1).  Slices of 32 k go through two LDS buffers, the next slice's loads on their way
// while one is multiplied.  A row of a slice takes 36 floats of LDS, so that the 16-byte reads of 16 neighbouring rows fall on different
// banks; lane (row, half) reads four k at once and the matrix instructions take k in that order, the same for both operands.  Every slice
// is summed on its own and then added.
// Bound by the matrix instructions (64 cycles a tile and two k) where the tiles fill the chip.
// Measured: 695 x 6,144 x 1,024 in 104 us (84 TFLOP/s), 2,048 x 32,768 x 1,024 in 1.12 ms (122 TFLOP/s; a library product of 8,192
// cubed reaches 154); 695 x 1,024 x 3,072 in 70 us, 87 with one group of waves a workgroup.
#define F32_SLICE 32
#define F32_STRIDE 36

template <int B, int KG, bool ACCUMULATE>
__global__ __launch_bounds__(256 * KG) void gemm_f32_tiles_kernel(const float* __restrict__ a, const float* __restrict__ w,
                                                                  float* __restrict__ c, int M, int N, int K) {
  constexpr int TILE = 64 * B, LOADS = TILE / 32;
  __shared__ __attribute__((aligned(16))) float slices[KG][2][2][TILE * F32_STRIDE];   // [group][buffer][activations, weights]
  const int tid = threadIdx.x & 255, lane = tid & 63, wave = tid >> 6, group = threadIdx.x >> 8;
  auto& lds = slices[group];
  const int m0 = blockIdx.y * TILE, n0 = blockIdx.x * TILE;
  const int l_row = tid >> 3, l_k = 4 * (tid & 7);
  const float *a_from[LOADS], *w_from[LOADS];
#pragma unroll
  for (int s = 0; s < LOADS; ++s) {
    a_from[s] = a + (size_t)min(m0 + l_row + 32 * s, M - 1) * K + l_k;
    w_from[s] = w + (size_t)min(n0 + l_row + 32 * s, N - 1) * K + l_k;
  }
  floatx4 next_a[LOADS], next_w[LOADS];
  auto fetch = [&](int k0) {
    const bool inside = k0 + l_k < K;      // K is a multiple of 4
#pragma unroll
    for (int s = 0; s < LOADS; ++s) {
      next_a[s] = inside ? load4(a_from[s] + k0) : floatx4{0.f, 0.f, 0.f, 0.f};
      next_w[s] = inside ? load4(w_from[s] + k0) : floatx4{0.f, 0.f, 0.f, 0.f};
    }
  };
  auto put = [&](int buffer) {
#pragma unroll
    for (int s = 0; s < LOADS; ++s) {
      *reinterpret_cast<floatx4*>(&lds[buffer][0][(l_row + 32 * s) * F32_STRIDE + l_k]) = next_a[s];
      *reinterpret_cast<floatx4*>(&lds[buffer][1][(l_row + 32 * s) * F32_STRIDE + l_k]) = next_w[s];
    }
  };
  const int wm = (wave >> 1) * 32 * B, wn = (wave & 1) * 32 * B;
  const int half = lane >> 5, at_row = lane & 31;
  floatx16 acc[B][B] = {};
  fetch(F32_SLICE * group);
  put(0);
  __syncthreads();
  int buffer = 0;
  for (int k0 = 0; k0 < K; k0 += KG * F32_SLICE, buffer ^= 1) {     // every group as often; a slice beyond K is zeros
    const bool more = k0 + KG * F32_SLICE < K;
    if (more) fetch(k0 + (KG + group) * F32_SLICE);
    const float* as = &lds[buffer][0][(wm + at_row) * F32_STRIDE + 4 * half];
    const float* ws = &lds[buffer][1][(wn + at_row) * F32_STRIDE + 4 * half];
    floatx16 part[B][B] = {};
#pragma unroll
    for (int kk = 0; kk < F32_SLICE; kk += 8) {
      floatx4 av[B], wv[B];
#pragma unroll
      for (int x = 0; x < B; ++x) {
        av[x] = load4(as + 32 * x * F32_STRIDE + kk);
        wv[x] = load4(ws + 32 * x * F32_STRIDE + kk);
      }
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int x = 0; x < B; ++x)
#pragma unroll
          for (int y = 0; y < B; ++y) part[x][y] = __builtin_amdgcn_mfma_f32_32x32x2f32(av[x][t], wv[y][t], part[x][y], 0, 0, 0);
    }
#pragma unroll
    for (int x = 0; x < B; ++x)
#pragma unroll
      for (int y = 0; y < B; ++y) acc[x][y] += part[x][y];
    if (more) put(buffer ^ 1);     // its readers passed the barrier that ended the slice before
    __syncthreads();
  }
  if constexpr (KG > 1) {          // the groups' sums, lane by lane, through their own slices' memory
    floatx16* mine = reinterpret_cast<floatx16*>(&slices[group][0][0][0]) + tid;
    if (group > 0) *mine = acc[0][0];
    __syncthreads();
    if (group > 0) return;
#pragma unroll
    for (int s = 1; s < KG; ++s) acc[0][0] += *(reinterpret_cast<const floatx16*>(&slices[s][0][0][0]) + tid);
  }
#pragma unroll
  for (int x = 0; x < B; ++x)
#pragma unroll
    for (int y = 0; y < B; ++y) {
      const int n = n0 + wn + 32 * y + at_row;
      if (n >= N) continue;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int m = m0 + wm + 32 * x + 8 * (r >> 2) + 4 * half + (r & 3);
        if (m >= M) continue;
        const size_t to = (size_t)m * N + n;
        c[to] = ACCUMULATE ? acc[x][y][r] + c[to] : acc[x][y][r];
      }
    }
}

// ---- which products go where ---------------------------------------------------------------------------

bool bh_gemm_f32_takes(const void* a, const void* w, const void* c, int K) {
  return K % 4 == 0 && (((uintptr_t)a | (uintptr_t)w) % 16) == 0 && ((uintptr_t)c % 4) == 0;
}

template <int R, int C, bool GATED, bool NORM>
static void few_waves(const float* a, const float* w, float* c, int M, int N, int K, int accumulate, GateForm form, RowNorm norm, hipStream_t stream) {
  const int outputs = 4 * (GATED ? R / 2 : R), blocks = (N + outputs - 1) / outputs;
  if constexpr (R == 4) {
    // Many rows: a wave alone walks all of K, so that its loads run on behind one another (32,768 x 1,024 at 32 rows 61 us, 105
    // where four waves share K), as long as that leaves four workgroups a compute unit.
    if (blocks >= 4 * bh_compute_units()) {
      gemm_f32_few_kernel<R, C, 1, GATED, NORM><<<blocks, 64, 0, stream>>>(a, w, c, M, N, K, accumulate, form, norm);
      return;
    }
  } else if constexpr (!NORM || C < 8) {      // (norms of more than 16 rows: short K only, bh_gemm_f32_takes_norm)
    // Eight waves share a long K where four would leave a compute unit with fewer than two workgroups.
    if (K >= 2048 && blocks < 2 * bh_compute_units()) {
      gemm_f32_few_kernel<R, C, 8, GATED, NORM><<<blocks, 512, 0, stream>>>(a, w, c, M, N, K, accumulate, form, norm);
      return;
    }
  }
  gemm_f32_few_kernel<R, C, 4, GATED, NORM><<<blocks, 256, 0, stream>>>(a, w, c, M, N, K, accumulate, form, norm);
}

template <int R, bool GATED, bool NORM = false>
static void few_rows(const float* a, const float* w, float* c, int M, int N, int K, int accumulate, GateForm form, hipStream_t stream,
                     RowNorm norm = RowNorm{}) {
  if (M <= 4) few_waves<R, 1, GATED, NORM>(a, w, c, M, N, K, accumulate, form, norm, stream);
  else if (M <= 8) few_waves<R, 2, GATED, NORM>(a, w, c, M, N, K, accumulate, form, norm, stream);
  else if (M <= 16) few_waves<R, 4, GATED, NORM>(a, w, c, M, N, K, accumulate, form, norm, stream);
  else few_waves<R, 8, GATED, NORM>(a, w, c, M, N, K, accumulate, form, norm, stream);
}

int bh_gemm_f32(const float* a, const float* w, float* c, int accumulate, int M, int N, int K, hipStream_t stream) {
  const int units = bh_compute_units();
  if (M <= BH_F32_FEW_ROWS) {
    const GateForm none = {0.f, 0.f};
    // as many weight rows a workgroup as leave two workgroups a compute unit
    if (N >= 32 * units) few_rows<4, false>(a, w, c, M, N, K, accumulate, none, stream);
    else if (N >= 16 * units) few_rows<2, false>(a, w, c, M, N, K, accumulate, none, stream);
    else few_rows<1, false>(a, w, c, M, N, K, accumulate, none, stream);
    return bh_check_launch("gemm_f32_few");
  }
  // Few slices in more than one round: a workgroup of the ring pays for its start (three slices asked for, the shares' sums) what it saves
  // behind it, and the tiles are ahead where they are not the wide ones.  Ring / tiles, us: 4,096 rows of 1,024 x 32 11.6 / 9.8, x 128
  // 22.4 / 19.7, x 192 26.6 / 25.7, x 256 29.4 / 30.4; 600 of 4,096 x 128 18.4 / 13.8, x 192 21.3 / 17.8; 1,500 of 1,024 x 64 10.0 / 7.9; one
  // round, 1,000 of 1,024 x 64 6.4 / 6.4, 300 of 1,024 x 128 6.2 / 7.1; wide ones, 4,096 of 4,096 x 128 64 / 83.
  const long wide = (long)((N + 127) / 128) * ((M + 127) / 128);      // tiles of 128 x 128
  const bool short_k = K < 256 && (long)((N + 63) / 64) * ((M + 63) / 64) > units && wide < 4L * units;
  if (K % 32 == 0 && !short_k && (M + 31) / 32 <= 65535) {
    // The waves' split with the least estimated time: rounds of workgroups, one a compute unit at a time (two share it and take as long),
    // of so many slices at what a slice takes, and the start; a smaller tile has to be 5 % ahead, for it reads more.  64 x 64 / 32 x 64 /
    // 32 x 32 outputs, us, weights from memory (1 to 3 % less than now, before the sums of even and odd steps were kept apart), in
    // brackets the tiles of gemm_f32_tiles: 744 rows of 6,144 x 1,024 104 / 106 / 173 (120), of 2,048 x 1,024 42 / 38 / 55 (49), of
    // 1,024 x 3,072 66 / 67 / 72 (75); 1,500 of 1,024 x 3,072 112 / 97 / 139 (132); 300 of 1,024 x 3,072 63 / 38 / 48 (74); 100 of it
    // 60 / 35 / 22 (71); 64 of 3,000 x 1,024 22 / 14 / 11 (26); 3,200 of 6,144 x 1,024 334 / 373 / 629 (392); 2,048 of 4,096 x 4,096
    // 563 / 608 / 803 (620), 122 TFLOP/s.
    const auto rounds = [&](int rows, int columns) {
      return (double)(((long)((M + rows - 1) / rows) * ((N + columns - 1) / columns) + units - 1) / units);
    };
    const double whole = rounds(64, 64) * ((K / 32) * 0.58 + 1.0) + 3.0;
    const double in_two = K % 64 ? 1e30 : rounds(32, 64) * ((K / 64) * 0.64 + 1.0) + 3.0;
    const double in_four = K % 128 ? 1e30 : rounds(32, 32) * ((K / 128) * 0.75 + 4.0);
#define BH_F32_RING(WM, WN, KG, R)                                                                                                 \
  do {                                                                                                                             \
    const dim3 grid((N + 32 * WN - 1) / (32 * WN), (M + 32 * WM - 1) / (32 * WM));                                                 \
    if (accumulate) gemm_f32_ring_kernel<WM, WN, KG, R, true><<<grid, 256, 0, stream>>>(a, w, c, M, N, K);                         \
    else gemm_f32_ring_kernel<WM, WN, KG, R, false><<<grid, 256, 0, stream>>>(a, w, c, M, N, K);                                   \
    return bh_check_launch("gemm_f32_ring");                                                                                       \
  } while (0)
    if (in_four < 0.95 * in_two && in_four < 0.95 * whole) BH_F32_RING(1, 1, 4, 4);      // rings of 128, 72 and 48 KB
    if (in_two < 0.95 * whole) BH_F32_RING(1, 2, 2, 3);
    BH_F32_RING(2, 2, 1, 3);
#undef BH_F32_RING
  }
  // Other K, and those few slices.
  // Tiles of 128 x 128 read half as much a product, but only four of them a compute unit and more level out (695 x 6,144 x 1,024,
  // 1.1 a unit: 141 us, 104 in tiles of 64 x 64); where tiles of 64 x 64 are not even two a unit, a second group of waves hides the
  // first one's waits for its slices.
  const bool big = wide >= 4L * units;
  const int tile = big ? 128 : 64;
  BH_REQUIRE((M + tile - 1) / tile <= 65535, "gemm: M=%d needs more than 65535 row tiles", M);
  const dim3 grid((N + tile - 1) / tile, (M + tile - 1) / tile);
  const bool groups = (long)grid.x * grid.y < 2L * units && K >= 4 * F32_SLICE;
#define BH_F32_TILES(B, KG)                                                                                          \
  do {                                                                                                               \
    if (accumulate) gemm_f32_tiles_kernel<B, KG, true><<<grid, 256 * KG, 0, stream>>>(a, w, c, M, N, K);             \
    else gemm_f32_tiles_kernel<B, KG, false><<<grid, 256 * KG, 0, stream>>>(a, w, c, M, N, K);                       \
  } while (0)
  if (big) BH_F32_TILES(2, 1);
  else if (groups) BH_F32_TILES(1, 2);
  else BH_F32_TILES(1, 1);
#undef BH_F32_TILES
  return bh_check_launch("gemm_f32_tiles");
}

// The gated form of few rows in one launch.  bh_gemm_f32_takes_gated: whether these sizes go (else: the product, then its activation).
extern "C" int bh_gemm_f32_takes_gated(int M, int F, int K) { return M > 0 && M <= BH_F32_FEW_ROWS && F > 0 && K > 0 && K % 4 == 0 ? 1 : 0; }
extern "C" int bh_gemm_f32_gated(const float* a, const float* w, float* out, int M, int F, int K, int gate, hipStream_t stream) {
  BH_REQUIRE(bh_gemm_f32_takes_gated(M, F, K) && bh_gemm_f32_takes(a, w, out, K),
             "gemm: a gated float32 product takes up to %d rows, K a multiple of 4 and 16-byte aligned operands (M=%d K=%d)",
             BH_F32_FEW_ROWS, M, K);
  const GateForm form = bh_gate_form(gate);
  if (F >= 16 * bh_compute_units()) few_rows<4, true>(a, w, out, M, F, K, 0, form, stream);
  else few_rows<2, true>(a, w, out, M, F, K, 0, form, stream);
  return bh_check_launch("gemm_f32_few");
}

// The same products of RMSNorm(a; norm_weight, eps) in place of a, which is a residual as it stands, by one launch: c[M, N] = norm(a) W^T, or
// gated (`gate`, a BhGate; N outputs).
// bh_gemm_f32_takes_norm: whether these sizes go.  It saves a launch of 2.5 us and costs every workgroup the squares of the rows and a
// register or two for each number of them.  us, norm and product / one launch, chains of products of cold weights:
//   up to 4 rows it wins at all sizes (1 x 7,268 x 748 9.4 / 7.2, 4 x 9,412 x 3,072 32.1 / 28.6, gated 4 x 1,848 x 6,044 26.3 / 23.7);
//   up to 16 rows where a wave takes one or two groups of four outputs or a gated pair of them (8 x 2,608 x 668 7.7 / 5.6, 16 x 2,864 x 924
//   11.2 / 9.7, 10 x 904 x 6,144 16.8 / 14.8, gated 8 x 2,720 x 1,564 15.2 / 13.2, 12 x 1,704 x 4,560 27.9 / 26.0); with more of them
//   its registers leave room for a wave a SIMD less (gated 6 x 8,672 x 3,756 59.7 / 87.9, 12 x 11,000 x 260 11.1 / 15.0);
//   up to 32 rows, whose squares are as much work as the products of a group, only where a wave has few of them and one workgroup is
//   all that a compute unit has (24 x 448 x 140 6.4 / 5.7, gated 24 x 372 x 324 9.5 / 8.6; 28 x 1,488 x 2,600 22.2 / 26.4, 20 x 2,732 x 404
//   9.6 / 14.0).
// What does not go has its norm in front.
extern "C" int bh_gemm_f32_takes_norm(int M, int N, int K, int gated) {
  if (!bh_gemm_f32_takes_gated(M, N, K)) return 0;
  if (M <= 4) return 1;
  const int units = bh_compute_units(), group = (N + 3) / 4;      // groups of four outputs: of one a workgroup
  if (M <= 16) return N < (gated ? 16 : 32) * units ? 1 : 0;
  return group <= units && K <= 768 ? 1 : 0;
}
extern "C" int bh_gemm_f32_normed(const float* a, const float* norm_weight, float eps, const float* w, float* c, int M, int N, int K, int gate,
                                  hipStream_t stream) {
  BH_REQUIRE(bh_gemm_f32_takes_norm(M, N, K, gate != 0) && bh_gemm_f32_takes(a, w, c, K) && ((uintptr_t)norm_weight % 16) == 0,
             "gemm: a float32 product of M=%d N=%d K=%d that norms its rows (bh_gemm_f32_takes_norm), from 16-byte aligned operands", M, N, K);
  BH_REQUIRE(norm_weight != nullptr && eps >= 0.f, "gemm: a norm has a weight, and an epsilon that is not negative");
  BH_REQUIRE(gate == 0 || gate == BH_GATE_SILU || gate == BH_GATE_GELU_TANH, "gemm: unknown activation %d", gate);
  const GateForm form = bh_gate_form(gate);
  const RowNorm norm = {norm_weight, eps};
  const int units = bh_compute_units();
  if (gate && N >= 16 * units) few_waves<4, 1, true, true>(a, w, c, M, N, K, 0, form, norm, stream);
  else if (gate) few_rows<2, true, true>(a, w, c, M, N, K, 0, form, stream, norm);
  else if (N >= 32 * units) few_waves<4, 1, false, true>(a, w, c, M, N, K, 0, form, norm, stream);
  else if (N < 16 * units) few_rows<1, false, true>(a, w, c, M, N, K, 0, form, stream, norm);
  else if (M <= 4) few_waves<2, 1, false, true>(a, w, c, M, N, K, 0, form, norm, stream);
  else if (M <= 8) few_waves<2, 2, false, true>(a, w, c, M, N, K, 0, form, norm, stream);
  else few_waves<2, 4, false, true>(a, w, c, M, N, K, 0, form, norm, stream);
  return bh_check_launch("gemm_f32_few");
}
