// bfloat16 matrix products of many rows, C[M, N] (+)= A[M, K] * W[N, K]^T with W in the tiles layout (gemm_bf16.hip) and A in blocks of
// 16 rows x 32 k in operand order (bh_blocked_index): prompts from 129 rows on.
//
// A workgroup of WM x WN waves owns a tile of 16 XB WM rows x 16 YB WN weight rows and walks over k in steps of 32, the k that one
// 16x16x32 MFMA takes.  A step's operands are pieces of 1 KB (16 rows x 32 k in lane order) that global memory hands to LDS directly
// (16-byte loads that write LDS at the wave's base + 16 * lane), so that reading one back is one conflict-free 16-byte read a lane.
// LDS holds a ring of R steps: while step j is multiplied from registers, the wave reads the operands of step j + 1 from LDS into the
// other set of registers and asks for step j + R - 1, whose place in the ring step j - 1 has left.  Reads, loads and MFMAs are issued
// alternately (one operand read, at most one or two loads, a group of MFMAs, and a fence for the compiler between the groups), so that
// the matrix cores never wait for a burst of either; one barrier a step.
//
// What bounds it: operands on their way from L2 and memory for the tiles it is compiled for (128 x 128 asks for 64 bytes per clock and
// compute unit at the matrix cores' full rate, all that L2 gives; 131 GB/s a compute unit measured), the matrix cores, and the clock that
// their power leaves (1.85 to 2.0 GHz of 2.4, a shader clock counter beside the wall clock in the running kernel).  Tiles of 256 x 192 and
// 256 x 256, which the power bounds alone, run on the kernel of gemm_bf16_turns.hip.
// Measured against what these sizes ran on before (the widest tiles with K in parts and a finishing kernel), every product alone in a
// captured graph, weights from memory, us:  2,048 rows: 2,048 x 2,048 47.2 -> 24.6, 2,048 x 6,144 70.6 -> 59.1, 4,096 x 4,096 82.8 -> 69.9;
// 2,096 rows: 3,072 x 2,048 47.8 -> 33.0, 2,048 x 2,048 40.4 -> 31.9; 192 rows of 32,768 x 2,048 51.9 -> 44.6.  The vendor library's product
// (torch.matmul) takes 24, 62, 62, 32.5 and 24.5 at the first five.
// Tried and left out: the 32x32x16 MFMA (half the MFMAs, the same LDS reads: 8 to 12 % slower, the clock falls to 1.75 GHz), waves of
// 128 x 128 (256 accumulators, which the compiler moves between register files), a raised wave priority around the MFMAs, tiles of
// 192 x 128 (no faster than 128 x 128 and 256 x 128 at any size) and 256 x 160.
#include "gemm_bf16_ring.h"
#include "gemm_bf16_turns.h"
#include <type_traits>

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));

namespace {

__device__ inline bf16x8_t as_bf16x8(u32x4_t v) { return __builtin_bit_cast(bf16x8_t, v); }

// s_waitcnt of gfx9 (vmcnt in bits 3:0 and 15:14, expcnt 6:4, lgkmcnt 11:8): all LDS reads are back, and at most `vm` of the wave's
// global loads are still on their way.
#define WAIT_VM_LGKM0(vm) __builtin_amdgcn_s_waitcnt(((vm) & 15) | (((vm) >> 4) << 14) | (7 << 4) | (0 << 8))
// Every wave has waited for its loads.  Nothing may be moved across it by the compiler.
#define MEET()                            \
  do {                                    \
    __builtin_amdgcn_sched_barrier(0);    \
    __builtin_amdgcn_s_barrier();         \
    __builtin_amdgcn_sched_barrier(0);    \
  } while (0)

// Which tile (and part of K) a workgroup takes.  Workgroups go to the eight XCDs in turn (workgroup i to XCD i % 8), each with an L2 of
// its own: an XCD takes a run of neighbours in an order that goes through the tiles in blocks of BM row tiles x BN weight tiles, so
// that the 32 (or 64) workgroups that walk over k there together ask that L2 for few different bytes (8 x 4 tiles: 12 slices for 32
// tiles, where a column of row tiles under one weight tile would fetch 33).  Only speed depends on where the workgroups really run.
template <int BM, int BN>
__device__ inline void tile_of_workgroup(int n_tiles, int m_tiles, int parts, int* tile_n, int* tile_m, int* part) {
  const int tiles = n_tiles * m_tiles, total = tiles * parts, xcd = blockIdx.x % 8, each = total / 8, more = total % 8;
  int v = xcd * each + min(xcd, more) + blockIdx.x / 8;
  *part = v / tiles;
  v %= tiles;
  const int whole_columns = n_tiles / BN;                   // groups of BN weight tiles
  int first_n = 0, columns = BN;
  if (v >= whole_columns * BN * m_tiles) {                  // the weight tiles that fill no group
    v -= whole_columns * BN * m_tiles;
    first_n = whole_columns * BN;
    columns = n_tiles - first_n;
  } else {
    first_n = (v / (BN * m_tiles)) * BN;
    v %= BN * m_tiles;
  }
  const int chunk = v / (BM * columns), within = v % (BM * columns);   // chunks of BM row tiles; the last may be shorter
  const int rows = min(BM, m_tiles - chunk * BM);
  *tile_m = chunk * BM + within % rows;
  *tile_n = first_n + within / rows;
}

// MODE 0: bfloat16 output.  1: float32 output, optionally added to what is there; with parts, part p leaves the bare sums of its share
// of k at c + p M N.  2: gated (the gate as `form` says), bfloat16 output of N columns; W has 2 N rows, gate rows then up rows, and a
// wave's weight rows are the gate and the up rows of the same outputs.  3: as 0, squared behind a ReLU.  4: as 2, clamped (gate_mul).  c_blocked (MODE 2 to 4): the
// output in blocks of 16 rows.
// A tile that sticks out of the matrix repeats its last blocks and stores only what exists; no block of A beyond the last row's is read.
// K a multiple of 64 per part, so that a part has an even number of steps.
// KG = 2: two such groups of waves, each with a ring of its own, take half of k each, and the second hands its sums to the first through
// LDS at the end: what two workgroups of the tile with K in two parts would do on one compute unit, without the sums' way through memory.
template <int MODE, int XB, int YB, int WM, int WN, int R, int KG, int BM, int BN>
__global__ __launch_bounds__(64 * WM * WN * KG, 2) void gemm_ring_kernel(const uint16_t* __restrict__ a, const uint16_t* __restrict__ w,
                                                                    void* __restrict__ c, int M, int N, int K, int parts, int accumulate,
                                                                    int c_blocked, GateForm form) {
  constexpr int WAVES = WM * WN, A_PIECES = XB * WM, W_PIECES = YB * WN, PIECES = A_PIECES + W_PIECES;
  constexpr int EACH = (PIECES + WAVES - 1) / WAVES;   // a wave's pieces of a step; those beyond the last repeat it, so that every wave's count of loads says how far they are
  constexpr bool GATED = MODE == 2 || MODE == 4;
  constexpr int ROWS = 16 * A_PIECES, OUTS = (GATED ? 8 : 16) * W_PIECES;
  static_assert(!GATED || YB % 2 == 0, "a wave's weight rows are gate and up rows of the same outputs");
  static_assert(R >= 4 && EACH * (R - 3) < 64, "the count of loads on their way fits s_waitcnt");
  __shared__ __attribute__((aligned(16))) u32x4_t rings[KG][R * PIECES * 64];     // [group][step in turn][A pieces, then W pieces][lane]
  const int lane = threadIdx.x % 64, wave_of_all = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
  const int wave = wave_of_all % WAVES, group = wave_of_all / WAVES;
  const int wm = wave / WN, wn = wave % WN;
  u32x4_t* const ring = rings[group];
  int tile_n, tile_m, part;
  tile_of_workgroup<BM, BN>((N + OUTS - 1) / OUTS, (M + ROWS - 1) / ROWS, parts, &tile_n, &tile_m, &part);
  const int k_part = K / parts / KG, k_first = (part * KG + group) * k_part, steps = k_part / 32;

  // In W's tiles layout the 32 k of a step are the 16-byte pieces 4 v + q of a row (v: first or second step of a 64-wide chunk, q the
  // lane's group), piece p at half p % 2, lane 16 (p / 2) + r.
  const int w_lane = ((lane / 16) % 2) * 512 + (16 * (lane / 32) + lane % 16) * 8;   // + 256 elements for the second step
  const uint16_t* from[EACH];
  bool of_w[EACH];
  int to[EACH];
#pragma unroll
  for (int i = 0; i < EACH; ++i) {
    const int piece = min(wave + i * WAVES, PIECES - 1);
    to[i] = piece * 64;
    of_w[i] = piece >= A_PIECES;
    if (!of_w[i]) {
      const int block = min(tile_m * A_PIECES + piece, (M - 1) / 16);
      from[i] = a + ((size_t)block * (K / 32) + k_first / 32) * 512 + lane * 8;
    } else {
      const int b = piece - A_PIECES, column = b / YB, y = b % YB;
      const int block = GATED ? (y < YB / 2 ? 0 : N / 16) + min(tile_n * (W_PIECES / 2) + (YB / 2) * column + y % (YB / 2), N / 16 - 1)
                                  : min(tile_n * W_PIECES + b, N / 16 - 1);
      from[i] = w + ((size_t)block * (K / 64) + k_first / 64) * 1024 + w_lane;
    }
  }
  auto ask_piece = [&](int i, int step, int place) {
    const size_t at = of_w[i] ? (size_t)(step >> 1) * 1024 + (step & 1) * 256 : (size_t)step * 512;
    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(from[i] + at),
                                     (__attribute__((address_space(3))) void*)&ring[place * PIECES * 64 + to[i]], 16, 0, 0);
  };
  auto ask = [&](int step, int place) {
#pragma unroll
    for (int i = 0; i < EACH; ++i) ask_piece(i, step, place);
  };

  f32x4_t acc[XB][YB];
#pragma unroll
  for (int x = 0; x < XB; ++x)
#pragma unroll
    for (int y = 0; y < YB; ++y) acc[x][y] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  u32x4_t af[2][XB], wf[2][YB];            // the operands of an even and of an odd step
  int place = 0;                           // of the step that is multiplied
  for (int j = 0; j < R - 1 && j < steps; ++j) ask(j, j);
  WAIT_VM_LGKM0(0);
  MEET();
#pragma unroll
  for (int y = 0; y < YB; ++y) wf[0][y] = ring[(A_PIECES + wn * YB + y) * 64 + lane];
#pragma unroll
  for (int x = 0; x < XB; ++x) af[0][x] = ring[(wm * XB + x) * 64 + lane];
  // Step j, its operands in registers or on their way there.  STEADY: step j + R - 1 is asked for, and the steps after j + 1 may still
  // be on their way; otherwise everything asked for is waited for (the last R steps).
  // The place that is loaded again held step j - 1: every wave waited for its reads of it before the barrier that began step j - 1.
  auto multiply = [&](int j, auto odd, auto steady) {
    constexpr int U = decltype(odd)::value;
    constexpr bool STEADY = decltype(steady)::value;
    if (STEADY) WAIT_VM_LGKM0(EACH * (R - 3));
    else WAIT_VM_LGKM0(0);
    MEET();
    const int next = place == R - 1 ? 0 : place + 1, left = place == 0 ? R - 1 : place - 1;
    constexpr int READS = XB + YB, MFMAS = XB * YB, GROUP = (MFMAS + READS - 1) / READS;
#pragma unroll
    for (int g = 0; g < READS; ++g) {
      // (beyond the last step this reads what an earlier one has left there, and nobody uses it)
      if (g < YB) wf[1 - U][g] = ring[(next * PIECES + A_PIECES + wn * YB + g) * 64 + lane];
      else af[1 - U][g - YB] = ring[(next * PIECES + wm * XB + g - YB) * 64 + lane];
      if (STEADY) {
#pragma unroll
        for (int i = 0; i < EACH; ++i)
          if (i * READS / EACH == g) ask_piece(i, j + R - 1, left);
      }
#pragma unroll
      for (int q = g * GROUP; q < (g + 1) * GROUP && q < MFMAS; ++q)
        acc[q / YB][q % YB] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(wf[U][q % YB]), as_bf16x8(af[U][q / YB]), acc[q / YB][q % YB], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    }
    place = next;
  };
  const std::integral_constant<int, 0> even;
  const std::integral_constant<int, 1> odd;
  int j = 0;
  for (; j + R < steps; j += 2) {
    multiply(j, even, std::true_type());
    multiply(j + 1, odd, std::true_type());
  }
  if (j + R - 1 < steps) ask(j + R - 1, place == 0 ? R - 1 : place - 1);   // at most one step is still to be asked for
  for (; j < steps; j += 2) {
    multiply(j, even, std::false_type());
    multiply(j + 1, odd, std::false_type());
  }

  if constexpr (KG > 1) {
    static_assert(KG == 2 && WAVES * XB * YB <= R * PIECES, "the second group's sums fit where its operands stood");
    f32x4_t* handed = reinterpret_cast<f32x4_t*>(rings[1]) + wave * (XB * YB * 64) + lane;
    MEET();      // the second group has read its last step
    if (group == 1) {
#pragma unroll
      for (int x = 0; x < XB; ++x)
#pragma unroll
        for (int y = 0; y < YB; ++y) handed[(x * YB + y) * 64] = acc[x][y];
    }
    WAIT_VM_LGKM0(0);
    MEET();
    if (group == 1) return;
#pragma unroll
    for (int x = 0; x < XB; ++x)
#pragma unroll
      for (int y = 0; y < YB; ++y) acc[x][y] += handed[(x * YB + y) * 64];
  }
  // acc[x][y][i]: row 16 (XB wm + x) + lane % 16 of the tile, weight row 16 (YB wn + y) + 4 (lane / 16) + i
  const int m0 = tile_m * ROWS + 16 * XB * wm + lane % 16;
#pragma unroll
  for (int x = 0; x < XB; ++x) {
    const int row = m0 + 16 * x;
    if (row >= M) continue;
#pragma unroll
    for (int y = 0; y < (GATED ? YB / 2 : YB); ++y) {
      const int n = tile_n * OUTS + (GATED ? 8 : 16) * YB * wn + 16 * y + 4 * (lane / 16);
      if (n >= N) continue;
      if (MODE == 1) {
        f32x4_t* at = reinterpret_cast<f32x4_t*>(reinterpret_cast<float*>(c) + ((size_t)part * M + row) * N + n);
        f32x4_t v = acc[x][y];
        if (accumulate) v += *at;
        *at = v;
      } else {
        float v[4];
#pragma unroll
        for (int i = 0; i < 4; ++i)
          v[i] = GATED ? gate_mul<MODE == 4>(acc[x][y][i], acc[x][GATED ? y + YB / 2 : y][i], form) : MODE == 3 ? relu_squared(acc[x][y][i]) : acc[x][y][i];
        u32x2_t packed;
        packed[0] = f32_to_bf16_bits(v[0]) | ((uint32_t)f32_to_bf16_bits(v[1]) << 16);
        packed[1] = f32_to_bf16_bits(v[2]) | ((uint32_t)f32_to_bf16_bits(v[3]) << 16);
        *reinterpret_cast<u32x2_t*>(reinterpret_cast<uint16_t*>(c) +
                                    (MODE >= 2 && c_blocked ? (size_t)bh_blocked_index(row, n, N) : (size_t)row * N + n)) = packed;
      }
    }
  }
}
#undef WAIT_VM_LGKM0
#undef MEET

// A tile's sizes, what a step of 32 k costs a compute unit that has one, or two, workgroups of it, and what their start and end cost (us).
// Two workgroups of the tile of four waves share a compute unit.  From the times of every tile and cut of K for 34 products of 1,024 to
// 17,408 weight rows and 17 numbers of rows from 129 to 4,100 (625 sizes, weights from memory, with the norm, finishing or rotation
// behind them): what this chooses there takes 1 % (float32), 2 % (bfloat16) and 1 % (gated) longer than the best of them on average.
// One process differs from another by up to 8 % where a product takes more than 80 us (the clock that the power leaves).
struct TileShape {
  int rows, columns, share;
  double step, step_shared, start_and_end;
};
constexpr TileShape SHAPES[RING_TILES] = {
    {128, 128, 2, 0.245, 0.43, 4.0}, {128, 128, 1, 0.23, 0., 5.0}, {256, 128, 1, 0.36, 0., 4.0}, {256, 192, 1, 0.51, 0., 5.3}, {256, 256, 1, 0.594, 0., 5.0}};
constexpr int MOST_PARTS = 8;

double cost_us(int tile, int parts, int M, int W, int K, RingOutput output) {
  const TileShape& s = SHAPES[tile];
  const long units = bh_compute_units(), workgroups = (long)((M + s.rows - 1) / s.rows) * ((W + s.columns - 1) / s.columns) * parts;
  const double steps = K / 32.0 / parts, alone = steps * s.step + s.start_and_end;
  double t;
  if (s.share == 1) {
    t = (double)((workgroups + units - 1) / units) * alone;
  } else {      // whole rounds of two a compute unit, then a last one: of two, which take as long on some units as on all, or of one
    const double both = steps * s.step_shared + s.start_and_end;
    const long rest = workgroups % (2 * units);
    t = (double)(workgroups / (2 * units)) * both + (rest > units ? both : rest > 0 ? alone : 0.);
  }
  if (parts == 1) return t;
  // The parts' sums on their way to memory and back.  float32: the finishing kernel takes the place of the norm's launch.  bfloat16: it
  // is a launch more; wide products are the queries', keys' and values' projection as a rule, whose reader takes the parts as they are
  // (gemm_ring_bare_plan), and at those what hides behind the next tiles is more: cheaper from 6,144 weight rows and k of 2,048 on
  // (rather than at the price of the others: 768 x 7,168 x 5,120 75.9 against 79.9 us, 1,000 x 6,144 x 4,096 70.1 against 69.5).
  const double sums = parts * (double)M * W * 4.0;
  return t + (output == RING_F32 ? sums / 3.0e6 : W >= 6144 && K >= 2048 ? sums / 6.4e6 : sums / 3.8e6 + 4.0);
}

template <int MODE>
int launch(int tile, int parts, const void* a, const void* w, void* c, int M, int N, int K, int accumulate, int c_blocked, GateForm form,
           hipStream_t stream) {
  const int outs = SHAPES[tile].columns / (MODE == 2 || MODE == 4 ? 2 : 1), rows = SHAPES[tile].rows;
  const dim3 grid((unsigned)((long)((N + outs - 1) / outs) * ((M + rows - 1) / rows) * parts));
#define BH_RING(XB, YB, WM, WN, R, KG, BM, BN)                                                                                 \
  gemm_ring_kernel<MODE, XB, YB, WM, WN, R, KG, BM, BN><<<grid, 64 * WM * WN * KG, 0, stream>>>(                               \
      (const uint16_t*)a, (const uint16_t*)w, c, M, N, K, parts, accumulate, c_blocked, form)
  switch (tile) {       // rings of 80, twice 80 and 144 KB
    case RING_128x128: BH_RING(4, 4, 2, 2, 5, 1, 8, 8); break;
    case RING_128x128_HALVES: BH_RING(4, 4, 2, 2, 5, 2, 8, 4); break;
    case RING_256x128: BH_RING(4, 4, 4, 2, 6, 1, 8, 4); break;
    default: return gemm_turns_launch(a, w, c, MODE, accumulate, M, N, K, tile == RING_256x256 ? 8 : 6, parts, c_blocked, form, stream);
  }
#undef BH_RING
  return bh_check_launch("gemm_ring");
}

}  // namespace

// The tile and the parts of K with the least of the estimate above.
static RingPlan best_plan(int M, int N, int K, RingOutput output) {
  RingPlan plan = {-1, 1};
  const int W = output == RING_GATED ? 2 * N : N;
  for (int tile = 0; tile < RING_TILES; ++tile) {
    if (tile == RING_128x128_HALVES && (K % 128 != 0 || K < 512)) continue;
    const int mode = output == RING_GATED ? 2 : output == RING_F32 ? 1 : 0, blocks = tile == RING_256x256 ? 8 : 6;
    // K is cut where the tiles alone would leave compute units idle
    const long tiles = (long)((M + SHAPES[tile].rows - 1) / SHAPES[tile].rows) * ((W + SHAPES[tile].columns - 1) / SHAPES[tile].columns);
    const int most = output == RING_GATED || tile == RING_128x128_HALVES || tiles >= 2L * bh_compute_units() ? 1 : MOST_PARTS;
    for (int parts = 1; parts <= most; ++parts) {
      if (parts > 1 && (K % (64 * parts) != 0 || K / parts < 256)) continue;
      if (tile >= RING_256x192 && !gemm_turns_can(M, N, K, parts > 1 ? 1 : mode, blocks, parts)) continue;
      const double cost = cost_us(tile, parts, M, W, K, output);
      if (plan.tile < 0 || cost < plan.us) plan = {tile, parts, cost};
    }
  }
  return plan;
}

// Up to 256 rows, for short K or few outputs there, a norm may ride on the product (gemm_bf16.hip), which this kernel does not carry; up
// to 128 rows the kernel of gemm_bf16_slices.hip is the faster one.
// A product asks for its plan several times and a model for the same few over and over; a search takes 0.3 us of the host, which is what
// bounds a step of few rows.  So a thread keeps the last plans it was asked for.
RingPlan gemm_ring_plan(int M, int N, int K, int layout, RingOutput output) {
  if (layout != 1 || M <= 128 || N % 16 != 0 || K % 64 != 0 || K < 128 || N < 128) return {-1, 1};
  if (M <= 256 && (K < 1024 || (output == RING_GATED ? 2 * N : N) < 1024)) return {-1, 1};
  struct Kept {
    int M, N, K, output;
    RingPlan plan;
  };
  static thread_local Kept kept[64] = {};
  Kept& one = kept[((unsigned)M * 31u + (unsigned)(N / 16) * 17u + (unsigned)(K / 64) * 7u + (unsigned)output) % 64];
  if (one.M != M || one.N != N || one.K != K || one.output != output) one = {M, N, K, output, best_plan(M, N, K, output)};
  return one.plan;
}

RingPlan gemm_ring_bare_plan(int M, int N, int K, int layout) {
  const RingPlan plan = gemm_ring_plan(M, N, K, layout, RING_BF16);
  return plan.tile == RING_128x128_HALVES ? RingPlan{RING_128x128, 2, plan.us} : plan;
}

static bool ring_can(int M, int N, int K, int tile, int parts) {
  return M > 0 && N > 0 && N % 16 == 0 && K > 0 && parts >= 1 && K % (64 * parts * (tile == RING_128x128_HALVES ? 2 : 1)) == 0 && tile >= 0 && tile < RING_TILES &&
         (long)((N + 63) / 64) * ((M + 127) / 128) * parts < (1L << 31);
}

int gemm_ring_launch_parts(const void* a, const void* w, float* sums, int M, int N, int K, const RingPlan& plan, hipStream_t stream) {
  BH_REQUIRE(ring_can(M, N, K, plan.tile, plan.parts), "gemm_ring: M=%d N=%d K=%d cannot be multiplied in %d parts of K", M, N, K, plan.parts);
  BH_REQUIRE(((uintptr_t)a | (uintptr_t)w | (uintptr_t)sums) % 16 == 0, "gemm_ring: operands must be 16-byte aligned");
  return launch<1>(plan.tile, plan.parts, a, w, sums, M, N, K, 0, 0, GateForm{}, stream);
}

int gemm_ring_launch(const void* a, const void* w, void* c, int c_dtype, int accumulate, int M, int N, int K, int activation, int tile,
                     int c_blocked, GateForm form, hipStream_t stream) {
  BH_REQUIRE(ring_can(M, N, K, tile, 1), "gemm_ring: a product of M=%d N=%d K=%d is not one this kernel takes (K a multiple of 64, N of 16)", M, N, K);
  BH_REQUIRE(c_dtype == BH_F32 || (c_dtype == BH_BF16 && !accumulate), "gemm_ring: output float32, or bfloat16 without accumulation");
  BH_REQUIRE(!activation || c_dtype == BH_BF16, "gemm_ring: a gated product writes bfloat16");
  BH_REQUIRE(((uintptr_t)a | (uintptr_t)w | (uintptr_t)c) % 16 == 0, "gemm_ring: operands and output must be 16-byte aligned");
  BH_REQUIRE(!form.squared || (!activation && c_dtype == BH_BF16), "gemm_ring: a plain product squares its bfloat16 output");
  BH_REQUIRE(!c_blocked || ((activation || form.squared) && N % 32 == 0),
             "gemm_ring: only a gated or squared product writes its output in blocks, and N=%d must be a multiple of 32", N);
  if (activation == GATED_CLAMPED) return launch<4>(tile, 1, a, w, c, M, N, K, 0, c_blocked, form, stream);
  if (activation) return launch<2>(tile, 1, a, w, c, M, N, K, 0, c_blocked, form, stream);
  if (c_dtype == BH_F32) return launch<1>(tile, 1, a, w, c, M, N, K, accumulate, 0, form, stream);
  if (form.squared) return launch<3>(tile, 1, a, w, c, M, N, K, 0, c_blocked, form, stream);
  return launch<0>(tile, 1, a, w, c, M, N, K, 0, 0, form, stream);
}

// For tests and measurements: the tiles of 256 rows at a given width of 32 `blocks` weight rows, whatever gemm_ring_plan would choose.
extern "C" int bh_gemm_bf16_turns(const void* a, const void* w, void* c, int c_dtype, int accumulate, int M, int N, int K, int activation,
                                  int blocks, int c_blocked, hipStream_t stream) {
  const int outs = (activation ? 16 : 32) * blocks;
  BH_REQUIRE((blocks == 8 || blocks == 6 || blocks == 4) && M >= 256 && N >= outs && N % 16 == 0 && K >= 128 && K % 128 == 0,
             "gemm_turns: a product of M=%d N=%d K=%d with %d blocks per wave is not one this kernel takes "
             "(M >= 256, K a multiple of 128, N a multiple of 16 and at least a tile)", M, N, K, blocks);
  return gemm_ring_launch(a, w, c, c_dtype, accumulate, M, N, K, activation != 0, blocks == 8 ? RING_256x256 : blocks == 6 ? RING_256x192 : RING_256x128,
                          c_blocked, bh_gate_form(activation), stream);
}
