// The routed experts' products of a step of many rows on the matrix cores, from weights in the tiles layout (gemm_bf16.hip: blocks
// of 16 weight rows x 64 k in operand order), all experts in one launch and nothing decided on the host.
//   experts_many   what experts_tiles (experts_tiles.hip) computes, for experts of many pairs
// A workgroup of four waves owns 32 XB pairs of one expert and 128 of its weight rows (gated: the gate and the up rows of the same 64
// outputs, so that a lane holds both sums of an output), a wave 16 XB pairs x 64 weight rows.  Which ones, every workgroup finds by
// itself from the experts' counts: the grid is as large as the pairs allow at most, and what lies beyond the last tile ends at once.
// Operands go from global memory straight to LDS (1 KB a load): a pair's input row, found through its list, in units of 64 k, so that a
// load takes whole cache lines, into a ring of three; weight rows in steps of 32 k, the k of one matrix instruction, in lane order into a
// ring of four.  While step j is multiplied from registers, the operands of step j + 1 are read from LDS into the other set of registers
// and what comes up to four steps later is asked for, a read, a load and a group of MFMAs in turn; a barrier a step.  Two workgroups
// share a compute unit and hide each other's barriers.  (Tiles of 64 pairs take 56 KB of LDS for it, so that two share one too; with three
// steps of weights three could, which with few workgroups is slower: 8 experts 34.7 -> 40 us.)
// Bound by the operands' way from the L2 and memory: weights are read once a tile of pairs, and neighbours on an XCD are the tiles
// of pairs of the same weight rows.  Tiles of few steps (down: 24 for ff 768) pay for their start and their float32 output beside it.
// Measured (32 experts, gate and up / down, us), in brackets with rows loaded in steps of 32 k, half a line a row and load, whose other
// half came from the L2 once more, and each step's operands read from LDS before its MFMAs: width 2,048, ff 768, 263 pairs an expert
// 87 / 63 (116 / 74), 0.61 and 0.42 PFLOP/s; 512 pairs 139 / 100 (176 / 117); 16 pairs 45 / 21 (47 / 21; 201 MB at 4.5 TB/s), where
// experts_tiles, which reads the weights once for 16 pairs, takes 56 / 35 and is ahead up to 8 pairs.  Width 4,096, ff 1,536, 256 pairs
// 290 / 170 (372 / 210).  8 experts, width 4,096, ff 4,096, 1,024 pairs 573 / 305 (748 / 405), 0.96 and 0.90 PFLOP/s.  The registers
// in turn without the whole lines: 112 / 75 at the first size.
#include "common.h"
#include <cmath>
#include <type_traits>

typedef __bf16 xm_bf16x8_t __attribute__((ext_vector_type(8)));
typedef float xm_f32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t xm_u32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t xm_u32x2_t __attribute__((ext_vector_type(2)));

namespace {

__device__ inline xm_bf16x8_t as_operand(xm_u32x4_t v) { return __builtin_bit_cast(xm_bf16x8_t, v); }

__device__ inline float activation(float g, float u, float limit, float alpha, float shift) {
  g = fminf(g, limit);
  u = fminf(fmaxf(u, -limit), limit);
  return g / (1.0f + expf(-alpha * g)) * (u + shift);
}

// s_waitcnt of gfx9: vmcnt in bits 3:0 and 15:14, expcnt 6:4, lgkmcnt 11:8; waits for all LDS reads and until at most `vm` of the
// wave's global loads are on their way.
#define XM_WAIT(vm) __builtin_amdgcn_s_waitcnt(((vm) & 15) | (((vm) >> 4) << 14) | (7 << 4) | (0 << 8))
// Every wave has waited for its loads.  Nothing may be moved across it by the compiler.
#define XM_MEET()                         \
  do {                                    \
    __builtin_amdgcn_sched_barrier(0);    \
    __builtin_amdgcn_s_barrier();         \
    __builtin_amdgcn_sched_barrier(0);    \
  } while (0)

template <bool GATED, int XB>
__global__ __launch_bounds__(256, 2) void experts_many_kernel(const uint16_t* __restrict__ in, int in_div, const int32_t* __restrict__ list,
                                                           int capacity, const int32_t* __restrict__ counts, int E,
                                                           const uint16_t* __restrict__ w, void* __restrict__ out_raw, int K, int N,
                                                           float limit, float alpha, float shift, const float* __restrict__ in_weights) {
  constexpr int ROWS = 32 * XB, OUTS = GATED ? 64 : 128, STEPS = 4;
  // [3 units of 64 k in turn][block of 16 pairs][16 rows x 8 pieces], then [STEPS steps of 32 k in turn][block of 16 weight rows][lane]; one
  // array, for before a read from one of two arrays the compiler waits for all loads on their way to that one
  __shared__ __attribute__((aligned(16))) xm_u32x4_t lds[3 * 2 * XB * 128 + STEPS * 8 * 64];
  constexpr int W_RING = 3 * 2 * XB * 128;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n_tiles = (N + OUTS - 1) / OUTS;

  // Tiles of pairs of all experts: a wave adds up 64 experts at a time.  Every wave of the workgroup finds the same.
  int total = 0;
  for (int e0 = 0; e0 < E; e0 += 64) total += e0 + lane < E ? (counts[e0 + lane] + ROWS - 1) / ROWS : 0;
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) total += __shfl_xor(total, off, BH_WAVE);
  total *= n_tiles;
  // workgroups go to the eight XCDs in turn; every XCD takes a stretch of (expert, weight tile, tile of pairs) in this order
  const int each = (total + 7) / 8, turn = blockIdx.x / 8;
  const int id = (blockIdx.x % 8) * each + turn;
  if (turn >= each || id >= total) return;      // the whole workgroup
  int expert = -1, before = 0, count = 0, at = 0;
  for (int e0 = 0; e0 < E && expert < 0; e0 += 64) {
    const int mine = e0 + lane < E ? counts[e0 + lane] : 0, tiles = (mine + ROWS - 1) / ROWS * n_tiles;
    int upto = tiles;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const int lower = __shfl_up(upto, off, BH_WAVE);
      if (lane >= off) upto += lower;
    }
    const unsigned long long behind = __ballot(before + upto > id);
    if (behind) {
      const int l = __ffsll(behind) - 1;
      expert = e0 + l;
      count = __shfl(mine, l, BH_WAVE);
      at = id - before - (__shfl(upto, l, BH_WAVE) - __shfl(tiles, l, BH_WAVE));
    } else {
      before += __shfl(upto, 63, BH_WAVE);
    }
  }
  expert = __builtin_amdgcn_readfirstlane(expert);
  count = __builtin_amdgcn_readfirstlane(count);
  at = __builtin_amdgcn_readfirstlane(at);
  const int row_tiles = (count + ROWS - 1) / ROWS;
  const int p0 = (at % row_tiles) * ROWS, n0 = (at / row_tiles) * OUTS;
  const int32_t* pairs = list + (size_t)expert * capacity;

  // What this wave brings: of the pairs, XB / 2 blocks of 16 rows x a unit of 64 k, a whole cache line of eight rows a load (32 k would be
  // half a line, whose other half the next step fetches from the L2 again); of the weights two blocks of 16 rows x a step of 32 k in
  // the weights' own operand order: lane (r = lane % 16, q = lane / 16) takes the pieces 4 v + q of row r (v: first or second step of a
  // chunk of 64), piece p at half p % 2, lane 16 (p / 2) + r.  Pairs beyond the last one and weight rows beyond the last block repeat it.
  // The 16-byte piece c of row r of a block of pairs lies at place c ^ (r % 8) ^ (r / 8) of the row's eight, so that the 16 rows whose
  // piece c a quarter of a wave reads lie in different banks.
  constexpr int AL = XB / 2, EACH = AL + 2;      // a wave's loads a step: half its blocks' rows of a unit, and its weights of a step
  const uint16_t* from_in[AL][2];
#pragma unroll
  for (int b = 0; b < AL; ++b)
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      const int p = min(p0 + 16 * (AL * wave + b) + 8 * half + lane / 8, count - 1);
      from_in[b][half] = in + (size_t)(pairs[p] / in_div) * K + 8 * ((lane % 8) ^ (lane / 8) ^ half);
    }
  const uint16_t* from_w[2];
#pragma unroll
  for (int b = 0; b < 2; ++b) {
    const int y = 2 * wave + b, half = y / 4;      // blocks 0..3 are the first pair of waves' columns, 4..7 the second's
    int block;
    if (GATED) block = min(n0 / 16 + 2 * half + y % 2, N / 16 - 1) + (y % 4 < 2 ? 0 : N / 16);
    else block = min(n0 / 16 + y, N / 16 - 1);
    from_w[b] = w + ((size_t)expert * (GATED ? 2 : 1) * (N / 16) + block) * (K / 64) * 1024 + ((lane / 16) % 2) * 512 +
                (16 * (lane / 32) + lane % 16) * 8;
  }
  auto ask_rows = [&](int b, int half, int unit, int place) {
    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(from_in[b][half] + (size_t)unit * 64),
                                     (__attribute__((address_space(3))) void*)&lds[((place * 2 * XB + AL * wave + b) * 2 + half) * 64], 16, 0, 0);
  };
  auto ask_weights = [&](int b, int step) {
    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(from_w[b] + (size_t)(step >> 1) * 1024 + (step & 1) * 256),
                                     (__attribute__((address_space(3))) void*)&lds[W_RING + ((step % STEPS) * 8 + 2 * wave + b) * 64], 16, 0, 0);
  };

  const int wm = wave / 2, wn = wave % 2, steps = K / 32, units = K / 64;
  xm_f32x4_t acc[XB][4];
#pragma unroll
  for (int x = 0; x < XB; ++x)
#pragma unroll
    for (int y = 0; y < 4; ++y) acc[x][y] = xm_f32x4_t{0.f, 0.f, 0.f, 0.f};
  xm_u32x4_t af[2][XB], wf[2][4];      // the operands of an even and of an odd step
  // The first two units and half of the third, and four steps of weights; what follows is asked for as places become free.  In the order
  // of their use, so that the first step waits for its own only.
  auto ask_unit = [&](int unit) {
#pragma unroll
    for (int b = 0; b < AL; ++b) {
      ask_rows(b, 0, unit, unit);
      if (unit < 2) ask_rows(b, 1, unit, unit);
    }
  };
  auto ask_step = [&](int step) {
#pragma unroll
    for (int b = 0; b < 2; ++b) ask_weights(b, step);
  };
  ask_unit(0);
  ask_step(0);
  ask_step(1);
  if (units >= 3) {
    ask_unit(1);
    ask_step(2);
    ask_unit(2);
    ask_step(3);
    XM_WAIT(2 + 2 * AL + 2 + AL + 2);
  } else {
    if (units == 2) {
      ask_unit(1);
      ask_step(2);
      ask_step(3);
    }
    XM_WAIT(0);
  }
  XM_MEET();
  const int r = lane % 16, read_at = (r / 8) * 64 + (r % 8) * 8 + ((lane / 16) ^ (r % 8) ^ (r / 8));     // ^ 4 for a unit's second step
#pragma unroll
  for (int y = 0; y < 4; ++y) wf[0][y] = lds[W_RING + (4 * wn + y) * 64 + lane];
#pragma unroll
  for (int x = 0; x < XB; ++x) af[0][x] = lds[(XB * wm + x) * 128 + read_at];
  int unit_place = 0;      // of the unit of the step that is multiplied
  // Step j, its operands in registers or on their way there; it reads those of step j + 1.  STEADY: it asks for the weights of step
  // j + 4, in the place of step j's, and for half a unit of rows: in an even step the second half of the unit two ahead of its own, in
  // an odd step the first half of the unit three ahead, which takes its own unit's place (beyond the last unit that one again, which
  // nobody reads).  Every wave waited for its reads of either place before the barrier here.  What step j + 1 needs was asked for in
  // step j - 3 or before, so the loads of two steps may still be on their way.
  auto multiply = [&](int j, auto odd, auto steady) {
    constexpr int U = decltype(odd)::value;
    constexpr bool STEADY = decltype(steady)::value;
    if (STEADY) XM_WAIT(2 * EACH);
    else XM_WAIT(0);
    XM_MEET();
    const int after = unit_place == 2 ? 0 : unit_place + 1, ahead = unit_place == 0 ? 2 : unit_place - 1;
    const int rows_at = (U == 0 ? unit_place : after) * XB * 256 + (U == 0 ? read_at ^ 4 : read_at);
    constexpr int READS = XB + 4, MFMAS = XB * 4, GROUP = (MFMAS + READS - 1) / READS;
#pragma unroll
    for (int g = 0; g < READS; ++g) {
      // (beyond the last step this reads what an earlier one has left there, and nobody uses it)
      if (g < 4) wf[1 - U][g] = lds[W_RING + (((j + 1) % STEPS) * 8 + 4 * wn + g) * 64 + lane];
      else af[1 - U][g - 4] = lds[rows_at + (XB * wm + g - 4) * 128];
      if (STEADY) {
#pragma unroll
        for (int i = 0; i < EACH; ++i)
          if (i * READS / EACH == g) {
            if (i < 2) ask_weights(i, j + STEPS);
            else if (U == 0) ask_rows(i - 2, 1, j / 2 + 2, ahead);
            else ask_rows(i - 2, 0, min(j / 2 + 3, units - 1), unit_place);
          }
      }
#pragma unroll
      for (int q = g * GROUP; q < (g + 1) * GROUP && q < MFMAS; ++q)
        acc[q / 4][q % 4] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_operand(wf[U][q % 4]), as_operand(af[U][q / 4]), acc[q / 4][q % 4], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    }
    if (U == 1) unit_place = after;
  };
  const std::integral_constant<int, 0> even;
  const std::integral_constant<int, 1> odd;
  int j = 0;
  for (; j + STEPS < steps; j += 2) {
    multiply(j, even, std::true_type());
    multiply(j + 1, odd, std::true_type());
  }
  for (; j < steps; j += 2) {
    multiply(j, even, std::false_type());
    multiply(j + 1, odd, std::false_type());
  }

  // acc[x][y][i]: pair 16 (XB wm + x) + lane % 16 of the tile, row 4 (lane / 16) + i of the wave's y-th block of weight rows
#pragma unroll
  for (int x = 0; x < XB; ++x) {
    const int p = p0 + 16 * (XB * wm + x) + lane % 16;
    if (p >= count) continue;
    const int pair = pairs[p];
    if (GATED) {
      const float weight = in_weights ? in_weights[pair] : 1.0f;
#pragma unroll
      for (int y = 0; y < 2; ++y) {
        const int n = n0 + 32 * wn + 16 * y + 4 * (lane / 16);
        if (n >= N) continue;
        uint32_t bits[4];
#pragma unroll
        for (int i = 0; i < 4; ++i)
          bits[i] = f32_to_bf16_bits(activation(acc[x][y][i] * weight, acc[x][y + 2][i] * weight, limit, alpha, shift));
        *reinterpret_cast<xm_u32x2_t*>(reinterpret_cast<uint16_t*>(out_raw) + (size_t)pair * N + n) =
            xm_u32x2_t{bits[0] | (bits[1] << 16), bits[2] | (bits[3] << 16)};
      }
    } else {
#pragma unroll
      for (int y = 0; y < 4; ++y) {
        const int n = n0 + 64 * wn + 16 * y + 4 * (lane / 16);
        if (n < N) *reinterpret_cast<xm_f32x4_t*>(reinterpret_cast<float*>(out_raw) + (size_t)pair * N + n) = acc[x][y];
      }
    }
  }
}
#undef XM_WAIT
#undef XM_MEET

// Whether tiles of 128 pairs are the faster ones.  They read the weights half as often as tiles of 64, and a compute unit that has one of
// either takes 1.12 times as long for it; one that has two takes 1.3 times as long as for one.  So it is the rounds of two a compute
// unit that decide, at as many tiles an expert as the average lets expect (counts differ: from about 0.81 of a tile on some experts
// need one more, behind that half a tile more).  Gate and up + down, tiles of 64 / 128, us, 32 experts: width 1,024, ff 384 at 56 pairs
// 25.5 / 27.5, at 80 27.9 / 28.5, at 128 33.7 / 39.0, at 192 44.7 / 40.2; width 2,048, ff 768 at 48 70.5 / 76.0, at 56 46.8 + 29.0 /
// 51.1 + 24.1, at 64 89.2 / 77.2, at 128 112 / 115; width 4,096, ff 1,536 at 56 264 / 251, at 96 316 / 268.
// With more tiles than places and k of 4,096 the weights' way from memory is the time, and the wider tiles' steps hide more of it: 16
// pairs 158 / 149 (768 tiles), where 128 experts of 2,048 x 768 take 146 / 148 (1,536).
bool tiles_of_128(int pairs, int E, int K, int n_tiles) {
  const double units = bh_compute_units(), average = (double)pairs / E;
  const auto tiles = [&](int size) {
    const double q = average / size, spill = 0.81;
    return (double)E * n_tiles * (q <= spill ? 1.0 : q < 1.0 ? 1.0 + 0.5 * (q - spill) / (1.0 - spill) : q + 0.5);
  };
  const auto time = [&](double count) {
    const double r = count / units, full = std::floor(r / 2.0), rest = r - 2.0 * full;
    return 1.3 * full + (rest < 0.02 ? 0.0 : rest <= 1.0 ? 1.0 : 1.3);
  };
  return (K >= 4096 && (double)E * n_tiles > 2.0 * units) || 1.12 * time(tiles(128)) < time(tiles(64));
}

template <bool GATED, int XB>
int launch(const void* in, int in_div, const int32_t* list, int capacity, const int32_t* counts, const void* w, void* out, int pairs, int E,
           int K, int N, float limit, float alpha, float shift, const float* in_weights, hipStream_t stream) {
  constexpr int ROWS = 32 * XB, OUTS = GATED ? 64 : 128;
  // every expert's last tile may be a part of one: at most so many, rounded up to whole rounds over the XCDs
  const long tiles = ((long)pairs / ROWS + (E < pairs ? E : pairs)) * ((N + OUTS - 1) / OUTS);
  const long grid = (tiles + 7) / 8 * 8;
  BH_REQUIRE(grid < (1L << 31), "experts_many: too many tiles");
  experts_many_kernel<GATED, XB><<<(unsigned)grid, 256, 0, stream>>>((const uint16_t*)in, in_div, list, capacity, counts, E, (const uint16_t*)w, out,
                                                                    K, N, limit, alpha, shift, in_weights);
  return bh_check_launch("experts_many");
}

}  // namespace

// As bh_experts_tiles; `pairs`: how many pairs all experts have together at most (identity experts' may be missing from the lists).
// For tests: the pairs of a tile.
extern "C" int bh_experts_many_tile(int pairs, int E, int K, int N, int gated) {
  return pairs > 0 && E > 0 && N > 0 && tiles_of_128(pairs, E, K, gated ? (N + 63) / 64 : (N + 127) / 128) ? 128 : 64;
}
extern "C" int bh_experts_many(const void* in, int in_div, const int32_t* list, int capacity, const int32_t* counts, const void* w, void* out,
                               int pairs, int E, int K, int N, int gated, float limit, float alpha, float shift, const float* in_weights,
                               hipStream_t stream) {
  BH_REQUIRE(E > 0 && in_div > 0 && capacity > 0 && pairs > 0 && K >= 64 && N >= 16 && K % 64 == 0 && N % 16 == 0,
             "experts_many: K must be a multiple of 64 and N of 16, got %d and %d", K, N);
  BH_REQUIRE(((uintptr_t)in | (uintptr_t)w | (uintptr_t)out) % 16 == 0, "experts_many: operands must be 16-byte aligned");
  BH_REQUIRE(gated || in_weights == nullptr, "experts_many: weights on the input go with the gated product");
  const bool wide = tiles_of_128(pairs, E, K, gated ? (N + 63) / 64 : (N + 127) / 128);
#define BH_XM(GATED, XB) launch<GATED, XB>(in, in_div, list, capacity, counts, w, out, pairs, E, K, N, limit, alpha, shift, in_weights, stream)
  if (gated) return wide ? BH_XM(true, 4) : BH_XM(true, 2);
  return wide ? BH_XM(false, 4) : BH_XM(false, 2);
#undef BH_XM
}
