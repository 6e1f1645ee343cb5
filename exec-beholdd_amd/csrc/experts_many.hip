// The routed experts' products of a step of many rows on the matrix cores, from weights in the tiles layout (gemm_bf16.hip: blocks
// of 16 weight rows x 64 k in operand order), all experts in one launch and nothing decided on the host.
//   experts_many   what experts_tiles (experts_tiles.hip) computes, for experts of many pairs
// A workgroup of four waves owns 32 XB pairs of one expert and 128 of its weight rows (gated: the gate and the up rows of the same 64
// outputs, so that a lane holds both sums of an output), a wave 16 XB pairs x 64 weight rows.  Which ones, every workgroup finds by
// itself from the experts' counts: the grid is as large as the pairs allow at most, and what lies beyond the last tile ends at once.
// A step is 32 k: operands go from global memory straight to LDS in lane order (1 KB a load; a pair's input row is found through
// its list, 64 bytes of it a load), three steps ahead in a ring of four, a barrier a step; two workgroups share a compute unit and
// hide each other's barriers.
// Bound by the operands' way from the L2 and memory: weights are read once a tile of pairs, and neighbours on an XCD are the tiles
// of pairs of the same weight rows.
// Measured (32 experts, gate and up / down, us): width 2,048, ff 768, 262 pairs an expert 112 / 71 (0.47 and 0.37 PFLOP/s), 474 / 239
// in the tiles of experts_mfma.hip from row-major matrices, whose 128 weight rows a slice of k lie 4 KB apart; 16 pairs 45 / 21
// (201 MB at 4.5 TB/s), 56 / 35 with experts_tiles, which reads the weights once for 16 pairs and is still ahead at 8 (35 / 21
// against 42 / 21).  Width 4,096, ff 1,536, 256 pairs 379 / 219, where a product an expert of the kernels for one matrix took about
// 25 us each; those reach twice the rate on large matrices, and the caller takes them there.
#include "common.h"

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

template <bool GATED, int XB>
__global__ __launch_bounds__(256) void experts_many_kernel(const uint16_t* __restrict__ in, int in_div, const int32_t* __restrict__ list,
                                                           int capacity, const int32_t* __restrict__ counts, int E,
                                                           const uint16_t* __restrict__ w, void* __restrict__ out_raw, int K, int N,
                                                           float limit, float alpha, float shift, const float* __restrict__ in_weights) {
  constexpr int ROWS = 32 * XB, OUTS = GATED ? 64 : 128, REGIONS = 4, CHUNKS = 2 * XB + 8;
  __shared__ __attribute__((aligned(16))) xm_u32x4_t lds[REGIONS * CHUNKS * 64];   // [region][2 XB blocks of pairs, 8 of weights][lane]
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n_tiles = (N + OUTS - 1) / OUTS;

  // Tiles of pairs of all experts: a wave adds up 64 experts at a time.  Every wave of the workgroup finds the same.
  int total = 0;
  for (int e0 = 0; e0 < E; e0 += 64) total += e0 + lane < E ? (counts[e0 + lane] + ROWS - 1) / ROWS : 0;
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) total += __shfl_xor(total, off, BH_WAVE);
  total *= n_tiles;
  // workgroups go to the eight XCDs in turn; every XCD takes a stretch of (expert, weight tile, tile of pairs) in this order
  const int each = (total + 7) / 8, place = blockIdx.x / 8;
  const int id = (blockIdx.x % 8) * each + place;
  if (place >= each || id >= total) return;      // the whole workgroup
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

  // What this wave brings every step: XB / 2 blocks of 16 pairs and two of 16 weight rows.  Lane (r = lane % 16, q = lane / 16) holds
  // k 8 q .. 8 q + 7 of row r; in the weights' layout those are the pieces 4 v + q of the row (v: first or second step of a chunk of
  // 64), piece p at half p % 2, lane 16 (p / 2) + r.  Pairs beyond the last one and weight rows beyond the last block repeat it.
  constexpr int AL = XB / 2;
  const uint16_t* from_in[AL];
#pragma unroll
  for (int b = 0; b < AL; ++b) {
    const int p = min(p0 + 16 * (AL * wave + b) + lane % 16, count - 1);
    from_in[b] = in + (size_t)(pairs[p] / in_div) * K + 8 * (lane / 16);
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
  auto fetch = [&](int j) {
    const int region = (j & (REGIONS - 1)) * CHUNKS;
#pragma unroll
    for (int b = 0; b < AL; ++b)
      __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(from_in[b] + j * 32),
                                       (__attribute__((address_space(3))) void*)&lds[(region + AL * wave + b) * 64], 16, 0, 0);
#pragma unroll
    for (int b = 0; b < 2; ++b)
      __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(from_w[b] + (size_t)(j >> 1) * 1024 + (j & 1) * 256),
                                       (__attribute__((address_space(3))) void*)&lds[(region + 2 * XB + 2 * wave + b) * 64], 16, 0, 0);
  };

  const int wm = wave / 2, wn = wave % 2, J = K / 32;
  xm_f32x4_t acc[XB][4];
#pragma unroll
  for (int x = 0; x < XB; ++x)
#pragma unroll
    for (int y = 0; y < 4; ++y) acc[x][y] = xm_f32x4_t{0.f, 0.f, 0.f, 0.f};
  // K is a multiple of 64: at least two steps
  for (int j = 0; j < 3 && j < J; ++j) fetch(j);
  constexpr int EACH = AL + 2;      // a wave's loads a step
  for (int j = 0; j < J; ++j) {
    // step j has landed for this wave when at most the later steps' loads are on their way, and for all behind the barrier, which
    // every wave reaches with its reads of step j - 1 done: that region is asked for again
    const int later = min(2, J - 1 - j);
    if (later == 2) XM_WAIT(2 * EACH);
    else if (later == 1) XM_WAIT(EACH);
    else XM_WAIT(0);
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    if (j + 3 < J) fetch(j + 3);
    const int region = (j & (REGIONS - 1)) * CHUNKS;
    xm_u32x4_t af[XB], wf[4];
#pragma unroll
    for (int x = 0; x < XB; ++x) af[x] = lds[(region + XB * wm + x) * 64 + lane];
#pragma unroll
    for (int y = 0; y < 4; ++y) wf[y] = lds[(region + 2 * XB + 4 * wn + y) * 64 + lane];
#pragma unroll
    for (int x = 0; x < XB; ++x)
#pragma unroll
      for (int y = 0; y < 4; ++y) acc[x][y] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_operand(wf[y]), as_operand(af[x]), acc[x][y], 0, 0, 0);
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
extern "C" int bh_experts_many(const void* in, int in_div, const int32_t* list, int capacity, const int32_t* counts, const void* w, void* out,
                               int pairs, int E, int K, int N, int gated, float limit, float alpha, float shift, const float* in_weights,
                               hipStream_t stream) {
  BH_REQUIRE(E > 0 && in_div > 0 && capacity > 0 && pairs > 0 && K >= 64 && N >= 16 && K % 64 == 0 && N % 16 == 0,
             "experts_many: K must be a multiple of 64 and N of 16, got %d and %d", K, N);
  BH_REQUIRE(((uintptr_t)in | (uintptr_t)w | (uintptr_t)out) % 16 == 0, "experts_many: operands must be 16-byte aligned");
  BH_REQUIRE(gated || in_weights == nullptr, "experts_many: weights on the input go with the gated product");
  // Tiles of 128 pairs read the weights half as often as tiles of 64, which leave less of a last tile empty.  Gate and up,
  // tiles of 64 / 128, us: width 2,048 at 48 pairs an expert 49 / 55, at 96 58 / 63, at 192 107 / 86; width 4,096 at 48 152 / 181,
  // at 96 213 / 183, at 192 349 / 289.
  const bool wide = (long)pairs >= 96L * E;
#define BH_XM(GATED, XB) launch<GATED, XB>(in, in_div, list, capacity, counts, w, out, pairs, E, K, N, limit, alpha, shift, in_weights, stream)
  if (gated) return wide ? BH_XM(true, 4) : BH_XM(true, 2);
  return wide ? BH_XM(false, 4) : BH_XM(false, 2);
#undef BH_XM
}
