// bfloat16 matrix products of many rows, C[M, N] (+)= A[M, K] * W[N, K]^T with W in the tiles layout
// (see gemm_bf16.hip), for the shapes where a 256-row tile fills the chip: prompts from 129 tokens on.
//
// A workgroup of eight waves owns 256 rows x 32 YB weight rows.  Its waves form two groups of four (one wave
// of each group per SIMD) that take turns: while one group multiplies (32 or 24 MFMAs on operands it holds
// in registers), the other reads its next operands from LDS and asks for data that is three steps ahead; a
// barrier ends every turn.  So the matrix cores always have one wave per SIMD that does nothing but multiply,
// and no wave waits for memory in the middle of its multiplies.  A step is half a 64-wide k slice: the 32 k
// values that one 16x16x32 MFMA takes.
//
// Global memory goes to LDS directly (16-byte loads that write LDS at the wave's base + 16 * lane): 1 KB per
// load, which is one operand of 16 rows x 32 k in lane order, so that reading it back is one conflict-free
// 16-byte read per lane.  A lies in blocks of 16 rows x 32 k in operand order (bh_blocked_index in layout.h; the
// kernels that produce activations write it that way for this reader), so that an operand is 1 KB of contiguous
// memory like W's; from plain rows, of which a quarter of a wave touched 16 cache lines for a quarter of their
// bytes each, gate/up at 2,048 rows took 333 us instead of 293 (1.41 PFLOP/s).  The vendor library's
// product (torch.matmul, bfloat16) takes 287 us for the gate/up shape without the gate (1.44 PFLOP/s), 81 us for qkv,
// and reaches 1.51 to 1.55 at its best shapes (4,096 and 8,192 rows): that, not 2.5, is what these matrix cores
// give with operands from memory.
// LDS holds four steps (4 x (16 + 2 YB) KB); a step's region is loaded again as soon as both groups have read
// it, which is five to six turns before it is read next.
//
// It stands beside the ring of gemm_bf16_ring.hip, which keeps both waves of a SIMD busy at once: with tiles of 256 x 256 and 256 x 192 the
// matrix cores' power sets the clock, and taking turns is the more frugal way (8,160 rows, us here / there: gate and up of 12,288 x 4,096
// 1,170 / 1,235, 4,096 x 12,288 551 / 585, 6,144 x 4,096 293 / 303; 2,048 x 8,192 x 2,048 56 / 58); with narrower tiles, which wait for their
// operands more than for the matrix cores, the ring wins (256 x 128 at 2,048 x 4,096 x 4,096: 84 / 63).
#include "gemm_bf16_turns.h"
#include <type_traits>

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));

namespace {

__device__ inline bf16x8_t as_bf16x8(u32x4_t v) { return __builtin_bit_cast(bf16x8_t, v); }

// s_waitcnt immediates of gfx9: vmcnt in bits 3:0 and 15:14, expcnt 6:4, lgkmcnt 11:8.  Both wait for all
// LDS reads; the first also until at most `vm` of the wave's global loads are still on their way.
#define WAIT_VM_LGKM0(vm) __builtin_amdgcn_s_waitcnt(((vm) & 15) | (((vm) >> 4) << 14) | (7 << 4) | (0 << 8))
#define WAIT_LGKM0() __builtin_amdgcn_s_waitcnt(15 | (3 << 14) | (7 << 4) | (0 << 8))
// The end of a turn.  Nothing may be moved across it by the compiler.
#define TICK()                            \
  do {                                    \
    __builtin_amdgcn_sched_barrier(0);    \
    __builtin_amdgcn_s_barrier();         \
    __builtin_amdgcn_sched_barrier(0);    \
  } while (0)

// Which tile a workgroup takes.  Workgroups go to the eight XCDs in turn (workgroup i to XCD i % 8), and each
// XCD has an L2 of its own: neighbours in the order below are workgroups of one XCD, and the 32 of them that
// run at one time (one per compute unit, walking over k in step) should ask that L2 for as few different bytes
// as possible.  So the order goes through the tiles in blocks of 8 row tiles x 4 weight tiles (row tiles
// first): a slice of rows is then fetched once for four compute units and a slice of weights once for eight,
// 12 slices for 32 tiles, where a whole column of row tiles under one weight tile would fetch 33 (measured
// with the chip full: L2 delivers 26 TB/s to the compute units, what lies beyond it 7; at 149,070 rows x
// 51,200 weight rows the column order read 305 GB per product and ran at 1.14 PFLOP/s).  At 8,192 rows x 4,096
// the gate and up product went from 1,245 to 1,165 us (1.42 PFLOP/s) and the down projection from 600 to 563 us
// (1.46).  Only speed depends on where the workgroups really run.
__device__ inline void tile_of_workgroup(int n_tiles, int m_tiles, int* tile_n, int* tile_m) {
  constexpr int BM = 8, BN = 4;
  const int total = n_tiles * m_tiles, xcd = blockIdx.x % 8, each = total / 8, more = total % 8;
  int v = xcd * each + min(xcd, more) + blockIdx.x / 8;
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

// MODE 0: bfloat16 output.  1: float32 output, optionally added to what is there.  2: SwiGLU (the gate as `form` says), bfloat16 output
// (N outputs; W has 2 N rows, gate rows then up rows; a wave's weight rows are the gate and the up rows of
// the same outputs).  3: as 0, squared behind a ReLU.  YB: blocks of 16 weight rows per wave.
// A tile that would stick out of the weight rows is moved back inside and stores only what it owns.
// A's buffer holds whole tiles of 256 rows, and a tile that sticks out below stays where it is and stores only the rows
// that exist.  4: as 2, clamped (gate_mul).  c_blocked (MODE 2 to 4): the output lies in blocks of 16 rows.
template <int MODE, int YB>
__global__ __launch_bounds__(512) void gemm_turns_kernel(const uint16_t* __restrict__ a, const uint16_t* __restrict__ w,
                                                      void* __restrict__ c, int M, int N, int K, int accumulate,
                                                      int c_blocked, GateForm form) {
  constexpr bool GATED = MODE == 2 || MODE == 4;
  constexpr int OUTS = GATED ? 16 * YB : 32 * YB;
  constexpr int CHUNKS = 16 + 2 * YB;
  constexpr int WL = YB / 2;   // W chunks per loading wave
  constexpr int R = 4;                 // steps that LDS holds (with five or six of them it ran no faster)
  __shared__ __attribute__((aligned(16))) u32x4_t lds[R * CHUNKS * 64];   // [region][16 A blocks, then 2 YB W blocks][lane]
  const int tid = threadIdx.x, lane = tid % 64;
  const int wave = __builtin_amdgcn_readfirstlane(tid / 64);
  const int g = wave / 4, i4 = wave % 4;
  int tile_n, tile_m;
  tile_of_workgroup((N + OUTS - 1) / OUTS, (M + 255) / 256, &tile_n, &tile_m);
  const int m0 = tile_m * 256, n_own = tile_n * OUTS, n0 = min(n_own, N - OUTS);
  // K in parts (blockIdx.y, MODE 1 only): part p multiplies its share of k and leaves the bare sums at
  // c + p * M * N for the finishing kernel of gemm_bf16.hip; one part is the whole product.
  const int k_part = K / gridDim.y, k_first = blockIdx.y * k_part;
  const int J = k_part / 32;   // steps: half slices; k_part % 128 == 0

  // The first group brings A (four blocks of 16 rows per wave), the second W (YB / 2 blocks per wave).
  // A step takes 32 consecutive k: lane (row r = lane % 16, group q = lane / 16) holds k 8 q .. 8 q + 7 of them,
  // 1 KB of contiguous memory of a block of A.  In W's tiles layout those are the 16-byte pieces
  // 4 v + q of the row (v: first or second step of the slice), piece p at half p % 2, lane 16 (p / 2) + r.
  const uint16_t* a_src = a + ((size_t)((m0 + 64 * i4) / 16) * (K / 32) + k_first / 32) * 512 + lane * 8;
  const size_t a_block = (size_t)(K / 32) * 512;   // from 16 rows to the next
  const int w_lane = ((lane / 16) % 2) * 512 + (16 * (lane / 32) + lane % 16) * 8;   // + 256 elements for the second step
  const uint16_t* w_src[WL];
#pragma unroll
  for (int b = 0; b < WL; ++b) {
    const int rb = i4 * WL + b, gg = rb / YB, y = rb % YB;
    const int nb = GATED ? (y < YB / 2 ? 0 : N / 16) + n0 / 16 + (YB / 2) * gg + y % (YB / 2) : n0 / 16 + rb;
    w_src[b] = w + ((size_t)nb * (K / 64) + k_first / 64) * 1024 + w_lane;
  }
  auto fetch_a = [&](int j, int region) {
#pragma unroll
    for (int b = 0; b < 4; ++b)
      __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(a_src + b * a_block + j * 512),
                                       (__attribute__((address_space(3))) void*)&lds[(region * CHUNKS + 4 * i4 + b) * 64], 16, 0, 0);
  };
  auto fetch_w = [&](int j, int region) {   // step j = half u of slice s
    const int s = j >> 1, u = j & 1;
#pragma unroll
    for (int b = 0; b < WL; ++b)
      __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(w_src[b] + (size_t)s * 1024 + u * 256),
                                       (__attribute__((address_space(3))) void*)&lds[(region * CHUNKS + 16 + i4 * WL + b) * 64], 16, 0, 0);
  };

  f32x4_t acc[4][YB];
#pragma unroll
  for (int x = 0; x < 4; ++x)
#pragma unroll
    for (int y = 0; y < YB; ++y) acc[x][y] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  u32x4_t af[4], wf[YB];

  auto read_operands = [&](int region) {
#pragma unroll
    for (int x = 0; x < 4; ++x) af[x] = lds[(region * CHUNKS + 4 * i4 + x) * 64 + lane];
#pragma unroll
    for (int y = 0; y < YB; ++y) wf[y] = lds[(region * CHUNKS + 16 + YB * g + y) * 64 + lane];
  };
  auto multiply = [&]() {
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int x = 0; x < 4; ++x)
#pragma unroll
      for (int y = 0; y < YB; ++y)
        acc[x][y] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(wf[y]), as_bf16x8(af[x]), acc[x][y], 0, 0, 0);
    __builtin_amdgcn_s_setprio(0);
  };

  // Step j lies in region j % R.  A wave asks for step j + R - 1 while it reads step j (into the region that
  // step j - 1 has left); before the turn in which the first group reads step j + 1, all that was asked for
  // it must have landed: what may still be on its way are the loads of the steps after it.
  auto wait_for_next = [&](int j, auto per_step) {   // per_step: this wave's loads per step
    constexpr int each = decltype(per_step)::value;
    const int later = min(R - 2, J - 2 - j);   // steps after j + 1 that have been asked for
    if (later >= 2) WAIT_VM_LGKM0(2 * each);
    else if (later == 1) WAIT_VM_LGKM0(each);
    else WAIT_VM_LGKM0(0);
  };
  static_assert(R == 4, "wait_for_next knows of two steps on their way after the next");
  if (g == 0) {
    for (int j = 0; j < R - 1 && j < J; ++j) fetch_a(j, j);
    WAIT_VM_LGKM0(0);
    TICK();
    int region = 0;
    for (int j = 0; j < J; ++j) {
      if (j + R - 1 < J) fetch_a(j + R - 1, region == 0 ? R - 1 : region - 1);
      read_operands(region);
      WAIT_LGKM0();
      TICK();
      multiply();
      wait_for_next(j, std::integral_constant<int, 4>());
      TICK();
      region = region == R - 1 ? 0 : region + 1;
    }
    TICK();
  } else {
    for (int j = 0; j < R - 1 && j < J; ++j) fetch_w(j, j);
    WAIT_VM_LGKM0(0);
    TICK();
    TICK();   // the second group runs one tick behind
    int region = 0;
    for (int j = 0; j < J; ++j) {
      if (j + R - 1 < J) fetch_w(j + R - 1, region == 0 ? R - 1 : region - 1);
      read_operands(region);
      wait_for_next(j, std::integral_constant<int, WL>());
      TICK();
      multiply();
      TICK();
      region = region == R - 1 ? 0 : region + 1;
    }
  }
  // acc[x][y][i]: row 64 i4 + 16 x + lane % 16 of the tile, weight row 16 (YB g + y) + 4 (lane / 16) + i
  const int m = m0 + 64 * i4 + lane % 16;
  if (GATED) {
    uint16_t* out = reinterpret_cast<uint16_t*>(c);
#pragma unroll
    for (int x = 0; x < 4; ++x) {
      const int row = m + 16 * x;
      if (row >= M) continue;
#pragma unroll
      for (int y = 0; y < YB / 2; ++y) {
        const int n = n0 + 8 * YB * g + 16 * y + 4 * (lane / 16);
        if (n < n_own) continue;
        u32x2_t packed;
        packed[0] = f32_to_bf16_bits(gate_mul<MODE == 4>(acc[x][y][0], acc[x][y + YB / 2][0], form)) | ((uint32_t)f32_to_bf16_bits(gate_mul<MODE == 4>(acc[x][y][1], acc[x][y + YB / 2][1], form)) << 16);
        packed[1] = f32_to_bf16_bits(gate_mul<MODE == 4>(acc[x][y][2], acc[x][y + YB / 2][2], form)) | ((uint32_t)f32_to_bf16_bits(gate_mul<MODE == 4>(acc[x][y][3], acc[x][y + YB / 2][3], form)) << 16);
        *reinterpret_cast<u32x2_t*>(out + (c_blocked ? (size_t)bh_blocked_index(row, n, N) : (size_t)row * N + n)) = packed;
      }
    }
  } else {
#pragma unroll
    for (int x = 0; x < 4; ++x) {
      const int row = m + 16 * x;
      if (row >= M) continue;
#pragma unroll
      for (int y = 0; y < YB; ++y) {
        const int n = n0 + 16 * YB * g + 16 * y + 4 * (lane / 16);
        if (n < n_own) continue;
        if (MODE == 1) {
          f32x4_t* at = reinterpret_cast<f32x4_t*>(reinterpret_cast<float*>(c) + ((size_t)blockIdx.y * M + row) * N + n);
          f32x4_t v = acc[x][y];
          if (accumulate) v += *at;
          *at = v;
        } else {
          float v[4];
#pragma unroll
          for (int i = 0; i < 4; ++i) v[i] = MODE == 3 ? relu_squared(acc[x][y][i]) : acc[x][y][i];
          u32x2_t packed;
          packed[0] = f32_to_bf16_bits(v[0]) | ((uint32_t)f32_to_bf16_bits(v[1]) << 16);
          packed[1] = f32_to_bf16_bits(v[2]) | ((uint32_t)f32_to_bf16_bits(v[3]) << 16);
          *reinterpret_cast<u32x2_t*>(reinterpret_cast<uint16_t*>(c) + (MODE == 3 && c_blocked ? (size_t)bh_blocked_index(row, n, N) : (size_t)row * N + n)) = packed;
        }
      }
    }
  }
}


#undef WAIT_VM_LGKM0
#undef WAIT_LGKM0
#undef TICK

template <int MODE>
void launch(const void* a, const void* w, void* c, int blocks, int M, int N, int K, int accumulate, int parts, int c_blocked, GateForm form,
            hipStream_t stream) {
  const int outs = (MODE == 2 || MODE == 4 ? 16 : 32) * blocks;
  dim3 grid(((N + outs - 1) / outs) * ((M + 255) / 256), parts);
  if (blocks == 8)
    gemm_turns_kernel<MODE, 8><<<grid, 512, 0, stream>>>((const uint16_t*)a, (const uint16_t*)w, c, M, N, K, accumulate, c_blocked, form);
  else
    gemm_turns_kernel<MODE, 6><<<grid, 512, 0, stream>>>((const uint16_t*)a, (const uint16_t*)w, c, M, N, K, accumulate, c_blocked, form);
}

}  // namespace

bool gemm_turns_can(int M, int N, int K, int mode, int blocks, int parts) {
  if (blocks != 8 && blocks != 6) return false;
  const int outs = (mode == 2 || mode == 4 ? 16 : 32) * blocks;
  return M > 0 && N >= outs && N % 16 == 0 && parts >= 1 && (mode == 1 || parts == 1) && K >= 128 * parts && K % (128 * parts) == 0 &&
         (long)((N + outs - 1) / outs) * ((M + 255) / 256) < (1L << 31);   // offsets into A, W and C are 64-bit
}

int gemm_turns_launch(const void* a, const void* w, void* c, int mode, int accumulate, int M, int N, int K, int blocks, int parts,
                      int c_blocked, GateForm form, hipStream_t stream) {
  BH_REQUIRE(gemm_turns_can(M, N, K, mode, blocks, parts), "gemm_turns: M=%d N=%d K=%d with %d blocks per wave in %d parts of K is not a product this kernel takes", M, N, K, blocks, parts);
  if (mode == 2) launch<2>(a, w, c, blocks, M, N, K, 0, 1, c_blocked, form, stream);
  else if (mode == 4) launch<4>(a, w, c, blocks, M, N, K, 0, 1, c_blocked, form, stream);
  else if (mode == 1) launch<1>(a, w, c, blocks, M, N, K, accumulate, parts, 0, form, stream);
  else if (mode == 3) launch<3>(a, w, c, blocks, M, N, K, 0, 1, c_blocked, form, stream);
  else launch<0>(a, w, c, blocks, M, N, K, 0, 1, 0, form, stream);
  return bh_check_launch("gemm_turns");
}
