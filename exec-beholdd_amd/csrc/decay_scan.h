// A linear recurrence with a scalar decay per row and head, for prompts, on the float32 matrix instructions:
//   S_t = d_t S_(t-1) + w_t k_t v_t^T,   o_t = S_t^T q_t + skip v_t          S [D][V] per (sequence, head)
// (lightning attention: d the head's constant, w 1, no skip; the state-space recurrence: d and w from the row's step size.)
//
// With the rows in chunks of 64 and D(t, j) = d_(j+1) .. d_t, a chunk that starts from the state E has
//   o_t = D(t, start) E^T q_t + sum_(j <= t) D(t, j) w_j (q_t . k_j) v_j + skip v_t,   S_end = D(end, start) E + sum_j D(end, j) w_j k_j v_j^T,
// so that all of it but the chain of states is products of matrices, for all chunks at the same time:
//   scan_states    a workgroup a (chunk, head): Z = sum_j D(end, j) w_j k_j v_j^T and the chunk's whole decay
//   scan_combine   goes through a sequence's chunks in order: E_(c+1) = D E_c + Z_c, from and to the sequence's region; a thread four elements
//   scan_outputs   a workgroup a (chunk, head): scores q k^T, times their decays and weights below the diagonal, times v, and E^T q
// Every product and sum is 32-bit; decays are differences of logarithms summed in 64 bits (or powers of the constant), so that
// no row's decay is a chain of roundings.  A walk row by row (lightning_scan, ssm_chunk) has the same sums in another order, but as a
// serial chain of FMAs.
// A sequence's chunks have places of their own, floor(first row / 64) + sequence onward, which overlap no other sequence's: a step
// needs rows / 64 + sequences places, and a window of them at a time has memory for its states.
// Bound by the matrix instructions, of which lightning attention's outputs need 11 us below, and by what comes before and behind them: all
// workgroups are at the same of a chunk's four phases at a time, and loads and stores alone take 17 us of the outputs' 34.  A state is
// written once and read twice.
// Measured, bfloat16 projections, one sequence of 2,048 rows: lightning attention with 16 heads of 128 x 128 70 us in all (25 + 11 +
// 34), 240 as a walk of chunks; the state-space recurrence with 64 heads of 128 x 64 148 us, 610.  (88 and 165 with states by rows,
// loads waited for one piece after the other, and heads of a group on different XCDs.)  With the values in LDS beside the keys, one
// workgroup a compute unit, about 20 and 50 us more.
#pragma once

#include "common.h"

#include <type_traits>

#define DS_ROWS 64                    // rows of a chunk
#define DS_MOST_VALUES 256             // elements of a value
#define DS_PSTRIDE 20                   // floats from one row of a 16 x 16 tile of scores to the next: 16 rows' 16 bytes on all banks
#define DS_SCORES (10 * 16 * DS_PSTRIDE) // the tiles on and below the diagonal, (row, column) at place row (row + 1) / 2 + column
#define DS_SCRATCH_FLOATS (24L << 20) // states that a window of places may take: 96 MB (36: 8,192 rows of 32 heads 621 -> 878 us)

typedef float ds_f32x4_t __attribute__((ext_vector_type(4)));

struct ScanChunk {
  int seq, chunk, first, rows;
};

__device__ inline int ds_place_of(const int32_t* seq_start, int seq) { return seq_start[seq] / DS_ROWS + seq; }

// The chunk at a place; rows 0 where no sequence has one there.  The same for the whole workgroup.
__device__ inline ScanChunk ds_find(const int32_t* __restrict__ seq_start, int n_seqs, int place) {
  const int lane = threadIdx.x & 63;
  int upto = 0;      // sequences whose places start at this one or before
  for (int s0 = 0; s0 < n_seqs; s0 += 64) {
    const int s = s0 + lane;
    upto += __popcll(__ballot(s < n_seqs && ds_place_of(seq_start, s < n_seqs ? s : 0) <= place));
  }
  ScanChunk at = {0, 0, 0, 0};
  if (upto == 0) return at;      // a place before the first sequence's, where rows of nobody lie ahead of it
  at.seq = __builtin_amdgcn_readfirstlane(upto - 1);
  at.chunk = place - ds_place_of(seq_start, at.seq);
  at.first = seq_start[at.seq] + at.chunk * DS_ROWS;
  at.rows = min(DS_ROWS, seq_start[at.seq + 1] - at.first);
  if (at.rows < 0) at.rows = 0;
  return at;
}

// Rows' decays within a chunk.  POWERS: of one number, pow[n] = d^n; otherwise from the rows' logarithms, summed in 64 bits.
template <bool POWERS>
struct ScanDecays;
template <>
struct ScanDecays<true> {
  float pow[DS_ROWS + 1];
  __device__ float between(int t, int j) const { return pow[t - j]; }
  __device__ float from_start(int t) const { return pow[t + 1]; }
};
template <>
struct ScanDecays<false> {
  double sum[DS_ROWS];
  // e^x of a 64-bit number: what 32 bits of it leave out is below 2^-24 of it, so that one term of the series is enough
  static __device__ float exponential(double x) {
    const float head = (float)x, power = expf(head);
    return fmaf(power, (float)(x - head), power);
  }
  __device__ float between(int t, int j) const { return exponential(sum[t] - sum[j]); }
  __device__ float from_start(int t) const { return exponential(sum[t]); }
};

// The place (of `places`) and head of a workgroup.  Heads that share their keys and queries (`shared` in a row) run at one place on one
// XCD, one after the other, so that its L2 holds them (64 heads of 128 x 64 in groups of eight, 2,103 rows of three sequences: 164 -> 154 us); workgroups go to
// the eight XCDs in turn.  The grid is of whole rounds (ds_grid); those beyond the last place and head have nothing to do.
__device__ inline bool ds_where(int places, int H, int shared, int& place, int& head) {
  const int turn = blockIdx.x / 8, unit = turn / shared * 8 + blockIdx.x % 8;
  place = unit % places;
  head = unit / places * shared + turn % shared;
  return head < H;
}
inline unsigned ds_grid(int places, int H, int shared) { return ((unsigned)(places * (H / shared)) + 7) / 8 * 8 * shared; }

// Where a workgroup's 512 threads find four neighbouring elements of the chunk's 64 vectors of 4 * `pieces` each: thread, then 512 on.
struct ScanPieces {
  int row, piece, pieces;
  __device__ ScanPieces(int pieces) : row(threadIdx.x / pieces), piece(threadIdx.x % pieces), pieces(pieces) {}
  __device__ void next() {
    row += 512 / pieces;
    piece += 512 % pieces;
    if (piece >= pieces) piece -= pieces, ++row;
  }
};

// A state lies in scratch memory as the matrix instructions hand it out and take it: 16 x 16 tiles, column after column of them, and in
// a tile lane (j, g)'s four elements (rows 4 g .. + 3, column j) side by side, so that every load and store of one is 1 KB in a piece (by
// rows, 64 bytes at a time, lightning attention's three kernels of 16 heads of 128 x 128 and 2,048 rows took 25 + 18 + 41 us).
__device__ inline size_t ds_tile(int column_tile, int row_tile, int D) { return ((size_t)column_tile * (D / 16) + row_tile) * 256; }

// In: what the recurrence reads.  POWERS, SKIPS (with skip(head)), shared() (heads in a row with the same keys and queries), Raw q4 / k4 / v4(row, head, i) (elements i .. i + 3 of the head's vector as
// memory holds them) with float4 open(Raw), and prepare(decays, weights, chunk, head): called by a whole workgroup, which it leaves with
// a barrier to come.  WIDE: vectors of more than 128 elements.  All of a chunk's loads are asked for before the first is waited for.
template <class In, bool WIDE>
__global__ __launch_bounds__(512) void scan_states_kernel(In in, const int32_t* __restrict__ seq_start, int n_seqs, int place0, int places,
                                                          float* __restrict__ states, float* __restrict__ factors, int H, int D, int V) {
  extern __shared__ __align__(16) float ds_lds[];
  __shared__ ScanDecays<In::POWERS> decays;
  __shared__ float weights[DS_ROWS];
  constexpr int STEPS = WIDE ? 9 : 4;      // D of up to 288 fits the LDS
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  int place, head;
  if (!ds_where(places, H, in.shared(), place, head)) return;
  const ScanChunk at = ds_find(seq_start, n_seqs, place0 + place);
  if (at.rows == 0) return;
  const int ks = D + 4, vs = V + 4;
  float* k_lds = ds_lds;
  float* v_lds = k_lds + DS_ROWS * ks;
  typename In::Raw k_raw[STEPS], v_raw[STEPS];
  {
    ScanPieces k_at(D / 4), v_at(V / 4);
#pragma unroll
    for (int u = 0; u < STEPS; ++u, k_at.next(), v_at.next()) {
      if (k_at.row < at.rows) k_raw[u] = in.k4(at.first + k_at.row, head, 4 * k_at.piece);
      if (v_at.row < at.rows) v_raw[u] = in.v4(at.first + v_at.row, head, 4 * v_at.piece);
    }
  }
  in.prepare(decays, weights, at, head);
  __syncthreads();
  const float4 none = make_float4(0.f, 0.f, 0.f, 0.f);
  ScanPieces k_at(D / 4), v_at(V / 4);
#pragma unroll
  for (int u = 0; u < STEPS; ++u, k_at.next(), v_at.next()) {
    if (k_at.row < DS_ROWS) {
      float4 k = none;
      if (k_at.row < at.rows) {
        k = in.open(k_raw[u]);
        const float w = weights[k_at.row] * decays.between(at.rows - 1, k_at.row);
        k = make_float4(k.x * w, k.y * w, k.z * w, k.w * w);
      }
      *reinterpret_cast<float4*>(k_lds + k_at.row * ks + 4 * k_at.piece) = k;
    }
    if (v_at.row < DS_ROWS) *reinterpret_cast<float4*>(v_lds + v_at.row * vs + 4 * v_at.piece) = v_at.row < at.rows ? in.open(v_raw[u]) : none;
  }
  if (tid == 0) factors[(size_t)place * H + head] = decays.from_start(at.rows - 1);
  __syncthreads();
  // Z [D][V]: 32 x 16 elements at a time, rows of the chunk as the products' depth; a wave's values stay in registers while its columns
  // do (V of 16, 32, 64, 128: always)
  const int j = lane & 15, g = lane >> 4, columns = V / 16;
  float* out = states + ((size_t)place * H + head) * D * V;
  float v[DS_ROWS / 4];
  int held = -1;
  for (int unit = wave; unit < D / 32 * columns; unit += 8) {
    const int d0 = unit / columns * 32, column = unit % columns;
    if (column != held) {
      held = column;
#pragma unroll
      for (int s = 0; s < DS_ROWS / 4; ++s) v[s] = v_lds[(16 * (s / 4) + 4 * g + s % 4) * vs + 16 * column + j];
    }
    ds_f32x4_t acc[2] = {};
#pragma unroll
    for (int s = 0; s < DS_ROWS / 4; ++s) {
      const int row = 16 * (s / 4) + 4 * g + s % 4;      // four rows of 4 D + 16 floats apart: on banks of their own
      const float* k_row = k_lds + row * ks + d0 + j;
      acc[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(k_row[0], v[s], acc[0], 0, 0, 0);
      acc[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(k_row[16], v[s], acc[1], 0, 0, 0);
    }
#pragma unroll
    for (int x = 0; x < 2; ++x) *reinterpret_cast<ds_f32x4_t*>(out + ds_tile(column, d0 / 16 + x, D) + 4 * lane) = acc[x];
  }
}

// grid (sequences, heads, elements / 1024)
template <int UNUSED = 0>
__global__ __launch_bounds__(256) void scan_combine_kernel(const int32_t* __restrict__ seq_start, const int32_t* __restrict__ seq_slot, const int32_t* __restrict__ seq_to,
                                                           int place0, int places, float* __restrict__ states,
                                                           const float* __restrict__ factors, float* __restrict__ home, long slot_stride,
                                                           int H, int D, int V) {
  constexpr int AHEAD = 8;
  const int seq = blockIdx.x, head = blockIdx.y, size = D * V, e = 4 * (blockIdx.z * 256 + threadIdx.x);
  if (e >= size) return;
  const int base = ds_place_of(seq_start, seq), chunks = (seq_start[seq + 1] - seq_start[seq] + DS_ROWS - 1) / DS_ROWS;
  const int from = max(0, place0 - base), upto = min(chunks, place0 + places - base);
  if (from >= upto) return;
  // the thread's four elements of a tile (ds_tile) in the sequence's region, which lies by rows
  const int tile = e / 256, lane = e % 256 / 4, d = tile % (D / 16) * 16 + lane / 16 * 4, v = tile / (D / 16) * 16 + lane % 16;
  float* left = home + (size_t)seq_to[seq] * slot_stride + (size_t)head * size + (size_t)d * V + v;
  // (a launch that goes on with a sequence goes on from what the one before left)
  const float* mine = from > 0 ? left : home + (size_t)seq_slot[seq] * slot_stride + (size_t)head * size + (size_t)d * V + v;
  const size_t apart = (size_t)H * size;
  float* z = states + ((size_t)(base + from - place0) * H + head) * size + e;
  const float* f = factors + (size_t)(base + from - place0) * H + head;
  float4 state = make_float4(mine[0], mine[V], mine[2 * V], mine[3 * V]);
  float4 own[2][AHEAD];
  float factor[2][AHEAD];
  auto ask = [&](int side, int c) {      // (beyond the last chunk the last one's again, which nobody uses)
#pragma unroll
    for (int u = 0; u < AHEAD; ++u) {
      const int at = min(c + u, upto - from - 1);
      own[side][u] = *reinterpret_cast<const float4*>(z + at * apart);
      factor[side][u] = f[(size_t)at * H];
    }
  };
  ask(0, 0);
  for (int c0 = 0; c0 < upto - from; c0 += 2 * AHEAD)
#pragma unroll
    for (int side = 0; side < 2; ++side) {
      const int c = c0 + side * AHEAD;
      if (c >= upto - from) break;
      if (c + AHEAD < upto - from) ask(1 - side, c + AHEAD);      // while this side's chunks are joined
#pragma unroll
      for (int u = 0; u < AHEAD; ++u) {
        if (c + u >= upto - from) break;
        *reinterpret_cast<float4*>(z + (c + u) * apart) = state;      // what this chunk starts from
        state.x = fmaf(factor[side][u], state.x, own[side][u].x);
        state.y = fmaf(factor[side][u], state.y, own[side][u].y);
        state.z = fmaf(factor[side][u], state.z, own[side][u].z);
        state.w = fmaf(factor[side][u], state.w, own[side][u].w);
      }
    }
  left[0] = state.x, left[V] = state.y, left[2 * V] = state.z, left[3 * V] = state.w;
}

template <class In, bool WIDE>
__global__ __launch_bounds__(512, WIDE ? 2 : 4) void scan_outputs_kernel(In in, const int32_t* __restrict__ seq_start, int n_seqs, int place0,
                                                                         int places, const float* __restrict__ states, float* __restrict__ out,
                                                                         int H, int D, int V) {
  extern __shared__ __align__(16) float ds_lds[];
  __shared__ ScanDecays<In::POWERS> decays;
  __shared__ float weights[DS_ROWS];
  __shared__ int any_spoilt;      // whether a value of the chunk is not finite
  constexpr int STEPS = WIDE ? 9 : 4, DEPTH = WIDE ? 18 : 8;      // D of up to 288 fits the LDS
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  int place, head;
  if (!ds_where(places, H, in.shared(), place, head)) return;
  const ScanChunk at = ds_find(seq_start, n_seqs, place0 + place);
  if (at.rows == 0) return;
  const int qs = D + 4, vs = V + 4;
  // The scores and the values take the keys' place once those have been multiplied (the values wait in registers), which lets two
  // workgroups of heads of 128 share a compute unit.
  float* q_lds = ds_lds;
  float* k_lds = q_lds + DS_ROWS * qs;
  float* p_lds = k_lds;
  float* v_lds = p_lds + DS_SCORES;
  const float4 none = make_float4(0.f, 0.f, 0.f, 0.f);
  typename In::Raw v_raw[STEPS];
  // the state that the chunk starts from: a wave's columns of it, asked for here and needed last
  const float* start = states + ((size_t)place * H + head) * D * V;
  const int columns = V / 16, halves = columns >= 8 ? 1 : 2;      // a wave has both halves of the rows where there are columns for every wave
  ds_f32x4_t e[DEPTH];
  auto ask_state = [&](int column) {
#pragma unroll
    for (int b = 0; b < DEPTH; ++b)
      if (16 * b < D) e[b] = *reinterpret_cast<const ds_f32x4_t*>(start + ds_tile(column, b, D) + 4 * lane);
  };
  {
    typename In::Raw q_raw[STEPS], k_raw[STEPS];
    ScanPieces asked(D / 4), v_at(V / 4), put(D / 4);
#pragma unroll
    for (int u = 0; u < STEPS; ++u, asked.next()) {
      if (asked.row < at.rows) {
        q_raw[u] = in.q4(at.first + asked.row, head, 4 * asked.piece);
        k_raw[u] = in.k4(at.first + asked.row, head, 4 * asked.piece);
      }
    }
#pragma unroll
    for (int u = 0; u < STEPS; ++u, v_at.next())
      if (v_at.row < at.rows) v_raw[u] = in.v4(at.first + v_at.row, head, 4 * v_at.piece);
    in.prepare(decays, weights, at, head);
#pragma unroll
    for (int u = 0; u < STEPS; ++u, put.next()) {
      if (put.row >= DS_ROWS) continue;
      const bool there = put.row < at.rows;
      *reinterpret_cast<float4*>(q_lds + put.row * qs + 4 * put.piece) = there ? in.open(q_raw[u]) : none;
      *reinterpret_cast<float4*>(k_lds + put.row * qs + 4 * put.piece) = there ? in.open(k_raw[u]) : none;
    }
  }
  if (tid == 0) any_spoilt = 0;
  if (wave < halves * columns) ask_state(wave / halves);
  __syncthreads();
  // scores: the ten 16 x 16 tiles on and below the diagonal, a wave one or two.  A lane's 16 bytes are k 16 b + 4 g .. + 3 of its row
  // for either operand, which the matrix instructions take in turn.
  const int j = lane & 15, g = lane >> 4;
  ds_f32x4_t score[2];
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const int tile = wave + 8 * u;
    score[u] = ds_f32x4_t{0.f, 0.f, 0.f, 0.f};
    if (tile >= 10) continue;
    const int tr = tile < 1 ? 0 : tile < 3 ? 1 : tile < 6 ? 2 : 3, tc = tile - tr * (tr + 1) / 2;
    const float* q_row = q_lds + (16 * tr + j) * qs + 4 * g;
    const float* k_row = k_lds + (16 * tc + j) * qs + 4 * g;
    ds_f32x4_t chain[4] = {};      // four sums side by side, added at the end
#pragma unroll 2
    for (int b = 0; b < D; b += 32) {
      const ds_f32x4_t q0 = *reinterpret_cast<const ds_f32x4_t*>(q_row + b), k0 = *reinterpret_cast<const ds_f32x4_t*>(k_row + b);
      const ds_f32x4_t q1 = *reinterpret_cast<const ds_f32x4_t*>(q_row + b + 16), k1 = *reinterpret_cast<const ds_f32x4_t*>(k_row + b + 16);
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        chain[t & 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(q0[t], k0[t], chain[t & 1], 0, 0, 0);
        chain[2 + (t & 1)] = __builtin_amdgcn_mfma_f32_16x16x4f32(q1[t], k1[t], chain[2 + (t & 1)], 0, 0, 0);
      }
    }
    score[u] = (chain[0] + chain[1]) + (chain[2] + chain[3]);
  }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const int tile = wave + 8 * u;
    if (tile >= 10) continue;
    const int tr = tile < 1 ? 0 : tile < 3 ? 1 : tile < 6 ? 2 : 3, tc = tile - tr * (tr + 1) / 2;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int t = 16 * tr + 4 * g + r, c = 16 * tc + j;
      float p = 0.f;
      if (c <= t && t < at.rows) {
        p = score[u][r] * decays.between(t, c) * weights[c];
      }
      p_lds[tile * 16 * DS_PSTRIDE + (4 * g + r) * DS_PSTRIDE + j] = p;
    }
  }
  float zero = 0.f;      // zero times every value: NaN where one is not finite
  ScanPieces v_at(V / 4);
#pragma unroll
  for (int u = 0; u < STEPS; ++u, v_at.next()) {
    if (v_at.row >= DS_ROWS) continue;
    const float4 value = v_at.row < at.rows ? in.open(v_raw[u]) : none;
    *reinterpret_cast<float4*>(v_lds + v_at.row * vs + 4 * v_at.piece) = value;
    zero = fmaf(value.w, 0.f, fmaf(value.z, 0.f, fmaf(value.y, 0.f, fmaf(value.x, 0.f, zero))));
  }
  if (zero != 0.f) any_spoilt = 1;
  __syncthreads();
  const bool spoilt = any_spoilt;
  // outputs: 32 rows x 16 columns at a time
  auto outputs = [&](int r0, int c0) {
    ds_f32x4_t carried[2];
    {
      ds_f32x4_t from_state[2][2] = {};      // [side]: two sums side by side
      const float* q_row = q_lds + (r0 + j) * qs + 4 * g;
#pragma unroll
      for (int b = 0; b < DEPTH; ++b) {
        if (16 * b >= D) break;
        __builtin_amdgcn_sched_barrier(0);      // not all rows of q in registers at once
        ds_f32x4_t q[2];
#pragma unroll
        for (int x = 0; x < 2; ++x) q[x] = *reinterpret_cast<const ds_f32x4_t*>(q_row + 16 * x * qs + 16 * b);
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
          for (int x = 0; x < 2; ++x) from_state[t & 1][x] = __builtin_amdgcn_mfma_f32_16x16x4f32(q[x][t], e[b][t], from_state[t & 1][x], 0, 0, 0);
      }
#pragma unroll
      for (int x = 0; x < 2; ++x) carried[x] = from_state[0][x] + from_state[1][x];
    }
    ds_f32x4_t acc[2][2] = {};
    const int tile0 = r0 / 16;
    auto p_tile = [&](int x, int column) { return p_lds + ((tile0 + x) * (tile0 + x + 1) / 2 + column) * 16 * DS_PSTRIDE; };
    auto add_rows = [&](auto guarded) {
#pragma unroll 1
      for (int b = 0; b < r0 + 32; b += 16) {
        float v[4], own[4];      // own: what the tile on the diagonal takes
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          v[t] = v_lds[(b + 4 * g + t) * vs + c0 + j];
          own[t] = !guarded || isfinite(v[t]) ? v[t] : 0.f;
        }
#pragma unroll
        for (int x = 0; x < 2; ++x) {
          if (b > r0 + 16 * x) continue;      // rows see no later ones
          const ds_f32x4_t p = *reinterpret_cast<const ds_f32x4_t*>(p_tile(x, b / 16) + j * DS_PSTRIDE + 4 * g);
#pragma unroll
          for (int t = 0; t < 4; ++t)
            acc[t & 1][x] = __builtin_amdgcn_mfma_f32_16x16x4f32(p[t], guarded && b == r0 + 16 * x ? own[t] : v[t], acc[t & 1][x], 0, 0, 0);
        }
      }
    };
    if (!spoilt) {
      add_rows(std::false_type{});
    } else {
      // Scores above the diagonal are zeros, but zero times infinity is not: a value that is not finite stays out of the product of
      // its own rows' tile and is added by itself, to its row and the later ones.
      add_rows(std::true_type{});
#pragma unroll
      for (int x = 0; x < 2; ++x) {
        for (int c = 0; c < 16; ++c) {
          const float v = v_lds[(r0 + 16 * x + c) * vs + c0 + j];
          if (isfinite(v)) continue;
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const float added = fmaf(p_tile(x, tile0 + x)[(4 * g + r) * DS_PSTRIDE + c], v, acc[0][x][r]);
            if (c <= 4 * g + r) acc[0][x][r] = added;
          }
        }
      }
    }
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int t = r0 + 16 * x + 4 * g + r;
        if (t >= at.rows) continue;
        float total = fmaf(carried[x][r], decays.from_start(t), acc[0][x][r] + acc[1][x][r]);
        if (In::SKIPS) total = fmaf(in.skip(head), v_lds[t * vs + c0 + j], total);
        out[((size_t)(at.first + t) * H + head) * V + c0 + j] = total;
      }
  };
  for (int unit = wave; unit < halves * columns; unit += 8) {
    if (unit != wave) ask_state(unit / halves);
    const int first = halves == 2 ? unit % 2 * 32 : 0, last = halves == 2 ? first : 32;
#pragma unroll 1
    for (int r0 = first; r0 <= last; r0 += 32) outputs(r0, unit / halves * 16);
  }
}

__device__ inline float4 ds_raw4(const float* p) { return *reinterpret_cast<const float4*>(p); }
__device__ inline uint2 ds_raw4(const bf16_t* p) { return *reinterpret_cast<const uint2*>(p); }
__device__ inline float4 ds_widen(float4 raw) { return raw; }
__device__ inline float4 ds_widen(uint2 raw) {
  return make_float4(bf16_bits_to_f32((uint16_t)raw.x), bf16_bits_to_f32((uint16_t)(raw.x >> 16)), bf16_bits_to_f32((uint16_t)raw.y),
                     bf16_bits_to_f32((uint16_t)(raw.y >> 16)));
}

// ---- host side -----------------------------------------------------------------------------------------

inline long ds_places(int n_seqs, int n_rows) {
  return n_seqs == 1 ? ((long)n_rows + DS_ROWS - 1) / DS_ROWS : (long)n_rows / DS_ROWS + n_seqs;
}
inline size_t ds_states_lds(int D, int V) { return ((size_t)DS_ROWS * (D + 4) + (size_t)DS_ROWS * (V + 4)) * sizeof(float); }
inline size_t ds_outputs_lds(int D, int V) {
  const size_t keys = (size_t)DS_ROWS * (D + 4), behind = DS_SCORES + (size_t)DS_ROWS * (V + 4);
  return ((size_t)DS_ROWS * (D + 4) + (keys > behind ? keys : behind)) * sizeof(float);
}
// Floats of scratch memory that a step of these sizes takes; 0 where this form does not take it: sizes have to be whole tiles and
// fit a workgroup's LDS.
inline long ds_scratch_floats(int n_seqs, int n_rows, int H, int D, int V) {
  if (V > DS_MOST_VALUES || D % 32 || V % 16 || D < 64 || H > 65535 ||
      ds_outputs_lds(D, V) > 150 * 1024 || ds_states_lds(D, V) > 150 * 1024)
    return 0;
  const long places = ds_places(n_seqs, n_rows), one = (long)H * ((long)D * V + 1);
  const long most = DS_SCRATCH_FLOATS / one > 1 ? DS_SCRATCH_FLOATS / one : 1;
  return (places < most ? places : most) * one;
}

template <class In, bool WIDE>
int ds_launch_as(const In& in, const int32_t* seq_start, const int32_t* seq_slot, const int32_t* seq_to, float* home, long slot_stride, float* out, float* scratch,
              long scratch_floats, int n_seqs, int n_rows, int H, int D, int V, hipStream_t stream) {
  const long one = (long)H * ((long)D * V + 1), places = ds_places(n_seqs, n_rows);
  const int window = (int)(scratch_floats / one < places ? scratch_floats / one : places);
  BH_REQUIRE(window > 0, "scan: no scratch memory for a chunk's states");
  BH_REQUIRE((long)window * H < (1L << 30) && ((long)D * V + 1023) / 1024 <= 65535, "scan: a state of %d x %d is too large", D, V);
  const size_t states_lds = ds_states_lds(D, V), outputs_lds = ds_outputs_lds(D, V);
  bh_allow_lds<scan_states_kernel<In, WIDE>>(states_lds);
  bh_allow_lds<scan_outputs_kernel<In, WIDE>>(outputs_lds);
  float* factors = scratch + (size_t)window * H * D * V;
  for (long place = 0; place < places; place += window) {
    const int here = (int)(places - place < window ? places - place : window);
    scan_states_kernel<In, WIDE><<<ds_grid(here, H, in.shared()), 512, states_lds, stream>>>(in, seq_start, n_seqs, (int)place, here, scratch, factors, H, D, V);
    if (int status = bh_check_launch("scan_states")) return status;
    scan_combine_kernel<0><<<dim3(n_seqs, H, (D * V + 1023) / 1024), 256, 0, stream>>>(seq_start, seq_slot, seq_to, (int)place, here, scratch, factors, home,
                                                                                     slot_stride, H, D, V);
    if (int status = bh_check_launch("scan_combine")) return status;
    scan_outputs_kernel<In, WIDE><<<ds_grid(here, H, in.shared()), 512, outputs_lds, stream>>>(in, seq_start, n_seqs, (int)place, here, scratch, out, H, D, V);
    if (int status = bh_check_launch("scan_outputs")) return status;
  }
  return 0;
}

template <class In>
int ds_launch(const In& in, const int32_t* seq_start, const int32_t* seq_slot, const int32_t* seq_to, float* home, long slot_stride, float* out, float* scratch,
              long scratch_floats, int n_seqs, int n_rows, int H, int D, int V, hipStream_t stream) {
  return D > 128 || V > 128
             ? ds_launch_as<In, true>(in, seq_start, seq_slot, seq_to, home, slot_stride, out, scratch, scratch_floats, n_seqs, n_rows, H, D, V, stream)
             : ds_launch_as<In, false>(in, seq_start, seq_slot, seq_to, home, slot_stride, out, scratch, scratch_floats, n_seqs, n_rows, H, D, V, stream);
}
