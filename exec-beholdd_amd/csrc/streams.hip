// Several residual streams side by side, and the small elementwise steps of layers that keep their sublayer's
// result apart from the residual: the residual of a row is x[S][D] (S streams of width D, float32); a sublayer reads
// one weighted sum of the streams through an RMSNorm and its result y[D] goes back into every stream,
//   x_t <- sum_s mix[s][t] x_s + give[t] * scale[i] * y[i]        (all streams at once, from the old ones).
// With S = 1, mix = give = 1 this is a plain residual with a per-channel scale on the sublayer's result.
// Everything here is float32 arithmetic; only a norm's output takes the activation type.
#include "common.h"

#define BH_STREAMS_MOST 16

// ---- open: every stream starts as the same row -------------------------------------------------------------
__global__ void streams_open_kernel(const float* __restrict__ src, float* __restrict__ dst, int width, int streams) {
  const int row = blockIdx.x;
  const float* from = src + (size_t)row * width;
  float* to = dst + (size_t)row * streams * width;
  for (int i = threadIdx.x; i < width; i += blockDim.x) {
    const float v = from[i];
    for (int s = 0; s < streams; ++s) to[(size_t)s * width + i] = v;
  }
}

extern "C" int bh_streams_open(const float* src, float* dst, int n_rows, int width, int streams, hipStream_t stream) {
  BH_REQUIRE(n_rows > 0 && width > 0 && streams > 0, "streams_open: rows %d, width %d and streams %d must be positive",
             n_rows, width, streams);
  streams_open_kernel<<<dim3(n_rows), dim3(256), 0, stream>>>(src, dst, width, streams);
  return bh_check_launch("streams_open");
}

// ---- read: RMSNorm of a weighted sum of the streams --------------------------------------------------------
// out[r, i] = u[i] / sqrt(mean(u^2) + eps) * w[i],  u = sum_s take[s] * x[src, s, :]  (take == null: every stream once),
// src = rows ? rows[r] : r.  PER > 0: the row fits PER elements a thread and u stays in registers; PER == 0: u is
// formed twice.
template <typename TO, int PER>
__global__ void streams_rmsnorm_kernel(const float* __restrict__ x, const int32_t* __restrict__ rows,
                                       const float* __restrict__ take, const float* __restrict__ w, TO* __restrict__ out,
                                       int width, int streams, float eps, int block_rows) {
  __shared__ float scratch[16];
  __shared__ float share[BH_STREAMS_MOST];
  const int r = blockIdx.x;
  const int src = rows ? rows[r] : r;
  const float* xr = x + (size_t)src * streams * width;
  if (threadIdx.x < streams) share[threadIdx.x] = take ? take[threadIdx.x] : 1.f;
  __syncthreads();
  auto mixed = [&](int i) {
    float u = 0.f;
    for (int s = 0; s < streams; ++s) u = fmaf(share[s], xr[(size_t)s * width + i], u);
    return u;
  };
  auto at = [&](int i) { return out + bh_rows_index(block_rows, r, i, width); };
  float ss = 0.f;
  if (PER > 0) {
    float uv[PER > 0 ? PER : 1];
#pragma unroll
    for (int j = 0; j < PER; ++j) {
      const int i = threadIdx.x + j * blockDim.x;
      uv[j] = i < width ? mixed(i) : 0.f;
      ss += uv[j] * uv[j];
    }
    ss = block_sum(ss, scratch);
    const float inv = 1.0f / sqrtf(ss / (float)width + eps);
#pragma unroll
    for (int j = 0; j < PER; ++j) {
      const int i = threadIdx.x + j * blockDim.x;
      if (i < width) *at(i) = from_f32<TO>(uv[j] * inv * (w ? w[i] : 1.f));
    }
    return;
  }
  for (int i = threadIdx.x; i < width; i += blockDim.x) {
    const float u = mixed(i);
    ss += u * u;
  }
  ss = block_sum(ss, scratch);
  const float inv = 1.0f / sqrtf(ss / (float)width + eps);
  for (int i = threadIdx.x; i < width; i += blockDim.x) *at(i) = from_f32<TO>(mixed(i) * inv * (w ? w[i] : 1.f));
}

template <typename TO>
static void launch_streams_rmsnorm(const float* x, const int32_t* rows, const float* take, const float* w, void* out,
                                   int n_rows, int width, int streams, float eps, int block_rows, hipStream_t stream) {
  const int threads = width >= 4096 ? 1024 : (width >= 1024 ? 512 : 256);
  const int per = (width + threads - 1) / threads;
  dim3 grid(n_rows), block(threads);
#define BH_SNORM(PER) \
  streams_rmsnorm_kernel<TO, PER><<<grid, block, 0, stream>>>(x, rows, take, w, (TO*)out, width, streams, eps, block_rows)
  if (per <= 4) BH_SNORM(4);
  else if (per <= 8) BH_SNORM(8);
  else BH_SNORM(0);
#undef BH_SNORM
}

extern "C" int bh_streams_rmsnorm(const float* x, const int32_t* rows, const float* take, const float* w, void* out,
                                  int out_dtype, int n_rows, int width, int streams, float eps, int out_block_rows,
                                  hipStream_t stream) {
  BH_REQUIRE(n_rows > 0 && width > 0, "streams_rmsnorm: rows %d and width %d must be positive", n_rows, width);
  BH_REQUIRE(streams >= 1 && streams <= BH_STREAMS_MOST, "streams_rmsnorm: 1 to %d streams, not %d", BH_STREAMS_MOST, streams);
  BH_REQUIRE(eps >= 0.f, "streams_rmsnorm: eps must not be negative");
  BH_REQUIRE(out_block_rows == 0 || ((out_block_rows == 8 || out_block_rows == 16) && out_dtype == BH_BF16 && width % 32 == 0),
             "streams_rmsnorm: rows in blocks of %d need bfloat16 and a width that is a multiple of 32 (got %d)",
             out_block_rows, width);
  if (out_dtype == BH_F32) launch_streams_rmsnorm<float>(x, rows, take, w, out, n_rows, width, streams, eps, out_block_rows, stream);
  else if (out_dtype == BH_BF16) launch_streams_rmsnorm<bf16_t>(x, rows, take, w, out, n_rows, width, streams, eps, out_block_rows, stream);
  else return bh_fail("streams_rmsnorm: unknown output dtype %d", out_dtype);
  return bh_check_launch("streams_rmsnorm");
}

// ---- write: a sublayer's result goes back into every stream ------------------------------------------------
__global__ __launch_bounds__(256) void streams_update_kernel(float* __restrict__ x, const float* __restrict__ y,
                                                             const float* __restrict__ mix, const float* __restrict__ give,
                                                             const float* __restrict__ scale, int width, int streams,
                                                             size_t total) {
  __shared__ float m[BH_STREAMS_MOST * BH_STREAMS_MOST];
  __shared__ float g[BH_STREAMS_MOST];
  for (int e = threadIdx.x; e < streams * streams; e += blockDim.x) m[e] = mix ? mix[e] : (e / streams == e % streams ? 1.f : 0.f);
  if (threadIdx.x < streams) g[threadIdx.x] = give ? give[threadIdx.x] : 1.f;
  __syncthreads();
  const size_t at = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (at >= total) return;
  const size_t row = at / width;
  const int i = (int)(at % width);
  float* xr = x + row * streams * width + i;
  float old[BH_STREAMS_MOST];
  for (int s = 0; s < streams; ++s) old[s] = xr[(size_t)s * width];
  const float add = (scale ? scale[i] : 1.f) * y[at];
  for (int t = 0; t < streams; ++t) {
    float v = 0.f;
    for (int s = 0; s < streams; ++s) v = fmaf(m[s * streams + t], old[s], v);
    xr[(size_t)t * width] = fmaf(g[t], add, v);
  }
}

// The same for up to four streams whose width is a multiple of 4, a 16-byte piece of a row a thread.
template <int S>
__global__ __launch_bounds__(256) void streams_update_wide_kernel(float* __restrict__ x, const float* __restrict__ y, const float* __restrict__ mix,
                                                                  const float* __restrict__ give, const float* __restrict__ scale, int pieces) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= pieces) return;
  float4* xr = reinterpret_cast<float4*>(x) + (size_t)blockIdx.y * S * pieces + i;
  float4 old[S];
#pragma unroll
  for (int s = 0; s < S; ++s) old[s] = xr[s * pieces];
  const float4 c = scale ? reinterpret_cast<const float4*>(scale)[i] : float4{1.f, 1.f, 1.f, 1.f};
  float4 a = reinterpret_cast<const float4*>(y)[(size_t)blockIdx.y * pieces + i];
  a = float4{c.x * a.x, c.y * a.y, c.z * a.z, c.w * a.w};
#pragma unroll
  for (int t = 0; t < S; ++t) {
    const float g = give ? give[t] : 1.f;
    float4 v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < S; ++s) {
      const float m = mix ? mix[s * S + t] : (s == t ? 1.f : 0.f);
      v = float4{fmaf(m, old[s].x, v.x), fmaf(m, old[s].y, v.y), fmaf(m, old[s].z, v.z), fmaf(m, old[s].w, v.w)};
    }
    xr[t * pieces] = float4{fmaf(g, a.x, v.x), fmaf(g, a.y, v.y), fmaf(g, a.z, v.z), fmaf(g, a.w, v.w)};
  }
}

extern "C" int bh_streams_update(float* x, const float* y, const float* mix, const float* give, const float* scale,
                                 int n_rows, int width, int streams, hipStream_t stream) {
  BH_REQUIRE(n_rows > 0 && width > 0, "streams_update: rows %d and width %d must be positive", n_rows, width);
  BH_REQUIRE(streams >= 1 && streams <= BH_STREAMS_MOST, "streams_update: 1 to %d streams, not %d", BH_STREAMS_MOST, streams);
  if (streams <= 4 && width % 4 == 0 && n_rows <= 65535 && (((uintptr_t)x | (uintptr_t)y | (uintptr_t)scale) % 16) == 0) {
    const dim3 grid((width / 4 + 255) / 256, n_rows);
    if (streams == 1) streams_update_wide_kernel<1><<<grid, 256, 0, stream>>>(x, y, mix, give, scale, width / 4);
    else if (streams == 2) streams_update_wide_kernel<2><<<grid, 256, 0, stream>>>(x, y, mix, give, scale, width / 4);
    else if (streams == 3) streams_update_wide_kernel<3><<<grid, 256, 0, stream>>>(x, y, mix, give, scale, width / 4);
    else streams_update_wide_kernel<4><<<grid, 256, 0, stream>>>(x, y, mix, give, scale, width / 4);
    return bh_check_launch("streams_update");
  }
  const size_t total = (size_t)n_rows * width;
  const size_t blocks = (total + 255) / 256;
  BH_REQUIRE(blocks <= 2147483647u, "streams_update: too many elements");
  streams_update_kernel<<<dim3((unsigned)blocks), dim3(256), 0, stream>>>(x, y, mix, give, scale, width, streams, total);
  return bh_check_launch("streams_update");
}

// ---- write, and read for the sublayer that follows, in one pass ---------------------------------------------------
// streams_update for one row, then streams_rmsnorm of the row as it has become (with the next sublayer's `take` and
// norm weight): a workgroup per row; a thread keeps the next sublayer's sum of its elements while it writes the streams.
template <typename TO, int PER>
__global__ void streams_update_rmsnorm_kernel(float* __restrict__ x, const float* __restrict__ y, const float* __restrict__ mix,
                                              const float* __restrict__ give, const float* __restrict__ scale,
                                              const float* __restrict__ take, const float* __restrict__ w, TO* __restrict__ out,
                                              int width, int streams, float eps, int block_rows) {
  __shared__ float scratch[16];
  __shared__ float m[BH_STREAMS_MOST * BH_STREAMS_MOST];
  __shared__ float g[BH_STREAMS_MOST], share[BH_STREAMS_MOST];
  const int r = blockIdx.x;
  for (int e = threadIdx.x; e < streams * streams; e += blockDim.x) m[e] = mix ? mix[e] : (e / streams == e % streams ? 1.f : 0.f);
  if (threadIdx.x < streams) {
    g[threadIdx.x] = give ? give[threadIdx.x] : 1.f;
    share[threadIdx.x] = take ? take[threadIdx.x] : 1.f;
  }
  __syncthreads();
  float* xr = x + (size_t)r * streams * width;
  const float* yr = y + (size_t)r * width;
  auto renew = [&](int i) {      // the streams' element i as it becomes, written; returns the next sublayer's sum of it
    float old[BH_STREAMS_MOST];
    for (int s = 0; s < streams; ++s) old[s] = xr[(size_t)s * width + i];
    const float add = (scale ? scale[i] : 1.f) * yr[i];
    float u = 0.f;
    for (int t = 0; t < streams; ++t) {
      float v = 0.f;
      for (int s = 0; s < streams; ++s) v = fmaf(m[s * streams + t], old[s], v);
      v = fmaf(g[t], add, v);
      xr[(size_t)t * width + i] = v;
      u = fmaf(share[t], v, u);
    }
    return u;
  };
  auto at = [&](int i) { return out + bh_rows_index(block_rows, r, i, width); };
  float ss = 0.f;
  if (PER > 0) {
    float uv[PER > 0 ? PER : 1];
#pragma unroll
    for (int j = 0; j < PER; ++j) {
      const int i = threadIdx.x + j * blockDim.x;
      uv[j] = i < width ? renew(i) : 0.f;
      ss += uv[j] * uv[j];
    }
    ss = block_sum(ss, scratch);
    const float inv = 1.0f / sqrtf(ss / (float)width + eps);
#pragma unroll
    for (int j = 0; j < PER; ++j) {
      const int i = threadIdx.x + j * blockDim.x;
      if (i < width) *at(i) = from_f32<TO>(uv[j] * inv * (w ? w[i] : 1.f));
    }
    return;
  }
  for (int i = threadIdx.x; i < width; i += blockDim.x) {
    const float u = renew(i);
    ss += u * u;
  }
  ss = block_sum(ss, scratch);
  const float inv = 1.0f / sqrtf(ss / (float)width + eps);
  for (int i = threadIdx.x; i < width; i += blockDim.x) {      // a thread reads back what it wrote itself
    float u = 0.f;
    for (int t = 0; t < streams; ++t) u = fmaf(share[t], xr[(size_t)t * width + i], u);
    *at(i) = from_f32<TO>(u * inv * (w ? w[i] : 1.f));
  }
}

// The same for up to four streams whose width is a multiple of 4, in 16-byte pieces: a thread keeps PER pieces between the statistic
// and the write, and has all of its loads on their way together.
// Bound by the streams' way from memory and back.  Measured, two streams, bfloat16 out: 2,048 rows of 2,048 19 us (31 with an element a
// load and a loop over the streams), 16 rows of 4,096 4.9 us (12.2).
template <typename TO, int S, int PER, bool SPREAD>
__global__ void streams_update_rmsnorm_wide_kernel(float* __restrict__ x, const float* __restrict__ y, const float* __restrict__ mix,
                                                   const float* __restrict__ give, const float* __restrict__ scale,
                                                   const float* __restrict__ take, const float* __restrict__ w, TO* __restrict__ out,
                                                   int n_rows, int width, float eps, int block_rows) {
  __shared__ float scratch[16];
  const int r = bh_row_of_block<SPREAD>(), pieces = width / 4;
  if (SPREAD && r >= n_rows) return;
  float4* xr = reinterpret_cast<float4*>(x + (size_t)r * S * width);
  const float4* yr = reinterpret_cast<const float4*>(y + (size_t)r * width);
  const float4* scales = reinterpret_cast<const float4*>(scale);
  const float4* weights = reinterpret_cast<const float4*>(w);
  constexpr bool SOON = S <= 2;      // whether the registers hold the scales beside the streams
  float4 old[PER][S], add[PER], by[SOON ? PER : 1];
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    const int i = threadIdx.x + j * blockDim.x;
    if (i < pieces) {
#pragma unroll
      for (int s = 0; s < S; ++s) old[j][s] = xr[s * pieces + i];
      add[j] = yr[i];
      if constexpr (SOON) by[j] = scales ? scales[i] : float4{1.f, 1.f, 1.f, 1.f};
    }
  }
  float m[S][S], g[S], share[S];
#pragma unroll
  for (int t = 0; t < S; ++t) {
    g[t] = give ? give[t] : 1.f;
    share[t] = take ? take[t] : 1.f;
#pragma unroll
    for (int s = 0; s < S; ++s) m[s][t] = mix ? mix[s * S + t] : (s == t ? 1.f : 0.f);
  }
  float4 kept[PER];
  float ss = 0.f;
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    const int i = threadIdx.x + j * blockDim.x;
    kept[j] = float4{0.f, 0.f, 0.f, 0.f};
    if (i < pieces) {
      float4 c;
      if constexpr (SOON) c = by[j];
      else c = scales ? scales[i] : float4{1.f, 1.f, 1.f, 1.f};
      const float4 a = {c.x * add[j].x, c.y * add[j].y, c.z * add[j].z, c.w * add[j].w};
#pragma unroll
      for (int t = 0; t < S; ++t) {
        float4 v = {m[0][t] * old[j][0].x, m[0][t] * old[j][0].y, m[0][t] * old[j][0].z, m[0][t] * old[j][0].w};
#pragma unroll
        for (int s = 1; s < S; ++s)
          v = float4{fmaf(m[s][t], old[j][s].x, v.x), fmaf(m[s][t], old[j][s].y, v.y), fmaf(m[s][t], old[j][s].z, v.z), fmaf(m[s][t], old[j][s].w, v.w)};
        v = float4{fmaf(g[t], a.x, v.x), fmaf(g[t], a.y, v.y), fmaf(g[t], a.z, v.z), fmaf(g[t], a.w, v.w)};
        xr[t * pieces + i] = v;
        kept[j] = float4{fmaf(share[t], v.x, kept[j].x), fmaf(share[t], v.y, kept[j].y), fmaf(share[t], v.z, kept[j].z), fmaf(share[t], v.w, kept[j].w)};
      }
    }
    ss += fmaf(kept[j].w, kept[j].w, fmaf(kept[j].z, kept[j].z, fmaf(kept[j].x, kept[j].x, kept[j].y * kept[j].y)));
  }
  ss = block_sum(ss, scratch);
  const float inv = 1.0f / sqrtf(ss / (float)width + eps);
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    const int i = threadIdx.x + j * blockDim.x;
    if (i < pieces) {
      const float4 c = weights ? weights[i] : float4{1.f, 1.f, 1.f, 1.f};
      // four neighbouring columns lie together in rows and in blocks alike
      store_four(out + bh_rows_index(block_rows, r, 4 * i, width), kept[j].x * inv * c.x, kept[j].y * inv * c.y, kept[j].z * inv * c.z, kept[j].w * inv * c.w);
    }
  }
}

extern "C" int bh_streams_update_rmsnorm(float* x, const float* y, const float* mix, const float* give, const float* scale,
                                         const float* take, const float* w, void* out, int out_dtype, int n_rows, int width,
                                         int streams, float eps, int out_block_rows, hipStream_t stream) {
  BH_REQUIRE(n_rows > 0 && width > 0, "streams_update_rmsnorm: rows %d and width %d must be positive", n_rows, width);
  BH_REQUIRE(streams >= 1 && streams <= BH_STREAMS_MOST, "streams_update_rmsnorm: 1 to %d streams, not %d", BH_STREAMS_MOST, streams);
  BH_REQUIRE(eps >= 0.f, "streams_update_rmsnorm: eps must not be negative");
  BH_REQUIRE(out_block_rows == 0 || ((out_block_rows == 8 || out_block_rows == 16) && out_dtype == BH_BF16 && width % 32 == 0),
             "streams_update_rmsnorm: rows in blocks of %d need bfloat16 and a width that is a multiple of 32 (got %d)",
             out_block_rows, width);
  const bool on16 = (((uintptr_t)x | (uintptr_t)y | (uintptr_t)scale | (uintptr_t)w | (uintptr_t)out) % 16) == 0;
  if (streams <= 4 && on16 && width % 4 == 0 && width <= 4 * 8 * 256 && (out_dtype == BH_F32 || out_dtype == BH_BF16)) {
    // few rows: many waves a row; many rows fill the chip by themselves (several streams of the widest rows in four pieces a thread,
    // which is what the registers hold)
    const int pieces = width / 4, most = n_rows < bh_compute_units() / 4 ? 1024 : streams > 1 && pieces > 1024 ? 512 : 256;
    const int threads = pieces >= most ? most : (pieces + BH_WAVE - 1) / BH_WAVE * BH_WAVE, per = (pieces + threads - 1) / threads;
#define BH_WIDE(TO, S, PER)                                                                                                          \
  BH_BY_ROWS(TO, n_rows, out_block_rows, threads, stream, (x, y, mix, give, scale, take, w, (TO*)out, n_rows, width, eps, out_block_rows), \
             streams_update_rmsnorm_wide_kernel, TO, S, PER)
#define BH_WIDE_SIZES(TO, S)            \
  do {                                  \
    if (per == 1) BH_WIDE(TO, S, 1);    \
    else if (per == 2) BH_WIDE(TO, S, 2); \
    else if (S > 1 || per <= 4) BH_WIDE(TO, S, 4); \
    else BH_WIDE(TO, S, (S > 1 ? 4 : 8)); \
  } while (0)
#define BH_WIDE_STREAMS(TO)                  \
  do {                                       \
    if (streams == 1) BH_WIDE_SIZES(TO, 1);  \
    else if (streams == 2) BH_WIDE_SIZES(TO, 2); \
    else if (streams == 3) BH_WIDE_SIZES(TO, 3); \
    else BH_WIDE_SIZES(TO, 4);               \
  } while (0)
    if (out_dtype == BH_F32) BH_WIDE_STREAMS(float);
    else BH_WIDE_STREAMS(bf16_t);
#undef BH_WIDE_STREAMS
#undef BH_WIDE_SIZES
#undef BH_WIDE
    return bh_check_launch("streams_update_rmsnorm");
  }
  const int threads = width >= 4096 ? 1024 : (width >= 1024 ? 512 : 256);
  const int per = (width + threads - 1) / threads;
  dim3 grid(n_rows), block(threads);
#define BH_SUN(TO, PER)                                                                                                  \
  streams_update_rmsnorm_kernel<TO, PER><<<grid, block, 0, stream>>>(x, y, mix, give, scale, take, w, (TO*)out, width, streams, \
                                                                     eps, out_block_rows)
#define BH_SUN_SIZES(TO)           \
  do {                             \
    if (per <= 4) BH_SUN(TO, 4);   \
    else if (per <= 8) BH_SUN(TO, 8); \
    else BH_SUN(TO, 0);            \
  } while (0)
  if (out_dtype == BH_F32) BH_SUN_SIZES(float);
  else if (out_dtype == BH_BF16) BH_SUN_SIZES(bf16_t);
  else return bh_fail("streams_update_rmsnorm: unknown output dtype %d", out_dtype);
#undef BH_SUN_SIZES
#undef BH_SUN
  return bh_check_launch("streams_update_rmsnorm");
}

// ---- small elementwise steps ---------------------------------------------------------------------------------
__global__ void scale_kernel(float* __restrict__ x, float factor, size_t total) {
  const size_t at = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (at < total) x[at] *= factor;
}

extern "C" int bh_scale(float* x, long total, float factor, hipStream_t stream) {
  BH_REQUIRE(total > 0, "scale: nothing to scale");
  const size_t blocks = ((size_t)total + 255) / 256;
  BH_REQUIRE(blocks <= 2147483647u, "scale: too many elements");
  scale_kernel<<<dim3((unsigned)blocks), dim3(256), 0, stream>>>(x, factor, (size_t)total);
  return bh_check_launch("scale");
}

// out <- max(x, 0)^2 (out may be x itself), in float32 whatever the element type; the output's rows one after the other
// or in blocks of rows (bh_rows_index)
template <typename T>
__global__ void relu_squared_kernel(const T* __restrict__ x, T* __restrict__ out, int width, size_t total, int block_rows) {
  const size_t at = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (at >= total) return;
  const float v = fmaxf(to_f32(x[at]), 0.f);
  const size_t to = block_rows ? (size_t)bh_rows_index(block_rows, (int)(at / width), (int)(at % width), width) : at;
  out[to] = from_f32<T>(v * v);
}

// The same in pieces of 16 bytes (4 or 8 neighbouring columns, which lie together in rows and in blocks alike): a thread one piece.
// 2,048 x 6,144 bfloat16 into blocks 13 us, 32 with an element a thread (a division and a 2-byte store each).
template <typename T>
__global__ __launch_bounds__(256) void relu_squared_pieces_kernel(const T* __restrict__ x, T* __restrict__ out, int n_rows, int width, int block_rows) {
  constexpr int N = 16 / sizeof(T);
  const int row = bh_row_of_block(block_rows), i = N * (blockIdx.y * blockDim.x + threadIdx.x);
  if (row >= n_rows || i >= width) return;
  union {
    uint4 raw;
    T v[N];
  } piece;
  piece.raw = *reinterpret_cast<const uint4*>(x + (size_t)row * width + i);
#pragma unroll
  for (int e = 0; e < N; ++e) {
    const float v = fmaxf(to_f32(piece.v[e]), 0.f);
    piece.v[e] = from_f32<T>(v * v);
  }
  *reinterpret_cast<uint4*>(out + bh_rows_index(block_rows, row, i, width)) = piece.raw;
}

extern "C" int bh_relu_squared(const void* x, void* out, int dtype, int n_rows, int width, int out_block_rows, hipStream_t stream) {
  BH_REQUIRE(n_rows > 0 && width > 0, "relu_squared: nothing to do");
  BH_REQUIRE(out_block_rows == 0 || ((out_block_rows == 8 || out_block_rows == 16) && dtype == BH_BF16 && width % 32 == 0 && x != out),
             "relu_squared: rows in blocks of %d need bfloat16, a width that is a multiple of 32 (got %d) and an output of their own",
             out_block_rows, width);
  // (rows of bfloat16 that are less than a wave's pieces: 8,160 x 256 4.0 us an element a thread, 4.3 in pieces)
  if ((dtype == BH_F32 || (bh_pieces_pay((long)n_rows * width) && (out_block_rows || width >= 8 * BH_WAVE))) && width <= 8 * 256 * 65535 / 2 && (((uintptr_t)x | (uintptr_t)out) % 16) == 0 && ((dtype == BH_F32 && width % 4 == 0) || (dtype == BH_BF16 && width % 8 == 0))) {
    const int pieces = width / (dtype == BH_F32 ? 4 : 8);
    const dim3 grid(bh_rows_grid(n_rows, out_block_rows), (pieces + 255) / 256), block(bh_piece_threads(pieces));
    if (dtype == BH_F32) relu_squared_pieces_kernel<float><<<grid, block, 0, stream>>>((const float*)x, (float*)out, n_rows, width, out_block_rows);
    else relu_squared_pieces_kernel<bf16_t><<<grid, block, 0, stream>>>((const bf16_t*)x, (bf16_t*)out, n_rows, width, out_block_rows);
    return bh_check_launch("relu_squared");
  }
  const size_t total = (size_t)n_rows * width;
  const size_t blocks = (total + 255) / 256;
  BH_REQUIRE(blocks <= 2147483647u, "relu_squared: too many elements");
  if (dtype == BH_F32)
    relu_squared_kernel<float><<<dim3((unsigned)blocks), dim3(256), 0, stream>>>((const float*)x, (float*)out, width, total, out_block_rows);
  else if (dtype == BH_BF16)
    relu_squared_kernel<bf16_t><<<dim3((unsigned)blocks), dim3(256), 0, stream>>>((const bf16_t*)x, (bf16_t*)out, width, total, out_block_rows);
  else return bh_fail("relu_squared: unknown dtype %d", dtype);
  return bh_check_launch("relu_squared");
}
