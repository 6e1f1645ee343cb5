// The state of a short convolution over time (short_conv.hip), as the kernels that make the convolution leave it on their way.
#pragma once
#include "common.h"

#define SC_MAX_TAPS 16

// What the next step's convolution of channel c starts with, the last taps - 1 inputs of a sequence whose rows of this step are start ..
// start + n_new - 1: from them and, where they are fewer, from `old`.  `to` may be `old`: all is read before anything is written.
template <typename T>
__device__ inline void sc_leave_inputs(const T* __restrict__ u, int row_stride, int column, int start, int n_new, int taps, const float* old, float* to,
                                       int channels, int c) {
  const int keep = taps - 1;
  float next[SC_MAX_TAPS];
#pragma unroll
  for (int s = 0; s < SC_MAX_TAPS; ++s) {
    if (s >= keep) break;
    const int at = n_new + s - keep;        // index into the step's rows; negative: still an old input
    next[s] = at >= 0 ? to_f32(u[(size_t)(start + at) * row_stride + column]) : old[(size_t)(n_new + s) * channels + c];
  }
#pragma unroll
  for (int s = 0; s < SC_MAX_TAPS; ++s) {
    if (s >= keep) break;
    to[(size_t)s * channels + c] = next[s];
  }
}
