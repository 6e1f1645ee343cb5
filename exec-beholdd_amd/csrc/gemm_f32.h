// Products of float32 operands on the float32 matrix instructions (gemm_f32.hip), for bh_gemm_generic.
#pragma once

#include <hip/hip_runtime.h>

#define BH_F32_FEW_ROWS 32   // up to so many activation rows a product is bound by its weights' stream

// Whether these operands go: 16-byte loads along K.
bool bh_gemm_f32_takes(const void* a, const void* w, const void* c, int K);
int bh_gemm_f32(const float* a, const float* w, float* c, int accumulate, int M, int N, int K, hipStream_t stream);
