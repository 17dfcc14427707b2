// The float32 product on the matrix cores (gemm_f32.hip), for the entry point in gemm_tiled.hip.
#pragma once

#include "common.h"

bool gemm_f32_takes(const void* x, const void* w, int K, long long ldx, long long ldw);
bool gemm_f32_launch(float* out, const float* x, const float* w, int M, int N, int K, long long ldx, long long ldw,
                     long long ldo, hipStream_t stream);
