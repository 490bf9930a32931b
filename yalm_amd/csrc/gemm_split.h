// Float32 products of more than 64 rows by bfloat16 terms (gemm_split.hip), for gemm_f32.hip, which asks before it takes a
// product itself.
#pragma once
#include "common.h"

// The tile whose estimated time is the least and below `than` us, or -1: none is (or the product is not one for this kernel).
int yalm_gemm_split_choose(int M, int N, int K, bool gate, double than);
// K a multiple of 32, A and W on 16 bytes, `tile` as chosen; epilogues as yalm_gemm.
int yalm_gemm_split(int tile, const float* A, const float* W, float* C, int M, int N, int K, int epilogue, GateOut H, hipStream_t stream);
