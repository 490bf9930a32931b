// The sum of squares that a row's RMS norm divides by, in one order wherever it is formed: a norm that a kernel in front applies
// on its way has the bits of the norm's own kernel (a faint read-out behind it magnifies a last bit a thousandfold).
#pragma once
#include "common.h"

// Rows of more than 1,024 to 8,192 elements, a multiple of 4 on 16 bytes: four waves, 16 bytes a load, the row kept in registers.
// Other rows: element by element, four waves, or one wave up to 1,024 elements.
constexpr int RMS_VEC_MAX = 8;
inline bool rms_row_vec(const void* x, const void* out, int D) {
  return D % 4 == 0 && D > 1024 && D <= 256 * 4 * RMS_VEC_MAX && !((uintptr_t)x & 15) && !((uintptr_t)out & 15);
}

__device__ __forceinline__ float rms_add4(float ss, float4 v) {      // written out: which product is rounded by itself is not left open
  return ss + fmaf(v.w, v.w, fmaf(v.z, v.z, fmaf(v.y, v.y, v.x * v.x)));
}

// This thread's part of the sum over x[D] (element by element; tid of n threads)
__device__ __forceinline__ float rms_part(const float* x, int D, int tid, int n) {
  float ss = 0.f;
  for (int i = tid; i < D; i += n) ss = fmaf(x[i], x[i], ss);
  return ss;
}

// The whole sum for a row in LDS, by the first waves of a workgroup; every thread of the workgroup gets it.  VEC: rms_row_vec.
// red: four floats.
__device__ __forceinline__ float rms_sum_of_lds(const float* x, int D, bool vec, float* red) {
  const int tid = threadIdx.x, waves = D > 1024 ? 4 : 1;
  float ss = 0.f;
  if (tid < waves * WAVE) {
    if (vec) {
      const float4* x4 = reinterpret_cast<const float4*>(x);
#pragma unroll
      for (int u = 0; u < RMS_VEC_MAX; ++u) {
        const int i = tid + u * 256;
        ss = rms_add4(ss, i < D / 4 ? x4[i] : make_float4(0.f, 0.f, 0.f, 0.f));
      }
    } else {
      ss = rms_part(x, D, tid, waves * WAVE);
    }
    ss = wave_sum(ss);
    if (tid % WAVE == 0) red[tid / WAVE] = ss;
  }
  __syncthreads();
  if (waves == 1) return red[0];
  float s = 0.f;
#pragma unroll
  for (int i = 0; i < 4; ++i) s += red[i];
  return s;
}
