// The gated linear recurrence whose forget gate also decides what is written (HGRN2).  Per head, with the state S
// [d, dv] in float32:
//     q = silu(z_q),  f = l + (1 - l) sigmoid(z_f + b)          (l the gate's lower bound, per head and channel)
//     S <- diag(f) S + (1 - f) v^T,   o = S^T q
// and each head's o is divided by its root mean square over dv and multiplied by a weight shared by the heads.
// Everything behind the projections z_q | z_f | v (float32) is float32; the walk over the tokens is diag_scan.h's, but in a step of
// one token a sequence (hgrn2_step_kernel).
#include <climits>
#include "diag_scan.h"
#include "yalm_hip.h"

namespace {
struct Hgrn2Op {
  static constexpr bool KEYS = false, LOW = false;
  struct Row { float bias, lower; };
  const float* proj;
  const float* f_bias;
  const float* lower;
  int Hd, N, d, dv;                               // heads * d; from one token's projections to the next one's
  __device__ Row begin(int h, int r, bool ok) const {
    return {ok ? f_bias[h * d + r] : 0.f, ok ? lower[h * d + r] : 0.f};
  }
  __device__ void fetch(int t, int h, int r, float* z) const {
    z[0] = proj[(size_t)t * N + h * d + r];
    z[1] = proj[(size_t)t * N + Hd + h * d + r];
  }
  __device__ void form(const Row& m, const float* z, const float*, float& q, float& f, float&) const {
    q = z[0] / (1.0f + expf(-z[0]));
    f = m.lower + (1.0f - m.lower) / (1.0f + expf(-(z[1] + m.bias)));
  }
  __device__ float value(int t, int h, int j) const { return proj[(size_t)t * N + 2 * Hd + h * dv + j]; }
  __device__ static float act(float v) { return v; }
  __device__ int low_size() const { return 0; }
  __device__ float low(int, int) const { return 0.f; }
};

// A step of one token a sequence (of few: it walks what it is given): a workgroup has a head's whole state in registers, eight lanes a
// column, so that the head's norm needs no launch of its own.  Bound by one trip of the state from memory and back behind one of
// the slot's number: the operands of the token are asked for beside the state.  d and dv multiples of 4 to 128.
// Eight rows (five live), 32 heads of 128 x 128, 6.3 us (21 MB of state); diag_scan_kernel and heads_norm_kernel
// took 12.2 and 4.7.  Two columns a lane group: 512 threads for 128 columns, 128 for 32, so that many small heads share a compute unit
// (800 sequences of 8 heads of 16 x 16 9.3 us, with 512 threads each 23.3, those two kernels 13.8).
constexpr int HS_MAX = 128;

template <typename T, int THREADS>
__global__ __launch_bounds__(THREADS) void hgrn2_step_kernel(Hgrn2Op op, float* __restrict__ state, const float* __restrict__ w_norm,
                                                                T* __restrict__ out, const int* __restrict__ cu_seqlens,
                                                                const int* __restrict__ seq_slot, int n_heads, int d, int dv, float eps) {
  constexpr int LANES = 8, GROUPS = THREADS / LANES, NC = 2, NV = HS_MAX / (4 * LANES);
  constexpr int VALUES = THREADS > HS_MAX ? HS_MAX : 0;       // the first of the threads that fetch a token's values
  __shared__ __attribute__((aligned(16))) float s_q[HS_MAX], s_f[HS_MAX], s_v[HS_MAX], s_o[HS_MAX];
  const int h = blockIdx.x, b = blockIdx.y, tid = threadIdx.x, group = tid / LANES, rl = tid % LANES;
  const int slot = seq_slot[b], t0 = cu_seqlens[b], t1 = cu_seqlens[b + 1], HV = n_heads * dv;
  const typename Hgrn2Op::Row mine = op.begin(h, min(tid, d - 1), tid < HS_MAX);
  if (slot < 0) {                                  // a padding row: no state is touched, its result is zeros
    for (int t = t0; t < t1; ++t)
      if (tid < dv) out[(size_t)t * HV + h * dv + tid] = from_f32<T>(0.f);
    return;
  }
  float* sp = state + ((size_t)slot * n_heads + h) * dv * d;
  float4 s[NC][NV];
#pragma unroll
  for (int c = 0; c < NC; ++c)
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int j = group + c * GROUPS, r = 4 * (rl + i * LANES);
      s[c][i] = *reinterpret_cast<const float4*>(sp + (size_t)min(j, dv - 1) * d + min(r, d - 4));      // (what lies behind is not used)
    }
  const float w0 = w_norm[min(tid % WAVE, dv - 1)], w1 = w_norm[min(tid % WAVE + WAVE, dv - 1)];
  for (int t = t0; t < t1; ++t) {
    if (tid < HS_MAX) {
      float z[2], q, f, k;
      op.fetch(t, h, min(tid, d - 1), z);
      op.form(mine, z, nullptr, q, f, k);
      s_q[tid] = tid < d ? q : 0.f;
      s_f[tid] = tid < d ? f : 0.f;
    }
    if (tid >= VALUES && tid < VALUES + HS_MAX) s_v[tid - VALUES] = op.value(t, h, min(tid - VALUES, dv - 1));
    lds_barrier();
    float sum[NC];
#pragma unroll
    for (int c = 0; c < NC; ++c) sum[c] = 0.f;
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int r = 4 * (rl + i * LANES);
      const float4 f4 = *reinterpret_cast<const float4*>(&s_f[r]), q4 = *reinterpret_cast<const float4*>(&s_q[r]);
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        const float v = s_v[group + c * GROUPS];
        float4& x = s[c][i];
        x.x = fmaf(f4.x, x.x - v, v);              // f S + (1 - f) v
        x.y = fmaf(f4.y, x.y - v, v);
        x.z = fmaf(f4.z, x.z - v, v);
        x.w = fmaf(f4.w, x.w - v, v);
        if (r < d) sum[c] += fmaf(x.w, q4.w, fmaf(x.z, q4.z, fmaf(x.y, q4.y, x.x * q4.x)));
      }
    }
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      sum[c] += quad_swap<0xB1>(sum[c]);           // lane ^ 1
      sum[c] += quad_swap<0x4E>(sum[c]);           // lane ^ 2
      sum[c] += __shfl_xor(sum[c], 4, WAVE);
      if (rl == 0) s_o[group + c * GROUPS] = sum[c];
    }
    lds_barrier();
    if (tid < WAVE) {                              // heads_norm_kernel's sum
      const float a = tid < dv ? s_o[tid] : 0.f, bb = tid + WAVE < dv ? s_o[tid + WAVE] : 0.f;
      const float f = 1.0f / sqrtf(wave_sum(fmaf(bb, bb, a * a)) / (float)dv + eps);
      T* o = out + (size_t)t * HV + h * dv + tid;
      if (tid < dv) o[0] = from_f32<T>(a * f * w0);
      if (tid + WAVE < dv) o[WAVE] = from_f32<T>(bb * f * w1);
    }
  }
#pragma unroll
  for (int c = 0; c < NC; ++c)
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int j = group + c * GROUPS, r = 4 * (rl + i * LANES);
      if (j < dv && r < d) *reinterpret_cast<float4*>(sp + (size_t)j * d + r) = s[c][i];
    }
}
}  // namespace

extern "C" int yalm_hgrn2(const float* proj, long proj_row, const float* f_bias, const float* lower, const float* w_norm, float* state,
                          float* raw, const int* cu_seqlens, const int* seq_slot, void* out, int T, int B, int n_heads,
                          int d, int dv, float eps, int out_dtype, hipStream_t stream) {
  if (T <= 0 || B <= 0) return YALM_OK;
  if (n_heads <= 0 || d <= 0 || d > 256 || dv <= 0) return YALM_ERR_ARG;
  if (out_dtype != YALM_F32 && out_dtype != YALM_BF16) return YALM_ERR_DTYPE;
  if (proj_row < 2 * n_heads * d + n_heads * dv || proj_row > INT_MAX) return YALM_ERR_ARG;
  const Hgrn2Op op = {proj, f_bias, lower, n_heads * d, (int)proj_row, d, dv};
  // one token a sequence, as the numbers say (the kernel walks whatever cu_seqlens holds; eight tokens of one sequence and none of seven
  // others, which no step of the engine is, take it 12 us and diag_scan_kernel 6)
  if (T == B && n_heads <= 65535 && B <= 65535 && d <= HS_MAX && dv <= HS_MAX && d % 4 == 0 && dv % 4 == 0 && ((uintptr_t)state & 15) == 0) {
    const dim3 grid(n_heads, B);
#define STEP(T_, THREADS_) \
  hgrn2_step_kernel<T_, THREADS_><<<grid, THREADS_, 0, stream>>>(op, state, w_norm, (T_*)out, cu_seqlens, seq_slot, n_heads, d, dv, eps)
#define STEP_OF(T_) \
  if (dv <= 32) STEP(T_, 128); else if (dv <= 64) STEP(T_, 256); else STEP(T_, 512)
    if (out_dtype == YALM_F32) { STEP_OF(float); }
    else { STEP_OF(bf16); }
#undef STEP_OF
#undef STEP
    return launch_status();
  }
  int rc;
#define SCAN(NR_, LANES_, NC_, TOK_) \
  rc = diag_scan_launch<Hgrn2Op, NR_, LANES_, NC_, TOK_>(op, state, raw, cu_seqlens, seq_slot, B, n_heads, d, dv, 0, stream)
  if (d <= 32) SCAN(4, 8, 1, 16);
  else if (d <= 64) SCAN(8, 8, 1, 16);
  // Two columns a lane group halve the reads of the operands from LDS, and pay where more than three workgroups of 32 columns share a
  // compute unit (nine prompts of 700 tokens, 32 heads of 128 x 128: 617 -> 527 us, twenty of 64 126 -> 100); with few the walk waits for itself, and
  // longer with two (2,048 tokens 534 -> 780; 640 workgroups 239 and 238).  The sums are the same.
  else if (d <= 128 && (long)B * n_heads * ceil_div(dv, 32) > 3L * compute_units()) SCAN(16, 8, 2, 16);
  else if (d <= 128) SCAN(16, 8, 1, 16);
  else SCAN(32, 8, 1, 16);
#undef SCAN
  if (rc != YALM_OK) return rc;
  return heads_norm_launch(raw, w_norm, nullptr, 0, out, T, n_heads, dv, eps, out_dtype, stream);
}
