// The gated linear recurrence whose forget gate also decides what is written (HGRN2).  Per head, with the state S
// [d, dv] in float32:
//     q = silu(z_q),  f = l + (1 - l) sigmoid(z_f + b)          (l the gate's lower bound, per head and channel)
//     S <- diag(f) S + (1 - f) v^T,   o = S^T q
// and each head's o is divided by its root mean square over dv and multiplied by a weight shared by the heads.
// Everything behind the projections z_q | z_f | v (float32) is float32; the walk over the tokens is diag_scan.h's, but in a step of
// one token a sequence (hgrn2_step_kernel).
//
// Prompts go a tile of 64 tokens at a time on the matrix cores, in float32 (v_mfma_f32_16x16x4_f32).  With F(s, t) the product of the
// gates of the tokens behind s up to and including t (a number a channel),
//     o_t = (q_t F(start, t)) S_0 + sum over s <= t of (sum over channels of q_t F(s, t) (1 - f_s)) v_s,
//     S_64 = diag(F(start, 63)) S_0 + sum over s of (F(s, 63) (1 - f_s)) v_s^T.
// Every F is a product of gates, formed factor by factor: no quotient, no logarithm, so that gates of 0 and of 1 and runs of small ones
// are exact where the walk is.  hgrn2_tiles_kernel (every tile and head at once) makes the scaled operands and the second sum of o;
// tile_scan.h's walk over the tiles the products with S_0 and the state.  Between two tokens of different blocks F is cut at the blocks'
// borders into factors of the one, of the blocks between and of the other, which makes the sum over channels a matrix product: blocks of 16
// tokens, halves of one and quarters of one; inside four tokens every pair's product is carried on from token to token.
#include <cfloat>
#include <climits>
#include "tile_scan.h"
#include "yalm_hip.h"

namespace {
struct Hgrn2Op {
  static constexpr bool KEYS = false, LOW = false;
  struct Row { float bias, lower; };
  const float* proj;
  const float* f_bias;
  const float* lower;
  int Hd, N, d, dv, Hv;                           // heads * d; from one token's projections to the next one's; heads * dv
  __device__ Row begin(int h, int r, bool ok) const {
    return {ok ? f_bias[h * d + r] : 0.f, ok ? lower[h * d + r] : 0.f};
  }
  __device__ void fetch(int t, int h, int r, float* z) const {
    z[0] = proj[(size_t)t * N + h * d + r];
    z[1] = proj[(size_t)t * N + Hd + h * d + r];
  }
  // k = 1 - f as (1 - lower) e / (1 + e), e = e^-z, where that keeps digits: of an f close to one the rounding would be most of 1 - f
  __device__ void form(const Row& m, const float* z, const float*, float& q, float& f, float& k) const {
    q = z[0] / (1.0f + expf(-z[0]));
    const float e = expf(-(z[1] + m.bias)), free = 1.0f - m.lower, open = free / (1.0f + e);
    f = m.lower + open;
    k = e > 1.0f ? free - open : open * e;
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

// The gate of a result that stands beside the recurrence's (yalm_sigmoid_gate's: o *= sigmoid(g)), done by further workgroups of a step's
// launch: both wait for nothing but the product in front, and alone each is a launch of 4.6 us and more that moves next to nothing (five
// tokens, 32 heads of 128: 5.9 + 4.6 -> 6.4 us).
template <typename T>
struct SideGate {
  T* o;
  const float* g;
  long g_stride;
  int n_heads, dv, pad, blocks;                   // blocks: workgroups a token, behind the heads' (0: none)
};

template <typename T, int THREADS>
__global__ __launch_bounds__(THREADS) void hgrn2_step_kernel(Hgrn2Op op, float* __restrict__ state, const float* __restrict__ w_norm,
                                                                T* __restrict__ out, const int* __restrict__ cu_seqlens,
                                                                const int* __restrict__ seq_slot, int n_heads, int d, int dv, float eps,
                                                                SideGate<T> gate) {
  constexpr int LANES = 8, GROUPS = THREADS / LANES, NC = 2, NV = HS_MAX / (4 * LANES);
  constexpr int VALUES = THREADS > HS_MAX ? HS_MAX : 0;       // the first of the threads that fetch a token's values
  __shared__ __attribute__((aligned(16))) float s_q[HS_MAX], s_f[HS_MAX], s_v[HS_MAX], s_o[HS_MAX];
  const int h = blockIdx.x, b = blockIdx.y, tid = threadIdx.x, group = tid / LANES, rl = tid % LANES;
  if (h >= n_heads) {                              // token b's gate, 16 bytes of the result a thread
    constexpr int VEC = 16 / sizeof(T);
    const int i = ((h - n_heads) * THREADS + tid) * VEC;
    if (i >= gate.n_heads * gate.dv) return;
    T* p = gate.o + ((size_t)b * gate.n_heads + i / gate.dv) * gate.pad + i % gate.dv;
    const float* g = gate.g + (size_t)b * gate.g_stride + i;
    typedef __attribute__((ext_vector_type(VEC))) T Vec;
    Vec v = *reinterpret_cast<const Vec*>(p);
    float z[VEC];
#pragma unroll
    for (int k = 0; k < VEC; k += 4) {
      const float4 z4 = *reinterpret_cast<const float4*>(g + k);
      z[k] = z4.x, z[k + 1] = z4.y, z[k + 2] = z4.z, z[k + 3] = z4.w;
    }
#pragma unroll
    for (int k = 0; k < VEC; ++k) v[k] = from_f32<T>(to_f32(static_cast<T>(v[k])) / (1.0f + expf(-z[k])));
    *reinterpret_cast<Vec*>(p) = v;
    return;
  }
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

namespace {
constexpr int HT_HALF = 8, HT_QUAD = 4;          // tokens of half a block, of a quarter

size_t hgrn2_tiles_lds(int dp) { return ((size_t)4 * GT * (dp + 4) + GNB * dp + (size_t)GT * GA_ROW) * sizeof(float); }

// qd [tile][head][64][DP], kd [tile][head][DP][64] and gd [tile][head][DP] as tile_scan.h wants them; raw = the second sum of o.
// A thread owns one channel of one block of 16 tokens.  LDS (155 KB at DP 128: a workgroup of eight waves a compute unit): four rows
// a token, first q, 1 - f and f; then q F(block's start, t), (1 - f) F(t, block's end) and, for the halves of a block, q F(half's start, t)
// in the second and (1 - f) F(t, half's end) in the first, and the same for the quarters of a half.
// Bound by its phases one behind the other, 18 us a workgroup: the operands' way in 3, their gates 5 (the walk's own form, two exponentials and
// two divisions), the scaled rows through LDS 4, the products 2, the rest barriers and the way out (five prompts of 255 to 509 tokens, 32 heads
// of 128 x 128, 960 workgroups, inside a step: 92 us, the walk over the tiles behind it 100, the heads' norm 10; one behind the other with warm
// caches 174 in all, token by token 228).  Errors against 64 bits, relative, of
// the normed heads: ordinary gates 8.4e-8 (token by token 8.5e-8), gates close to one 1.0e-7 (8.2e-7), small ones 6.6e-8 (7.0e-8); of
// the state 8.2e-8 (1.4e-7), 2.2e-7 (2.8e-6), 3.3e-8 (2.7e-8: there 1 - f is close to one and rounded, which the walk's f (S - v) + v is not).
template <int DP>
__global__ __launch_bounds__(GNB * DP) void hgrn2_tiles_kernel(Hgrn2Op op, float* __restrict__ raw, float* __restrict__ qd,
                                                               float* __restrict__ kd, float* __restrict__ gd,
                                                               const int* __restrict__ cu_seqlens, const int* __restrict__ seq_tile0,
                                                               int B, int n_heads) {
  constexpr int ROW = DP + 4, NWAVES = GNB * DP / WAVE, CH = DP / 16, CV = CH < 4 ? CH : 4;      // channels a lane of the pairs inside four tokens, and a load
  extern __shared__ __attribute__((aligned(16))) float lds[];
  float* s_q = lds;                               // [64][ROW]
  float* s_k = s_q + GT * ROW;                    // [64][ROW]
  float* s_f = s_k + GT * ROW;                    // [64][ROW]
  float* s_e = s_f + GT * ROW;                    // [64][ROW]
  float* s_tot = s_e + GT * ROW;                  // [4][DP]  the product of a block's gates
  float* s_a = s_tot + GNB * DP;                  // [64][GA_ROW] scores
  auto load_v = [](float* to, const float* from) {
    typedef __attribute__((ext_vector_type(CV))) float vec;
    const vec x = *reinterpret_cast<const vec*>(from);
#pragma unroll
    for (int u = 0; u < CV; ++u) to[u] = x[u];
  };
  const int gt = blockIdx.x, h = blockIdx.y, tid = threadIdx.x;
  const int b = seq_of_tile(seq_tile0, B, gt);
  const int p0 = (gt - seq_tile0[b]) * GT, first = cu_seqlens[b] + p0, n = min(GT, cu_seqlens[b + 1] - first);
  if (n <= 0) return;
  const int ch = tid % DP, sb = tid / DP, lane = tid % WAVE, li = lane % 16, lq = lane / 16;
  const int wave = __builtin_amdgcn_readfirstlane(tid / WAVE);
  const int d = op.d, dv = op.dv;
  const bool ch_ok = ch < d;
  // the values of the wave's first columns, in the order of the last product's operand: asked for first, needed last
  const int n_cols = (dv + 15) / 16;
  float vb[GT / 4];
  auto load_values = [&](int col) {
    const int j = min(col * 16 + li, dv - 1);
#pragma unroll
    for (int i = 0; i < GT / 4; ++i) {
      const int s = 16 * (i / 4) + 4 * lq + i % 4;
      vb[i] = op.value(first + min(s, n - 1), h, j);           // behind the text the score is zero
    }
  };
  float q[GB], k[GB], f[GB];
  {
    float z[GB][2];
#pragma unroll
    for (int u = 0; u < GB; ++u) op.fetch(first + min(sb * GB + u, n - 1), h, min(ch, d - 1), z[u]);
    if (wave < n_cols) load_values(wave);
    const Hgrn2Op::Row mine = op.begin(h, ch, ch_ok);
#pragma unroll
    for (int u = 0; u < GB; ++u) {
      float qq, ff, kk;
      op.form(mine, z[u], nullptr, qq, ff, kk);
      const bool ok = ch_ok && sb * GB + u < n;    // what lies behind the text or the head adds nothing and forgets nothing
      q[u] = ok ? qq : 0.f;
      f[u] = ok ? ff : 1.f;
      k[u] = ok ? kk : 0.f;
    }
  }
  float total = 1.f;
#pragma unroll
  for (int u = 0; u < GB; ++u) {
    const int at = (sb * GB + u) * ROW + ch;
    s_q[at] = q[u], s_k[at] = k[u], s_f[at] = f[u];
    total *= f[u];
  }
  s_tot[sb * DP + ch] = total;
  lds_barrier();
  float before = 1.f, after = 1.f, whole = 1.f;    // the gates of the blocks before and behind this thread's, of all
#pragma unroll
  for (int i = 0; i < GNB; ++i) {
    const float t = s_tot[i * DP + ch];
    if (i < sb) before *= t;
    if (i > sb) after *= t;
    whole *= t;
  }
  {
    const size_t at = (size_t)gt * n_heads + h;
    float* qo = qd + (at * GT + sb * GB) * DP + ch;
    float* ko = kd + (at * DP + ch) * GT + sb * GB;
    float c = before;
#pragma unroll
    for (int u = 0; u < GB; ++u) {
      c *= f[u];
      qo[(size_t)u * DP] = q[u] * c;
    }
    float e = after;
#pragma unroll
    for (int u = GB - 4; u >= 0; u -= 4) {
      float4 o;
      o.w = k[u + 3] * e, e *= f[u + 3];
      o.z = k[u + 2] * e, e *= f[u + 2];
      o.y = k[u + 1] * e, e *= f[u + 1];
      o.x = k[u] * e, e *= f[u];
      *reinterpret_cast<float4*>(ko + u) = o;
    }
    if (sb == 0) gd[at * DP + ch] = whole;
  }
  // Scores inside four tokens: a lane a token s and CH channels, whose product it carries on to the tokens s, s + 1, ...; the sixteen
  // lanes of a token are four apart.
  for (int quad = wave; quad < GT / HT_QUAD; quad += NWAVES) {
    const int s = lane % HT_QUAD, e0 = lane / HT_QUAD * CH, row0 = quad * HT_QUAD;
    float p[CH], sum[HT_QUAD];
#pragma unroll
    for (int i = 0; i < CH; i += CV) load_v(p + i, s_k + (row0 + s) * ROW + e0 + i);
#pragma unroll
    for (int step = 0; step < HT_QUAD; ++step) {
      const int at = (row0 + min(s + step, HT_QUAD - 1)) * ROW + e0;
      float acc[2] = {0.f, 0.f}, a[CH], g[CH];
#pragma unroll
      for (int i = 0; i < CH; i += CV) {
        load_v(a + i, s_q + at + i);
        if (step > 0) load_v(g + i, s_f + at + i);
      }
#pragma unroll
      for (int i = 0; i < CH; ++i) {
        if (step > 0) p[i] *= g[i];
        acc[i & 1] = fmaf(a[i], p[i], acc[i & 1]);
      }
      sum[step] = acc[0] + acc[1];
    }
#pragma unroll
    for (int step = 0; step < HT_QUAD; ++step) {
#pragma unroll
      for (int o = HT_QUAD; o < WAVE; o *= 2) sum[step] += __shfl_xor(sum[step], o, WAVE);
    }
    // the lanes of a token share its four results: one a lane, and the zeros of the tokens that do not see it
    const int mine = lane / HT_QUAD;
    const float r = mine == 0 ? sum[0] : mine == 1 ? sum[1] : mine == 2 ? sum[2] : sum[3];
    const int t = s + mine;
    if (mine < HT_QUAD) s_a[(row0 + t % HT_QUAD) * GA_ROW + row0 + s] = t < HT_QUAD ? r : 0.f;
  }
  lds_barrier();
  {
    float c = 1.f, c8 = 1.f, c4 = 1.f, e = 1.f, e8 = 1.f, e4 = 1.f;
#pragma unroll
    for (int u = 0; u < GB; ++u) {
      const int at = (sb * GB + u) * ROW + ch;
      c *= f[u];
      s_q[at] = q[u] * c;
      if (u & HT_HALF) {
        c8 *= f[u];
        s_f[at] = q[u] * c8;
      }
      if (u & HT_QUAD) {
        c4 = (u & (HT_QUAD - 1)) == 0 ? f[u] : c4 * f[u];
        s_e[at] = q[u] * c4;
      }
    }
#pragma unroll
    for (int u = GB - 1; u >= 0; --u) {
      const int at = (sb * GB + u) * ROW + ch;
      s_k[at] = k[u] * e;
      e *= f[u];
      if (!(u & HT_HALF)) {
        s_f[at] = k[u] * e8;
        e8 *= f[u];
      }
      if (!(u & HT_QUAD)) {
        if ((u & (HT_QUAD - 1)) == HT_QUAD - 1) e4 = 1.f;
        s_e[at] = k[u] * e4;
        e4 *= f[u];
      }
    }
  }
  lds_barrier();
  // scores between the blocks i > j (jobs 0 .. 5), between the halves of block i (6 .. 9) and between the quarters of its halves (the others);
  // the rows of the last two are both operands: the later part's the queries, the earlier part's the keys
  constexpr int PAIRS = GNB * (GNB - 1) / 2;
  for (int job = wave; job < PAIRS + 2 * GNB; job += NWAVES) {
    const int part = job < PAIRS ? 0 : job < PAIRS + GNB ? HT_HALF : HT_QUAD;      // tokens of a part
    const int i = part ? (job - PAIRS) % GNB : job < 1 ? 1 : job < 3 ? 2 : 3, j = part ? i : job - i * (i - 1) / 2;
    const float* pa = (part == 0 ? s_q : part == HT_HALF ? s_f : s_e) + (i * GB + li) * ROW + 4 * lq;
    const float* px = part == 0 ? s_k + (j * GB + li) * ROW + 4 * lq : pa;
    gf32x4 acc[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) acc[r] = (gf32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll 2
    for (int m = 0; m < DP / 16; ++m) {
      float4 a = *reinterpret_cast<const float4*>(pa + 16 * m);
      const float4 x = *reinterpret_cast<const float4*>(px + 16 * m);
      for (int g = j + 1; g < i; ++g) {            // the blocks between
        const float4 t = *reinterpret_cast<const float4*>(s_tot + g * DP + 16 * m + 4 * lq);
        a.x *= t.x, a.y *= t.y, a.z *= t.z, a.w *= t.w;
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) acc[r] = mfma4(el(a, r), el(x, r), acc[r]);
    }
    const gf32x4 sum = (acc[0] + acc[1]) + (acc[2] + acc[3]);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int t = 4 * lq + r, s = li;
      float* to = s_a + (i * GB + t) * GA_ROW + j * GB + s;
      if (part == 0) {
        *to = sum[r];
      } else if (t / (2 * part) == s / (2 * part)) {
        if ((t & part) && !(s & part)) *to = sum[r];
        else if (!(t & part) && (s & part)) *to = 0.f;           // the earlier part does not see the later one
      }
    }
  }
  lds_barrier();
  for (int col = wave; col < n_cols; col += NWAVES) {
    if (col != wave) load_values(col);
    const int j = col * 16 + li;
    // Where a value is not finite, the zeros of the tokens that do not see it would make their results NaN: the tokens of one block then
    // meet one by one.
    bool all_finite = true;
#pragma unroll
    for (int i = 0; i < GT / 4; ++i) all_finite = all_finite && fabsf(vb[i]) <= FLT_MAX;
    const bool one_by_one = __any(!all_finite);
#pragma unroll
    for (int i = 0; i < GNB; ++i) {
      gf32x4 acc[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) acc[r] = (gf32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int m = 0; m <= i; ++m) {
        if (m == i && one_by_one) break;
        const float4 a = *reinterpret_cast<const float4*>(s_a + (i * GB + li) * GA_ROW + 16 * m + 4 * lq);
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[r] = mfma4(el(a, r), vb[4 * m + r], acc[r]);
      }
      gf32x4 sum;                                  // (in 64 bits: two roundings less, a twentieth of the heads' error)
#pragma unroll
      for (int r = 0; r < 4; ++r) sum[r] = (float)(((double)acc[0][r] + (double)acc[1][r]) + ((double)acc[2][r] + (double)acc[3][r]));
      if (one_by_one) {
#pragma unroll
        for (int s = 0; s < GB; ++s) {
          const float v = __shfl(vb[4 * i + s % 4], s / 4 * 16 + li, WAVE);
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int t = 4 * lq + r;
            if (t >= s) sum[r] = fmaf(s_a[(i * GB + t) * GA_ROW + i * GB + s], v, sum[r]);
          }
        }
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int t = i * GB + 4 * lq + r;
        if (t < n && j < dv) raw[(size_t)(first + t) * op.Hv + h * dv + j] = sum[r];
      }
    }
  }
}

int hgrn2_padded_dim(int d) { return d <= 0 ? 0 : d <= 32 ? 32 : d <= 64 ? 64 : d <= 128 ? 128 : 0; }

template <int DP>
int hgrn2_tiles_launch(const Hgrn2Op& op, float* state, float* raw, float* qd, float* kd, float* gd, const int* cu_seqlens,
                       const int* seq_slot, const int* seq_tile0, int n_tiles, int B, int n_heads, hipStream_t stream) {
  static LdsAllowance allowance;
  const size_t lds = hgrn2_tiles_lds(DP);
  int rc = allow_dynamic_lds(allowance, reinterpret_cast<const void*>(hgrn2_tiles_kernel<DP>), (int)lds);
  if (rc != YALM_OK) return rc;
  hgrn2_tiles_kernel<DP><<<dim3(n_tiles, n_heads), GNB * DP, lds, stream>>>(op, raw, qd, kd, gd, cu_seqlens, seq_tile0, B, n_heads);
  rc = launch_status();
  if (rc != YALM_OK) return rc;
  return scan_carry_launch<DP>(op, state, raw, qd, kd, gd, cu_seqlens, seq_slot, seq_tile0, B, n_heads, stream);
}
}  // namespace

extern "C" int yalm_hgrn2_tiles_fit(int d) { return hgrn2_padded_dim(d); }

extern "C" int yalm_hgrn2_tiles(const float* proj, long proj_row, const float* f_bias, const float* lower, const float* w_norm,
                                float* state, float* raw, float* qd, float* kd, float* gd, const int* cu_seqlens, const int* seq_slot,
                                const int* seq_tile0, int n_tiles, void* out, int T, int B, int n_heads, int d, int dv, float eps,
                                int out_dtype, hipStream_t stream) {
  if (T <= 0 || B <= 0 || n_tiles <= 0) return YALM_OK;
  const int dp = hgrn2_padded_dim(d);
  if (n_heads <= 0 || n_heads > 65535 || B > 65535 || dp == 0 || dv <= 0 || ceil_div(dv, 16) > 65535 ||
      ((((uintptr_t)qd) | ((uintptr_t)kd) | ((uintptr_t)gd)) & 15))
    return YALM_ERR_ARG;
  if (out_dtype != YALM_F32 && out_dtype != YALM_BF16) return YALM_ERR_DTYPE;
  if (proj_row < 2 * n_heads * d + n_heads * dv || proj_row > INT_MAX) return YALM_ERR_ARG;
  const Hgrn2Op op = {proj, f_bias, lower, n_heads * d, (int)proj_row, d, dv, n_heads * dv};
  const int rc = dp == 32   ? hgrn2_tiles_launch<32>(op, state, raw, qd, kd, gd, cu_seqlens, seq_slot, seq_tile0, n_tiles, B, n_heads, stream)
                 : dp == 64 ? hgrn2_tiles_launch<64>(op, state, raw, qd, kd, gd, cu_seqlens, seq_slot, seq_tile0, n_tiles, B, n_heads, stream)
                            : hgrn2_tiles_launch<128>(op, state, raw, qd, kd, gd, cu_seqlens, seq_slot, seq_tile0, n_tiles, B, n_heads, stream);
  if (rc != YALM_OK) return rc;
  return heads_norm_launch(raw, w_norm, nullptr, 0, out, T, n_heads, dv, eps, out_dtype, stream);
}

static int hgrn2_gated(const float* proj, long proj_row, const float* f_bias, const float* lower, const float* w_norm, float* state,
                       float* raw, const int* cu_seqlens, const int* seq_slot, void* out, int T, int B, int n_heads, int d, int dv, float eps,
                       void* gate_o, const float* gate, long gate_stride, int gate_heads, int gate_dv, int gate_pad, int out_dtype,
                       hipStream_t stream) {
  if (T <= 0 || B <= 0) return YALM_OK;
  if (n_heads <= 0 || d <= 0 || d > 256 || dv <= 0) return YALM_ERR_ARG;
  if (out_dtype != YALM_F32 && out_dtype != YALM_BF16) return YALM_ERR_DTYPE;
  if (proj_row < 2 * n_heads * d + n_heads * dv || proj_row > INT_MAX) return YALM_ERR_ARG;
  const Hgrn2Op op = {proj, f_bias, lower, n_heads * d, (int)proj_row, d, dv, n_heads * dv};
  // one token a sequence, as the numbers say (the kernel walks whatever cu_seqlens holds; eight tokens of one sequence and none of seven
  // others, which no step of the engine is, take it 12 us and diag_scan_kernel 6)
  const bool step = T == B && n_heads <= 65535 && B <= 65535 && d <= HS_MAX && dv <= HS_MAX && d % 4 == 0 && dv % 4 == 0 && ((uintptr_t)state & 15) == 0;
  // the gate goes along where a thread's part of it lies on 16 bytes; else it is a launch of its own
  const int vec = out_dtype == YALM_BF16 ? 8 : 4, threads = dv <= 32 ? 128 : dv <= 64 ? 256 : 512;
  int blocks = 0;
  if (gate_o != nullptr) {
    if (gate_heads <= 0 || gate_dv <= 0 || gate_pad < gate_dv || gate_stride < (long)gate_heads * gate_dv) return YALM_ERR_ARG;
    if (step && gate_dv % vec == 0 && gate_pad % vec == 0 && gate_stride % 4 == 0 && (((uintptr_t)gate_o | (uintptr_t)gate) & 15) == 0) {
      blocks = ceil_div((long)gate_heads * gate_dv, (long)threads * vec);
    } else {
      const int rc = yalm_sigmoid_gate(gate_o, gate, gate_stride, T, gate_heads, gate_dv, gate_pad, out_dtype, stream);
      if (rc != YALM_OK) return rc;
    }
  }
  if (step) {
    const dim3 grid(n_heads + blocks, B);
#define STEP(T_, THREADS_)                                                                                                                   \
  hgrn2_step_kernel<T_, THREADS_><<<grid, THREADS_, 0, stream>>>(op, state, w_norm, (T_*)out, cu_seqlens, seq_slot, n_heads, d, dv, eps, \
                                                                 SideGate<T_>{(T_*)gate_o, gate, gate_stride, gate_heads, gate_dv, gate_pad, blocks})
#define STEP_OF(T_) \
  if (threads == 128) STEP(T_, 128); else if (threads == 256) STEP(T_, 256); else STEP(T_, 512)
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

extern "C" int yalm_hgrn2(const float* proj, long proj_row, const float* f_bias, const float* lower, const float* w_norm, float* state,
                          float* raw, const int* cu_seqlens, const int* seq_slot, void* out, int T, int B, int n_heads,
                          int d, int dv, float eps, int out_dtype, hipStream_t stream) {
  return hgrn2_gated(proj, proj_row, f_bias, lower, w_norm, state, raw, cu_seqlens, seq_slot, out, T, B, n_heads, d, dv, eps, nullptr, nullptr, 0,
                     0, 0, 0, out_dtype, stream);
}

extern "C" int yalm_hgrn2_gated(const float* proj, long proj_row, const float* f_bias, const float* lower, const float* w_norm, float* state,
                                float* raw, const int* cu_seqlens, const int* seq_slot, void* out, int T, int B, int n_heads, int d, int dv,
                                float eps, void* gate_o, const float* gate, long gate_stride, int gate_heads, int gate_dv, int gate_pad,
                                int out_dtype, hipStream_t stream) {
  if (gate_o == nullptr || gate == nullptr) return YALM_ERR_ARG;
  return hgrn2_gated(proj, proj_row, f_bias, lower, w_norm, state, raw, cu_seqlens, seq_slot, out, T, B, n_heads, d, dv, eps, gate_o, gate,
                     gate_stride, gate_heads, gate_dv, gate_pad, out_dtype, stream);
}
