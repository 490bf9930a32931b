// What stands between the q/k/v product and an attention without rotation: biases, RMS norms over the WHOLE query
// and key projections (all heads at once), a query factor that grows with the position, the blend of the values
// with those an earlier layer made for the same token, and the way into the cache.  A workgroup a token; the row
// waits in LDS between its sums and its results.
//
// The rows of qkv are qkv_row apart (a product may hold more behind them).
//   q = (qkv[:Q] + b_q);  q <- q / rms(q) * w_q            (w_q null: no norm)
//   q <- q * (1 + coef ln(floor((p + 1) / every) + 1)) * q_scale      (every 0: no factor)
//   k likewise with w_k (no factor);  v = qkv[Q + K:] + b_v
//   blend 1: v_first <- v;   blend 2: v <- (1 - lam) v + lam v_first      (lam a number on the device)
// head_norm: the norms run a head at a time instead (over the head's d elements, w_q and w_k of d elements shared by
// the heads).  v_from_k: the product has no value part; a head's values are its keys as projected, before their norm
// (dv = d).  rot_dims > 0: behind the norms, of each query and key head's first rot_dims elements the neighbours (2p,
// 2p + 1) are turned by the angle of pair p at the token's position (cos_sin [positions][rot_dims / 2]).
// Heads are written `pad` elements wide (key size d and value size dv may differ; zeros behind): q_out [T, heads,
// pad], keys into their page and the step's staging tile [row][pad], values transposed [pad][row].
#include "common.h"
#include "yalm_hip.h"

namespace {
// a row of a few hundred numbers takes 256 threads, a real model's thousands 1,024 (a decode step has few tokens, and a
// thread's loads wait for each other's results in turn: the fewer rounds the better).  Few tokens are dealt to several workgroups each
// (blockIdx.y), which all read the row and form its sums and write a share of the results (8 tokens of 6,144 numbers 10.1 -> 8.2 us).  What a thread's
// first results need beside the row is asked for in front of the sums, which share their barriers (5 tokens 7.7 -> 7.4).
template <typename T, int PACK_THREADS>
__global__ __launch_bounds__(PACK_THREADS) void qkv_pack_kernel(
    const float* __restrict__ qkv, long qkv_row, const float* __restrict__ bias, const float* __restrict__ w_q,
    const float* __restrict__ w_k, float eps, float temp_coef, int temp_every, float q_scale, float* __restrict__ v_first,
    int blend, const float* __restrict__ lam_p, T* __restrict__ q_out, T* __restrict__ k_stage, T* __restrict__ v_stage,
    const int* __restrict__ seq_tile0, T* __restrict__ k_pages, T* __restrict__ v_pages,
    const int* __restrict__ block_table, int table_stride, int ring_pages, const int* __restrict__ tok_seq,
    const int* __restrict__ tok_pos, const int* __restrict__ seq_slot, const int* __restrict__ seq_len, int n_heads,
    int n_kv_heads, int d, int dv, int pad, int n_pages, int page_layout, T* __restrict__ v_rows, int head_norm,
    int v_from_k, const float2* __restrict__ cos_sin, int rot_dims, int n_positions) {
  extern __shared__ float row[];                  // [Q + K + V], then a factor for every query and key head
  __shared__ float2 red[PACK_THREADS / WAVE];
  const int t = blockIdx.x, tid = threadIdx.x, part = blockIdx.y, parts = gridDim.y;
  const int Q = n_heads * d, K = n_kv_heads * d, V = n_kv_heads * dv, N = Q + K + (v_from_k ? 0 : V);
  float* head_f = row + N;                        // head_norm: 1 / rms of each query head, then of each key head
  const float* src = qkv + (size_t)t * qkv_row;
  // the row is asked for first: the chain of loads below, to where the token's key and value go, passes while it comes
  constexpr int AHEAD = 8;
  float v[AHEAD];
#pragma unroll
  for (int k = 0; k < AHEAD; ++k) {
    const int i = min(tid + k * PACK_THREADS, N - 1);
    v[k] = src[i] + (bias != nullptr ? bias[i] : 0.f);
  }
  const int pos = tok_pos[t];
  const int b = tok_seq[t];
  const int slot = b >= 0 ? seq_slot[b] : -1;
  const int r = pos & (PAGE - 1);
  long page = -1, tile = -1;                       // its page in the cache (a ring keeps the last pages only) and the step's tile
  if (slot >= 0 && pos >= 0 && k_pages != nullptr) {
    const int ap = pos / PAGE, last_ap = (seq_len[b] - 1) / PAGE;
    if (ap > last_ap - ring_pages) {
      const int phys = block_table[(size_t)slot * table_stride + (ap % ring_pages)];
      if (phys >= 0 && phys < n_pages) page = phys;
    }
  }
  if (k_stage != nullptr && b >= 0 && pos >= 0) tile = (long)seq_tile0[b] + pos / PAGE;
  float sq = 0.f, sk = 0.f;
  auto take = [&](int i, float x) {
    row[i] = x;
    if (i < Q) sq = fmaf(x, x, sq);
    else if (i < Q + K) sk = fmaf(x, x, sk);
  };
#pragma unroll
  for (int k = 0; k < AHEAD; ++k)
    if (tid + k * PACK_THREADS < N) take(tid + k * PACK_THREADS, v[k]);
  for (int i = tid + AHEAD * PACK_THREADS; i < N; i += PACK_THREADS) take(i, src[i] + (bias != nullptr ? bias[i] : 0.f));
  // the norm weights and the rotation of this thread's first query and key come while the sums are formed
  const float2* cs = rot_dims > 0 ? cos_sin + (size_t)min(max(pos, 0), n_positions - 1) * (rot_dims / 2) : nullptr;
  struct Ahead {
    float w, w_other;                             // of the element, and of the other one of its pair
    float2 c;
  };
  auto ask = [&](const float* w, int head, int e) {
    Ahead a = {1.0f, 1.0f, make_float2(1.0f, 0.0f)};
    if (e < d) {
      const bool turned = e < rot_dims;
      if (w != nullptr) a.w = w[head_norm ? e : head * d + e];
      if (w != nullptr && turned) a.w_other = w[head_norm ? e ^ 1 : head * d + (e ^ 1)];
      if (turned) a.c = cs[e >> 1];
    }
    return a;
  };
  const int first = part * PACK_THREADS + tid, step = parts * PACK_THREADS;
  Ahead aq = ask(w_q, first / pad, first < n_heads * pad ? first % pad : d), ak = ask(w_k, first / pad, first < n_kv_heads * pad ? first % pad : d);
  const float2 both = block_sum2<PACK_THREADS / WAVE>(sq, sk, red);
  sq = both.x;
  sk = both.y;
  if (head_norm) {                                // a wave a head: the sum of its squares
    for (int hh = tid / WAVE; hh < n_heads + n_kv_heads; hh += PACK_THREADS / WAVE) {
      float s = 0.f;
      for (int e = tid % WAVE; e < d; e += WAVE) s = fmaf(row[hh * d + e], row[hh * d + e], s);
      s = wave_sum(s);
      if (tid % WAVE == 0) head_f[hh] = 1.0f / sqrtf(s / (float)d + eps);
    }
    __syncthreads();
  }

  // the queries
  float fq = q_scale;
  if (w_q != nullptr && !head_norm) fq *= 1.0f / sqrtf(sq / (float)Q + eps);
  if (temp_every > 0) fq *= 1.0f + temp_coef * logf((float)((pos + 1) / temp_every) + 1.0f);
  for (int i = first; i < n_heads * pad; i += step) {
    const int h = i / pad, e = i - h * pad;
    if (i != first) aq = ask(w_q, h, e);
    float v = 0.f;
    if (e < d) {
      const float f = head_norm && w_q != nullptr ? fq * head_f[h] : fq;
      v = row[h * d + e] * f * aq.w;
      if (e < rot_dims) {
        const float2 c = aq.c;
        const float other = row[h * d + (e ^ 1)] * f * aq.w_other;
        v = (e & 1) ? fmaf(v, c.x, other * c.y) : fmaf(v, c.x, -other * c.y);
      }
    }
    q_out[(size_t)t * n_heads * pad + i] = from_f32<T>(v);
  }

  const float fk = w_k != nullptr && !head_norm ? 1.0f / sqrtf(sk / (float)K + eps) : 1.0f;
  const float lam = blend == 2 ? lam_p[0] : 0.f;
  for (int i = first; i < n_kv_heads * pad; i += step) {
    const int g = i / pad, e = i - g * pad;
    if (i != first) ak = ask(w_k, g, e);
    float kv = 0.f, vv = 0.f;
    if (e < d) {
      const float f = head_norm && w_k != nullptr ? head_f[n_heads + g] : fk;
      kv = row[Q + g * d + e] * f * ak.w;
      if (e < rot_dims) {
        const float2 c = ak.c;
        const float other = row[Q + g * d + (e ^ 1)] * f * ak.w_other;
        kv = (e & 1) ? fmaf(kv, c.x, other * c.y) : fmaf(kv, c.x, -other * c.y);
      }
    }
    if (e < dv) {
      vv = v_from_k ? row[Q + g * d + e] : row[Q + K + g * dv + e];
      float* first = v_first != nullptr ? v_first + (size_t)t * V + g * dv + e : nullptr;
      if (blend == 1) *first = vv;
      else if (blend == 2) vv = (1.0f - lam) * vv + lam * *first;
    }
    const T kt = from_f32<T>(kv), vt = from_f32<T>(vv);
    // v_rows: the values go there row by row, and a kernel that works a tile of 64 tokens at a time brings them into the
    // transposed places (whole lines instead of two bytes at a time)
    if (v_rows != nullptr) v_rows[(size_t)t * n_kv_heads * pad + i] = vt;
    if (tile >= 0) {
      const size_t base = ((size_t)tile * n_kv_heads + g) * PAGE * pad;
      k_stage[base + (size_t)r * pad + e] = kt;
      if (v_rows == nullptr) v_stage[base + (size_t)e * PAGE + r] = vt;
    }
    if (page >= 0) {
      const size_t base = ((size_t)page * n_kv_heads + g) * PAGE * pad;
      k_pages[base + page_k_offset(page_layout, r, e, pad)] = kt;
      if (v_rows == nullptr) v_pages[base + page_v_offset(page_layout, r, e, pad)] = vt;
    }
  }
}

// The same work four elements a thread, the token's row in registers between its sums and its results: one exchange for both sums and
// no row in LDS.  The sums are formed as one wave alone forms them, 256 elements after 256 in every lane, whatever the number of waves: the
// bits of a row's norm do not hang on it (what the waves hand each other is a sum of four squares an element's thread; the exchange is
// level with one of the waves' sums: 1,909 rows of 6,144 20.9 and 21.1 us).  For rows whose parts and heads are multiples of four elements (a thread takes four consecutive ones at a time) and at most
// 1,024 * NV elements.  A workgroup of four waves a token: with a wave a token, 24 rounds of a row of 6,144 and its weights were 250
// registers, two waves a SIMD and too few loads in flight (1,909 tokens inside a step 43.8 -> 31.1 us; 32
// tokens alone 19.8 -> 7.2, 1,909 29.5 -> 21; rows of 1,536 7.3 -> 4.9 and 10.5 -> 9.1).  Rows of up to 256 are a wave's (2,048 of them 4.2 us, with four waves 5.5), and so are those of up to
// 2,048 where tokens are many: each of the four has next to nothing to load and the chip holds 2,048 workgroups of four.  us with four waves, two
// and one, rows of 384: 1,000 tokens 4.5 4.1 4.3, 1,909 6.0 5.0 4.6, 4,000 9.7 7.5 6.2; of 1,024 4.8 4.6 5.0, 6.8 6.2 6.6, 11.5 9.5 9.0; of 1,344
// 5.7 5.7 7.1, 9.6 7.9 8.9, 14.4 12.8 11.7; of 2,048 7.3 7.7 9.8, 11.4 10.1 11.0, 18.4 16.9 15.9; of 2,304 and more four are the soonest or level.
template <typename T> struct Pack4;
template <> struct Pack4<float> {
  static __device__ __forceinline__ void store(float* p, float a, float b, float c, float d) {
    *reinterpret_cast<float4*>(p) = make_float4(a, b, c, d);
  }
};
template <> struct Pack4<bf16> {
  typedef __attribute__((ext_vector_type(4))) __bf16 bf16x4;
  static __device__ __forceinline__ void store(bf16* p, float a, float b, float c, float d) {
    *reinterpret_cast<bf16x4*>(p) = (bf16x4){static_cast<bf16>(a), static_cast<bf16>(b), static_cast<bf16>(c), static_cast<bf16>(d)};
  }
};

// SHAPED: with norms a head, values that are the keys, or the rotation (the other models run the code without them)
template <typename T, int NV, bool SHAPED, int PV_THREADS>
__global__ __launch_bounds__(PV_THREADS) void qkv_pack_vec_kernel(
    const float* __restrict__ qkv, long qkv_row, const float* __restrict__ bias, const float* __restrict__ w_q,
    const float* __restrict__ w_k, float eps, float temp_coef, int temp_every, float q_scale, float* __restrict__ v_first,
    int blend, const float* __restrict__ lam_p, T* __restrict__ q_out, T* __restrict__ k_stage, T* __restrict__ v_stage,
    const int* __restrict__ seq_tile0, T* __restrict__ k_pages, T* __restrict__ v_pages,
    const int* __restrict__ block_table, int table_stride, int ring_pages, const int* __restrict__ tok_seq,
    const int* __restrict__ tok_pos, const int* __restrict__ seq_slot, const int* __restrict__ seq_len,
    int n_heads, int n_kv_heads, int d, int dv, int pad, int n_pages, int page_layout, T* __restrict__ v_rows,
    int head_norm_, int v_from_k_, const float2* __restrict__ cos_sin, int rot_dims_, int n_positions) {
  // head_norm here: d a power of two from 4 to 256, so that a head's elements lie in d / 4 neighbouring lanes of one round
  const int head_norm = SHAPED ? head_norm_ : 0, v_from_k = SHAPED ? v_from_k_ : 0, rot_dims = SHAPED ? rot_dims_ : 0;
  constexpr int WAVES = PV_THREADS / WAVE, ROUNDS = NV * WAVES;      // a round: 256 elements in their order
  constexpr int AT_ONCE = ROUNDS < 8 ? ROUNDS : 8;
  __shared__ float round_ss[WAVES > 1 ? ROUNDS : 1][WAVE], sums[2];
  const int t = blockIdx.x, tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid / WAVE), lane = tid % WAVE;
  const int pos = tok_pos[t];
  const int b = tok_seq[t];
  const int Q = n_heads * d, K = n_kv_heads * d, V = n_kv_heads * dv, N = Q + K + (v_from_k ? 0 : V);
  const float* src = qkv + (size_t)t * qkv_row;
  // Heads that divide a round's elements: a thread has the same place in the head in every round, and its two angles are asked for
  // once, in front of the row
  const float2* cs = rot_dims > 0 ? cos_sin + (size_t)min(max(pos, 0), n_positions - 1) * (rot_dims / 2) : nullptr;
  const bool same_place = (PV_THREADS * 4) % d == 0;
  float2 turn0 = make_float2(1.0f, 0.0f), turn1 = turn0;
  if (SHAPED && same_place && cs != nullptr) {
    const int e = tid * 4 % d;
    if (e < rot_dims) turn0 = cs[e >> 1];
    if (e + 2 < rot_dims) turn1 = cs[(e >> 1) + 1];
  }
  float4 r[NV], wt[NV];                           // the row and the norm weights of its elements: every load asked for at once
  const bool row_norm = !head_norm && (w_q != nullptr || w_k != nullptr);
  float sq = 0.f, sk = 0.f;
#pragma unroll
  for (int j = 0; j < NV; ++j) {
    const int i = (j * PV_THREADS + tid) * 4;
    wt[j] = make_float4(1.f, 1.f, 1.f, 1.f);
    if (i < Q && w_q != nullptr) wt[j] = *reinterpret_cast<const float4*>(w_q + (head_norm ? i % d : i));
    else if (i >= Q && i < Q + K && w_k != nullptr) wt[j] = *reinterpret_cast<const float4*>(w_k + (head_norm ? (i - Q) % d : i - Q));
  }

#pragma unroll
  for (int j = 0; j < NV; ++j) {
    const int i = (j * PV_THREADS + tid) * 4;
    float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
    if (i < N) {
      v = *reinterpret_cast<const float4*>(src + i);
      if (bias != nullptr) {
        const float4 b4 = *reinterpret_cast<const float4*>(bias + i);
        v.x += b4.x; v.y += b4.y; v.z += b4.z; v.w += b4.w;
      }
      const float ss = v.x * v.x + v.y * v.y + v.z * v.z + v.w * v.w;
      if constexpr (WAVES > 1) {
        if (row_norm) round_ss[j * WAVES + wave][lane] = ss;
      } else {
        if (i < Q) sq += ss;
        else if (i < Q + K) sk += ss;
      }
    }
    r[j] = v;
    if constexpr (SHAPED) {
      if (head_norm) {                            // the sum over the head's lanes (neighbours: exchanges inside their group);
        float ss = i < Q + K ? v.x * v.x + v.y * v.y + v.z * v.z + v.w * v.w : 0.f;      // 1 / rms rides on the norm's weights
        for (int o = 1; o < d / 4; o <<= 1) ss += __shfl_xor(ss, o, WAVE);
        const float f = 1.0f / sqrtf(ss / (float)d + eps);
        wt[j].x *= f, wt[j].y *= f, wt[j].z *= f, wt[j].w *= f;
      }
    }
  }
  if (row_norm) {                                 // the rounds are added in their order, lane by lane, as one wave alone does it
    if constexpr (WAVES > 1) {
      lds_barrier();
      if (wave < 2) {                             // the first wave the queries', the second the keys'
        const int lo = wave == 0 ? 0 : Q, hi = wave == 0 ? Q : Q + K;
        float s = 0.f;
        for (int j0 = lo / (WAVE * 4); j0 * WAVE * 4 < hi; j0 += AT_ONCE) {
          float part[AT_ONCE];
#pragma unroll
          for (int u = 0; u < AT_ONCE; ++u) part[u] = round_ss[min(j0 + u, ROUNDS - 1)][lane];
#pragma unroll
          for (int u = 0; u < AT_ONCE; ++u) {
            const int i = ((j0 + u) * WAVE + lane) * 4;
            s += i >= lo && i < hi ? part[u] : 0.f;
          }
        }
        s = wave_sum(s);
        if (lane == 0) sums[wave] = s;
      }
      lds_barrier();
      sq = sums[0];
      sk = sums[1];
    } else {
      sq = wave_sum(sq);
      sk = wave_sum(sk);
    }
  }
  const int slot = b >= 0 ? seq_slot[b] : -1;
  float fq = q_scale;
  if (w_q != nullptr && !head_norm) fq *= 1.0f / sqrtf(sq / (float)Q + eps);
  if (temp_every > 0) fq *= 1.0f + temp_coef * logf((float)((pos + 1) / temp_every) + 1.0f);
  const float fk = w_k != nullptr && !head_norm ? 1.0f / sqrtf(sk / (float)K + eps) : 1.0f;
  const float lam = blend == 2 ? lam_p[0] : 0.f;
  const int row = pos & (PAGE - 1);
  // the lane's four elements e .. e + 3 of a head are two of the rotation's pairs.  Which product is rounded before the other joins it
  // is said here and not left to the compiler: the sine's, and of bfloat16 queries the cosine's
  auto turn_pair = [](bool q, const float2& c, float& a0, float& a1) {
    float x, y;
    if (q && sizeof(T) == 2) x = fmaf(-a1, c.y, a0 * c.x), y = fmaf(a0, c.y, a1 * c.x);
    else x = fmaf(a0, c.x, -(a1 * c.y)), y = fmaf(a1, c.x, a0 * c.y);
    a0 = x, a1 = y;
  };
  auto turn = [&](bool q, int e, float& a0, float& a1, float& a2, float& a3) {
    if (same_place) {                             // two ways, so that this one waits for no load (and for no store in front of it)
      if (e < rot_dims) turn_pair(q, turn0, a0, a1);
      if (e + 2 < rot_dims) turn_pair(q, turn1, a2, a3);
    } else {
      if (e < rot_dims) turn_pair(q, cs[e >> 1], a0, a1);
      if (e + 2 < rot_dims) turn_pair(q, cs[(e >> 1) + 1], a2, a3);
    }
  };
  long page = -1, tile = -1;
  if (slot >= 0 && pos >= 0 && k_pages != nullptr) {
    const int ap = pos / PAGE, last_ap = (seq_len[b] - 1) / PAGE;
    if (ap > last_ap - ring_pages) {
      const int phys = block_table[(size_t)slot * table_stride + (ap % ring_pages)];
      if (phys >= 0 && phys < n_pages) page = phys;
    }
  }
  if (k_stage != nullptr && b >= 0 && pos >= 0) tile = (long)seq_tile0[b] + pos / PAGE;
  T* qo = q_out + (size_t)t * n_heads * pad;
#pragma unroll
  for (int j = 0; j < NV; ++j) {
    const int i = (j * PV_THREADS + tid) * 4;
    if (i >= N) continue;
    float4 v = r[j];
    if (i < Q) {
      const int h = i / d, e = i - h * d;
      const float4 w4 = wt[j];
      float a0 = v.x * fq * w4.x, a1 = v.y * fq * w4.y, a2 = v.z * fq * w4.z, a3 = v.w * fq * w4.w;
      if constexpr (SHAPED) turn(true, e, a0, a1, a2, a3);
      Pack4<T>::store(qo + h * pad + e, a0, a1, a2, a3);
    } else if (i < Q + K) {
      const int ik = i - Q, g = ik / d, e = ik - g * d;
      const float4 w4 = wt[j];
      float a0 = v.x * fk * w4.x, a1 = v.y * fk * w4.y, a2 = v.z * fk * w4.z, a3 = v.w * fk * w4.w;
      if constexpr (SHAPED) turn(false, e, a0, a1, a2, a3);
      if (SHAPED && v_from_k) {                             // the key as projected is the value
        if (v_rows != nullptr) {
          Pack4<T>::store(v_rows + (size_t)t * n_kv_heads * pad + g * pad + e, v.x, v.y, v.z, v.w);
        } else {
          const float vals[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            const T vt = from_f32<T>(vals[u]);
            if (tile >= 0) v_stage[((size_t)tile * n_kv_heads + g) * PAGE * pad + (size_t)(e + u) * PAGE + row] = vt;
            if (page >= 0) v_pages[((size_t)page * n_kv_heads + g) * PAGE * pad + page_v_offset(page_layout, row, e + u, pad)] = vt;
          }
        }
      }
      if (tile >= 0) Pack4<T>::store(k_stage + ((size_t)tile * n_kv_heads + g) * PAGE * pad + (size_t)row * pad + e, a0, a1, a2, a3);
      if (page >= 0)                              // four consecutive elements lie together in either layout
        Pack4<T>::store(k_pages + ((size_t)page * n_kv_heads + g) * PAGE * pad + page_k_offset(page_layout, row, e, pad), a0, a1, a2, a3);
    } else {
      const int iv = i - Q - K, g = iv / dv, e = iv - g * dv;
      if (blend == 1) {
        *reinterpret_cast<float4*>(v_first + (size_t)t * V + iv) = v;
      } else if (blend == 2) {
        const float4 f4 = *reinterpret_cast<const float4*>(v_first + (size_t)t * V + iv);
        v.x = (1.0f - lam) * v.x + lam * f4.x; v.y = (1.0f - lam) * v.y + lam * f4.y;
        v.z = (1.0f - lam) * v.z + lam * f4.z; v.w = (1.0f - lam) * v.w + lam * f4.w;
      }
      if (v_rows != nullptr) {
        Pack4<T>::store(v_rows + (size_t)t * n_kv_heads * pad + g * pad + e, v.x, v.y, v.z, v.w);
      } else {
        const float vals[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const T vt = from_f32<T>(vals[u]);
          if (tile >= 0) v_stage[((size_t)tile * n_kv_heads + g) * PAGE * pad + (size_t)(e + u) * PAGE + row] = vt;
          if (page >= 0) v_pages[((size_t)page * n_kv_heads + g) * PAGE * pad + page_v_offset(page_layout, row, e + u, pad)] = vt;
        }
      }
    }
  }
  // the heads' elements behind the key and the value size are zeros
  const T zero = from_f32<T>(0.f);
  if (pad > d) {
    const int extra = pad - d;
    for (int i = tid; i < n_heads * extra; i += PV_THREADS) qo[(i / extra) * pad + d + i % extra] = zero;
    for (int i = tid; i < n_kv_heads * extra; i += PV_THREADS) {
      const int g = i / extra, e = d + i % extra;
      if (tile >= 0) k_stage[((size_t)tile * n_kv_heads + g) * PAGE * pad + (size_t)row * pad + e] = zero;
      if (page >= 0) k_pages[((size_t)page * n_kv_heads + g) * PAGE * pad + page_k_offset(page_layout, row, e, pad)] = zero;
    }
  }
  if (pad > dv) {
    const int extra = pad - dv;
    for (int i = tid; i < n_kv_heads * extra; i += PV_THREADS) {
      const int g = i / extra, e = dv + i % extra;
      if (v_rows != nullptr) {
        v_rows[(size_t)t * n_kv_heads * pad + g * pad + e] = zero;
      } else {
        if (tile >= 0) v_stage[((size_t)tile * n_kv_heads + g) * PAGE * pad + (size_t)e * PAGE + row] = zero;
        if (page >= 0) v_pages[((size_t)page * n_kv_heads + g) * PAGE * pad + page_v_offset(page_layout, row, e, pad)] = zero;
      }
    }
  }
}

// The values of a step of whole prompts from rows [T, G, pad] into the transposed staging tiles and cache pages: a
// workgroup a (tile of 64 tokens, KV head), through LDS, so that every write is a run of consecutive rows.
constexpr int VT_THREADS = 256;
template <typename T>
__global__ __launch_bounds__(VT_THREADS) void v_tiles_kernel(
    const T* __restrict__ v_rows, T* __restrict__ v_stage, T* __restrict__ v_pages, const int* __restrict__ cu_seqlens,
    const int* __restrict__ seq_tile0, const int* __restrict__ block_table, int table_stride, int ring_pages,
    const int* __restrict__ seq_slot, const int* __restrict__ seq_len, int B, int n_kv_heads, int pad, int n_pages,
    int page_layout) {
  constexpr int VEC = 16 / sizeof(T);             // elements of a 16-byte access (pad is a multiple of 16)
  struct __attribute__((aligned(16))) Chunk { T v[VEC]; };
  extern __shared__ __attribute__((aligned(16))) unsigned char vt_raw[];
  T* tl = reinterpret_cast<T*>(vt_raw);           // [PAGE][pad + VEC]
  const int tile = blockIdx.x, g = blockIdx.y, tid = threadIdx.x;
  int lo = 0, hi = B - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (seq_tile0[mid] <= tile) lo = mid; else hi = mid - 1;
  }
  const int b = lo, tq = tile - seq_tile0[b];
  const int start = cu_seqlens[b], len = cu_seqlens[b + 1] - start;
  const int n_rows = min(PAGE, len - tq * PAGE);
  const int row_w = pad + VEC, per_row = pad / VEC;
  for (int i = tid; i < PAGE * per_row; i += VT_THREADS) {
    const int r = i / per_row, c = i - r * per_row;
    Chunk ch;
#pragma unroll
    for (int u = 0; u < VEC; ++u) ch.v[u] = from_f32<T>(0.f);
    if (r < n_rows)
      ch = *reinterpret_cast<const Chunk*>(v_rows + ((size_t)(start + tq * PAGE + r) * n_kv_heads + g) * pad + c * VEC);
    *reinterpret_cast<Chunk*>(tl + r * row_w + c * VEC) = ch;
  }
  __syncthreads();
  T* vp = nullptr;
  const int slot = seq_slot[b];
  if (v_pages != nullptr && slot >= 0 && n_rows > 0) {
    const int last_ap = (seq_len[b] - 1) / PAGE;
    if (tq > last_ap - ring_pages) {
      const int phys = block_table[(size_t)slot * table_stride + (tq % ring_pages)];
      if (phys >= 0 && phys < n_pages) vp = v_pages + ((size_t)phys * n_kv_heads + g) * PAGE * pad;
    }
  }
  T* vs = v_stage + ((size_t)tile * n_kv_heads + g) * PAGE * pad;
  constexpr int RC = PAGE / VEC;                  // runs of VEC consecutive rows in a tile
  for (int i = tid; i < pad * RC; i += VT_THREADS) {
    const int e = i / RC, r0 = (i % RC) * VEC;
    Chunk ch;
#pragma unroll
    for (int u = 0; u < VEC; ++u) ch.v[u] = tl[(r0 + u) * row_w + e];
    *reinterpret_cast<Chunk*>(vs + (size_t)e * PAGE + r0) = ch;      // rows behind the sequence's end are zeros
    // a run of consecutive rows lies together in either page layout; rows behind the end belong to tokens still to
    // come, which write them before anyone reads them
    if (vp != nullptr && r0 < n_rows) *reinterpret_cast<Chunk*>(vp + page_v_offset(page_layout, r0, e, pad)) = ch;
  }
}
}  // namespace

// v_rows `dtype` [T, G, pad] (what yalm_qkv_pack left) into v_stage [n_tiles, G, pad, 64] and the cache pages (null: none).
extern "C" int yalm_v_tiles(const void* v_rows, void* v_stage, void* v_pages, const int* cu_seqlens, const int* seq_tile0,
                            const int* block_table, int table_stride, int ring_pages, const int* seq_slot,
                            const int* seq_len, int B, int n_tiles, int n_kv_heads, int pad, int n_pages, int page_layout,
                            int dtype, hipStream_t stream) {
  if (n_tiles <= 0 || B <= 0) return YALM_OK;
  if (n_kv_heads <= 0 || n_kv_heads > 65535 || pad <= 0 || v_rows == nullptr || v_stage == nullptr ||
      (v_pages != nullptr && (block_table == nullptr || ring_pages <= 0 || seq_len == nullptr)) ||
      !page_layout_ok(page_layout, pad) || (dtype != YALM_F32 && dtype != YALM_BF16))
    return YALM_ERR_ARG;
  if (pad % 16 != 0 || ((((uintptr_t)v_rows) | ((uintptr_t)v_stage) | ((uintptr_t)v_pages)) & 15)) return YALM_ERR_ARG;
  const size_t lds = (size_t)PAGE * (pad + (dtype == YALM_F32 ? 4 : 8)) * (dtype == YALM_F32 ? 4 : 2);
  if (lds > 64 * 1024) return YALM_ERR_ARG;
  dim3 grid(n_tiles, n_kv_heads);
  if (dtype == YALM_F32)
    v_tiles_kernel<float><<<grid, VT_THREADS, lds, stream>>>((const float*)v_rows, (float*)v_stage, (float*)v_pages, cu_seqlens,
                                                             seq_tile0, block_table, table_stride, ring_pages, seq_slot,
                                                             seq_len, B, n_kv_heads, pad, n_pages, page_layout);
  else
    v_tiles_kernel<bf16><<<grid, VT_THREADS, lds, stream>>>((const bf16*)v_rows, (bf16*)v_stage, (bf16*)v_pages, cu_seqlens,
                                                            seq_tile0, block_table, table_stride, ring_pages, seq_slot, seq_len,
                                                            B, n_kv_heads, pad, n_pages, page_layout);
  return launch_status();
}

extern "C" int yalm_qkv_pack(const float* qkv, long qkv_row, const float* bias, const float* w_q, const float* w_k, float eps,
                             float temp_coef, int temp_every, float q_scale, float* v_first, int blend,
                             const float* lam, void* q_out, void* k_stage, void* v_stage, const int* seq_tile0,
                             void* k_pages, void* v_pages, const int* block_table, int table_stride, int ring_pages,
                             const int* tok_seq, const int* tok_pos, const int* seq_slot, const int* seq_len, int T,
                             int n_heads, int n_kv_heads, int d, int dv, int pad, int n_pages, int page_layout,
                             int dtype, void* v_rows, int head_norm, int v_from_k, const float* cos_sin, int rot_dims,
                             int n_positions, hipStream_t stream) {
  if (T <= 0) return YALM_OK;
  if ((v_from_k && (d != dv || blend != 0)) || rot_dims < 0 || rot_dims % 2 || rot_dims > d ||
      (rot_dims > 0 && (cos_sin == nullptr || n_positions <= 0)))
    return YALM_ERR_ARG;
  if (n_heads <= 0 || n_kv_heads <= 0 || d <= 0 || dv <= 0 || pad < d || pad < dv || temp_every < 0 || blend < 0 ||
      blend > 2 || (blend != 0 && v_first == nullptr) || (blend == 2 && lam == nullptr) ||
      (k_stage != nullptr && (v_stage == nullptr || seq_tile0 == nullptr)) ||
      (k_pages != nullptr && (v_pages == nullptr || block_table == nullptr || ring_pages <= 0 || seq_len == nullptr)) ||
      !page_layout_ok(page_layout, pad))
    return YALM_ERR_ARG;
  const int n_row = n_heads * d + n_kv_heads * (d + (v_from_k ? 0 : dv));
  const size_t lds = (size_t)(n_row + n_heads + n_kv_heads) * sizeof(float);
  if (lds > 64 * 1024 || qkv_row < n_row) return YALM_ERR_ARG;
  // four elements a thread where the row's parts allow it and the row fits the registers, and where the tokens
  // are many.  A few tokens alone take much the same either way (5 of 6,144 numbers 6.8 us with the row in LDS and 6.6 in registers, with
  // norms a head 7.3 and 8.2, rows of 8,192 8.3 and 10.9, of 1,536 4.9 and 3.5); inside a step, where the row and the weights come from
  // memory, the shares of several workgroups are sooner (requests of 255 to 509 tokens and 12 steps on four Rekirax layers 12.18 ms and 12.33)
  const bool heads_fit = !head_norm || (d >= 4 && d <= 256 && (d & (d - 1)) == 0);      // a head in neighbouring lanes
  const bool by_fours = heads_fit && T >= 32 && d % 4 == 0 && dv % 4 == 0 && qkv_row % 4 == 0 && n_row <= 256 * 32 &&
                       ((((uintptr_t)qkv) | ((uintptr_t)bias) | ((uintptr_t)w_q) | ((uintptr_t)w_k) | ((uintptr_t)v_first) |
                         ((uintptr_t)q_out) | ((uintptr_t)k_stage) | ((uintptr_t)k_pages) | ((uintptr_t)v_rows)) & 15) == 0;
  if (by_fours) {
    const bool shaped = head_norm || v_from_k || rot_dims > 0;
#define YALM_PACK_W(TYPE, NV_, TH_)                                                                                      \
  do { if (shaped) YALM_PACK_WS(TYPE, NV_, true, TH_); else YALM_PACK_WS(TYPE, NV_, false, TH_); } while (0)
#define YALM_PACK_WS(TYPE, NV_, SHAPED_, TH_)                                                                               \
  qkv_pack_vec_kernel<TYPE, NV_, SHAPED_, TH_><<<T, TH_, 0, stream>>>(                                               \
      qkv, qkv_row, bias, w_q, w_k, eps, temp_coef, temp_every, q_scale, v_first, blend, lam, (TYPE*)q_out, (TYPE*)k_stage,        \
      (TYPE*)v_stage, seq_tile0, (TYPE*)k_pages, (TYPE*)v_pages, block_table, table_stride, ring_pages, tok_seq,         \
      tok_pos, seq_slot, seq_len, n_heads, n_kv_heads, d, dv, pad, n_pages, page_layout, (TYPE*)v_rows, head_norm,       \
      v_from_k, (const float2*)cos_sin, rot_dims, n_positions)
#define YALM_PACK_WN(TYPE)                                                                                               \
  if (n_row <= 256) YALM_PACK_W(TYPE, 1, 64);                                                                            \
  else if (n_row <= 1024 && T > 1024) YALM_PACK_W(TYPE, 4, 64);                                                          \
  else if (n_row <= 1024) YALM_PACK_W(TYPE, 1, 256);                                                                     \
  else if (n_row <= 1024 * 2 && T > 3072) YALM_PACK_W(TYPE, 8, 64);                                                      \
  else if (n_row <= 1024 * 2 && T > 1536) YALM_PACK_W(TYPE, 4, 128);                                                     \
  else if (n_row <= 1024 * 2) YALM_PACK_W(TYPE, 2, 256);                                                                 \
  else if (n_row <= 1024 * 4) YALM_PACK_W(TYPE, 4, 256);                                                                 \
  else if (n_row <= 1024 * 6) YALM_PACK_W(TYPE, 6, 256);                                                                 \
  else YALM_PACK_W(TYPE, 8, 256)
    if (dtype == YALM_F32) {
      YALM_PACK_WN(float);
    } else if (dtype == YALM_BF16) {
      YALM_PACK_WN(bf16);
    } else {
      return YALM_ERR_DTYPE;
    }
#undef YALM_PACK_WN
#undef YALM_PACK_W
#undef YALM_PACK_WS
    return launch_status();
  }
  const bool wide = n_row >= 2048;
#define YALM_PACK(TYPE)                                                                                              \
  if (wide) YALM_PACK_N(TYPE, 1024); else YALM_PACK_N(TYPE, 256)
#define YALM_PACK_N(TYPE, NT)                                                                                        \
  qkv_pack_kernel<TYPE, NT><<<dim3(T, T <= 32 ? min(8, ceil_div((long)max(n_heads, n_kv_heads) * pad, NT)) : 1), NT, lds, stream>>>(                                                                 \
      qkv, qkv_row, bias, w_q, w_k, eps, temp_coef, temp_every, q_scale, v_first, blend, lam, (TYPE*)q_out, (TYPE*)k_stage,    \
      (TYPE*)v_stage, seq_tile0, (TYPE*)k_pages, (TYPE*)v_pages, block_table, table_stride, ring_pages, tok_seq,     \
      tok_pos, seq_slot, seq_len, n_heads, n_kv_heads, d, dv, pad, n_pages, page_layout, (TYPE*)v_rows, head_norm,    \
      v_from_k, (const float2*)cos_sin, rot_dims, n_positions)
  if (dtype == YALM_F32) {
    YALM_PACK(float);
  } else if (dtype == YALM_BF16) {
    YALM_PACK(bf16);
  } else {
    return YALM_ERR_DTYPE;
  }
#undef YALM_PACK
#undef YALM_PACK_N
  return launch_status();
}
