// The merge of a decode step's attention splits inside the attention kernel: the workgroup that arrives last of a (sequence,
// KV head)'s splits merges their partial results, in one order whoever is last, so that no kernel of its own does
// (4.7 us a layer of a decode step, most of it a launch).  counters: an int for each (sequence, blockIdx.y), zero before
// the launch and behind it, each in a line of memory of its own (arrivals at counters of one line wait for each other: eight rows
// in 16 splits 9.1 us with them side by side, 8.4 apart).
//
// The partial results pass between XCDs, whose second-level caches do not see each other's lines: they are stored and loaded
// as relaxed atomics of agent scope, which go through to where all XCDs see them and are not served from a cache that does
// not; every wave waits until its stores have got there before the workgroup's barrier, and the counter is raised behind
// that.  (An acquire-release exchange instead writes back and drops the whole cache, once a workgroup: a step of
// thirty-two layers at batch 8 took 3.60 ms that way, with the kernel that merges 3.40.)
#pragma once
#include <float.h>
#include "common.h"

#if defined(__HIP_DEVICE_COMPILE__) && !defined(__gfx950__)
#error "this exchange rests on how gfx950 carries out accesses of agent scope, not on the order of the language"
#endif

constexpr int COUNTER_STRIDE = 32;               // ints
typedef unsigned long long pair_bits;            // two floats

// Whether the last workgroup to arrive should merge the splits of its heads (of `heads` of a KV head, at most 16): a wave takes
// a head, so where there is one for each the merge costs the last workgroup less than a launch behind it, and where the waves
// take several in turn more.  Merged inside against by the kernel behind, us, at 4 / 16 / 64 splits of 256 keys and one sequence:
// four waves and 4 heads of 128 7.1 / 7.6 / 11.3 against 8.0 / 8.4 / 18.6; 8 heads 8.6 / 9.5 / 15.6 against 8.0 / 8.4 / 17.9;
// 16 heads 11.1 / 12.8 / 24.3 against 8.1 / 8.6 / 18.1; two waves and 4 heads of 256 11.5 / 12.8 / 21.4 against 10.9 / 11.4 / 27.0.
inline bool merges_inside(int heads, int waves) { return heads <= waves; }

__device__ __forceinline__ void store_pair(float* p, float a, float b) {
  const pair_bits v = (pair_bits)__float_as_uint(a) | ((pair_bits)__float_as_uint(b) << 32);
  __hip_atomic_store(reinterpret_cast<pair_bits*>(p), v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ float2 load_pair(const float* p) {
  const pair_bits v = __hip_atomic_load(reinterpret_cast<const pair_bits*>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  return make_float2(__uint_as_float((unsigned)v), __uint_as_float((unsigned)(v >> 32)));
}

// True in every thread of the one workgroup that arrives last of `n`; what the others stored with store_pair is there then.
__device__ __forceinline__ bool last_to_arrive(int* counter, int n) {
  __shared__ int last;
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  if (threadIdx.x == 0) {
    last = __hip_atomic_fetch_add(counter, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == n - 1;
    if (last) __hip_atomic_store(counter, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);     // for the next launch
  }
  __syncthreads();
  return last;
}

// partial: [B, n_heads, n_splits, HD + 2] = (sum[HD], maximum, denominator), on 8 bytes; BASE2: maxima are exponents of 2, else
// of e.  The workgroup's NW waves take the heads h0 ... h0 + G - 1 of row b in turn.  The sums run in the order of
// attn_decode_combine_kernel, so that it does not show in a result which of the two merged: the denominators a lane a split,
// the weighted sums in four chains of every fourth split.
template <int HD, int NW, bool BASE2, typename T>
__device__ __forceinline__ void merge_splits(const float* partial, T* __restrict__ out, float* __restrict__ lse, int b, int n_heads,
                                             int h0, int G, int n_splits, const float* __restrict__ sink_logit, int wave, int lane) {
  constexpr int EL = (HD / 2 + WAVE - 1) / WAVE, PRE = 8, CHAINS = 4;      // pairs of elements a lane; splits asked for together
  static_assert(PRE % CHAINS == 0 && WAVE % PRE == 0, "a split's chain and its lane follow from its place in a run");
  auto weight = [](float d) { return BASE2 ? exp2f(d) : expf(d); };
  for (int hh = wave; hh < G; hh += NW) {
    const int h = h0 + hh;
    const float* part = partial + ((size_t)b * n_heads + h) * n_splits * (HD + 2);
    auto maximum_of = [&](int s) { return s < n_splits ? load_pair(part + (size_t)s * (HD + 2) + HD) : make_float2(-FLT_MAX, 0.f); };
    float2 v[2][PRE][EL];
    int none = 0;                                  // zero in a vector register: the splits' places are worked out a lane, from one
    asm("" : "+v"(none));                          // base, and take no scalar registers from the attention's loops
    auto ask = [&](int buf, int s0) {
#pragma unroll
      for (int u = 0; u < PRE; ++u) {
        const int ps = min(s0 + u + none, n_splits - 1) * (HD + 2);
#pragma unroll
        for (int e = 0; e < EL; ++e) v[buf][u][e] = load_pair(part + (unsigned)(ps + 2 * min(lane + e * WAVE, HD / 2 - 1)));
      }
    };
    float2 ml = maximum_of(lane);                  // of split lane
    ask(0, 0);
    if (n_splits > PRE) ask(1, PRE);
    float m = ml.x;
    for (int s = lane + WAVE; s < n_splits; s += WAVE) m = fmaxf(m, maximum_of(s).x);
    m = wave_max(m);
    const float logit = sink_logit != nullptr ? sink_logit[h] * (BASE2 ? 1.4426950408889634f : 1.0f) : -FLT_MAX;
    if (sink_logit != nullptr) m = fmaxf(m, logit);
    float f = weight(ml.x - m);                    // of split lane
    float l = lane < n_splits ? ml.y * f : 0.f;
    for (int s = lane + WAVE; s < n_splits; s += WAVE) {
      const float2 other = maximum_of(s);
      l = fmaf(other.y, weight(other.x - m), l);
    }
    l = wave_sum(l);
    if (sink_logit != nullptr && l > 0.f) l += weight(logit - m);
    float2 acc[CHAINS][EL];
#pragma unroll
    for (int c = 0; c < CHAINS; ++c)
#pragma unroll
      for (int e = 0; e < EL; ++e) acc[c][e] = make_float2(0.f, 0.f);
    auto add = [&](int buf, int s0) {
      if (s0 != 0 && s0 % WAVE == 0) f = weight(maximum_of(s0 + lane).x - m);
#pragma unroll
      for (int u = 0; u < PRE; ++u) {
        const float fs = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(f), (s0 + u) % WAVE));
        if (s0 + u < n_splits) {
#pragma unroll
          for (int e = 0; e < EL; ++e) {
            acc[u % CHAINS][e].x = fmaf(v[buf][u][e].x, fs, acc[u % CHAINS][e].x);
            acc[u % CHAINS][e].y = fmaf(v[buf][u][e].y, fs, acc[u % CHAINS][e].y);
          }
        }
      }
    };
    for (int s0 = 0; s0 < n_splits; s0 += 2 * PRE) {
      add(0, s0);
      if (s0 + 2 * PRE < n_splits) ask(0, s0 + 2 * PRE);
      if (s0 + PRE < n_splits) {
        add(1, s0 + PRE);
        if (s0 + 3 * PRE < n_splits) ask(1, s0 + 3 * PRE);
      }
    }
    const float inv_l = l > 0.f ? 1.0f / l : 0.f;
    T* row = out + ((size_t)b * n_heads + h) * HD;
#pragma unroll
    for (int e = 0; e < EL; ++e) {
      const int p = lane + e * WAVE;
      if (p < HD / 2) {
        row[2 * p] = from_f32<T>((((acc[0][e].x + acc[1][e].x) + acc[2][e].x) + acc[3][e].x) * inv_l);
        row[2 * p + 1] = from_f32<T>((((acc[0][e].y + acc[1][e].y) + acc[2][e].y) + acc[3][e].y) * inv_l);
      }
    }
    if (lse != nullptr && lane == 0)
      lse[(size_t)b * n_heads + h] = l > 0.f ? (BASE2 ? m * 0.6931471805599453f : m) + logf(l) : -FLT_MAX;
  }
}
