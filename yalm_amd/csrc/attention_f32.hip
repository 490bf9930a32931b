// Attention of the true 32-bit path on the matrix cores (v_mfma_f32_16x16x4_f32), softmax state and expf in float32:
// head sizes of 64 to 128 in steps of 16, every shape of the scores.  The kernels of attention_simple.hip take the others.
// Smaller heads stay there for their bits, not for their time: both sum to about 3e-7, in another order, and a model of heads of 8
// to 24 with a recurrent head beside the attention read a nearly empty recurrent state there, which magnifies a last bit a
// thousandfold: 1.1e-4 off in the logits with these kernels, 2.7e-5 with the general ones.  Heads of 32 and 48 have not been
// compared and stay with them too.
//
//   scores^T[key, query] = K[key, :] . Q[query, :]        A = 16 key rows x 4 elements, B = 16 queries
//   out^T[elem, query]  += V^T[elem, key] P^T[key, query]  A = 16 elements x 4 keys, B = P^T
//
// Lane (lq, l16) reads four consecutive elements of a key row (of its query) at once and feeds them to four products; the
// first product leaves it four consecutive keys of one query, and product r of the second takes key r of all four lq: the
// probabilities never leave their registers, and a lane reads the four keys of its V^T row at once.
// A tile's part of out is summed from zero and joins the total once (o <- o corr + part), as attention_simple.hip sums.
//
// Probabilities of zero still multiply their value there, and 0 times infinity is no number.  Keys whose values are not all
// finite are mixed one by one instead, zeros left out.
//
// 701 tokens, 24 heads of 128: 2,564 -> 87 us a layer; a decode step of 4 sequences of 20 to 36 tokens, 4 heads of 128:
// 24 -> 8 us, and no kernel that merges splits behind it where there is one; 8 sequences of 4,000 tokens 666 -> 46 us.
#include <float.h>
#include <type_traits>
#include "common.h"
#include "attention_merge.h"
#include "sinks.h"
#include "yalm_hip.h"

namespace {

typedef __attribute__((ext_vector_type(4))) float f32x4;

__device__ __forceinline__ f32x4 ld4(const float* p) { return *reinterpret_cast<const f32x4*>(p); }
__device__ __forceinline__ f32x4 mfma4(float a, float b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }

// the score of a scaled product at a distance
__device__ __forceinline__ float shaped(const ScoreShape& sh, float s, int head, int distance) {
  if (sh.softcap > 0.f) s = sh.softcap * tanhf(s / sh.softcap);
  float term = sh.bias != nullptr ? sh.bias[(size_t)head * sh.n_bias + min(max(distance, 0), sh.n_bias - 1)] : 0.f;
  if (sh.slope != nullptr) term -= sh.slope[head] * (float)distance;
  if (sh.log_a != nullptr) term -= sh.log_a[head] * log1pf(sh.log_b[head] * (float)max(distance, 0));
  return s + term;
}

// ---------------------------------------------------------------------------
// prefill: a workgroup of four waves takes 64 query positions of one head, a wave 16 of them; key and value tiles of 64 go
// through LDS once a workgroup, the next one's loads in flight meanwhile.  Grid (head, tile): the tiles that see the most
// keys start first; the heads of a group run together and share their keys in the cache.  Bound by the matrix cores: a tile
// of 64 keys is 256 products of 32 clocks a wave at head size 128.
// ---------------------------------------------------------------------------
template <int HD, bool SHAPED>
__global__ __launch_bounds__(256, 2) void attn_prefill_f32_kernel(
    const float* __restrict__ q, const float* __restrict__ k_stage, const float* __restrict__ v_stage,
    float* __restrict__ out, float* __restrict__ out_f32, float* __restrict__ lse, const int* __restrict__ cu_seqlens,
    const int* __restrict__ seq_tile0, int B, int n_heads, int n_kv_heads, int window, ScoreShape sh) {
  constexpr int DT = HD / 16, KROW = HD + 4, VROW = PAGE + 4, NLOAD = HD / 16;
  extern __shared__ __attribute__((aligned(16))) float smem[];
  float* ks = smem;                                // [64][KROW]
  float* vs = smem + PAGE * KROW;                  // [HD][VROW]
  __shared__ int odd_values[2];                    // a value of the (even, odd) tile is not finite
  const int h = blockIdx.x, gt = (int)gridDim.y - 1 - (int)blockIdx.y;
  const int tid = threadIdx.x, lane = tid % WAVE, l16 = lane % 16, lq = lane / 16;
  const int wave = __builtin_amdgcn_readfirstlane(tid / WAVE);
  int b = 0;
  for (int hi = B - 1; b < hi;) {                  // the last sequence whose first tile is not behind this one
    const int mid = (b + hi + 1) >> 1;
    if (seq_tile0[mid] <= gt) b = mid; else hi = mid - 1;
  }
  const int tile0 = seq_tile0[b], start = cu_seqlens[b], len = cu_seqlens[b + 1] - start;
  const int blk0 = (gt - tile0) * PAGE;
  if (blk0 >= len) return;
  const int g = h / (n_heads / n_kv_heads);
  const int pos0 = blk0 + wave * 16, pos = pos0 + l16;
  const bool live = pos < len;
  const int lo = first_visible(pos, window, sh.block), wave_lo = first_visible(pos0, window, sh.block);
  const int wave_last = min(pos0 + 15, len - 1);
  const float inv = sqrtf((float)HD);

  f32x4 qv[DT];
  {
    const float* qr = q + ((size_t)(start + (live ? pos : len - 1)) * n_heads + h) * HD + lq * 4;
#pragma unroll
    for (int s = 0; s < DT; ++s) qv[s] = ld4(qr + s * 16);
  }
  float m = -FLT_MAX, l = 0.f;                     // l: this lane's keys only
  f32x4 o[DT];
#pragma unroll
  for (int d = 0; d < DT; ++d) o[d] = (f32x4){0.f, 0.f, 0.f, 0.f};

  const int kt_lo = first_visible(blk0, window, sh.block) / PAGE, kt_hi = min(blk0 + PAGE - 1, len - 1) / PAGE;
  f32x4 rk[NLOAD], rv[NLOAD];
  auto load_tile = [&](int kt) {
    const size_t at = ((size_t)(tile0 + kt) * n_kv_heads + g) * PAGE * HD;
#pragma unroll
    for (int p = 0; p < NLOAD; ++p) {
      rk[p] = ld4(k_stage + at + (size_t)(tid + p * 256) * 4);
      rv[p] = ld4(v_stage + at + (size_t)(tid + p * 256) * 4);
    }
  };
  // keys as they lie; values with zeros behind the sequence's end, where anything may lie.  True: some value is not finite
  auto store_tile = [&](int kt) {
    bool odd = false;
#pragma unroll
    for (int p = 0; p < NLOAD; ++p) {
      const int c = tid + p * 256, row = c / (HD / 4), col = c % (HD / 4) * 4;
      *reinterpret_cast<f32x4*>(ks + row * KROW + col) = rk[p];
      const int vrow = c / (PAGE / 4), vcol = c % (PAGE / 4) * 4;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if (kt * PAGE + vcol + e >= len) rv[p][e] = 0.f;
        odd = odd || !(fabsf(rv[p][e]) <= FLT_MAX);
      }
      *reinterpret_cast<f32x4*>(vs + vrow * VROW + vcol) = rv[p];
    }
    return odd;
  };

  load_tile(kt_lo);
  if (tid < 2) odd_values[tid] = 0;
  for (int kt = kt_lo; kt <= kt_hi; ++kt) {
    __syncthreads();                               // the tile before has been read
    if (tid == 0) odd_values[(kt + 1) & 1] = 0;
    if (store_tile(kt)) odd_values[kt & 1] = 1;
    if (kt < kt_hi) load_tile(kt + 1);
    lds_barrier();
    const int base = kt * PAGE;
    if (pos0 >= len || base > wave_last || base + PAGE - 1 < wave_lo) continue;       // the same for the whole wave
    f32x4 sc[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      f32x4 even = {0.f, 0.f, 0.f, 0.f}, uneven = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < DT; ++s) {
        const f32x4 kf = ld4(ks + (t * 16 + l16) * KROW + s * 16 + lq * 4);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          if (s % 2 == 0) even = mfma4(kf[e], qv[s][e], even);
          else uneven = mfma4(kf[e], qv[s][e], uneven);
        }
      }
      sc[t] = even + uneven;
    }
    // lane (lq, l16) holds the keys base + 16 t + 4 lq + r of query l16
    const bool edge = base + PAGE - 1 > pos0 || base < first_visible(wave_last, window, sh.block);
    float mx = -FLT_MAX;
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int j = base + t * 16 + lq * 4 + r;
        float s = sc[t][r] / inv;
        if constexpr (SHAPED) s = shaped(sh, s, h, pos - j);
        if (edge && (j > pos || j < lo)) s = -INFINITY;
        sc[t][r] = s;
        mx = fmaxf(mx, s);
      }
    mx = fmaxf(mx, __shfl_xor(mx, 16, WAVE));
    mx = fmaxf(mx, __shfl_xor(mx, 32, WAVE));
    const float m_new = fmaxf(m, mx), corr = expf(m - m_new);
    float psum = 0.f;
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        sc[t][r] = expf(sc[t][r] - m_new);
        psum += sc[t][r];
      }
    l = l * corr + psum;
    m = m_new;
    if (odd_values[kt & 1]) {
#pragma unroll
      for (int d = 0; d < DT; ++d) o[d] *= corr;
      for (int j = 0; j < PAGE; ++j) {
        float p = 0.f;                             // key j of query l16: in lane (j / 4 mod 4, l16), tile j / 16, place j mod 4
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const float v = __shfl(sc[t][r], (j / 4 % 4) * 16 + l16, WAVE);
            if (j / 16 == t && j % 4 == r) p = v;
          }
        if (p != 0.f) {
#pragma unroll
          for (int d = 0; d < DT; ++d)
#pragma unroll
            for (int r = 0; r < 4; ++r) o[d][r] = fmaf(p, vs[(d * 16 + lq * 4 + r) * VROW + j], o[d][r]);
        }
      }
    } else {
#pragma unroll
      for (int d = 0; d < DT; ++d) {
        f32x4 part = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          const f32x4 vf = ld4(vs + (d * 16 + l16) * VROW + t * 16 + lq * 4);
#pragma unroll
          for (int r = 0; r < 4; ++r) part = mfma4(vf[r], sc[t][r], part);
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) o[d][r] = fmaf(o[d][r], corr, part[r]);
      }
    }
  }
  l += __shfl_xor(l, 16, WAVE);
  l += __shfl_xor(l, 32, WAVE);
  if (SHAPED && sh.sink_logit != nullptr) {        // the learned logit counts in the denominator only
    const float sk = sh.sink_logit[h], m_new = fmaxf(m, sk), corr = expf(m - m_new);
    l = l * corr + expf(sk - m_new);
    m = m_new;
#pragma unroll
    for (int d = 0; d < DT; ++d) o[d] *= corr;
  }
  if (!live) return;
  // lane (lq, l16) holds the elements 16 d + 4 lq + r of query l16
  const size_t row = (size_t)(start + pos) * n_heads + h;
#pragma unroll
  for (int d = 0; d < DT; ++d) {
    f32x4 v;
#pragma unroll
    for (int r = 0; r < 4; ++r) v[r] = o[d][r] / l;
    *reinterpret_cast<f32x4*>(out + row * HD + d * 16 + lq * 4) = v;
    if (out_f32 != nullptr) *reinterpret_cast<f32x4*>(out_f32 + row * HD + d * 16 + lq * 4) = v;
  }
  // natural logarithm of the sum of exp(score) over the keys seen: for a later mix with further keys
  if (lse != nullptr && lq == 0) lse[row] = m + logf(l);
}

// ---------------------------------------------------------------------------
// decode: one query a sequence over the pages of the cache; grid (split, KV head and up to 16 of its query heads, sequence).
// Each of the four waves takes a quarter of every page of the split (the 16 key rows that lie together where pages are in
// blocks), so that a short context is worked by all of them; the next page's keys are in flight while a page is mixed, and the
// waves' results are merged in LDS.  Bound by memory for long contexts, by a page's chain of loads, products and
// exponentials for short ones.
// ---------------------------------------------------------------------------
template <int HD, bool BLOCKS, bool SHAPED>
__global__ __launch_bounds__(256, 2) void attn_decode_f32_kernel(
    const float* __restrict__ q, const float* __restrict__ k_pages, const float* __restrict__ v_pages,
    const int* __restrict__ block_table, int table_stride, int ring_pages, const int* __restrict__ seq_slot,
    const int* __restrict__ seq_len, float* __restrict__ partial, float* __restrict__ out, float* __restrict__ lse,
    int n_heads, int n_kv_heads, int window, int n_splits, int n_pages, const int* __restrict__ seq_order, ScoreShape sh, int* __restrict__ counters) {
  constexpr int DT = HD / 16, NW = 4, LAYOUT = BLOCKS ? YALM_PAGE_BLOCKS : YALM_PAGE_ROWS;
  __shared__ float sm_m[NW][16], sm_l[NW][16];
  __shared__ f32x4 sm_o[NW][DT][WAVE];
  const int Gall = n_heads / n_kv_heads, parts_g = (Gall + 15) / 16;
  const int split = blockIdx.x, g = (int)blockIdx.y / parts_g, h0 = g * Gall + ((int)blockIdx.y % parts_g) * 16;
  const int b = seq_order != nullptr ? min(max(seq_order[blockIdx.z], 0), (int)gridDim.z - 1) : (int)blockIdx.z;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x / WAVE), lane = threadIdx.x % WAVE;
  const int l16 = lane % 16, lq = lane / 16;
  const int G = min(16, (g + 1) * Gall - h0);      // heads of this workgroup, the first being head h0
  const int h = h0 + min(l16, G - 1);              // of this lane's column
  const int slot = seq_slot[b], L = slot >= 0 ? seq_len[b] : 0;
  float m = -FLT_MAX, l = 0.f;
  f32x4 o[DT];
#pragma unroll
  for (int d = 0; d < DT; ++d) o[d] = (f32x4){0.f, 0.f, 0.f, 0.f};

  if (L > 0) {
    const int lo = first_visible(L - 1, window, sh.block), first_page = lo / PAGE, last_page = (L - 1) / PAGE;
    // cut by the sequence's own length: in float32 its sums hang on no other sequence of the step
    const int per = (last_page - first_page + n_splits) / n_splits;
    const int p_begin = first_page + split * per, p_end = min(last_page + 1, p_begin + per);
    const float inv = sqrtf((float)HD);
    const size_t page_elems = (size_t)n_kv_heads * PAGE * HD;
    const int* table = block_table + (size_t)slot * table_stride;
    // the wave's key rows: row0 + 8 (i / 4) + i mod 4 for i < 16 (page_row_place's 16 wave ... 16 wave + 15)
    const int row0 = 32 * (wave >> 1) + 4 * (wave & 1);
    const int k_row = row0 + 8 * (l16 >> 2) + (l16 & 3), v_row = row0 + 8 * lq;
    f32x4 qv[DT], kf[DT], vf[DT];
#pragma unroll
    for (int s = 0; s < DT; ++s) qv[s] = ld4(q + ((size_t)b * n_heads + h) * HD + s * 16 + lq * 4);
    // a page that does not exist (never the case for a live sequence) is seen by nobody; some other is read in its place
    auto page_at = [&](int phys) { return (size_t)min(max(phys, 0), n_pages - 1) * page_elems + (size_t)g * PAGE * HD; };
    auto load_keys = [&](size_t at) {
#pragma unroll
      for (int s = 0; s < DT; ++s) kf[s] = ld4(k_pages + at + page_k_offset(LAYOUT, k_row, s * 16 + lq * 4, HD));
    };
    int phys = 0;                                  // the page
    // one page; has_next is a compile-time tag (std::true_type: the next page's keys are asked for)
    auto one_page = [&](int ap, auto has_next) {
      constexpr bool NEXT = decltype(has_next)::value;
      const int phys_next = NEXT ? table[(ap + 1) % ring_pages] : 0;
      const size_t at_v = page_at(phys);
      const bool there = phys >= 0 && phys < n_pages;
#pragma unroll
      for (int d = 0; d < DT; ++d) vf[d] = ld4(v_pages + at_v + page_v_offset(LAYOUT, v_row, d * 16 + l16, HD));
      __builtin_amdgcn_sched_barrier(0);           // the values are asked for before the keys are waited for
      f32x4 even = {0.f, 0.f, 0.f, 0.f}, uneven = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < DT; ++s)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          if (s % 2 == 0) even = mfma4(kf[s][e], qv[s][e], even);
          else uneven = mfma4(kf[s][e], qv[s][e], uneven);
        }
      f32x4 sc = even + uneven;
      if constexpr (NEXT) {
        load_keys(page_at(phys_next));             // in flight while this page is mixed
        phys = phys_next;
        __builtin_amdgcn_sched_barrier(0);
      }
      const int pos0 = ap * PAGE + v_row;          // lane (lq, l16) holds the keys pos0 + r of head l16
      float mx = -FLT_MAX;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const bool seen = there && pos0 + r >= lo && pos0 + r < L;
        float s = sc[r] / inv;
        if constexpr (SHAPED) s = shaped(sh, s, h, L - 1 - pos0 - r);
        sc[r] = seen ? s : -INFINITY;
        mx = fmaxf(mx, sc[r]);
#pragma unroll
        for (int d = 0; d < DT; ++d)               // rows that nobody sees may hold anything
          if (!seen) vf[d][r] = 0.f;
      }
      mx = fmaxf(mx, __shfl_xor(mx, 16, WAVE));
      mx = fmaxf(mx, __shfl_xor(mx, 32, WAVE));
      const float m_new = fmaxf(m, mx), corr = expf(m - m_new);
      float psum = 0.f;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        sc[r] = expf(sc[r] - m_new);
        psum += sc[r];
      }
      l = l * corr + psum;
      m = m_new;
      f32x4 part[DT];
      float z = 0.f;                               // no number if some part is not finite
#pragma unroll
      for (int d = 0; d < DT; ++d) {
        part[d] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int r = 0; r < 4; ++r) part[d] = mfma4(vf[d][r], sc[r], part[d]);
#pragma unroll
        for (int r = 0; r < 4; ++r) z = fmaf(part[d][r], 0.f, z);
      }
      if (__any(z != 0.f)) {                       // key by key, probabilities of zero left out
#pragma unroll
        for (int d = 0; d < DT; ++d) part[d] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
        for (int key = 0; key < 16; ++key) {       // key 4 k + r in lane (k, l16), place r
          const int r = key & 3;
          const float p = __shfl(r < 2 ? (r == 0 ? sc[0] : sc[1]) : (r == 2 ? sc[2] : sc[3]), key / 4 * 16 + l16, WAVE);
          if (p != 0.f) {
#pragma unroll
            for (int d = 0; d < DT; ++d)
#pragma unroll
              for (int e = 0; e < 4; ++e)
                part[d][e] = fmaf(p, v_pages[at_v + page_v_offset(LAYOUT, row0 + 8 * (key / 4) + r, d * 16 + lq * 4 + e, HD)], part[d][e]);
          }
        }
      }
#pragma unroll
      for (int d = 0; d < DT; ++d)
#pragma unroll
        for (int r = 0; r < 4; ++r) o[d][r] = fmaf(o[d][r], corr, part[d][r]);
    };
    if (p_begin < p_end) {
      phys = table[p_begin % ring_pages];
      load_keys(page_at(phys));
      int ap = p_begin;
      for (; ap + 1 < p_end; ++ap) one_page(ap, std::true_type{});
      one_page(ap, std::false_type{});
    }
  }

  l += __shfl_xor(l, 16, WAVE);                    // the four lanes of a column hold parts of its sum; then the waves merge
  l += __shfl_xor(l, 32, WAVE);
  if (lq == 0) sm_m[wave][l16] = m;
  __syncthreads();
  float m_all = sm_m[0][l16];
#pragma unroll
  for (int w = 1; w < NW; ++w) m_all = fmaxf(m_all, sm_m[w][l16]);
  const float scale = expf(m - m_all);
#pragma unroll
  for (int d = 0; d < DT; ++d) sm_o[wave][d][lane] = o[d] * scale;
  if (lq == 0) sm_l[wave][l16] = l * scale;
  __syncthreads();
  float lt = (sm_l[0][l16] + sm_l[1][l16]) + (sm_l[2][l16] + sm_l[3][l16]);
  float keep = 1.0f;
  float* to;
  if (n_splits == 1 && out != nullptr) {           // one split: this is the result
    to = out + ((size_t)b * n_heads + h) * HD;
    if (SHAPED && sh.sink_logit != nullptr && lt > 0.f) {     // the learned logit: in the denominator only
      const float sk = sh.sink_logit[h], m_new = fmaxf(m_all, sk);
      keep = expf(m_all - m_new);
      lt = lt * keep + expf(sk - m_new);
      m_all = m_new;
    }
    keep = lt > 0.f ? keep / lt : 0.f;
    if (lse != nullptr && wave == 0 && lq == 0 && l16 < G) lse[(size_t)b * n_heads + h] = lt > 0.f ? m_all + logf(lt) : -FLT_MAX;
  } else {
    to = partial + (((size_t)b * n_heads + h) * n_splits + split) * (HD + 2);
    if (wave == 0 && lq == 0 && l16 < G) {
      if (counters != nullptr) {
        store_pair(to + HD, m_all, lt);
      } else {
        to[HD] = m_all;
        to[HD + 1] = lt;
      }
    }
  }
#pragma unroll
  for (int d = 0; d < DT; ++d)
    if (d % NW == wave && l16 < G) {
      const f32x4 v = (sm_o[0][d][lane] + sm_o[1][d][lane]) + (sm_o[2][d][lane] + sm_o[3][d][lane]);
      if (counters != nullptr) {
        store_pair(to + d * 16 + lq * 4, v[0], v[1]);
        store_pair(to + d * 16 + lq * 4 + 2, v[2], v[3]);
      } else {
#pragma unroll
        for (int r = 0; r < 4; ++r) to[d * 16 + lq * 4 + r] = v[r] * keep;       // a partial row need not lie on 16 bytes
      }
    }
  if (counters != nullptr && last_to_arrive(counters + ((size_t)blockIdx.z * gridDim.y + blockIdx.y) * COUNTER_STRIDE, n_splits))
    merge_splits<HD, NW, false>(partial, out, lse, b, n_heads, h0, G, n_splits, sh.sink_logit, wave, lane);
}

template <int HD>
int launch_prefill(const float* q, const float* k_stage, const float* v_stage, float* out, float* out_f32, float* lse,
                   const int* cu_seqlens, const int* seq_tile0, int B, int n_tiles, int n_heads, int n_kv_heads,
                   int window, const ScoreShape& shape, hipStream_t stream) {
  constexpr int lds = (PAGE * (HD + 4) + HD * (PAGE + 4)) * (int)sizeof(float);
  const dim3 grid(n_heads, n_tiles);
  auto run = [&](auto kernel, LdsAllowance& allowed) -> int {
    if (lds > 60 * 1024)
      if (int rc = allow_dynamic_lds(allowed, (const void*)kernel, lds); rc != YALM_OK) return rc;
    kernel<<<grid, 256, lds, stream>>>(q, k_stage, v_stage, out, out_f32, lse, cu_seqlens, seq_tile0, B, n_heads,
                                       n_kv_heads, window, shape);
    return launch_status();
  };
  static LdsAllowance plain_allowed, shaped_allowed;
  if (shape.any()) return run(&attn_prefill_f32_kernel<HD, true>, shaped_allowed);
  return run(&attn_prefill_f32_kernel<HD, false>, plain_allowed);
}

bool takes(int head_dim, const void* a, const void* b, const void* c, const void* d) {
  return head_dim >= 64 && head_dim <= 128 && head_dim % 16 == 0 &&
         (((uintptr_t)a | (uintptr_t)b | (uintptr_t)c | (uintptr_t)d) & 15) == 0;
}

}  // namespace

// YALM_ERR_ARG: not taken (the caller runs the kernel of attention_simple.hip)
int yalm_attn_prefill_f32_mfma(const void* q, const void* k_stage, const void* v_stage, void* out, float* out_f32, float* lse,
                               const int* cu_seqlens, const int* seq_tile0, int B, int n_tiles, int n_heads,
                               int n_kv_heads, int head_dim, int window, const ScoreShape& shape, hipStream_t stream) {
  if (!takes(head_dim, q, k_stage, v_stage, out) || ((uintptr_t)out_f32 & 15) || B <= 0 || n_tiles > 65535) return YALM_ERR_ARG;
#define YALM_HD(HD_)                                                                                                     \
  case HD_:                                                                                                              \
    return launch_prefill<HD_>((const float*)q, (const float*)k_stage, (const float*)v_stage, (float*)out, out_f32, lse, \
                               cu_seqlens, seq_tile0, B, n_tiles, n_heads, n_kv_heads, window, shape, stream)
  switch (head_dim) {
    YALM_HD(64);
    YALM_HD(80);
    YALM_HD(96);
    YALM_HD(112);
    YALM_HD(128);
  }
#undef YALM_HD
  return YALM_ERR_ARG;
}

// out null: the splits' partial results are merged by the caller; with counters the kernel merges them.  YALM_ERR_ARG: not taken
int yalm_attn_decode_f32_mfma(const void* q, const void* k_pages, const void* v_pages, const int* block_table,
                              int table_stride, int ring_pages, const int* seq_slot, const int* seq_len, void* out, float* lse,
                              float* partial, int B, int n_heads, int n_kv_heads, int head_dim, int window, int n_splits,
                              int n_pages, int page_layout, const int* seq_order, const ScoreShape& shape, int* counters,
                              hipStream_t stream) {
  const int parts_g = (n_heads / n_kv_heads + 15) / 16;
  const bool blocks = page_layout == YALM_PAGE_BLOCKS;
  if (!takes(head_dim, q, k_pages, v_pages, nullptr) || (long)n_kv_heads * parts_g > 65535 || B > 65535 ||
      (blocks && head_dim % 32 != 0) || (out == nullptr && partial == nullptr) || (out == nullptr && counters != nullptr))
    return YALM_ERR_ARG;
  const dim3 grid(n_splits, n_kv_heads * parts_g, B);
#define YALM_RUN(HD_, BLOCKS_, SHAPED_)                                                                                  \
  attn_decode_f32_kernel<HD_, BLOCKS_, SHAPED_><<<grid, 256, 0, stream>>>(                                               \
      (const float*)q, (const float*)k_pages, (const float*)v_pages, block_table, table_stride, ring_pages, seq_slot,    \
      seq_len, partial, (float*)out, lse, n_heads, n_kv_heads, window, n_splits, n_pages, seq_order, shape, counters)
#define YALM_HD16(HD_)                                                                                                   \
  case HD_:                                                                                                              \
    if (shape.any()) YALM_RUN(HD_, false, true);                                                                         \
    else YALM_RUN(HD_, false, false);                                                                                    \
    break
#define YALM_HD32(HD_)                                                                                                   \
  case HD_:                                                                                                              \
    if (blocks && shape.any()) YALM_RUN(HD_, true, true);                                                                \
    else if (blocks) YALM_RUN(HD_, true, false);                                                                         \
    else if (shape.any()) YALM_RUN(HD_, false, true);                                                                    \
    else YALM_RUN(HD_, false, false);                                                                                    \
    break
  switch (head_dim) {
    YALM_HD32(64);
    YALM_HD16(80);
    YALM_HD32(96);
    YALM_HD16(112);
    YALM_HD32(128);
  }
#undef YALM_HD32
#undef YALM_HD16
#undef YALM_RUN
  return launch_status();
}
