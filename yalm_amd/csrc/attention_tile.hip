// Attention of a step whose prompts are one tile (64 positions) each, from the sums of the q/k/v product to the heads' results:
// the rotation, the cache write and the attention of attention_mfma_prefill.hip in one launch (see attention_mfma.h for the
// products' layout).
#include "attention_mfma.h"

namespace {

// Where the value of row `row` lies in an element's LDS row: groups of 8 rows, turned by the element's place, so that the lanes that store
// neighbouring elements of a row meet in pairs and not in eights
__device__ __forceinline__ int v_place(int el, int row) { return row ^ ((el >> 4) & 7) << 3; }

// A workgroup takes a query head of a sequence: its waves (eight for heads of 64, sixteen for 128) add the product's K slices and
// rotate q, k and v of that head on their way into LDS, then the waves share the queries in columns of 16, all of them the scores of
// every key, each a part of the result's elements.  The first head of a group writes the cache.  What bounds it is no rate but the way of one launch:
// memory, LDS, two chains of products, memory; with many slices what a compute unit takes in (a slice of 64 tokens is 98 KB a workgroup,
// 1 us).  So one launch in the place of two, keys and values formed again by every head of a group (from the second-level cache) rather
// than handed over through memory, and all loads of a slice asked for before the first is added (two slices at a time gave nothing; eight waves for heads
// of 128 have no registers left for it and took 7.8 us for 5.5).  The bits are those of yalm_rope_kv_write with yalm_attn_prefill behind it.
// us, those two (the rotation by tiles from 320 tokens on) and this, 32 heads of 128 in 8 groups but where stated:
//   33 tokens, 1 slice 8.9 5.5   2 slices 9.1 6.1   4 slices 9.9 7.6   8 slices 11.2 9.7        9 tokens, 24 heads 8.0 5.1
//   64 tokens, 2 slices 9.7 7.6   4 slices 11.0 9.9   8 slices 11.9 14.4       4 x 40 tokens, 1 slice 13.8 6.5   4 slices 14.6 10.0
//   8 x 50, 24 heads 18.7 7.7   40 x 50, 24 heads 37.7 26.6   128 x 64, 2 slices 170 167      heads of 64: 30 tokens 7.5 4.1   100 x 50 46 34
// Where it is behind (many slices of long prompts, many sequences of wide groups) its caller takes the two (one_tile_pays in parts/attention.py).
template <int HD>
__global__ __launch_bounds__(HD * 8) void attn_tile_kernel(
    const float* __restrict__ qkv, bf16* __restrict__ out, bf16* __restrict__ k_pages, bf16* __restrict__ v_pages,
    const int* __restrict__ block_table, int table_stride, const int* __restrict__ cu_seqlens, const int* __restrict__ seq_slot,
    const float2* __restrict__ cos_sin, int n_positions, int n_heads, int n_kv_heads, int rotary_dim, int n_pages, int page_layout,
    int slices, long plane) {
  constexpr int KS = HD / 32, DT = HD / 16;
  constexpr int NT = HD * 8, ROWS = NT / (HD / 4);   // threads, and the rows that they take at a time, four elements a thread
  constexpr int PARTS = NT / 256;                 // waves that share the elements of 16 queries' results
  constexpr int PASSES = PAGE / ROWS;
  constexpr int KROW = HD + 8, VROW = PAGE + 8;   // LDS rows with 16 bytes of padding
  static_assert(HD == 64 || HD == 128, "built for heads of 64 and 128");
  typedef __attribute__((ext_vector_type(4))) __bf16 bf16x4;
  __shared__ __attribute__((aligned(16))) bf16 qs[PAGE * KROW];
  __shared__ __attribute__((aligned(16))) bf16 ks[PAGE * KROW];
  __shared__ __attribute__((aligned(16))) bf16 vs[HD * VROW];

  const int h = blockIdx.x, b = blockIdx.y, group = n_heads / n_kv_heads, g = h / group;
  const int start = cu_seqlens[b], len = min(cu_seqlens[b + 1] - start, PAGE);
  if (len <= 0) return;
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid / WAVE), lane = tid % WAVE, qd = lane / 16, j = lane % 16;
  const int width = (n_heads + 2 * n_kv_heads) * HD;
  const int e = (tid % (HD / 4)) * 4, row0 = tid / (HD / 4), half_rot = rotary_dim / 2;

  bf16 *kpage = nullptr, *vpage = nullptr;
  if (h % group == 0 && k_pages != nullptr) {
    const int slot = seq_slot[b];
    const int phys = slot >= 0 ? block_table[(size_t)slot * table_stride] : -1;
    if (phys >= 0 && phys < n_pages) {
      kpage = k_pages + ((size_t)phys * n_kv_heads + g) * PAGE * HD;
      vpage = v_pages + ((size_t)phys * n_kv_heads + g) * PAGE * HD;
    }
  }

  // the sums of the slices, in their order; rows behind the sequence's end are zeros
  f32x4 a[3][PASSES];
  const float* from[3] = {qkv + (size_t)start * width + h * HD + e, qkv + (size_t)start * width + (n_heads + g) * HD + e,
                          qkv + (size_t)start * width + (n_heads + n_kv_heads + g) * HD + e};
  float2 cs[PASSES][2];
#pragma unroll
  for (int p = 0; p < PASSES; ++p) {
    const int row = p * ROWS + row0;
#pragma unroll
    for (int w = 0; w < 3; ++w)
      a[w][p] = row < len ? *reinterpret_cast<const f32x4*>(from[w] + (size_t)row * width) : (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int u = 0; u < 2; ++u)
      cs[p][u] = cos_sin != nullptr && row < len && row < n_positions && e / 2 + u < half_rot ? cos_sin[(size_t)row * half_rot + e / 2 + u]
                                                                                            : make_float2(1.f, 0.f);
  }
  for (int s = 1; s < slices; ++s) {
    f32x4 more[3][PASSES];
#pragma unroll
    for (int p = 0; p < PASSES; ++p)
#pragma unroll
      for (int w = 0; w < 3; ++w) {
        const int row = p * ROWS + row0;
        more[w][p] = row < len ? *reinterpret_cast<const f32x4*>(from[w] + s * plane + (size_t)row * width) : (f32x4){0.f, 0.f, 0.f, 0.f};
      }
#pragma unroll
    for (int p = 0; p < PASSES; ++p)
#pragma unroll
      for (int w = 0; w < 3; ++w) a[w][p] += more[w][p];
  }
#pragma unroll
  for (int p = 0; p < PASSES; ++p) {
    const int row = p * ROWS + row0;
    const bool turn = cos_sin != nullptr && row < n_positions;
    bf16x4 r[2];                                  // q, k
#pragma unroll
    for (int w = 0; w < 2; ++w)
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        float x0 = a[w][p][2 * u], x1 = a[w][p][2 * u + 1];
        if (turn && e / 2 + u < half_rot) {
          const float y0 = rotate_one(x0, x1, false, cs[p][u]), y1 = rotate_one(x1, x0, true, cs[p][u]);
          x0 = y0;
          x1 = y1;
        }
        r[w][2 * u] = static_cast<bf16>(x0);
        r[w][2 * u + 1] = static_cast<bf16>(x1);
      }
    *reinterpret_cast<bf16x4*>(qs + row * KROW + e) = r[0];
    *reinterpret_cast<bf16x4*>(ks + row * KROW + e) = r[1];
    if (kpage != nullptr && row < len) *reinterpret_cast<bf16x4*>(kpage + page_k_offset(page_layout, row, e, HD)) = r[1];
#pragma unroll
    for (int i = 0; i < 4; ++i) vs[(e + i) * VROW + v_place(e + i, row)] = static_cast<bf16>(a[2][p][i]);
  }
  __syncthreads();

  if (vpage != nullptr)                           // 8 rows of an element at a time; the page is the sequence's own to its end
    for (int c = tid; c < HD * ((len + 7) / 8); c += NT) {
      const int el = c % HD, r = c / HD * 8;
      *reinterpret_cast<bf16x8*>(vpage + page_v_offset(page_layout, r, el, HD)) = *reinterpret_cast<const bf16x8*>(vs + el * VROW + v_place(el, r));
    }

  const int pos = (wave % 4) * 16 + j, dt0 = wave / 4 * (DT / PARTS);
  if ((wave % 4) * 16 >= len) return;
  const float score_scale = 1.4426950408889634f / sqrtf((float)HD);   // log2(e) / sqrt(head_dim)
  bf16x8 qv[KS];
#pragma unroll
  for (int k = 0; k < KS; ++k) qv[k] = *reinterpret_cast<const bf16x8*>(qs + pos * KROW + k * 32 + qd * 8);
  f32x4 sc[4];
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    sc[t] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int k = 0; k < KS; ++k) {
      const bf16x8 kf = *reinterpret_cast<const bf16x8*>(ks + key_row(t, j) * KROW + k * 32 + qd * 8);
      sc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf, qv[k], sc[t], 0, 0, 0);
    }
  }
  float mx = -FLT_MAX;
#pragma unroll
  for (int t = 0; t < 4; ++t)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float v = 32 * (t >> 1) + 8 * qd + 4 * (t & 1) + r <= pos ? sc[t][r] : -INFINITY;
      sc[t][r] = v;
      mx = fmaxf(mx, v);
    }
  mx = fmaxf(mx, __shfl_xor(mx, 16, WAVE));
  mx = fmaxf(mx, __shfl_xor(mx, 32, WAVE));
  const float m = fmaxf(-FLT_MAX, mx * score_scale);
  float l = 0.f;
  bf16x8 pb[2];
#pragma unroll
  for (int s2 = 0; s2 < 2; ++s2)
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float p = __builtin_amdgcn_exp2f(fmaf(sc[2 * s2 + (i >> 2)][i & 3], score_scale, -m));
      l += p;
      pb[s2][i] = static_cast<bf16>(p);
    }
  l += __shfl_xor(l, 16, WAVE);
  l += __shfl_xor(l, 32, WAVE);
  const float inv_l = 1.0f / l;
  bf16* orow = out + ((size_t)(start + min(pos, len - 1)) * n_heads + h) * HD;
#pragma unroll
  for (int d = 0; d < DT / PARTS; ++d) {
    const int dt = dt0 + d;
    f32x4 o = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s2 = 0; s2 < 2; ++s2) {
      const bf16x8 vf = *reinterpret_cast<const bf16x8*>(vs + (dt * 16 + j) * VROW + v_place(dt * 16 + j, s2 * 32 + qd * 8));
      o = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf, pb[s2], o, 0, 0, 0);
    }
    if (pos < len) {
      bf16x4 w;
#pragma unroll
      for (int r = 0; r < 4; ++r) w[r] = static_cast<bf16>(o[r] * inv_l);
      *reinterpret_cast<bf16x4*>(orow + dt * 16 + 4 * qd) = w;
    }
  }
}

}  // namespace

extern "C" int yalm_attn_tile(const float* qkv, void* out, void* k_pages, void* v_pages, const int* block_table, int table_stride,
                              const int* cu_seqlens, const int* seq_slot, const float* cos_sin, int n_positions, int T, int B, int n_tiles,
                              int n_heads, int n_kv_heads, int head_dim, int rotary_dim, int n_pages, int page_layout, int slices,
                              hipStream_t stream) {
  if (T <= 0 || B <= 0) return YALM_OK;
  if (n_tiles != B || B > 65535 || n_heads <= 0 || n_kv_heads <= 0 || n_heads % n_kv_heads != 0 || (head_dim != 64 && head_dim != 128) ||
      rotary_dim < 0 || (rotary_dim & 1) || rotary_dim > head_dim || slices < 1 || !page_layout_ok(page_layout, head_dim) ||
      (((uintptr_t)qkv | (uintptr_t)out | (uintptr_t)k_pages | (uintptr_t)v_pages) & 15) || (k_pages == nullptr) != (v_pages == nullptr))
    return YALM_ERR_ARG;
  const long plane = (long)T * (n_heads + 2 * n_kv_heads) * head_dim;
  const dim3 grid(n_heads, B);
#define YALM_TILE(HD_)                                                                                                                  \
  attn_tile_kernel<HD_><<<grid, HD_ * 8, 0, stream>>>(qkv, (bf16*)out, (bf16*)k_pages, (bf16*)v_pages, block_table, table_stride, cu_seqlens, \
                                                  seq_slot, (const float2*)cos_sin, n_positions, n_heads, n_kv_heads, rotary_dim, n_pages, \
                                                  page_layout, slices, plane)
  if (head_dim == 128)
    YALM_TILE(128);
  else
    YALM_TILE(64);
#undef YALM_TILE
  return launch_status();
}
