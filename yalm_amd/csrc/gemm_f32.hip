// C = epilogue(A[M,K] * W[N,K]^T) in float32 on the matrix cores (v_mfma_f32_16x16x4_f32: products and sums in
// float32, as a chain of fused multiply-adds): the products of the true 32-bit path.
//
// More than 64 rows and K 512 and more go to gemm_split.hip where that is sooner (all but small products).
//
// gemm_f32_kernel, from some 64 rows on bound by the matrix cores (157 TFLOP/s: the vector units' own rate, but an operand
// register serves 16 products where gemm_simple_kernel reads LDS for every eight).  A workgroup of four waves owns a
// tile of 32 FA x 32 FB; a wave FA x FB products of 16 x 16.  k tiles of 32 floats go straight into LDS (128-byte rows,
// 16-byte chunks XOR-swizzled by the row, as in gemm_dma.hip); a lane reads four consecutive k of a row at once and feeds
// them to four products one after the other: which k stands in which place of a product does not matter as long as both
// operands agree.  It reaches 119 to 138 TFLOP/s (rocBLAS 129 to 153); 701 rows against gemm_simple_kernel: 16,384 x 3,072
// 2,250 -> 552 us, 128,256 x 3,072 16.3 -> 4.0 ms, 3,072 x 8,192 1,740 -> 290 us.
//
// gemm_few_f32_kernel and small tiles take a decode step's rows, which the vector units' kernel (gemm_rows_f32_kernel) had
// multiplied at a fraction of memory's rate: 16 rows, 4,096 x 4,096 54 -> 19 us, 128,256 x 3,072 725 -> 276 us; one row,
// 4,096 x 4,096 23 -> 16 us, 128,256 x 3,072 263 -> 257 us.
//
// Sums over short runs of k join a total of their own: short chains of additions lie closer to 64 bits than one over K (a relative
// error of 3.0e-7 at 701 rows and K 8,192, where gemm_simple_kernel's was 1.6e-6; at most 64 rows 0.6e-7 at K 32 to 1.3e-7 at K
// 3,072 and 1.6e-7 at K 14,336, gemm_rows_f32_kernel's 0.6e-7, 1.4e-7 and 2.8e-7).
#include "common.h"
#include "gemm_split.h"
#include "rms_row.h"
#include "yalm_hip.h"

namespace {

typedef __attribute__((ext_vector_type(4))) float f32x4;

constexpr int TK = 32;                           // floats of k a tile
constexpr int ROWB = TK * 4;
constexpr int CPR = ROWB / 16;                   // 16-byte chunks a row
constexpr int RPI = WAVE / CPR;                  // rows one wave instruction brings
constexpr int NW = 4;

__device__ __forceinline__ int swizzle_of(int row) { return (row >> 1) & (CPR - 1); }

__device__ __forceinline__ f32x4 mfma4(float a, float b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }

// The products of the 16 k that a wave's lanes hold, four by four, joined in a tree
__device__ __forceinline__ f32x4 sum_of_products(f32x4 a, f32x4 b) {
  f32x4 p[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) p[e] = mfma4(a[e], b[e], (f32x4){0.f, 0.f, 0.f, 0.f});
  return (p[0] + p[1]) + (p[2] + p[3]);
}

// at most N_ of this wave's loads in flight, and none of its LDS reads
template <int N_>
__device__ __forceinline__ void wait_loads() {
  __builtin_amdgcn_s_waitcnt((N_ & 0xF) | ((N_ >> 4) << 14) | (0x7 << 4) | (0x0 << 8));
}

// stages of LDS: as many as leave room for two workgroups a CU, four at most
constexpr int stages_of(int FA, int FB) { return 640 / (32 * (FA + FB)) < 4 ? 640 / (32 * (FA + FB)) : 4; }
constexpr int GROUP = 4;                         // tile columns that an XCD walks together

// FINE: four chains of sums, one for each of the k that a lane holds side by side, joined every four k tiles and added to a sum
// that joins the total every sixteen: chains of 32, 4 and K / 512 additions.  Else one chain, added to the total every eight k tiles.
template <int EPI, int FA, int FB, bool FINE>
__global__ __launch_bounds__(256, 2) void gemm_f32_kernel(const float* __restrict__ A, const float* __restrict__ W,
                                                          float* __restrict__ C, int M, int N, int K, GateOut H) {
  constexpr int TM = 32 * FA, TN = 32 * FB, ROWS = TM + TN, STAGE_B = ROWS * ROWB, S = stages_of(FA, FB);
  constexpr int L = ROWS / (RPI * NW);           // load instructions a wave and stage
  constexpr int CH = FINE ? 4 : 1, FOLD = FINE ? 4 : 8;
  static_assert(S >= 2 && (S - 1) * L < 64, "vmcnt holds 6 bits");
  static_assert(!gated(EPI) || FB % 2 == 0, "the gated epilogue pairs column tiles");
  extern __shared__ __attribute__((aligned(1024))) unsigned char stages[];
  const int tid = threadIdx.x, lane = tid % WAVE;
  const int wave = __builtin_amdgcn_readfirstlane(tid / WAVE);
  const int wm = wave / 2, wn = wave % 2;
  const int l16 = lane % 16, lq = lane / 16;
  // Workgroup i runs on XCD i mod 8: every XCD takes a run of the tiles (groups of GROUP columns, in a group the columns
  // fastest), so that the tiles it works on at a time share rows and columns in its second-level cache.
  const int mt = (M + TM - 1) / TM, nt = (N + TN - 1) / TN, tiles = mt * nt, chunk = (tiles + 7) / 8;
  const int i0 = blockIdx.x, t = (i0 % 8) * chunk + i0 / 8;
  if (t >= tiles || i0 / 8 >= chunk) return;
  const int per_group = mt * GROUP, g = t / per_group, r0 = t % per_group, width = min(GROUP, nt - g * GROUP);
  const int m0 = (r0 / width) * TM, n0 = (g * GROUP + r0 % width) * TN;

  const float* gp[L];
#pragma unroll
  for (int i = 0; i < L; ++i) {
    const int row = (i * NW + wave) * RPI + lane / CPR;
    const float* base = row < TM ? A + (size_t)min(m0 + row, M - 1) * K          // rows past the edge repeat the last
                                 : W + (size_t)min(n0 + row - TM, N - 1) * K;    // one and are never stored
    gp[i] = base + ((lane % CPR) ^ swizzle_of(row)) * 4;
  }
  auto issue = [&](int kt, int stage, int i) {
#if defined(__HIP_DEVICE_COMPILE__)   // the host pass drops a template that names this builtin, and its launch stub with it
    const float* from = gp[i] + (size_t)kt * TK;
    unsigned char* to = stages + stage * STAGE_B + (i * NW + wave) * 1024;
    // weights that at most 64 rows need are not kept in the caches (2: non-temporal): 4 rows, 128,256 x 3,072 273 -> 254 us
    if (FINE && i >= TM / (RPI * NW)) __builtin_amdgcn_global_load_lds(from, to, 16, 0, 2);
    else __builtin_amdgcn_global_load_lds(from, to, 16, 0, 0);
#endif
  };
  auto issue_all = [&](int kt, int stage) {
#pragma unroll
    for (int i = 0; i < L; ++i) issue(kt, stage, i);
  };

  f32x4 acc[CH][FA][FB], some[FINE ? FA : 1][FINE ? FB : 1], total[FA][FB];
#pragma unroll
  for (int a = 0; a < FA; ++a)
#pragma unroll
    for (int b = 0; b < FB; ++b) {
      total[a][b] = (f32x4){0.f, 0.f, 0.f, 0.f};
      if constexpr (FINE) some[a][b] = total[a][b];
#pragma unroll
      for (int c = 0; c < CH; ++c) acc[c][a][b] = (f32x4){0.f, 0.f, 0.f, 0.f};
    }

  // fragments: address in a stage row * 128 + ((4 s + lq) ^ swizzle) * 16 for step s; tiles 16 rows apart share the swizzle
  const int a_row = wm * (TM / 2) + l16, w_row = wn * (TN / 2) + l16;
  int a_at[2], w_at[2];
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    a_at[s] = a_row * ROWB + (((4 * s + lq) ^ swizzle_of(a_row)) << 4);
    w_at[s] = (TM + w_row) * ROWB + (((4 * s + lq) ^ swizzle_of(TM + w_row)) << 4);
  }

  // Tile kt lies in stage kt mod S; S tiles are in LDS or on their way.  The barrier of a tile stands between its two
  // steps: the second step's fragments are in registers by then, so nobody reads the tile's stage any more and tile
  // kt + S is asked for at once, a load behind every few products; the first fragments of tile kt + 1 are read in front
  // of the last products of tile kt.
  const int nk = K / TK;
#pragma unroll
  for (int s = 0; s < S; ++s)
    if (s < nk) issue_all(s, s);
  if (nk >= S) wait_loads<(S - 1) * L>(); else wait_loads<0>();
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  f32x4 fa[2][FA], fw[2][FB];
  auto read_frags = [&](int stage, int s) {
    const unsigned char* at = stages + stage * STAGE_B;
#pragma unroll
    for (int a = 0; a < FA; ++a) fa[s][a] = *reinterpret_cast<const f32x4*>(at + a_at[s] + a * 16 * ROWB);
#pragma unroll
    for (int b = 0; b < FB; ++b) fw[s][b] = *reinterpret_cast<const f32x4*>(at + w_at[s] + b * 16 * ROWB);
  };
  read_frags(0, 0);
  int stage = 0;
  for (int kt = 0; kt < nk; ++kt) {
    const int next = stage + 1 == S ? 0 : stage + 1;
    read_frags(stage, 1);
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int a = 0; a < FA; ++a)
#pragma unroll
        for (int b = 0; b < FB; ++b)
          acc[e % CH][a][b] = mfma4(fa[0][a][e], fw[0][b][e], acc[e % CH][a][b]);
    __builtin_amdgcn_sched_barrier(0);
    // tile kt + 1 has landed when at most the loads of the S - 2 tiles behind it are in flight
    if (kt + S - 1 < nk) wait_loads<(S - 2) * L>(); else wait_loads<0>();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    read_frags(next, 0);                           // behind the last tile: whatever lies there, never used
    const bool more = kt + S < nk;
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int a = 0; a < FA; ++a)
#pragma unroll
        for (int b = 0; b < FB; ++b) {
          acc[e % CH][a][b] = mfma4(fa[1][a][e], fw[1][b][e], acc[e % CH][a][b]);
          const int j = (e * FA + a) * FB + b;
#pragma unroll
          for (int i = 0; i < L; ++i)
            if (j == (i + 1) * 4 * FA * FB / (L + 1) - 1) {
              if (more) issue(kt + S, stage, i);
              __builtin_amdgcn_sched_barrier(0);
            }
        }
    stage = next;
    if ((kt + 1) % FOLD == 0 || kt + 1 == nk) {
#pragma unroll
      for (int a = 0; a < FA; ++a)
#pragma unroll
        for (int b = 0; b < FB; ++b) {
          if constexpr (FINE) {
            some[a][b] += (acc[0][a][b] + acc[1][a][b]) + (acc[2][a][b] + acc[3][a][b]);
            if ((kt + 1) % (4 * FOLD) == 0 || kt + 1 == nk) {
              total[a][b] += some[a][b];
              some[a][b] = (f32x4){0.f, 0.f, 0.f, 0.f};
            }
          } else {
            total[a][b] += acc[0][a][b];
          }
#pragma unroll
          for (int c = 0; c < CH; ++c) acc[c][a][b] = (f32x4){0.f, 0.f, 0.f, 0.f};
        }
    }
  }

  // lane (lq, l16) holds rows 4 lq .. 4 lq + 3 of column l16 of every 16 x 16
#pragma unroll
  for (int a = 0; a < FA; ++a)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int m = m0 + wm * (TM / 2) + a * 16 + 4 * lq + r;
      if (m >= M) continue;
      if (gated(EPI)) {                              // weight rows: 16 gate rows, 16 up rows, ...: even tiles gate, odd tiles up
#pragma unroll
        for (int p = 0; p < FB / 2; ++p) {
          const int hcol = (n0 + wn * (TN / 2)) / 2 + p * 16 + l16;
          if (hcol < H) C[(size_t)m * H + hcol] = gate_value<EPI>(total[a][2 * p][r], total[a][2 * p + 1][r], H, gate_bias<EPI>(H, hcol));
        }
      } else {
#pragma unroll
        for (int b = 0; b < FB; ++b) {
          const int n = n0 + wn * (TN / 2) + b * 16 + l16;
          if (n >= N) continue;
          const size_t o = (size_t)m * N + n;
          if (EPI == 2) C[o] += total[a][b][r];
          else C[o] = total[a][b][r];
        }
      }
    }
}

// ---------------------------------------------------------------------------
// At most 64 rows (a decode step of the 32-bit path): bound by the weights' one trip from memory.  A workgroup owns
// 16 NB weight rows and 16 MB rows of A; its waves take every NWV-th block of 32 k (128 bytes of each row, whole
// lines), a block's eight products are joined in a tree, and the waves' sums in a tree in LDS: at K 32 NWV, chains of 4 + 3 + 3
// additions.  Weights and A go from memory straight into registers, the next block's while one is multiplied (two blocks ahead
// measured the same).
//
// NORM (a decode step of up to 16 rows): A is the residual stream and its norm is applied on the way: the rows' sums of squares
// first, by every workgroup (a wave a row, in the order of the norm's own kernel, so that its bits come out), then x * scale * weight
// in front of every product.  EPI 4: the q/k/v product of a decode step, rotated and written to the pages of the cache as
// rope_kv_write_kernel does.  A launch less each, seven of a small model's 24 a step (two layers of 256, steps queued: one row 82 -> 70
// us, three 92 -> 80, sixteen 99 -> 88; a step of four 7B layers at one row 974 -> 955 us, at 16 rows 1,152 -> 1,137; of 3B layers at
// 8 rows 857 -> 846).  norm_pays says where.
// ---------------------------------------------------------------------------
constexpr int NWV = 8;
constexpr int EPI_QKV = 4;

struct NormIn {
  const float* w;                                // [K]
  float eps;
};
struct QkvOut {
  float *q_out, *k_pages, *v_pages;
  const int *block_table, *tok_pos, *seq_slot;
  const float2* cos_sin;
  int table_stride, ring_pages, n_positions, n_heads, n_kv_heads, hd, rotary_dim, n_pages, page_layout;
};

// 1 / rms of row x[K], by one wave: the sum of squares as rms_row.h forms it over one or four waves
__device__ __forceinline__ float row_scale(const float* x, int K, bool vec, float eps, int lane) {
  float ss = 0.f;
  if (K <= 1024) {
    ss = wave_sum(rms_part(x, K, lane, WAVE));
  } else {
    float part[4];
#pragma unroll
    for (int p = 0; p < 4; ++p) {
      const int tid = p * WAVE + lane;
      if (vec) {
        part[p] = 0.f;
#pragma unroll
        for (int u = 0; u < RMS_VEC_MAX; ++u) {
          const int i = tid + u * 256;
          part[p] = rms_add4(part[p], i < K / 4 ? reinterpret_cast<const float4*>(x)[i] : make_float4(0.f, 0.f, 0.f, 0.f));
        }
      } else {
        part[p] = rms_part(x, K, tid, 256);
      }
    }
#pragma unroll
    for (int p = 0; p < 4; ++p) ss += wave_sum(part[p]);
  }
  return 1.0f / sqrtf(ss / (float)K + eps);
}

template <int EPI, int MB, int NB, bool NORM>
__global__ __launch_bounds__(NWV * WAVE, 2) void gemm_few_f32_kernel(const float* __restrict__ A, const float* __restrict__ W,
                                                                    float* __restrict__ C, int M, int N, int K, GateOut H, NormIn norm,
                                                                    QkvOut out) {
  static_assert(!gated(EPI) || NB == 2, "a block of gate rows and its up rows");
  static_assert((!NORM && EPI != EPI_QKV) || MB == 1, "up to 16 rows");
  __shared__ f32x4 sums[NWV][MB * NB][WAVE];
  __shared__ float scales[16];
  const int tid = threadIdx.x, lane = tid % WAVE;
  const int wave = __builtin_amdgcn_readfirstlane(tid / WAVE);
  const int l16 = lane % 16, lq = lane / 16;
  const int n0 = blockIdx.x * 16 * NB, m0 = blockIdx.y * 16 * MB;
  A += (size_t)m0 * K;
  C += (size_t)m0 * (gated(EPI) ? (int)H : N);
  M -= m0;
  const float* wp[NB];
  const float* ap[MB];
#pragma unroll
  for (int b = 0; b < NB; ++b) wp[b] = W + (size_t)min(n0 + b * 16 + l16, N - 1) * K + lq * 4;    // rows past the edge repeat the
#pragma unroll
  for (int a = 0; a < MB; ++a) ap[a] = A + (size_t)min(a * 16 + l16, M - 1) * K + lq * 4;         // last one, never stored
  f32x4 acc[MB][NB];
#pragma unroll
  for (int a = 0; a < MB; ++a)
#pragma unroll
    for (int b = 0; b < NB; ++b) acc[a][b] = (f32x4){0.f, 0.f, 0.f, 0.f};

  const int blocks = K / TK, mine = (blocks - wave + NWV - 1) / NWV;     // this wave's: wave, wave + NWV, ...
  f32x4 w[2][NB][2], x[2][MB][2], nw[2][2];
  float scale = 1.f;
  auto load = [&](int buf, int i) {                // block i of this wave
    const size_t k = (size_t)(i * NWV + wave) * TK;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      if (NORM) nw[buf][h] = *(const f32x4*)(norm.w + k + h * 16 + lq * 4);
#pragma unroll
      for (int b = 0; b < NB; ++b) w[buf][b][h] = __builtin_nontemporal_load((const f32x4*)(wp[b] + k + h * 16));
#pragma unroll
      for (int a = 0; a < MB; ++a) x[buf][a][h] = *(const f32x4*)(ap[a] + k + h * 16);
    }
  };
  auto multiply = [&](int buf) {
    if (NORM)
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int e = 0; e < 4; ++e) x[buf][0][h][e] = x[buf][0][h][e] * scale * nw[buf][h][e];
#pragma unroll
    for (int a = 0; a < MB; ++a)
#pragma unroll
      for (int b = 0; b < NB; ++b)
        acc[a][b] += sum_of_products(x[buf][a][0], w[buf][b][0]) + sum_of_products(x[buf][a][1], w[buf][b][1]);
  };
  if (mine > 0) load(0, 0);
  if (NORM) {                                      // while the first weights are on their way
    const bool vec = K <= 256 * 4 * RMS_VEC_MAX;   // (rms_row_vec: A lies on 16 bytes)
    for (int m = wave; m < M; m += NWV) {
      const float s = row_scale(A + (size_t)m * K, K, vec, norm.eps, lane);
      if (lane == 0) scales[m] = s;
    }
    lds_barrier();
    scale = scales[min(l16, M - 1)];
  }
  if (mine > 0) {
    int i = 0;
    for (; i + 2 < mine; i += 2) {
      load(1, i + 1);
      multiply(0);
      load(0, i + 2);
      multiply(1);
    }
    if (i + 1 < mine) load(1, i + 1);
    multiply(0);
    if (i + 1 < mine) multiply(1);
  }
#pragma unroll
  for (int a = 0; a < MB; ++a)
#pragma unroll
    for (int b = 0; b < NB; ++b) sums[wave][a * NB + b][lane] = acc[a][b];
  __syncthreads();

  // lane (lq, l16) of a 16 x 16 holds rows 4 lq .. 4 lq + 3 of column l16
  constexpr int UNITS = gated(EPI) ? MB : MB * NB;
  for (int e = tid; e < UNITS * WAVE; e += NWV * WAVE) {
    const int at = e % WAVE, unit = e / WAVE, col = at % 16, row = 4 * (at / 16);
    auto total = [&](int t) {
      return ((sums[0][t][at] + sums[1][t][at]) + (sums[2][t][at] + sums[3][t][at])) +
             ((sums[4][t][at] + sums[5][t][at]) + (sums[6][t][at] + sums[7][t][at]));
    };
    if constexpr (gated(EPI)) {
      const f32x4 gt = total(unit * 2), up = total(unit * 2 + 1);
      const int hcol = blockIdx.x * 16 + col;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int m = unit * 16 + row + r;
        if (m < M && hcol < H) C[(size_t)m * H + hcol] = gate_value<EPI>(gt[r], up[r], H, gate_bias<EPI>(H, hcol));
      }
    } else if constexpr (EPI == EPI_QKV) {
      const f32x4 v = total(unit);
      const int n = n0 + unit * 16 + col, Q = out.n_heads * out.hd, KV = out.n_kv_heads * out.hd;
      const int region = n < Q ? 0 : n < Q + KV ? 1 : 2, within = n - (region == 0 ? 0 : region == 1 ? Q : Q + KV);
      const int head = within / out.hd, i = within % out.hd, pair = i >> 1;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int m = row + r;
        const float other = __shfl_xor(v[r], 1, WAVE);                       // the pair's other element, in the next lane
        if (m >= M || n >= N) continue;
        const int pos = out.tok_pos[m];
        float y = v[r];
        if (region < 2 && out.cos_sin != nullptr && pair < out.rotary_dim / 2 && pos >= 0 && pos < out.n_positions) {
          const float2 c = out.cos_sin[(size_t)pos * (out.rotary_dim / 2) + pair];
          y = rotate_one(v[r], other, (i & 1) != 0, c);
        }
        if (region == 0) {
          out.q_out[(size_t)m * Q + n] = y;
          continue;
        }
        const int slot = out.seq_slot[m];
        if (slot < 0 || pos < 0) continue;
        const int phys = out.block_table[(size_t)slot * out.table_stride + (pos / PAGE) % out.ring_pages];
        if (phys < 0 || phys >= out.n_pages) continue;
        const size_t base = ((size_t)phys * out.n_kv_heads + head) * PAGE * out.hd;
        if (region == 1) out.k_pages[base + page_k_offset(out.page_layout, pos & (PAGE - 1), i, out.hd)] = y;
        else out.v_pages[base + page_v_offset(out.page_layout, pos & (PAGE - 1), i, out.hd)] = y;
      }
    } else {
      const f32x4 v = total(unit);
      const int n = n0 + (unit % NB) * 16 + col;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int m = (unit / NB) * 16 + row + r;
        if (m >= M || n >= N) continue;
        const size_t o = (size_t)m * N + n;
        if (EPI == 2) C[o] += v[r];
        else C[o] = v[r];
      }
    }
  }
}

template <int EPI, int MB, int NB, bool NORM = false>
int launch_few(const float* A, const float* W, float* C, int M, int N, int K, GateOut H, hipStream_t stream, NormIn norm = {},
               QkvOut out = {}) {
  gemm_few_f32_kernel<EPI, MB, NB, NORM>
      <<<dim3(ceil_div(N, 16 * NB), ceil_div(M, 16 * MB)), NWV * WAVE, 0, stream>>>(A, W, C, M, N, K, H, norm, out);
  return launch_status();
}

template <int EPI, int FA, int FB, bool FINE>
int launch_f32(const float* A, const float* W, float* C, int M, int N, int K, GateOut H, hipStream_t stream) {
  const int tiles = ceil_div(M, 32 * FA) * ceil_div(N, 32 * FB), lds = stages_of(FA, FB) * 32 * (FA + FB) * ROWB;
  auto kernel = &gemm_f32_kernel<EPI, FA, FB, FINE>;
  if (lds > 64 * 1024) {
    static LdsAllowance allowed;
    if (int rc = allow_dynamic_lds(allowed, (const void*)kernel, lds); rc != YALM_OK) return rc;
  }
  kernel<<<8 * ceil_div(tiles, 8), 256, lds, stream>>>(A, W, C, M, N, K, H);
  return launch_status();
}

// Estimated time in us of one of the tile's kernel: f = FA FB products of 16 x 16 a wave.  Measured: a k tile takes 0.13 +
// 0.116 f us of a workgroup that has a CU to itself and 0.055 + 0.118 f of a CU's time where several share it (K 3,072 and
// 4,096: 4x4 249 us, 3x3 111, 2x4 102, 2x2 73, 2x1 45, 1x1 32 alone); a last round on a fraction of the CUs costs half a
// round and half its fraction.
double tile_time(int M, int N, int K, int fa, int fb) {
  const double f = fa * fb, per = (double)ceil_div(M, 32 * fa) * ceil_div(N, 32 * fb) / compute_units(), k = K / TK;
  if (per <= 1.0) return (0.13 + 0.116 * f) * k;
  const long whole = (long)per;
  const double rest = per - (double)whole;
  return (0.055 + 0.118 * f) * k * ((double)whole + (rest > 0.0 ? 0.5 + 0.5 * rest : 0.0));
}

struct Choice {
  enum Kernel { FEW, FINE, COARSE } kernel;
  int a, b;                                        // MB and NB, or FA and FB
};

// How many of the rows and weight rows a workgroup of gemm_few_f32_kernel takes (no sum depends on it).  Every 16 rows by
// themselves where that leaves no CU two workgroups (64 rows, 1,024 x 1,024 6.8 us; 2 and 4 times 16 8.9 and 13.1), else 32, and
// 64 of up to 4,096 columns (64 rows, 4,096 x 4,096 42 against 51 us with 32).  Two blocks of weight rows save reading A, which
// pays from 8 rows of many columns on (5,120 x 3,072: 4 rows 22.1 us with one, 22.8 with two, 16 rows 28.1 and 25.7).
Choice choose_few(int M, int N, bool gate) {
  const bool alone = M <= 16 || (long)ceil_div(N, gate ? 32 : 16) * ceil_div(M, 16) <= compute_units();
  if (gate) return {Choice::FEW, alone ? 1 : 2, 2};
  if (alone) return {Choice::FEW, 1, M > 7 && N > 4096 ? 2 : 1};
  if (N > 4096) return {Choice::FEW, 2, 2};
  return {Choice::FEW, M <= 32 ? 2 : 4, 1};
}

// The fastest tile by the estimate (701 rows, N x K: 16,384 x 3,072 takes 2x4 555 us, 128,256 x 3,072 2x4 4.0 ms, 3,072 x 8,192
// 3x3 288 us on exactly 256 tiles, 2x4 would be 24 % slower).  Up to 64 rows the small tiles' FINE form (2x4 would spill
// registers: 128,256 x 3,072 at 64 rows 446 against 459 us with 2x2, 16,384 x 3,072 114 against 66).
Choice choose_tile(int M, int N, int K, bool gate) {
  static constexpr int shapes[][2] = {{1, 1}, {1, 2}, {2, 1}, {2, 2}, {2, 4}, {3, 3}, {3, 4}, {4, 4}};
  const bool fine = M <= 64;
  int best = -1;
  double best_t = 0.0;
  for (int i = 0; i < (fine ? 4 : 8); ++i) {
    if (gate && shapes[i][1] % 2) continue;
    const double t = tile_time(M, N, K, shapes[i][0], shapes[i][1]);
    if (best < 0 || t < best_t) { best = i; best_t = t; }
  }
  return {fine ? Choice::FINE : Choice::COARSE, shapes[best][0], shapes[best][1]};
}

// Up to 64 rows the form of a sum follows from N and K alone, so that a row's results do not change with the number of rows
// beside it.  gemm_few_f32_kernel takes what is narrow (the tiles' kernel would leave CUs without work, and walks K alone where
// eight waves share it: 16 rows, 4,096 x 4,096 19 against 33 us, 3,072 x 8,192 34 against 60; 64 rows 42 and 81 against 33 and 61)
// and short sums, where the FINE chains would lie further from 64 bits than gemm_rows_f32_kernel's (a relative error at K 1,024 of
// 1.2e-7 against 1.0e-7, its own 0.9e-7; at K 2,560 1.26e-7 against 1.33e-7).  The rest goes to the tiles, which read A once for 32
// weight rows and more (16,384 x 3,072: one row 43 us, 16 rows 42, 64 rows 66; gemm_few_f32_kernel 45, 51 and 127).
Choice choose(int M, int N, int K, bool gate) {
  return M <= 64 && (N < 8192 || K <= 2048) ? choose_few(M, N, gate) : choose_tile(M, N, K, gate);
}

// The tile of gemm_split.hip that is sooner by the estimates than the tile chosen here, or -1 (5,120 x 3,072: 65 rows 41 us here, 47
// there; 128 rows 59 and 53; of 398 sizes that it takes there four are up to 5 % slower than here).  tile_time compares tiles with
// each other and leaves out a launch's start and end, some 5 us, and a tenth that broken rounds take longer (up to 40 % just above one
// round: 65 rows, 3,072 x 8,192 69 us for 98 measured).
int split_tile(int M, int N, int K, bool gate) {
  const Choice c = choose(M, N, K, gate);
  return c.kernel == Choice::COARSE ? yalm_gemm_split_choose(M, N, K, gate, 5.0 + 1.1 * tile_time(M, N, K, c.a, c.b)) : -1;
}

// A norm is folded into the products of gemm_few_f32_kernel of up to 16 rows
bool takes_norm(int M, int N, int K, bool gate) {
  return M >= 1 && M <= 16 && N > 0 && K > 0 && K % TK == 0 && choose(M, N, K, gate).kernel == Choice::FEW;
}
// Whether a step is sooner with it than with the norm's kernel in front (and the rotation's behind, `qkv`): every workgroup forms the
// rows' sums of squares anew, which pays while there are at most two of them a CU, one in the wide form, and without the rotation's launch
// while a wave takes a row at once (K to 1,024).  us folded and apart, one row and 16: 4,096 x 1,024 8.4 and 10.7, 11.3 and 12.2; 8,192
// x 1,024 12.7 and 13.9, 15.3 and 16.0; gated 12.9 and 14.4, 15.6 and 16.3.  More weight rows: 10,240 x 512 11.0 and 9.9, gated 13.2 and
// 11.4; 128,256 x 2,048 246 and 191, 287 and 237.  Longer rows: 4,096 x 1,056 8.1 and 8.1, 11.4 and 10.1; 2,048 x 2,048 10.5 and
// 10.1, 15.2 and 13.0.  q/k/v: 6,144 x 1,024 12.6 and 16.3, 17.3 and 18.8; 6,144 x 4,096 33.1 and 35.2, 39.2 and 38.5 (a step of four
// 7B layers 955 and 974, 1,137 and 1,152); 12,288 x 2,048 32.8 and 29.0, 44.7 and 38.6.
bool norm_pays(int M, int N, int K, bool gate, bool qkv) {
  return takes_norm(M, N, K, gate) && N <= 32L * compute_units() && (qkv || K <= 1024);
}
template <int EPI>
int launch_norm(const float* x, const float* W, float* C, int M, int N, int K, GateOut H, NormIn norm, QkvOut out, hipStream_t stream) {
  if constexpr (gated(EPI)) return launch_few<EPI, 1, 2, true>(x, W, C, M, N, K, H, stream, norm, out);
  else if (choose(M, N, K, false).b == 2) return launch_few<EPI, 1, 2, true>(x, W, C, M, N, K, H, stream, norm, out);
  else return launch_few<EPI, 1, 1, true>(x, W, C, M, N, K, H, stream, norm, out);
}

template <int EPI>
int launch(const float* A, const float* W, float* C, int M, int N, int K, GateOut H, hipStream_t stream) {
  const Choice c = choose(M, N, K, gated(EPI));
#define YALM_TAKE(KERNEL_, A_, B_, CALL_) \
  if (c.kernel == Choice::KERNEL_ && c.a == A_ && c.b == B_) return CALL_(A, W, C, M, N, K, H, stream)
  YALM_TAKE(FEW, 1, 2, (launch_few<EPI, 1, 2>));
  YALM_TAKE(FEW, 2, 2, (launch_few<EPI, 2, 2>));
  YALM_TAKE(FINE, 1, 2, (launch_f32<EPI, 1, 2, true>));
  YALM_TAKE(FINE, 2, 2, (launch_f32<EPI, 2, 2, true>));
  YALM_TAKE(COARSE, 1, 2, (launch_f32<EPI, 1, 2, false>));
  YALM_TAKE(COARSE, 2, 2, (launch_f32<EPI, 2, 2, false>));
  YALM_TAKE(COARSE, 2, 4, (launch_f32<EPI, 2, 4, false>));
  YALM_TAKE(COARSE, 3, 4, (launch_f32<EPI, 3, 4, false>));
  YALM_TAKE(COARSE, 4, 4, (launch_f32<EPI, 4, 4, false>));
  if constexpr (!gated(EPI)) {                     // an odd number of column tiles
    YALM_TAKE(FEW, 1, 1, (launch_few<EPI, 1, 1>));
    YALM_TAKE(FEW, 2, 1, (launch_few<EPI, 2, 1>));
    YALM_TAKE(FEW, 4, 1, (launch_few<EPI, 4, 1>));
    YALM_TAKE(FINE, 1, 1, (launch_f32<EPI, 1, 1, true>));
    YALM_TAKE(FINE, 2, 1, (launch_f32<EPI, 2, 1, true>));
    YALM_TAKE(COARSE, 1, 1, (launch_f32<EPI, 1, 1, false>));
    YALM_TAKE(COARSE, 2, 1, (launch_f32<EPI, 2, 1, false>));
    YALM_TAKE(COARSE, 3, 3, (launch_f32<EPI, 3, 3, false>));
  }
#undef YALM_TAKE
  return YALM_ERR_ARG;
}

}  // namespace

// Which tile of gemm_split.hip a product takes, or -1: it stays here
extern "C" int yalm_gemm_f32_split_choice(int M, int N, int K, int gate) {
  if (M <= 0 || N <= 0 || K <= 0 || K % TK != 0) return -1;
  return split_tile(M, N, K, gate != 0);
}

// Which kernel and tile of this file a product takes (that gemm_split.hip does not): 100 kernel (0 gemm_few_f32_kernel, 1 FINE tiles,
// 2 tiles) + 10 a + b
extern "C" int yalm_gemm_f32_choice(int M, int N, int K, int gate) {
  if (M <= 0 || N <= 0 || K <= 0 || K % TK != 0) return -1;
  const Choice c = choose(M, N, K, gate != 0);
  return 100 * c.kernel + 10 * c.a + c.b;
}

// Whether yalm_gemm_norm_f32 (and the q/k/v form) takes the product
extern "C" int yalm_gemm_norm_f32_takes(int M, int N, int K, int gate) { return takes_norm(M, N, K, gate != 0); }

// Whether it is sooner than the kernels one by one; what: 0 a plain product, 1 a gated one, 2 q/k/v
extern "C" int yalm_gemm_norm_f32_pays(int M, int N, int K, int what) { return norm_pays(M, N, K, what == 1, what == 2); }

static bool norm_operands_ok(const float* x, const float* norm_w, const float* W) {
  return x != nullptr && norm_w != nullptr && W != nullptr && !((uintptr_t)x & 15) && !((uintptr_t)norm_w & 15) && !((uintptr_t)W & 15);
}

// yalm_gemm_norm with float32 weights and results: C = epilogue(rmsnorm(x, norm_w, eps) W^T), epilogue 0 or a gated one
extern "C" int yalm_gemm_norm_f32(const float* x, const float* norm_w, float eps, const float* W, float* C, int M, int N, int K, int epilogue,
                                  int hidden, hipStream_t stream) {
  if (!takes_norm(M, N, K, gated(epilogue)) || !norm_operands_ok(x, norm_w, W) || C == nullptr) return YALM_ERR_ARG;
  const GateOut H(hidden);
  const NormIn norm = {norm_w, eps};
  if (gated(epilogue) && (hidden <= 0 || N != 32 * ((hidden + 15) / 16))) return YALM_ERR_ARG;
  switch (epilogue) {
    case 0: return launch_norm<0>(x, W, C, M, N, K, H, norm, QkvOut{}, stream);
    case 3: return launch_norm<3>(x, W, C, M, N, K, H, norm, QkvOut{}, stream);
    case 5: return launch_norm<5>(x, W, C, M, N, K, H, norm, QkvOut{}, stream);
  }
  return YALM_ERR_ARG;
}

// yalm_gemm_norm_qkv_rope with everything in float32
extern "C" int yalm_gemm_norm_qkv_rope_f32(const float* x, const float* norm_w, float eps, const float* Wqkv, float* q_out, float* k_pages,
                                           float* v_pages, const int* block_table, int table_stride, int ring_pages, const int* tok_pos,
                                           const int* seq_slot, const float* cos_sin, int n_positions, int M, int K, int n_heads,
                                           int n_kv_heads, int head_dim, int rotary_dim, int n_pages, int page_layout, hipStream_t stream) {
  const int N = (n_heads + 2 * n_kv_heads) * head_dim;
  if (head_dim <= 0 || head_dim % 16 != 0 || rotary_dim < 0 || (rotary_dim & 1) || rotary_dim > head_dim || n_heads <= 0 || n_kv_heads <= 0 ||
      ring_pages <= 0 || n_pages <= 0 || !page_layout_ok(page_layout, head_dim) || block_table == nullptr || tok_pos == nullptr ||
      seq_slot == nullptr || q_out == nullptr || k_pages == nullptr || v_pages == nullptr)
    return YALM_ERR_ARG;
  if (!takes_norm(M, N, K, false) || !norm_operands_ok(x, norm_w, Wqkv)) return YALM_ERR_ARG;
  const QkvOut out = {q_out, k_pages, v_pages, block_table, tok_pos, seq_slot, (const float2*)cos_sin, table_stride, ring_pages, n_positions,
                      n_heads, n_kv_heads, head_dim, rotary_dim, n_pages, page_layout};
  return launch_norm<EPI_QKV>(x, Wqkv, nullptr, M, N, K, GateOut(0), NormIn{norm_w, eps}, out, stream);
}

// K a multiple of 32 and 16-byte aligned operands; YALM_ERR_ARG: not taken.
int yalm_gemm_f32_mfma(const void* A, const void* W, void* C, int M, int N, int K, int epilogue, GateOut H, hipStream_t stream) {
  if (M <= 0 || N <= 0 || K <= 0 || K % TK != 0 || ((uintptr_t)A & 15) || ((uintptr_t)W & 15)) return YALM_ERR_ARG;
  const float *a = (const float*)A, *w = (const float*)W;
  float* c = (float*)C;
  if (const int tile = split_tile(M, N, K, gated(epilogue)); tile >= 0) return yalm_gemm_split(tile, a, w, c, M, N, K, epilogue, H, stream);
  switch (epilogue) {
    case 0:
    case 1: return launch<0>(a, w, c, M, N, K, H, stream);
    case 2: return launch<2>(a, w, c, M, N, K, H, stream);
    case 3: return launch<3>(a, w, c, M, N, K, H, stream);
    case 5: return launch<5>(a, w, c, M, N, K, H, stream);
    case 6: return launch<6>(a, w, c, M, N, K, H, stream);
  }
  return YALM_ERR_ARG;
}
