// C = epilogue(A[M,K] * W[N,K]^T) in float32, more than 64 rows, on the matrix cores' bfloat16 products: a float is the sum
// of three bfloat16 numbers (8 + 8 + 8 significant bits), and of the nine products of two such sums the six largest are made and
// added in float32, the smallest first (the way of Henry, Tang and Heinecke, "Leveraging the bfloat16 artificial intelligence
// datatype for higher-precision computations", 2019).  The three left out are below 2^-25 of the product, under the rounding of one
// addition.  v_mfma_f32_16x16x32_bf16 takes 32 products in the time in which v_mfma_f32_16x16x4_f32 takes 2, so six of them still
// leave a factor of 2.7 over gemm_f32.hip's tiles.
//
// A bfloat16 number has float32's exponents, so the last terms of a float below 2^-108 would fall off their end (an operand of 2^-120
// kept 14 bits).  Both operands are therefore split at 2^24 times their size, where every float, a subnormal one too, is the sum of its
// terms exactly (no bit of a float is below 2^-149, none there below 2^-125), and a fold's sums come back by 2^-48 as they join the
// total.  What that leaves no room for (an operand from about 2^104 on, a fold's sum from 2^80 on) comes out as no finite number, and
// is made again with float32 products like an infinity (a product of nothing else: 366 us where gemm_f32_kernel takes 117).
//
// The error against 64 bits is smaller than gemm_f32_kernel's, whose sums are chains of four products at a time: relative, K 512
// 1.6e-7 (2.9e-7), 3,072 1.7 to 1.8e-7 (2.95e-7), 8,192 1.9 to 2.1e-7 (3.05e-7), 14,336 2.1 to 2.5e-7 (3.2e-7).  The instruction drops the
// bits that it shifts out of a sum's addends towards minus infinity: all results of a product would lie low by 2e-8 (K 512) to 1.2e-7
// (K 14,336) of their size, and what every number of a stream is off by alike does not average out in the layers behind it
// (probabilities of a scored text 5.5e-7 off, with gemm_f32_kernel 4.6e-7).  So every second fold of k tiles is summed with A's signs
// turned and subtracted: the means are 1e-10 of a size then.  Operands of one sign, of exponents spread over 2^+-24 and with a few numbers a
// thousand times the others are no further off than there either; rows of one number that is not zero are (3.5e-8, 4.3e-8 here), and
// rows of eight (5.1 to 6.1e-8, 6.2 to 7.0e-8), whose sums have hardly any rounding but the products' own.
//
// A row's sums hang on how many rows stand beside it, by which tile they choose: gemm_f32_kernel's, one of one group of waves and
// one of two add in three orders.
//
// Bound by the power that the matrix cores may draw (full rounds of 128 x 256: 1.45 PFLOP/s of bfloat16 products) and by
// rounds of tiles that do not come out even.  Every element is split once a workgroup, on its way from registers into LDS
// (the next k tile's, a vector instruction or two behind every matrix product): split by each wave that multiplies it, straight
// from fragments of float32, the vector instructions take as long as the products (701 rows, 16,384 x 3,072 415 us against 365).
// 701 rows against gemm_f32_kernel, us: 16,384 x 3,072 573 -> 372, 128,256 x 3,072 4,130 -> 2,753, 5,120 x 3,072 195 -> 137, 3,072 x 8,192
// 304 -> 222, 3,072 x 3,072 117 -> 85 (1 to 2 % of it the scale of W's elements).
#include "common.h"
#include "gemm_split.h"

namespace {

typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(2))) float f32x2;
typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;
typedef __attribute__((ext_vector_type(4))) unsigned u32x4;

constexpr int TK = 32;                           // k a tile
constexpr int ROWB = TK * 2;                     // bytes of a row in one of the three planes of terms
constexpr int TERMS = 3;
constexpr int GROUP = 4;                         // tile columns that an XCD walks together
constexpr int FOLD = 4;                          // k tiles whose sums join before they are added to the total (8: the errors 1.4 times these, 2 % sooner)

constexpr float UP = 0x1p24f, DOWN = 0x1p-48f;   // the operands' scale on the way into terms, and the sums' on the way back

struct Terms { u32x4 t[TERMS]; };

// Four floats into dwords 2 h and 2 h + 1 of each term: each rounded to bfloat16, the rest to the next term (differences exact)
__device__ __forceinline__ void split4(Terms& out, int h, f32x4 v) {
  float x[4] = {v[0], v[1], v[2], v[3]};
#pragma unroll
  for (int p = 0; p < TERMS; ++p)
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      const unsigned w = __builtin_bit_cast(unsigned, __builtin_convertvector((f32x2){x[2 * e], x[2 * e + 1]}, bf16x2));
      out.t[p][2 * h + e] = w;
      if (p + 1 < TERMS) {
        x[2 * e] -= __uint_as_float(w << 16);
        x[2 * e + 1] -= __uint_as_float(w & 0xffff0000u);
      }
    }
}

// WM x WN waves of FA x FB products of 16 x 16 make a tile; KG groups of such waves take its k tiles in turn (two groups
// where a tile has only four waves: a SIMD needs a second wave to have products to make while the first one waits).
// A k tile lies in LDS as three planes of terms, rows of 64 bytes whose 16-byte chunks are XOR-swizzled by the row (eight rows'
// reads fall on different banks), twice: one is multiplied while the next one is split into the other.  VPM: vector
// instructions that the schedule puts behind each matrix product.
template <int EPI, int FA, int FB, int WM, int WN, int KG, int VPM>
__global__ __launch_bounds__(WM * WN * KG * WAVE, 2) void gemm_split_kernel(const float* __restrict__ A, const float* __restrict__ W,
                                                                           float* __restrict__ C, int M, int N, int K, GateOut H) {
  constexpr int NW = WM * WN, NT = NW * WAVE;
  constexpr int TM = 16 * FA * WM, TN = 16 * FB * WN, ROWS = TM + TN, PLANE = ROWS * ROWB, BUF = TERMS * PLANE;
  constexpr int U = (ROWS * 4 + NT - 1) / NT;     // shares of 8 k of a row that a thread splits
  static_assert(ROWS * 4 % WAVE == 0 && NW * KG == 8 && (KG == 1 || KG == 2), "whole waves' shares; two waves a SIMD");
  static_assert(!gated(EPI) || FB % 2 == 0, "the gated epilogue pairs column tiles");
  extern __shared__ __attribute__((aligned(1024))) unsigned char lds[];          // [KG][2][BUF]
  const int grp = KG == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x / NT);
  const int tid = threadIdx.x - grp * NT, lane = tid % WAVE;
  const int wave = __builtin_amdgcn_readfirstlane(tid / WAVE);
  const int wm = wave / WN, wn = wave % WN;
  const int l16 = lane % 16, lq = lane / 16;
  unsigned char* bufs = lds + grp * 2 * BUF;
  // Workgroup i runs on XCD i mod 8: every XCD takes a run of the tiles (groups of GROUP columns, in a group the columns
  // fastest), so that the tiles it works on at a time share rows and columns in its second-level cache.
  const int mt = (M + TM - 1) / TM, nt = (N + TN - 1) / TN, tiles = mt * nt, chunk = (tiles + 7) / 8;
  const int i0 = blockIdx.x, t = (i0 % 8) * chunk + i0 / 8;
  if (t >= tiles || i0 / 8 >= chunk) return;
  const int per_group = mt * GROUP, g = t / per_group, r0 = t % per_group, width = min(GROUP, nt - g * GROUP);
  const int m0 = (r0 / width) * TM, n0 = (g * GROUP + r0 % width) * TN;

  const float* from[U];
  int to[U];
#pragma unroll
  for (int i = 0; i < U; ++i) {
    const int u = min(tid + i * NT, ROWS * 4 - 1), row = u / 4, c = u % 4;
    from[i] = (row < TM ? A + (size_t)min(m0 + row, M - 1) * K                    // rows past the edge repeat the last
                        : W + (size_t)min(n0 + row - TM, N - 1) * K) + c * 8;     // one and are never stored
    to[i] = row * ROWB + ((c ^ ((row >> 2) & 3)) << 4);
  }
  f32x4 raw[U][2];
  auto load = [&](int kt) {
#pragma unroll
    for (int i = 0; i < U; ++i)
#pragma unroll
      for (int h = 0; h < 2; ++h) raw[i][h] = *reinterpret_cast<const f32x4*>(from[i] + (size_t)kt * TK + h * 4);
  };
  float a_scale = UP;                              // A's scale in the tile that is stored, with the sign that it takes there
  auto store = [&](int buf, int i) {
    if ((i + 1) * NT > ROWS * 4 && (wave + i * NW) * WAVE >= ROWS * 4) return;    // a last share that only some waves have
    // rows of A or of W (whole waves')
    const float by = i * NT < TM * 4 && ((i + 1) * NT <= TM * 4 || (wave + i * NW) * WAVE < TM * 4) ? a_scale : UP;
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int e = 0; e < 4; ++e) raw[i][h][e] *= by;
    Terms s;
    split4(s, 0, raw[i][0]);
    split4(s, 1, raw[i][1]);
#pragma unroll
    for (int p = 0; p < TERMS; ++p) *reinterpret_cast<u32x4*>(bufs + buf * BUF + p * PLANE + to[i]) = s.t[p];
  };

  f32x4 acc[FA][FB], total[FA][FB];
#pragma unroll
  for (int a = 0; a < FA; ++a)
#pragma unroll
    for (int b = 0; b < FB; ++b) total[a][b] = acc[a][b] = (f32x4){0.f, 0.f, 0.f, 0.f};
  const int a_row = wm * 16 * FA + l16, w_row = TM + wn * 16 * FB + l16;
  const int a_at = a_row * ROWB + ((lq ^ ((a_row >> 2) & 3)) << 4), w_at = w_row * ROWB + ((lq ^ ((w_row >> 2) & 3)) << 4);
  bf16x8 pa[FA][TERMS], pw[TERMS];
  auto read_w = [&](int buf, bf16x8 (&v)[TERMS], int b) {
#pragma unroll
    for (int p = 0; p < TERMS; ++p) v[p] = *reinterpret_cast<const bf16x8*>(bufs + buf * BUF + p * PLANE + w_at + b * 16 * ROWB);
  };
  auto read_a = [&](int buf, int a) {
#pragma unroll
    for (int p = 0; p < TERMS; ++p) pa[a][p] = *reinterpret_cast<const bf16x8*>(bufs + buf * BUF + p * PLANE + a_at + a * 16 * ROWB);
  };
  constexpr int a_term[6] = {2, 0, 1, 1, 0, 0}, w_term[6] = {0, 2, 1, 0, 1, 0};   // the smallest products first

  const int nk = K / TK, mine = (nk - grp + KG - 1) / KG, most = (nk + KG - 1) / KG;     // this group's k tiles: grp, grp + KG, ...
  auto tile_of = [&](int i) { return min(grp + i * KG, nk - 1); };               // (behind the last one: read again, not used)
  auto turned = [&](int i) { return ((i / FOLD + grp) & 1) != 0; };               // whether tile i's fold takes A with its signs turned
  load(tile_of(0));
  a_scale = turned(0) ? -UP : UP;
#pragma unroll
  for (int i = 0; i < U; ++i) store(0, i);
  load(tile_of(1));
  lds_barrier();
  read_w(0, pw, 0);
#pragma unroll
  for (int a = 0; a < FA; ++a) read_a(0, a);
  // Tile i is multiplied column by column out of buffer `buf` while tile i + 1 goes from registers into the other one.
  // The barrier stands in front of the last column's products: by then nobody reads `buf` any more, the next tile is whole, and
  // its first fragments are read among these products.
  auto one_tile = [&](int i, int buf) {
    a_scale = turned(i + 1) ? -UP : UP;
#pragma unroll
    for (int b = 0; b < FB - 1; ++b) {
      bf16x8 next[TERMS];
      read_w(buf, next, b + 1);
#pragma unroll
      for (int c = 0; c < 6; ++c)
#pragma unroll
        for (int a = 0; a < FA; ++a)
          acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(pa[a][a_term[c]], pw[w_term[c]], acc[a][b], 0, 0, 0);
#pragma unroll
      for (int u = b * U / (FB - 1); u < (b + 1) * U / (FB - 1); ++u) store(buf ^ 1, u);
#pragma unroll
      for (int p = 0; p < TERMS; ++p) pw[p] = next[p];
#pragma unroll
      for (int j = 0; j < FA * 6; ++j) {
        __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x2, VPM, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    load(tile_of(i + 2));
    lds_barrier();
    bf16x8 next[TERMS];
    read_w(buf ^ 1, next, 0);
#pragma unroll
    for (int a0 = 0; a0 < FA; a0 += 2) {
#pragma unroll
      for (int c = 0; c < 6; ++c)
#pragma unroll
        for (int a = a0; a < (a0 + 2 < FA ? a0 + 2 : FA); ++a)
          acc[a][FB - 1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(pa[a][a_term[c]], pw[w_term[c]], acc[a][FB - 1], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int a = a0; a < (a0 + 2 < FA ? a0 + 2 : FA); ++a) read_a(buf ^ 1, a);
    }
#pragma unroll
    for (int p = 0; p < TERMS; ++p) pw[p] = next[p];
  };
  for (int k0 = 0; k0 < mine; k0 += FOLD) {
    const int k1 = min(k0 + FOLD, mine);
    for (int i = k0; i < k1; ++i) one_tile(i, i & 1);
    const float back = turned(k0) ? -DOWN : DOWN;
#pragma unroll
    for (int a = 0; a < FA; ++a)
#pragma unroll
      for (int b = 0; b < FB; ++b) {
        asm volatile("" : "+v"(acc[a][b]));        // added here, not in every turn of the loop
#pragma unroll
        for (int r = 0; r < 4; ++r) total[a][b][r] = fmaf(acc[a][b][r], back, total[a][b][r]);
        acc[a][b] = (f32x4){0.f, 0.f, 0.f, 0.f};
      }
  }
  if constexpr (KG == 2) {                         // the groups' sums meet in LDS
    static_assert(FA * FB * NT * 16 <= 2 * KG * BUF, "the second group's sums fit where the tiles were");
    if (mine < most) lds_barrier();                // one for each tile of the group that has more
    lds_barrier();                                 // the fragments read ahead are there
    f32x4* other = reinterpret_cast<f32x4*>(lds);
    if (grp == 1)
#pragma unroll
      for (int a = 0; a < FA; ++a)
#pragma unroll
        for (int b = 0; b < FB; ++b) other[(a * FB + b) * NT + tid] = total[a][b];
    lds_barrier();
    if (grp == 1) return;
#pragma unroll
    for (int a = 0; a < FA; ++a)
#pragma unroll
      for (int b = 0; b < FB; ++b) total[a][b] += other[(a * FB + b) * NT + tid];
  }

  // An infinity, a NaN, or a number that is infinite at 2^24 times its size makes every sum that it enters a NaN (infinity less
  // infinity in its terms), and a fold's sum that has no room is infinite.  Sums that are no finite numbers are made again with float32
  // products, chains as in gemm_f32_kernel, 16 rows at a time; the sums beside them stay as they are.
  auto finite = [](float v) { return (__float_as_uint(v) & 0x7f800000u) != 0x7f800000u; };
#pragma unroll
  for (int a = 0; a < FA; ++a) {
    bool all = true;
#pragma unroll
    for (int b = 0; b < FB; ++b)
#pragma unroll
      for (int r = 0; r < 4; ++r) all &= finite(total[a][b][r]);
    if (__all(all)) continue;
    const float *ra = A + (size_t)min(m0 + (wm * FA + a) * 16 + l16, M - 1) * K + lq * 4, *rw[FB];
    f32x4 again[FB], fold[FB];
#pragma unroll
    for (int b = 0; b < FB; ++b) {
      rw[b] = W + (size_t)min(n0 + (wn * FB + b) * 16 + l16, N - 1) * K + lq * 4;
      again[b] = fold[b] = (f32x4){0.f, 0.f, 0.f, 0.f};
    }
    for (int k = 0; k < K; k += 16) {
      const f32x4 va = *reinterpret_cast<const f32x4*>(ra + k);
      f32x4 vw[FB];
#pragma unroll
      for (int b = 0; b < FB; ++b) vw[b] = *reinterpret_cast<const f32x4*>(rw[b] + k);
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int b = 0; b < FB; ++b) fold[b] = __builtin_amdgcn_mfma_f32_16x16x4f32(va[e], vw[b][e], fold[b], 0, 0, 0);
      if ((k + 16) % (FOLD * TK) == 0 || k + 16 == K)
#pragma unroll
        for (int b = 0; b < FB; ++b) {
          again[b] += fold[b];
          fold[b] = (f32x4){0.f, 0.f, 0.f, 0.f};
        }
    }
#pragma unroll
    for (int b = 0; b < FB; ++b)
#pragma unroll
      for (int r = 0; r < 4; ++r) total[a][b][r] = finite(total[a][b][r]) ? total[a][b][r] : again[b][r];
  }

  // lane (lq, l16) holds rows 4 lq .. 4 lq + 3 of column l16 of every 16 x 16
#pragma unroll
  for (int a = 0; a < FA; ++a)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int m = m0 + (wm * FA + a) * 16 + 4 * lq + r;
      if (m >= M) continue;
      if (gated(EPI)) {                              // weight rows: 16 gate rows, 16 up rows, ...: even tiles gate, odd tiles up
#pragma unroll
        for (int p = 0; p < FB / 2; ++p) {
          const int hcol = (n0 + wn * 16 * FB) / 2 + p * 16 + l16;
          if (hcol < H) C[(size_t)m * H + hcol] = gate_value<EPI>(total[a][2 * p][r], total[a][2 * p + 1][r], H, gate_bias<EPI>(H, hcol));
        }
      } else {
#pragma unroll
        for (int b = 0; b < FB; ++b) {
          const int n = n0 + (wn * FB + b) * 16 + l16;
          if (n >= N) continue;
          const size_t o = (size_t)m * N + n;
          if (EPI == 2) C[o] += total[a][b][r];
          else C[o] = total[a][b][r];
        }
      }
    }
}

template <int EPI, int FA, int FB, int WM, int WN, int KG, int VPM>
int launch_split(const float* A, const float* W, float* C, int M, int N, int K, GateOut H, hipStream_t stream) {
  constexpr int TM = 16 * FA * WM, TN = 16 * FB * WN, bytes = KG * 2 * TERMS * (TM + TN) * ROWB;
  static_assert(bytes <= 160 * 1024, "the LDS of a CU");
  const int tiles = ceil_div(M, TM) * ceil_div(N, TN);
  auto kernel = &gemm_split_kernel<EPI, FA, FB, WM, WN, KG, VPM>;
  static LdsAllowance allowed;
  if (int rc = allow_dynamic_lds(allowed, (const void*)kernel, bytes); rc != YALM_OK) return rc;
  kernel<<<8 * ceil_div(tiles, 8), WM * WN * KG * WAVE, bytes, stream>>>(A, W, C, M, N, K, H);
  return launch_status();
}

// The tiles, and us a k tile of a workgroup that few others run beside (the slope between K 3,072 and 8,192 of one round on
// part of the chip).
struct Tile { int rows, cols; double us; };
constexpr Tile tiles_of[] = {{64, 64, 0.43}, {64, 128, 0.63}, {96, 96, 0.72}, {128, 128, 1.12}, {192, 128, 1.59}, {128, 256, 1.74}};
constexpr int N_TILES = sizeof(tiles_of) / sizeof(Tile);

// Estimated us of a product: rounds of a workgroup a CU.  A full chip draws so much power that a round takes 18 % longer (128 x
// 256 2.1 us a k tile); 5 us of start and end.  700 rows, 6,144 x 4,096 with 96 x 96: 221 (measured 208 to 218); 300 rows, 28,672 x
// 4,096 with 192 x 128, 128 x 256, 128 x 128: 476, 503, 501 (448, 495, 485).
double split_time(const Tile& t, int M, int N, int K) {
  const double per = (double)ceil_div(M, t.rows) * ceil_div(N, t.cols) / compute_units();
  const double whole = (double)(long)per, rest = per - whole;
  return 5.0 + t.us * (K / TK) * (whole * 1.18 + (rest > 0.0 ? 1.0 + 0.18 * rest : 0.0));
}

template <int EPI>
int launch(int tile, const float* A, const float* W, float* C, int M, int N, int K, GateOut H, hipStream_t stream) {
  switch (tile) {
    case 0: return launch_split<EPI, 2, 2, 2, 2, 2, 3>(A, W, C, M, N, K, H, stream);
    case 1: return launch_split<EPI, 2, 4, 2, 2, 2, 3>(A, W, C, M, N, K, H, stream);
    case 2:
      if constexpr (!gated(EPI)) return launch_split<EPI, 3, 3, 2, 2, 2, 3>(A, W, C, M, N, K, H, stream);
      break;
    case 3: return launch_split<EPI, 2, 4, 4, 2, 1, 3>(A, W, C, M, N, K, H, stream);
    case 4: return launch_split<EPI, 3, 4, 4, 2, 1, 4>(A, W, C, M, N, K, H, stream);
    case 5: return launch_split<EPI, 4, 4, 2, 4, 1, 3>(A, W, C, M, N, K, H, stream);
  }
  return YALM_ERR_ARG;
}

}  // namespace

int yalm_gemm_split_choose(int M, int N, int K, bool gate, double than) {
  // Up to 64 rows a row's results do not hang on the rows beside it: gemm_f32.hip's kernels keep them.  Short sums stay with
  // its tiles too: a product of few k tiles is its start and its end (700 rows, 3,072 x 128: 9.6 against 10.1 us).
  if (M <= 64 || K < 512 || K % TK != 0) return -1;
  int best = -1;
  for (int i = 0; i < N_TILES; ++i) {
    if (gate && i == 2) continue;
    const double t = split_time(tiles_of[i], M, N, K);
    if (t < than) {
      best = i;
      than = t;
    }
  }
  return best;
}

int yalm_gemm_split(int tile, const float* A, const float* W, float* C, int M, int N, int K, int epilogue, GateOut H, hipStream_t stream) {
  switch (epilogue) {
    case 0:
    case 1: return launch<0>(tile, A, W, C, M, N, K, H, stream);
    case 2: return launch<2>(tile, A, W, C, M, N, K, H, stream);
    case 3: return launch<3>(tile, A, W, C, M, N, K, H, stream);
    case 5: return launch<5>(tile, A, W, C, M, N, K, H, stream);
    case 6: return launch<6>(tile, A, W, C, M, N, K, H, stream);
  }
  return YALM_ERR_ARG;
}
