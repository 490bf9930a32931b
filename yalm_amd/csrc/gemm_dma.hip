// GEMMs of more than 64 rows whose k tiles go from global memory straight into LDS:
// C = epilogue(A[M,K] * W[N,K]^T), bfloat16 operands, float32 accumulation.
//
// A workgroup owns a tile of C.  Its waves issue global_load_lds_dwordx4 (16 bytes a lane, a
// wave's 64 lanes land as 1 KB contiguous in LDS) for later k tiles while they multiply the
// current one; no register or LDS write instruction stands between memory and the matrix
// cores.  Rows are kept unpadded (128 bytes for 64 k) and the 16-byte chunks of a row are
// XOR-swizzled by the row number, which every lane applies to the GLOBAL address it asks
// for, so that the b128 fragment reads of 16 consecutive rows fall on different banks.  The
// compiler does not know that these loads write LDS: the kernels wait for them themselves
// (s_waitcnt vmcnt) and use the bare s_barrier, because __syncthreads() carries a fence that
// would wait for the loads of all stages.
//
// gemm_stages_kernel (256, 192, 128 or 64 rows x 128 columns, whole k tiles of both operands as stages, three to six of them) serves
// the short and middle prompts and what whole rounds of large tiles leave; gemm_ring16_kernel (256 x 256 and 256 x 192, five slots in
// turn) the long ones.  With few tiles K is split over the grid as well: every slice writes its float32 partial product, and
// yalm_splitk_reduce (or the consumer) adds them in order and applies the epilogue.  tile_plan says which.
//
// Takes any M and N and K % 64 == 0; other shapes are refused (YALM_ERR_ARG) and the
// caller runs the kernel of gemm_mfma.hip.  Sums are in a fixed order for a given shape.
#include "common.h"
#include "yalm_hip.h"
#include <type_traits>

int yalm_splitk_reduce(const float* partial, void* C, int M, int N, GateOut H, int slices, int epilogue,
                       hipStream_t stream);                                  // gemm_batch.hip

namespace {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) float f32x4;

constexpr int TK = 64;
constexpr int ROWB = TK * 2;                     // bytes a row of a stage
constexpr int CPR = ROWB / 16;                   // 16-byte chunks a row
constexpr int RPI = WAVE / CPR;                  // rows one wave instruction brings

__device__ __forceinline__ int swizzle_of(int row) { return (row >> 1) & (CPR - 1); }

template <int N_>
__device__ __forceinline__ void wait_vmcnt() {   // vmcnt only: expcnt and lgkmcnt fields at their maxima
  __builtin_amdgcn_s_waitcnt((N_ & 0xF) | ((N_ >> 4) << 14) | (0x7 << 4) | (0xF << 8));
}

// ---------------------------------------------------------------------------
// The kernel for many tiles: 256 x TN tiles, 8 waves, and a ring of five 32 KB slots that holds the k tiles of
// W and of A in turn (W0 A0 W1 A1 W2 ...; tile t has W in slot 2t mod 5 and A in slot (2t + 1) mod 5), so that
// two and a half k tiles are in flight or in use.  What it does beside a plain double buffer, each measured:
//  * a vector memory instruction holds its wave for tens of clocks, more while the memory system is busy; issued
//    as a burst behind the barrier they stall every wave at once and the matrix cores idle.  Here a wave issues
//    one DMA instruction in every few products, all through the iteration, and each has a k step or more to land;
//  * the barrier stands in front of a tile's last products: their fragments are in registers by
//    then, so nobody reads the tile's slots any more and they are refilled at once, and the first fragments
//    of the next tile are read while the last products of this one run;
//  * the fragments of a k step are read during the products of the one before (two register sets);
//  * the DMA takes its base from scalar registers and a 32-bit offset a lane (inline asm: the compiler would
//    add a 64-bit pair a lane for every instruction).
// The order of statements in the loop is the order of the instructions: a scheduling fence follows each.
// ---------------------------------------------------------------------------
constexpr int RING_SLOT = 32768, RING_SLOTS = 5, RING_TM = 256;

__device__ __forceinline__ void wait_lgkmcnt0() { __builtin_amdgcn_s_waitcnt(0x3F | (0x7 << 4) | (0x0 << 8) | (0x3 << 14)); }

// the product index of a k step (of n_products) behind which DMA instruction d of n_dma is issued
// (evenly spread: 2 of 8 go behind products 1 and 4)
__host__ __device__ constexpr int dma_place(int d, int n_dma, int n_products) {
  const int at = (d + 1) * n_products / (n_dma + 1) - 1;
  return at < 0 ? 0 : at;
}

// ---------------------------------------------------------------------------
// Tiles of TM x 128 with TM 256, 192, 128 or 64: as many whole k tiles (A rows, then W rows: (TM + 128) x 128 bytes) as LDS holds, all but
// one in flight.  A prompt of 65 to some 1,000 rows has too few tiles of 256 x 256 to fill the chip, and what bounds it is the way of
// the operands into a CU (192 rows of 4,096 x 28,672: 60 us; without its products and fragment reads 57, without its loads 41), so the
// tile is cut to the rows there are and the depth of the ring hides the memory's latency.  The timetable is the one above: a wave issues
// its DMA instructions between the products of a k step, the barrier stands between the two k steps of a tile (the fragments of the
// last one are in registers by then), and fragments are read one k step ahead.
// us before (tiles of 128 x 128 with two stages below 160 rows, the ring of five slots above) and with this kernel, slices unadded:
//   28,672 x 4,096 gated  150 rows 88.0 57.9   192 rows 70.9 59.5   256 rows 73.0 66.6
//   4,096 x 14,336        150 rows 45.2 36.3   384 rows 68.6 51.2   448 rows 72.4 57.0
//   16,384 x 3,072 gated  150 rows 42.4 36.5   256 rows 53.1 39.7   384 rows 55.0 47.6
//   4,096 x 4,096         150 rows 19.5 15.0   256 rows 23.5 17.8   640 rows 31.5 30.6
// ---------------------------------------------------------------------------
template <int TM> struct StageTiling;               // waves over rows and columns, stages
template <> struct StageTiling<256> { static constexpr int NWM = 4, NWN = 2, S = 3; };
template <> struct StageTiling<192> { static constexpr int NWM = 4, NWN = 2, S = 4; };
template <> struct StageTiling<128> { static constexpr int NWM = 4, NWN = 2, S = 5; };
template <> struct StageTiling<64> { static constexpr int NWM = 2, NWN = 4, S = 6; };
constexpr int STAGES_TN = 128, TILE_GROUP = 4;      // columns a tile; tile columns whose tiles follow each other

template <int EPI, int TM>
__global__ __launch_bounds__(512, 1) void gemm_stages_kernel(const bf16* __restrict__ A, const bf16* __restrict__ W,
                                                             void* __restrict__ Cv, int M, int N, int K, GateOut H, int n_tile0,
                                                             int n_tiles, float* __restrict__ partial, int tiles_per_slice) {
  constexpr int NWM = StageTiling<TM>::NWM, NWN = StageTiling<TM>::NWN, S = StageTiling<TM>::S, TN = STAGES_TN, NW = NWM * NWN;
  constexpr int WM = TM / NWM, WN = TN / NWN, FA = WM / 16, FB = WN / 16, NMF = FA * FB;
  constexpr int STAGE = (TM + TN) * ROWB, L = (TM + TN) / (8 * NW);      // bytes a stage; DMA instructions (8 rows each) a wave and stage
  static_assert(NW == 8 && (TM + TN) % (8 * NW) == 0 && TM % (8 * NW) == 0, "an instruction of all waves lies in one operand");
  static_assert(S * STAGE <= 160 * 1024 && (S - 1) * L < 64, "the ring fits the LDS of a CU; vmcnt holds 6 bits");
  static_assert(FA + FB <= NMF && L <= NMF, "a fragment read and a DMA instruction follow a product");
  static_assert(!gated(EPI) || FB % 2 == 0, "the gated epilogue pairs column tiles");
  extern __shared__ __attribute__((aligned(1024))) unsigned char stages[];
  const int tid = threadIdx.x, lane = tid % WAVE;
  const int wave = __builtin_amdgcn_readfirstlane(tid / WAVE);
  const int wm = wave / NWN, wn = wave % NWN, l16 = lane % 16, lq = lane / 16;
  // blocks of tiles for every XCD (workgroup L runs on XCD L mod 8): TILE_GROUP tile columns, all rows of one block after the other
  const int mt = (M + TM - 1) / TM, T = mt * n_tiles, chunk = (T + 7) / 8;
  const int Lb = blockIdx.x, t = (Lb % 8) * chunk + Lb / 8;
  if (t >= T || Lb / 8 >= chunk) return;
  const int per_group = mt * TILE_GROUP, g = t / per_group, rest = t % per_group, width = min(TILE_GROUP, n_tiles - g * TILE_GROUP);
  const int m0 = (rest / width) * TM, n0 = (n_tile0 + g * TILE_GROUP + rest % width) * TN;
  const int slice = blockIdx.y, n_slices = gridDim.y, kt0 = slice * tiles_per_slice;
  const int nk = min(K / TK - kt0, tiles_per_slice);

  // instruction i of a wave brings rows (i * NW + wave) * 8 ... + 7 of a stage; rows past the edge repeat the last one
  constexpr int LA = TM / (8 * NW);                         // the first LA instructions bring rows of A
  unsigned off[L];
  const char* a_base = (const char*)(A + (size_t)m0 * K + (size_t)kt0 * TK);
  const char* w_base = (const char*)(W + (size_t)n0 * K + (size_t)kt0 * TK);
#pragma unroll
  for (int i = 0; i < L; ++i) {
    const int row = (i * NW + wave) * RPI + lane / CPR;
    const int there = i < LA ? min(row, M - 1 - m0) : min(row - TM, N - 1 - n0);
    off[i] = (unsigned)(((size_t)there * K + ((lane % CPR) ^ swizzle_of(row)) * 8) * 2);
  }
  const unsigned lds0 = (unsigned)(uintptr_t)stages + (unsigned)(wave * 1024);
  auto dma = [&](int kt, int slot, int i) {
    const char* base = (i < LA ? a_base : w_base) + (size_t)kt * ROWB;
    const unsigned at = lds0 + (unsigned)slot * STAGE;
    asm volatile("s_add_u32 m0, %0, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
                 : : "s"(at), "v"(off[i]), "s"(base), "s"((unsigned)(i * NW * 1024)) : "memory", "m0", "scc");
  };

  // the running sums go into the whole ones every FOLD k tiles, the last ones included: no sum is a chain of more than 512 products and of one
  // for every FOLD k tiles, which rounds as little as the finest slices of K
  f32x4 acc[FA][FB], run[FA][FB];
#pragma unroll
  for (int a = 0; a < FA; ++a)
#pragma unroll
    for (int b = 0; b < FB; ++b) acc[a][b] = run[a][b] = (f32x4){0.f, 0.f, 0.f, 0.f};
  auto fold = [&]() {
#pragma unroll
    for (int a = 0; a < FA; ++a)
#pragma unroll
      for (int b = 0; b < FB; ++b) {
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[a][b][r] += run[a][b][r];
        run[a][b] = (f32x4){0.f, 0.f, 0.f, 0.f};
      }
  };
  const int a_row = wm * WM + l16, w_row = TM + wn * WN + l16;
  int a_at[2], w_at[2];
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    a_at[s] = a_row * ROWB + (((4 * s + lq) ^ swizzle_of(a_row)) << 4);
    w_at[s] = w_row * ROWB + (((4 * s + lq) ^ swizzle_of(w_row)) << 4);
  }
  auto frag_a = [&](const unsigned char* st, int s, int a) { return *reinterpret_cast<const bf16x8*>(st + a_at[s] + a * 16 * ROWB); };
  auto frag_w = [&](const unsigned char* st, int s, int b) { return *reinterpret_cast<const bf16x8*>(st + w_at[s] + b * 16 * ROWB); };

#pragma unroll
  for (int p = 0; p < S - 1; ++p)
    if (p < nk)
#pragma unroll
      for (int i = 0; i < L; ++i) dma(p, p, i);
  if (nk >= S - 1) wait_vmcnt<(S - 2) * L>(); else wait_vmcnt<0>();
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_sched_barrier(0);
  bf16x8 fa[2][FA], fw[2][FB];
#pragma unroll
  for (int a = 0; a < FA; ++a) fa[0][a] = frag_a(stages, 0, a);
#pragma unroll
  for (int b = 0; b < FB; ++b) fw[0][b] = frag_w(stages, 0, b);
  int slot = 0;
  auto iteration = [&](int kt, auto more) {                 // more: k tile kt + S - 1 exists and is asked for here
    constexpr bool MORE = decltype(more)::value;
    const int next = slot + 1 == S ? 0 : slot + 1, last = slot == 0 ? S - 1 : slot - 1;
    const unsigned char *cur = stages + slot * STAGE, *nx = stages + next * STAGE;
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      if (s == 1) {                                         // nobody reads the tile any more, and the next one has landed
        wait_lgkmcnt0();
        if (MORE) wait_vmcnt<(S - 2) * L>(); else wait_vmcnt<0>();
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int j = 0; j < NMF; ++j) {
        const int a = j % FA, b = j / FA;
        run[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fa[s][a], fw[s][b], run[a][b], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
        // (behind the last tile the next slot's fragments are read as they lie and not used)
        if (j < FA) fa[s ^ 1][j] = s == 0 ? frag_a(cur, 1, j) : frag_a(nx, 0, j);
        else if (j < FA + FB) fw[s ^ 1][j - FA] = s == 0 ? frag_w(cur, 1, j - FA) : frag_w(nx, 0, j - FA);
        if (s == 0 && MORE) {                               // into the slot of tile kt - 1, free since that tile's barrier
#pragma unroll
          for (int i = 0; i < L; ++i)
            if (j == dma_place(i, L, NMF)) dma(kt + S - 1, last, i);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    slot = next;
  };
  constexpr int FOLD = 8;
  int kt = 0;
  for (; kt + S - 1 < nk; ++kt) {
    iteration(kt, std::true_type{});
    if (kt % FOLD == FOLD - 1) fold();
  }
  for (; kt < nk; ++kt) {
    iteration(kt, std::false_type{});
    if (kt % FOLD == FOLD - 1) fold();
  }
  fold();
  wait_vmcnt<0>();                                 // nothing of this workgroup is on its way into LDS when it ends

  // C: lane (lq, l16) holds rows 4 lq .. 4 lq + 3 of column l16 of every tile
  if (n_slices > 1) {                              // a slice of K: the plain sums, column n = weight row n
    float* plane = partial + (size_t)slice * M * N;
#pragma unroll
    for (int a = 0; a < FA; ++a)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int m = m0 + wm * WM + a * 16 + 4 * lq + r;
        if (m >= M) continue;
#pragma unroll
        for (int b = 0; b < FB; ++b) {
          const int nn = n0 + wn * WN + b * 16 + l16;
          if (nn < N) plane[(size_t)m * N + nn] = acc[a][b][r];
        }
      }
    return;
  }
  GateBias gb[FB / 2 + 1];
  if (EPI == EPI_GATED_BIAS)
#pragma unroll
    for (int pp = 0; pp < FB / 2; ++pp) gb[pp] = gate_bias<EPI>(H, (n0 + wn * WN) / 2 + pp * 16 + l16);
#pragma unroll
  for (int a = 0; a < FA; ++a) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int m = m0 + wm * WM + a * 16 + 4 * lq + r;
      if (m >= M) continue;
      if (gated(EPI)) {                              // weight rows: 16 gate rows, 16 up rows, ...: even tiles gate, odd tiles up
#pragma unroll
        for (int pp = 0; pp < FB / 2; ++pp) {
          const int hcol = (n0 + wn * WN) / 2 + pp * 16 + l16;
          if (hcol < H)
            ((bf16*)Cv)[(size_t)m * H + hcol] = static_cast<bf16>(gate_value<EPI>(acc[a][2 * pp][r], acc[a][2 * pp + 1][r], H, gb[pp]));
        }
      } else {
#pragma unroll
        for (int b = 0; b < FB; ++b) {
          const int nn = n0 + wn * WN + b * 16 + l16;
          if (nn >= N) continue;
          const size_t o = (size_t)m * N + nn;
          if (EPI == 0) ((float*)Cv)[o] = acc[a][b][r];
          if (EPI == 1) ((bf16*)Cv)[o] = static_cast<bf16>(acc[a][b][r]);
          if (EPI == 2) ((float*)Cv)[o] += acc[a][b][r];
        }
      }
    }
  }
}

// ---------------------------------------------------------------------------
// The ring for tiles of 256 and 192 columns.  It uses v_mfma_f32_16x16x32_bf16: the chip is power-bound under
// this loop (the shader clock falls to 1.5-1.8 GHz), and on random operands the 16x16x32 instruction does about a
// sixth more products for the same power than 32x32x16 (2.16 against 1.83 PFLOP/s out of registers: it moves a
// quarter of the accumulator registers per product); the whole GEMM gains 5-10 %.
// A wave owns 64 rows x TN/2 columns: 4 x FB tiles of 16x16.  A tile's 64 k are two k steps of 32; a k step is FB
// groups of four products that share one W fragment.  The W fragments come from LDS through a ring of four, three
// groups ahead of their use; the A fragments of a k step are read during the one before.  The barrier stands in
// front of the group behind which no fragment of the tile is read any more (the ring holds the last three); behind
// it the first fragments of the next tile are read.
// ---------------------------------------------------------------------------
template <int EPI, int TN, int MAP>
__global__ __launch_bounds__(512, 1) void gemm_ring16_kernel(const bf16* __restrict__ A, const bf16* __restrict__ W,
                                                             void* __restrict__ Cv, int M, int N, int K, GateOut H,
                                                             int n_tile0, int n_tiles, float* __restrict__ partial,
                                                             int tiles_per_slice) {
  constexpr int TM = RING_TM, NW = 8, NWM = 4, NWN = 2, WM = TM / NWM, WN = TN / NWN, FA = WM / 16, FB = WN / 16;
  constexpr int DA = (TM / 8) / NW, DW = (TN / 8) / NW;     // DMA instructions (8 rows each) a wave and slot
  constexpr int DA1 = DA / 2, DW1 = (DW + 1) / 2;           // of them in the first of the two quarters that issue them
  constexpr int RB = 4;                                     // the ring of W fragments
  constexpr int NG = 2 * FB;                                // groups a tile
  constexpr int GB = NG - (RB - 1);                         // the barrier stands in front of this group
  constexpr int QG = NG / 4;                                // groups a quarter of the tile (the DMA's timetable)
  constexpr int G3 = GB > 3 * QG ? GB : 3 * QG;             // the first group of the last quarter behind the barrier
  static_assert(FA == 4 && NG % RB == 0 && NG % 4 == 0, "64 rows a wave; the ring goes round whole times a tile");
  static_assert(2 * QG <= GB && NG - G3 >= 1, "W(kt + 2) is issued in front of the barrier, half of A(kt + 2) behind it");
  static_assert(!gated(EPI) || FB % 2 == 0, "the gated epilogue pairs column tiles");
  extern __shared__ __attribute__((aligned(1024))) unsigned char stages[];
  const int tid = threadIdx.x, lane = tid % WAVE;
  const int wave = __builtin_amdgcn_readfirstlane(tid / WAVE);
  const int wm = wave / NWN, wn = wave % NWN;
  const int l16 = lane % 16, lq = lane / 16;
  int tile_m, tile_n;
  if (MAP == 0) {
    tile_m = blockIdx.y;
    tile_n = blockIdx.x + n_tile0;
  } else {                                                  // blocks of tiles for every XCD, as in gemm_stages_kernel
    const int mt = (M + TM - 1) / TM, T = mt * n_tiles, chunk = (T + 7) / 8;
    const int L = blockIdx.x, t = (L % 8) * chunk + L / 8;
    if (t >= T || L / 8 >= chunk) return;
    const int per_group = mt * MAP, g = t / per_group, r = t % per_group;
    const int width = min(MAP, n_tiles - g * MAP);
    tile_n = n_tile0 + g * MAP + r % width;
    tile_m = r / width;
  }
  const int m0 = tile_m * TM, n0 = tile_n * TN;
  const int slice = MAP == 0 ? blockIdx.z : blockIdx.y, n_slices = MAP == 0 ? gridDim.z : gridDim.y;
  const int kt0 = slice * tiles_per_slice;
  const int nk = min(K / TK - kt0, tiles_per_slice);

  unsigned off_a[DA], off_w[DW];
  const char* a_base = (const char*)(A + (size_t)m0 * K + (size_t)kt0 * TK);
  const char* w_base = (const char*)(W + (size_t)n0 * K + (size_t)kt0 * TK);
#pragma unroll
  for (int i = 0; i < DA; ++i) {
    const int row = (i * NW + wave) * RPI + lane / CPR;
    off_a[i] = (unsigned)(((size_t)min(row, M - 1 - m0) * K + ((lane % CPR) ^ swizzle_of(row)) * 8) * 2);
  }
#pragma unroll
  for (int i = 0; i < DW; ++i) {
    const int row = (i * NW + wave) * RPI + lane / CPR;
    off_w[i] = (unsigned)(((size_t)min(row, N - 1 - n0) * K + ((lane % CPR) ^ swizzle_of(row)) * 8) * 2);
  }
  // the LDS address of this wave's first row block of a slot (scalar); instruction i lies i * 8 KB further
  const unsigned lds0 = (unsigned)(uintptr_t)stages + (unsigned)(wave * 1024);
  auto slot_addr = [&](int slot) { return lds0 + (unsigned)slot * RING_SLOT; };
  auto dma = [&](const char* base, unsigned off, unsigned lds_slot, int i) {
    const unsigned add = (unsigned)(i * NW * 1024);
    asm volatile("s_add_u32 m0, %0, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
                 : : "s"(lds_slot), "v"(off), "s"(base), "s"(add) : "memory", "m0", "scc");
  };

  f32x4 acc[FA][FB];
#pragma unroll
  for (int a = 0; a < FA; ++a)
#pragma unroll
    for (int b = 0; b < FB; ++b) acc[a][b] = (f32x4){0.f, 0.f, 0.f, 0.f};

  // fragments (operand rows = lane % 16, 8 k at k offset 8 * (lane / 16)): address in a slot row * 128 +
  // ((4 s + lq) ^ swizzle) * 16 for k step s; tiles 16 rows apart share the swizzle
  const int a_row = wm * WM + l16, w_row = wn * WN + l16;
  int a_at[2], w_at[2];
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    a_at[s] = a_row * ROWB + (((4 * s + lq) ^ swizzle_of(a_row)) << 4);
    w_at[s] = w_row * ROWB + (((4 * s + lq) ^ swizzle_of(w_row)) << 4);
  }
  auto frag_a = [&](int slot, int s, int a) {
    return *reinterpret_cast<const bf16x8*>(stages + slot * RING_SLOT + a_at[s] + a * 16 * ROWB);
  };
  auto frag_w = [&](int slot, int s, int b) {
    return *reinterpret_cast<const bf16x8*>(stages + slot * RING_SLOT + w_at[s] + b * 16 * ROWB);
  };

  // before the loop: W0 A0 W1 and the first half of A1 (what iterations -2 and -1 would have issued)
#pragma unroll
  for (int i = 0; i < DW; ++i) dma(w_base, off_w[i], slot_addr(0), i);
#pragma unroll
  for (int i = 0; i < DA; ++i) dma(a_base, off_a[i], slot_addr(1), i);
  if (nk > 1) {
#pragma unroll
    for (int i = 0; i < DW; ++i) dma(w_base + ROWB, off_w[i], slot_addr(2), i);
#pragma unroll
    for (int i = 0; i < DA1; ++i) dma(a_base + ROWB, off_a[i], slot_addr(3), i);
    wait_vmcnt<DW + DA1>();
  } else {
    wait_vmcnt<0>();
  }
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_sched_barrier(0);
  bf16x8 fa[2][FA], fb[RB];
#pragma unroll
  for (int a = 0; a < FA; ++a) fa[0][a] = frag_a(1, 0, a);
#pragma unroll
  for (int g = 0; g < RB - 1; ++g) fb[g] = frag_w(0, g / FB, g % FB);

  int ws = 0, as = 1;                              // slots of the tile that is multiplied
  // one k tile; T1 / T2: tiles kt + 1 / kt + 2 exist (the loop's last two iterations stand apart, so that the
  // others carry no branch)
  auto iteration = [&](int kt, auto t1_, auto t2_) {
    constexpr bool T1 = decltype(t1_)::value, T2 = decltype(t2_)::value;
    const int ws1 = ws + 2 >= RING_SLOTS ? ws + 2 - RING_SLOTS : ws + 2;          // of tile kt + 1
    const int as1 = as + 2 >= RING_SLOTS ? as + 2 - RING_SLOTS : as + 2;
    const int ws2 = ws1 + 2 >= RING_SLOTS ? ws1 + 2 - RING_SLOTS : ws1 + 2;       // of tile kt + 2
    const int as2 = as1 + 2 >= RING_SLOTS ? as1 + 2 - RING_SLOTS : as1 + 2;
    const unsigned l_as1 = slot_addr(as1), l_ws2 = slot_addr(ws2), l_as2 = slot_addr(as2);
    const char* a1 = a_base + (size_t)(kt + 1) * ROWB;
    const char* a2 = a_base + (size_t)(kt + 2) * ROWB;
    const char* w2 = w_base + (size_t)(kt + 2) * ROWB;
#pragma unroll
    for (int g = 0; g < NG; ++g) {                 // group g: W fragment b of k step s against the four A fragments
      const int s = g / FB, b = g % FB;
      if (g == GB) {
        // No fragment of tile kt is read from here on; this wave's share of tile kt + 1 has landed (W(kt + 2) may
        // still be on its way).  Behind the barrier that holds for all waves.
        wait_lgkmcnt0();
        if (T2) wait_vmcnt<DW>(); else wait_vmcnt<0>();
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int a = 0; a < FA; ++a) {
        acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fa[s][a], fb[g % RB], acc[a][b], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
        if (a == 0) {                                // the W fragment RB - 1 groups ahead (behind the barrier: of the next tile;
          const int gn = g + RB - 1;                 // behind the last tile: read, never used)
          if (gn < NG) fb[gn % RB] = frag_w(ws, gn / FB, gn % FB);
          else fb[gn % RB] = frag_w(ws1, (gn - NG) / FB, (gn - NG) % FB);
        }
        if (a == 2 && s == 0 && b >= FB - FA)        // the A fragments of k step 1, in the last four groups of k step 0
          fa[1][b - (FB - FA)] = frag_a(as, 1, b - (FB - FA));
        if (a >= 2 && g >= GB && (g - GB) * 2 + (a - 2) < FA)      // those of the next tile behind the barrier, two a group
          fa[0][(g - GB) * 2 + (a - 2)] = frag_a(as1, 0, (g - GB) * 2 + (a - 2));
        // DMA by quarters of the tile: the second half of A(kt + 1); W(kt + 2) in two halves; behind the barrier the
        // first half of A(kt + 2); behind the second and the fourth product of a group
        if (a == 1 || a == 3) {
          const int q = g / QG, d = (g % QG) * 2 + (a == 3);
          if (q == 0) { if (T1 && d < DA - DA1) dma(a1, off_a[DA1 + d], l_as1, DA1 + d); }
          else if (q == 1) { if (T2 && d < DW1) dma(w2, off_w[d], l_ws2, d); }
          else if (q == 2) { if (T2 && d < DW - DW1) dma(w2, off_w[DW1 + d], l_ws2, DW1 + d); }
          if (g >= G3) {
            const int d2 = (g - G3) * 2 + (a == 3);
            if (T2 && d2 < DA1) dma(a2, off_a[d2], l_as2, d2);
          }
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    ws = ws1;
    as = as1;
  };
  int kt = 0;
  for (; kt + 2 < nk; ++kt) iteration(kt, std::true_type{}, std::true_type{});
  if (kt + 1 < nk) { iteration(kt, std::true_type{}, std::false_type{}); ++kt; }
  if (kt < nk) iteration(kt, std::false_type{}, std::false_type{});
  wait_vmcnt<0>();                                 // nothing of this workgroup is on its way into LDS when it ends

  // C: lane (lq, l16) holds rows 4 lq .. 4 lq + 3 of column l16 of every tile
  if (n_slices > 1) {                              // a slice of K: the plain sums, column n = weight row n
    float* plane = partial + (size_t)slice * M * N;
#pragma unroll
    for (int a = 0; a < FA; ++a)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int m = m0 + wm * WM + a * 16 + 4 * lq + r;
        if (m >= M) continue;
#pragma unroll
        for (int b = 0; b < FB; ++b) {
          const int nn = n0 + wn * WN + b * 16 + l16;
          if (nn < N) plane[(size_t)m * N + nn] = acc[a][b][r];
        }
      }
    return;
  }
  GateBias gb[FB / 2 + 1];
  if (EPI == EPI_GATED_BIAS)
#pragma unroll
    for (int pp = 0; pp < FB / 2; ++pp) gb[pp] = gate_bias<EPI>(H, (n0 + wn * WN) / 2 + pp * 16 + l16);
#pragma unroll
  for (int a = 0; a < FA; ++a) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int m = m0 + wm * WM + a * 16 + 4 * lq + r;
      if (m >= M) continue;
      if (gated(EPI)) {                              // weight rows: 16 gate rows, 16 up rows, ...: even tiles gate, odd tiles up
#pragma unroll
        for (int pp = 0; pp < FB / 2; ++pp) {
          const int hcol = (n0 + wn * WN) / 2 + pp * 16 + l16;
          if (hcol < H)
            ((bf16*)Cv)[(size_t)m * H + hcol] = static_cast<bf16>(gate_value<EPI>(acc[a][2 * pp][r], acc[a][2 * pp + 1][r], H, gb[pp]));
        }
      } else {
#pragma unroll
        for (int b = 0; b < FB; ++b) {
          const int nn = n0 + wn * WN + b * 16 + l16;
          if (nn >= N) continue;
          const size_t o = (size_t)m * N + nn;
          if (EPI == 0) ((float*)Cv)[o] = acc[a][b][r];
          if (EPI == 1) ((bf16*)Cv)[o] = static_cast<bf16>(acc[a][b][r]);
          if (EPI == 2) ((float*)Cv)[o] += acc[a][b][r];
        }
      }
    }
  }
}

// column tiles n_tile0 ... n_tile0 + n_tiles - 1 (n_tiles < 0: to the last) of a TM x TN tiling
// (slices > 1: the slices of K go to `partial` as [slices][M][N], unadded)
template <int EPI, int TM, int TN, int MAP>
int launch_tiles(const bf16* A, const bf16* W, void* C, int M, int N, int K, GateOut H, hipStream_t stream, int n_tile0 = 0,
                 int n_tiles = -1, float* partial = nullptr, int slices = 1) {
  if (n_tiles < 0) n_tiles = ceil_div(N, TN) - n_tile0;
  const int mt = ceil_div(M, TM);
  const int tiles_per_slice = ceil_div(K / TK, slices);
  slices = ceil_div(K / TK, tiles_per_slice);
  const dim3 grid = MAP == 0 ? dim3(n_tiles, mt, slices) : dim3(8 * ceil_div(mt * n_tiles, 8), slices, 1);
  void (*kernel)(const bf16*, const bf16*, void*, int, int, int, GateOut, int, int, float*, int);
  size_t lds;
  if constexpr (TN == STAGES_TN) {
    static_assert(MAP == TILE_GROUP, "the kernel's own order of tiles");
    kernel = &gemm_stages_kernel<EPI, TM>;
    lds = (size_t)StageTiling<TM>::S * (TM + TN) * ROWB;
  } else {
    static_assert(TM == RING_TM, "the ring's rows");
    kernel = &gemm_ring16_kernel<EPI, TN, MAP>;
    lds = (size_t)RING_SLOTS * RING_SLOT;
  }
  static LdsAllowance allowed;                     // more than 64 KB of LDS has to be asked for once a device
  if (int rc = allow_dynamic_lds(allowed, (const void*)kernel, (int)lds); rc != YALM_OK) return rc;
  kernel<<<grid, 512, lds, stream>>>(A, W, C, M, N, K, H, n_tile0, n_tiles, partial, tiles_per_slice);
  return launch_status();
}

// A tiling and what a launch of it takes, in us: `start` for the first workgroup's loads and the last one's end, `round` more for every
// round of workgroups on all 256 compute units before the last one; an iteration (64 k) of such a round `full`, of the last round on the
// fraction f of the units f last + (1 - f) alone (fewer units have more of the memory and clock higher each); and `out` for a million
// floats written.  Two fits (least squares of the relative errors):
//  * from K = 1,024 on to 2,362 launches: 12 shapes of 1,024 to 28,672 weight rows and K to 14,336, 129 to 8,192 rows, 1 to 12 slices of K;
//    errors 6 to 10 %.  What the plan picks by it is 1 % slower than the fastest of them in the mean and 16 % at worst.  Its terms are the fit's,
//    not the chip's (`out` of 64 x 128 would be stores of 23 TB/s, and rounds start for nothing): bounded to what the chip can
//    do, with a start a round, it fits as well and picks worse (of 51 products where the two differ 31 are slower, up to 12 %, and 10 faster).
//  * below it, where a workgroup's few iterations stand behind each other's starts and ends, to 750 launches: 14 shapes of 512 to 32,000 weight
//    rows and K of 64 to 960, `out` at least 0.3; errors 6 to 12 %, the picks 1 % slower in the mean and, but for one shape (2,048
//    rows of 4,096 x 512), 12 % at worst.  The first fit gave nearly all of these tiles of 64 x 128: 2,048 rows of 28,672 x 128 81 us
//    and now 54, 4,096 of 6,144 x 192 41 and 27, 1,100 of 24,000 x 256 49 and 31.
// Those launches were short bursts.  In the long
// products of a prompt, layer after layer, the power the chip may take sets its clock, and a narrower tile moves more operands for a product:
// `warm` is what a product of several rounds, or of more than 1,024 rows, takes longer then (six layers of 7B sizes with 1,536 tokens whose down
// products went one round of 192 x 128, 170 us for 175 by themselves, took 3 % longer; a step of 28 layers of 3B sizes with 3,641 tokens: q/k/v on 192 x 128
// 103 us by itself against 116 in two launches, and the step 20,750 us against 20,000).
struct TileTimes {
  double start, round, full, last, alone, out;
};
struct Tiling {
  int tm, tn;
  double warm;
  TileTimes long_k, short_k;
};
constexpr int LONG_K = 1024;
constexpr Tiling TILINGS[] = {
    {256, 256, 1.0, {7.74, 0.0, 1.438, 1.301, 1.069, 0.586}, {7.672, 4.099, 1.535, 1.350, 0.956, 0.392}},
    {256, 192, 1.06, {6.13, 0.0, 1.170, 1.157, 0.967, 0.531}, {6.271, 3.445, 1.241, 1.245, 0.710, 0.416}},
    {256, 128, 1.12, {5.33, 0.0, 0.827, 0.820, 0.648, 0.734}, {5.429, 1.301, 1.029, 0.847, 0.523, 0.490}},
    {192, 128, 1.12, {4.98, 0.0, 0.641, 0.656, 0.514, 0.928}, {5.290, 1.983, 0.865, 0.729, 0.351, 0.339}},
    {128, 128, 1.12, {3.68, 0.0, 0.546, 0.567, 0.391, 1.157}, {4.569, 1.582, 0.653, 0.515, 0.273, 0.334}},
    {64, 128, 1.12, {4.22, 0.0, 0.401, 0.435, 0.305, 0.170}, {3.931, 1.499, 0.373, 0.338, 0.214, 0.300}}};
constexpr int N_TILINGS = sizeof(TILINGS) / sizeof(TILINGS[0]);

// What a prompt step's GEMM is launched as: the tiling, the slices of K, and whether whole rounds of 256 x 256
// tiles are followed by a second launch of narrower tiles for the remaining columns.
struct TilePlan {
  int tiling = 0, slices = 1, nt_main = 0;       // nt_main > 0: two launches, the first over nt_main tile columns; `tiling` is the second's
};

// Estimated time in us of `tiles` workgroups of `iters` k tiles each that write `floats` numbers in all, of a product of M rows and K.
double tiles_time(const Tiling& tiling, int M, int K, long tiles, int iters, double floats) {
  const TileTimes& t = K >= LONG_K ? tiling.long_k : tiling.short_k;
  const long rounds = (tiles - 1) / 256;           // before the last one
  const double f = (double)(tiles - 256 * rounds) / 256.0;
  const double iter = (double)rounds * t.full + f * t.last + (1.0 - f) * t.alone;
  return t.start + rounds * t.round + iters * iter * (rounds > 0 || M > 1024 ? tiling.warm : 1.0) + floats * 1e-6 * t.out;
}

// Splits K where the tiles alone leave most CUs without work (short prompts, narrow outputs): a second kernel then
// adds the slices (about (slices + 2) * M * N * 4 bytes at 4 TB/s).  residual: the product is added to the float32
// residual stream.  Unsplit, the tiles read and write that stream in their epilogue, M * N * 8 bytes that no loop
// hides (2,048 x 4,096 x 4,096 on tiles of 128 columns: 87 us, the same tiles with the gated epilogue 65); split,
// the kernel that adds the slices also does the norm behind them, whose own pass (M * N * 6 bytes) is saved.
// consumer: who takes the product.  TAKES_PLAIN: the epilogue, or a kernel that adds the slices; TAKES_RESIDUAL:
// as described above; TAKES_READER: a kernel that reads the product anyway adds the slices as it reads (the
// rotation kernel behind q/k/v), a slice more is M * N * 4 bytes more for it to read.
enum { TAKES_PLAIN = 0, TAKES_RESIDUAL = 1, TAKES_READER = 2 };
TilePlan tile_plan(int M, int N, int K, long workspace_floats, int consumer) {
  const bool residual = consumer == TAKES_RESIDUAL;
  const int nk = K / TK;
  const double MN = (double)M * N;
  TilePlan best;
  double best_t = 1e30;
  const double in_epilogue = residual ? MN * 8.0 / 4.0e6 : 0.0;
  const double norm_saved = residual ? MN * 6.0 / 5.0e6 : 0.0;
  for (int i = 0; i < N_TILINGS; ++i) {
    const long tiles = (long)ceil_div(M, TILINGS[i].tm) * ceil_div(N, TILINGS[i].tn);
    for (int want : {1, 2, 3, 4, 6, 8, 12}) {
      if (want > 1 && (tiles * want > 256 || nk / want < 6 || (long)want * M * N > workspace_floats)) break;
      const int iters = ceil_div(nk, want), s = ceil_div(nk, iters);
      const double adding = consumer == TAKES_READER ? (s - 1) * MN * 4.0 / 5.0e6 : 3.0 + (s + 2) * MN * 4.0 / 4.0e6 - norm_saved;
      const double t = tiles_time(TILINGS[i], M, K, tiles * s, iters, MN * s) + (s > 1 ? adding : in_epilogue);
      if (t < best_t) { best_t = t; best.tiling = i; best.slices = s; best.nt_main = 0; }
    }
  }
  const int mt = ceil_div(M, 256), nt = ceil_div(N, 256);
  const int nt_main = (int)(((long)mt * nt / 256) * 256 / mt);
  TilePlan main;
  double main_t = 1e30;
  if (nt_main > 0 && nt_main < nt)
    for (int i = 2; i < N_TILINGS; ++i) {
      const long rest = (long)ceil_div(M, TILINGS[i].tm) * (ceil_div(N, STAGES_TN) - 2 * nt_main);
      const double t = tiles_time(TILINGS[0], M, K, (long)mt * nt_main, nk, 256.0 * nt_main * M) +
                       tiles_time(TILINGS[i], M, K, rest, nk, MN - 256.0 * nt_main * M) + in_epilogue;
      if (t < main_t) { main_t = t; main.tiling = i; main.nt_main = nt_main; }
    }
  // (a second launch waits for the first one's last tile: for a gain of 3 % and more; 6,000 rows of 4,096 x 28,672 1,054 us in one
  // launch and 1,122 in two that the estimate has level, 2,048 rows 393 and 383 where it has 5 %)
  return main_t < 0.97 * best_t ? main : best;
}

template <int EPI>
int launch_tiling(int tiling, const bf16* A, const bf16* W, void* C, int M, int N, int K, GateOut H, hipStream_t stream, int n_tile0 = 0,
                  float* partial = nullptr, int slices = 1) {
  switch (tiling) {
    case 0: return launch_tiles<EPI, 256, 256, 4>(A, W, C, M, N, K, H, stream, n_tile0, -1, partial, slices);
    case 1: return launch_tiles<EPI, 256, 192, 0>(A, W, C, M, N, K, H, stream, n_tile0, -1, partial, slices);
    case 2: return launch_tiles<EPI, 256, STAGES_TN, TILE_GROUP>(A, W, C, M, N, K, H, stream, n_tile0, -1, partial, slices);
    case 3: return launch_tiles<EPI, 192, STAGES_TN, TILE_GROUP>(A, W, C, M, N, K, H, stream, n_tile0, -1, partial, slices);
    case 4: return launch_tiles<EPI, 128, STAGES_TN, TILE_GROUP>(A, W, C, M, N, K, H, stream, n_tile0, -1, partial, slices);
    case 5: return launch_tiles<EPI, 64, STAGES_TN, TILE_GROUP>(A, W, C, M, N, K, H, stream, n_tile0, -1, partial, slices);
  }
  return YALM_ERR_ARG;
}

// partial: scratch for the slices of K (the plan was made with its size); with slices_out the product's slices
// stay there unadded, *slices_out says how many
template <int EPI>
int launch(const bf16* A, const bf16* W, void* C, float* partial, long partial_floats, int M, int N, int K,
           GateOut H, hipStream_t stream, int* slices_out = nullptr, int consumer = EPI == 2 ? TAKES_RESIDUAL : TAKES_PLAIN) {
  const bool keep = slices_out != nullptr;
  const TilePlan p = tile_plan(M, N, K, partial != nullptr ? partial_floats : 0, consumer);
  if (keep) *slices_out = p.slices;
  if (p.nt_main > 0) {
    int rc = launch_tiles<EPI, 256, 256, 4>(A, W, C, M, N, K, H, stream, 0, p.nt_main);
    if (rc != YALM_OK) return rc;
    return launch_tiling<EPI>(p.tiling, A, W, C, M, N, K, H, stream, 2 * p.nt_main);
  }
  int rc = launch_tiling<EPI>(p.tiling, A, W, C, M, N, K, H, stream, 0, partial, p.slices);
  if (rc != YALM_OK || p.slices == 1 || keep) return rc;
  return yalm_splitk_reduce(partial, C, M, N, H, p.slices, EPI, stream);
}

}  // namespace

// floats of scratch with which yalm_gemm_bf16_dma would split K (0: it would not) as a product that is added to
// the residual stream; other products split as much or less
long yalm_gemm_bf16_dma_workspace(int M, int N, int K) {
  if (M <= 64 || K < TK || K % TK != 0) return 0;
  const int s = max(tile_plan(M, N, K, (long)1 << 40, TAKES_RESIDUAL).slices, tile_plan(M, N, K, (long)1 << 40, TAKES_READER).slices);
  return s > 1 ? (long)s * M * N : 0;
}

extern "C" int yalm_gemm_bf16_dma_choice(int M, int N, int K, long workspace_floats, int consumer) {
  if (M <= 64 || N <= 0 || K < TK || K % TK != 0 || consumer < TAKES_PLAIN || consumer > TAKES_READER) return -1;
  const TilePlan p = tile_plan(M, N, K, workspace_floats, consumer);
  return (p.nt_main > 0 ? 1000 : 0) + 10 * p.slices + p.tiling;
}

// The product's K slices, left unadded, as [*slices][M][N] float32 in the workspace (one slice: the product
// itself), for a consumer that adds them.  More than 64 rows, K a multiple of 64, at least M * N floats.
// residual: the consumer adds them to the residual stream; else it is a kernel that reads the product anyway
// (see tile_plan).
int yalm_gemm_bf16_dma_partial(const void* A, const void* W, float* workspace, long workspace_floats, int M, int N,
                               int K, int* slices_out, int residual, hipStream_t stream) {
  if (M <= 64 || K < TK || K % TK != 0 || ((uintptr_t)A & 15) || ((uintptr_t)W & 15) || workspace == nullptr ||
      workspace_floats < (long)M * N || slices_out == nullptr)
    return YALM_ERR_ARG;
  const bf16* a = (const bf16*)A;
  const bf16* w = (const bf16*)W;
  const int consumer = residual ? TAKES_RESIDUAL : TAKES_READER;
  const TilePlan p = tile_plan(M, N, K, workspace_floats, consumer);
  if (p.slices == 1) {              // the kernel stores the product itself, to the workspace
    *slices_out = 1;
    return launch<0>(a, w, workspace, nullptr, 0, M, N, K, GateOut(0), stream);
  }
  return launch<0>(a, w, nullptr, workspace, workspace_floats, M, N, K, GateOut(0), stream, slices_out, consumer);
}

int yalm_gemm_bf16_dma(const void* A, const void* W, void* C, float* workspace, long workspace_floats, int M, int N,
                       int K, int epilogue, GateOut H, hipStream_t stream) {
  if (M <= 64 || K < TK || K % TK != 0 || ((uintptr_t)A & 15) || ((uintptr_t)W & 15)) return YALM_ERR_ARG;
  const bf16* a = (const bf16*)A;
  const bf16* w = (const bf16*)W;
  switch (epilogue) {
    case 0: return launch<0>(a, w, C, workspace, workspace_floats, M, N, K, H, stream);
    case 1: return launch<1>(a, w, C, workspace, workspace_floats, M, N, K, H, stream);
    case 2: return launch<2>(a, w, C, workspace, workspace_floats, M, N, K, H, stream);
    case 3: return launch<3>(a, w, C, workspace, workspace_floats, M, N, K, H, stream);
    case 5: return launch<5>(a, w, C, workspace, workspace_floats, M, N, K, H, stream);
    case 6: return launch<6>(a, w, C, workspace, workspace_floats, M, N, K, H, stream);
  }
  return YALM_ERR_ARG;
}
