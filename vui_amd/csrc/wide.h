// The main loop of the large-tile products (token-model and prompt passes): C (M x N) = X (M x K) W^T (N x K), both operands
// in the layout of tile.h, bf16 (W may be int8: one 1 KiB piece per 16 rows x 64 columns, the 16 bytes of a lane in column
// order), four waves on a tile of (16 MBW WM) x (16 NBW WN).
//
// A product of many rows is bound by the matrix instructions only if a tile is large enough for what feeds it: with K split
// over the waves of a 32 x 32 or 64 x 64 tile every wave fetches all its operands from L2 (16 flops per byte).  Here the
// waves share a tile through LDS; S stages of KS x 32 columns each are in flight, written to LDS by the loads themselves (a
// piece of the layout is 1 KiB in lane order on both sides), and a wave waits only for the oldest.
// 1024 x 11776 x 2048 without an epilogue: 63 us = 780 TFLOP/s (62 with one chain of sums; hipBLASLt reaches 1125 at 8192^3).
#pragma once
#include "tile.h"

// 16 bytes per lane from g to LDS at byte `at` + 16 lane (wave-uniform; taken from m0, which the compiler loads and so
// knows to be overwritten).  There is no register for the compiler to wait for: the loop counts these loads itself (vmcnt).
// Through the builtin the compiler waited for all of them in front of every LDS read.
__device__ __forceinline__ void wide_to_lds(const char* g, uint32_t at) {
  asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"{m0}"(at), "v"(g) : "memory");
}

// eight int8 -> four packed bf16 pairs, exact
__device__ __forceinline__ uint4 widen8_i8(uint32_t lo, uint32_t hi) {
  uint4 r;
  r.x = f2bf2((float)(int8_t)(lo & 0xff), (float)(int8_t)((lo >> 8) & 0xff));
  r.y = f2bf2((float)(int8_t)((lo >> 16) & 0xff), (float)(int8_t)(lo >> 24));
  r.z = f2bf2((float)(int8_t)(hi & 0xff), (float)(int8_t)((hi >> 8) & 0xff));
  r.w = f2bf2((float)(int8_t)((hi >> 16) & 0xff), (float)(int8_t)(hi >> 24));
  return r;
}

template <int MBW_, int NBW_, int WM_, int WN_, int S_, int KS_, bool I8_ = false>
struct WideTile {
  static constexpr int MBW = MBW_, NBW = NBW_, WM = WM_, WN = WN_, S = S_, KS = KS_;
  static constexpr bool I8 = I8_;
  static constexpr int MB = MBW * WM, NB = NBW * WN;        // 16-row blocks of X and of W
  static constexpr int WK = I8 ? 1 : KS;                    // pieces of a block of W per step
  static constexpr int PIECES = MB * KS + NB * WK, L = PIECES / 4, LDS = S * PIECES * 1024;
  static_assert(WM * WN == 4 && PIECES % 4 == 0, "four waves, the same number of pieces each");
  static_assert(!I8 || KS == 2, "an int8 piece covers 64 columns");

  const char* src[L];
  int stride[L];
  uint32_t lds0;
  char* lds;
  int wave, lane;

  // x(i): byte address of row block i of the tile (all its K columns), w(i) the same for W; lane offsets are added here
  template <typename FX, typename FW>
  __device__ __forceinline__ void begin(char* lds_, int wave_, int lane_, FX&& x, FW&& w) {
    lds = lds_; wave = wave_; lane = lane_;
    lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)lds_;
#pragma unroll
    for (int i = 0; i < L; ++i) {  // pieces wave, wave + 4, ... of a stage are this wave's
      const int q = wave + 4 * i;
      if (q < MB * KS) { src[i] = x(q / KS) + q % KS * 1024 + lane * 16; stride[i] = KS * 1024; }
      else { src[i] = w((q - MB * KS) / WK) + (q - MB * KS) % WK * 1024 + lane * 16; stride[i] = WK * 1024; }
    }
  }
  __device__ __forceinline__ void issue(int slot) {
#pragma unroll
    for (int i = 0; i < L; ++i) {
      wide_to_lds(src[i], lds0 + (uint32_t)(slot * PIECES + wave + 4 * i) * 1024u);
      src[i] += stride[i];
    }
  }
  // the first stages; loads of the caller's own may follow
  __device__ __forceinline__ void prologue(int Q) {
#pragma unroll
    for (int q = 0; q < S - 1; ++q)
      if (q < Q) issue(q);
  }
  // The sums of a quarter of K each (in whole 64 columns) are added in order, as the waves of a K-splitting workgroup leave
  // them, so that a chain of fp32 sums is no longer than there and both forms give the same bits.
  __device__ __forceinline__ void run(int Q, tl_f32x4 (&sum)[NBW][MBW]) {
    tl_f32x4 acc[NBW][MBW];
    steps(0, Q, Q, Q * KS / 2, 1, sum, acc);
#pragma unroll
    for (int i = 0; i < NBW; ++i)
#pragma unroll
      for (int j = 0; j < MBW; ++j) sum[i][j] += acc[i][j];
  }
  // Steps first ... first + Q - 1 of K = 64 n64 columns, which begin with quarter `part` - 1: `acc` is left with the sums of the last
  // quarter, `sum` with those before it.  All waves of the workgroup meet `rounds` >= Q times.
  __device__ __forceinline__ void steps(int first, int Q, int rounds, int n64, int part, tl_f32x4 (&sum)[NBW][MBW], tl_f32x4 (&acc)[NBW][MBW]) {
    const int wm = wave % WM, wn = wave / WM;
    const tl_f32x4 zero = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < NBW; ++i)
#pragma unroll
      for (int j = 0; j < MBW; ++j) acc[i][j] = sum[i][j] = zero;
    int slot = 0, end = (n64 * part >> 2) * 2 / KS - first;  // the first step behind this quarter
    for (int q = 0; q < Q; ++q) {
      // the oldest stage has landed once no more than the stages behind it are outstanding, for every wave behind the
      // barrier; the fragments read from the slot that is filled next have arrived as well
      if (q + S - 1 <= Q) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"((S - 2) * L) : "memory");
      else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      if (q + S - 1 < Q) issue(slot == 0 ? S - 1 : slot - 1);
      const char* st = lds + slot * PIECES * 1024 + lane * 16;
      uint4 xa[KS][MBW], wa[KS][NBW];
#pragma unroll
      for (int k = 0; k < KS; ++k)
#pragma unroll
        for (int j = 0; j < MBW; ++j) xa[k][j] = *reinterpret_cast<const uint4*>(st + ((wm * MBW + j) * KS + k) * 1024);
      if constexpr (I8) {
#pragma unroll
        for (int i = 0; i < NBW; ++i) {
          const uint4 b = *reinterpret_cast<const uint4*>(st + (MB * KS + wn * NBW + i) * 1024);
          wa[0][i] = widen8_i8(b.x, b.y);
          wa[KS - 1][i] = widen8_i8(b.z, b.w);
        }
      } else {
#pragma unroll
        for (int k = 0; k < KS; ++k)
#pragma unroll
          for (int i = 0; i < NBW; ++i) wa[k][i] = *reinterpret_cast<const uint4*>(st + (MB * KS + (wn * NBW + i) * KS + k) * 1024);
      }
      if (q == end) {  // while the fragments arrive
#pragma unroll
        for (int i = 0; i < NBW; ++i)
#pragma unroll
          for (int j = 0; j < MBW; ++j) { sum[i][j] += acc[i][j]; acc[i][j] = zero; }
        do end = (n64 * ++part >> 2) * 2 / KS - first;
        while (end == q);
      }
#pragma unroll
      for (int k = 0; k < KS; ++k)
#pragma unroll
        for (int i = 0; i < NBW; ++i)
#pragma unroll
          for (int j = 0; j < MBW; ++j) acc[i][j] = Tl<bf16_t>::mma(wa[k][i], xa[k][j], acc[i][j]);
      slot = slot == S - 1 ? 0 : slot + 1;
    }
    for (int q = Q; q < rounds; ++q) __builtin_amdgcn_s_barrier();
  }
};

// Which tile takes an M x N x K product, or none (the K-splitting kernels: quicker for the smaller products, at 0.38 us per
// thousand 32 x 32 tiles and 64 columns, and kept unless `keep` of that is still more).  Estimated microseconds besides the launch and the
// epilogue (MI355X): a step of 32 columns takes a tile `wait` us when its CU has nothing else to do and `work` us per tile
// when it has.  Measured (us, K-splitting with its epilogue / quickest large tile without): 1024 x 11776 x 2048 147 / 63,
// 1024 x 2048 x 6144 82 / 40, 1024 x 5120 x 768 26 / 18, 1024 x 768 x 2816 16 / 14, 300 x 768 x 2816 9 / 14.  The prompt pass of the
// backbone has estimates of its own.
enum { WIDE_NONE = -1, WIDE_128 = 0, WIDE_64x128 = 1, WIDE_64 = 2, WIDE_64x128_2 = 3, WIDE_64_2 = 4 };
static inline int wide_pick(int M, int N, int K, double keep) {
  static const struct { int bm, bn; double wait, work; } tile[] = {{128, 128, 0.335, 0.144}, {64, 128, 0.21, 0.08}, {64, 64, 0.17, 0.059}};
  double cost = keep * 0.38e-3 * ((M + 31) / 32) * ((N + 31) / 32) * (K / 64);
  if (M < 128) return WIDE_NONE;
  bool large = false;
  for (int i = 0; i < 3; ++i) {
    const long tiles = (long)((M + tile[i].bm - 1) / tile[i].bm) * ((N + tile[i].bn - 1) / tile[i].bn);
    const double work = (double)((tiles + 255) / 256) * tile[i].work, c = (K / 32) * (work > tile[i].wait ? work : tile[i].wait);
    if (c < cost) large = true;
  }
  if (!large) return WIDE_NONE;
  // Which one is measured beside each other: a step takes `wait` us alone on a CU and `work` for each of more tiles, of which a last round
  // that is nearly empty costs little (workgroups start as others end); `base` us of a launch differ by tile.  Fitted to the three tiles
  // of 107 products (150 ... 1999 rows, the projections of both designs, 768 to 2048 wide): the tile taken is 0.4 us above the quickest on average,
  // by the estimates above 1.7.  us, by those / so: 1300 x 2048 x 6144 70.5 / 57.2, 500 x 6144 x 2048 35.7 / 28, 1999 x 3136 x 2048
  // 56 / 48, 650 x 4224 x 1024 19.2 / 17.4.
  static const struct { double base, wait, work; } each[] = {{0.7, 0.136, 0.145}, {0, 0.12, 0.079}, {-0.35, 0.057, 0.065}};
  int best = 0;
  for (int i = 0; i < 3; ++i) {
    const long tiles = (long)((M + tile[i].bm - 1) / tile[i].bm) * ((N + tile[i].bn - 1) / tile[i].bn);
    const double rounds = tiles <= 256 ? 0 : 0.9 * (tiles / 256.0) + 0.1 * ((tiles + 255) / 256), work = rounds * each[i].work;
    const double c = each[i].base + (K / 32) * (work > each[i].wait ? work : each[i].wait);
    if (i == 0 || c < cost) { best = i; cost = c; }
  }
  return best;
}
