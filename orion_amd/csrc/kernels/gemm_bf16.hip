// High-priority co-location kernel: C[M,N] = A[M,K] * B[N,K]^T, bf16 inputs,
// fp32 accumulation on the gfx950 matrix cores, bf16 or fp32 output.
//
// MFMA-bound: 2*M*N*K flops against (M*K + N*K) * 2 + M*N * sizeof(out)
// algorithmic bytes.  Both operands are K-contiguous, so one 16-byte load gives
// a lane the eight consecutive K values v_mfma_f32_16x16x32_bf16 wants.
//
// Tiling (64-wide wavefronts, one workgroup resident per CU):
//   workgroup  256 x 256 x 64   4 wavefronts, 2 x 2
//   wavefront  128 x 128        8 x 8 tiles of v_mfma_f32_16x16x32_bf16, 256
//                               accumulators; a k-tile is two MFMA k-steps
//   LDS        2 stages x (A 32 KiB + B 32 KiB) = 128 KiB of the CU's 160 KiB,
//              filled straight from global memory (global_load_lds_dwordx4)
// An LDS row is one 128-byte cache line of an operand row (eight 16-byte
// chunks); chunk c of row r sits at position c ^ (r & 7), so the 16-byte
// fragment reads of any eight consecutive lanes (eight consecutive rows, same
// logical chunk) cover all banks exactly once.
//
// What shaped it, measured on MI355X at 8192^3 (the GPU sits at its 1400 W
// power limit throughout, so speed is energy per flop as much as overlap):
// v_mfma_f32_16x16x32_bf16 sustains 15 % more than 32x32x16 on random data;
// loading whole 128-byte lines per row (k-tile 64) instead of half lines took
// the global->LDS stream alone from 0.64 to 0.44 ms; with one wave per SIMD the
// matrix core idles whenever the wave issues anything else for longer than one
// MFMA runs, so every other instruction sits alone between two MFMAs.
//
// The reference system has no device code of its own; this kernel stands in for
// the compute-bound half of its toy co-location pair
// (benchmarking/benchmark_suite/toy_models/conv_trainer.py:20-27).

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "kernels.h"
#include "mfma_tile.h"
#include "stream_units.h"

namespace {

using mfma_tile::bf16x2;
using mfma_tile::bf16x8;
using mfma_tile::f32x2;
using mfma_tile::f32x4;
using mfma_tile::u32x2;
using mfma_tile::u32x4;

constexpr int BM = 256;
constexpr int BN = 256;
constexpr int BK = 64;
constexpr int kThreads = 256;
constexpr int kStages = 2;
constexpr int kMatBytes = BM * BK * 2;      // 32 KiB per operand and stage
constexpr int kStageBytes = 2 * kMatBytes;  // A then B

// c += a * b on the matrix core; c lives in accumulator registers and is
// updated in place (as a builtin call the register allocator shuffles the 256
// accumulators between register files in every iteration).
__device__ __forceinline__ void mfma_16x16x32(f32x4& c, const bf16x8& a, const bf16x8& b) {
  asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b));
}

// Four consecutive elements of a row of C from one accumulator tile.
__device__ __forceinline__ void store_quad(float* p, const f32x4& v) {
  *reinterpret_cast<f32x4*>(p) = v;
}
// bf16: round to nearest even (v_cvt_pk_bf16_f32 on gfx950), two per register.
__device__ __forceinline__ void store_quad(uint16_t* p, const f32x4& v) {
  const f32x2 lo = {v[0], v[1]}, hi = {v[2], v[3]};
  u32x2 packed;
  packed[0] = __builtin_bit_cast(uint32_t, __builtin_convertvector(lo, bf16x2));
  packed[1] = __builtin_bit_cast(uint32_t, __builtin_convertvector(hi, bf16x2));
  *reinterpret_cast<u32x2*>(p) = packed;
}

// Workgroup id -> output tile.  Hardware hands consecutive workgroup ids to the
// eight XCDs in turn, each with a private L2, and 256 workgroups (one per CU)
// run at a time.  When the tile grid divides into 16 x 16 super-tiles, every
// such round of 256 workgroups covers one super-tile (16 A panels + 16 B panels
// enter the chip per round instead of 32 + 8 per band), and inside it XCD x owns
// the 4 x 8 block at rows (x / 2) * 4, columns (x % 2) * 8, so the 32 CUs of an
// XCD share 4 A panels and 8 B panels in that XCD's L2.  Other grids fall back
// to bands of kGroupM tile rows per XCD.
constexpr int kXcds = 8;
constexpr int kGroupM = 4;
constexpr int kSuper = 16;

__device__ __forceinline__ void tile_of_block(int bid, int tiles_m, int tiles_n,
                                              int* tm, int* tn) {
  const int total = tiles_m * tiles_n;
  if (tiles_m % kSuper == 0 && tiles_n % kSuper == 0) {
    const int xcd = bid % kXcds;
    const int seq = bid / kXcds;       // order of this workgroup within its XCD
    const int super = seq / 32;        // 32 tiles of every super-tile per XCD
    const int local = seq % 32;
    const int supers_n = tiles_n / kSuper;
    // super-tiles in boustrophedon order: consecutive rounds share their A or
    // their B panels, which the memory-side cache still holds
    const int sr = super / supers_n;
    const int sc = (sr & 1) ? supers_n - 1 - super % supers_n : super % supers_n;
    *tm = sr * kSuper + (xcd / 2) * 4 + local % 4;
    *tn = sc * kSuper + (xcd % 2) * 8 + local / 4;
    return;
  }
  int lid = bid;
  if (total % kXcds == 0) lid = (bid % kXcds) * (total / kXcds) + bid / kXcds;
  const int band = kGroupM * tiles_n;
  const int g = lid / band;
  const int first_m = g * kGroupM;
  const int rows = (tiles_m - first_m < kGroupM) ? (tiles_m - first_m) : kGroupM;
  const int in_band = lid - g * band;
  *tm = first_m + in_band % rows;
  *tn = in_band / rows;
}

template <typename OutT>
__global__ __launch_bounds__(kThreads, 1) void gemm_bf16_nt_kernel(
    const uint16_t* __restrict__ A, const uint16_t* __restrict__ B,
    OutT* __restrict__ C, int M, int N, int K) {
  __shared__ __attribute__((aligned(16))) unsigned char lds[kStages * kStageBytes];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // wave-uniform
  const int wm = wave >> 1;
  const int wn = wave & 1;
  const int l16 = lane & 15;  // row (A, B) or column (C) within a 16x16 tile
  const int lq = lane >> 4;   // 16-byte k chunk of a fragment; row group of C

  int tm, tn;
  tile_of_block(blockIdx.x, M / BM, N / BN, &tm, &tn);
  const size_t row0_a = (size_t)tm * BM;
  const size_t row0_b = (size_t)tn * BN;

  // Global -> LDS without a stop in registers: global_load_lds_dwordx4 writes
  // the 16 bytes a lane loads to LDS at (wave-uniform base) + lane * 16, so one
  // instruction of a wave fills eight 128-byte rows, each a whole cache line of
  // the operand.  Lane l owns row l / 8, PHYSICAL chunk l % 8 and fetches the
  // logical chunk the swizzle stores there, (l % 8) ^ (l / 8).  Wave w issues row
  // blocks w, w + 4, ..., w + 28 of A and of B.
  const int l_chunk = (lane & 7) ^ (lane >> 3);
  const int l_row = wave * 8 + (lane >> 3);
  const uint16_t* gA = A + (row0_a + l_row) * (size_t)K + l_chunk * 8;
  const uint16_t* gB = B + (row0_b + l_row) * (size_t)K + l_chunk * 8;
  const size_t g_step = (size_t)32 * K;  // 32 rows between a wave's row blocks

  // idx 0..7: row blocks of A, 8..15: of B
  auto load_one = [&](int kt, int stage, int idx) {
    const int i = idx & 7;
    const uint16_t* p = (idx < 8 ? gA : gB) + (size_t)kt * BK + i * g_step;
    unsigned char* d = lds + stage * kStageBytes + (idx < 8 ? 0 : kMatBytes) +
                       (i * 4 + wave) * 1024;
    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)p,
                                     (__attribute__((address_space(3))) void*)d, 16, 0, 0);
  };

  f32x4 acc[8][8];
#pragma unroll
  for (int i = 0; i < 8; ++i)
#pragma unroll
    for (int j = 0; j < 8; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) acc[i][j][r] = 0.0f;

  // Fragment reads.  Fragment i of a wave covers rows base + i*16 + l16; of each
  // 128-byte row, k-step ks uses logical chunks ks*4 .. ks*4+3 and lane group lq
  // takes chunk ks*4 + lq.  base and i*16 are multiples of 8, so the swizzle term
  // is l16 % 8.
  const int fr_a = (wm * 128 + l16) * 128;
  const int fr_b = kMatBytes + (wn * 128 + l16) * 128;
  const int fr_k0 = (lq ^ (l16 & 7)) << 4;
  const int fr_k1 = ((4 + lq) ^ (l16 & 7)) << 4;
  // Two fragment register sets, one per k-step of a tile.
  bf16x8 fa[2][8], fb[2][8];
  auto read_one = [&](auto ks_c, int stage, int r) {
    constexpr int KS = decltype(ks_c)::value;
    const unsigned char* st = lds + stage * kStageBytes + (KS ? fr_k1 : fr_k0);
    if (r < 8) fb[KS][r] = *reinterpret_cast<const bf16x8*>(st + fr_b + r * 2048);
    else fa[KS][r - 8] = *reinterpret_cast<const bf16x8*>(st + fr_a + (r - 8) * 2048);
  };
  using KS0 = std::integral_constant<int, 0>;
  using KS1 = std::integral_constant<int, 1>;

  const int KT = K / BK;
#pragma unroll
  for (int idx = 0; idx < 16; ++idx) load_one(0, 0, idx);
  if (KT > 1) {
#pragma unroll
    for (int idx = 0; idx < 16; ++idx) load_one(1, 1, idx);
    __builtin_amdgcn_s_waitcnt(0x4070);  // vmcnt(16): tile 0 has landed
  } else {
    __builtin_amdgcn_s_waitcnt(0x0070);  // vmcnt(0)
  }
  __builtin_amdgcn_s_barrier();
#pragma unroll
  for (int r = 0; r < 16; ++r) read_one(KS0{}, 0, r);

  // One k-tile = two MFMA k-steps of 64 MFMAs.  With one wave per SIMD the
  // matrix core idles whenever the wave issues anything else for longer than one
  // MFMA runs (16 cycles), so every other instruction sits alone between two
  // MFMAs: a fragment read after every third MFMA (all sixteen are out by the
  // 47th, the last sixteen MFMAs cover their latency), a global->LDS load after
  // every fourth in the second k-step.
  //
  // On entry set 0 holds the first k-step of tile kt and every load of tile
  // kt + 1 has been issued.  First k-step: fragment reads of the second.  The
  // wait + barrier after it mean that every wave has all of tile kt in
  // registers and that tile kt + 1 has landed.  Second k-step: first fragment
  // reads of tile kt + 1, loads of tile kt + 2 into the stage tile kt has left.
  auto read_slot = [&](auto ks_c, int stage, int m) {
    // B fragments first: every MFMA row of the next k-step needs all of them
    if (m % 3 == 1) read_one(ks_c, stage, m / 3);
  };
  auto k_tile = [&](int kt, auto has_next, auto has_loads) {
    constexpr bool kNext = decltype(has_next)::value;
    constexpr bool kLoads = decltype(has_loads)::value;
    const int cur = kt & 1, nxt = cur ^ 1;
    __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): set 0 is complete
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int m = 0; m < 64; ++m) {
      mfma_16x16x32(acc[m >> 3][m & 7], fb[0][m & 7], fa[0][m >> 3]);
      read_slot(KS1{}, cur, m);
      __builtin_amdgcn_sched_barrier(0);
    }
    __builtin_amdgcn_s_waitcnt(0x0070);  // vmcnt(0) lgkmcnt(0)
    if (kNext) __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int m = 0; m < 64; ++m) {
      mfma_16x16x32(acc[m >> 3][m & 7], fb[1][m & 7], fa[1][m >> 3]);
      if (kNext) read_slot(KS0{}, nxt, m);
      if (kLoads && (m & 3) == 2) load_one(kt + 2, cur, m >> 2);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  int kt = 0;
  for (; kt + 2 < KT; ++kt) k_tile(kt, std::true_type{}, std::true_type{});
  if (kt + 1 < KT) { k_tile(kt, std::true_type{}, std::false_type{}); ++kt; }
  k_tile(kt, std::false_type{}, std::false_type{});

  // The MFMAs above are opaque to the compiler's hazard handling: give the last
  // ones time to write their accumulators before anything reads them.
  asm volatile("s_nop 15\n\ts_nop 15\n\ts_nop 15" ::: "memory");

  // Epilogue.  The MFMAs ran with the B fragment as first operand, so a lane's
  // four accumulators of tile (i, j) are four CONSECUTIVE columns of one row of
  // C: row i*16 + l16, columns j*16 + lq*4 .. +3.  They are converted, packed
  // and written as one 8- or 16-byte piece into the wave's own quarter of the
  // LDS (free now); whole rows are then read back and stored 16 bytes per lane,
  // so every store instruction covers full cache lines.  A row is cut into
  // 16-byte slots; slot s of row R sits at s ^ (R & 15), which keeps the sixteen
  // rows one write instruction touches apart.
  __builtin_amdgcn_s_waitcnt(0xc07f);
  __builtin_amdgcn_s_barrier();  // every wave has read its last fragments
  constexpr int kElt = (int)sizeof(OutT);
  constexpr int kRowB = 128 * kElt;          // bytes of one row of the block
  constexpr int kPassRows = 32768 / kRowB;   // rows that fit the wave's quarter
  constexpr int kPasses = 128 / kPassRows;   // 1 (bf16) or 2 (fp32)
  constexpr int kIPerPass = 8 / kPasses;
  constexpr int kSlots = kRowB / 16;         // 16-byte slots per row
  constexpr int kRowsPerStore = 64 / kSlots;
  unsigned char* ep = lds + wave * 32768;
  const int st_row = lane / kSlots;
  const int st_slot = lane % kSlots;
  OutT* c_block = C + (row0_a + wm * 128) * (size_t)N + row0_b + wn * 128;
#pragma unroll
  for (int pass = 0; pass < kPasses; ++pass) {
#pragma unroll
    for (int ii = 0; ii < kIPerPass; ++ii)
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int byte = (j * 16 + lq * 4) * kElt;
        unsigned char* dst = ep + (ii * 16 + l16) * kRowB +
                             (((byte >> 4) ^ l16) << 4) + (byte & 15);
        store_quad(reinterpret_cast<OutT*>(dst), acc[pass * kIPerPass + ii][j]);
      }
#pragma unroll
    for (int it = 0; it < kPassRows / kRowsPerStore; ++it) {
      const int R = it * kRowsPerStore + st_row;
      const u32x4 v = *reinterpret_cast<const u32x4*>(ep + R * kRowB +
                                                      ((st_slot ^ (R & 15)) << 4));
      __builtin_nontemporal_store(
          v, reinterpret_cast<u32x4*>(c_block + (size_t)(pass * kPassRows + R) * N) + st_slot);
    }
  }
}

// Other tiles, for products that 256 x 256 tiles would spread badly over the compute units:
// mfma_tile.h's pipeline (HALVES: the one by k-steps, where two k-tiles' fragments would
// fill the registers), GROUPS groups of four waves that take every GROUPS-th k-tile (their
// sums meet in LDS).  Tiles whose rows do not divide 256 reach past the last one.
// Small products are bound by the latency of a k-tile's way to the MFMAs, 0.12 to 0.34 us
// by tile against 0.06 to 0.22 of matrix core time; those that fill the chip by its clock
// (1.9 instead of 2.4 GHz) and by LDS.  Measured, by 256 x 256, by 128 x 128 and smaller
// ones only, and now, us:
//   256 x 512 x 256      8.9   3.6   3.6      2304 x 2304 x 2048  38.5  31.0  23.6
//   1024 x 1024 x 1024  19.7   5.8   5.8      2560 x 2560 x 4096  68.0  56.6  49.3
//   3072 x 1024 x 1024  20.1  10.2   9.7
//   3072 x 1024 x 4096  65.7  26.9  26.6
__device__ __forceinline__ void small_tile_of_block(int bid, int tiles_m, int tiles_n, int* tm,
                                                    int* tn) {
  // a contiguous range of tiles per XCD, bands of kGroupM tile rows
  const int total = tiles_m * tiles_n, per = total / kXcds, extra = total % kXcds;
  const int xcd = bid % kXcds;
  const int lid = xcd * per + (xcd < extra ? xcd : extra) + bid / kXcds;
  const int band = kGroupM * tiles_n;
  const int first_m = lid / band * kGroupM;
  const int rows = tiles_m - first_m < kGroupM ? tiles_m - first_m : kGroupM;
  const int in_band = lid % band;
  *tm = first_m + in_band % rows;
  *tn = in_band / rows;
}

template <int TM, int TN, int NS, int GROUPS, bool HALVES, typename OutT>
__global__ __launch_bounds__(GROUPS * 256, 1) void gemm_bf16_nt_tile_kernel(
    const uint16_t* __restrict__ A, const uint16_t* __restrict__ B, OutT* __restrict__ C, int M,
    int N, int K) {
  using namespace mfma_tile;
  constexpr int kI = TM / 32, kJ = TN / 32;
  constexpr int kGroupLds = NS * (Rows<TM>::kBytes + Rows<TN>::kBytes);
  constexpr int kSumLds = (GROUPS - 1) * TM * TN * 4;
  constexpr int kWaveRows = TM / 2, kWaveCols = TN / 2;
  // rows of a wave's block on their way out, 16 bytes apart so that the sixteen rows that
  // one instruction writes keep to banks of their own
  constexpr int kRowB = kWaveCols * (int)sizeof(OutT), kRowLds = kRowB + 16;
  constexpr int kPassI = kI < 3 ? kI : 3, kPassRows = kPassI * 16;
  constexpr int kOutLds = 4 * kPassRows * kRowLds;
  constexpr int kLds = GROUPS * kGroupLds > kSumLds
                           ? (GROUPS * kGroupLds > kOutLds ? GROUPS * kGroupLds : kOutLds)
                           : (kSumLds > kOutLds ? kSumLds : kOutLds);
  __shared__ __attribute__((aligned(16))) unsigned char lds[kLds];
  const int lane = threadIdx.x & 63;
  const int wave_all = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wave = wave_all & 3, group = wave_all >> 2;
  const int wm = wave >> 1, wn = wave & 1;
  const int l16 = lane & 15, lq = lane >> 4;
  int tm, tn;
  small_tile_of_block(blockIdx.x, (M + TM - 1) / TM, (N + TN - 1) / TN, &tm, &tn);
  static_assert(256 % TN == 0, "no tile reaches past the last column");
  // a tile may reach past the last row, which it then reads again
  const int row0 = tm * TM, col0 = tn * TN;
  Rows<TM> a;
  Rows<TN> b;
  a.init(wave, lane, [&](int r) {
    return A + (size_t)(256 % TM == 0 || row0 + r < M ? row0 + r : M - 1) * K + group * kTileK;
  });
  b.init(wave, lane, [&](int r) { return B + (size_t)(col0 + r) * K + group * kTileK; });
  f32x4 acc[kI][kJ];
  clear(acc);
  if constexpr (HALVES)
    stream_product_halves<TM, TN, NS>(acc, lds, K / kTileK, a, b, wm, wn, lane);
  else
    stream_product<TM, TN, NS, (GROUPS > 1)>(
        acc, lds + group * kGroupLds, (K / kTileK + GROUPS - 1) / GROUPS, GROUPS * kTileK, a, b, wm,
        wn, lane, (K / kTileK - group + GROUPS - 1) / GROUPS);
  block_sync();                        // the stages are free
  if (GROUPS > 1) {
    f32x4* other = reinterpret_cast<f32x4*>(lds) + wave * 64 + lane;
    if (group == 1) {
#pragma unroll
      for (int i = 0; i < kI; ++i)
#pragma unroll
        for (int j = 0; j < kJ; ++j) other[(i * kJ + j) * 256] = acc[i][j];
    }
    block_sync();
    if (group == 0) {
#pragma unroll
      for (int i = 0; i < kI; ++i)
#pragma unroll
        for (int j = 0; j < kJ; ++j) acc[i][j] += other[(i * kJ + j) * 256];
    }
    block_sync();
    if (group == 1) return;
  }
  // whole rows of the wave's block leave as 16-byte pieces, three rows of fragments at a time
  constexpr int kSlots = kRowB / 16, kPerSlot = 16 / (int)sizeof(OutT);
  unsigned char* ep = lds + wave * kPassRows * kRowLds;
  const int row_w = row0 + wm * kWaveRows, col_w = col0 + wn * kWaveCols;
#pragma unroll
  for (int i0 = 0; i0 < kI; i0 += kPassI) {
    constexpr int kAll = kPassRows * kSlots;
    static_assert(16 * kSlots % 64 == 0, "whole instructions");
    const int rows = (kI - i0 < kPassI ? kI - i0 : kPassI) * 16;
#pragma unroll
    for (int i = i0; i < i0 + kPassI && i < kI; ++i)
#pragma unroll
      for (int j = 0; j < kJ; ++j)
        store_quad(reinterpret_cast<OutT*>(ep + ((i - i0) * 16 + l16) * kRowLds) + j * 16 + lq * 4,
                   acc[i][j]);
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront", "local");
#pragma unroll
    for (int first = 0; first < kAll; first += 64) {
      const int at = first + lane, R = at / kSlots, slot = at % kSlots;
      if (first >= rows * kSlots) break;
      const int row = row_w + i0 * 16 + R, col = col_w + slot * kPerSlot;
      if (256 % TM != 0 && row >= M) continue;
      const u32x4 v = *reinterpret_cast<const u32x4*>(ep + R * kRowLds + slot * 16);
      *reinterpret_cast<u32x4*>(C + (size_t)row * N + col) = v;
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront", "local");
  }
}

// What a launch of each tile takes, us: 1.5 + rounds of as many workgroups as the stream
// has compute units * (fixed + per_tile * k-tiles), fitted on the whole GPU, with operands
// in the caches, to 150 products drawn from 256 x 256 x 64 to 8192 x 8192 x 8192.  For
// nine in ten the estimate of the chosen tile is 0.64 to 1.15 of its time, lowest for large
// products, which take the clock down; what counts is the order: over the drawn products
// the choice takes 0.9 % longer in the geometric mean than the best of these tiles each time
// would, and 15 % at most.  The large tile's estimate counts 0.9 because a round of it keeps
// the whole chip busy where one of the others waits (8192 x 2560 x 1024: 48 us by 256 x 256
// tiles, 52 by 128 x 128, 61 with operands out of the caches, estimated at 42 and 42).
// 96 x 128 lies closest to another tile, 128 x 128, so its costs follow a sweep of those two
// at ten sizes from 512 x 4352 to 5888 x 512, with operands in the caches and out of them:
// 8 k-tiles 3 % faster to 3 % slower, 16 8 % faster to 2 % slower, 24 10 % faster to 2 %
// slower, 32 6 to 14 % faster; at 24 sizes of 33 to 128 k-tiles 23 % faster to 2 % slower.
// They cross at 17 k-tiles.
// Streams limited to some compute units have costs of their own, and only the tiles that
// were measured there.  With the whole GPU's, 3 % of the products drawn for 32, 64 and 128
// units went from 128 x 128 to 256 x 256, which takes longer (us, these and the whole GPU's
// choice: 768 x 2816 x 384 on 128 units 9.9 and 11.2, 6656 x 256 x 448 on 64 units 10.4 and
// 11.9, 256 x 2816 x 256 on 32 units 8.2 and 9.1; 5 to 18 % at 16 such products, with
// operands in the caches and out of them).
struct Cost {
  double fixed, per_tile;
};
struct TileCost {
  int tm, tn, groups;     // of waves, which take turns at the k-tiles
  Cost whole, limited;
};
constexpr Cost kUnmeasured = {0.0, 0.0};
constexpr TileCost kTiles[] = {
    {256, 256, 1, {4.65, 0.958}, {4.0, 1.10}},
    {256, 128, 1, {3.44, 0.584}, kUnmeasured},
    {192, 128, 1, {3.92, 0.470}, kUnmeasured},
    {128, 128, 1, {2.80, 0.336}, {2.0, 0.42}},
    {96, 128, 1, {3.33, 0.305}, kUnmeasured},
    {128, 64, 1, {1.7, 0.28}, {1.7, 0.28}},
    {64, 64, 1, {1.5, 0.19}, {1.5, 0.19}},
    {32, 64, 2, {1.5, 0.125}, {1.5, 0.125}},
};

// k-tiles from which on a group of waves may have one less than the other.  By 64 x 64 tiles
// and by 32 x 64, us: 512 x 1024 x 320 3.7 and 3.9, 256 x 512 x 448 3.8 and 3.8, 512 x 512 x
// 576 4.1 and 4.0, 512 x 1024 x 1088 5.4 and 5.2, 512 x 512 x 2112 7.4 and 5.9, 256 x 1280 x
// 4160 11.6 and 9.0, 256 x 512 x 8128 24.7 and 17.1.
constexpr int kLeastUneven = 9;

int tile_for(int M, int N, int K, int cus) {
  int best = 0;
  double best_us = 0.0;
  for (int i = 0; i < (int)(sizeof(kTiles) / sizeof(kTiles[0])); ++i) {
    const TileCost& t = kTiles[i];
    const Cost& c = cus == stream_units::kWholeGpu ? t.whole : t.limited;
    if ((K / BK % t.groups != 0 && K / BK < kLeastUneven) || c.per_tile == 0.0) continue;
    const long long blocks = (long long)((M + t.tm - 1) / t.tm) * ((N + t.tn - 1) / t.tn);
    const int k_tiles = (K / BK + t.groups - 1) / t.groups * t.groups;
    const double us = 1.5 + (double)((blocks + cus - 1) / cus) * (c.fixed + c.per_tile * k_tiles);
    if (i == 0 || us < best_us) {
      best = i;
      best_us = i == 0 ? 0.9 * us : us;
    }
  }
  return best;
}

// The tile for a stream.  On some of the compute units the smaller tiles' workgroups
// only take turns (64 of them, us by 256 x 256 and by the whole GPU's choice: 2048^3
// 36.8 and 51.4; 1024 x 4096 x 512 13.7 and 23.5), so where the whole GPU's choice is
// a smaller one the stream is asked for its mask and the rounds are counted with that.
int tile_for_stream(int M, int N, int K, hipStream_t stream) {
  using stream_units::kWholeGpu;
  const int tile = tile_for(M, N, K, kWholeGpu);
  if (tile == 0) return tile;
  const int cus = stream_units::compute_units_of(stream);
  return cus == kWholeGpu ? tile : tile_for(M, N, K, cus);
}

template <int TM, int TN, int NS, int GROUPS, bool HALVES, typename OutT>
void launch_tiles(const uint16_t* A, const uint16_t* B, OutT* C, int M, int N, int K,
                  hipStream_t stream) {
  const dim3 grid((unsigned)((M + TM - 1) / TM * ((N + TN - 1) / TN)));
  hipLaunchKernelGGL((gemm_bf16_nt_tile_kernel<TM, TN, NS, GROUPS, HALVES, OutT>), grid,
                     dim3(GROUPS * 256), 0, stream, A, B, C, M, N, K);
}

template <typename OutT>
void launch_gemm(const uint16_t* A, const uint16_t* B, OutT* C, int M, int N, int K,
                 hipStream_t stream) {
  switch (tile_for_stream(M, N, K, stream)) {
    case 1: return launch_tiles<256, 128, 3, 1, true>(A, B, C, M, N, K, stream);
    case 2: return launch_tiles<192, 128, 4, 1, true>(A, B, C, M, N, K, stream);
    case 3: return launch_tiles<128, 128, 4, 1, true>(A, B, C, M, N, K, stream);
    case 4: return launch_tiles<96, 128, 4, 1, false>(A, B, C, M, N, K, stream);
    case 5: return launch_tiles<128, 64, 4, 1, false>(A, B, C, M, N, K, stream);
    case 6: return launch_tiles<64, 64, 4, 1, false>(A, B, C, M, N, K, stream);
    case 7: return launch_tiles<32, 64, 4, 2, false>(A, B, C, M, N, K, stream);
    default:
      hipLaunchKernelGGL(gemm_bf16_nt_kernel<OutT>, dim3((unsigned)((M / BM) * (N / BN))),
                         dim3(kThreads), 0, stream, A, B, C, M, N, K);
  }
}

}  // namespace

extern "C" int orion_gemm_bf16_nt(const void* A, const void* B, void* C, int M,
                                  int N, int K, int out_is_f32, void* stream) {
  if (M == 0 || N == 0) return ORION_OK;
  if (A == nullptr || B == nullptr || C == nullptr) return ORION_ERR_ARG;
  if (M < 0 || N < 0 || K <= 0) return ORION_ERR_ARG;
  if (M % BM != 0 || N % BN != 0 || K % BK != 0) return ORION_ERR_SHAPE;
  if ((((uintptr_t)A | (uintptr_t)B | (uintptr_t)C) & 15u) != 0)
    return ORION_ERR_ALIGN;
  const long long tiles = (long long)(M / BM) * (N / BN);
  if (tiles > 0x7fffffffLL) return ORION_ERR_SHAPE;
  if (out_is_f32)
    launch_gemm((const uint16_t*)A, (const uint16_t*)B, (float*)C, M, N, K, (hipStream_t)stream);
  else
    launch_gemm((const uint16_t*)A, (const uint16_t*)B, (uint16_t*)C, M, N, K,
                (hipStream_t)stream);
  return hipGetLastError() == hipSuccess ? ORION_OK : ORION_ERR_LAUNCH;
}
