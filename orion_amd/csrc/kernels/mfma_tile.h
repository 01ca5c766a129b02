// Building blocks of the bf16 matrix-core kernels whose output tile is smaller
// than gemm_bf16.hip's 256 x 256: four wavefronts as 2 x 2 over a BM x BN tile,
// both operands K-contiguous, fp32 accumulation with v_mfma_f32_16x16x32_bf16.
//
// A k-tile is 64 elements: one 128-byte line of every operand row.  In LDS the
// 16-byte chunk c of row r sits at position c ^ (r & 7), so the fragment reads of
// eight consecutive lanes (eight rows, one logical chunk) cover all banks once.
// Operands go global -> LDS directly, NS k-tiles ahead of the one in work, with one
// barrier a k-tile.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>
#include <utility>

namespace mfma_tile {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

constexpr int kTileK = 64;
constexpr int kRowBytes = kTileK * 2;

// At most N of this wave's vector memory operations are still in flight.
template <int N>
__device__ __forceinline__ void wait_vm() {
  static_assert(N < 64, "six bits");
  asm volatile("" ::: "memory");        // the loads issued so far stay before it
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | 0x0f70);
  asm volatile("" ::: "memory");
}

// Workgroup barrier that orders LDS accesses and leaves global loads in flight (a
// workgroup fence would wait for every global -> LDS load too).
__device__ __forceinline__ void block_sync() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt(0xc07f);   // lgkmcnt(0)
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// 16 bytes per lane from global memory to LDS at dst (wave-uniform) + lane * 16.
__device__ __forceinline__ void load_to_lds(const void* src, unsigned char* dst) {
  __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)src,
                                   (__attribute__((address_space(3))) void*)dst, 16, 0, 0);
}

__device__ __forceinline__ f32x4 mfma(bf16x8 a, bf16x8 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// The same in place and opaque to the compiler, which shuffles larger sets of
// accumulators between registers in every k-tile when it allocates them itself
// (128 x 128 tiles, 8192 deep: 55 us against 48).  At least three other MFMAs have
// to lie between two that use the same accumulators, and `settle` between the last
// one and what reads them.
__device__ __forceinline__ void mfma_in_place(const bf16x8& a, const bf16x8& b, f32x4& c) {
  asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b));
}

// Two floats to bf16, nearest even, in one register.
__device__ __forceinline__ uint32_t pack_bf16(float lo, float hi) {
  const f32x2 v = {lo, hi};
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2));
}

__device__ __forceinline__ float bf16_lo(uint32_t v) { return __builtin_bit_cast(float, v << 16); }
__device__ __forceinline__ float bf16_hi(uint32_t v) {
  return __builtin_bit_cast(float, v & 0xffff0000u);
}

// A k-tile of ROWS rows on its way to LDS.  Wave w of the group issues the
// 8-row blocks w, w + 4, ...; lane l fetches row l / 8's logical chunk
// (l % 8) ^ (l / 8), which lands at physical chunk l % 8.
template <int ROWS>
struct Rows {
  static constexpr int kLoads = ROWS / 32;   // per wave and k-tile
  static constexpr int kBytes = ROWS * kRowBytes;
  const uint16_t* p[kLoads];
  int wave;

  // row_at(r): the address of the first element of the tile's row r, which has to
  // be readable for every r < ROWS
  template <typename RowAt>
  __device__ __forceinline__ void init(int wave_, int lane, RowAt row_at) {
    wave = wave_;
    const int chunk = (lane & 7) ^ (lane >> 3);
#pragma unroll
    for (int i = 0; i < kLoads; ++i) p[i] = row_at((i * 4 + wave) * 8 + (lane >> 3)) + chunk * 8;
  }
  __device__ __forceinline__ void issue_one(int i, int k, unsigned char* stage) const {
    load_to_lds(p[i] + k, stage + (i * 4 + wave) * 1024);
  }
  __device__ __forceinline__ void issue(int k, unsigned char* stage) const {
#pragma unroll
    for (int i = 0; i < kLoads; ++i) issue_one(i, k, stage);
  }
};

// The fragments of one k-tile that wave (wm, wn) of 2 x 2 needs; it owns rows
// wm * BM / 2, columns wn * BN / 2.  The B fragment is the MFMA's first operand, so
// a lane's four accumulators of tile (i, j) are four consecutive columns of one
// row: row i * 16 + lane % 16, columns j * 16 + lane / 16 * 4 .. + 3.
template <int BM, int BN>
struct Fragments {
  static constexpr int kI = BM / 32, kJ = BN / 32;
  static constexpr int kReads = 2 * (kI + kJ);
  bf16x8 a[2][kI], b[2][kJ];
  __device__ __forceinline__ void read_one(int r, const unsigned char* ta, const unsigned char* tb,
                                           int wm, int wn, int lane) {
    const int ks = r / (kI + kJ), x = r % (kI + kJ);
    const int l16 = lane & 15;
    const int at = ((ks * 4 + (lane >> 4)) ^ (l16 & 7)) << 4;
    if (x < kJ)
      b[ks][x] = *reinterpret_cast<const bf16x8*>(tb + (wn * (BN / 2) + x * 16 + l16) * kRowBytes +
                                                  at);
    else
      a[ks][x - kJ] = *reinterpret_cast<const bf16x8*>(
          ta + (wm * (BM / 2) + (x - kJ) * 16 + l16) * kRowBytes + at);
  }
  __device__ __forceinline__ void read(const unsigned char* ta, const unsigned char* tb, int wm,
                                       int wn, int lane) {
#pragma unroll
    for (int r = 0; r < kReads; ++r) read_one(r, ta, tb, wm, wn, lane);
  }
};

// acc += the fragments' product.  `kReads` reads and `kLoads` loads of what comes
// next are issued one by one between the MFMAs, the reads in the first three
// quarters: a wave that issues them in a row leaves its matrix core idle meanwhile
// (128 x 128 tiles, 8192 deep, one workgroup a compute unit: 68 us; the loads alone
// 40, everything else 49).
// (Each product is a template of its own: loops of this size are not unrolled any more, and
// operands picked at run time go through memory.)
template <int BM, int BN, int kReads, int kLoads, typename Read, typename Load, int... kAt>
__device__ __forceinline__ void multiply(f32x4 (&acc)[BM / 32][BN / 32],
                                         const Fragments<BM, BN>& f, Read read, Load load,
                                         std::integer_sequence<int, kAt...>) {
  constexpr int kI = BM / 32, kJ = BN / 32, kM = 2 * kI * kJ;
  constexpr int kSpan = kM * 3 / 4 > 0 ? kM * 3 / 4 : 1;
  auto product = [&](auto at) {
    constexpr int m = decltype(at)::value;
    constexpr int ks = m / (kI * kJ), i = m / kJ % kI, j = m % kJ;
    if constexpr (kI * kJ >= 4) mfma_in_place(f.b[ks][j], f.a[ks][i], acc[i][j]);
    else acc[i][j] = mfma(f.b[ks][j], f.a[ks][i], acc[i][j]);
    constexpr int kRead = (m * kReads + kSpan - 1) / kSpan;
    constexpr int kReadEnd = ((m + 1) * kReads + kSpan - 1) / kSpan;
#pragma unroll
    for (int x = kRead; x < (kReadEnd < kReads ? kReadEnd : kReads); ++x) read(x);
    constexpr int kLoad = (m * kLoads + kM - 1) / kM, kLoadEnd = ((m + 1) * kLoads + kM - 1) / kM;
#pragma unroll
    for (int x = kLoad; x < (kLoadEnd < kLoads ? kLoadEnd : kLoads); ++x) load(x);
    __builtin_amdgcn_sched_barrier(0);
  };
  (product(std::integral_constant<int, kAt>{}), ...);
}
template <int BM, int BN, int kReads, int kLoads, typename Read, typename Load>
__device__ __forceinline__ void multiply(f32x4 (&acc)[BM / 32][BN / 32],
                                         const Fragments<BM, BN>& f, Read read, Load load) {
  multiply<BM, BN, kReads, kLoads>(
      acc, f, read, load, std::make_integer_sequence<int, 2 * (BM / 32) * (BN / 32)>{});
}
template <int BM, int BN>
__device__ __forceinline__ void multiply(f32x4 (&acc)[BM / 32][BN / 32],
                                         const Fragments<BM, BN>& f) {
  multiply<BM, BN, 0, 0>(acc, f, [](int) {}, [](int) {});
}

// Whatever wrote the accumulators is done with them, and what follows comes after.
template <int I, int J>
__device__ __forceinline__ void settle(f32x4 (&acc)[I][J]) {
#pragma unroll
  for (int i = 0; i < I; ++i)
#pragma unroll
    for (int j = 0; j < J; ++j) asm volatile("" : "+a"(acc[i][j]));
  asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");
#pragma unroll
  for (int i = 0; i < I; ++i)
#pragma unroll
    for (int j = 0; j < J; ++j) asm volatile("" : "+a"(acc[i][j]));
}

template <int I, int J>
__device__ __forceinline__ void clear(f32x4 (&acc)[I][J]) {
#pragma unroll
  for (int i = 0; i < I; ++i)
#pragma unroll
    for (int j = 0; j < J; ++j) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  settle(acc);
}

// acc += A * B^T over KT >= 1 k-tiles that lie k_step elements apart, both operands
// staged through NS stages at `lds`.  The fragments of a whole k-tile are read
// while the one before it is multiplied: behind the barrier the next tile has
// landed, and every wave has this one in registers, so its stage is filled again.
// kShared: groups of waves that meet at the same barriers take turns at the k-tiles, and
// this one has `own` of them, KT or KT - 1 and at least one; for the one that it lacks it
// loads its last one again, and does not multiply it.
template <int BM, int BN, int NS, bool kShared = false>
__device__ __forceinline__ void stream_product(f32x4 (&acc)[BM / 32][BN / 32],
                                               unsigned char* lds, int KT, int k_step,
                                               const Rows<BM>& a, const Rows<BN>& b, int wm,
                                               int wn, int lane, int own = 0) {
  constexpr int kStage = Rows<BM>::kBytes + Rows<BN>::kBytes;
  constexpr int kLoads = Rows<BM>::kLoads + Rows<BN>::kLoads;
  auto k_of = [&](int kt) { return (kShared && kt >= own ? own - 1 : kt) * k_step; };
  auto issue = [&](int kt, unsigned char* s) {
    a.issue(k_of(kt), s);
    b.issue(k_of(kt), s + Rows<BM>::kBytes);
  };
  auto read = [&](Fragments<BM, BN>& f, unsigned char* s) {
    f.read(s, s + Rows<BM>::kBytes, wm, wn, lane);
  };
#pragma unroll
  for (int s = 0; s < NS; ++s)
    if (s < KT) issue(s, lds + s * kStage);
  if (KT >= NS) wait_vm<kLoads*(NS - 1)>();
  else wait_vm<0>();
  block_sync();
  Fragments<BM, BN> even, odd;
  read(even, lds);
  unsigned char* cur = lds;
  // kMore: there is a tile to load into the freed stage
  auto step = [&](const Fragments<BM, BN>& now, Fragments<BM, BN>& next, int kt, auto more) {
    constexpr bool kMore = decltype(more)::value;
    // the loads of the tiles after the next one may still be in flight
    if (kMore || KT - kt >= NS) wait_vm<kLoads*(NS - 2)>();
    else wait_vm<0>();
    block_sync();
    unsigned char* freed = cur;
    cur = cur + kStage == lds + NS * kStage ? lds : cur + kStage;
    if (!kMore && kt + NS < KT) issue(kt + NS, freed);
    __builtin_amdgcn_sched_barrier(0);
    multiply<BM, BN, Fragments<BM, BN>::kReads, kMore ? kLoads : 0>(
        acc, now,
        [&](int r) { next.read_one(r, cur, cur + Rows<BM>::kBytes, wm, wn, lane); },
        [&](int l) {
          if (l < Rows<BM>::kLoads) a.issue_one(l, k_of(kt + NS), freed);
          else b.issue_one(l - Rows<BM>::kLoads, k_of(kt + NS), freed + Rows<BM>::kBytes);
        });
  };
  // between these parts the compiler may move accumulators and fragments
  int kt = 0;
  for (; kt + 1 + NS < KT; kt += 2) {
    step(even, odd, kt, std::true_type{});
    step(odd, even, kt + 1, std::true_type{});
  }
  settle(acc);
  for (; kt + 2 < KT; kt += 2) {
    step(even, odd, kt, std::false_type{});
    step(odd, even, kt + 1, std::false_type{});
  }
  settle(acc);
  if (kt + 1 < KT) {
    step(even, odd, kt, std::false_type{});
    settle(acc);
    block_sync();                      // odd has arrived
    even = odd;
  }
  settle(acc);
  if (!kShared || own == KT) multiply(acc, even);
  settle(acc);
}

// The same for tiles whose fragments of two whole k-tiles do not fit the registers: two
// sets of one k-step (half a k-tile) each.  While the first k-step is multiplied the second
// is read; behind the barrier every wave has all of this tile in registers and the next
// one has landed; while the second k-step is multiplied the next tile's first is read and
// this one's stage is filled again.  Bound as above, with LDS busy most of the time; by
// 128 x 128 tiles 3072 x 1024 x 1024 takes 9.7 us so and 10.2 with whole k-tiles, 2560 x
// 2560 x 4096 57.4 and 56.6.
template <int BM, int BN>
struct HalfFragments {
  static constexpr int kI = BM / 32, kJ = BN / 32, kReads = kI + kJ;
  bf16x8 a[kI], b[kJ];
  // B first: every row of products needs all of it
  template <int kStep>
  __device__ __forceinline__ void read_one(int r, const unsigned char* ta, const unsigned char* tb,
                                           int wm, int wn, int lane) {
    const int l16 = lane & 15;
    const int at = ((kStep * 4 + (lane >> 4)) ^ (l16 & 7)) << 4;
    if (r < kJ)
      b[r] = *reinterpret_cast<const bf16x8*>(tb + (wn * (BN / 2) + r * 16 + l16) * kRowBytes + at);
    else
      a[r - kJ] = *reinterpret_cast<const bf16x8*>(
          ta + (wm * (BM / 2) + (r - kJ) * 16 + l16) * kRowBytes + at);
  }
};

template <int BM, int BN, int kReads, int kLoads, typename Read, typename Load, int... kAt>
__device__ __forceinline__ void multiply_half(f32x4 (&acc)[BM / 32][BN / 32],
                                              const HalfFragments<BM, BN>& f, Read read, Load load,
                                              std::integer_sequence<int, kAt...>) {
  constexpr int kJ = BN / 32, kM = (BM / 32) * kJ, kSpan = kM * 3 / 4;
  auto product = [&](auto at) {
    constexpr int m = decltype(at)::value;
    mfma_in_place(f.b[m % kJ], f.a[m / kJ], acc[m / kJ][m % kJ]);
    constexpr int kRead = (m * kReads + kSpan - 1) / kSpan;
    constexpr int kReadEnd = ((m + 1) * kReads + kSpan - 1) / kSpan;
#pragma unroll
    for (int x = kRead; x < (kReadEnd < kReads ? kReadEnd : kReads); ++x) read(x);
    constexpr int kLoad = (m * kLoads + kM - 1) / kM, kLoadEnd = ((m + 1) * kLoads + kM - 1) / kM;
#pragma unroll
    for (int x = kLoad; x < (kLoadEnd < kLoads ? kLoadEnd : kLoads); ++x) load(x);
    __builtin_amdgcn_sched_barrier(0);
  };
  (product(std::integral_constant<int, kAt>{}), ...);
}

template <int BM, int BN, int NS>
__device__ __forceinline__ void stream_product_halves(f32x4 (&acc)[BM / 32][BN / 32],
                                                      unsigned char* lds, int KT,
                                                      const Rows<BM>& a, const Rows<BN>& b, int wm,
                                                      int wn, int lane) {
  constexpr int kStage = Rows<BM>::kBytes + Rows<BN>::kBytes;
  constexpr int kLoads = Rows<BM>::kLoads + Rows<BN>::kLoads;
  constexpr int kReads = HalfFragments<BM, BN>::kReads;
  constexpr std::make_integer_sequence<int, (BM / 32) * (BN / 32)> kProducts{};
#pragma unroll
  for (int s = 0; s < NS; ++s)
    if (s < KT) {
      a.issue(s * kTileK, lds + s * kStage);
      b.issue(s * kTileK, lds + s * kStage + Rows<BM>::kBytes);
    }
  if (KT >= NS) wait_vm<kLoads*(NS - 1)>();
  else wait_vm<0>();
  block_sync();
  HalfFragments<BM, BN> first, second;
#pragma unroll
  for (int r = 0; r < kReads; ++r)
    first.template read_one<0>(r, lds, lds + Rows<BM>::kBytes, wm, wn, lane);
  unsigned char* cur = lds;
  // kMore: there is a tile to load into the freed stage; kNext: one to read from
  auto step = [&](int kt, auto more, auto next) {
    constexpr bool kMore = decltype(more)::value, kNext = decltype(next)::value;
    multiply_half<BM, BN, kReads, 0>(
        acc, first,
        [&](int r) {
          second.template read_one<1>(r, cur, cur + Rows<BM>::kBytes, wm, wn, lane);
        },
        [](int) {}, kProducts);
    unsigned char* freed = cur;
    if constexpr (kNext) {
      if (kMore || KT - kt >= NS) wait_vm<kLoads*(NS - 2)>();
      else wait_vm<0>();
      block_sync();
      cur = cur + kStage == lds + NS * kStage ? lds : cur + kStage;
    }
    __builtin_amdgcn_sched_barrier(0);
    multiply_half<BM, BN, kNext ? kReads : 0, kMore ? kLoads : 0>(
        acc, second,
        [&](int r) {
          first.template read_one<0>(r, cur, cur + Rows<BM>::kBytes, wm, wn, lane);
        },
        [&](int l) {
          if (l < Rows<BM>::kLoads) a.issue_one(l, (kt + NS) * kTileK, freed);
          else b.issue_one(l - Rows<BM>::kLoads, (kt + NS) * kTileK, freed + Rows<BM>::kBytes);
        },
        kProducts);
  };
  int kt = 0;
  for (; kt + NS < KT; ++kt) step(kt, std::true_type{}, std::true_type{});
  settle(acc);
  for (; kt + 1 < KT; ++kt) step(kt, std::false_type{}, std::true_type{});
  settle(acc);
  step(kt, std::false_type{}, std::false_type{});
  settle(acc);
}

}  // namespace mfma_tile
