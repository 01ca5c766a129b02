// Building blocks of the bf16 matrix-core kernels whose output tile is smaller
// than gemm_bf16.hip's 256 x 256: four wavefronts as 2 x 2 over a BM x BN tile,
// both operands K-contiguous, fp32 accumulation with v_mfma_f32_16x16x32_bf16.
//
// A k-tile is 64 elements: one 128-byte line of every operand row.  In LDS the
// 16-byte chunk c of row r sits at position c ^ (r & 7), so the fragment reads of
// eight consecutive lanes (eight rows, one logical chunk) cover all banks once.
// Operands go global -> LDS directly; NS stages keep NS - 1 k-tiles in flight and
// one barrier a k-tile is enough: the stage a wave fills after the barrier is the
// one that all waves had finished reading before it.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

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
  __device__ __forceinline__ void issue(int k, unsigned char* stage) const {
#pragma unroll
    for (int i = 0; i < kLoads; ++i) load_to_lds(p[i] + k, stage + (i * 4 + wave) * 1024);
  }
};

// acc += A tile * B tile over one k-tile in LDS.  Wave (wm, wn) of 2 x 2 owns rows
// wm * BM / 2, columns wn * BN / 2.  The B fragment is the first operand, so a
// lane's four accumulators of tile (i, j) are four consecutive columns of one row:
// row i * 16 + lane % 16, columns j * 16 + lane / 16 * 4 .. + 3.
template <int BM, int BN>
__device__ __forceinline__ void tile_step(f32x4 (&acc)[BM / 32][BN / 32], const unsigned char* a,
                                          const unsigned char* b, int wm, int wn, int lane) {
  const int l16 = lane & 15, lq = lane >> 4;
  const unsigned char* pa = a + (wm * (BM / 2) + l16) * kRowBytes;
  const unsigned char* pb = b + (wn * (BN / 2) + l16) * kRowBytes;
#pragma unroll
  for (int ks = 0; ks < 2; ++ks) {
    const int at = ((ks * 4 + lq) ^ (l16 & 7)) << 4;
    bf16x8 fa[BM / 32], fb[BN / 32];
#pragma unroll
    for (int i = 0; i < BM / 32; ++i)
      fa[i] = *reinterpret_cast<const bf16x8*>(pa + i * 16 * kRowBytes + at);
#pragma unroll
    for (int j = 0; j < BN / 32; ++j)
      fb[j] = *reinterpret_cast<const bf16x8*>(pb + j * 16 * kRowBytes + at);
#pragma unroll
    for (int i = 0; i < BM / 32; ++i)
#pragma unroll
      for (int j = 0; j < BN / 32; ++j) acc[i][j] = mfma(fb[j], fa[i], acc[i][j]);
  }
}

template <int I, int J>
__device__ __forceinline__ void clear(f32x4 (&acc)[I][J]) {
#pragma unroll
  for (int i = 0; i < I; ++i)
#pragma unroll
    for (int j = 0; j < J; ++j) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
}

// acc += A * B^T over KT >= 1 k-tiles that lie k_step elements apart, both operands
// staged through NS stages at `lds`.
template <int BM, int BN, int NS>
__device__ __forceinline__ void stream_product(f32x4 (&acc)[BM / 32][BN / 32],
                                               unsigned char* lds, int KT, int k_step,
                                               const Rows<BM>& a, const Rows<BN>& b, int wm,
                                               int wn, int lane) {
  constexpr int kStage = Rows<BM>::kBytes + Rows<BN>::kBytes;
  constexpr int kLoads = Rows<BM>::kLoads + Rows<BN>::kLoads;
  auto issue = [&](int kt, int stage) {
    unsigned char* s = lds + stage * kStage;
    a.issue(kt * k_step, s);
    b.issue(kt * k_step, s + Rows<BM>::kBytes);
  };
#pragma unroll
  for (int s = 0; s < NS - 1; ++s)
    if (s < KT) issue(s, s);
  int cur = 0, fill = NS - 1;
  for (int kt = 0; kt < KT; ++kt) {
    // the loads of the k-tiles after this one may still be in flight
    if (KT - 1 - kt >= NS - 2) wait_vm<kLoads*(NS - 2)>();
    else wait_vm<0>();
    block_sync();
    if (kt + NS - 1 < KT) issue(kt + NS - 1, fill);
    const unsigned char* s = lds + cur * kStage;
    tile_step<BM, BN>(acc, s, s + Rows<BM>::kBytes, wm, wn, lane);
    cur = cur + 1 == NS ? 0 : cur + 1;
    fill = fill + 1 == NS ? 0 : fill + 1;
  }
}

}  // namespace mfma_tile
