// Forward pass of the Transformer-XL inference client in bf16: the layers of
// relative attention and feed-forward (Dai et al., 2019), and the per-token losses
// of the adaptive softmax (Grave et al., 2017).  The reference's client runs the
// same model as framework operations
// (benchmarking/benchmark_suite/transformer_trainer.py:63-86, :144).
//
// A request is small (768 token rows at batch 4: 0.2 TFLOP, half of it in the
// vocabulary) and a chain of 16 layers, so what bounds it is the number of
// dependent steps and the latency inside each, not a rate.  Two launches a layer (of
// at most 3840 rows); whatever does not depend on the chain runs before it, for all
// layers at once:
//
//   before      positions (sinusoids); keys and values of the memory and the
//               projected positions of every layer; [q k v] = x_0 Wqkv^T
//   layer i     attention                                   txl_attention
//               y = x_i + att Wo^T                          txl_layer, four products
//               x' = LN(y), h = relu(x' W1^T + b1)
//               y = x' + h W2^T + b2
//               x_i+1 = LN(y), [q k v] = x_i+1 Wqkv^T
//   after       hidden = LN(y)
//
// The layer norm rides in the product that reads it: a workgroup has 48 whole rows
// of 512, so it normalises them itself on the way into LDS, from means and squares
// that the product before left for every 32 columns (every workgroup of a row panel
// repeats that; each writes a share of the rows, for the residual and the memory).
// y stays fp32.
//
// Sums are fp32 throughout; activations are rounded to bf16 where the model's
// own operations rounded them, less y, the two query biases (added in fp32) and
// the position scores, which stay fp32 here.

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>
#include <type_traits>

#include "kernels.h"
#include "mfma_tile.h"

namespace {

using namespace mfma_tile;

constexpr int kD = 512;               // model width: the length of a norm's row
constexpr int kHead = 64;             // head width
constexpr int kPanelTiles = kD / kTileK;
constexpr int kMaxJobs = 64;
constexpr int kThreads = 256;

__device__ __forceinline__ void store_bf16x4(uint16_t* p, const f32x4& v) {
  u32x2 packed;
  packed[0] = pack_bf16(v[0], v[1]);
  packed[1] = pack_bf16(v[2], v[3]);
  *reinterpret_cast<u32x2*>(p) = packed;
}

__device__ __forceinline__ u32x4 pack_bf16x8(const f32x4& a, const f32x4& b) {
  return u32x4{pack_bf16(a[0], a[1]), pack_bf16(a[2], a[3]), pack_bf16(b[0], b[1]),
               pack_bf16(b[2], b[3])};
}

__device__ __forceinline__ f32x4 unpack_bf16x4(const u32x2& v) {
  return f32x4{bf16_lo(v[0]), bf16_hi(v[0]), bf16_lo(v[1]), bf16_hi(v[1])};
}

// Sum over the sixteen lanes of a row of lanes, by rotations within it.
__device__ __forceinline__ float sum16(float v) {
  auto rotated = [](float x, auto by) {
    return __builtin_bit_cast(
        float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x),
                                           0x120 + decltype(by)::value, 0xf, 0xf, true));
  };
  v += rotated(v, std::integral_constant<int, 8>{});
  v += rotated(v, std::integral_constant<int, 4>{});
  v += rotated(v, std::integral_constant<int, 2>{});
  v += rotated(v, std::integral_constant<int, 1>{});
  return v;
}

// The values of lanes l, l ^ 16, l ^ 32, l ^ 48 joined: v_permlane*_swap of a register with
// a copy of itself leaves a pair's two halves in the two registers, which takes a few
// cycles where a shuffle goes through LDS.  (In assembly: the builtins' second result came
// out as the first one here.  What was just written needs two cycles before the swap.)
template <typename Join>
__device__ __forceinline__ float over_rows(float v, Join join) {
  float other = v;
  asm volatile("s_nop 1\n\tv_permlane16_swap_b32 %0, %1" : "+v"(v), "+v"(other));
  v = other = join(v, other);
  asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %1" : "+v"(v), "+v"(other));
  return join(v, other);
}
__device__ __forceinline__ float max_over_rows(float v) {
  return over_rows(v, [](float a, float b) { return __builtin_fmaxf(a, b); });
}
__device__ __forceinline__ float sum_over_rows(float v) {
  return over_rows(v, [](float a, float b) { return a + b; });
}

// n / d and n % d in scalar registers, given ~0u / d; the compiler's own division begins with
// a reciprocal in vector ones and takes four times as many instructions.
struct Divided {
  uint32_t quotient, rest;
};
__device__ __forceinline__ Divided divide(uint32_t n, uint32_t d, uint32_t inverse) {
  uint32_t q = __umulhi(n, inverse);               // or one more
  if (n - q * d >= d) ++q;
  return {q, n - q * d};
}

struct Norm {
  const uint16_t* w;
  const uint16_t* b;
  const float2* parts;
  float eps;
};

// A row's layer norm starts from the mean and the sum of squared distances from it
// of each of its sixteen parts of 32 elements, left by the product that made the row.
constexpr int kParts = 16, kPartLen = kD / kParts;

// A row's mean and 1 / deviation, from a part in each of sixteen lanes.
__device__ __forceinline__ float2 row_stats(const float2& part, float eps) {
  const float mean = sum16(part.x) * (1.0f / kParts);
  const float d = part.x - mean;
  const float squares = sum16(__builtin_fmaf((float)kPartLen * d, d, part.y));
  const float variance = squares * (1.0f / kD) + eps;
  // one step of Newton's from the instruction's value (but from zero and infinity, of an
  // infinite variance and of none): two roundings as a square root and a division have, a
  // tenth of the instructions.  The instruction takes a subnormal variance for zero.
  const bool small = variance < 0x1p-126f;
  const float scaled = small ? variance * 0x1p48f : variance;
  const float r = __builtin_amdgcn_rsqf(scaled);
  const float off = __builtin_fmaf(-scaled * r, r, 1.0f);
  const float rstd = r == 0.0f || r == __builtin_inff() ? r : __builtin_fmaf(0.5f * r, off, r);
  return make_float2(mean, small ? rstd * 0x1p24f : rstd);
}

// Eight elements of a row, normalised.  The mean comes off before the scale: as x * rstd -
// mean * rstd, one instruction less an element (the layers of a batch-4 request 540 us instead
// of 545), elements many deviations from zero lose what they differ in.
__device__ __forceinline__ u32x4 norm_chunk(const f32x4 (&v)[2], float mean, float rstd,
                                            const u32x4& w, const u32x4& b) {
  u32x4 out;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const f32x4& x = v[e >> 1];
    out[e] = pack_bf16(
        __builtin_fmaf((x[e * 2 & 3] - mean) * rstd, bf16_lo(w[e]), bf16_lo(b[e])),
        __builtin_fmaf((x[(e * 2 + 1) & 3] - mean) * rstd, bf16_hi(w[e]), bf16_hi(b[e])));
  }
  return out;
}

// A row of 512 for layer norm, sixteen lanes a row: lane l % 16 holds the elements
// of the 16-byte bf16 chunks l % 16 + 16 * j, and one of the parts.
struct NormRow {
  f32x4 v[4][2];
  float2 part;
  __device__ __forceinline__ void load(const float* y, const Norm& norm, int row, int cl) {
    part = norm.parts[(size_t)row * kParts + cl];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float* p = y + (size_t)row * kD + (cl + 16 * j) * 8;
      v[j][0] = *reinterpret_cast<const f32x4*>(p);
      v[j][1] = *reinterpret_cast<const f32x4*>(p + 4);
    }
  }
};

// Weights and biases of the chunks first + 64 / J * j.
template <int J>
struct NormWeights {
  u32x4 w[J], b[J];
  __device__ __forceinline__ void load(const Norm& norm, int first) {
#pragma unroll
    for (int j = 0; j < J; ++j) {
      w[j] = *reinterpret_cast<const u32x4*>(norm.w + (first + 64 / J * j) * 8);
      b[j] = *reinterpret_cast<const u32x4*>(norm.b + (first + 64 / J * j) * 8);
    }
  }
};

__device__ __forceinline__ void norm_row(const NormRow& row, const NormWeights<4>& weights,
                                         float eps, u32x4 (&out)[4]) {
  const float2 stats = row_stats(row.part, eps);
#pragma unroll
  for (int j = 0; j < 4; ++j)
    out[j] = norm_chunk(row.v[j], stats.x, stats.y, weights.w[j], weights.b[j]);
}

// Rows of the normalised (or given) input that later launches and the caller read.
struct RowsOut {
  uint16_t* x;         // [M, 512], may be null
  uint16_t* mem;       // rows mem_from.. of [M, 512], may be null
  int mem_from;
};

__device__ __forceinline__ void put_row(const RowsOut& out, int row, int chunk, const u32x4& v) {
  if (out.x) *reinterpret_cast<u32x4*>(out.x + (size_t)row * kD + chunk * 8) = v;
  if (out.mem && row >= out.mem_from)
    *reinterpret_cast<u32x4*>(out.mem + (size_t)(row - out.mem_from) * kD + chunk * 8) = v;
}

// Workgroup -> tile.  The eight XCDs, each with an L2 of its own, are given workgroups in
// turn; each takes an even, contiguous share of the tiles counted along the rows' columns, so
// that an XCD reads its own rows only.
struct TileMap {
  unsigned tiles, tiles_n;
  __host__ TileMap(size_t tiles_m, size_t tiles_n)
      : tiles((unsigned)(tiles_m * tiles_n)), tiles_n((unsigned)tiles_n) {}
  __host__ unsigned blocks() const { return tiles; }
  __device__ __forceinline__ void tile(unsigned block, int* tm, int* tn) const {
    const unsigned xcd = block % 8, extra = tiles % 8;
    const unsigned at = xcd * (tiles / 8) + (xcd < extra ? xcd : extra) + block / 8;
    *tm = at / tiles_n;
    *tn = at % tiles_n;
  }
};

// C[M, N] = A[M, 512] * W[N, 512]^T with the whole A panel of a workgroup in LDS.  Two
// groups of four waves take the even and the odd k-tiles, W streaming through kPanelStages
// stages each, and their sums meet in LDS.  N is a multiple of BN; rows past M are computed
// from the last row and not written.
constexpr int kPanelThreads = 2 * kThreads;
constexpr int kPanelStages = 3;

template <int BM, int BN>
constexpr int panel_lds() {
  return BM * kD * 2 + 2 * kPanelStages * Rows<BN>::kBytes;
}

template <int BM, int BN, typename Epi>
__device__ __forceinline__ void panel_gemm(unsigned char* lds, const uint16_t* A,
                                           const uint16_t* W, int M, int tm, int tn, int tiles_n,
                                           const RowsOut& out, const Epi& epi) {
  constexpr int NS = kPanelStages, kSteps = kPanelTiles / 2;
  constexpr int kI = BM / 32, kJ = BN / 32;
  static_assert(kI == 2, "each group of waves finishes one of two row tiles");
  const int lane = threadIdx.x & 63;
  const int wave8 = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wave = wave8 & 3, group = wave8 >> 2;
  const int wm = wave >> 1, wn = wave & 1;
  const int l16 = lane & 15, lq = lane >> 4;
  const int row0 = tm * BM;
  unsigned char* stages = lds + BM * kD * 2 + group * NS * Rows<BN>::kBytes;
  // k-tile 2 * step + group
  unsigned char* panel = lds + group * Rows<BM>::kBytes;
  auto k_of = [&](int step) { return (2 * step + group) * kTileK; };
  Rows<BN> b;
  b.init(wave, lane, [&](int r) { return W + (size_t)(tn * BN + r) * kD; });
  // the rows are written by one column of workgroups each
  const int writers = tiles_n < 16 ? tiles_n : 16;

  Rows<BM> a;
  a.init(wave, lane, [&](int r) {
    const int row = row0 + r < M ? row0 + r : M - 1;
    return A + (size_t)row * kD;
  });
#pragma unroll
  for (int s = 0; s < kSteps; ++s) a.issue(k_of(s), panel + s * 2 * Rows<BM>::kBytes);
#pragma unroll
  for (int s = 0; s < NS; ++s) b.issue(k_of(s), stages + s * Rows<BN>::kBytes);
  const int col0 = tn * BN + wn * (BN / 2) + lq * 4;
  typename Epi::Ahead ahead[kJ];
#pragma unroll
  for (int j = 0; j < kJ; ++j) ahead[j] = epi.ahead(col0 + j * 16);

  f32x4 acc[kI][kJ];
  clear(acc);
  Fragments<BM, BN> f[2];
  wait_vm<Rows<BN>::kLoads*(NS - 1)>();
  block_sync();
  f[0].read(panel, stages, wm, wn, lane);
  auto step = [&](auto step_c) {                   // as in stream_product
    constexpr int st = decltype(step_c)::value;
    constexpr bool kMore = st + NS < kSteps;
    wait_vm<kSteps - st >= NS ? Rows<BN>::kLoads*(NS - 2) : 0>();
    block_sync();
    __builtin_amdgcn_sched_barrier(0);
    multiply<BM, BN, Fragments<BM, BN>::kReads, kMore ? Rows<BN>::kLoads : 0>(
        acc, f[st & 1],
        [&](int r) {
          f[(st + 1) & 1].read_one(r, panel + (st + 1) * 2 * Rows<BM>::kBytes,
                                   stages + (st + 1) % NS * Rows<BN>::kBytes, wm, wn, lane);
        },
        [&](int l) { b.issue_one(l, k_of(st + NS), stages + st % NS * Rows<BN>::kBytes); });
  };
  static_assert(kSteps == 4, "the steps");
  step(std::integral_constant<int, 0>{});
  step(std::integral_constant<int, 1>{});
  step(std::integral_constant<int, 2>{});
  multiply(acc, f[1]);
  settle(acc);

  if (out.mem) {                          // sixteen lanes a row
#pragma unroll
    for (int it = 0; it < BM / 32; ++it) {
      const int r = wave8 * (BM / 8) + it * 4 + (lane >> 4);
      if ((wave8 * (BM / 32) + it) % writers != tn || row0 + r >= M) continue;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int chunk = l16 + 16 * j;
        put_row(out, row0 + r, chunk,
                *reinterpret_cast<const u32x4*>(lds + (chunk >> 3) * Rows<BM>::kBytes +
                                                r * kRowBytes + (((chunk & 7) ^ (r & 7)) << 4)));
      }
    }
  }
  block_sync();                           // the panel and the stages have been read
  // group g finishes row tile g of its waves' two
  f32x4* meet = reinterpret_cast<f32x4*>(lds) + wave * 64 + lane;
  if (group == 0) {
#pragma unroll
    for (int j = 0; j < kJ; ++j) meet[(kJ + j) * 256] = acc[1][j];
  } else {
#pragma unroll
    for (int j = 0; j < kJ; ++j) meet[j * 256] = acc[0][j];
  }
  block_sync();
  const int row = row0 + wm * (BM / 2) + group * 16 + l16;
  if (row >= M) return;
#pragma unroll
  for (int j = 0; j < kJ; ++j) {
    const f32x4 mine = group == 0 ? acc[0][j] : acc[1][j];
    epi(row, col0 + j * 16, mine + meet[(group * kJ + j) * 256], ahead[j]);
  }
}

// What is done with four columns of a row of C; `ahead` is what that needs from
// memory, asked for before the product.

// [q k v]: the query leaves twice, with each of the two learned biases.
struct QkvEpi {
  uint16_t *qu, *qv, *kv;
  const uint16_t *u, *v;
  int proj;
  struct Ahead {
    u32x2 u, v;
  };
  __device__ __forceinline__ Ahead ahead(int col) const {
    const int at = col < proj ? col : 0;
    return {*reinterpret_cast<const u32x2*>(u + at), *reinterpret_cast<const u32x2*>(v + at)};
  }
  __device__ __forceinline__ void operator()(int row, int col, const f32x4& x, Ahead a) const {
    if (col >= proj) {
      store_bf16x4(kv + (size_t)row * (2 * proj) + (col - proj), x);
    } else {
      store_bf16x4(qu + (size_t)row * proj + col, x + unpack_bf16x4(a.u));
      store_bf16x4(qv + (size_t)row * proj + col, x + unpack_bf16x4(a.v));
    }
  }
  // the same for eight columns
  struct Needs {
    u32x4 u, v;
  };
  __device__ __forceinline__ Needs needs(int col) const {
    const int at = col < proj ? col : 0;
    return {*reinterpret_cast<const u32x4*>(u + at), *reinterpret_cast<const u32x4*>(v + at)};
  }
  __device__ __forceinline__ void operator()(int row, int col, const f32x4& left,
                                             const f32x4& right, const Needs& a) const {
    auto with = [&](const u32x4& b) {
      return pack_bf16x8(left + unpack_bf16x4(u32x2{b[0], b[1]}),
                         right + unpack_bf16x4(u32x2{b[2], b[3]}));
    };
    if (col >= proj) {
      *reinterpret_cast<u32x4*>(kv + (size_t)row * (2 * proj) + (col - proj)) =
          pack_bf16x8(left, right);
    } else {
      *reinterpret_cast<u32x4*>(qu + (size_t)row * proj + col) = with(a.u);
      *reinterpret_cast<u32x4*>(qv + (size_t)row * proj + col) = with(a.v);
    }
  }
};

template <int BM, int BN, typename Epi>
__global__ __launch_bounds__(kPanelThreads, 1) void txl_panel_gemm_kernel(
    const uint16_t* A, const uint16_t* W, int M, TileMap map, RowsOut out, Epi epi) {
  __shared__ __attribute__((aligned(16))) unsigned char lds[panel_lds<BM, BN>()];
  int tm, tn;
  map.tile(blockIdx.x, &tm, &tn);
  panel_gemm<BM, BN>(lds, A, W, M, tm, tn, map.tiles_n, out, epi);
}

// Independent products with the same inner length, one launch: workgroups
// first_block[i] .. first_block[i + 1] of the grid are job i's.  A workgroup takes 256
// columns, 32 a wave, whose weights stay in registers as the MFMA's fragments over
// kJobPanels panels of 32 rows, which come to LDS four panels ahead.  N is a multiple
// of 32.  As 64 x 128 tiles that each brought their own weights the launch took 50 us of
// a batch-4 request, bound by a workgroup's start (2 us of 6, in 7.5 rounds); so 30, a
// panel bound by the LDS reads of its rows, which every wave needs whole (256 KiB).  The
// weights come by whole lines through LDS: loaded as fragments, where lanes side by side
// are different rows, they take the address unit four times as long (32 us).
struct Job {
  const uint16_t *A, *W;
  uint16_t* out;
  int M, N;
};
struct Jobs {
  Job job[kMaxJobs];
  uint32_t first_block[kMaxJobs + 1];
  int count;
};
constexpr int kJobThreads = 512, kJobM = 32, kJobN = 256, kJobPanels = 8;
constexpr int kJobPanelBytes = kJobM * kD * 2;
constexpr int kJobWaveN = kJobN / 8;
constexpr int kJobPassTiles = kPanelTiles / 2;     // k-tiles of weights in LDS at a time
constexpr int kJobPassBytes = kJobPassTiles * kJobWaveN * kRowBytes;   // of a wave
constexpr int kJobRing = 5;                        // panels; the weights lie in the last four
constexpr int kJobLds = kJobRing * kJobPanelBytes;
static_assert(8 * kJobPassBytes == 4 * kJobPanelBytes, "the weights' place");

__global__ __launch_bounds__(kJobThreads, 1) void txl_jobs_kernel(Jobs jobs) {
  __shared__ __attribute__((aligned(16))) unsigned char lds[kJobLds];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l16 = lane & 15, lq = lane >> 4;
  // Each XCD (they get workgroups in turn) takes a contiguous share of the jobs, so that a
  // layer's memory and weights go to one or two of them: with workgroups in order a batch-4
  // request took 714 us, 709 so.
  const unsigned xcd = blockIdx.x % 8, each = gridDim.x / 8, extra = gridDim.x % 8;
  const unsigned block = xcd * each + (xcd < extra ? xcd : extra) + blockIdx.x / 8;
  const bool before = lane < jobs.count && jobs.first_block[lane] <= block;
  const int i = __builtin_amdgcn_readfirstlane(__popcll(__ballot(before)) - 1);
  const Job job = jobs.job[i];
  const int local = block - jobs.first_block[i];
  const int tiles_n = (job.N + kJobN - 1) / kJobN;
  const int tn = local % tiles_n, row0 = local / tiles_n * (kJobPanels * kJobM);
  const int want = tn * kJobN + wave * kJobWaveN;
  const int col0 = want < job.N ? want : job.N - kJobWaveN;
  const int chunk = ((lane & 7) ^ (lane >> 3)) * 8;
  unsigned char* mine = lds + kJobPanelBytes + wave * kJobPassBytes;
  const uint16_t* weights = job.W + (size_t)(col0 + (lane >> 3)) * kD + chunk;
  // wave w brings the w-th k-tile of the rows, eight rows an instruction; past the last
  // row that one again
  auto fetch = [&](int panel) {
#pragma unroll
    for (int b = 0; b < kJobM / 8; ++b) {
      int row = row0 + panel * kJobM + b * 8 + (lane >> 3);
      row = row < job.M ? row : job.M - 1;
      load_to_lds(job.A + (size_t)row * kD + wave * kTileK + chunk,
                  lds + panel % kJobRing * kJobPanelBytes + (wave * kJobM + b * 8) * kRowBytes);
    }
  };
  auto fragment = [&](const unsigned char* base, int row, int ks) {
    return *reinterpret_cast<const bf16x8*>(base + row * kRowBytes +
                                            (((ks * 4 + lq) ^ (row & 7)) << 4));
  };
  // the first half of the weights straight to LDS, the other through registers, so that
  // both are on their way at once
  constexpr int kBlocks = kJobWaveN / 8;
  u32x4 later[kJobPassTiles][kBlocks];
#pragma unroll
  for (int t = 0; t < kJobPassTiles; ++t)
#pragma unroll
    for (int b = 0; b < kBlocks; ++b)
      load_to_lds(weights + (size_t)b * 8 * kD + t * kTileK,
                  mine + (t * kJobWaveN + b * 8) * kRowBytes);
#pragma unroll
  for (int t = 0; t < kJobPassTiles; ++t)
#pragma unroll
    for (int b = 0; b < kBlocks; ++b)
      later[t][b] = *reinterpret_cast<const u32x4*>(weights + (size_t)b * 8 * kD +
                                                    (kJobPassTiles + t) * kTileK);
  fetch(0);
  bf16x8 w[2 * kPanelTiles][2];                    // [k-step][columns]
  auto read_weights = [&](int first) {
#pragma unroll
    for (int t = 0; t < kJobPassTiles; ++t)
#pragma unroll
      for (int ks = 0; ks < 2; ++ks)
#pragma unroll
        for (int j = 0; j < 2; ++j)
          w[(first + t) * 2 + ks][j] = fragment(mine + t * kJobWaveN * kRowBytes, j * 16 + l16, ks);
    __builtin_amdgcn_s_waitcnt(0xc07f);            // read before anything overwrites it
    __builtin_amdgcn_sched_barrier(0);
  };
  wait_vm<0>();
  read_weights(0);
#pragma unroll
  for (int t = 0; t < kJobPassTiles; ++t)
#pragma unroll
    for (int b = 0; b < kBlocks; ++b)
      *reinterpret_cast<u32x4*>(mine + (t * kJobWaveN + b * 8) * kRowBytes + lane * 16) =
          later[t][b];
  __builtin_amdgcn_s_waitcnt(0xc07f);
  __builtin_amdgcn_sched_barrier(0);
  read_weights(kJobPassTiles);
  const int left = (job.M - row0 + kJobM - 1) / kJobM;
  const int panels = left < kJobPanels ? left : kJobPanels;
  // every panel leaves four stores a wave behind
  const bool whole = want < job.N && row0 + panels * kJobM <= job.M;
  for (int p = 0; p < panels; ++p) {
    // A panel's four loads are followed by at least twelve more and four stores (the
    // loads of the three panels after it, the stores of one) when its turn comes.
    if (whole && p > 0) wait_vm<16>();
    else wait_vm<0>();
    block_sync();                      // this panel is whole, the one before has been read
    if (p == 0)
      for (int n = 1; n < kJobRing - 1; ++n) fetch(n);
    fetch(p + kJobRing - 1);
    f32x4 acc[2][2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    // the next four k-steps' rows on their way while four are multiplied
    constexpr int kAhead = 4, kGroups = 2 * kPanelTiles / kAhead;
    bf16x8 a[2][kAhead][2];
    auto read = [&](int g) {
#pragma unroll
      for (int s = 0; s < kAhead; ++s)
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          const int ks = g * kAhead + s;
          a[g & 1][s][i] =
              fragment(lds + p % kJobRing * kJobPanelBytes + (ks >> 1) * kJobM * kRowBytes,
                       i * 16 + l16, ks & 1);
        }
    };
    read(0);
#pragma unroll
    for (int g = 0; g < kGroups; ++g) {
      if (g + 1 < kGroups) read(g + 1);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int s = 0; s < kAhead; ++s)
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int j = 0; j < 2; ++j)
            acc[i][j] = mfma(w[g * kAhead + s][j], a[g & 1][s][i], acc[i][j]);
      __builtin_amdgcn_sched_barrier(0);
    }
    if (want >= job.N) continue;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int row = row0 + p * kJobM + i * 16 + l16;
      if (row >= job.M) continue;
#pragma unroll
      for (int j = 0; j < 2; ++j)
        store_bf16x4(job.out + (size_t)row * job.N + col0 + j * 16 + lq * 4, acc[i][j]);
    }
  }
  wait_vm<0>();                        // nothing lands in LDS that is no longer ours
}

// One launch a layer behind attention: attention's projection, the feed-forward layer and
// the next layer's queries, keys and values.  As launches of their own, with 64 x 96, 64 x
// 128 and 32 x 64 tiles, the four products took 32 us of a batch-4 request's layer: a launch
// begins 2 us after the last one ends, waits 2 us for its first data and reads weights only
// then.  So 24: 4 for the first product, 6.5, 5.5 and 5.5 for the others (a request 664 us
// instead of 801; batch 1, 16 tokens without memory 529 and 644).
//
// Rows come in panels of up to 48.  The work is a list of tasks, 32 or 128 columns of a
// product for a panel; a task that reads what others of its panel write waits until a
// counter says that they are done.  Its weights, 128 KiB, come meanwhile: a compute unit
// takes in 60 to 100 KiB a us, and as much again of rows.  (16 rows more a panel and half the
// columns a task than 32 rows and 64 or 256, which need twice the weights: 772 us a request
// instead of 803.)  Panels are dealt out to one to eight groups of workgroups (with eight one
// an XCD, which get workgroups in turn), evenly by 16 rows.
//
// Every wait ends, on any number of compute units and beside any other kernel: a group's
// tasks are taken from a counter in the order of the products, a task waits only for tasks
// of its own group before it, and a task that has been taken is run by a workgroup that is
// running.  (The first task not finished waits for nothing; a workgroup takes its next task
// ahead, but that comes after the one that it runs.)
//
// What one workgroup writes and another reads within the launch is written through to
// memory (sc1, agent scope), and a counter is raised when its workgroup's stores have been
// acknowledged.  Readers may cache it: a line of it is one workgroup's (Pieces), no one reads
// it in this launch before the counter says so, and caches start a launch without lines of the
// launches before.  Only the means and squares of a row's parts lie sixteen workgroups to a
// line; a cache that holds the line because it wrote a part of it must not answer for the
// others, so they are read past the caches.  So nothing depends on where a workgroup runs.  A
// stage whose 192 workgroups hand on 32 KiB a panel takes 1.6 us so (2.0 with a panel's
// workgroups on all XCDs), 4.3 (6.8) with release and acquire fences, 2.5 to 2.9 as a launch.
constexpr int kLayerThreads = 512;
constexpr int kGroups = 8;
constexpr int kPanelTiles16 = 3, kPanelRows = 16 * kPanelTiles16;
constexpr int kRowTileBytes = kPanelRows * kRowBytes;        // a panel's k-tile
constexpr int kUnits4 = 4, kUnitCols = 32;           // a wave's weights: four k-tiles of 32 columns
constexpr int kUnitBytes = kUnitCols * kRowBytes, kUnitLoads = kUnitBytes / 1024;
constexpr int kOwn = 159 * 128;                      // a wave's share of the LDS
constexpr int kLayerLds = 8 * kOwn;
constexpr int kResCols = 32, kNormCols = 128;        // of a task
constexpr int kResTasks = kD / kResCols;
constexpr int kLine = 32;                            // counters lie a 128-byte line apart
constexpr int kCoherent = 16;                        // sc1

// Memory that other workgroups of the launch write or read; offsets in bytes.  What lies
// past `bytes` reads as zero and is not written.
struct Shared {
  __amdgpu_buffer_rsrc_t r;
  __device__ __forceinline__ Shared(const void* p, int bytes)
      : r(__builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, bytes, 0x00020000)) {}
  __device__ __forceinline__ u32x4 load16(int at) const {
    return __builtin_amdgcn_raw_buffer_load_b128(r, at, 0, 0);
  }
  __device__ __forceinline__ u32x2 load8(int at) const {
    return __builtin_amdgcn_raw_buffer_load_b64(r, at, 0, 0);
  }
  // past the caches, for lines that several workgroups write a part of
  __device__ __forceinline__ u32x2 fresh8(int at) const {
    return __builtin_amdgcn_raw_buffer_load_b64(r, at, 0, kCoherent);
  }
  __device__ __forceinline__ void store16(int at, const u32x4& v) const {
    __builtin_amdgcn_raw_buffer_store_b128(v, r, at, 0, kCoherent);
  }
  __device__ __forceinline__ void store8(int at, const u32x2& v) const {
    __builtin_amdgcn_raw_buffer_store_b64(v, r, at, 0, kCoherent);
  }
};

__device__ __forceinline__ bf16x8 panel_fragment(const unsigned char* base, int row, int ks,
                                                 int lq) {
  return *reinterpret_cast<const bf16x8*>(base + row * kRowBytes +
                                          (((ks * 4 + lq) ^ (row & 7)) << 4));
}

// The weights of a wave's next task: k-tiles of 32 columns that come by whole lines through
// LDS into registers, as the MFMA's fragments.  Fragment j of a k-tile takes the columns
// 8 * (i / 4) + 4 * j + i % 4, so that a lane's accumulators of both are eight columns in a row.
struct Plan {
  const uint16_t* W;            // 32 columns
  int even, odd;                // this lane's chunk of rows lane / 8 and 8 + lane / 8, bytes
  int ld, first, last;          // k-tiles: this wave's first, the last of all (past it that again)
  int units;                    // of the four that there are
};

// The range check counts `at`, the scalar offset, too (seen on the device, to LDS and to
// registers): a row of a panel that is not full is not read wherever it would lie.
__device__ __forceinline__ void buffer_to_lds(const Shared& from, int lane_at, int at,
                                              unsigned char* to) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(
      from.r, (__attribute__((address_space(3))) void*)to, 16, lane_at, at, 0, 0);
}

__device__ __forceinline__ Plan plan_of(const uint16_t* W, int ld, int first, int units,
                                        int lane) {
  const int at = (lane >> 3) * ld * 2, chunk = (lane & 7) ^ ((lane >> 3) & 3);
  return {W,  at + chunk * 16, at + 16 * ld + (chunk ^ 4) * 16, ld, first, ld / kTileK - 1, units};
}

// Half h (sixteen rows) of unit u.
__device__ __forceinline__ void issue_half(const Plan& plan, int u, int h, unsigned char* to) {
  if (u >= plan.units) return;
  const Shared W(plan.W, kUnitCols * plan.ld * 2);
  const int tile = plan.first + u < plan.last ? plan.first + u : plan.last;
  const int at = h * 32 * plan.ld + tile * kRowBytes;
  buffer_to_lds(W, plan.even, at, to);
  buffer_to_lds(W, plan.odd, at, to + 8 * kRowBytes);
}
__device__ __forceinline__ void issue_unit(const Plan& plan, int u, unsigned char* to) {
  issue_half(plan, u, 0, to);
  issue_half(plan, u, 1, to + kUnitBytes / 2);
}

typedef bf16x8 Weights[kUnits4][2][2];               // [k-tile][k-step][fragment]

// A unit's first sixteen rows lie at `from`, the others 2 KiB or `apart` behind them.
__device__ __forceinline__ void take_unit(Weights& w, int u, const unsigned char* from, int lane,
                                          int apart = kUnitBytes / 2) {
  const int l16 = lane & 15, lq = lane >> 4;
  from += l16 < 8 ? 0 : apart - kUnitBytes / 2;
#pragma unroll
  for (int ks = 0; ks < 2; ++ks)
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int row = (l16 >> 2) * 8 + j * 4 + (l16 & 3);
      w[u][ks][j] = *reinterpret_cast<const bf16x8*>(from + row * kRowBytes +
                                                     (((ks * 4 + lq) ^ (l16 & 7)) << 4));
    }
}

// Sum over eight lanes that lie side by side.
__device__ __forceinline__ float sum8(float v) {
  auto moved = [](float x, auto how) {
    return __builtin_bit_cast(
        float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), decltype(how)::value,
                                           0xf, 0xf, true));
  };
  v += moved(v, std::integral_constant<int, 0xb1>{});     // lane ^ 1
  v += moved(v, std::integral_constant<int, 0x4e>{});     // lane ^ 2
  v += moved(v, std::integral_constant<int, 0x141>{});    // 7 - lane
  return v;
}

struct Panel {
  int row0, rows;
};

// The thread, anew for each task: what is computed from it then belongs to the task (kept
// over all of them it fills the registers).
__device__ __forceinline__ int thread_of_task() {
  int thread = threadIdx.x;
  asm volatile("" : "+v"(thread));
  return thread;
}

constexpr int kSumBytes = 7168;        // of a wave's own: its sums in a residual task

// LDS in a norm task, and where the next task's weights go meanwhile.
struct NormPlaces {
  static constexpr int kPanel = kPanelRows * kD * 2;         // bytes of the normalised rows
  static constexpr int kMeet = 6 * 4 * 1024;                 // and of the halves' sums behind them
  static constexpr int kFree = (8 * kOwn - kPanel - kMeet) / 8 / 128 * 128;
  static constexpr int kDead = kPanel / 8;                   // free once the rows have been read
  static_assert(kFree >= 5 * kUnitBytes / 2 && kDead >= 3 * kUnitBytes / 2, "four units a wave");
  // units 0 and 1 and half of 3 in the free part, unit 2 and the other half in the rows' place
  static __device__ __forceinline__ int of(int unit, int wave) {
    return unit == 2 ? wave * kDead
                     : kPanel + kMeet + wave * kFree + (unit == 3 ? 2 : unit) * kUnitBytes;
  }
  static __device__ __forceinline__ int rest_of_last(int wave) { return wave * kDead + kUnitBytes; }
};

// Where a task's weights wait for it: as its workgroup's first, or as the task before left them.
enum class Place { kFirst, kBehindNorm, kBehindSum };

// What a workgroup carries from task to task.
struct Run {
  unsigned char* lds;
  uint32_t* next;               // the group's counter of tasks
  uint32_t* taken;              // in LDS: what it said last
  Place place;

  __device__ __forceinline__ uint32_t take() const {
    return __hip_atomic_fetch_add(next, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  __device__ __forceinline__ int wave() const {
    return __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  }
  __device__ __forceinline__ unsigned char* own() const { return lds + wave() * kOwn; }
  // A task's weights, and what it waits for (nothing for a null counter); after it everyone
  // knows the next task.  loads(): exactly kLoads loads, which are not waited for.
  template <int kLoads, typename Loads>
  __device__ __forceinline__ void wait_for(Weights& w, int lane, const uint32_t* counter,
                                           uint32_t target, Loads loads) {
    uint32_t seen = target, coming = 0;
    if (threadIdx.x == 0) {
      coming = take();
      if (counter) seen = __hip_atomic_load(counter, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    loads();
    wait_vm<kLoads>();
    if (place == Place::kBehindNorm) {
#pragma unroll
      for (int u = 0; u < kUnits4; ++u)
        take_unit(w, u, lds + NormPlaces::of(u, wave()), lane,
                  u < 3 ? kUnitBytes / 2
                        : NormPlaces::rest_of_last(wave()) - NormPlaces::of(3, wave()));
    } else {
      const int at = place == Place::kFirst ? 0 : kSumBytes;
#pragma unroll
      for (int u = 0; u < kUnits4; ++u)
        take_unit(w, u, own() + (u < 3 ? at + u * kUnitBytes : at ? 0 : 3 * kUnitBytes), lane);
    }
    if (threadIdx.x == 0) {
      while ((int)(seen - target) < 0)
        seen = __hip_atomic_load(counter, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      *taken = coming;
    }
    block_sync();
  }
};

// y = x + bias + A W^T for 32 columns of a panel, in fp32, with the means and squares of the
// part that they are.  The eight waves share the depth, KT k-tiles each at a time, and their
// sums meet in LDS: so a wave's rows and weights pass through LDS once and no wave waits for
// another before the end.  K is a multiple of 64.  kWait: A and x come from this launch.
// ahead(step): 0, the next task is known; 1, the stores are on their way and three units of its
// weights may go to LDS from kSumBytes on.
template <int KT, bool kWait, typename Ahead, int... kTile>
__device__ __forceinline__ void residual_task(Run& run, const Plan& plan, const Panel& panel,
                                              int tn, const uint16_t* A, int K,
                                              const uint16_t* bias, const uint16_t* x, float* y,
                                              float2* parts, const uint32_t* counter,
                                              uint32_t target, Ahead ahead,
                                              std::integer_sequence<int, kTile...>) {
  constexpr int kSumRow = kResCols + 4;            // floats
  constexpr int kI = kPanelTiles16, kJ = kResCols / 16;
  // rows that need not be waited for lie beside the weights on their way
  constexpr int kRowsAt = kWait ? 0 : KT * kUnitBytes;
  constexpr int kFit = (kOwn - kRowsAt) / kRowTileBytes, kAhead = kFit < KT ? kFit : KT;
  static_assert(kAhead > 0 && (kWait || kAhead == KT), "");
  static_assert(kPanelRows * kSumRow * 4 <= kSumBytes && kSumBytes + 3 * kUnitBytes <= kOwn, "");
  const int thread = thread_of_task(), lane = thread & 63;
  const int wave = __builtin_amdgcn_readfirstlane(thread >> 6);
  const int l16 = lane & 15, lq = lane >> 4;
  unsigned char* own = run.lds + wave * kOwn;
  const int tiles = K / kTileK, col0 = tn * kResCols;
  // the element that this thread finishes (of the first 384)
  const int r = thread >> 3, col = col0 + (thread & 7) * 4;
  const int at = r < panel.rows ? r : panel.rows - 1;
  const u32x2 add_b = bias ? *reinterpret_cast<const u32x2*>(bias + col) : u32x2{0, 0};
  u32x2 add_x = {0, 0};
  if constexpr (!kWait)
    add_x = *reinterpret_cast<const u32x2*>(x + (size_t)(panel.row0 + at) * kD + col);
  // rows past the last one are not read
  const Shared rows(A + (size_t)panel.row0 * K, panel.rows * K * 2);
  const int rows_at = (lane >> 3) * K * 2 + ((lane & 7) ^ (lane >> 3)) * 16;
  Weights w;
  f32x4 acc[kI][kJ];
#pragma unroll
  for (int i = 0; i < kI; ++i)
#pragma unroll
    for (int j = 0; j < kJ; ++j) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  for (int base = 0; base < tiles; base += 8 * KT) {
    const int mine = base + wave * KT;
    // past the last k-tile that one again, not multiplied
    auto issue_rows = [&](int kt) {
      const int tile = mine + kt < tiles ? mine + kt : tiles - 1;
#pragma unroll
      for (int b = 0; b < kPanelRows / 8; ++b)
        buffer_to_lds(rows, rows_at, b * 16 * K + tile * kRowBytes,
                    own + kRowsAt + kt % kAhead * kRowTileBytes + b * 8 * kRowBytes);
    };
    // what need not be waited for is on its way with a first task's weights
    const bool at_once = !kWait && (base > 0 || run.place == Place::kFirst);
    if (at_once) {
#pragma unroll
      for (int kt = 0; kt < kAhead; ++kt) issue_rows(kt);
    }
    if (base == 0) {
      run.wait_for<0>(w, lane, kWait ? counter : nullptr, target, [] {});
      if constexpr (kWait)
        add_x =
            Shared(x + (size_t)panel.row0 * kD, panel.rows * kD * 2).load8((at * kD + col) * 2);
    } else {
      Plan more = plan;
      more.first = mine;
#pragma unroll
      for (int u = 0; u < KT; ++u) issue_unit(more, u, own + u * kUnitBytes);
      wait_vm<0>();
#pragma unroll
      for (int u = 0; u < KT; ++u) take_unit(w, u, own + u * kUnitBytes, lane);
      __builtin_amdgcn_s_waitcnt(0xc07f);
      __builtin_amdgcn_sched_barrier(0);
    }
    if (!at_once) {
#pragma unroll
      for (int kt = 0; kt < kAhead; ++kt) issue_rows(kt);
    }
    if (base == 0) ahead(0);
    auto multiply_tile = [&](auto tile) {
      constexpr int kt = decltype(tile)::value;
      constexpr int kIssued = kt + kAhead < KT ? kt + kAhead : KT;
      wait_vm<kWait ? (kIssued - kt - 1) * (kPanelRows / 8) : 0>();
      bf16x8 a[2][kI];
#pragma unroll
      for (int ks = 0; ks < 2; ++ks)
#pragma unroll
        for (int i = 0; i < kI; ++i)
          a[ks][i] = panel_fragment(own + kRowsAt + kt % kAhead * kRowTileBytes, i * 16 + l16, ks,
                                    lq);
      if constexpr (kt + kAhead < KT) {
        __builtin_amdgcn_s_waitcnt(0xc07f);        // read before it is overwritten
        __builtin_amdgcn_sched_barrier(0);
        issue_rows(kt + kAhead);
      }
      if (mine + kt >= tiles) return;
#pragma unroll
      for (int ks = 0; ks < 2; ++ks)
#pragma unroll
        for (int i = 0; i < kI; ++i)
#pragma unroll
          for (int j = 0; j < kJ; ++j) acc[i][j] = mfma(w[kt][ks][j], a[ks][i], acc[i][j]);
    };
    (multiply_tile(std::integral_constant<int, kTile>{}), ...);
    __builtin_amdgcn_s_waitcnt(0xc07f);
    __builtin_amdgcn_sched_barrier(0);
  }
#pragma unroll
  for (int i = 0; i < kI; ++i)
#pragma unroll
    for (int j = 0; j < kJ; ++j)
      *reinterpret_cast<f32x4*>(own + ((i * 16 + l16) * kSumRow + lq * 8 + j * 4) * 4) = acc[i][j];
  block_sync();
  if (r < kPanelRows) {
    f32x4 product = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int w = 0; w < 8; ++w)
      product += *reinterpret_cast<const f32x4*>(run.lds + w * kOwn +
                                                 (r * kSumRow + (thread & 7) * 4) * 4);
    const f32x4 v = product + unpack_bf16x4(add_b) + unpack_bf16x4(add_x);
    Shared(y + (size_t)panel.row0 * kD, panel.rows * kD * 4)
        .store16((r * kD + col) * 4, __builtin_bit_cast(u32x4, v));
    // eight threads hold the part
    static_assert(kResCols == kPartLen, "a task's columns are a part");
    const float mean = sum8(v[0] + v[1] + v[2] + v[3]) * (1.0f / kPartLen);
    float squares = 0.0f;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float d = v[e] - mean;
      squares = __builtin_fmaf(d, d, squares);
    }
    squares = sum8(squares);
    if ((thread & 7) == 0)
      Shared(parts + (size_t)panel.row0 * kParts, panel.rows * kParts * 8)
          .store8((r * kParts + tn) * 8, u32x2{__builtin_bit_cast(uint32_t, mean),
                                               __builtin_bit_cast(uint32_t, squares)});
  }
  ahead(1);
}

// 128 columns of LN(y) W^T for a panel: wave (c, g) takes 32 of the columns and half of the
// depth.  put(row, chunk, values): normalised rows, of which each task writes a share;
// needs(column): what finish(row, column, left, right, needs) wants from memory for eight
// columns; ahead(step): 0, the next task is known; 1, its weights may go to
// the free part of NormPlaces, and 2, behind the stores, to the rows' place.
template <typename PutRow, typename Needs, typename Finish, typename Ahead>
__device__ __forceinline__ void norm_task(Run& run, const Panel& panel, int tn, int tasks,
                                          const float* y, const Norm& norm,
                                          const uint32_t* counter, uint32_t target, PutRow put,
                                          Needs needs, Finish finish, Ahead ahead) {
  constexpr int KT = kUnits4, kI = kPanelTiles16, kJ = 2, kPasses = kPanelRows / 16;
  const int thread = thread_of_task(), lane = thread & 63;
  const int wave = __builtin_amdgcn_readfirstlane(thread >> 6);
  const int l16 = lane & 15, lq = lane >> 4, cg = wave & 3, kg = wave >> 2;
  const int col0 = tn * kNormCols + cg * 32;
  const int cl = lane & 31;                        // 32 lanes a row, two rows at a time
  unsigned char* lds = run.lds;
  NormWeights<2> weights;
  Weights w;
  run.wait_for<4>(w, lane, counter, target, [&] { weights.load(norm, cl); });
  {
    const Shared rows(y + (size_t)panel.row0 * kD, panel.rows * kD * 4);
    const Shared sums(norm.parts + (size_t)panel.row0 * kParts, panel.rows * kParts * 8);
    __builtin_amdgcn_sched_barrier(0);
    // rows past the last one are zeros
    constexpr int kRows = 2 * kPasses;             // of a wave
    const int first = wave * kRows;
    f32x2 part[2];                                 // of rows 0 to 3, and of 4 and 5
#pragma unroll
    for (int h = 0; h < 2; ++h)
      part[h] = __builtin_bit_cast(
          f32x2, sums.fresh8(((first + (h ? 4 + (lq & 1) : lq)) * kParts + l16) * 8));
    f32x4 v[kPasses][2][2];
#pragma unroll
    for (int it = 0; it < kPasses; ++it)
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int h = 0; h < 2; ++h)
          v[it][j][h] = __builtin_bit_cast(
              f32x4, rows.load16(((first + it * 2 + (lane >> 5)) * kD + (cl + 32 * j) * 8 + h * 4) *
                                 4));
    ahead(0);
    float mean[kRows], rstd[kRows];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const float2 stats = row_stats(make_float2(part[h][0], part[h][1]), norm.eps);
#pragma unroll
      for (int i = 0; i < (h ? 2 : 4); ++i) {
        mean[h * 4 + i] = __builtin_bit_cast(
            float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, stats.x), i * 16));
        rstd[h * 4 + i] = __builtin_bit_cast(
            float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, stats.y), i * 16));
      }
    }
#pragma unroll
    for (int it = 0; it < kPasses; ++it)           // the rows are here
#pragma unroll
      for (int j = 0; j < 2; ++j) asm volatile("" ::"v"(v[it][j][0]), "v"(v[it][j][1]));
    ahead(1);
#pragma unroll
    for (int it = 0; it < kPasses; ++it) {
      __builtin_amdgcn_sched_barrier(0);
      const bool second = lane >= 32;
      const int r = first + it * 2 + second;
      const float m = second ? mean[it * 2 + 1] : mean[it * 2];
      const float s = second ? rstd[it * 2 + 1] : rstd[it * 2];
      u32x4 out[2];
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const int chunk = cl + 32 * j;
        out[j] = norm_chunk(v[it][j], m, s, weights.w[j], weights.b[j]);
        *reinterpret_cast<u32x4*>(lds + (chunk >> 3) * kRowTileBytes + r * kRowBytes +
                                  (((chunk & 7) ^ (r & 7)) << 4)) = out[j];
      }
      if ((wave * kPasses + it) % tasks == tn && r < panel.rows) {
        put(r, cl, out[0]);
        put(r, cl + 32, out[1]);
      }
    }
  }
  const auto needed = needs(col0 + lq * 8);
  block_sync();
  f32x4 acc[kI][kJ];
#pragma unroll
  for (int i = 0; i < kI; ++i)
#pragma unroll
    for (int j = 0; j < kJ; ++j) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  bf16x8 a[2][2][kI];                  // the next k-tile's while one is multiplied
  auto read = [&](int kt) {
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
      for (int i = 0; i < kI; ++i)
        a[kt & 1][ks][i] =
            panel_fragment(lds + (kg * KT + kt) * kRowTileBytes, i * 16 + l16, ks, lq);
  };
  read(0);
#pragma unroll
  for (int kt = 0; kt < KT; ++kt) {
    if (kt + 1 < KT) read(kt + 1);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
      for (int i = 0; i < kI; ++i)
#pragma unroll
        for (int j = 0; j < kJ; ++j) acc[i][j] = mfma(w[kt][ks][j], a[kt & 1][ks][i], acc[i][j]);
    __builtin_amdgcn_sched_barrier(0);
  }
  // Half g finishes row tile g, and row tile 2 of every second four waves' columns.
  f32x4* meet = reinterpret_cast<f32x4*>(lds + NormPlaces::kPanel) + cg * 64 + lane;
  const bool both = (cg & 1) == kg;                // this wave finishes two row tiles
#pragma unroll
  for (int j = 0; j < kJ; ++j) {
    meet[(kg * 2 + j) * 256] = kg ? acc[0][j] : acc[1][j];
    if (!both) meet[(4 + j) * 256] = acc[2][j];
  }
  block_sync();
  const f32x4* other = meet + (1 - kg) * 2 * 256;
  finish(kg * 16 + l16, col0 + lq * 8, (kg ? acc[1][0] : acc[0][0]) + other[0],
         (kg ? acc[1][1] : acc[0][1]) + other[256], needed);
  if (both)
    finish(32 + l16, col0 + lq * 8, acc[2][0] + meet[4 * 256], acc[2][1] + meet[5 * 256], needed);
  ahead(2);
}

struct Layer {
  struct Product {
    const uint16_t* W;
    int ld, columns;                      // of a task
    int tasks;                            // of a panel
    uint32_t inverse;                     // ~0u over them
  } product[4];                           // out, ff1, ff2, the next layer's qkv
  int products;                           // 4, in the last layer 3
  const uint16_t *att, *x, *ff1_b, *ff2_b;
  Norm norm1, norm2;                      // the parts of y1 and y2
  float *y1, *y2;
  float2 *parts1, *parts2;
  uint16_t *x2, *h;
  RowsOut rows_out;                       // the next layer's input
  QkvEpi qkv;
  uint32_t* counters;                     // kLine apart: 8 of tasks, then 3 a panel
  int rows, inner, proj, panels;          // panels a group has counters for
};

// What a workgroup needs before it has a task comes first, by value, in registers; the
// workgroup asks for its first task with it and reads the rest meanwhile (a batch-4 request
// 669 us so and 684 with all of it in the structure, batch 1, 16 tokens 519 and 531).
struct alignas(8) LayerStart {
  uint32_t* counters;
  int group_mask, group_shift;            // of 1, 2, 4 or 8 groups
  int tiles16, layer;                     // tiles of 16 rows; of the layers
};
// The other arguments, read anew where they are needed (from the scalar cache): sixty
// registers of them do not fit, and the compiler would keep them in lanes of vector ones.
__device__ __forceinline__ const Layer& arguments() {
  auto at = (const __attribute__((address_space(4))) char*)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(at));
  return *(const Layer*)(at + sizeof(LayerStart));
}

__global__ __launch_bounds__(kLayerThreads, 1) void txl_layer_kernel(
    uint32_t* all_counters, int group_mask, int group_shift, int all16, int layer, Layer) {
  // LayerStart, which has to arrive in registers, and behind it the structure
  __shared__ __attribute__((aligned(16))) unsigned char lds[kLayerLds + 16];
  const int group = blockIdx.x & group_mask;
  // this group's share of the row tiles, and its panels': even ones
  int first16, tiles16, panels;
  int ff1_at, ff2_at, qkv_at, tasks;     // tasks before each product's
  uint32_t before;                       // taken in the layers before
  Run run;
  run.lds = lds;
  run.taken = reinterpret_cast<uint32_t*>(lds + kLayerLds);
  run.place = Place::kFirst;
  run.next = all_counters + group * kLine;
  uint32_t first_taken = 0;
  if (threadIdx.x == 0) first_taken = run.take();
  {
    const Layer& a = arguments();
    const int each = all16 >> group_shift, extra = all16 & group_mask;
    tiles16 = each + (group < extra ? 1 : 0);
    first16 = group * each + (group < extra ? group : extra);
    panels = (tiles16 + kPanelTiles16 - 1) / kPanelTiles16;
    ff1_at = panels * kResTasks;
    ff2_at = ff1_at + panels * a.product[1].tasks;
    qkv_at = ff2_at + ff1_at;
    const int all = qkv_at + panels * a.product[3].tasks;
    tasks = a.products == 4 ? all : qkv_at;
    before = (uint32_t)layer * (all + (gridDim.x >> group_shift));
    // every cache line of the arguments
    auto line = [&](int i) {
      return *reinterpret_cast<const int*>(reinterpret_cast<const char*>(&a) + 64 * i);
    };
    static_assert(sizeof(Layer) > 5 * 64 && sizeof(Layer) <= 6 * 64, "six lines");
    asm volatile("" ::"s"(line(0)), "s"(line(1)), "s"(line(2)), "s"(line(3)), "s"(line(4)),
                 "s"(line(5)));
  }
  if (threadIdx.x == 0) *run.taken = first_taken;
  // tiles16 / panels, of the fewest panels that hold them
  const int share = panels == 1 ? tiles16 : kPanelTiles16 - (tiles16 < kPanelTiles16 * panels);
  const int larger = tiles16 - share * panels;
  struct Task {
    int number, stage, panel, tn;
  };
  auto task_of = [&](int number, Plan* plan) {
    const int stage = (number >= ff1_at) + (number >= ff2_at) + (number >= qkv_at);
    const unsigned at =
        number - (stage < 2 ? (stage == 0 ? 0 : ff1_at) : stage == 2 ? ff2_at : qkv_at);
    const Layer::Product& product = arguments().product[stage];
    const Divided by_tasks = divide(at, product.tasks, product.inverse);
    const int panel = by_tasks.quotient, tn = by_tasks.rest, wave = run.wave();
    const int col0 = tn * product.columns + (stage & 1 ? (wave & 3) * kUnitCols : 0);
    // a sum's waves share the depth, a norm's two halves
    const int first = stage == 0 ? wave : (stage == 2 ? wave : wave >> 2) * kUnits4;
    *plan = plan_of(product.W + (size_t)col0 * product.ld, product.ld, first,
                    stage == 0 ? 1 : kUnits4, thread_of_task() & 63);
    return Task{number, stage, panel, tn};
  };
  block_sync();
  const int number = (int)(__builtin_amdgcn_readfirstlane(*run.taken) - before);
  if (number >= tasks) return;
  Plan plan;
  Task task = task_of(number, &plan);
#pragma unroll
  for (int u = 0; u < kUnits4; ++u) issue_unit(plan, u, run.own() + u * kUnitBytes);
  block_sync();                          // everyone knows its task
  while (true) {
    const Layer& a = arguments();
    const int tn = task.tn, p = task.panel;
    const int from16 = first16 + p * share + (p < larger ? p : larger);
    const int end = (from16 + share + (p < larger ? 1 : 0)) * 16;
    const Panel panel = {from16 * 16, (end < a.rows ? end : a.rows) - from16 * 16};
    uint32_t* const counters = a.counters + (size_t)(kGroups + (group * a.panels + p) * 3) * kLine;
    const uint32_t times = layer + 1;
    Task coming = {tasks, 0, 0, 0};
    Plan then = {};
    auto look_ahead = [&]() {
      coming.number = (int)(__builtin_amdgcn_readfirstlane(*run.taken) - before);
      if (coming.number >= tasks) return;
      coming = task_of(coming.number, &then);
    };
    // Once the stores are on their way the next weights follow them; wait_vm counts what may
    // still be in flight when the stores have arrived.
    auto stores_first = [] {
      asm volatile("" ::: "memory");
      __builtin_amdgcn_sched_barrier(0);
    };
    auto ahead_of_sum = [&](int step) {
      if (step == 0) return look_ahead();
      stores_first();
      if (then.units == kUnits4) {
#pragma unroll
        for (int u = 0; u < kUnits4 - 1; ++u)
          issue_unit(then, u, run.own() + kSumBytes + u * kUnitBytes);
        wait_vm<(kUnits4 - 1) * kUnitLoads>();
      } else {
        issue_unit(then, 0, run.own() + kSumBytes);
        wait_vm<0>();
      }
    };
    auto ahead_of_norm = [&](int step) {
      if (step == 0) return look_ahead();
      if (step == 1) {
        issue_unit(then, 0, lds + NormPlaces::of(0, run.wave()));
        issue_unit(then, 1, lds + NormPlaces::of(1, run.wave()));
        issue_half(then, 3, 0, lds + NormPlaces::of(3, run.wave()));
        return;
      }
      stores_first();
      if (then.units == kUnits4) {
        issue_unit(then, 2, lds + NormPlaces::of(2, run.wave()));
        issue_half(then, 3, 1, lds + NormPlaces::rest_of_last(run.wave()));
        wait_vm<kUnitLoads + kUnitLoads / 2>();
      } else {
        wait_vm<0>();
      }
    };
    const bool sum = (task.stage & 1) == 0;
    uint32_t* raise = nullptr;
    if (task.stage == 0) {
      residual_task<1, false>(run, plan, panel, tn, a.att, a.proj, nullptr, a.x, a.y1,
                              a.parts1, nullptr, 0, ahead_of_sum,
                              std::make_integer_sequence<int, 1>{});
      raise = counters;
    } else if (task.stage == 1) {
      const Shared x2(a.x2 + (size_t)panel.row0 * kD, panel.rows * kD * 2);
      const Shared out(a.h + (size_t)panel.row0 * a.inner, panel.rows * a.inner * 2);
      norm_task(
          run, panel, tn, a.product[1].tasks, a.y1, a.norm1, counters, times * kResTasks,
          [&](int r, int chunk, const u32x4& v) { x2.store16((r * kD + chunk * 8) * 2, v); },
          [&](int col) { return *reinterpret_cast<const u32x4*>(a.ff1_b + col); },
          [&](int r, int col, f32x4 left, f32x4 right, const u32x4& bias) {
            left += unpack_bf16x4(u32x2{bias[0], bias[1]});
            right += unpack_bf16x4(u32x2{bias[2], bias[3]});
#pragma unroll
            for (int e = 0; e < 4; ++e) {                      // a NaN stays one
              left[e] = left[e] < 0.0f ? 0.0f : left[e];
              right[e] = right[e] < 0.0f ? 0.0f : right[e];
            }
            out.store16((r * a.inner + col) * 2, pack_bf16x8(left, right));
          },
          ahead_of_norm);
      raise = counters + kLine;
    } else if (task.stage == 2) {
      residual_task<kUnits4, true>(run, plan, panel, tn, a.h, a.inner, a.ff2_b, a.x2, a.y2,
                                   a.parts2, counters + kLine, times * a.product[1].tasks,
                                   ahead_of_sum, std::make_integer_sequence<int, kUnits4>{});
      raise = counters + 2 * kLine;
    } else {
      norm_task(
          run, panel, tn, a.product[3].tasks, a.y2, a.norm2, counters + 2 * kLine,
          times * kResTasks,
          [&](int r, int chunk, const u32x4& v) { put_row(a.rows_out, panel.row0 + r, chunk, v); },
          [&](int col) { return a.qkv.needs(col); },
          [&](int r, int col, const f32x4& left, const f32x4& right, const QkvEpi::Needs& biases) {
            if (r < panel.rows) a.qkv(panel.row0 + r, col, left, right, biases);
          },
          ahead_of_norm);
    }
    block_sync();                        // every wave's stores have arrived
    if (raise && threadIdx.x == 0)
      __hip_atomic_fetch_add(raise, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (coming.number >= tasks) return;
    // the sums have been read: room for the last unit
    if (sum) issue_unit(then, kUnits4 - 1, run.own());
    run.place = sum ? Place::kBehindSum : Place::kBehindNorm;
    task = coming;
    plan = then;
  }
}

// hidden = LN(y), one wave for four rows.
__global__ __launch_bounds__(kThreads) void txl_norm_kernel(const float* y, Norm norm,
                                                            uint16_t* hidden, int M) {
  const int row = blockIdx.x * (kThreads / 16) + (threadIdx.x >> 4);
  const int at = row < M ? row : M - 1;
  NormRow in;
  NormWeights<4> weights;
  u32x4 v[4];
  in.load(y, norm, at, threadIdx.x & 15);
  weights.load(norm, threadIdx.x & 15);
  norm_row(in, weights, norm.eps, v);
  if (row >= M) return;
#pragma unroll
  for (int j = 0; j < 4; ++j)
    *reinterpret_cast<u32x4*>(hidden + (size_t)row * kD + ((threadIdx.x & 15) + 16 * j) * 8) = v[j];
}

// table[distance] = [sin, cos](distance * 10000^(-2c/512)), bf16; and the counters at zero.
__global__ __launch_bounds__(kD / 2) void txl_positions_kernel(uint16_t* table,
                                                               uint32_t* counters, int count) {
  const int c = threadIdx.x;
  for (int i = blockIdx.x * (kD / 2) + c; i < count; i += gridDim.x * (kD / 2)) counters[i] = 0;
  const double rate = exp2(-13.287712379549449391 * (2.0 * c / kD));   // log2(10000)
  const double angle = blockIdx.x * rate;
  const uint32_t v = pack_bf16((float)sin(angle), (float)cos(angle));
  table[(size_t)blockIdx.x * kD + c] = (uint16_t)v;
  table[(size_t)blockIdx.x * kD + kD / 2 + c] = (uint16_t)(v >> 16);
}

// Relative attention of 32 queries of one head of one sequence.
//
//   score(i, j) = ((q_i + u) k_j + (q_i + v) r_(m + i - j)) / 8,   j <= m + i
//
// with m rows of memory in front of the segment.  Eight waves: wave w takes
// queries 16 (w % 2) .. + 15 and one quarter of each stage of 128 keys (online
// softmax; the quarters meet in LDS at the end).  K and R are the first
// MFMA operand, so a lane's values belong to ONE query (lane % 16) and to four
// consecutive keys or distances: the softmax needs two swaps of lanes a maximum, and the
// probabilities are already where the second product wants its operand, given V
// transposed and its keys taken in the same order.
//
// The shift by relative distance is a shear: the wave computes the 48 distances
// that its 16 x 32 block of pairs touches, keeps them in LDS as fp32 and each lane
// picks entry (query - key + 31) of its row.  A stage's R rows are the 160
// distances from the workgroup's first query to the stage's last key on.
//
// Bound by LDS and by the softmax's arithmetic, of two waves a SIMD: at batch 4 (192
// workgroups, 384 keys, 3 stages) a stage takes 1.6 us of every wave and a
// launch 8.0; with 64 queries a workgroup, 96 of them, 2.1 and 10.1.  The next stage's rows
// travel through registers while this one is worked on.  The arguments that the first stage's
// loads need are the leading ones, which arrive in registers (fourteen of them); the queries
// are asked for behind those loads (a batch-4 request 658 us so, 671 with a wait for arguments
// before the first load and two divisions there; batch 1, 16 tokens 515 and 520).
constexpr int kAttnThreads = 512;
constexpr int kQ = 32, kKeys = 128;
constexpr int kParts4 = 4, kPartKeys = kKeys / kParts4;
constexpr int kDistances = kQ + kKeys;         // a stage's R rows
constexpr int kVtRow = (kKeys / 2 + 2) * 4;    // bytes of a row of V transposed
constexpr int kShearRow = 52;                  // floats of a row of position scores
constexpr int kAttnR = kKeys * kRowBytes;
constexpr int kAttnV = kAttnR + kDistances * kRowBytes;
constexpr int kAttnShear = kAttnV + kHead * kVtRow;
constexpr int kAttnLds = kAttnShear + 8 * 16 * kShearRow * 4;
constexpr int kMeetRow = 20;                   // floats a lane leaves at the end
static_assert(8 * 64 * kMeetRow * 4 <= kAttnLds, "in place of the stage");
constexpr size_t kAttnMost = (1u << 23) - 1024;   // workgroups: a grid has less than 2^32 threads

// Weights of the launches that follow, read by workgroups of their own on compute units
// that attention leaves idle, so that they come from the memory-side cache then: a
// request's vocabulary has pushed them out since they were last used.  A layer launch reads its
// weights a task ahead, but its first ones and each product's would come from memory.  us a
// request so and without: batch 4, 192 tokens 688 and 712, 2 x 192 650 and 675, 1 x 64 579 and
// 608, 1 x 16 without memory 530 and 528.  Each of these workgroups reads 192 KiB, about what
// fits attention's time: 32 of them a layer of the client's, more for wider ones while units
// are left (at an inner width of 65536, two layers, batch 4 797 so and 805 without, 1 x 64 462
// and 457).  How many follows attention's size alone, not the compute units of the stream: they
// are the last of the grid, and on streams of 32 to 128 units, where they wait for attention's
// own, requests take between 4 % less (2 x 192 on 64) and 6 % more (2 x 64 on 32) time than
// without.  Beside a GEMM or a triad on another stream (16 pairs of masks and sizes) they take
// between 3 % less and 8 % more, the other's rate is the same within 4 %.
constexpr uint32_t kTouchBytes = 192 << 10, kUnits = 256;
struct Coming {
  const uint16_t* p[4];
  uint32_t bytes[4];                   // multiples of 16
};
__device__ __forceinline__ void touch(const Coming& coming, uint32_t first_block) {
  constexpr uint32_t kEach = kAttnThreads * 16, kUnroll = 4;
  const uint32_t step = (gridDim.x - first_block) * kEach;
  const uint32_t mine = (blockIdx.x - first_block) * kEach + threadIdx.x * 16;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const char* p = reinterpret_cast<const char*>(coming.p[i]);
    for (uint32_t at = mine; at < coming.bytes[i]; at += kUnroll * step) {
      u32x4 v[kUnroll];
#pragma unroll
      for (uint32_t u = 0; u < kUnroll; ++u) {
        const uint32_t to = at + u * step;
        v[u] = *reinterpret_cast<const u32x4*>(p + (to < coming.bytes[i] ? to : at));
      }
#pragma unroll
      for (uint32_t u = 0; u < kUnroll; ++u) asm volatile("" ::"v"(v[u]));
    }
  }
}

__global__ __launch_bounds__(kAttnThreads, 1) void txl_attention_kernel(
    const uint16_t* __restrict__ kv_mem, const uint16_t* __restrict__ kv_x,
    const uint16_t* __restrict__ r, int qlen, int mlen, int batch, int heads, uint32_t first,
    uint32_t own, uint32_t inverse_heads, uint32_t inverse_batch,
    const uint16_t* __restrict__ qu, const uint16_t* __restrict__ qv, uint16_t* __restrict__ out,
    Coming coming) {
  __shared__ __attribute__((aligned(16))) unsigned char lds[kAttnLds];
  if (blockIdx.x >= own) {
    touch(coming, own);
    return;
  }
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l16 = lane & 15, lq = lane >> 4;
  const uint32_t block = first + blockIdx.x;
  const Divided by_heads = divide(block, heads, inverse_heads);
  const Divided by_batch = divide(by_heads.quotient, batch, inverse_batch);
  const int head = by_heads.rest, b = by_batch.rest;
  const int q0 = by_batch.quotient * kQ;
  const int klen = mlen + qlen;
  const int proj = heads * kHead;
  const int qt = wave & 1, part = wave >> 1;

  const size_t key_step = (size_t)batch * (2 * proj);
  const uint16_t* in_mem = kv_mem + (size_t)b * (2 * proj) + head * kHead;
  const uint16_t* in_x = kv_x + (size_t)b * (2 * proj) + head * kHead;
  auto key_row = [&](int j) {
    j = j < klen ? j : klen - 1;
    return j < mlen ? in_mem + (unsigned)j * key_step : in_x + (unsigned)(j - mlen) * key_step;
  };
  // this thread's share of a stage
  u32x4 nk[2], nr[3], nv[2];
  auto fetch = [&](int j0) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int u = i * kAttnThreads + threadIdx.x;
      nk[i] = *reinterpret_cast<const u32x4*>(key_row(j0 + (u >> 3)) + (u & 7) * 8);
    }
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      const int u = i * kAttnThreads + threadIdx.x;
      if (u >= kDistances * 8) break;
      int d = mlen + q0 - (j0 + kKeys - 1) + (u >> 3);
      d = d < 0 ? 0 : d < klen ? d : klen - 1;
      nr[i] = *reinterpret_cast<const u32x4*>(r + (size_t)d * proj + head * kHead + (u & 7) * 8);
    }
#pragma unroll
    for (int i = 0; i < 2; ++i)
      nv[i] = *reinterpret_cast<const u32x4*>(key_row(j0 + (threadIdx.x >> 3) * 2 + i) + proj +
                                              (threadIdx.x & 7) * 8);
  };
  auto put = [&]() {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int u = i * kAttnThreads + threadIdx.x, row = u >> 3;
      *reinterpret_cast<u32x4*>(lds + row * kRowBytes + (((u & 7) ^ (row & 7)) << 4)) = nk[i];
    }
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      const int u = i * kAttnThreads + threadIdx.x, row = u >> 3;
      if (u >= kDistances * 8) break;
      *reinterpret_cast<u32x4*>(lds + kAttnR + row * kRowBytes + (((u & 7) ^ (row & 7)) << 4)) =
          nr[i];
    }
    // two keys of a head column side by side
    unsigned char* vt = lds + kAttnV + (threadIdx.x & 7) * 8 * kVtRow + (threadIdx.x >> 3) * 4;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      *reinterpret_cast<uint32_t*>(vt + (2 * e) * kVtRow) =
          (nv[0][e] & 0xffffu) | (nv[1][e] << 16);
      *reinterpret_cast<uint32_t*>(vt + (2 * e + 1) * kVtRow) =
          (nv[0][e] >> 16) | (nv[1][e] & 0xffff0000u);
    }
  };

  fetch(0);
  __builtin_amdgcn_sched_barrier(0);
  const int qi = q0 + qt * 16 + l16;            // this lane's query
  bf16x8 fqu[2], fqv[2];
  {
    const int q = qi < qlen ? qi : qlen - 1;
    const size_t at = ((size_t)q * batch + b) * proj + head * kHead + lq * 8;
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      fqu[ks] = *reinterpret_cast<const bf16x8*>(qu + at + ks * 32);
      fqv[ks] = *reinterpret_cast<const bf16x8*>(qv + at + ks * 32);
    }
  }
  auto fragment = [&](int base, int row, int ks) {
    return *reinterpret_cast<const bf16x8*>(lds + base + row * kRowBytes +
                                            (((ks * 4 + lq) ^ (row & 7)) << 4));
  };
  float* shear = reinterpret_cast<float*>(lds + kAttnShear) + (wave * 16 + l16) * kShearRow;

  constexpr float kExp = 0.125f * 1.44269504088896340736f;   // 1 / sqrt(64), base 2
  const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
  f32x4 o[4] = {zero, zero, zero, zero};
  float m = -__builtin_inff(), l = 0.0f;
  const int last_query = q0 + kQ <= qlen ? q0 + kQ - 1 : qlen - 1;
  const int stages = (mlen + last_query) / kKeys + 1;
  for (int st = 0; st < stages; ++st) {
    const int j0 = st * kKeys;
    if (st > 0) block_sync();                   // everyone is done with the last stage
    put();
    block_sync();
    if (st + 1 < stages) fetch(j0 + kKeys);
    const int jw = j0 + kPartKeys * part;       // this wave's first key
    if (jw > mlen + q0 + qt * 16 + 15) continue;   // all of them in the future

    // Everything this wave takes from the stage, in one go: read one by one between the
    // MFMAs, each waits for LDS by itself (a stage took 1.5 us of which 0.1 are products).
    bf16x8 fr[3][2], fk[2][2];
    u32x2 fv[4][2];
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
#pragma unroll
      for (int t = 0; t < 3; ++t)
        fr[t][ks] = fragment(kAttnR, 16 * qt + 96 - kPartKeys * part + 16 * t + l16, ks);
#pragma unroll
      for (int t = 0; t < 2; ++t) fk[t][ks] = fragment(0, kPartKeys * part + 16 * t + l16, ks);
    }
#pragma unroll
    for (int d = 0; d < 4; ++d) {
      const unsigned char* vt =
          lds + kAttnV + (16 * d + l16) * kVtRow + (kPartKeys * part + lq * 4) * 2;
      fv[d][0] = *reinterpret_cast<const u32x2*>(vt);
      fv[d][1] = *reinterpret_cast<const u32x2*>(vt + 32);
    }
    __builtin_amdgcn_sched_barrier(0);
    f32x4 g[3] = {zero, zero, zero}, s[2] = {zero, zero};
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
#pragma unroll
      for (int t = 0; t < 3; ++t) g[t] = mfma(fr[t][ks], fqv[ks], g[t]);
#pragma unroll
      for (int t = 0; t < 2; ++t) s[t] = mfma(fk[t][ks], fqu[ks], s[t]);
    }
#pragma unroll
    for (int t = 0; t < 3; ++t) *reinterpret_cast<f32x4*>(shear + 16 * t + lq * 4) = g[t];
    // the rows of position scores cross lanes of this wave only
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront", "local");
    float by_distance[2][4];
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int e = 0; e < 4; ++e) by_distance[t][e] = shear[l16 + 31 - (16 * t + lq * 4 + e)];
    __builtin_amdgcn_sched_barrier(0);
    const int last = mlen + qi - jw - lq * 4;     // of this lane's keys, counted from its first
    float top = -__builtin_inff();
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float v = s[t][e] + by_distance[t][e];
        s[t][e] = 16 * t + e <= last ? v : -__builtin_inff();
        top = __builtin_fmaxf(top, s[t][e]);
      }
    top = max_over_rows(top);
    const float m_new = __builtin_fmaxf(m, top);
    const float base = m_new == -__builtin_inff() ? 0.0f : m_new;
    const float scale = __builtin_amdgcn_exp2f((m - base) * kExp);
    m = m_new;
    l *= scale;
#pragma unroll
    for (int d = 0; d < 4; ++d) o[d] *= scale;
    u32x4 p;
#pragma unroll
    for (int t = 0; t < 2; ++t) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        s[t][e] = __builtin_amdgcn_exp2f((s[t][e] - base) * kExp);
        l += s[t][e];
      }
      p[2 * t] = pack_bf16(s[t][0], s[t][1]);
      p[2 * t + 1] = pack_bf16(s[t][2], s[t][3]);
    }
#pragma unroll
    for (int d = 0; d < 4; ++d) {
      const u32x4 f = {fv[d][0][0], fv[d][0][1], fv[d][1][0], fv[d][1][1]};
      o[d] = mfma(__builtin_bit_cast(bf16x8, f), __builtin_bit_cast(bf16x8, p), o[d]);
    }
  }
  // l holds this lane's keys only
  l = sum_over_rows(l);
  block_sync();
  // the quarters meet: wave (qt, part) finishes head columns 16 * part .. + 15
  float* meet = reinterpret_cast<float*>(lds);
  {
    float* mine = meet + (wave * 64 + lane) * kMeetRow;
    mine[0] = m;
    mine[1] = l;
#pragma unroll
    for (int d = 0; d < 4; ++d) *reinterpret_cast<f32x4*>(mine + 4 + d * 4) = o[d];
  }
  block_sync();
  if (qi >= qlen) return;
  float ms[kParts4], top = -__builtin_inff();
#pragma unroll
  for (int p = 0; p < kParts4; ++p) {
    ms[p] = meet[((p * 2 + qt) * 64 + lane) * kMeetRow];
    top = __builtin_fmaxf(top, ms[p]);
  }
  float all = 0.0f;
  f32x4 sum = zero;
#pragma unroll
  for (int p = 0; p < kParts4; ++p) {
    const float* of = meet + ((p * 2 + qt) * 64 + lane) * kMeetRow;
    const float a = ms[p] == top ? 1.0f : __builtin_amdgcn_exp2f((ms[p] - top) * kExp);
    all = __builtin_fmaf(of[1], a, all);
    sum += *reinterpret_cast<const f32x4*>(of + 4 + part * 4) * a;
  }
  store_bf16x4(out + ((size_t)qi * batch + b) * proj + head * kHead + 16 * part + lq * 4,
               sum * (1.0f / all));
}

// ---------------------------------------------------------------------------
// Adaptive softmax losses.  The logits (n x 267,735 at the client's vocabulary)
// never reach memory: a workgroup takes 256 rows and a chunk of a cluster's columns, in
// tiles of 64, and leaves one (reference, sum of exponentials) pair a row; the last
// kernel joins a row's pairs and computes the target's own logits and the head's entries
// for the tails as plain dot products.

constexpr int kMaxTails = 7;
constexpr int kCritM = 256, kCritN = 64, kCritStages = 16;
constexpr int kCritWaveM = kCritM / 4;
constexpr int kCritLeast = 4, kCritMost = 64;    // tiles of a chunk
constexpr int kCritBlocks = 256;                 // one a compute unit
constexpr int kGroupThreads = 1024;

// The work as it turns out on the device: every cluster's columns in chunks of the same
// number of tiles, an item for each chunk and 256 rows.
struct CritPlan {
  int chunk;                       // tiles
  int chunks[kMaxTails + 1];       // of the head and of each tail
  int row_tiles[kMaxTails + 1];
  int first_item[kMaxTails + 2];
};

struct Crit {
  const uint16_t* hidden;          // [n, 512]
  const uint16_t *weight, *bias;   // [n_token, 512], [n_token]
  const uint16_t *tail_weight, *tail_bias;   // the head's entries for the tails
  const int64_t* target;
  int n, tails;
  int edge[kMaxTails + 2];         // 0, cutoffs, n_token
  int least;                       // tiles of a chunk, at least
  int stride[kMaxTails + 1];       // chunks that a row's pairs have room for
  // workspace
  CritPlan* plan;
  int* count;                      // [tails] rows of each tail
  int* place;                      // [n] a row's place within its tail
  int* rows;                       // [tails][n] the rows, in order
  float2* pairs[kMaxTails + 1];    // [rows][stride]
};

// Tail of a target (0: in the head or outside the vocabulary).
__device__ __forceinline__ int tail_of(const Crit& c, int64_t t) {
  int tail = 0;
  for (int k = 1; k <= c.tails; ++k)
    if (t >= c.edge[k] && t < c.edge[k + 1]) tail = k;
  return tail;
}

// One workgroup: the rows of every tail, in their order, and the plan: chunks of the fewest
// tiles that leave no more items than compute units (an item starts with its rows, 7 us,
// and a second round of a few takes as long as the first).
__global__ __launch_bounds__(kGroupThreads) void crit_group_kernel(Crit c) {
  constexpr int kWaves = kGroupThreads / 64;
  __shared__ int wave_count[kMaxTails][kWaves];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  int seen[kMaxTails] = {0};
  for (int base = 0; base < c.n; base += kGroupThreads) {
    const int row = base + threadIdx.x;
    const int tail = row < c.n ? tail_of(c, c.target[row]) : 0;
    int before = 0;
#pragma unroll
    for (int k = 1; k <= kMaxTails; ++k) {
      if (k > c.tails) break;
      const uint64_t mine = __ballot(tail == k);
      if (tail == k) before = __popcll(mine & ((1ull << lane) - 1));
      if (lane == 0) wave_count[k - 1][wave] = __popcll(mine);
    }
    __syncthreads();
#pragma unroll
    for (int k = 1; k <= kMaxTails; ++k) {
      if (k > c.tails) break;
      int at = seen[k - 1], all = 0;
      for (int w = 0; w < kWaves; ++w) {
        if (w < wave) at += wave_count[k - 1][w];
        all += wave_count[k - 1][w];
      }
      if (tail == k) {
        c.place[row] = at + before;
        c.rows[(size_t)(k - 1) * c.n + at + before] = row;
      }
      seen[k - 1] += all;
    }
    __syncthreads();
  }
  if (threadIdx.x >= 64) return;
  int row_tiles[kMaxTails + 1], cols[kMaxTails + 1];
  int64_t all = 0;
  const int mine = c.least + lane;                 // tiles: every lane tries another number
  static_assert(kCritMost - kCritLeast < 64, "a lane for each");
#pragma unroll
  for (int k = 0; k <= kMaxTails; ++k) {
    const int rows = k == 0 ? c.n : k <= c.tails ? seen[k > 0 ? k - 1 : 0] : 0;
    if (k > 0 && k <= c.tails && lane == 0) c.count[k - 1] = rows;
    row_tiles[k] = (rows + kCritM - 1) / kCritM;
    cols[k] = k <= c.tails ? (c.edge[k + 1] - c.edge[k] + kCritN - 1) / kCritN : 0;
    all += (int64_t)row_tiles[k] * ((cols[k] + mine - 1) / mine);
  }
  const uint64_t enough = __ballot(all <= kCritBlocks || mine >= kCritMost);
  const int chunk = c.least + __builtin_ctzll(enough);   // the last lane's is past kCritMost
  if (lane != 0) return;
  CritPlan& plan = *c.plan;
  plan.chunk = chunk;
  int items = 0;
#pragma unroll
  for (int k = 0; k <= kMaxTails; ++k) {
    plan.chunks[k] = (cols[k] + chunk - 1) / chunk;
    plan.row_tiles[k] = row_tiles[k];
    plan.first_item[k] = items;
    items += row_tiles[k] * ((cols[k] + chunk - 1) / chunk);
  }
  plan.first_item[kMaxTails + 1] = items;
}

// Wave w owns rows 64 w .. + 63 (or 32 w .. + 31 of an item of up to 128 rows), whose 512
// elements stay in registers (all 256 accumulator ones), and all 64 columns of a tile; only
// the weights go through LDS, sixteen k-tiles ahead and from one column tile straight on to
// the next.  A wave reads one fragment for four products (with 32 rows a wave, two, LDS reads
// alone took as long as the products), a barrier stands between two k-tiles of sixty-four,
// and the epilogue is six instructions an element: the bias is one more product behind the
// others (in front of them every partial sum would be rounded at its magnitude), and the
// exponentials are taken against the lane's first tile's maximum, which is only replaced
// when a sum gets out of hand.  A batch-4 request's logits take 101 us, in which the matrix
// cores are busy for half of the time and 306 MB are read; 155 with 128 rows a workgroup,
// tiles of 128 columns one after the other and chunks of eight.  What stays of a lane's
// values does not fit the registers: eight of them lie in scratch, written once and read at
// most twice an item, outside the loop over the tiles.
__device__ __forceinline__ void mfma_by_kept(const bf16x8& a, const bf16x8& kept, f32x4& c) {
  asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+v"(c) : "v"(a), "a"(kept));
}
__device__ __forceinline__ void first_by_kept(const bf16x8& a, const bf16x8& kept, f32x4& c) {
  asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, 0" : "=&v"(c) : "v"(a), "a"(kept));
}

template <int I, int J>
__device__ __forceinline__ void settle_vector(f32x4 (&acc)[I][J]) {   // mfma_tile.h's settle
#pragma unroll
  for (int i = 0; i < I; ++i)
#pragma unroll
    for (int j = 0; j < J; ++j) asm volatile("" : "+v"(acc[i][j]));
  asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");
#pragma unroll
  for (int i = 0; i < I; ++i)
#pragma unroll
    for (int j = 0; j < J; ++j) asm volatile("" : "+v"(acc[i][j]));
}

template <int kWaveM>
__device__ __forceinline__ void crit_item(const Crit& c, unsigned char* lds, int k, int chunk,
                                          int row0, int rows, int width) {
  constexpr int NS = kCritStages, kStage = Rows<kCritN>::kBytes, kLoads = Rows<kCritN>::kLoads;
  constexpr int kI = kWaveM / 16, kJ = kCritN / 16, kM = 2 * kI * kJ;   // products a k-tile
  static_assert(NS == 2 * kPanelTiles && kPanelTiles % 2 == 0, "the order of the loads");
  static_assert(kCritMost * kCritN * 2 <= 4 * kWaveM * kRowBytes, "the biases' place");
  const int* list = k == 0 ? nullptr : c.rows + (size_t)(k - 1) * c.n;
  const int lo = c.edge[k] + chunk * width;                  // this chunk's tokens
  const int left = c.edge[k + 1] - lo;
  const int tokens = left < width ? left : width;
  const int tiles = (tokens + kCritN - 1) / kCritN;
  const int last_token = lo + tokens - 1;

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l16 = lane & 15, lq = lane >> 4;
  // rows of weights past the chunk are its last one again (masked below)
  struct Source {
    const uint16_t* p[kLoads];
  };
  auto source = [&](int tile) {
    Source s;
#pragma unroll
    for (int i = 0; i < kLoads; ++i) {
      int token = lo + tile * kCritN + (i * 4 + wave) * 8 + (lane >> 3);
      token = token < last_token ? token : last_token;
      s.p[i] = c.weight + (size_t)token * kD + ((lane & 7) ^ (lane >> 3)) * 8;
    }
    return s;
  };
  auto issue_one = [&](const Source& s, int i, int kt, int stage) {
    load_to_lds(s.p[i] + kt * kTileK, lds + stage * kStage + (i * 4 + wave) * 1024);
  };
  {
    const Source s0 = source(0), s1 = source(1);
#pragma unroll
    for (int q = 0; q < NS - 1; ++q)
#pragma unroll
      for (int i = 0; i < kLoads; ++i)
        issue_one(q < kPanelTiles ? s0 : s1, i, q % kPanelTiles, q);
    __builtin_amdgcn_sched_barrier(0);
  }
  // the chunk's biases: loads of them in the loop would be waited for together with every
  // other load in flight
  constexpr int kBiasLoads = kCritMost * kCritN / kThreads;
  uint16_t bias_line[kBiasLoads];

  // The wave's rows, by whole lines, and through LDS into the fragments' order.
  unsigned char* own = lds + NS * kStage + wave * kWaveM * kRowBytes;
  bf16x8 fa[kI][2 * kPanelTiles];
  {
    int from[kWaveM / 8];
#pragma unroll
    for (int g = 0; g < kWaveM / 8; ++g) {
      const int at = row0 + wave * kWaveM + g * 8 + (lane >> 3);
      from[g] = at < rows ? at : rows - 1;
    }
    if (list) {
#pragma unroll
      for (int g = 0; g < kWaveM / 8; ++g) from[g] = list[from[g]];
    }
    constexpr int kHalf = kPanelTiles / 2, kLines = kWaveM / 8;
    u32x4 line[kHalf][kLines];                      // half of the k-tiles at a time
    auto load = [&](int kt, int g) {
      line[kt % kHalf][g] = *reinterpret_cast<const u32x4*>(
          c.hidden + (size_t)from[g] * kD + ((lane & 7) ^ (lane >> 3)) * 8 + kt * kTileK);
    };
#pragma unroll
    for (int g = 0; g < kLines; ++g) {
#pragma unroll
      for (int kt = 0; kt < kHalf; ++kt) load(kt, g);
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int b = 0; b < kBiasLoads; ++b) {
      const int token = lo + b * kThreads + threadIdx.x;
      bias_line[b] = c.bias[token < last_token ? token : last_token];
    }
#pragma unroll
    for (int kt = 0; kt < kPanelTiles; ++kt) {
#pragma unroll
      for (int g = 0; g < kLines; ++g)
        *reinterpret_cast<u32x4*>(own + g * 8 * kRowBytes + lane * 16) = line[kt % kHalf][g];
#pragma unroll
      for (int i = 0; i < kI; ++i)
#pragma unroll
        for (int ks = 0; ks < 2; ++ks)
          fa[i][kt * 2 + ks] = *reinterpret_cast<const bf16x8*>(
              own + (i * 16 + l16) * kRowBytes + (((ks * 4 + lq) ^ (l16 & 7)) << 4));
      if (kt == kHalf - 1) {
#pragma unroll
        for (int next = kHalf; next < kPanelTiles; ++next)
#pragma unroll
          for (int g = 0; g < kLines; ++g) load(next, g);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  block_sync();
  uint16_t* biases = reinterpret_cast<uint16_t*>(lds + NS * kStage);   // in the rows' place
#pragma unroll
  for (int b = 0; b < kBiasLoads; ++b) biases[b * kThreads + threadIdx.x] = bias_line[b];
  bf16x8 fb[2][2 * kJ];                             // [even, odd k-tile][k-step, columns]
  // from here on a read is an offset from one of four addresses
  const unsigned char* place[2][2];
#pragma unroll
  for (int half = 0; half < 2; ++half)
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
      place[half][ks] = lds + half * kPanelTiles * kStage + l16 * kRowBytes +
                        (((ks * 4 + lq) ^ (l16 & 7)) << 4);
  auto read_one = [&](auto odd, int r, int stage) {
    fb[decltype(odd)::value][r] = *reinterpret_cast<const bf16x8*>(
        place[stage / kPanelTiles][r / kJ] + stage % kPanelTiles * kStage +
        r % kJ * 16 * kRowBytes);
  };
  wait_vm<0>();
  block_sync();
#pragma unroll
  for (int r = 0; r < 2 * kJ; ++r) read_one(std::integral_constant<int, 0>{}, r, 0);

  constexpr float kLog2e = 1.44269504088896340736f;
  const float kNone = -__builtin_inff();
  float ref[kI], sum[kI];
  float base[kI];                                   // the reference, or 0 without one
#pragma unroll
  for (int i = 0; i < kI; ++i) {
    ref[i] = kNone;
    sum[i] = base[i] = 0.0f;
  }
  // The bias is a product by a row of ones: only the first of a fragment's 32 elements
  // counts, lane group 0's first.
  const u32x4 one = {lq == 0 ? 0x3f80u : 0u, 0, 0, 0};
  const uint32_t first = lq == 0 ? 0xffffu : 0u;
  uint32_t bias[kJ];
  auto read_bias = [&](int tile) {
#pragma unroll
    for (int j = 0; j < kJ; ++j) bias[j] = biases[tile * kCritN + j * 16 + l16];
  };
  auto term = [&](float v, int i) { return __builtin_amdgcn_exp2f((v - base[i]) * kLog2e); };
  // a tile's exponentials `part` (a lane's own columns; lanes meet at the end) to the sums;
  // without a reference, or with one so far below that the sum might overflow, they are
  // taken again against a new one
  auto take = [&](const f32x4 (&acc)[kI][kJ], float (&part)[kI]) {
#pragma unroll
    for (int i = 0; i < kI; ++i) {
      if (__any(ref[i] == kNone || part[i] > 0x1p60f)) {
        float m = ref[i];
#pragma unroll
        for (int j = 0; j < kJ; ++j)
#pragma unroll
          for (int e = 0; e < 4; ++e) m = __builtin_fmaxf(m, acc[i][j][e]);
        base[i] = m == kNone ? 0.0f : m;
        sum[i] *= term(ref[i], i);
        ref[i] = m;
        part[i] = 0.0f;
#pragma unroll
        for (int j = 0; j < kJ; ++j)
#pragma unroll
          for (int e = 0; e < 4; ++e) part[i] += term(acc[i][j][e], i);
      }
      sum[i] += part[i];
    }
  };
  Source next = source(1);
  // Tile t's products, between them the exponentials of the tile before.
  auto tile = [&](int t, auto parity, f32x4 (&acc)[kI][kJ], f32x4 (&old)[kI][kJ]) {
    constexpr int half = decltype(parity)::value ? kPanelTiles : 0;   // this tile's first stage
    const Source after = source(t + 2);
    float part[kI], one_term = 0.0f;
#pragma unroll
    for (int i = 0; i < kI; ++i) part[i] = 0.0f;
    // k-tiles 2 * pair and the next.  Behind the barrier every wave has read the first of
    // them and the two after it have landed, so the stage before them and the first one's
    // are filled again; twelve k-tiles may be in flight.
    auto step = [&](auto pair_c) {
      constexpr int kFirst = decltype(pair_c)::value * 2;
      wait_vm<kLoads*(NS - 4)>();
      block_sync();
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int kt = kFirst + h;
#pragma unroll
        for (int m = 0; m < kM; ++m) {
          const int ks = m / (kI * kJ), i = m / kJ % kI, j = m % kJ;
          if (kt == 0 && ks == 0) first_by_kept(fb[h][j], fa[i][0], acc[i][j]);
          else mfma_by_kept(fb[h][ks * kJ + j], fa[i][kt * 2 + ks], acc[i][j]);
          // the next k-tile's fragments, in the first three quarters
          const bool reads = kI == 4 ? m % 3 == 1 : m % 3 != 1;
          const int r = kI == 4 ? m / 3 : m - (m + 2) / 3;
          if (reads && r < 2 * kJ) {
            const int stage = kt + 1 < kPanelTiles ? half + kt + 1 : kPanelTiles - half;
            if (h == 0) read_one(std::integral_constant<int, 1>{}, r, stage);
            else read_one(std::integral_constant<int, 0>{}, r, stage);
          }
          if (h == 0 && m % (kM / 4) == kI / 2) {
            const int x = m / (kM / 4);             // two loads for each stage
            if (x < kLoads) {
              if (kFirst == 0) issue_one(next, x, kPanelTiles - 1, 2 * kPanelTiles - half - 1);
              else issue_one(after, x, kFirst - 1, half + kFirst - 1);
            } else {
              issue_one(after, x - kLoads, kFirst, half + kFirst);
            }
          }
          // an element of the old tile every four products, one instruction behind each of
          // them: in a row they would wait for each other
          const int at = kt * kM + m;
          static_assert(kPanelTiles * 2 == 4 * 4, "four products an element");
          const int x = at / 4, oi = x / (kJ * 4);
          if (at % 4 == 0) one_term = old[oi][x / 4 % kJ][x % 4] - base[oi];
          else if (at % 4 == 1) one_term *= kLog2e;
          else if (at % 4 == 2) one_term = __builtin_amdgcn_exp2f(one_term);
          else part[oi] += one_term;
          if (at % 4 < 3) asm volatile("" : "+v"(one_term));
          else asm volatile("" : "+v"(part[oi]));
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    };
    step(std::integral_constant<int, 0>{});
    read_bias(t);
    step(std::integral_constant<int, 1>{});
    step(std::integral_constant<int, 2>{});
    step(std::integral_constant<int, 3>{});
#pragma unroll
    for (int j = 0; j < kJ; ++j) {
      const u32x4 b = {bias[j] & first, 0, 0, 0};
#pragma unroll
      for (int i = 0; i < kI; ++i)
        asm volatile("s_nop 1\n\tv_mfma_f32_16x16x32_bf16 %0, %1, %2, %0"
                     : "+v"(acc[i][j]) : "v"(b), "v"(one));
    }
    next = after;
    take(old, part);
    // written before anything reads them: their exponentials start behind the next product
    asm volatile("s_nop 15" ::: "memory");
#pragma unroll
    for (int i = 0; i < kI; ++i)
#pragma unroll
      for (int j = 0; j < kJ; ++j) asm volatile("" : "+v"(acc[i][j]));
  };
  auto last_tile = [&](f32x4 (&acc)[kI][kJ]) {
    settle_vector(acc);
    float part[kI];
#pragma unroll
    for (int i = 0; i < kI; ++i) {
      part[i] = 0.0f;
#pragma unroll
      for (int j = 0; j < kJ; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int token = lo + (tiles - 1) * kCritN + j * 16 + lq * 4 + e;
          if (token > last_token) acc[i][j][e] = kNone;
          part[i] += term(acc[i][j][e], i);
        }
    }
    take(acc, part);
  };
  f32x4 even[kI][kJ], odd[kI][kJ];
#pragma unroll
  for (int i = 0; i < kI; ++i)
#pragma unroll
    for (int j = 0; j < kJ; ++j)       // before the first
      odd[i][j] = f32x4{kNone, kNone, kNone, kNone};
  int t = 0;
  for (; t + 1 < tiles; t += 2) {
    tile(t, std::integral_constant<int, 0>{}, even, odd);
    tile(t + 1, std::integral_constant<int, 1>{}, odd, even);
  }
  if (t < tiles) {
    tile(t, std::integral_constant<int, 0>{}, even, odd);
    last_tile(even);
  } else {
    last_tile(odd);
  }
  wait_vm<0>();                        // nothing lands in LDS that is no longer ours
#pragma unroll
  for (int i = 0; i < kI; ++i) {
    float m = ref[i], s = sum[i];
#pragma unroll
    for (int d = 16; d < 64; d <<= 1) {
      const float om = __shfl_xor(m, d), os = __shfl_xor(s, d);
      const float t = __builtin_fmaxf(m, om);
      s = s * (m == t ? 1.0f : __expf(m - t)) + os * (om == t ? 1.0f : __expf(om - t));
      m = t;
    }
    const int at = row0 + wave * kWaveM + i * 16 + l16;
    if (lq == 0 && at < rows) c.pairs[k][(size_t)at * c.stride[k] + chunk] = make_float2(m, s);
  }
}

__global__ __launch_bounds__(kThreads, 1) void crit_logits_kernel(Crit c) {
  // the stages, and 8 KiB for each wave's rows on their way to registers (one array: with
  // two the compiler waits for the loads in flight before every read)
  constexpr int kLds = kCritStages * Rows<kCritN>::kBytes + 4 * kCritWaveM * kRowBytes;
  __shared__ __attribute__((aligned(16))) unsigned char lds[kLds];
  auto uniform = [](int v) { return __builtin_amdgcn_readfirstlane(v); };
  const CritPlan& plan = *c.plan;
  const int items = uniform(plan.first_item[kMaxTails + 1]);
  for (int item = blockIdx.x; item < items; item += kCritBlocks) {
    int k = 0;
    while (k < c.tails && item >= uniform(plan.first_item[k + 1])) ++k;
    // eight chunks, then their next rows: an XCD (of eight, in turn) takes all the rows of a
    // chunk and brings its weights once
    const int local = item - uniform(plan.first_item[k]);
    const int row_tiles = uniform(plan.row_tiles[k]), width = uniform(plan.chunk) * kCritN;
    const int group = local / (8 * row_tiles), in_group = local % (8 * row_tiles);
    const int others = uniform(plan.chunks[k]) - group * 8, abreast = others < 8 ? others : 8;
    const int chunk = group * 8 + in_group % abreast;
    const int row0 = in_group / abreast * kCritM;
    const int rows = k == 0 ? c.n : uniform(c.count[k - 1]);
    // Rows that fit 128 are multiplied by 32 a wave.  By 64, half of them for nothing, a
    // request on a stream of few compute units waits for the products: 16 rows of the
    // client's vocabulary on 32 units 402 us, so 244; 64 units 209 and 131, 256 units 76 and
    // 57.  Rows that do not fit keep 64 a wave: by 32 their weights would come twice (256
    // rows on 32 units 589 with items of 128, 387 so).
    if (rows - row0 <= kCritM / 2) crit_item<kCritWaveM / 2>(c, lds, k, chunk, row0, rows, width);
    else crit_item<kCritWaveM>(c, lds, k, chunk, row0, rows, width);
    block_sync();                      // the next item's loads land where this one's were read
  }
}

// The pair of a row's pairs, by one wave; (maximum, sum) of the lanes' own to start.
__device__ __forceinline__ float join_pairs(const float2* pairs, int count, int lane, float top,
                                            float sum) {
  for (int i = lane; i < count; i += 64) {
    const float2 p = pairs[i];
    const float t = __builtin_fmaxf(top, p.x);
    sum = sum * (top == t ? 1.0f : __expf(top - t)) + p.y * (p.x == t ? 1.0f : __expf(p.x - t));
    top = t;
  }
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const float ot = __shfl_xor(top, d), os = __shfl_xor(sum, d);
    const float t = __builtin_fmaxf(top, ot);
    sum = sum * (top == t ? 1.0f : __expf(top - t)) + os * (ot == t ? 1.0f : __expf(ot - t));
    top = t;
  }
  return top + logf(sum);
}

// weight . x + bias by one wave, eight elements of the row a lane.
__device__ __forceinline__ float logit_of(const uint16_t* weight, const uint16_t* bias,
                                          const u32x4& x, int lane) {
  const u32x4 w = *reinterpret_cast<const u32x4*>(weight + lane * 8);
  float s = 0.0f;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    s = __builtin_fmaf(bf16_lo(w[e]), bf16_lo(x[e]), s);
    s = __builtin_fmaf(bf16_hi(w[e]), bf16_hi(x[e]), s);
  }
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) s += __shfl_xor(s, d);
  return s + __builtin_bit_cast(float, (uint32_t)*bias << 16);
}

__global__ __launch_bounds__(kThreads) void crit_losses_kernel(Crit c, uint16_t* nll) {
  static_assert(kD == 64 * 8, "logit_of's row");
  const int lane = threadIdx.x & 63;
  const int row = blockIdx.x * (kThreads / 64) + (threadIdx.x >> 6);
  if (row >= c.n) return;
  const int64_t t = c.target[row];
  float loss = 0.0f;                               // a target outside the vocabulary: 0
  if (t >= 0 && t < c.edge[c.tails + 1]) {
    const u32x4 x = *reinterpret_cast<const u32x4*>(c.hidden + (size_t)row * kD + lane * 8);
    const int k = tail_of(c, t);
    const float own = logit_of(c.weight + (size_t)t * kD, c.bias + t, x, lane);
    // the head's entries for the tails: lane j starts from the j-th
    float head = own, top = -__builtin_inff(), sum = 0.0f;
    for (int j = 0; j < c.tails; ++j) {
      const float v = logit_of(c.tail_weight + (size_t)j * kD, c.tail_bias + j, x, lane);
      if (lane == j) {
        top = v;
        sum = v == -__builtin_inff() ? 0.0f : 1.0f;
      }
      if (j == k - 1) head = v;
    }
    // a NaN among them has to reach the sum: its maximum does not carry it
    if (top != top) {
      top = -__builtin_inff();
      sum = __builtin_nanf("");
    }
    loss = join_pairs(c.pairs[0] + (size_t)row * c.stride[0], c.plan->chunks[0], lane, top, sum) -
           head;
    if (k)
      loss += join_pairs(c.pairs[k] + (size_t)c.place[row] * c.stride[k], c.plan->chunks[k], lane,
                         -__builtin_inff(), 0.0f) -
              own;
  }
  if (lane == 0) nll[row] = (uint16_t)pack_bf16(loss, 0.0f);
}

// Pieces of a workspace, each in cache lines of its own whatever the workspace's alignment (16
// bytes at least): a layer launch's visibility needs that.  With no base only their sizes add up.
struct Pieces {
  static constexpr size_t kAlign = 128;
  char* base;
  size_t used = 0;
  explicit Pieces(void* workspace)
      : base((char*)(((uintptr_t)workspace + kAlign - 1) & ~(uintptr_t)(kAlign - 1))) {}
  size_t bytes() const { return used + kAlign - 16; }
  template <typename T>
  T* take(size_t count) {
    T* p = base ? reinterpret_cast<T*>(base + used) : nullptr;
    used += (count * sizeof(T) + 255) & ~(size_t)255;
    return p;
  }
};

size_t tiles(size_t n, size_t tile) { return (n + tile - 1) / tile; }

struct Buffers {
  uint16_t *x[2], *x2, *qu, *qv, *att, *h, *kv_x, *kv_mem, *table, *r;
  float *y, *y2;
  float2 *parts, *parts2;
  uint32_t* counters;
  size_t counts;
  size_t bytes;
};

// Panels of the largest of so many groups.
size_t group_panels(size_t rows, size_t groups) {
  return tiles(tiles(tiles(rows, 16), groups), kPanelTiles16);
}

// Groups of a layer launch, eight (an XCD each), four, two or one: those whose panels are the
// fewest, since a panel that is not full takes as long as a full one and reads all weights;
// as many as that allows.  us a request behind 192 tokens of memory on 32, 64, 128 and 256
// compute units, by eight groups (or as many as there are tiles of 16 rows) and so: batch 1, 64
// tokens 1120 and 880, 662 and 673, 580 and 590, 568 and 578; batch 2, 64 tokens 1618 and 1095,
// 944 and 710, 626 and 624, 600 and 598; batch 1, 192 tokens 1740 and 1311, 1017 and 767, 656
// and 646, 636 and 627; batch 3, 150 tokens 3350 and 2921, 1811 and 1618, 1060 and 959, 701
// and 701.  Three, five to seven groups are no better: XCDs share theirs unevenly.  Two or one
// are for rows that eight full panels hold: with more of them every XCD has work of every panel,
// and requests on the whole GPU take longer (by four groups and by one: batch 4, 100 tokens 617
// and 642, 120 tokens 635 and 682, batch 3, 160 tokens 641 and 709; batch 40, 200 tokens
// without memory 4539 and 4680).
size_t groups_of(size_t rows) {
  const bool few = rows <= kGroups * kPanelRows;
  size_t best = kGroups;
  for (size_t g = kGroups; g >= (few ? 1u : kGroups / 2); g /= 2)
    if (g * group_panels(rows, g) < best * group_panels(rows, best)) best = g;
  return best;
}

// Rows of one layer launch, a multiple of what full panels of all groups hold.  A launch cannot
// be held back once it has begun, and best-effort kernels run on budgets of 100 us and more, so
// none takes longer than that on the whole GPU: 3072 rows 79 us, 3840 96, 4608 114, 6144 145.
// What is cut off costs its beginning and end, us a request behind 192 tokens of memory in one
// launch a layer and so: batch 20 (3840 rows) 2555 and 2551, 21 2700 and 2884, 32 3877 and 4006,
// 40 4758 and 4888, 64 7556 and 7946.  A launch may be issued to another stream than its call
// names, so a stream's units are not asked: batch 4 takes 136 us a launch on 32 of them, 72 on
// 64.  (The logits' launch, which is not cut, takes 4 to 5 times as long as a layer's.)
constexpr size_t kFullRows = kGroups * kPanelRows, kLaunchRows = 10 * kFullRows;
size_t launch_rows(size_t rows) {
  return tiles(tiles(rows, tiles(rows, kLaunchRows)), kFullRows) * kFullRows;
}

// Counters of a layer launch of so many rows.
size_t counters_of(size_t rows) {
  const size_t groups = groups_of(rows);
  return kLine * (kGroups + 3 * groups * group_panels(rows, groups));
}

Buffers buffers_of(const orion_txl_dims& d, void* base) {
  const size_t rows = (size_t)d.q_len * d.batch, mem_rows = (size_t)d.m_len * d.batch;
  const size_t proj = (size_t)d.heads * kHead, k_len = (size_t)d.q_len + d.m_len;
  Pieces p(base);
  Buffers b;
  b.y = p.take<float>(rows * kD);
  b.parts = p.take<float2>(rows * kParts);
  b.y2 = p.take<float>(rows * kD);
  b.parts2 = p.take<float2>(rows * kParts);
  const size_t most = launch_rows(rows), rest = rows % most;
  b.counts = rows / most * counters_of(most) + (rest ? counters_of(rest) : 0);
  b.counters = p.take<uint32_t>(b.counts);
  b.x[0] = p.take<uint16_t>(rows * kD);
  b.x[1] = p.take<uint16_t>(rows * kD);
  b.x2 = p.take<uint16_t>(rows * kD);
  b.qu = p.take<uint16_t>(rows * proj);
  b.qv = p.take<uint16_t>(rows * proj);
  b.att = p.take<uint16_t>(rows * proj);
  b.h = p.take<uint16_t>(rows * d.inner);
  b.kv_x = p.take<uint16_t>(rows * 2 * proj);
  b.kv_mem = p.take<uint16_t>(d.layers * mem_rows * 2 * proj);
  b.table = p.take<uint16_t>(k_len * kD);
  b.r = p.take<uint16_t>(d.layers * k_len * proj);
  b.bytes = p.bytes();
  return b;
}

constexpr int kMostQueries = 65535 * 64;         // longer segments keep the operations

bool dims_fit(const orion_txl_dims& d) {
  return d.q_len > 0 && d.m_len >= 0 && d.batch > 0 && d.layers > 0 && d.heads > 0 &&
         d.heads % 2 == 0 && d.heads <= 1024 && d.inner > 0 && d.inner % 128 == 0 &&
         d.inner <= (1 << 20) && ((int64_t)d.q_len + d.m_len) * d.batch < (1 << 24) &&
         d.q_len <= kMostQueries;
}

bool lay_out(const orion_nll* a, void* base, Crit* c, size_t* bytes) {
  if (a->rows <= 0 || a->rows >= (1 << 24) || a->tails < 0 || a->tails > kMaxTails) return false;
  c->hidden = (const uint16_t*)a->hidden;
  c->weight = (const uint16_t*)a->weight;
  c->bias = (const uint16_t*)a->bias;
  c->tail_weight = (const uint16_t*)a->tail_weight;
  c->tail_bias = (const uint16_t*)a->tail_bias;
  c->target = (const int64_t*)a->target;
  c->n = a->rows;
  c->tails = a->tails;
  for (int k = 0; k <= a->tails + 1; ++k) {
    c->edge[k] = a->edges[k];
    if (k == 0 ? a->edges[0] != 0 : a->edges[k] <= a->edges[k - 1]) return false;
  }
  // every row is one of the head's, so chunks are at least as many tiles as its items ask for
  const size_t head = tiles(a->rows, kCritM) * tiles(a->edges[1], kCritN);
  const size_t least = tiles(head, kCritBlocks);
  c->least = (int)(least < kCritLeast ? kCritLeast : least > kCritMost ? kCritMost : least);
  Pieces p(base);
  c->plan = p.take<CritPlan>(1);
  c->count = p.take<int>(kMaxTails);
  c->place = p.take<int>(a->rows);
  c->rows = p.take<int>((size_t)a->tails * a->rows);
  for (int k = 0; k <= a->tails; ++k) {
    c->stride[k] = (int)tiles((size_t)c->edge[k + 1] - c->edge[k], kCritN * c->least);
    c->pairs[k] = p.take<float2>((size_t)a->rows * c->stride[k]);
  }
  *bytes = p.bytes();
  return true;
}

}  // namespace

extern "C" size_t orion_txl_workspace_bytes(const orion_txl_dims* dims) {
  return dims != nullptr && dims_fit(*dims) ? buffers_of(*dims, nullptr).bytes : 0;
}

extern "C" int orion_txl_hidden(const orion_txl_dims* dims, const orion_txl_layer* layers,
                                const void* u, const void* v, const void* x0, const void* mems,
                                size_t mem_stride, void* new_mems, size_t new_mem_stride,
                                int mem_rows_out, void* hidden, void* workspace,
                                size_t workspace_bytes, void* stream) {
  if (!dims || !layers || !u || !v || !x0 || !hidden || !workspace) return ORION_ERR_ARG;
  const orion_txl_dims& d = *dims;
  if (!dims_fit(d)) return ORION_ERR_SHAPE;
  if ((d.m_len > 0 && !mems) || (new_mems && (mem_rows_out <= 0 || mem_rows_out > d.q_len)))
    return ORION_ERR_ARG;
  uintptr_t all = (uintptr_t)u | (uintptr_t)v | (uintptr_t)x0 | (uintptr_t)mems |
                  (uintptr_t)new_mems | (uintptr_t)hidden | (uintptr_t)workspace |
                  (d.m_len > 0 ? mem_stride * 2 : 0) | (new_mems ? new_mem_stride * 2 : 0);
  for (int i = 0; i < d.layers; ++i) {
    const void* const* p = reinterpret_cast<const void* const*>(layers + i);
    for (size_t e = 0; e < sizeof(orion_txl_layer) / sizeof(void*); ++e) {
      if (!p[e]) return ORION_ERR_ARG;
      all |= (uintptr_t)p[e];
    }
  }
  if ((all & 15u) != 0) return ORION_ERR_ALIGN;
  if (workspace_bytes < buffers_of(d, nullptr).bytes) return ORION_ERR_ARG;

  const Buffers w = buffers_of(d, workspace);
  hipStream_t s = (hipStream_t)stream;
  const int rows = d.q_len * d.batch, mem_rows = d.m_len * d.batch, k_len = d.q_len + d.m_len;
  const int proj = d.heads * kHead;
  typedef const uint16_t* In;

  hipLaunchKernelGGL(txl_positions_kernel, dim3(k_len), dim3(kD / 2), 0, s, w.table,
                     w.counters, (int)w.counts);
  Jobs jobs;
  jobs.count = 0;
  uint64_t blocks = 0;
  auto flush = [&]() {
    if (jobs.count == 0) return;
    for (int i = jobs.count; i <= kMaxJobs; ++i) jobs.first_block[i] = (uint32_t)blocks;
    hipLaunchKernelGGL(txl_jobs_kernel, dim3((unsigned)blocks), dim3(kJobThreads), 0, s, jobs);
    jobs.count = 0;
    blocks = 0;
  };
  auto add = [&](In A, In W, uint16_t* out, int M, int N) {
    if (M == 0) return;
    jobs.job[jobs.count] = Job{A, W, out, M, N};
    jobs.first_block[jobs.count++] = (uint32_t)blocks;
    blocks += tiles(M, kJobM * kJobPanels) * tiles(N, kJobN);
    if (jobs.count == kMaxJobs) flush();
  };
  for (int i = 0; i < d.layers; ++i) {
    add(w.table, (In)layers[i].pos, w.r + (size_t)i * k_len * proj, k_len, proj);
    add((In)mems + i * mem_stride, (In)layers[i].qkv + (size_t)proj * kD,
        w.kv_mem + (size_t)i * mem_rows * 2 * proj, mem_rows, 2 * proj);
  }
  flush();

  const TileMap qkv_map(tiles(rows, 64), 3 * proj / 96);
  // a group has as many workgroups as a product has tasks there: with more, some would take
  // two tasks of one product while others wait for them
  size_t panel_tasks = kResTasks;
  for (size_t columns : {(size_t)d.inner, 3 * (size_t)proj})
    if (columns / kNormCols > panel_tasks) panel_tasks = columns / kNormCols;
  const size_t rows_each = launch_rows(rows);
  for (int i = 0; i < d.layers; ++i) {
    const orion_txl_layer& p = layers[i];
    // a layer's input also goes into the memory's last rows
    auto rows_out = [&](int layer) {
      RowsOut out = {};
      if (new_mems) {
        out.mem = (uint16_t*)new_mems + layer * new_mem_stride;
        out.mem_from = (d.q_len - mem_rows_out) * d.batch;
      }
      return out;
    };
    if (i == 0)
      hipLaunchKernelGGL((txl_panel_gemm_kernel<64, 96, QkvEpi>), dim3(qkv_map.blocks()),
                         dim3(kPanelThreads), 0, s, (In)x0, (In)p.qkv, rows, qkv_map,
                         rows_out(0), QkvEpi{w.qu, w.qv, w.kv_x, (In)u, (In)v, proj});
    const size_t attn_blocks = (size_t)d.heads * d.batch * tiles(d.q_len, kQ);
    Coming coming = {};
    size_t left = attn_blocks < kUnits ? (kUnits - attn_blocks) * kTouchBytes : 0, ahead = 0;
    int count = 0;
    auto add_coming = [&](const void* weights, size_t rows) {
      const size_t bytes = rows * kD * 2 < left ? rows * kD * 2 : left;
      coming.p[count] = (In)weights;
      coming.bytes[count++] = (uint32_t)bytes;
      left -= bytes;
      ahead += bytes;
    };
    add_coming(p.out, proj);
    add_coming(p.ff1_w, d.inner);
    add_coming(p.ff2_w, d.inner);
    if (i + 1 < d.layers) add_coming(layers[i + 1].qkv, 3 * (size_t)proj);
    for (size_t first = 0; first < attn_blocks; first += kAttnMost) {
      const size_t own = attn_blocks - first < kAttnMost ? attn_blocks - first : kAttnMost;
      hipLaunchKernelGGL(txl_attention_kernel,
                         dim3((unsigned)(own + tiles(ahead, kTouchBytes))), dim3(kAttnThreads), 0,
                         s, (In)(w.kv_mem + (size_t)i * mem_rows * 2 * proj), (In)w.kv_x,
                         (In)(w.r + (size_t)i * k_len * proj), d.q_len, d.m_len, d.batch, d.heads,
                         (uint32_t)first, (uint32_t)own, ~0u / (uint32_t)d.heads,
                         ~0u / (uint32_t)d.batch, (In)w.qu, (In)w.qv, w.att, coming);
    }
    Layer a = {};
    auto product = [&](int stage, const void* W, int ld, int columns, int tasks) {
      a.product[stage] = {(In)W, ld, columns, tasks, ~0u / (uint32_t)tasks};
    };
    product(0, p.out, proj, kResCols, kResTasks);
    product(1, p.ff1_w, kD, kNormCols, d.inner / kNormCols);
    product(2, p.ff2_w, d.inner, kResCols, kResTasks);
    product(3, i + 1 < d.layers ? layers[i + 1].qkv : nullptr, kD, kNormCols,
            3 * proj / kNormCols);
    a.products = i + 1 < d.layers ? 4 : 3;
    a.ff1_b = (In)p.ff1_b;
    a.ff2_b = (In)p.ff2_b;
    a.inner = d.inner;
    a.proj = proj;
    uint32_t* counters = w.counters;
    for (size_t row0 = 0; row0 < (size_t)rows; row0 += rows_each) {
      const size_t n = std::min(rows_each, rows - row0);
      const size_t groups = groups_of(n), panels = group_panels(n, groups);
      a.panels = (int)panels;
      a.rows = (int)n;
      a.att = w.att + row0 * proj;
      a.x = (i == 0 ? (In)x0 : w.x[i & 1]) + row0 * kD;
      a.parts1 = w.parts + row0 * kParts;
      a.parts2 = w.parts2 + row0 * kParts;
      a.norm1 = Norm{(In)p.norm1_w, (In)p.norm1_b, a.parts1, d.eps};
      a.norm2 = Norm{(In)p.norm2_w, (In)p.norm2_b, a.parts2, d.eps};
      a.y1 = w.y + row0 * kD;
      a.y2 = w.y2 + row0 * kD;
      a.x2 = w.x2 + row0 * kD;
      a.h = w.h + row0 * d.inner;
      if (i + 1 < d.layers) {
        a.rows_out = rows_out(i + 1);
        a.rows_out.x = w.x[(i + 1) & 1] + row0 * kD;
        a.rows_out.mem_from -= (int)row0;
        a.qkv = {w.qu + row0 * proj, w.qv + row0 * proj, w.kv_x + row0 * 2 * proj, (In)u, (In)v,
                 proj};
      }
      a.counters = counters;
      const size_t group_blocks = std::min(panel_tasks * panels, kUnits / groups);
      hipLaunchKernelGGL(txl_layer_kernel, dim3((unsigned)(groups * group_blocks)),
                         dim3(kLayerThreads), 0, s, counters, (int)groups - 1,
                         __builtin_ctz((unsigned)groups), (int)tiles(n, 16), i, a);
      counters += counters_of(n);
    }
  }
  const orion_txl_layer& last = layers[d.layers - 1];
  hipLaunchKernelGGL(txl_norm_kernel, dim3((unsigned)tiles(rows, kThreads / 16)), dim3(kThreads), 0,
                     s, (const float*)w.y2,
                     (Norm{(In)last.norm2_w, (In)last.norm2_b, w.parts2, d.eps}),
                     (uint16_t*)hidden, rows);
  return hipGetLastError() == hipSuccess ? ORION_OK : ORION_ERR_LAUNCH;
}

extern "C" size_t orion_nll_workspace_bytes(const orion_nll* args) {
  Crit c;
  size_t bytes = 0;
  return args != nullptr && lay_out(args, nullptr, &c, &bytes) ? bytes : 0;
}

extern "C" int orion_nll_bf16(const orion_nll* args, void* nll, void* workspace,
                              size_t workspace_bytes, void* stream) {
  if (!args || !nll || !workspace || !args->hidden || !args->weight || !args->bias ||
      !args->target || (args->tails > 0 && (!args->tail_weight || !args->tail_bias)))
    return ORION_ERR_ARG;
  Crit c;
  size_t bytes = 0;
  if (!lay_out(args, workspace, &c, &bytes)) return ORION_ERR_SHAPE;
  if (workspace_bytes < bytes) return ORION_ERR_ARG;
  if ((((uintptr_t)args->hidden | (uintptr_t)args->weight | (uintptr_t)args->tail_weight |
        (uintptr_t)workspace) & 15u) != 0)
    return ORION_ERR_ALIGN;
  hipStream_t s = (hipStream_t)stream;
  hipLaunchKernelGGL(crit_group_kernel, dim3(1), dim3(kGroupThreads), 0, s, c);
  hipLaunchKernelGGL(crit_logits_kernel, dim3(kCritBlocks), dim3(kThreads), 0, s, c);
  hipLaunchKernelGGL(crit_losses_kernel, dim3((unsigned)tiles(c.n, kThreads / 64)), dim3(kThreads),
                     0, s, c, (uint16_t*)nll);
  return hipGetLastError() == hipSuccess ? ORION_OK : ORION_ERR_LAUNCH;
}
