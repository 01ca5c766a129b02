// LAMB step over a list of fp32 tensors (the optimiser of the Transformer-XL
// training client; the reference's is related/baselines/transformer/lamb.py:108-144):
//
//   m = b1 m + (1 - b1) g          u = m / (sqrt(v) + eps) + decay w
//   v = b2 v + (1 - b2) g g        w = w - lr * min(|w|, 10) / (|u| + eps) * u
//
// HBM-bound.  w's update needs |u| over the whole tensor, so two passes: the
// first moves 24 bytes per element (reads g, m, v, w; writes m, v) and leaves
// one pair of partial sums per workgroup, the second 16 (reads m, v, w, computes
// the same u again, writes w).  40 bytes against the 28 that a step whose arrays
// all stayed on chip would move; as separate element-wise operations it is 100.
//
// Measured on the 16-layer, 267,735-token Transformer-XL (188 M parameters, 182
// tensors): 1.21 ms a step, 6.2 TB/s over the 40 bytes (1.31 with a contiguous chunk a
// workgroup, cached accesses and the tensor found by a vector load), against 5.2 ms for
// the element-wise operations.  The first pass has one 16-byte access per lane and array
// in flight and every wavefront a compute unit can hold (37 registers): 715 us for 188 M
// elements in launches of 5120 workgroups, 6.3 TB/s; four accesses a lane need 88
// registers, hold five wavefronts a SIMD and reach the same only bare of everything else
// (725).  The second is fastest with four (64 registers, 468 us, 6.4 TB/s), 10 % slower
// with one.  Both lose 2 to 4 us a launch on its beginning and end.
// Taking the tensors in groups small enough for the memory-side cache gains
// nothing over the launches it adds, so a group is as many tensors as the arguments
// hold, and its launches are cut by time only (kMomentsBlocks).
//
// The sums run in a fixed order (thread, wavefront, workgroup in fp32 over 4096
// elements, then fp64 over the workgroups), so a step gives the same bits twice.

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>

#include "kernels.h"

namespace {

constexpr int kMomentsThreads = 1024, kThreads = 256;
constexpr int kUnroll = 4;                            // 16-byte accesses per lane and array
constexpr int kChunk = kThreads * 4 * kUnroll;        // elements per workgroup
static_assert(kChunk == kMomentsThreads * 4, "");
constexpr int kMaxTensors = 64;
constexpr int kReduceThreads = 1024;
// Workgroups of one launch of each pass.  A launch cannot be held back once it has
// begun, and best-effort kernels run on budgets of 100 us and more, so none takes longer
// than that: 5120 (21 M elements) are 81 us of the first pass, 8192 (34 M) 84 us of the
// second.
constexpr uint64_t kMomentsBlocks = 5120, kUpdateBlocks = 8192;
// The second pass begins with the first one's last data, so a group's last launch of the first
// pass and the full one before it, 21 to 42 M elements, leave the moments (168 to 335 MB) in the
// memory-side cache (256 MB); all other accesses pass it by, gradients and weights among them.
// Where that is more than the cache holds, what it still has is what comes first.  us a step,
// nothing cached, and so: 13.7 M parameters 97 and 89, 23.9 M 165 and 152, 85 M 585 and 555,
// 192 M 1290 and 1245; the moments of all launches 1281, the second pass's accesses too 1366,
// the first one's weights too 1251.  With only the last launch's moments, with those of exactly
// the last 21 M elements, and so (eight tensors): 21.4 M 144, 134, 134; 41.5 M 260, 260, 256;
// 61.6 M 383, 384, 380; 88 M 566, 556, 554; 146 M 928, 931, 927.  The same rule serves groups of
// any size, the smallest whole.
constexpr uint64_t kKeptBlocks = 5120;

typedef float f32x4 __attribute__((ext_vector_type(4)));

// The tensors of some launches, by value in the kernel's arguments (2.9 KiB): nothing to
// upload, nothing that has to outlive the call.
struct Group {
  orion_lamb_tensor t[kMaxTensors];
  uint32_t first_block[kMaxTensors];       // workgroups before tensor i; past the last one all
  uint32_t every8[8];                      // first_block[8 * i]
  uint32_t blocks;
};

struct Coefs {
  float b1, b1c, b2, b2c, eps, decay;
};

// Tensor of this workgroup, between the launch's first one and its last one.  All of it stays
// in scalar registers and the scalar cache: a vector load, in which every lane compares an
// entry, waits behind the arrays' (a step 1.28 ms so instead of 1.26).
__device__ __forceinline__ int tensor_of_block(const Group& g, uint32_t block, int low, int high) {
  if (low == high) return low;
  int eight = 0, ti = 0;
#pragma unroll
  for (int i = 1; i < 8; ++i) eight += g.every8[i] <= block;
#pragma unroll
  for (int i = 1; i < 8; ++i) ti += g.first_block[eight * 8 + i] <= block;
  return eight * 8 + ti;
}

__device__ __forceinline__ bool aligned16(const orion_lamb_tensor& t) {
  return ((((uintptr_t)t.w | (uintptr_t)t.g | (uintptr_t)t.m | (uintptr_t)t.v) & 15u) == 0);
}

// Where a workgroup's elements lie: kChunk / 256 pieces of one wavefront's access each, `step`
// elements apart, U neighbours to a wavefront.  Eight workgroups in a row, which run on the
// eight XCDs, share a window of 8 * kChunk elements piece by piece, so that what is under way
// at a time lies close together in every array.  The accesses alone reach 6.4 TB/s so in the
// first pass and 6.6 in the second; with a chunk a workgroup 6.1 and 6.4, and with cached
// accesses 5.6 and 5.6.  A tensor's windows are counted from its start; in the last,
// incomplete one every workgroup has a chunk.
template <int U>
struct Pieces {
  uint64_t begin;                  // of the workgroup
  uint32_t step;
  bool whole;                      // no piece reaches past the tensor
  __device__ __forceinline__ Pieces(uint32_t block, uint64_t n) {
    const bool window = (uint64_t)((block | 7u) + 1) * kChunk <= n;
    begin = window ? (uint64_t)(block & ~7u) * kChunk + (block & 7u) * 256 : (uint64_t)block * kChunk;
    step = window ? 8 * 256 : 256;
    whole = (uint64_t)(block + 1) * kChunk <= n;
  }
  __device__ __forceinline__ uint64_t at(int u) const {
    return begin + ((threadIdx.x >> 6) * U + u) * step + (threadIdx.x & 63) * 4;
  }
};

// Without decay the weight is not in the update at all: 0 * w would be a NaN for an
// infinite weight, and through the norm for its whole tensor.
template <bool kDecay>
__device__ __forceinline__ float update_of(float w, float m, float v, const Coefs& c) {
  const float u = m / (__builtin_sqrtf(v) + c.eps);
  return kDecay ? __builtin_fmaf(c.decay, w, u) : u;
}

__device__ __forceinline__ void moments(float g, float& m, float& v, const Coefs& c) {
  m = __builtin_fmaf(c.b1c, g, c.b1 * m);
  v = __builtin_fmaf(c.b2c * g, g, c.b2 * v);
}

// Through the caches, or past them.
template <bool kCached>
__device__ __forceinline__ f32x4 load16(const float* p) {
  const f32x4* from = reinterpret_cast<const f32x4*>(p);
  return kCached ? *from : __builtin_nontemporal_load(from);
}
template <bool kCached>
__device__ __forceinline__ void store16(const f32x4& v, float* p) {
  f32x4* to = reinterpret_cast<f32x4*>(p);
  if (kCached) *to = v;
  else __builtin_nontemporal_store(v, to);
}

template <bool kDecay, bool kKept>
__global__ __launch_bounds__(kMomentsThreads) void lamb_moments_kernel(
    uint32_t first, int low, int high, float2* partials, Coefs c, Group g) {
  const uint32_t block = first + blockIdx.x;
  const int ti = tensor_of_block(g, block, low, high);
  const orion_lamb_tensor t = g.t[ti];
  const Pieces<1> pieces(block - g.first_block[ti], t.n);
  float sw = 0.0f, su = 0.0f;
  if (pieces.whole && aligned16(t)) {
    const uint64_t i = pieces.at(0);
    const f32x4 vg = load16<false>(t.g + i);
    f32x4 vm = load16<kKept>(t.m + i);
    f32x4 vv = load16<kKept>(t.v + i);
    const f32x4 vw = load16<false>(t.w + i);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      float m = vm[e], v = vv[e];
      moments(vg[e], m, v, c);
      vm[e] = m;
      vv[e] = v;
      const float w = vw[e], up = update_of<kDecay>(w, m, v, c);
      sw = __builtin_fmaf(w, w, sw);
      su = __builtin_fmaf(up, up, su);
    }
    store16<kKept>(vm, t.m + i);
    store16<kKept>(vv, t.v + i);
  } else {
    const uint64_t base = (uint64_t)(block - g.first_block[ti]) * kChunk;
    const uint64_t end = base + kChunk < t.n ? base + kChunk : t.n;
    for (uint64_t i = base + threadIdx.x; i < end; i += kMomentsThreads) {
      float m = t.m[i], v = t.v[i];
      moments(t.g[i], m, v, c);
      t.m[i] = m;
      t.v[i] = v;
      const float w = t.w[i], up = update_of<kDecay>(w, m, v, c);
      sw = __builtin_fmaf(w, w, sw);
      su = __builtin_fmaf(up, up, su);
    }
  }
#pragma unroll
  for (int d = 32; d > 0; d >>= 1) {
    sw += __shfl_xor(sw, d);
    su += __shfl_xor(su, d);
  }
  __shared__ float2 wave_sums[kMomentsThreads / 64];
  if ((threadIdx.x & 63) == 0) wave_sums[threadIdx.x >> 6] = make_float2(sw, su);
  __syncthreads();
  if (threadIdx.x == 0) {
    float2 s = wave_sums[0];
    for (int w = 1; w < kMomentsThreads / 64; ++w) {
      s.x += wave_sums[w].x;
      s.y += wave_sums[w].y;
    }
    partials[block] = s;
  }
}

// One workgroup per tensor: the factor that the update is added with.
__global__ __launch_bounds__(kReduceThreads) void lamb_ratio_kernel(
    const float2* __restrict__ partials, float* __restrict__ factor, double lr, double eps,
    Group g) {
  const int ti = blockIdx.x;
  double sw = 0.0, su = 0.0;
  const uint32_t end = ti + 1 < kMaxTensors ? g.first_block[ti + 1] : g.blocks;
  uint32_t b = g.first_block[ti] + threadIdx.x;
  // eight loads in flight: one after the other they are a chain of cache misses
  // (52 us for the 33,000 partial sums of a 137M-element tensor)
  for (; b + 7 * kReduceThreads < end; b += 8 * kReduceThreads) {
    float2 p[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) p[u] = partials[b + u * kReduceThreads];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      sw += (double)p[u].x;
      su += (double)p[u].y;
    }
  }
  for (; b < end; b += kReduceThreads) {
    sw += (double)partials[b].x;
    su += (double)partials[b].y;
  }
  __shared__ double lds[2][kReduceThreads];
  lds[0][threadIdx.x] = sw;
  lds[1][threadIdx.x] = su;
  __syncthreads();
  for (int d = kReduceThreads / 2; d > 0; d >>= 1) {
    if ((int)threadIdx.x < d) {
      lds[0][threadIdx.x] += lds[0][threadIdx.x + d];
      lds[1][threadIdx.x] += lds[1][threadIdx.x + d];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    double wn = sqrt(lds[0][0]);
    const double un = sqrt(lds[1][0]);
    if (wn > 10.0) wn = 10.0;              // a NaN stays one
    const double ratio = (wn == 0.0 || un == 0.0) ? 1.0 : wn / (un + eps);
    factor[ti] = (float)(-lr * ratio);
  }
}

template <bool kDecay>
__global__ __launch_bounds__(kThreads) void lamb_update_kernel(
    uint32_t last, int low, int high, const float* __restrict__ factor, Coefs c, Group g) {
  const uint32_t block = last - blockIdx.x;        // the first pass's last data first
  const int ti = tensor_of_block(g, block, low, high);
  const orion_lamb_tensor t = g.t[ti];
  const Pieces<kUnroll> pieces(block - g.first_block[ti], t.n);
  const float f = factor[ti];
  if (pieces.whole && aligned16(t)) {
    f32x4 vm[kUnroll], vv[kUnroll], vw[kUnroll];
#pragma unroll
    for (int u = 0; u < kUnroll; ++u) {
      const uint64_t i = pieces.at(u);
      vm[u] = load16<false>(t.m + i);
      vv[u] = load16<false>(t.v + i);
      vw[u] = load16<false>(t.w + i);
    }
#pragma unroll
    for (int u = 0; u < kUnroll; ++u) {
      const uint64_t i = pieces.at(u);
#pragma unroll
      for (int e = 0; e < 4; ++e)
        vw[u][e] = __builtin_fmaf(f, update_of<kDecay>(vw[u][e], vm[u][e], vv[u][e], c), vw[u][e]);
      store16<false>(vw[u], t.w + i);
    }
  } else {
    const uint64_t base = (uint64_t)(block - g.first_block[ti]) * kChunk;
    const uint64_t end = base + kChunk < t.n ? base + kChunk : t.n;
    for (uint64_t i = base + threadIdx.x; i < end; i += kThreads)
      t.w[i] = __builtin_fmaf(f, update_of<kDecay>(t.w[i], t.m[i], t.v[i], c), t.w[i]);
  }
}

uint64_t blocks_of(uint64_t n) { return (n + kChunk - 1) / kChunk; }

}  // namespace

// One factor per tensor of a launch and a pair of partial sums per workgroup.  The
// launches of one call run one after the other on one stream and share it.
extern "C" size_t orion_lamb_workspace_bytes(const orion_lamb_tensor* tensors, int count) {
  uint64_t blocks = 0;
  for (int i = 0; tensors != nullptr && i < count; ++i) blocks += blocks_of(tensors[i].n);
  return (size_t)(blocks * sizeof(float2) + kMaxTensors * sizeof(float));
}

extern "C" int orion_lamb_step(const orion_lamb_tensor* tensors, int count, double lr, double b1,
                               double b2, double eps, double decay, void* workspace,
                               size_t workspace_bytes, void* stream) {
  if (count < 0 || (count > 0 && (tensors == nullptr || workspace == nullptr)))
    return ORION_ERR_ARG;
  if (((uintptr_t)workspace & 7u) != 0) return ORION_ERR_ALIGN;
  if (workspace_bytes < orion_lamb_workspace_bytes(tensors, count)) return ORION_ERR_ARG;
  uint64_t all_blocks = 0;
  for (int i = 0; i < count; ++i) {
    const orion_lamb_tensor& t = tensors[i];
    if (t.n == 0) continue;
    if (!t.w || !t.g || !t.m || !t.v) return ORION_ERR_ARG;
    if ((((uintptr_t)t.w | (uintptr_t)t.g | (uintptr_t)t.m | (uintptr_t)t.v) & 3u) != 0)
      return ORION_ERR_ALIGN;
    all_blocks += blocks_of(t.n);
    if (all_blocks > 0x7fffffffu) return ORION_ERR_SHAPE;
  }
  const Coefs c = {(float)b1, (float)(1.0 - b1), (float)b2, (float)(1.0 - b2), (float)eps,
                   (float)decay};
  float* factor = (float*)workspace;
  float2* partials = (float2*)((char*)workspace + kMaxTensors * sizeof(float));
  hipStream_t s = (hipStream_t)stream;
  Group g;
  int next = 0;
  while (next < count) {
    int tensors_in = 0;
    uint64_t blocks = 0;
    for (; next < count && tensors_in < kMaxTensors; ++next) {
      const orion_lamb_tensor& t = tensors[next];
      if (t.n == 0) continue;
      g.t[tensors_in] = t;
      g.first_block[tensors_in++] = (uint32_t)blocks;
      blocks += blocks_of(t.n);
    }
    if (tensors_in == 0) break;
    for (int i = tensors_in; i < kMaxTensors; ++i) g.first_block[i] = (uint32_t)blocks;
    for (int i = 0; i < 8; ++i) g.every8[i] = g.first_block[8 * i];
    g.blocks = (uint32_t)blocks;
    auto tensor_at = [&](uint64_t block) {
      return (int)(std::upper_bound(g.first_block, g.first_block + tensors_in, (uint32_t)block) -
                   g.first_block) - 1;
    };
    for (uint64_t at = 0; at < blocks; at += kMomentsBlocks) {
      const uint64_t n = std::min(kMomentsBlocks, blocks - at);
      const bool kept = at + n + kKeptBlocks > blocks;
      hipLaunchKernelGGL(decay != 0.0 ? (kept ? lamb_moments_kernel<true, true>
                                              : lamb_moments_kernel<true, false>)
                                      : (kept ? lamb_moments_kernel<false, true>
                                              : lamb_moments_kernel<false, false>),
                         dim3((unsigned)n), dim3(kMomentsThreads), 0, s, (uint32_t)at, tensor_at(at),
                         tensor_at(at + n - 1), partials, c, g);
    }
    hipLaunchKernelGGL(lamb_ratio_kernel, dim3((unsigned)tensors_in), dim3(kReduceThreads), 0, s,
                       (const float2*)partials, factor, lr, eps, g);
    for (uint64_t end = blocks; end > 0;) {
      const uint64_t n = std::min(kUpdateBlocks, end);
      hipLaunchKernelGGL(decay != 0.0 ? lamb_update_kernel<true> : lamb_update_kernel<false>,
                         dim3((unsigned)n), dim3(kThreads), 0, s, (uint32_t)(end - 1),
                         tensor_at(end - n), tensor_at(end - 1), (const float*)factor, c, g);
      end -= n;
    }
  }
  return hipGetLastError() == hipSuccess ? ORION_OK : ORION_ERR_LAUNCH;
}
