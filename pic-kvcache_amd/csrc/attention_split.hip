// Split rule and merge of the side-forward attention's key ranges.
#include <hip/hip_bf16.h>
#include <hip/hip_fp16.h>

#include <algorithm>
#include <cmath>

#include "attention_split.hpp"

namespace cbk {
namespace {

constexpr uint32_t kMaxSplits = 32;
constexpr uint32_t kMinBlocksPerSplit = 3;
// float32: shorter ranges cost more in partials than they save
constexpr int64_t kMinKeysPerSplitF32 = 128;
constexpr int kMergeThreads = 256;

template <typename T> __device__ __forceinline__ T to_out(float v);
template <> __device__ __forceinline__ float to_out<float>(float v) { return v; }
template <> __device__ __forceinline__ __hip_bfloat16 to_out<__hip_bfloat16>(float v) { return __float2bfloat16(v); }
template <> __device__ __forceinline__ __half to_out<__half>(float v) { return __float2half(v); }

// 32 lanes per row. Lane s weighs range s, so a row's maximum and sum are
// lane reductions; then every lane sums N dims over the ranges with all the
// ranges' loads independent (one thread that read a row's ranges one after
// another took 0.3 us a range). N dims per lane: 4 at d = 128, 2 at 64, both
// one load; 0: any d, dims 32 apart.
template <typename T, int N>
__global__ __launch_bounds__(kMergeThreads) void attn_merge_kernel(const AttnParts parts, uint32_t nq, uint32_t hq,
                                                                   uint32_t d, const int64_t* pos, T* out,
                                                                   int64_t out_stride, bool nan_empty) {
  constexpr int E = N ? N : 4;  // d <= 128
  constexpr bool F32 = sizeof(T) == 4;
  typedef float VecN __attribute__((ext_vector_type(E)));
  const uint32_t lane = threadIdx.x & 31;
  const uint64_t rows = uint64_t(nq) * hq;
  const uint64_t row = uint64_t(blockIdx.x) * (kMergeThreads / 32) + (threadIdx.x >> 5);
  if (row >= rows) return;  // both halves' exchanges stay within their 32 lanes
  const uint32_t S = parts.splits;
  const float2 ml = lane < S ? parts.ml[lane * rows + row] : make_float2(-__builtin_inff(), 0.f);
  float m = ml.x;
#pragma unroll
  for (int off = 16; off >= 1; off >>= 1) m = fmaxf(m, __shfl_xor(m, off, 32));
  // a range without visible keys for the row: its sum is 0, its output may be
  // unwritten (never in float32)
  const float w = ml.y == 0.f ? 0.f : __builtin_amdgcn_exp2f((F32 ? 2.f : 1.f) * (ml.x - m));
  // every other output counts, also with a weight of 0 (an infinity in it is
  // NaN then, as in one range)
  const uint64_t any = __ballot(F32 || ml.y != 0.f);
  const uint32_t use = uint32_t((threadIdx.x & 32) ? any >> 32 : any);
  float l = ml.y == 0.f ? 0.f : w * ml.y;
#pragma unroll
  for (int off = 16; off >= 1; off >>= 1) l += __shfl_xor(l, off, 32);
  float acc[E];
#pragma unroll
  for (int e = 0; e < E; ++e) acc[e] = 0.f;
  const float* o = parts.o + row * d;
#pragma unroll 8
  for (uint32_t s = 0; s < S; ++s) {
    const float ws = __shfl(w, int(s), 32);
    const bool used = (use >> s) & 1u;
    if constexpr (N != 0) {
      const VecN v = used ? *reinterpret_cast<const VecN*>(o + s * rows * d + lane * N) : VecN(0.f);
#pragma unroll
      for (int e = 0; e < E; ++e) acc[e] = fmaf(ws, v[e], acc[e]);
    } else {
#pragma unroll
      for (int e = 0; e < E; ++e)
        if (used && lane + 32 * e < d) acc[e] = fmaf(ws, o[s * rows * d + lane + 32 * e], acc[e]);
    }
  }
  const uint32_t q = uint32_t(row / hq), h = uint32_t(row - uint64_t(q) * hq);
  const float empty = nan_empty && pos[q] >= 0 ? __uint_as_float(0x7fc00000u) : 0.f;
  const float inv = 1.f / l;
  T* dst = out + int64_t(q) * out_stride + int64_t(h) * d;
  T res[E];
#pragma unroll
  for (int e = 0; e < E; ++e) res[e] = to_out<T>(l == 0.f ? empty : acc[e] * inv);
  if constexpr (N != 0) {
    using V = typename Vec<int(N * sizeof(T))>::T;
    *reinterpret_cast<V*>(dst + lane * N) = *reinterpret_cast<const V*>(res);
  } else {
#pragma unroll
    for (int e = 0; e < E; ++e)
      if (lane + 32 * e < d) dst[lane + 32 * e] = res[e];
  }
}

template <typename T>
int launch_merge_t(const AttnParts& parts, uint32_t nq, uint32_t hq, uint32_t d, const int64_t* pos, T* out,
                   int64_t out_stride, bool nan_empty, hipStream_t stream) {
  constexpr uint64_t kRows = kMergeThreads / 32;
  const dim3 grid(uint32_t((uint64_t(nq) * hq + kRows - 1) / kRows));
  const bool aligned = out_stride % 4 == 0 && reinterpret_cast<uintptr_t>(out) % (4 * sizeof(T)) == 0;
#define CBK_MERGE(N)                                                                                             \
  hipLaunchKernelGGL((attn_merge_kernel<T, N>), grid, dim3(kMergeThreads), 0, stream, parts, nq, hq, d, pos, out, \
                     out_stride, nan_empty)
  if (d == 128 && aligned) CBK_MERGE(4);
  else if (d == 64 && aligned) CBK_MERGE(2);
  else CBK_MERGE(0);
#undef CBK_MERGE
  return launch_status("attention merge");
}

}  // namespace

uint32_t attn_splits(uint64_t groups, uint64_t rows, int64_t nk, int64_t d) {
  int cus = 0;
  if (groups == 0 || device_cus(&cus)) return 1;
  struct Cost { double start, step, share, merge, range, rate; };
  const Cost c = d == 64 ? Cost{6.5, 0.48, 0.146, 3.1, 0.21, 4.3e6} : Cost{8.1, 0.59, 0.25, 2.5, 0.16, 5.1e6};
  const double blocks = double((nk + kAttnKeyBlock - 1) / kAttnKeyBlock);
  const double busy = double(groups) * blocks * c.share / cus;
  auto cost = [&](uint32_t s) {
    const double chain = c.start + blocks / s * c.step;
    const double pass = std::sqrt(std::sqrt(chain * chain * chain * chain + busy * busy * busy * busy));
    return s == 1 ? pass : pass + c.merge + s * (c.range + double(rows) * double(d + 2) * 8 / c.rate);
  };
  uint32_t best = 1;
  double least = 0.97 * cost(1);  // no partials for less than 3%
  const uint32_t most = uint32_t(std::min<double>(kMaxSplits, blocks / kMinBlocksPerSplit));
  for (uint32_t s = 2; s <= most; ++s)
    if (const double t = cost(s); t < least) {
      least = t;
      best = s;
    }
  return best;
}

uint32_t attn_f32_splits(uint64_t groups, int64_t nk) {
  int cus = 0;
  if (groups == 0 || device_cus(&cus)) return 1;
  const uint64_t want = uint64_t(kAttnF32PerCu) * uint32_t(cus);
  // one round of workgroups where that takes three or more ranges; with fewer
  // the ranges are long, and two shorter rounds even out the tiles' lengths
  uint64_t s = want / groups;
  if (s < 3) s = 2 * want / groups;
  s = std::min<uint64_t>(s, uint64_t(nk / kMinKeysPerSplitF32));
  return uint32_t(std::max<uint64_t>(1, std::min<uint64_t>(s, kMaxSplits)));
}

size_t attn_parts_bytes(uint32_t splits, uint64_t rows, int64_t d) {
  if (splits <= 1) return 0;
  const uint64_t ml = (uint64_t(splits) * rows * sizeof(float2) + 255) & ~uint64_t(255);
  return size_t(ml + uint64_t(splits) * rows * uint64_t(d) * sizeof(float));
}

AttnParts attn_parts(uint32_t splits, uint64_t rows, void* workspace) {
  AttnParts p{splits, nullptr, nullptr};
  if (splits > 1) {
    p.ml = static_cast<float2*>(workspace);
    const uint64_t ml = (uint64_t(splits) * rows * sizeof(float2) + 255) & ~uint64_t(255);
    p.o = reinterpret_cast<float*>(static_cast<char*>(workspace) + ml);
  }
  return p;
}

int launch_attn_merge(const AttnParts& parts, uint32_t nq, uint32_t hq, uint32_t d, const int64_t* pos, void* out,
                      int64_t out_stride, int32_t dtype, bool nan_empty, hipStream_t stream) {
  switch (dtype) {
    case CBK_DTYPE_F32:
      return launch_merge_t(parts, nq, hq, d, pos, static_cast<float*>(out), out_stride, nan_empty, stream);
    case CBK_DTYPE_BF16:
      return launch_merge_t(parts, nq, hq, d, pos, static_cast<__hip_bfloat16*>(out), out_stride, nan_empty, stream);
    default:
      return launch_merge_t(parts, nq, hq, d, pos, static_cast<__half*>(out), out_stride, nan_empty, stream);
  }
}

}  // namespace cbk
