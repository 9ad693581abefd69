// Split rule and merge of the side-forward attention's key ranges.
#include <hip/hip_bf16.h>
#include <hip/hip_fp16.h>

#include <algorithm>

#include "attention_split.hpp"

namespace cbk {
namespace {

// A range holds at least 4 of the kernels' 32-key blocks of the longest row:
// shorter ones cost more in partials than they save.
constexpr uint32_t kMaxSplits = 32;
constexpr int64_t kMinKeysPerSplit = 128;
constexpr int kMergeThreads = 256;

__device__ __forceinline__ void store4(float* p, const float (&v)[4]) {
  *reinterpret_cast<float4*>(p) = make_float4(v[0], v[1], v[2], v[3]);
}
__device__ __forceinline__ void store4(__hip_bfloat16* p, const float (&v)[4]) {
  typedef float f4 __attribute__((ext_vector_type(4)));
  typedef __bf16 b4 __attribute__((ext_vector_type(4)));
  *reinterpret_cast<b4*>(p) = __builtin_convertvector((f4){v[0], v[1], v[2], v[3]}, b4);
}
__device__ __forceinline__ void store4(__half* p, const float (&v)[4]) {
  typedef float f4 __attribute__((ext_vector_type(4)));
  typedef _Float16 h4 __attribute__((ext_vector_type(4)));
  *reinterpret_cast<h4*>(p) = __builtin_convertvector((f4){v[0], v[1], v[2], v[3]}, h4);
}
__device__ __forceinline__ void store1(float* p, float v) { *p = v; }
__device__ __forceinline__ void store1(__hip_bfloat16* p, float v) { *p = __float2bfloat16(v); }
__device__ __forceinline__ void store1(__half* p, float v) { *p = __float2half(v); }

// One thread per (row, 4 dims): V of them per load where d and the output
// allow it (VEC), element by element otherwise. The partials were written by
// the launch before and are mostly still in the L2s and the last-level cache.
template <typename T, bool VEC>
__global__ __launch_bounds__(kMergeThreads) void attn_merge_kernel(const AttnParts parts, uint32_t nq, uint32_t hq,
                                                                   uint32_t d, const int64_t* pos, T* out,
                                                                   int64_t out_stride, bool nan_empty) {
  const uint32_t per_row = (d + 3) / 4;
  const uint64_t i = uint64_t(blockIdx.x) * kMergeThreads + threadIdx.x;
  const uint64_t rows = uint64_t(nq) * hq;
  const uint64_t row = i / per_row;
  if (row >= rows) return;
  const uint32_t dim = uint32_t(i - row * per_row) * 4;
  float m = -__builtin_inff();
  for (uint32_t s = 0; s < parts.splits; ++s) m = fmaxf(m, parts.ml[s * rows + row].x);
  const float ms = m == -__builtin_inff() ? 0.f : m;
  float l = 0.f, acc[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
  for (uint32_t s = 0; s < parts.splits; ++s) {
    const float2 ml = parts.ml[s * rows + row];
    const float* o = parts.o + (s * rows + row) * d + dim;
    if (ml.y == 0.f) continue;  // no visible keys: its output was not written
    const float w = __builtin_amdgcn_exp2f(ml.x - ms);
    l += w * ml.y;
    if constexpr (VEC) {
      const float4 v = *reinterpret_cast<const float4*>(o);
      acc[0] = fmaf(w, v.x, acc[0]);
      acc[1] = fmaf(w, v.y, acc[1]);
      acc[2] = fmaf(w, v.z, acc[2]);
      acc[3] = fmaf(w, v.w, acc[3]);
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (dim + e < d) acc[e] = fmaf(w, o[e], acc[e]);
    }
  }
  const uint32_t q = uint32_t(row / hq), h = uint32_t(row - uint64_t(q) * hq);
  const float empty = nan_empty && pos[q] >= 0 ? __uint_as_float(0x7fc00000u) : 0.f;
  const float inv = 1.f / l;
  T* dst = out + int64_t(q) * out_stride + int64_t(h) * d + dim;
#pragma unroll
  for (int e = 0; e < 4; ++e) acc[e] = l == 0.f ? empty : acc[e] * inv;
  if constexpr (VEC) {
    store4(dst, acc);
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (dim + e < d) store1(dst + e, acc[e]);
  }
}

template <typename T>
int launch_merge_t(const AttnParts& parts, uint32_t nq, uint32_t hq, uint32_t d, const int64_t* pos, T* out,
                   int64_t out_stride, bool nan_empty, hipStream_t stream) {
  const uint64_t threads = uint64_t(nq) * hq * ((d + 3) / 4);
  const dim3 grid(uint32_t((threads + kMergeThreads - 1) / kMergeThreads));
  const bool vec = d % 4 == 0 && out_stride % 4 == 0 && reinterpret_cast<uintptr_t>(out) % (4 * sizeof(T)) == 0;
  if (vec)
    hipLaunchKernelGGL((attn_merge_kernel<T, true>), grid, dim3(kMergeThreads), 0, stream, parts, nq, hq, d, pos,
                       out, out_stride, nan_empty);
  else
    hipLaunchKernelGGL((attn_merge_kernel<T, false>), grid, dim3(kMergeThreads), 0, stream, parts, nq, hq, d, pos,
                       out, out_stride, nan_empty);
  return launch_status("attention merge");
}

}  // namespace

uint32_t attn_splits(uint64_t groups, uint32_t per_cu, int64_t nk) {
  int cus = 0;
  if (groups == 0 || device_cus(&cus)) return 1;
  const uint64_t want = uint64_t(per_cu) * uint32_t(cus);
  uint64_t s = (want + groups - 1) / groups;
  s = std::min<uint64_t>(s, uint64_t(nk / kMinKeysPerSplit));
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
