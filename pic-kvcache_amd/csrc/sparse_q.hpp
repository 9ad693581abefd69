// Arguments and row statistics shared by the Sparse-Q score kernels.
#pragma once

#include <hip/hip_bf16.h>
#include <hip/hip_fp16.h>

#include "cbk_common.hpp"

namespace cbk {

constexpr int kThreads = 256;
constexpr int kQTile = 16;
constexpr float kLog2e = 1.4426950408889634f;
constexpr float kNegInf = -__builtin_inff();

struct SqArgs {
  const char* q;          // [*, Hq, D] rows
  int64_t q_stride;       // elements between query rows
  const int64_t* q_index; // [nq] rows of q that are sparse queries (nullable: 0..nq-1)
  const int64_t* pos;     // [*] absolute position of every q row (indexed like q)
  const char* k;          // [nk, Hkv, D]
  int64_t k_stride;       // elements between key rows
  uint32_t nq, nk, hq, hkv, d, groups;
  float c2;               // scale * log2(e)
  int32_t round_mode;     // 0 none, 1 bf16, 2 f16
  float2* stats;          // [hq][nq_pad] (m2 + log2(l), unused)
  float2* chunk_stats;    // [row_chunks][hq][nq_pad] (m2, l) of each key range, row_chunks > 1
  uint32_t row_chunks;    // key ranges per (query tile, kv head) in rowstats
  int32_t* tiles;         // [nq_pad / 16][32]: the 16 query positions (-1 past nq), min, max, unused
  float* partial;         // [col_splits][hkv][nk] column sums of each query range
  uint16_t* qdense;       // [hkv][nq_pad / 16][groups][16][D]: query rows in colsum's unit order
  uint32_t nq_pad;
  uint32_t col_splits;    // query-unit ranges per (key block, kv head) in colsum
};

__device__ __forceinline__ float round_logit(float x, int mode) {
  if (mode == 1) return __bfloat162float(__float2bfloat16(x));
  if (mode == 2) return __half2float(__float2half(x));
  return x;
}

__device__ __forceinline__ int32_t query_pos(const SqArgs& a, uint32_t qi) {
  if (qi >= a.nq) return -1;
  const int64_t row = a.q_index ? a.q_index[qi] : int64_t(qi);
  return int32_t(a.pos[row]);
}

__device__ __forceinline__ const char* query_row(const SqArgs& a, uint32_t qi, uint32_t h, uint32_t es) {
  const int64_t row = a.q_index ? a.q_index[qi] : int64_t(qi);
  return a.q + (row * a.q_stride + int64_t(h) * a.d) * es;
}

// Published per (head, query) row: x = m + log2(l), so that a probability
// is the single exp2(logit * scale * log2(e) - x) (+inf: an empty row).
__device__ __forceinline__ float2 row_stats(float m, float l) {
  return make_float2(l > 0.f ? m + log2f(l) : __builtin_inff(), 0.f);
}

// Online (max, sum) update in the log2 domain with -inf guards.
__device__ __forceinline__ void stats_merge(float& m, float& l, float m_o, float l_o) {
  const float mn = fmaxf(m, m_o);
  const float ms = mn == kNegInf ? 0.f : mn;
  l = l * __builtin_amdgcn_exp2f(m - ms) + l_o * __builtin_amdgcn_exp2f(m_o - ms);
  m = mn;
}

// Row and column pass on float32 inputs of any head size: sets the launch's
// key and query ranges in `a` and fills a.stats and a.partial.
int launch_sq_f32(SqArgs& a, hipStream_t stream);
// Merges the key ranges' statistics of every (head, query) row (row_chunks > 1).
void launch_sq_merge(const SqArgs& a, hipStream_t stream);

// Key ranges a (query tile, kv head) of the row pass may be split into, for
// `rows` = hq * nq_pad statistics: few rows leave most of the chip without a
// tile, and their ranges' statistics are small (16 MB at most past 8 ranges).
inline uint32_t max_row_chunks(uint64_t rows) {
  const uint64_t fit = (uint64_t(16) << 20) / (rows * sizeof(float2));
  return fit < 8 ? 8u : fit > 64 ? 64u : uint32_t(fit);
}
// Query ranges a (key block, kv head) of the column pass may be split into.
constexpr uint32_t kMaxColSplits = 4;

}  // namespace cbk
