// Key ranges of the side-forward attention: a launch with too few row tiles to
// fill the chip gives every tile's keys to several workgroups, each of which
// writes its rows' unnormalised output, maximum and sum; a second launch
// merges them.
#pragma once

#include "cbk_common.hpp"

namespace cbk {

// Partial results of `splits` key ranges: for range s and row r = query *
// hq + head, ml[s * rows + r] = (maximum in log2 units, sum of 2^(x - maximum))
// and o[(s * rows + r) * d ..] the sum of 2^(x - maximum) * value, float32.
struct AttnParts {
  uint32_t splits;  // 1: no partials, the workgroups write the output
  float2* ml;
  float* o;
};

// The ranges that bring a launch of `groups` workgroups to about `per_cu`
// workgroups per CU (1 where it has as many without), and the partials' bytes.
uint32_t attn_splits(uint64_t groups, uint32_t per_cu, int64_t nk);
size_t attn_parts_bytes(uint32_t splits, uint64_t rows, int64_t d);
AttnParts attn_parts(uint32_t splits, uint64_t rows, void* workspace);

// out[r] = the merged rows, in `dtype`; a row without visible keys (position
// below 0) is zero. nan_empty: a row whose visible keys all have a logit of
// -inf is NaN, as its softmax is; zero otherwise.
int launch_attn_merge(const AttnParts& parts, uint32_t nq, uint32_t hq, uint32_t d, const int64_t* pos, void* out,
                      int64_t out_stride, int32_t dtype, bool nan_empty, hipStream_t stream);

struct AttnF32Args {
  const float* q;
  const int64_t* pos;
  const float* k;
  const float* v;
  float* out;
  int64_t q_stride, k_stride, v_stride, out_stride;
  uint32_t nq, nk, hq, hkv, group, d;
  float scale;
  AttnParts parts;
};

// Rows (query, head of a KV head's group) per workgroup of the float32
// kernel, and the workgroups per CU its key ranges aim at: more than the two
// to four resident, so that the ranges of the latest tiles (most keys) do not
// run alone at the end. us a call at 1 / 2 / 3 / 4 / 6 / 8 / 12 ranges: 500 of
// 2047 keys, 16 heads over 8 x 128 (128 workgroups) 183 / 101 / 88 / 75 / 74 /
// 74 / 78; 400 of 2000, 40 over 8 x 128 (256) 182 / 132 / 119 / 116 / 119 /
// 125 / 139; 200 of 2047, 32 over 8 x 64 (104) 107 / 61 / 51 / 45 / 42 / 42 /
// 47.
constexpr uint32_t kAttnF32Rows = 64;
constexpr uint32_t kAttnF32PerCu = 3;
int launch_attn_f32(const AttnF32Args& a, hipStream_t stream);

}  // namespace cbk
