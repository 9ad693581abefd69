// Key ranges of the side-forward attention: a launch with too few row tiles to
// fill the chip gives every tile's keys to several workgroups, each of which
// writes its rows' unnormalised output, maximum and sum; a second launch
// merges them.
#pragma once

#include "cbk_common.hpp"

namespace cbk {

constexpr int kAttnKeyBlock = 32;  // keys per block of the attention kernels

// Partial results of `splits` key ranges: for range s and row r = query *
// hq + head, ml[s * rows + r] = (reference m in log2 units, sum of 2^(x - m))
// and o[(s * rows + r) * d ..] the sum of 2^(x - m) * value, float32. From
// float32 inputs m is halved: it holds every logit of the type that way.
struct AttnParts {
  uint32_t splits;  // 1: no partials, the workgroups write the output
  float2* ml;
  float* o;
};

// The ranges of a 16-bit launch of `groups` workgroups over `rows` (query,
// head) rows (1: none), the fewest us by this estimate: the longest workgroup
// takes `start` and a `step` per key block of its range; the CUs together are
// busy for `share` per block of all workgroups; the fourth root of the two
// fourth powers lies between them; the ranges add a launch, a little each and
// their partials written and read. Its six figures per head size are fitted to
// the calls below and 180 more (4% off in the mean): they take 1.2% longer
// than at the best count in the mean, 11% at the worst, and none longer than
// without ranges. The rule before it, as many ranges as fill the CUs' slots,
// took up to 53% longer than without (900 of 1000) and 6.7% than the best.
// us a call at 1 / 2 / 3 / 4 / 5 / 6 / 8 / 10 / 12 / 16 ranges, bf16, in groups
// without ranges (* taken):
//    8 (5 of 256, 32 heads over 8 x 128)      12.0*/ 12.7 / 12.4 / 12.1 / 12.3 / 12.7 / 12.7
//   32 (100 of 1000, 32 over 8 x 128)         26.2 / 22.2 / 19.5 / 19.0 / 18.6*/ 18.8 / 19.4 / 20.2 / 21.6 / 23.2
//   48 (190 of 12000, 32 over 8 x 128)         226 /  125 /   89 /   72 / 61.6 / 55.2 / 47.2 / 43.9 / 44.5*/ 49.2
//  104 (400 of 4000, 32 over 8 x 128)         78.6 / 51.6 / 43.2 / 39.9 / 38.3*/ 40.3 / 44.6 / 49.9 / 51.5 / 61.4
//  136 (520 of 12000, 32 over 8 x 128)         218 /  123 / 93.6 / 80.4 / 76.7 / 83.2*/ 84.3 / 89.9 / 96.5 /  109
//  176 (680 of 4000, 32 over 8 x 128)         80.2 / 58.1 / 49.1 / 52.0*/ 55.9 / 58.8 / 65.4 / 72.0 / 80.9
//  192 (760 of 12000, 32 over 8 x 128)         221 /  132 /  105 /  107*/  110 /  110 /  115 /  124 /  133
//  232 (900 of 1000, 32 over 8 x 128)         28.5*/ 34.3 / 38.7 / 42.8 / 48.3 / 53.0 / 62.6 / 69.5
//  256 (1000 of 4000, 32 over 8 x 128)        81.6 / 61.9 / 63.5*/ 65.0 / 69.3 / 73.5 / 85.3 / 97.0
//  256 (1000 of 4000, 32 over 8 x 64)         64.5 / 49.7 / 45.2*/ 45.0 / 47.7 / 49.0 / 55.4 / 60.9
//  400 (1600 of 16000, 32 over 8 x 128)        313 /  229 /  225*/  239 /  254 /  264
//  504 (2000 of 4000, 32 over 8 x 128)        91.7*/ 96.5 /  102 /  114 /  122
//  632 (2000 of 8000, 40 over 8 x 128)         184*/  191 /  201 /  218
//  704 (2800 of 16000, 32 over 8 x 128)        364*/  365 /  372
//  800 (3200 of 8000, 32 over 8 x 128)         217*/  237 /  256
// 1000 (4000 of 16000, 32 over 8 x 128)        519*/  513
uint32_t attn_splits(uint64_t groups, uint64_t rows, int64_t nk, int64_t d);
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
uint32_t attn_f32_splits(uint64_t groups, int64_t nk);
int launch_attn_f32(const AttnF32Args& a, hipStream_t stream);

}  // namespace cbk
