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

// The ranges of a launch of `groups` workgroups (1: none), so that about
// `per_cu` workgroups per CU run at once, and the partials' bytes. us a call
// at 1 / 2 / 3 / 4 / 6 / 8 / 10 / 16 ranges, D 128, in groups without ranges:
//   48 (180 queries of 8191 keys, 32 heads over 8)  167 / 94 / 69 / 57 / 44 / 41 / 38 / 47
//  104 (400 of 2000, 32 over 8)                      48 / 37 / 35 / 34 / 37 / 39 / 44 / 53
//  128 (500 of 4095, 32 over 4)                      89 / 57 / 47 / 43 / 50 / 50 / 57 / 73
//  248 (990 of 4095, 32 over 8, f16)                 94 / 74 / 73 / 72 / 80 / 89
//  256 (1000 of 32767, 32 over 8)                   648 / 371 / 337 / 330 / 336 / 344 / 357 / 398
//  376 (3000 of 16000, 16 over 8)                   333 / 243 / 239 / 242 / 260 / 283 / 307 / 388
//  500 (2000 of 12000, 32 over 4, f16)              277 / 251 / 250 / 259 / 279 / 309
// 1752 (7000 of 32767, 32 over 4)                  1860 / 1894 / - / 1972 / - / 2186
// A range more costs its partials' traffic: 16 MB each way a range and 32K rows.
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
