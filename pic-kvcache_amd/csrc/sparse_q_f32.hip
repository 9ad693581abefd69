// Sparse-Q attention-mass scores of float32 inputs for gfx950: the two passes
// of sparse_q.hip (row statistics, then column sums) on the float32 matrix
// cores, with the same ranges, merge and gather.
//
// Bound by the float32 matrix rate (v_mfma_f32_16x16x4_f32, 32 cycles each)
// over Q . K^T computed twice. Both passes stage one side's rows in LDS, 32
// at a time in two buffers (the next block's in registers meanwhile), and
// keep the other side's 16 rows per wave in registers:
//   row pass     keys in LDS, 64 (query, group head) rows per workgroup; a
//                lane holds 8 keys' logits of row lane % 16 and keeps that
//                row's (maximum, sum) over its own keys until the end
//   column pass  (query, group head) rows in LDS with their positions and
//                statistics, 64 keys per workgroup; a lane sums 8 rows'
//                probabilities of key lane % 16; every (key, range) belongs to
//                one wave, so the order of the sum is fixed
// A contraction step takes the dims in an order of its own (step e of a 16-dim
// group: dims 4 (lane / 16) + e), so that a lane's operands of 4 steps are one
// 16-byte read. One lane per logit with scalar dots took 1.65 ms + 8.9 ms on
// 256 queries of 2047 keys, 16 heads over 8 x 128 (2.0 GFLOP a pass).
// MFMA layout (checked on gfx950): A[i][k] in lane i + 16 k, B[k][j] in lane
// j + 16 k, D[i][j] in lane j + 16 (i / 4), register i % 4.
//
// Head sizes above 128, and more keys than one launch of the column pass
// holds, take one lane per logit.
#include <algorithm>

#include "sparse_q.hpp"

namespace cbk {
namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kBlock = 32;   // rows in LDS
constexpr int kTile = 64;    // rows in the workgroup's registers, 16 per wave
constexpr uint32_t kPerCu = 4;  // workgroups per CU that the ranges aim at

// 4 dims from `d0` on of a row of `d`, zeros past its end
template <bool VEC>
__device__ __forceinline__ f32x4 load4(const float* row, uint32_t d0, uint32_t d) {
  f32x4 w = f32x4{0.f, 0.f, 0.f, 0.f};
  if constexpr (VEC) {
    if (d0 < d) w = *reinterpret_cast<const f32x4*>(row + d0);
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (d0 + e < d) w[e] = row[d0 + e];
  }
  return w;
}

// The products of the block's 32 LDS rows with the wave's 16 register rows:
// register i of s[h] is LDS row 16 h + 4 (lane / 16) + i with register row lane % 16.
template <int DP>
__device__ __forceinline__ void block_products(const float* lds, const f32x4 (&reg)[DP / 16], f32x4 (&s)[2],
                                               uint32_t row, uint32_t grp) {
  constexpr int LD = DP + 4;
  s[0] = s[1] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int t = 0; t < DP / 16; ++t) {
    f32x4 w[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) w[h] = *reinterpret_cast<const f32x4*>(&lds[(16 * h + row) * LD + 16 * t + 4 * grp]);
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int h = 0; h < 2; ++h) s[h] = __builtin_amdgcn_mfma_f32_16x16x4f32(w[h][e], reg[t][e], s[h], 0, 0, 0);
  }
}

template <int DP, bool VEC>
__global__ __launch_bounds__(kThreads) void sq_rows_f32_kernel(const SqArgs a) {
  constexpr int LD = DP + 4;          // 16 rows' 16-byte reads fall on distinct banks
  constexpr int P = DP / 4;           // 16-byte pieces per row
  constexpr int ROWS = kThreads / P;  // rows loaded at a time
  constexpr int N = kBlock / ROWS;
  __shared__ __attribute__((aligned(16))) float kbuf[2][kBlock * LD];
  __shared__ int32_t s_max[4];
  const uint32_t lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t row = lane & 15, grp = lane >> 4;
  // workgroup -> (tile, key range, kv head), the kv head fastest and the
  // latest tiles (most keys) first
  const uint32_t g = __builtin_amdgcn_readfirstlane(blockIdx.x % a.hkv);
  const uint32_t rest = __builtin_amdgcn_readfirstlane(blockIdx.x / a.hkv);
  const uint32_t chunk = __builtin_amdgcn_readfirstlane(rest % a.row_chunks);
  const uint32_t nrows = a.nq * a.groups;
  const uint32_t ntiles = (nrows + kTile - 1) / kTile;
  const uint32_t r = (ntiles - 1 - rest / a.row_chunks) * kTile + wave * 16 + row;
  const bool valid = r < nrows;
  const uint32_t qi = valid ? r / a.groups : 0, h = g * a.groups + (valid ? r % a.groups : 0);
  const int32_t rpos = valid ? min(query_pos(a, qi), int32_t(a.nk) - 1) : -1;
  f32x4 qf[DP / 16];
  {
    const float* q = reinterpret_cast<const float*>(query_row(a, qi, h, 4));
#pragma unroll
    for (int t = 0; t < DP / 16; ++t)
      qf[t] = valid ? load4<VEC>(q, 16 * t + 4 * grp, a.d) : f32x4{0.f, 0.f, 0.f, 0.f};
  }
  int32_t wmax = rpos, wmin = valid ? rpos : 0x7fffffff;
#pragma unroll
  for (int off = 8; off >= 1; off >>= 1) {
    wmax = max(wmax, __shfl_xor(wmax, off));
    wmin = min(wmin, __shfl_xor(wmin, off));
  }
  wmax = __builtin_amdgcn_readfirstlane(wmax);
  wmin = __builtin_amdgcn_readfirstlane(wmin);
  if (lane == 0) s_max[wave] = wmax;
  __syncthreads();
  const int32_t gmax = __builtin_amdgcn_readfirstlane(max(max(s_max[0], s_max[1]), max(s_max[2], s_max[3])));
  const uint32_t nblocks = gmax < 0 ? 0u : uint32_t(gmax) / kBlock + 1;
  const int32_t b_lo = int32_t(uint64_t(nblocks) * chunk / a.row_chunks);
  const int32_t b_hi = int32_t(uint64_t(nblocks) * (chunk + 1) / a.row_chunks);

  const uint32_t lr = threadIdx.x / P, lp = threadIdx.x % P;
  f32x4 kreg[N];
  auto load = [&](int32_t b) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const uint32_t key = uint32_t(b) * kBlock + lr + ROWS * i;
      kreg[i] = f32x4{0.f, 0.f, 0.f, 0.f};
      if (key < a.nk)
        kreg[i] = load4<VEC>(reinterpret_cast<const float*>(a.k) + int64_t(key) * a.k_stride + int64_t(g) * a.d,
                             4 * lp, a.d);
    }
  };
  float m = kNegInf, l = 0.f;  // log2 units, over this lane's keys
  if (b_lo < b_hi) load(b_lo);
  for (int32_t b = b_lo; b < b_hi; ++b) {
    float* ks = kbuf[b & 1];
#pragma unroll
    for (int i = 0; i < N; ++i) *reinterpret_cast<f32x4*>(&ks[(lr + ROWS * i) * LD + 4 * lp]) = kreg[i];
    __syncthreads();  // block b is in LDS, and every wave is done with block b - 1's buffer
    if (b + 1 < b_hi) load(b + 1);
    const int32_t k0 = b * kBlock;
    if (wmax < k0) continue;  // no row of the wave sees the block
    f32x4 s[2];
    block_products<DP>(ks, qf, s, row, grp);
    float x[2][4], bm = kNegInf;
#pragma unroll
    for (int hh = 0; hh < 2; ++hh)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        x[hh][i] = (a.round_mode ? round_logit(s[hh][i], a.round_mode) : s[hh][i]) * a.c2;
        if (wmin < k0 + kBlock - 1 && k0 + 16 * hh + int32_t(4 * grp) + i > rpos) x[hh][i] = kNegInf;
        bm = fmaxf(bm, x[hh][i]);
      }
    const float mn = fmaxf(m, bm);
    const float ms = mn == kNegInf ? 0.f : mn;
    float sum = 0.f;
#pragma unroll
    for (int hh = 0; hh < 2; ++hh)
      sum += (__builtin_amdgcn_exp2f(x[hh][0] - ms) + __builtin_amdgcn_exp2f(x[hh][1] - ms)) +
             (__builtin_amdgcn_exp2f(x[hh][2] - ms) + __builtin_amdgcn_exp2f(x[hh][3] - ms));
    l = fmaf(l, __builtin_amdgcn_exp2f(m - ms), sum);
    m = mn;
  }
#pragma unroll
  for (int off = 16; off < 64; off <<= 1) {
    const float mo = __shfl_xor(m, off), lo = __shfl_xor(l, off);
    stats_merge(m, l, mo, lo);
  }
  if (grp == 0 && valid) {
    if (a.row_chunks == 1)
      a.stats[int64_t(h) * a.nq_pad + qi] = row_stats(m, l);
    else
      a.chunk_stats[(int64_t(chunk) * a.hq + h) * a.nq_pad + qi] = make_float2(m, l);
  }
}

template <int DP, bool VEC>
__global__ __launch_bounds__(kThreads) void sq_cols_f32_kernel(const SqArgs a) {
  constexpr int LD = DP + 4;
  constexpr int P = DP / 4;
  constexpr int ROWS = kThreads / P;
  constexpr int N = kBlock / ROWS;
  __shared__ __attribute__((aligned(16))) float qbuf[2][kBlock * LD];
  __shared__ __attribute__((aligned(16))) float s_stat[2][kBlock];
  __shared__ __attribute__((aligned(16))) int32_t s_pos[2][kBlock];
  const uint32_t lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t row = lane & 15, grp = lane >> 4;
  // workgroup -> (key tile, row range, kv head), the earliest keys (seen by
  // the most rows) first
  const uint32_t g = __builtin_amdgcn_readfirstlane(blockIdx.x % a.hkv);
  const uint32_t rest = __builtin_amdgcn_readfirstlane(blockIdx.x / a.hkv);
  const uint32_t split = __builtin_amdgcn_readfirstlane(rest % a.col_splits);
  const uint32_t kw0 = (rest / a.col_splits) * kTile + wave * 16;  // the wave's first key
  const uint32_t key = kw0 + row;
  f32x4 kf[DP / 16];
#pragma unroll
  for (int t = 0; t < DP / 16; ++t) {
    kf[t] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (key < a.nk)
      kf[t] = load4<VEC>(reinterpret_cast<const float*>(a.k) + int64_t(key) * a.k_stride + int64_t(g) * a.d,
                         16 * t + 4 * grp, a.d);
  }
  const uint32_t nrows = a.nq * a.groups;
  const uint32_t nblocks = (nrows + kBlock - 1) / kBlock;
  const uint32_t b_lo = uint32_t(uint64_t(nblocks) * split / a.col_splits);
  const uint32_t b_hi = uint32_t(uint64_t(nblocks) * (split + 1) / a.col_splits);
  const uint32_t lr = threadIdx.x / P, lp = threadIdx.x % P;
  f32x4 qreg[N];
  float stat = 0.f;   // threads below kBlock: row threadIdx.x of the block
  int32_t pos = -1;
  auto load = [&](uint32_t b) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const uint32_t r = b * kBlock + lr + ROWS * i;
      qreg[i] = f32x4{0.f, 0.f, 0.f, 0.f};
      if (r < nrows)
        qreg[i] = load4<VEC>(
            reinterpret_cast<const float*>(query_row(a, r / a.groups, g * a.groups + r % a.groups, 4)), 4 * lp, a.d);
    }
    if (threadIdx.x < kBlock) {
      const uint32_t r = b * kBlock + threadIdx.x;
      pos = -1;
      stat = 0.f;
      if (r < nrows) {
        const uint32_t qi = r / a.groups;
        pos = query_pos(a, qi);
        stat = a.stats[int64_t(g * a.groups + r % a.groups) * a.nq_pad + qi].x;
      }
    }
  };
  float acc = 0.f;
  if (b_lo < b_hi) load(b_lo);
  for (uint32_t b = b_lo; b < b_hi; ++b) {
    float* qs = qbuf[b & 1];
#pragma unroll
    for (int i = 0; i < N; ++i) *reinterpret_cast<f32x4*>(&qs[(lr + ROWS * i) * LD + 4 * lp]) = qreg[i];
    if (threadIdx.x < kBlock) {
      s_stat[b & 1][threadIdx.x] = stat;
      s_pos[b & 1][threadIdx.x] = pos;
    }
    __syncthreads();  // block b is in LDS, and every wave is done with block b - 1's buffers
    if (b + 1 < b_hi) load(b + 1);
    const int32_t lane_pos = s_pos[b & 1][lane % kBlock];
    if (!__any(lane_pos >= int32_t(kw0))) continue;  // no row of the block sees a key of the wave
    f32x4 s[2];
    block_products<DP>(qs, kf, s, row, grp);
#pragma unroll
    for (int hh = 0; hh < 2; ++hh) {
      const f32x4 st = *reinterpret_cast<const f32x4*>(&s_stat[b & 1][16 * hh + 4 * grp]);
      const int4 ps = *reinterpret_cast<const int4*>(&s_pos[b & 1][16 * hh + 4 * grp]);
      const int32_t p4[4] = {ps.x, ps.y, ps.z, ps.w};
      float p[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float x = (a.round_mode ? round_logit(s[hh][i], a.round_mode) : s[hh][i]) * a.c2;
        p[i] = int32_t(key) > p4[i] ? 0.f : __builtin_amdgcn_exp2f(x - st[i]);
      }
      acc += (p[0] + p[1]) + (p[2] + p[3]);
    }
  }
  acc += __shfl_xor(acc, 16);
  acc += __shfl_xor(acc, 32);
  if (grp == 0 && key < a.nk) a.partial[(int64_t(split) * a.hkv + g) * a.nk + key] = acc;
}

// ------------------------------------------------ one lane per logit

// rowstats: one wavefront per (query, head); lanes stride over keys.
__global__ __launch_bounds__(kThreads) void sq_rowstats_f32_kernel(const SqArgs a) {
  const uint32_t lane = threadIdx.x & 63;
  const uint32_t item = blockIdx.x * (kThreads / 64) + (threadIdx.x >> 6);
  if (item >= a.nq * a.hq) return;
  const uint32_t qi = item / a.hq, h = item % a.hq, g = h / a.groups;
  const int32_t pos = min(query_pos(a, qi), int32_t(a.nk) - 1);
  const float* qrow = reinterpret_cast<const float*>(query_row(a, qi, h, 4));
  float m = kNegInf, l = 0.f;
  for (int32_t key = int32_t(lane); key <= pos; key += 64) {
    const float* krow = reinterpret_cast<const float*>(a.k) + int64_t(key) * a.k_stride + int64_t(g) * a.d;
    float dot = 0.f;
    for (uint32_t e = 0; e < a.d; ++e) dot = fmaf(qrow[e], krow[e], dot);
    const float x = round_logit(dot, a.round_mode) * a.c2;
    stats_merge(m, l, x, 1.f);
  }
  for (int off = 1; off < 64; off <<= 1) {
    const float mo = __shfl_xor(m, off, 64), lo = __shfl_xor(l, off, 64);
    stats_merge(m, l, mo, lo);
  }
  if (lane == 0) a.stats[int64_t(h) * a.nq_pad + qi] = row_stats(m, l);
}

// colsum: one thread per (key, kv head), fixed query/head order.
__global__ __launch_bounds__(kThreads) void sq_colsum_f32_kernel(const SqArgs a) {
  const uint32_t t = blockIdx.x * kThreads + threadIdx.x;
  if (t >= a.nk * a.hkv) return;
  const uint32_t key = t % a.nk, g = t / a.nk;
  const float* krow = reinterpret_cast<const float*>(a.k) + int64_t(key) * a.k_stride + int64_t(g) * a.d;
  float acc = 0.f;
  for (uint32_t qi = 0; qi < a.nq; ++qi) {
    if (query_pos(a, qi) < int32_t(key)) continue;
    for (uint32_t hl = 0; hl < a.groups; ++hl) {
      const uint32_t h = g * a.groups + hl;
      const float* qrow = reinterpret_cast<const float*>(query_row(a, qi, h, 4));
      float dot = 0.f;
      for (uint32_t e = 0; e < a.d; ++e) dot = fmaf(qrow[e], krow[e], dot);
      const float2 st = a.stats[int64_t(h) * a.nq_pad + qi];
      acc += __builtin_amdgcn_exp2f(round_logit(dot, a.round_mode) * a.c2 - st.x);
    }
  }
  a.partial[int64_t(g) * a.nk + key] = acc;
}

template <int DP, bool VEC>
void launch_passes(const SqArgs& a, uint32_t g1, uint32_t g2, hipStream_t stream) {
  hipLaunchKernelGGL((sq_rows_f32_kernel<DP, VEC>), dim3(g1), dim3(kThreads), 0, stream, a);
  if (a.row_chunks > 1) launch_sq_merge(a, stream);
  hipLaunchKernelGGL((sq_cols_f32_kernel<DP, VEC>), dim3(g2), dim3(kThreads), 0, stream, a);
}

uint32_t ranges(uint64_t units, int cus, uint32_t most) {
  const uint64_t k = (uint64_t(kPerCu) * uint32_t(cus) + units - 1) / units;
  return uint32_t(std::max<uint64_t>(1, std::min<uint64_t>(k, most)));
}

}  // namespace

int launch_sq_f32(SqArgs& a, hipStream_t stream) {
  int cus = 0;
  if (int rc = device_cus(&cus)) return rc;
  const uint64_t rows = uint64_t(a.nq) * a.groups;
  const uint64_t u1 = (rows + kTile - 1) / kTile * a.hkv, u2 = (uint64_t(a.nk) + kTile - 1) / kTile * a.hkv;
  const uint32_t row_chunks = ranges(u1, cus, max_row_chunks(uint64_t(a.hq) * a.nq_pad));
  const uint32_t col_splits = ranges(u2, cus, kMaxColSplits);
  // a launch holds 2^32 threads: keys past 2^30 / hkv take a thread each
  if (a.d > 128 || rows >= (uint64_t(1) << 31) || u1 * row_chunks * kThreads >= (uint64_t(1) << 32) ||
      u2 * col_splits * kThreads >= (uint64_t(1) << 32)) {
    const uint64_t items = uint64_t(a.nq) * a.hq;
    hipLaunchKernelGGL(sq_rowstats_f32_kernel, dim3(uint32_t((items + 3) / 4)), dim3(kThreads), 0, stream, a);
    hipLaunchKernelGGL(sq_colsum_f32_kernel, dim3(uint32_t((uint64_t(a.nk) * a.hkv + kThreads - 1) / kThreads)),
                       dim3(kThreads), 0, stream, a);
    return CBK_OK;
  }
  a.row_chunks = row_chunks;
  a.col_splits = col_splits;
  const uint32_t g1 = uint32_t(u1 * row_chunks), g2 = uint32_t(u2 * col_splits);
  const int64_t align[5] = {a.q_stride * 4, a.k_stride * 4, int64_t(a.d) * 4,
                            int64_t(reinterpret_cast<uintptr_t>(a.q)), int64_t(reinterpret_cast<uintptr_t>(a.k))};
  const bool vec = common_vec_bytes(align, 5) == 16;
  if (a.d <= 64) {
    if (vec) launch_passes<64, true>(a, g1, g2, stream);
    else launch_passes<64, false>(a, g1, g2, stream);
  } else {
    if (vec) launch_passes<128, true>(a, g1, g2, stream);
    else launch_passes<128, false>(a, g1, g2, stream);
  }
  return CBK_OK;
}

}  // namespace cbk
