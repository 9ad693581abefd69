// float32 side-forward attention of the selected queries for gfx950: the
// float32 form of attention.hip (cacheblend_vllm/ascend.py:798-846 without
// the 16-bit roundings).
//
// Bound by the float32 matrix rate (v_mfma_f32_16x16x4_f32, 32 cycles each:
// 157 TFLOP/s nominal). One workgroup (4 waves) per (64 rows of (query, group
// head), key range, KV head); a wave takes 16 rows, so a K/V block staged in
// LDS serves 64. Per 32-key block:
//   S^T = K . Q^T  A = K rows from LDS, B = the wave's Q rows in registers.
//                  The contraction takes the dims in an order of its own --
//                  step e of a 16-dim group holds dims 4 (lane / 16) + e -- so
//                  that a lane's operands for 4 steps are one 16-byte read.
//   softmax        online maximum and sum per row; a lane holds 8 of the
//                  block's keys of row lane % 16
//   O += P . V     A = the S^T registers as they are (k-slot lane / 16 of
//                  step r is key 4 (lane / 16) + r); B = V rows from LDS, a
//                  16-byte read giving a lane 4 adjacent dims, one for each
//                  of 4 column tiles
// so that neither operand is transposed and every LDS read is 16 bytes. The
// next block's rows are loaded into registers while a block is computed and
// go to the other of two LDS buffers (one barrier a block).
// MFMA layout (checked on gfx950): A[i][k] in lane i + 16 k, B[k][j] in lane
// j + 16 k, D[i][j] in lane j + 16 (i / 4), register i % 4.
//
// Rows with a term that is not finite are computed again one by one, over
// their visible keys only: the blocks multiply a masked key's probability of
// zero with its value row, which may hold anything. So are rows without a
// sum, in natural units: logits past 1 / log2 e of the type's range.
#include <cmath>

#include "attention_split.hpp"

namespace cbk {
namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kWaves = 4;
constexpr int kThreads = 64 * kWaves;
constexpr int kKeys = kAttnKeyBlock;
constexpr float kLog2e = 1.4426950408889634f;
constexpr float kNegInf = -__builtin_inff();

__device__ __forceinline__ bool finite_bits(float x) { return (__float_as_uint(x) & 0x7f800000u) != 0x7f800000u; }

// One row's keys [k_lo, k_hi] by the whole wave: every lane two dims. The sum
// l and the maximum m (natural units) of the keys, o the lane's outputs.
__device__ void attend_row(const AttnF32Args& a, uint32_t qi, uint32_t h, int32_t k_lo, int32_t k_hi, uint32_t lane,
                           float& m, float& l, float& o0, float& o1) {
  const uint32_t kvh = h / a.group;
  const float* q = a.q + int64_t(qi) * a.q_stride + int64_t(h) * a.d;
  const float q0 = lane < a.d ? q[lane] : 0.f;
  const float q1 = lane + 64 < a.d ? q[lane + 64] : 0.f;
  m = kNegInf;
  l = o0 = o1 = 0.f;
  for (int32_t j = k_lo; j <= k_hi; ++j) {
    const float* kr = a.k + int64_t(j) * a.k_stride + int64_t(kvh) * a.d;
    const float* vr = a.v + int64_t(j) * a.v_stride + int64_t(kvh) * a.d;
    float dot = (lane < a.d ? q0 * kr[lane] : 0.f) + (lane + 64 < a.d ? q1 * kr[lane + 64] : 0.f);
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) dot += __shfl_xor(dot, off);
    const float x = dot * a.scale;
    const float mn = fmaxf(m, x);
    const float ms = mn == kNegInf ? 0.f : mn;
    const float alpha = expf(m - ms);
    const float p = expf(x - ms);
    l = l * alpha + p;
    o0 = o0 * alpha + p * (lane < a.d ? vr[lane] : 0.f);
    o1 = o1 * alpha + p * (lane + 64 < a.d ? vr[lane + 64] : 0.f);
    m = mn;
    if (l != l) {  // NaN from here on in every lane (uniform): a bad key that many rows see early
      o0 = o1 = l;
      return;
    }
  }
}

// Two workgroups per CU at DP 128 (66 KiB of LDS each).
template <int DP, bool VEC>
__global__ __launch_bounds__(kThreads, 2) void attn_f32_kernel(const AttnF32Args a) {
  constexpr int NT = DP / 16;        // 16-dim groups
  constexpr int CC = DP / 64;        // 64-dim column groups of the output
  constexpr int LD = DP + 4;         // LDS row: 16 rows' 16-byte reads fall on distinct banks
  constexpr int P = DP / 4;          // 16-byte pieces per row
  constexpr int ROWS = kThreads / P;  // rows the workgroup loads at a time
  constexpr int N = kKeys / ROWS;    // loads per thread and block, each of K and V
  __shared__ __attribute__((aligned(16))) float kbuf[2][kKeys * LD];
  __shared__ __attribute__((aligned(16))) float vbuf[2][kKeys * LD];
  __shared__ int32_t s_max[kWaves];
  const uint32_t lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t row = lane & 15, grp = lane >> 4;
  // workgroup -> (tile, key range, KV head), the KV head fastest and the
  // latest tiles (most keys) first
  const uint32_t S = a.parts.splits;
  const uint32_t kvh = __builtin_amdgcn_readfirstlane(blockIdx.x % a.hkv);
  const uint32_t rest = __builtin_amdgcn_readfirstlane(blockIdx.x / a.hkv);
  const uint32_t split = __builtin_amdgcn_readfirstlane(rest % S);
  const uint32_t nrows = a.nq * a.group;
  const uint32_t ntiles = (nrows + kAttnF32Rows - 1) / kAttnF32Rows;
  const uint32_t tile = __builtin_amdgcn_readfirstlane(ntiles - 1 - rest / S);
  const uint32_t r0 = tile * kAttnF32Rows + wave * 16;  // the wave's first row
  const uint32_t r = r0 + row;
  const bool valid = r < nrows;
  const uint32_t qi = valid ? r / a.group : 0;
  const uint32_t qh = kvh * a.group + (valid ? r % a.group : 0);
  const int32_t rpos = valid ? int32_t(max(min(a.pos[qi], int64_t(a.nk) - 1), int64_t(-1))) : -1;

  f32x4 qf[NT];
  {
    const float* q = a.q + int64_t(qi) * a.q_stride + int64_t(qh) * a.d;
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const uint32_t d0 = 16 * t + 4 * grp;
      qf[t] = f32x4{0.f, 0.f, 0.f, 0.f};
      if (!valid) continue;
      if constexpr (VEC) {
        if (d0 < a.d) qf[t] = *reinterpret_cast<const f32x4*>(q + d0);
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (d0 + e < a.d) qf[t][e] = q[d0 + e];
      }
    }
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
  // the workgroup's blocks: its share of the tile's
  const uint32_t nblocks = gmax < 0 ? 0u : uint32_t(gmax) / kKeys + 1;
  const int32_t b_lo = int32_t(uint64_t(nblocks) * split / S), b_hi = int32_t(uint64_t(nblocks) * (split + 1) / S);

  // this thread's pieces of a block: rows lr + ROWS i, dims 4 lp ..
  const uint32_t lr = threadIdx.x / P, lp = threadIdx.x % P;
  f32x4 kreg[N], vreg[N];
  auto piece = [&](const float* p) __attribute__((always_inline)) {
    f32x4 w = f32x4{0.f, 0.f, 0.f, 0.f};
    if constexpr (VEC) {
      if (4 * lp < a.d) w = *reinterpret_cast<const f32x4*>(p);
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (4 * lp + e < a.d) w[e] = p[e];
    }
    return w;
  };
  auto load = [&](int32_t b) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const int32_t key = b * kKeys + int32_t(lr) + ROWS * i;
      kreg[i] = vreg[i] = f32x4{0.f, 0.f, 0.f, 0.f};
      if (key < int32_t(a.nk)) {
        kreg[i] = piece(a.k + int64_t(key) * a.k_stride + int64_t(kvh) * a.d + 4 * lp);
        vreg[i] = piece(a.v + int64_t(key) * a.v_stride + int64_t(kvh) * a.d + 4 * lp);
      }
    }
  };

  f32x4 o[CC * 4];
#pragma unroll
  for (int c = 0; c < CC * 4; ++c) o[c] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m = kNegInf, l = 0.f;  // log2 units; l of this lane's keys only
  const float c2 = a.scale * kLog2e;
  if (b_lo < b_hi) load(b_lo);
  for (int32_t b = b_lo; b < b_hi; ++b) {
    float* ks = kbuf[b & 1];
    float* vs = vbuf[b & 1];
#pragma unroll
    for (int i = 0; i < N; ++i) {
      *reinterpret_cast<f32x4*>(&ks[(lr + ROWS * i) * LD + 4 * lp]) = kreg[i];
      *reinterpret_cast<f32x4*>(&vs[(lr + ROWS * i) * LD + 4 * lp]) = vreg[i];
    }
    __syncthreads();  // block b is in LDS, and every wave is done with block b - 1's buffer
    if (b + 1 < b_hi) load(b + 1);
    if (wmax < b * kKeys) continue;  // no row of the wave sees the block
    f32x4 s[2] = {f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      f32x4 kf[2];
#pragma unroll
      for (int h = 0; h < 2; ++h) kf[h] = *reinterpret_cast<const f32x4*>(&ks[(16 * h + row) * LD + 16 * t + 4 * grp]);
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int h = 0; h < 2; ++h) s[h] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[h][e], qf[t][e], s[h], 0, 0, 0);
    }
    float x[2][4], bm = kNegInf;
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        x[h][i] = s[h][i] * c2;
        if (wmin < b * kKeys + kKeys - 1 && b * kKeys + 16 * h + int32_t(4 * grp) + i > rpos) x[h][i] = kNegInf;
        bm = fmaxf(bm, x[h][i]);
      }
    bm = fmaxf(bm, __shfl_xor(bm, 16));
    bm = fmaxf(bm, __shfl_xor(bm, 32));
    if (__any(bm > m)) {  // some row's maximum rose
      const float mn = fmaxf(m, bm);
      const float alpha = mn == m ? 1.f : __builtin_amdgcn_exp2f(m - mn);
      m = mn;
      l *= alpha;
      float ao[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) ao[i] = __shfl(alpha, int(4 * grp + i));
#pragma unroll
      for (int c = 0; c < CC * 4; ++c)
#pragma unroll
        for (int i = 0; i < 4; ++i) o[c][i] *= ao[i];
    }
    const float ms = m == kNegInf ? 0.f : m;
    float p[2][4];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
#pragma unroll
      for (int i = 0; i < 4; ++i) p[h][i] = __builtin_amdgcn_exp2f(x[h][i] - ms);
      l += (p[h][0] + p[h][1]) + (p[h][2] + p[h][3]);
    }
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int c = 0; c < CC; ++c) {
          const f32x4 vf = *reinterpret_cast<const f32x4*>(&vs[(16 * h + 4 * grp + i) * LD + 64 * c + 4 * row]);
#pragma unroll
          for (int e = 0; e < 4; ++e)
            o[4 * c + e] = __builtin_amdgcn_mfma_f32_16x16x4f32(p[h][i], vf[e], o[4 * c + e], 0, 0, 0);
        }
  }
  l += __shfl_xor(l, 16);
  l += __shfl_xor(l, 32);

  // the wave's rows with a term that is not finite, or with keys but no sum
  // (logits that are finite by themselves, -inf times log2 e): redone below.
  // Rows past the last one count as little as their lanes do: their zeros
  // times a value that is not finite are NaN too, and nothing of theirs may be
  // read or written.
  uint32_t bad = 0;
  {
    const uint64_t lb = __ballot(!finite_bits(l) || (l == 0.f && b_lo < b_hi && rpos >= b_lo * kKeys));
    bad = uint32_t((lb | (lb >> 16) | (lb >> 32) | (lb >> 48)) & 0xffffu);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      bool f = true;
#pragma unroll
      for (int c = 0; c < CC * 4; ++c) f = f && finite_bits(o[c][i]);
      const uint64_t ob = __ballot(!f);
#pragma unroll
      for (int g = 0; g < 4; ++g)
        if ((ob >> (16 * g)) & 0xffffu) bad |= 1u << (4 * g + i);
    }
    bad &= uint32_t(__ballot(valid)) & 0xffffu;  // lanes 0..15 hold rows 0..15
  }
  const uint64_t rows_all = uint64_t(a.nq) * a.hq;
  // lane group grp holds rows 4 grp + i, dims 64 c + 4 (lane % 16) + e
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const uint32_t rr = 4 * grp + i, gr = r0 + rr;
    const float rl = __shfl(l, int(rr)), rm = __shfl(m, int(rr));
    const int32_t rp = __shfl(rpos, int(rr));
    if (gr >= nrows || ((bad >> rr) & 1u)) continue;
    const uint32_t oq = gr / a.group, oh = kvh * a.group + gr % a.group;
    float* dst;
    float f;
    if (S == 1) {
      dst = a.out + int64_t(oq) * a.out_stride + int64_t(oh) * a.d;
      // a sum of zero: no visible keys, or all their logits -inf (NaN)
      f = rl > 0.f ? 1.f / rl : rp >= 0 ? __uint_as_float(0x7fc00000u) : 0.f;
    } else {
      const uint64_t id = split * rows_all + uint64_t(oq) * a.hq + oh;
      dst = a.parts.o + id * a.d;
      f = 1.f;
      if (row == 0) a.parts.ml[id] = make_float2(0.5f * rm, rl);
    }
#pragma unroll
    for (int c = 0; c < CC; ++c) {
      const uint32_t d0 = 64 * c + 4 * row;
      const f32x4 w = f32x4{o[4 * c][i] * f, o[4 * c + 1][i] * f, o[4 * c + 2][i] * f, o[4 * c + 3][i] * f};
      if constexpr (VEC) {
        if (d0 < a.d) *reinterpret_cast<f32x4*>(dst + d0) = w;
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (d0 + e < a.d) dst[d0 + e] = w[e];
      }
    }
  }
  while (bad) {  // uniform
    const uint32_t rr = uint32_t(__builtin_ctz(bad)), gr = r0 + rr;
    bad &= bad - 1;
    const int32_t last = min(__builtin_amdgcn_readfirstlane(__shfl(rpos, int(rr))), b_hi * kKeys - 1);
    const uint32_t oq = gr / a.group, oh = kvh * a.group + gr % a.group;
    float fm, fl, o0, o1;
    attend_row(a, oq, oh, b_lo * kKeys, last, lane, fm, fl, o0, o1);
    float* dst;
    float f = 1.f;
    if (S == 1) {
      dst = a.out + int64_t(oq) * a.out_stride + int64_t(oh) * a.d;
      f = fl > 0.f ? 1.f / fl : last >= 0 ? __uint_as_float(0x7fc00000u) : 0.f;
    } else {
      const uint64_t id = split * rows_all + uint64_t(oq) * a.hq + oh;
      dst = a.parts.o + id * a.d;
      if (lane == 0) a.parts.ml[id] = make_float2(fm * (0.5f * kLog2e), fl);
    }
    if (lane < a.d) dst[lane] = o0 * f;
    if (lane + 64 < a.d) dst[lane + 64] = o1 * f;
  }
}

}  // namespace

int launch_attn_f32(const AttnF32Args& a, hipStream_t stream) {
  const uint64_t nrows = uint64_t(a.nq) * a.group;
  const uint64_t tiles = (nrows + kAttnF32Rows - 1) / kAttnF32Rows;
  const uint64_t groups = tiles * a.hkv * a.parts.splits;
  CBK_REQUIRE(groups * kThreads < (uint64_t(1) << 32), "blend attention f32: %llu workgroups exceed one launch",
              (unsigned long long)groups);
  const int64_t align[9] = {a.q_stride * 4, a.k_stride * 4, a.v_stride * 4, a.out_stride * 4, int64_t(a.d) * 4,
                            int64_t(reinterpret_cast<uintptr_t>(a.q)), int64_t(reinterpret_cast<uintptr_t>(a.k)),
                            int64_t(reinterpret_cast<uintptr_t>(a.v)), int64_t(reinterpret_cast<uintptr_t>(a.out))};
  const bool vec = common_vec_bytes(align, 9) == 16;
  const dim3 grid(static_cast<uint32_t>(groups)), block(kThreads);
  if (a.d <= 64) {
    if (vec) hipLaunchKernelGGL((attn_f32_kernel<64, true>), grid, block, 0, stream, a);
    else hipLaunchKernelGGL((attn_f32_kernel<64, false>), grid, block, 0, stream, a);
  } else {
    if (vec) hipLaunchKernelGGL((attn_f32_kernel<128, true>), grid, block, 0, stream, a);
    else hipLaunchKernelGGL((attn_f32_kernel<128, false>), grid, block, 0, stream, a);
  }
  return launch_status("blend attention f32");
}

}  // namespace cbk
