// Multi-row attention in fp32 at head_dim 64 on v_mfma_f32_16x16x4_f32 (fp32
// operands and accumulation; the rate of the 32 x 32 instruction).
//
// Workgroup: KS waves over RB blocks of 16 query rows of one (sequence, head);
// wave ks takes the key sub-tiles ks, ks + KS, ... (32 keys each) and the waves
// merge their (O, max, sum) through LDS at the end.  Blocks of 16 rows let the
// row count of a workgroup follow the launch: Whisper-tiny's encoder (6 heads x
// 1500 rows) is 192 workgroups of 48 rows, one per CU, where 282 of 32 rows
// left 26 CUs with twice the work of the others (49.1 against 63.7 us, 70 TFLOP/s
// of the 157 the instruction reaches); and the K and V operands are loaded once
// for RB * 16 rows.
//
// The products are the transposed ones of the other kernels:
//
//   S^T = K . Q^T    A = 16 keys x 4 head dims, B = Q^T: a lane's accumulators
//                    are keys 4 g + r of query row lane % 16 (g = lane / 16).
//   O^T = V^T . P^T  A = 16 head dims x 4 keys, B = P^T straight from the S^T
//                    accumulators: step r takes keys 4 g + r.
//
// Any assignment of head dims to the k slots (and of output rows to head dims)
// gives the same products, so both operands are 16-byte loads: step 4 j + e of
// S^T takes dim 16 j + 4 g + e, and V^T block e has dims 4 i + e (i = lane % 16),
// of which a lane's output registers hold runs of four.
//
// A sub-tile's K registers are free once its scores are done and take the next
// sub-tile's keys while the softmax and the value products run; V's likewise:
// no second set of operand registers.  The loads are unconditional; past the
// block's last key they read zeros.
//
// Softmax in base 2 with scale * log2(e) folded into one FMA per score; the
// running max is lazy (rescale only when a row's max grows by more than 2^8).
#include "common.hpp"
#include "fwd_common.hpp"
#include "kernels.hpp"
#include "ring_common.hpp"

namespace asrattn {
namespace {

typedef float f32x4_t __attribute__((ext_vector_type(4)));

__device__ __forceinline__ f32x4_t mfma16(float a, float b, const f32x4_t& c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ f32x4_t load4(__amdgpu_buffer_rsrc_t rsrc, uint32_t voffset) {
  return __builtin_bit_cast(f32x4_t, __builtin_amdgcn_raw_buffer_load_b128(rsrc, voffset, 0, 0));
}

constexpr int kHD = 64;
constexpr int kFewKeys = 512;

// x and its value in lanes l ^ 16, l ^ 32 and l ^ 48 (the lanes of the same
// query row), folded by `op`.
template <typename Op>
__device__ __forceinline__ float over_row(float x, Op op) {
  float a, b;
  lane_pair<16>(x, a, b);
  x = op(a, b);
  lane_pair<32>(x, a, b);
  return op(a, b);
}

template <int RB, int KS, bool WIN>
__global__ __launch_bounds__(64 * KS, 2) void fwd_f32row_kernel(const FwdArgs a, int q_tiles, int total) {
  constexpr int BM = 16 * RB;
  const asrattn_fwd_params& p = a.p;
  // Each XCD takes a contiguous range of (sequence, head, row block) items,
  // so a head's keys and values stay in that XCD's L2 for all its row blocks.
  const int item = ring::xcd_remap((int)blockIdx.x, total);
  const int qt = item % q_tiles;
  const int hq = (item / q_tiles) % p.heads_q;
  const int b = item / q_tiles / p.heads_q;
  const int hkv = hq / (p.heads_q / p.heads_kv);
  const SeqView sv = seq_view(p, b, hq, hkv);
  const int row0 = qt * BM;
  if (row0 >= sv.len_q) return;  // uniform over the workgroup
  const int len_c = (p.flags & ASRATTN_FWD_ZERO_PADDED_ROWS) != 0 ? min(sv.len_q, sv.n_k) : sv.len_q;
  const int tid = threadIdx.x;
  if (row0 >= len_c) {
    // Rows at or past the key count of a zero-padded batch: zeros.
    for (int i = tid; i < (min(row0 + BM, sv.len_q) - row0) * (kHD / 4); i += 64 * KS) {
      float* op = static_cast<float*>(p.out) + sv.o_off + (int64_t)(row0 + i / (kHD / 4)) * p.o_token_stride +
                  (i % (kHD / 4)) * 4;
      *reinterpret_cast<float4*>(op) = make_float4(0.f, 0.f, 0.f, 0.f);
    }
    return;
  }
  const int lane = tid & 63;
  const int ks = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int i16 = lane & 15;
  const int g = lane >> 4;

  const int kend = visible_keys(p, sv, min(row0 + BM, len_c) - 1);
  const int n_sub = (kend + 31) / 32;
  const int sub0 = WIN ? min(first_key(p, sv, row0), kend) / 32 : 0;  // the block's first sub-tile
  // Row lane % 16 of each block: its queries and the keys it sees.
  float q[RB][16];
  int row_lim[RB], row_lo[RB];
  bool row_ok[RB];
#pragma unroll
  for (int rb = 0; rb < RB; ++rb) {
    const int row = row0 + 16 * rb + i16;
    row_ok[rb] = row < len_c;
    row_lim[rb] = row_ok[rb] ? visible_keys(p, sv, row) : 0;
    row_lo[rb] = WIN ? first_key(p, sv, row) : 0;
    const float* qp =
        static_cast<const float*>(p.q) + sv.q_off + (int64_t)(row_ok[rb] ? row : 0) * p.q_token_stride + 4 * g;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float4 v = *reinterpret_cast<const float4*>(qp + 16 * j);
      q[rb][4 * j] = v.x;
      q[rb][4 * j + 1] = v.y;
      q[rb][4 * j + 2] = v.z;
      q[rb][4 * j + 3] = v.w;
    }
  }
  // Sub-tiles before `plain` hold only keys every row of the block sees (the
  // first row sees the fewest; with a window all take the mask).
  const int plain = WIN || row0 + BM > len_c ? 0 : visible_keys(p, sv, row0) / 32;

  const uint32_t kts = (uint32_t)p.k_token_stride * 4;
  const uint32_t vts = (uint32_t)p.v_token_stride * 4;
  const __amdgpu_buffer_rsrc_t krs = buffer_rsrc(static_cast<const float*>(p.k) + sv.k_off, (uint32_t)kend * kts);
  const __amdgpu_buffer_rsrc_t vrs = buffer_rsrc(static_cast<const float*>(p.v) + sv.v_off, (uint32_t)kend * vts);
  // K row i16 at head dims 16 j + 4 g; V row 4 g + r at head dims 4 i16.
  const uint32_t koff = (uint32_t)i16 * kts + (uint32_t)g * 16;
  const uint32_t voff = (uint32_t)(4 * g) * vts + (uint32_t)i16 * 16;
  f32x4_t kr[2][4], vr[2][4];
  auto load_k = [&](int sub) {
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int j = 0; j < 4; ++j) kr[kb][j] = load4(krs, (uint32_t)(sub * 32 + kb * 16) * kts + koff + (uint32_t)j * 64);
  };
  auto load_v = [&](int sub) {
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int r = 0; r < 4; ++r) vr[kb][r] = load4(vrs, (uint32_t)(sub * 32 + kb * 16 + r) * vts + voff);
  };

  f32x4_t o[4][RB];
  float m_run[RB], l_run[RB];
#pragma unroll
  for (int rb = 0; rb < RB; ++rb) {
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e][rb] = f32x4_t{};
    m_run[rb] = kNegInf;
    l_run[rb] = 0.f;
  }
  const float c = a.c;
  constexpr float kLazy = 8.f;

  load_k(sub0 + ks);
  load_v(sub0 + ks);
  for (int sub = sub0 + ks; sub < n_sub; sub += KS) {
    f32x4_t s[2][RB];
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int rb = 0; rb < RB; ++rb) s[kb][rb] = f32x4_t{};
#pragma unroll
    for (int t = 0; t < 16; ++t)
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int rb = 0; rb < RB; ++rb) s[kb][rb] = mfma16(kr[kb][t / 4][t % 4], q[rb][t], s[kb][rb]);
    load_k(sub + KS);
    if (sub >= plain) {
      // Keys outside the row's range -> -inf (register r of block kb: key
      // 32 sub + 16 kb + 4 g + r).
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int rb = 0; rb < RB; ++rb)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int key = sub * 32 + kb * 16 + 4 * g + r;
            if (key >= row_lim[rb] || (WIN && key < row_lo[rb])) s[kb][rb][r] = kNegInf;
          }
    }
    float mt[RB];
    bool grow = false;
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) {
      float x = fmaxf(s[0][rb][0], s[1][rb][0]);
#pragma unroll
      for (int r = 1; r < 4; ++r) x = fmaxf(x, fmaxf(s[0][rb][r], s[1][rb][r]));
      mt[rb] = over_row(x, [](float u, float v) { return fmaxf(u, v); }) * c;
      grow = grow || mt[rb] > m_run[rb] + kLazy;
    }
    if (__any(grow)) {
#pragma unroll
      for (int rb = 0; rb < RB; ++rb) {
        const float mn = fmaxf(m_run[rb], mt[rb]);
        const float alpha = mn == kNegInf ? 1.f : fast_exp2(m_run[rb] - mn);
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e][rb] *= alpha;
        l_run[rb] *= alpha;
        m_run[rb] = mn;
      }
    }
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) {
      const float mu = m_run[rb] == kNegInf ? 0.f : m_run[rb];
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          s[kb][rb][r] = fast_exp2(fmaf(s[kb][rb][r], c, -mu));
          l_run[rb] += s[kb][rb][r];
        }
    }
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
          for (int rb = 0; rb < RB; ++rb) o[e][rb] = mfma16(vr[kb][r][e], s[kb][rb][r], o[e][rb]);
    load_v(sub + KS);
  }

  // The lanes of a row hold disjoint keys of it.
#pragma unroll
  for (int rb = 0; rb < RB; ++rb) l_run[rb] = over_row(l_run[rb], [](float u, float v) { return u + v; });

  // Merge the key splits through LDS: every wave stores its (O^T, max, sum), and
  // wave r of the first four folds register r of every block and writes it
  // (register r of block e: head dim 4 (4 g + r) + e).
  static_assert(KS >= 4, "four waves write the output");
  constexpr int kPer = 18 * RB * 64;
  __shared__ float mf[KS * kPer];
  {
    float* dst = mf + ks * kPer + lane;
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) {
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int e = 0; e < 4; ++e) dst[(18 * rb + 4 * r + e) * 64] = o[e][rb][r];
      dst[(18 * rb + 16) * 64] = m_run[rb];
      dst[(18 * rb + 17) * 64] = l_run[rb];
    }
  }
  __syncthreads();
  if (ks >= 4) return;
#pragma unroll
  for (int rb = 0; rb < RB; ++rb) {
    const float* src = mf + 18 * rb * 64 + lane;
    float m[KS];
    float mx = kNegInf;
#pragma unroll
    for (int k = 0; k < KS; ++k) {
      m[k] = src[k * kPer + 16 * 64];
      mx = fmaxf(mx, m[k]);
    }
    const float mu = mx == kNegInf ? 0.f : mx;
    float l = 0.f, y[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int k = 0; k < KS; ++k) {
      const float w = fast_exp2(m[k] - mu);
      l = fmaf(src[k * kPer + 17 * 64], w, l);
#pragma unroll
      for (int e = 0; e < 4; ++e) y[e] = fmaf(src[k * kPer + (4 * ks + e) * 64], w, y[e]);
    }
    const int row = row0 + 16 * rb + i16;
    if (row >= sv.len_q) continue;
    const float inv = l > 0.f && row_ok[rb] ? 1.f / l : 0.f;  // rows past len_c get zeros
    float* op = static_cast<float*>(p.out) + sv.o_off + (int64_t)row * p.o_token_stride + 16 * g + 4 * ks;
    *reinterpret_cast<float4*>(op) = make_float4(y[0] * inv, y[1] * inv, y[2] * inv, y[3] * inv);
  }
}

template <int RB, int KS>
hipError_t launch_rb(const FwdArgs& a, hipStream_t stream) {
  const int q_tiles = (a.p.max_len_q + 16 * RB - 1) / (16 * RB);
  const long long total = (long long)q_tiles * a.p.heads_q * a.p.batch;
  if (total > 0x7fffffffLL) return hipErrorInvalidConfiguration;
  if (a.p.window > 0)
    hipLaunchKernelGGL((fwd_f32row_kernel<RB, KS, true>), dim3((unsigned)total), dim3(64 * KS), 0, stream, a, q_tiles,
                       (int)total);
  else
    hipLaunchKernelGGL((fwd_f32row_kernel<RB, KS, false>), dim3((unsigned)total), dim3(64 * KS), 0, stream, a, q_tiles,
                       (int)total);
  return hipGetLastError();
}

}  // namespace

// The 32-row kernel (fwd_f32mm.hip) is faster for launches of many row blocks
// over few keys, where the merge of this one's key splits weighs most: no
// window, at least 600 row blocks, and keys of two sub-tiles at most (64 rows, 20
// x 16 heads 13.5 us here, 11.2 there), or at most 512 (200 causal ones, the rows
// seeing half of them) while its waves -- a row block each, two where 2048 still
// hold them all -- fill at least 65% of the rounds they take: 260 rows, 12 x 16
// heads (1728 waves) 53.9 here, 51.0 there, 20 x 16 (2880) 81.5 and 76.8; 8 x 16
// (1152) 38.3 and 45.5.
bool fwd_f32row_takes(const asrattn_fwd_params& p) {
  if (p.window > 0 || p.max_len_k > kFewKeys) return true;
  const long long blocks = (long long)((p.max_len_q + 31) / 32) * p.heads_q * p.batch;
  if (blocks < 600) return true;
  if (p.max_len_k <= 64) return false;
  if (p.causal != ASRATTN_CAUSAL_NONE && p.max_len_k > 200) return true;
  const long long waves = blocks <= 1024 ? 2 * blocks : blocks;
  const long long rounds = (waves + 2047) / 2048;
  return waves * 100 < rounds * 2048 * 65;
}

hipError_t launch_fwd_f32row(const asrattn_fwd_params& p, hipStream_t stream) {
  FwdArgs a;
  a.p = p;
  a.c = p.scale * kLog2e;
  a.f = FsmnArgs{};
  // Rows per workgroup: the fewest 16-row blocks on the fullest CU, weighted by
  // what a block costs in workgroups of one, two and three.  Over many keys the
  // blocks of a workgroup share the operands' loads, eight percent each: us per
  // launch, 1500 rows and keys, 16 / 32 / 48 rows: 6 heads 51.7 / 59.7 / 49.1, 12
  // heads 79.4 / 87.6 / 85.2, 18 heads 107.9 / 113.0 / 123.9, 20 heads 122.5 /
  // 113.1 / 125.5, 24 heads 136.3 / 139.1 / 125.9, 64 heads 347.6 / 323.3 / 314.8.
  // Over few keys the loads come from the caches, and causal blocks of fewer rows
  // meet fewer masked keys (300 causal rows, 8 x 2 heads 11.1 / 13.0 / 16.9, 8 x 16
  // 35.7 / 38.3 / 41.5; 448, 8 x 16 58.1 / 58.2 / 65.2), while unmasked ones pay for
  // the merge more often (260 rows, 20 x 8 heads 41.9 / 40.4 / 39.0).
  const bool few = p.max_len_k <= kFewKeys;
  const int weight1 = !few ? 112 : p.causal != ASRATTN_CAUSAL_NONE ? 84 : 118;
  auto groups = [&](int rb) { return (long long)((p.max_len_q + 16 * rb - 1) / (16 * rb)) * p.heads_q * p.batch; };
  auto cost = [&](int rb) { return (groups(rb) + 255) / 256 * rb * (rb == 1 ? weight1 : rb == 2 ? 104 : 96); };
  int rb = 3;
  if (cost(2) < cost(rb)) rb = 2;
  if (cost(1) < cost(rb)) rb = 1;
  if (rb == 3) return launch_rb<3, 4>(a, stream);
  if (rb == 2) return launch_rb<2, 4>(a, stream);
  // Eight key splits where few workgroups walk many keys: 6 heads x 4 rows over
  // 1500 keys 22.6 -> 21.8 us; 192 heads x 4 rows 33.2 with four, 35.2 with
  // eight.
  if (groups(1) <= 128 && p.max_len_k > 256) return launch_rb<1, 8>(a, stream);
  return launch_rb<1, 4>(a, stream);
}

}  // namespace asrattn
