// A prompt pass's rows before its attention (asrlayer_prompt_rows).
//
// Bound by memory: every row (one head of one token) is read once and written
// once, keys and normalized values twice (packed for the attention, and to
// the cache).  As separate operations the same work reads and writes the rows
// some ten times: Qwen3's prompt pass of 8 x 400-430 tokens (16 + 2 x 8 heads
// of 128, bf16; 27 MB read, 34 MB written) took 215 us in 14 launches, and
// takes 16.4 here (3.7 TB/s; 19.0 with the tables loaded for every row, the
// slot looked up for every lane group and the values' norm computed unasked).
//
// A workgroup takes one token: its rotation tables are loaded once and its
// cache slot is looked up once.  A row of head_dim elements is held by LPK lanes
// of 16 bytes (two vectors a lane for float rows of 512); neighbouring lane
// groups take neighbouring rows, so a wave reads whole cache lines, and each
// group has two rows' loads in flight before it computes.
#include "kernels.hpp"
#include "layers.hpp"
#include "row_ops.hpp"

namespace asrattn {
namespace {

constexpr int kThreads = 256;

template <typename T, int HD>
struct PromptShape {
  static constexpr int kEPL = Elem<T>::kPerVec;
  static constexpr int kVecs = HD / kEPL > 64 ? HD / kEPL / 64 : 1;  // vectors per lane
  static constexpr int kLPK = HD / kEPL / kVecs;                     // lanes per row
  static constexpr int kGroups = kThreads / kLPK;                    // lane groups per workgroup
  static constexpr int kRows = kVecs > 1 ? 1 : 2;                    // rows a lane group has in flight
};

// Float rows of 512: vector v of a lane holds elements 256 v + 4 lane .. +3,
// so an element's rotation partner is in the lane's other vector.
__device__ __forceinline__ void wide_row(uint4* raw, bool norm, bool weighted, const uint4* w, bool rotated,
                                         const uint4* cs, const uint4* sn, float eps) {
  float x[8], wv[8], c[8], s[8];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    unpack<float>(raw[i], x + 4 * i);
    unpack<float>(w[i], wv + 4 * i);
    unpack<float>(cs[i], c + 4 * i);
    unpack<float>(sn[i], s + 4 * i);
  }
  float ss = 0.f;
#pragma unroll
  for (int e = 0; e < 8; ++e) ss = fmaf(x[e], x[e], ss);
  ss = group_sum<64>(ss);
  const float r = rsqrtf(ss * (1.f / 512) + eps);
#pragma unroll
  for (int e = 0; e < 8; ++e) x[e] = norm ? (weighted ? x[e] * r * wv[e] : x[e] * r) : x[e];
  float y[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const float a = x[e] * c[e];
    const float b = (e < 4 ? -x[e + 4] : x[e - 4]) * s[e];
    y[e] = rotated ? a + b : x[e];
  }
  raw[0] = pack<float>(y);
  raw[1] = pack<float>(y + 4);
}

template <typename T, int HD>
__global__ __launch_bounds__(kThreads) void prompt_rows_kernel(const asrlayer_prompt_params p) {
  using S = PromptShape<T, HD>;
  constexpr int EPL = S::kEPL, LPK = S::kLPK, NV = S::kVecs, NR = S::kRows, NG = S::kGroups;
  const int sub = threadIdx.x % LPK;
  const int group = threadIdx.x / LPK;
  const int tok = blockIdx.x;
  const int b = tok / p.tokens, t = tok % p.tokens;
  const int heads_kv = p.k != nullptr ? p.heads_kv : 0;
  const int rows = p.heads_q + 2 * heads_kv;  // queries, keys, values

  uint4 cs[NV], sn[NV];
  const int64_t rope = b * p.rope_batch_stride + t * p.rope_token_stride;
#pragma unroll
  for (int v = 0; v < NV; ++v) {
    const int at = (v * LPK + sub) * EPL;
    cs[v] = *reinterpret_cast<const uint4*>(static_cast<const T*>(p.cos) + rope + at);
    sn[v] = *reinterpret_cast<const uint4*>(static_cast<const T*>(p.sin) + rope + at);
  }

  // The token's slot in the cache (uniform).
  bool write = p.k_cache != nullptr;
  int64_t row = 0, pos = t;
  if (write) {
    row = load_uniform(p.rows + (p.positions != nullptr ? tok : b));
    if (p.positions != nullptr) pos = load_uniform(p.positions + tok);
    if (row < 0) row += p.cache_rows;
    write = row >= 0 && row < p.cache_rows;
    if (p.block_table != nullptr) {
      int64_t entry = pos >= 0 ? pos / p.page_size : -((-pos + p.page_size - 1) / p.page_size);
      pos -= entry * p.page_size;
      if (entry < 0) entry += p.bt_stride;
      write = write && entry >= 0 && entry < p.bt_stride;
      if (write) {
        const int32_t page = load_uniform(p.block_table + (row * p.bt_stride + entry));
        row = page >= 0 && page < p.num_pages ? page : p.num_pages;
      }
    } else {
      if (pos < 0) pos += p.cache_length;
      write = write && pos >= 0 && pos < p.cache_length;
    }
  }

  // Rows past the last repeat it (and are not stored): every lane takes part
  // in the row sums.
  for (int r0 = 0; r0 < rows; r0 += NR * NG) {
    uint4 raw[NR][NV], w[NR][NV];
    int index[NR];
#pragma unroll
    for (int i = 0; i < NR; ++i) {
      index[i] = r0 + i * NG + group;
      const int r = min(index[i], rows - 1);
      const bool is_q = r < p.heads_q, is_v = r >= p.heads_q + heads_kv;
      const int h = is_q ? r : r - p.heads_q - (is_v ? heads_kv : 0);
      const T* src = static_cast<const T*>(is_q ? p.q : is_v ? p.v : p.k);
      src += b * (is_q ? p.q_batch_stride : is_v ? p.v_batch_stride : p.k_batch_stride) +
             t * (is_q ? p.q_token_stride : is_v ? p.v_token_stride : p.k_token_stride) +
             h * (is_q ? p.q_head_stride : is_v ? p.v_head_stride : p.k_head_stride);
      const T* wp = static_cast<const T*>(is_q || p.k == nullptr ? p.q_norm : p.k_norm);
#pragma unroll
      for (int v = 0; v < NV; ++v) {
        const int at = (v * LPK + sub) * EPL;
        raw[i][v] = *reinterpret_cast<const uint4*>(src + at);
        w[i][v] = *reinterpret_cast<const uint4*>(wp + at);
      }
    }
#pragma unroll
    for (int i = 0; i < NR; ++i) {
      const int r = min(index[i], rows - 1);
      const bool is_q = r < p.heads_q, is_v = r >= p.heads_q + heads_kv;
      const int h = is_q ? r : r - p.heads_q - (is_v ? heads_kv : 0);
      const float eps = is_q ? p.q_eps : is_v ? p.v_eps : p.k_eps;
      const bool norm = !is_v || p.v_norm != 0;
      if (__any(norm)) {  // a wave of values alone copies them
        if constexpr (NV == 1)
          raw[i][0] = prologue_row<T, HD, LPK>(raw[i][0], true, norm, !is_v, w[i][0], true, !is_v, cs[0], sn[0], eps, sub);
        else
          wide_row(raw[i], norm, !is_v, w[i], !is_v, cs, sn, eps);
      }
      if (index[i] >= rows) continue;
      T* out = static_cast<T*>(is_q ? p.q_out : is_v ? p.v_out : p.k_out);
      if (out != nullptr) {
        out += ((int64_t)tok * (is_q ? p.heads_q : p.heads_kv) + h) * HD;
#pragma unroll
        for (int v = 0; v < NV; ++v) *reinterpret_cast<uint4*>(out + (v * LPK + sub) * EPL) = raw[i][v];
      }
      if (is_q || !write) continue;
      T* cache = static_cast<T*>(is_v ? p.v_cache : p.k_cache);
      cache += row * (is_v ? p.vc_row_stride : p.kc_row_stride) + pos * (is_v ? p.vc_pos_stride : p.kc_pos_stride) +
               h * (is_v ? p.vc_head_stride : p.kc_head_stride);
#pragma unroll
      for (int v = 0; v < NV; ++v) *reinterpret_cast<uint4*>(cache + (v * LPK + sub) * EPL) = raw[i][v];
    }
  }
}

template <typename T, int HD>
hipError_t launch_hd(const asrlayer_prompt_params& p, hipStream_t stream) {
  hipLaunchKernelGGL((prompt_rows_kernel<T, HD>), dim3((unsigned)(p.batch * p.tokens)), dim3(kThreads), 0, stream, p);
  return hipGetLastError();
}

template <typename T>
hipError_t launch_typed(const asrlayer_prompt_params& p, hipStream_t stream) {
  switch (p.head_dim) {
    case 64: return launch_hd<T, 64>(p, stream);
    case 128: return launch_hd<T, 128>(p, stream);
    case 256: return launch_hd<T, 256>(p, stream);
    default: return launch_hd<T, 512>(p, stream);
  }
}

}  // namespace

hipError_t launch_prompt_rows(const asrlayer_prompt_params& p, hipStream_t stream) {
  return p.dtype == ASRATTN_BF16 ? launch_typed<bf16_raw>(p, stream) : launch_typed<float>(p, stream);
}

}  // namespace asrattn
