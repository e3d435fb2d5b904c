// Decoder-step attention: one query per sequence over a key/value cache.
//
// The step is bound by HBM: every key and value of a sequence is read once
// and used for one (or, with grouped-query attention, g) dot products.  The
// kernel therefore streams K and V with 16-byte loads, keeps a second batch
// of loads in flight while it consumes the first, and does all arithmetic in
// registers:
//
//   * K and V are read once, with nontemporal loads (no L2 allocation).
//   * A key row (head_dim elements) is covered by LPK lanes, 16 bytes each;
//     a wave loads 64 / LPK key rows per instruction, so every load touches
//     whole rows.  Each group of LPK lanes runs its own online softmax over
//     the keys it reads (a "stream"); the g query heads sharing the kv head
//     ride along on the same loads.
//   * A workgroup of W waves covers one (sequence, kv head) -- or, for small
//     batches, one of `splits` key ranges of it.  Its streams merge first
//     inside each wave (a butterfly of lane swaps) and then across waves in
//     LDS.
//     With enough (sequence, kv head) pairs to fill the GPU there is one
//     split and the workgroup writes the output; otherwise each split writes
//     an unnormalized partial (o, max, sum) and the split that arrives last
//     folds them.  No workgroup waits on another.
//   * Sequence lengths are read from device memory (seqused_k or
//     positions + 1), and splits past a sequence's end write an empty
//     partial, so the grid depends only on shapes and the launch can be
//     replayed from a graph while lengths change.
//
// Softmax runs in base 2: each reduced score q . k is multiplied by
// scale * log2(e), so p = 2^(s - max) on v_exp_f32.
//
// Paged caches (asrattn_decode_paged): a load batch is U slices of NS
// consecutive keys (one key per stream), NS-aligned; with page sizes that
// are multiples of NS each slice lies in one page, whose pool index is one
// uniform (scalar) load from the block table.  The slice's buffer resource
// starts at that page and ends at the sequence's last key in it, so unused
// page slots and pages past the sequence are never read.
#pragma once

#include "common.hpp"
#include "decode_args.hpp"
#include "kernels.hpp"
#include "row_ops.hpp"

namespace asrattn {
namespace {


// s_waitcnt vmcnt(0) (gfx9 encoding; expcnt and lgkmcnt at their maxima).
constexpr int kWaitVmem = (0x7 << 4) | (0xF << 8);

template <typename T, int HD, int G, int W>
struct DecodeShape {
  static constexpr int kEPL = Elem<T>::kPerVec;   // elements per lane per load
  static constexpr int kLPK = HD / kEPL;          // lanes per key row
  static constexpr int kKPW = 64 / kLPK;          // key rows per wave load (streams per wave)
  static constexpr int kThreads = 64 * W;
  static constexpr int kStreams = W * kKPW;       // softmax streams per workgroup
  // Keys per stream per load batch; with four query heads per kv head the
  // batches are halved so that two of them fit beside the heads' state in
  // 128 VGPRs.
  static constexpr int kUnroll = G >= 4 || HD >= 256 ? 2 : 4;
  static constexpr int kStep = kStreams * kUnroll;  // keys per load batch
  // Plain (not append) kernels on 4-wave workgroups load two keys per
  // stream per batch instead of four: Qwen3's paged step 4.71 -> 4.93 TB/s,
  // its slab step +1%; the fused step lost 4% with two and keeps four.
  // Slab and paged variants sum in the same order either way.
  static constexpr int kPlainUnroll = W == 4 && kUnroll == 4 ? 2 : kUnroll;
  static constexpr int kPlainStep = kStreams * kPlainUnroll;
  // Waves per SIMD the register budget allows: four (128 VGPRs) up to four
  // query heads per kv head, two (256) for eight.
  static constexpr int kOcc = G >= 8 ? 2 : 4;
  // The cross-wave merge stages every wave's (G x HD) partial output in LDS.
  static constexpr bool kFits = W * G * HD * 4 <= 65536;
  static_assert(kLPK >= 1 && kLPK <= 64 && (64 % kLPK) == 0, "head_dim/lane mapping");
};

// q . k over one lane's 16-byte slices, accumulated in fp32.
template <typename T>
__device__ __forceinline__ float dot16(const uint4& q, const uint4& k);

template <>
__device__ __forceinline__ float dot16<float>(const uint4& q, const uint4& k) {
  float acc = __uint_as_float(q.x) * __uint_as_float(k.x);
  acc = fmaf(__uint_as_float(q.y), __uint_as_float(k.y), acc);
  acc = fmaf(__uint_as_float(q.z), __uint_as_float(k.z), acc);
  return fmaf(__uint_as_float(q.w), __uint_as_float(k.w), acc);
}

// bf16 pairs on v_dot2c_f32_bf16: the products of two bf16 values are exact
// in fp32, so this equals the unpacked fp32 dot product up to summation
// order.
template <>
__device__ __forceinline__ float dot16<bf16_raw>(const uint4& q, const uint4& k) {
  typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
  auto pair = [](uint32_t x) { return __builtin_bit_cast(bf16x2_t, x); };
  float acc = __builtin_amdgcn_fdot2_f32_bf16(pair(q.x), pair(k.x), 0.f, false);
  acc = __builtin_amdgcn_fdot2_f32_bf16(pair(q.y), pair(k.y), acc, false);
  acc = __builtin_amdgcn_fdot2_f32_bf16(pair(q.z), pair(k.z), acc, false);
  return __builtin_amdgcn_fdot2_f32_bf16(pair(q.w), pair(k.w), acc, false);
}

// Partials pass between workgroups on different XCDs, whose L2 caches are
// not coherent: agent-scope accesses go through to memory.
__device__ __forceinline__ void store_shared(float* p, float x) {
  __hip_atomic_store(p, x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ float load_shared(const float* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// p[0] and p[1], 8-byte aligned.
__device__ __forceinline__ void load_shared2(const float* p, float& first, float& second) {
  const float2 v = __builtin_bit_cast(float2, __hip_atomic_load(reinterpret_cast<const unsigned long long*>(p),
                                                                __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
  first = v.x;
  second = v.y;
}

// Online-softmax state of one stream for the G query heads of a kv head.
template <typename T, int HD, int G, int W>
struct Stream {
  using S = DecodeShape<T, HD, G, W>;
  static constexpr int EPL = S::kEPL;
  uint4 q[G];   // the lane's raw 16-byte slice of each query head
  float c;      // scale * log2(e), applied to the reduced score
  float m[G], l[G], o[G][EPL];

  // Starts the state from one key (k, v) when `mine`; the dot products run
  // on every lane (their reductions need the whole wave).
  __device__ __forceinline__ void seed(const uint4& k, const uint4& v, bool mine) {
    float vf[EPL];
    unpack<T>(v, vf);
#pragma unroll
    for (int g = 0; g < G; ++g) {
      const float s = group_sum<S::kLPK>(dot16<T>(q[g], k)) * c;
      if (mine) {
        m[g] = s;
        l[g] = 1.f;
#pragma unroll
        for (int e = 0; e < EPL; ++e) o[g][e] = vf[e];
      }
    }
  }

  __device__ __forceinline__ void init() {
#pragma unroll
    for (int g = 0; g < G; ++g) {
      m[g] = kNegInf;
      l[g] = 0.f;
#pragma unroll
      for (int e = 0; e < EPL; ++e) o[g][e] = 0.f;
    }
  }

  // Folds one load batch (raw 16-byte lane slices of K and V); key u is
  // valid when bit u of valid_mask is set.
  template <int U = S::kUnroll>
  __device__ __forceinline__ void consume(const uint4* kr, const uint4* vr, unsigned valid_mask) {
    float s[U][G];
#pragma unroll
    for (int u = 0; u < U; ++u) {
#pragma unroll
      for (int g = 0; g < G; ++g) {
        const float acc = group_sum<S::kLPK>(dot16<T>(q[g], kr[u]));
        s[u][g] = (valid_mask >> u) & 1u ? acc * c : kNegInf;
      }
    }
    float mu[G];
#pragma unroll
    for (int g = 0; g < G; ++g) {
      float mt = s[0][g];
#pragma unroll
      for (int u = 1; u < U; ++u) mt = fmaxf(mt, s[u][g]);
      const float mn = fmaxf(m[g], mt);
      mu[g] = mn == kNegInf ? 0.f : mn;
      const float alpha = fast_exp2(m[g] - mu[g]);
      l[g] *= alpha;
#pragma unroll
      for (int e = 0; e < EPL; ++e) o[g][e] *= alpha;
      m[g] = mn;
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      float vf[EPL];
      unpack<T>(vr[u], vf);
#pragma unroll
      for (int g = 0; g < G; ++g) {
        const float pu = fast_exp2(s[u][g] - mu[g]);
        l[g] += pu;
#pragma unroll
        for (int e = 0; e < EPL; ++e) o[g][e] = fmaf(pu, vf[e], o[g][e]);
      }
    }
  }

  // Merges the wave's streams (lane groups LPK apart) with a butterfly of
  // lane swaps (lane_pair: the Whisper steps 1-1.5% shorter than with
  // ds_bpermute shuffles, outputs bit-identical); afterwards the first group
  // (lanes 0 .. LPK - 1, the ones the workgroup merge reads) holds the
  // wave's state.
  template <int OFF>
  __device__ __forceinline__ void merge_from() {
    if constexpr (OFF < 64) {
#pragma unroll
      for (int g = 0; g < G; ++g) {
        float m1, m2, l1, l2;
        lane_pair<OFF>(m[g], m1, m2);
        lane_pair<OFF>(l[g], l1, l2);
        const float mn = fmaxf(m1, m2);
        const float mu = mn == kNegInf ? 0.f : mn;
        const float w1 = fast_exp2(m1 - mu);
        const float w2 = fast_exp2(m2 - mu);
        l[g] = l1 * w1 + l2 * w2;
#pragma unroll
        for (int e = 0; e < EPL; ++e) {
          float o1, o2;
          lane_pair<OFF>(o[g][e], o1, o2);
          o[g][e] = o1 * w1 + o2 * w2;
        }
        m[g] = mn;
      }
      merge_from<OFF * 2>();
    }
  }
  __device__ __forceinline__ void merge_wave() { merge_from<S::kLPK>(); }
};

// At most 128 VGPRs, so that four waves fit per SIMD (two 8-wave workgroups
// per CU).
//
// APPEND: the step's key and value join those of the cache, keys 0 ..
// positions[b] - 1 (the last split folds them into its state); the first
// split writes them to the cache at positions[b].  No workgroup reads that
// slot, so splits need no ordering among themselves.
//
// PRO: the prologue of asrattn_decode_append.  The G query rows, the step's
// key and its value are normalized and rotated once per workgroup, a lane
// group each, and shared through LDS (done by every lane group for all rows,
// the prologue's vector instructions took as long as the memory reads of a
// small batch).  Steps without norms and rotation (Whisper's) take the rows
// from memory, each lane its slices, without the barrier: 16 rows of 12 heads
// over 440 bf16 keys 7.01 -> 6.54 us, 13 of 20 over 223 6.07 -> 5.62, few
// float32 rows over 30 keys 3.8 -> 3.5; 0.95 of the time over 528 shapes, and 3%
// more at 260 to 320 pairs over 440 float32 keys.
//
// Splits: each stores its partial, waits until the stores have reached
// memory, and adds one to its pair's arrival word; the one that finds all
// others arrived folds the partials and clears the word.  The word lives in
// the caller's workspace, which holds anything before the launch: the splits
// tag it first (a launch's tag is its own), so no clearing pass is needed
// and a captured launch finds its word cleared or foreign on every replay.
//
// SPEC (plain launches with one split, no window, key counts in device
// memory and a cache of at least eight first batches; paged, a first page
// that holds the whole first batch; the launch chooses it): the first load
// batch, keys 0 .. STEP - 1, is issued before the row's key count is read,
// from buffer resources that end at the cache's capacity (paged: at the
// first page's end, the page read from the block table meanwhile); once the
// count is known, keys at or past it are masked and their values zeroed
// (cache slots past a row's keys may hold anything).
// The masked keys then add exactly zero, as the zeros of a resource ending
// at the count do, so the output is the same bit for bit; the launch is
// one round trip shorter at its start (Qwen3's step: 22.74 -> 22.37 us per
// launch, same box).  The fused step (its prologue's loads already cover
// that round trip) measured 2% slower with it and does not take it.
//
// PB (paged, one split, no window, pages of at least one load batch; SPEC
// on a paged cache implies it): batches start at multiples of STEP, and the
// page size is a power of two >= STEP, so each batch lies in one page: one
// block-table read and one pair of buffer resources per batch instead of
// one per slice (Qwen3's paged step 23.6 -> 22.9 us per launch, same box;
// the same loads in the same order, so the same bits).
template <typename T, int HD, int G, int W, bool APPEND, bool PAGED, bool SPEC = false, bool PB = false,
          bool PRO = APPEND>
__global__ __launch_bounds__(64 * W, (DecodeShape<T, HD, G, W>::kOcc)) void decode_kernel(const DecodeArgs a) {
  static_assert(!SPEC || !APPEND, "speculative first batch: plain launches");
  static_assert(!PB || PAGED, "page-sized batches: paged caches");
  static_assert(!PRO || APPEND, "the prologue belongs to appending launches");
  using S = DecodeShape<T, HD, G, W>;
  constexpr int EPL = S::kEPL, LPK = S::kLPK, NS = S::kStreams;
  // Keys per stream per load batch.
  constexpr int U = APPEND ? S::kUnroll : S::kPlainUnroll;
  constexpr int STEP = NS * U;
  constexpr bool kPageBatch = PAGED && (SPEC || PB);
  const asrattn_decode_params& p = a.p;

  const int split = blockIdx.x;
  const int hkv = blockIdx.y;
  const int b = blockIdx.z;
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int uwave = __builtin_amdgcn_readfirstlane(wave);
  const int sub = lane % LPK;
  const int stream = wave * S::kKPW + lane / LPK;
  const bool split_keys = !SPEC && !PB && a.splits > 1;  // both take one split
  unsigned long long* const arrive = a.ws_arrive + ((int64_t)b * p.heads_kv + hkv);
  unsigned long long arrive_old = 0;
  if (split_keys && threadIdx.x == 0)
    arrive_old = __hip_atomic_load(arrive, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);

  // K and V of this (sequence, kv head).
  const int64_t kbatch = PAGED ? 0 : (int64_t)b * p.k_batch_stride;
  const int64_t vbatch = PAGED ? 0 : (int64_t)b * p.v_batch_stride;
  const char* kbase =
      reinterpret_cast<const char*>(static_cast<const T*>(p.k) + kbatch + (int64_t)hkv * p.k_head_stride);
  const char* vbase =
      reinterpret_cast<const char*>(static_cast<const T*>(p.v) + vbatch + (int64_t)hkv * p.v_head_stride);
  const uint32_t kts = (uint32_t)(p.k_token_stride * (int64_t)sizeof(T));
  const uint32_t vts = (uint32_t)(p.v_token_stride * (int64_t)sizeof(T));
  const uint32_t lane_bytes = sub * EPL * (uint32_t)sizeof(T);

  // q is used raw (no unpacking), so its load latency overlaps the first
  // K/V batch's; it and the prologue's inputs load before the key count is
  // read, which none of them needs (Qwen3's step 21.4 -> 20.9 us per launch,
  // the fused step 23.1 -> 22.6).  SPEC issues the first K/V batch there
  // too; without the scheduling barrier below, the compiler moves the
  // count's load and its wait above those loads.
  Stream<T, HD, G, W> st;
  if constexpr (!PRO) {
    const T* qp = static_cast<const T*>(p.q) + (int64_t)b * p.q_batch_stride +
                  (int64_t)hkv * G * p.q_head_stride + sub * EPL;
#pragma unroll
    for (int g = 0; g < G; ++g) st.q[g] = *reinterpret_cast<const uint4*>(qp + (int64_t)g * p.q_head_stride);
  }
  st.c = a.c;
  st.init();
  // The prologue's inputs load here, before the first K/V batch; its
  // arithmetic runs after that batch is issued.  Row r of the prologue: query
  // head r (r < G), the new key (G), the new value (G + 1); lane group
  // `stream` takes rows stream, stream + NS, ... (past the last: the last).
  const asrattn_append_params& ap = a.ap;
  const bool has_norm = PRO && ap.q_norm != nullptr;
  const bool has_vnorm = PRO && ap.v_norm != 0;
  const bool has_rot = PRO && ap.cos != nullptr;
  constexpr int PR = G + 2;
  constexpr int kRounds = PRO ? (PR + NS - 1) / NS : 1;
  __shared__ uint4 sm_rows[PRO ? PR : 1][PRO ? LPK : 1];
  uint4 praw[kRounds], pw[kRounds], pcs = {}, psn = {}, knew = {}, vnew = {};
  if constexpr (APPEND) {
    const T* knp = static_cast<const T*>(ap.k_new) + (int64_t)b * ap.kn_batch_stride + (int64_t)hkv * ap.kn_head_stride;
    const T* vnp = static_cast<const T*>(ap.v_new) + (int64_t)b * ap.vn_batch_stride + (int64_t)hkv * ap.vn_head_stride;
    if constexpr (!PRO) {
      knew = *reinterpret_cast<const uint4*>(knp + sub * EPL);
      vnew = *reinterpret_cast<const uint4*>(vnp + sub * EPL);
    } else {
      const T* qp = static_cast<const T*>(p.q) + (int64_t)b * p.q_batch_stride + (int64_t)hkv * G * p.q_head_stride;
      // Absent weights or tables read k_new's slice instead (and are unused):
      // the loads stay unconditional, so no branch joins their registers and
      // forces a wait before the first K/V batch.
      const T* csp = has_rot ? static_cast<const T*>(ap.cos) + (int64_t)b * ap.rope_batch_stride : knp;
      const T* snp = has_rot ? static_cast<const T*>(ap.sin) + (int64_t)b * ap.rope_batch_stride : knp;
#pragma unroll
      for (int i = 0; i < kRounds; ++i) {
        const int r = min(stream + i * NS, PR - 1);
        const T* rp = r < G ? qp + (int64_t)r * p.q_head_stride : r == G ? knp : vnp;
        const T* wp = !has_norm || r > G ? knp : static_cast<const T*>(r < G ? ap.q_norm : ap.k_norm);
        praw[i] = *reinterpret_cast<const uint4*>(rp + sub * EPL);
        pw[i] = *reinterpret_cast<const uint4*>(wp + sub * EPL);
      }
      pcs = *reinterpret_cast<const uint4*>(csp + sub * EPL);
      psn = *reinterpret_cast<const uint4*>(snp + sub * EPL);
    }
  }

  // Two register batches in ping-pong: the next batch is in flight while the
  // current one is consumed.
  uint4 ka[U], va[U], kb[U], vb[U];
  // Paged: pool page of logical page pi of this sequence, or -1 when the
  // entry is missing or outside the pool (its keys are skipped).
  const int32_t* bt = PAGED ? a.pk.block_table + (int64_t)b * a.pk.bt_stride : nullptr;
  auto pool_page = [&](int pi) -> int {
    if (pi >= a.pk.bt_stride) return -1;
    const int e = load_uniform(bt + __builtin_amdgcn_readfirstlane(pi));
    return e >= 0 && e < a.pk.num_pages ? e : -1;
  };

  int page0 = 0;  // SPEC, paged: the sequence's first pool page (-1: none)
  if constexpr (SPEC) {
    // Slab: resources up to the cache's capacity.  Paged: over the first
    // page (the launch makes sure the batch fits in one).
    const char* kp = kbase;
    const char* vp = vbase;
    uint32_t keys = (uint32_t)p.max_len_k;
    if constexpr (PAGED) {
      page0 = pool_page(0);
      const int64_t pg = page0 >= 0 ? page0 : 0;
      kp = kbase + pg * a.pk.k_page_stride * (int64_t)sizeof(T);
      vp = vbase + pg * a.pk.v_page_stride * (int64_t)sizeof(T);
      keys = page0 >= 0 ? (uint32_t)a.pk.page_size : 0u;
    }
    const __amdgpu_buffer_rsrc_t kcap = buffer_rsrc(kp, keys * kts);
    const __amdgpu_buffer_rsrc_t vcap = buffer_rsrc(vp, keys * vts);
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const uint32_t j = (uint32_t)(u * NS + stream);
      ka[u] = buffer_load16_stream(kcap, j * kts + lane_bytes);
      va[u] = buffer_load16_stream(vcap, j * vts + lane_bytes);
    }
    __builtin_amdgcn_sched_barrier(0);  // the batch's issue stays above the count's load
  }

  const int64_t pos = APPEND ? load_uniform(p.positions + b) : 0;
  const int n = APPEND ? (int)min(max(pos, (int64_t)0), (int64_t)p.max_len_k)
                       : decode_key_count(p.seqused_k, p.positions, b, p.max_len_k);
  // Sliding window: the query sees its last `window` keys (with the append
  // variant the new key is one of them): cache keys kfirst .. n - 1.
  const int kfirst = p.window > 0 ? max(0, n + (APPEND ? 1 : 0) - p.window) : 0;
  // Paged: splits start NS-aligned (slices stay inside pages); keys before
  // kfirst are masked.
  const int kbeg = PAGED ? kfirst / NS * NS : kfirst;
  int chunk = (n - kbeg + a.splits - 1) / a.splits;
  if constexpr (PAGED) chunk = (chunk + NS - 1) / NS * NS;
  const int k0 = min(n, kbeg + split * chunk);
  const int k1 = min(n, k0 + chunk);

  // Buffer resources that end at the split's last key: loads past it return
  // zeros without a branch, so the two load batches stay in flight across
  // the loop.  (Paged: the pool, past the sequence's first page.)
  const __amdgpu_buffer_rsrc_t krs = buffer_rsrc(kbase, (uint32_t)k1 * kts);
  const __amdgpu_buffer_rsrc_t vrs = buffer_rsrc(vbase, (uint32_t)k1 * vts);

  // Key u of the batch starting at `base` is base + u * NS + stream.
  auto load = [&](uint4* kr, uint4* vr, int base) -> unsigned {
    unsigned mask = 0;
    // kPageBatch: the batch's page, its first key and its resources.
    int bfirst = 0, bpage = -1;
    __amdgpu_buffer_rsrc_t kb_rs = krs, vb_rs = vrs;
    if constexpr (kPageBatch) {
      const int pi = base >> a.page_shift;
      bfirst = pi << a.page_shift;
      bpage = pool_page(pi);
      const uint32_t keys = bpage >= 0 ? (uint32_t)min(max(k1 - bfirst, 0), a.pk.page_size) : 0u;
      const int64_t pg = bpage >= 0 ? bpage : 0;
      kb_rs = buffer_rsrc(kbase + pg * a.pk.k_page_stride * (int64_t)sizeof(T), keys * kts);
      vb_rs = buffer_rsrc(vbase + pg * a.pk.v_page_stride * (int64_t)sizeof(T), keys * vts);
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int j = base + u * NS + stream;
      if constexpr (kPageBatch) {
        kr[u] = buffer_load16_stream(kb_rs, (uint32_t)(j - bfirst) * kts + lane_bytes);
        vr[u] = buffer_load16_stream(vb_rs, (uint32_t)(j - bfirst) * vts + lane_bytes);
        mask |= (j < k1 && j >= kfirst && bpage >= 0 ? 1u : 0u) << u;
      } else if constexpr (PAGED) {
        const int j0 = base + u * NS;  // uniform; the slice lies in one page
        const int pi = j0 >> a.page_shift;
        const int first = pi << a.page_shift;
        const int page = pool_page(pi);
        const uint32_t keys = page >= 0 ? (uint32_t)min(max(k1 - first, 0), a.pk.page_size) : 0u;
        const int64_t pg = page >= 0 ? page : 0;
        const __amdgpu_buffer_rsrc_t kp = buffer_rsrc(kbase + pg * a.pk.k_page_stride * (int64_t)sizeof(T), keys * kts);
        const __amdgpu_buffer_rsrc_t vp = buffer_rsrc(vbase + pg * a.pk.v_page_stride * (int64_t)sizeof(T), keys * vts);
        kr[u] = buffer_load16_stream(kp, (uint32_t)(j - first) * kts + lane_bytes);
        vr[u] = buffer_load16_stream(vp, (uint32_t)(j - first) * vts + lane_bytes);
        mask |= (j < k1 && j >= kfirst && page >= 0 ? 1u : 0u) << u;
      } else {
        kr[u] = buffer_load16_stream(krs, (uint32_t)j * kts + lane_bytes);
        vr[u] = buffer_load16_stream(vrs, (uint32_t)j * vts + lane_bytes);
        mask |= (j < k1 ? 1u : 0u) << u;
      }
    }
    return mask;
  };

  // The first batch is issued unconditionally: with k0 >= k1 its offsets all
  // lie past the resource's end and read zeros.  SPEC's was issued above
  // (k0 = 0 with one split and no window); it is masked here.
  unsigned mb = 0;
  unsigned ma = 0;
  if constexpr (SPEC) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const bool valid = u * NS + stream < k1 && page0 >= 0;
      ma |= (valid ? 1u : 0u) << u;
      if (!valid) va[u] = make_uint4(0u, 0u, 0u, 0u);
    }
  } else {
    ma = load(ka, va, k0);
  }
  // Tag the pair's arrival word, whose load was issued first of all; the
  // answer is not waited for.
  if (split_keys && threadIdx.x == 0 && (arrive_old >> 16) != a.tag)
    __hip_atomic_compare_exchange_strong(arrive, &arrive_old, a.tag << 16, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                         __HIP_MEMORY_SCOPE_AGENT);
  if constexpr (PRO) {
    __builtin_amdgcn_sched_barrier(0);  // keep the prologue below the batch's issue
#pragma unroll
    for (int i = 0; i < kRounds; ++i) {
      if (uwave * S::kKPW + i * NS < PR) {  // uniform per wave
        const int r = min(stream + i * NS, PR - 1);
        sm_rows[r][sub] = prologue_row<T, HD, LPK>(praw[i], has_norm || has_vnorm, r <= G ? has_norm : has_vnorm,
                                                   r <= G, pw[i], has_rot, r <= G, pcs, psn, ap.eps, sub);
      }
    }
    // An LDS-only barrier: the K/V batch stays in flight across it.
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
#pragma unroll
    for (int g = 0; g < G; ++g) st.q[g] = sm_rows[g][sub];
    if (uwave == 0) st.seed(sm_rows[G][sub], sm_rows[G + 1][sub], split == a.splits - 1 && stream == 0);
  } else if constexpr (APPEND) {
    if (uwave == 0) st.seed(knew, vnew, split == a.splits - 1 && stream == 0);
  }
  for (int base = k0; base < k1; base += 2 * STEP) {
    mb = load(kb, vb, base + STEP);
    st.template consume<U>(ka, va, ma);
    if (base + STEP >= k1) break;
    ma = load(ka, va, base + 2 * STEP);
    st.template consume<U>(kb, vb, mb);
  }

  if constexpr (APPEND) {
    if (split == 0 && stream == 0 && pos >= 0 && pos < p.max_len_k) {
      int64_t koff = pos * kts, voff = pos * vts;
      bool write = true;
      if constexpr (PAGED) {
        const int pi = (int)(pos >> a.page_shift);
        const int page = pool_page(pi);
        const int64_t slot = pos - ((int64_t)pi << a.page_shift);
        write = page >= 0;
        koff = (int64_t)page * a.pk.k_page_stride * (int64_t)sizeof(T) + slot * kts;
        voff = (int64_t)page * a.pk.v_page_stride * (int64_t)sizeof(T) + slot * vts;
      }
      if (write) {
        *reinterpret_cast<uint4*>(const_cast<char*>(kbase) + koff + lane_bytes) = PRO ? sm_rows[G][sub] : knew;
        *reinterpret_cast<uint4*>(const_cast<char*>(vbase) + voff + lane_bytes) = PRO ? sm_rows[G + 1][sub] : vnew;
      }
    }
  }

  st.merge_wave();

  // Merge the waves in LDS.
  __shared__ float sm_m[W][G];
  __shared__ float sm_l[W][G];
  __shared__ float sm_o[W][G][HD];
  if (lane < LPK) {
#pragma unroll
    for (int g = 0; g < G; ++g) {
      if (lane == 0) {
        sm_m[wave][g] = st.m[g];
        sm_l[wave][g] = st.l[g];
      }
#pragma unroll
      for (int e = 0; e < EPL; ++e) sm_o[wave][g][sub * EPL + e] = st.o[g][e];
    }
  }
  __syncthreads();

  for (int t = threadIdx.x; t < G * HD; t += S::kThreads) {
    const int g = t / HD;
    const int d = t % HD;
    float mx = kNegInf;
#pragma unroll
    for (int w = 0; w < W; ++w) mx = fmaxf(mx, sm_m[w][g]);
    const float mxu = mx == kNegInf ? 0.f : mx;
    float lsum = 0.f, osum = 0.f;
#pragma unroll
    for (int w = 0; w < W; ++w) {
      const float wt = fast_exp2(sm_m[w][g] - mxu);
      lsum = fmaf(sm_l[w][g], wt, lsum);
      osum = fmaf(sm_o[w][g][d], wt, osum);
    }
    const int hq = hkv * G + g;
    if (!split_keys) {
      T* op = static_cast<T*>(p.out) + (int64_t)b * p.o_batch_stride + (int64_t)hq * p.o_head_stride + d;
      Elem<T>::store1(op, lsum > 0.f ? osum / lsum : 0.f);
    } else {
      const int64_t idx = ((int64_t)b * p.heads_q + hq) * a.splits + split;
      store_shared(a.ws_o + idx * HD + d, osum);
      if (d == 0) {
        store_shared(a.ws_ml + idx * 2, mx);
        store_shared(a.ws_ml + idx * 2 + 1, lsum);
      }
    }
  }
  if (!split_keys) return;

  // Arrive once every wave's partial stores are in memory.
  __builtin_amdgcn_s_waitcnt(kWaitVmem);
  __shared__ int sm_last;
  __syncthreads();
  if (threadIdx.x == 0) {
    const unsigned long long before =
        __hip_atomic_fetch_add(arrive, 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    sm_last = (int)(before & 0xffffull) == a.splits - 1;
    if (sm_last) __hip_atomic_store(arrive, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  __syncthreads();
  if (!sm_last) return;  // uniform over the workgroup

  // Fold the splits' partials into the output.  Bound by round trips to memory
  // (about a microsecond each): a head group of four outputs a thread and more
  // takes pairs of neighbours, up to eight of them a round (eight heads of 512 in
  // 16 splits: 36.5 -> 24.3 us a launch against one output a round; below that
  // line pairs took 0.2 us more).
  constexpr int kVec = G * HD >= 4 * S::kThreads ? 2 : 1;
  constexpr int kItems = G * HD / kVec;
  constexpr int kRound = kVec == 1 ? 1 : kItems >= 8 * S::kThreads ? 8 : kItems >= 4 * S::kThreads ? 4 : 2;
  constexpr int kBatch = kRound == 8 ? 4 : 8;  // splits whose partials are loaded in one round trip
  const int64_t row0 = ((int64_t)b * p.heads_q + hkv * G) * a.splits;
  for (int t0 = threadIdx.x; t0 < kItems; t0 += kRound * S::kThreads) {
    float mx[kRound], lsum[kRound], osum[kRound][kVec];
#pragma unroll
    for (int i = 0; i < kRound; ++i) {
      mx[i] = kNegInf;
      lsum[i] = 0.f;
#pragma unroll
      for (int e = 0; e < kVec; ++e) osum[i][e] = 0.f;
    }
    for (int s0 = 0; s0 < a.splits; s0 += kBatch) {
      float m[kRound][kBatch], l[kRound][kBatch], o[kRound][kBatch][kVec];
#pragma unroll
      for (int i = 0; i < kRound; ++i) {
        const int t = t0 + i * S::kThreads;  // below kItems, a multiple of kRound * kThreads if kRound > 1
        const int64_t idx0 = row0 + (int64_t)(t * kVec / HD) * a.splits;
#pragma unroll
        for (int s = 0; s < kBatch; ++s) {
          const int u = min(s0 + s, a.splits - 1);  // surplus slots repeat the last split
          if constexpr (kVec == 2) {
            load_shared2(a.ws_ml + (idx0 + u) * 2, m[i][s], l[i][s]);
            load_shared2(a.ws_o + (idx0 + u) * HD + t * kVec % HD, o[i][s][0], o[i][s][1]);
          } else {
            m[i][s] = load_shared(a.ws_ml + (idx0 + u) * 2);
            l[i][s] = load_shared(a.ws_ml + (idx0 + u) * 2 + 1);
            o[i][s][0] = load_shared(a.ws_o + (idx0 + u) * HD + t % HD);
          }
        }
      }
#pragma unroll
      for (int i = 0; i < kRound; ++i) {
        float mn = mx[i];
#pragma unroll
        for (int s = 0; s < kBatch; ++s) mn = fmaxf(mn, m[i][s]);
        const float mu = mn == kNegInf ? 0.f : mn;
        const float w0 = fast_exp2(mx[i] - mu);
        mx[i] = mn;
        lsum[i] *= w0;
#pragma unroll
        for (int e = 0; e < kVec; ++e) osum[i][e] *= w0;
#pragma unroll
        for (int s = 0; s < kBatch; ++s) {
          const float w = fast_exp2(m[i][s] - mu);
          const bool in = s0 + s < a.splits;  // a surplus slot's weight of 0 would turn an infinite partial into NaN
          lsum[i] = in ? fmaf(l[i][s], w, lsum[i]) : lsum[i];
#pragma unroll
          for (int e = 0; e < kVec; ++e) osum[i][e] = in ? fmaf(o[i][s][e], w, osum[i][e]) : osum[i][e];
        }
      }
    }
#pragma unroll
    for (int i = 0; i < kRound; ++i) {
      const int t = t0 + i * S::kThreads;
      T* op = static_cast<T*>(p.out) + (int64_t)b * p.o_batch_stride + (int64_t)(hkv * G + t * kVec / HD) * p.o_head_stride +
              t * kVec % HD;
#pragma unroll
      for (int e = 0; e < kVec; ++e) Elem<T>::store1(op + e, lsum[i] > 0.f ? osum[i][e] / lsum[i] : 0.f);
    }
  }
}

template <typename T, int HD, int G, int W>
hipError_t launch_typed(const DecodeArgs& a, bool append, hipStream_t stream) {
  const asrattn_decode_params& p = a.p;
  dim3 grid(a.splits, p.heads_kv, p.batch);
  const bool paged = a.pk.block_table != nullptr;
  // Key counts read from device memory, one split, no window, and a cache
  // of at least eight first batches: the first batch need not wait for the
  // count (SPEC).  Its resource ends at the capacity, not at the count, so a
  // batch as wide as the cache reads keys the row does not have: Whisper's
  // self-attention over a 256-key bucket, one 256-key batch, read 2.3x its
  // bytes and ran 3% slower with it.
  constexpr int kFirstBatch = DecodeShape<T, HD, G, W>::kPlainStep;
  const bool spec = !append && a.splits == 1 && p.window <= 0 &&
                    (p.seqused_k != nullptr || p.positions != nullptr) && p.max_len_k >= 8 * kFirstBatch &&
                    (!paged || a.pk.page_size >= kFirstBatch);
  // Paged appending steps whose batches each lie in one page (PB; the plain
  // steps get it with SPEC).
  const bool page_batch = paged && a.splits == 1 && p.window <= 0 &&
                          a.pk.page_size >= DecodeShape<T, HD, G, W>::kStep;
  const bool prologue = a.ap.q_norm != nullptr || a.ap.cos != nullptr || a.ap.v_norm != 0;
  if (append && paged && page_batch)
    hipLaunchKernelGGL((decode_kernel<T, HD, G, W, true, true, false, true>), grid, dim3(64 * W), 0, stream, a);
  else if (append && !paged && !prologue)
    hipLaunchKernelGGL((decode_kernel<T, HD, G, W, true, false, false, false, false>), grid, dim3(64 * W), 0, stream, a);
  else if (append && paged)
    hipLaunchKernelGGL((decode_kernel<T, HD, G, W, true, true>), grid, dim3(64 * W), 0, stream, a);
  else if (append)
    hipLaunchKernelGGL((decode_kernel<T, HD, G, W, true, false>), grid, dim3(64 * W), 0, stream, a);
  else if (paged && spec)
    hipLaunchKernelGGL((decode_kernel<T, HD, G, W, false, true, true>), grid, dim3(64 * W), 0, stream, a);
  else if (paged)
    hipLaunchKernelGGL((decode_kernel<T, HD, G, W, false, true>), grid, dim3(64 * W), 0, stream, a);
  else if (spec)
    hipLaunchKernelGGL((decode_kernel<T, HD, G, W, false, false, true>), grid, dim3(64 * W), 0, stream, a);
  else
    hipLaunchKernelGGL((decode_kernel<T, HD, G, W, false, false>), grid, dim3(64 * W), 0, stream, a);
  return hipGetLastError();
}

// waves: 4 or 8, lowered to what the merge's LDS allows.
template <typename T, int HD, int G>
hipError_t launch_waves(const DecodeArgs& a, int waves, bool append, hipStream_t stream) {
  if constexpr (DecodeShape<T, HD, G, 8>::kFits) {
    if (waves >= 8) return launch_typed<T, HD, G, 8>(a, append, stream);
  }
  static_assert(DecodeShape<T, HD, G, 4>::kFits, "four waves fit");
  return launch_typed<T, HD, G, 4>(a, append, stream);
}

template <typename T, int HD>
hipError_t launch_hd(const DecodeArgs& a, int group, int waves, bool append, hipStream_t stream) {
  switch (group) {
    case 1: return launch_waves<T, HD, 1>(a, waves, append, stream);
    case 2: return launch_waves<T, HD, 2>(a, waves, append, stream);
    case 4: return launch_waves<T, HD, 4>(a, waves, append, stream);
    case 8: return launch_waves<T, HD, 8>(a, waves, append, stream);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace
}  // namespace asrattn
