// Decoder-step attention: kernel choice and launch (the kernels live in
// decode_kernels.hpp, instantiated per element type in decode_bf16.hip and
// decode_f32.hip).
#include <atomic>
#include <chrono>

#include "decode_args.hpp"
#include "kernels.hpp"

namespace asrattn {

namespace {

// A tag no other launch of this process has had for 2^48 launches, and that
// neither a count nor a partial left in a reused workspace resembles: a
// counter from a start set by the clock, its bits mixed by an odd multiplier
// (a permutation of the 48-bit values).
unsigned long long launch_tag() {
  static std::atomic<unsigned long long> next{
      (unsigned long long)std::chrono::steady_clock::now().time_since_epoch().count()};
  constexpr unsigned long long kMask = (1ull << 48) - 1;
  unsigned long long tag = 0;
  while (tag == 0) tag = (next.fetch_add(1, std::memory_order_relaxed) * 0x9e3779b97f4a7c15ull) & kMask;
  return tag;
}

}  // namespace

bool decode_supported(int dtype, int head_dim, int group) {
  const bool dt = dtype == ASRATTN_F32 || dtype == ASRATTN_BF16;
  // A key row is read by at most one wave: 64 lanes x 16 bytes.
  const bool hd = head_dim == 64 || head_dim == 128 || head_dim == 256 || (head_dim == 512 && dtype == ASRATTN_BF16);
  const bool g = group == 1 || group == 2 || group == 4 || group == 8;
  return dt && hd && g;
}

int decode_keys_per_wave(int dtype, int head_dim) {
  return 64 / (head_dim * (dtype == ASRATTN_BF16 ? 2 : 4) / 16);
}

int decode_span(const asrattn_decode_params& p) {
  return p.window > 0 && p.window < p.max_len_k ? p.window : p.max_len_k;
}

int decode_waves(const asrattn_decode_params& p, int splits, int page_size) {
  // About 2048 waves over the grid (two per SIMD): on one MI355X, Qwen3's
  // 512 workgroups ran 6% faster on 4 waves than on 8.  Sixteen waves were
  // never faster than eight (each wave repeats the merge's vector work: split
  // launches of 6 to 64 pairs took 6.6-10.2 us with sixteen, 5.6-9.0 with
  // eight).
  const long long groups = (long long)p.batch * p.heads_kv * splits;
  const int keys_per_split = (decode_span(p) + splits - 1) / splits;
  int waves = groups * 8 > 2048 ? 4 : 8;
  // A wave loads 64 / LPK rows per instruction (8 for bf16 x 64, 4 for 128),
  // and a batch takes 4 of them (2 with four or more query heads per kv
  // head, or head_dim 256 and up: DecodeShape::kUnroll).  Four waves where
  // eight would load more than an unsplit row's keys at once, or where a
  // split's keys are two batches of four waves (Qwen3's 480 of 1024 slots in
  // eight splits: 6.4 us on four, 7.4 on eight; 900 slots: the same).
  const int rows_per_wave = 64 / (p.head_dim * (p.dtype == ASRATTN_BF16 ? 2 : 4) / 16);
  const int group = p.heads_q / p.heads_kv;
  const int batch = rows_per_wave * (group >= 4 || p.head_dim >= 256 ? 2 : 4);
  if (splits > 1 ? 8 * batch >= keys_per_split : 8 * batch > keys_per_split) waves = 4;
  // Paged: a slice (one key per stream of the workgroup) within one page.
  if (page_size > 0 && waves * rows_per_wave > page_size) waves = 4;
  return waves;
}

hipError_t launch_decode(const asrattn_decode_params& p, const asrattn_append_params* append,
                         const asrattn_paged_kv* paged, int splits, float* ws_o, float* ws_ml,
                         unsigned long long* ws_arrive, hipStream_t stream) {
  DecodeArgs a;
  a.p = p;
  a.ap = append != nullptr ? *append : asrattn_append_params{};
  a.pk = paged != nullptr ? *paged : asrattn_paged_kv{};
  a.page_shift = 0;
  while (paged != nullptr && (1 << a.page_shift) < paged->page_size) ++a.page_shift;
  const bool app = append != nullptr;
  a.ws_o = ws_o;
  a.ws_ml = ws_ml;
  a.ws_arrive = ws_arrive;
  a.tag = splits > 1 ? launch_tag() : 0;
  a.splits = splits;
  a.c = p.scale * kLog2e;
  const int group = p.heads_q / p.heads_kv;
  const int waves = decode_waves(p, splits, paged != nullptr ? paged->page_size : 0);
  return p.dtype == ASRATTN_BF16 ? launch_decode_bf16(a, p.head_dim, group, waves, app, stream)
                                 : launch_decode_f32(a, p.head_dim, group, waves, app, stream);
}

}  // namespace asrattn
