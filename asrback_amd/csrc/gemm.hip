// The projections around a module's attention over rows of bf16
// (asrlayer_gemm): x w^T, plus a bias or added to what the output holds.
//
// Two tilings, both on v_mfma_f32_32x32x16_bf16 with the weight rows as the
// first operand, so that a lane's accumulators are consecutive outputs of one
// row:
//
//   * Few rows: a workgroup takes 32 rows x 32 outputs, its four waves a
//     quarter of the reduction each, operands straight from memory into
//     registers, eight steps in flight.  A launch is one or two round trips to
//     memory, which is what bounds it (sixteen in flight in two register sets:
//     300 rows of 512 to 1536 outputs 7.2 -> 10.3 us).
//   * Many rows: 128 rows x 128 or 192 outputs, four waves of 64 rows x half the
//     outputs, 64-deep tiles of both operands moved into a two-stage LDS ring by
//     DMA (the attention's ring: chunks rotated within rows, so operand reads
//     are free of bank conflicts), 64 or 80 KB, two workgroups per CU.  Bound by
//     the matrix cores, their operand reads and the last round of workgroups.
//
// Rows at or past used[b] of batch entry b are neither read nor written:
// SenseVoice's padded frames (40% of the rows of a batch of 104-504 frames),
// whose queries, keys and values nothing reads.  32 x 504 frames of 512, 304 of
// them real on average, to 1536 outputs: 33.5 us, against 44 for the library's
// product of all rows (of all rows here: 40); to 512: 14.9 against 16.8.
#include "kernels.hpp"
#include "layers.hpp"
#include "ring_common.hpp"
#include "row_ops.hpp"

namespace asrattn {
namespace {

using namespace ring;

struct RowView {
  const bf16_raw* x;
  bf16_raw* out;
  int rows;  // rows computed
};

__device__ __forceinline__ RowView row_view(const asrlayer_gemm_params& p, int b) {
  RowView v;
  v.x = static_cast<const bf16_raw*>(p.x) + (int64_t)b * p.x_batch_stride;
  v.out = static_cast<bf16_raw*>(p.out) + (int64_t)b * p.out_batch_stride;
  v.rows = p.used != nullptr ? min(max(p.used[b], 0), p.rows) : p.rows;
  return v;
}

// Adds the bias or the held output to 4 * N sums of row `out`, columns from n0
// on, and stores them.
template <int N>
__device__ __forceinline__ void finish(const asrlayer_gemm_params& p, float* y, bf16_raw* out, int n0) {
  uint2 held[N] = {};
  const bf16_raw* add = p.accumulate ? out + n0 : p.bias != nullptr ? static_cast<const bf16_raw*>(p.bias) + n0 : nullptr;
  if (add != nullptr) {
#pragma unroll
    for (int i = 0; i < N; ++i) held[i] = *reinterpret_cast<const uint2*>(add + 4 * i);
  }
  uint2 r[N];
#pragma unroll
  for (int i = 0; i < N; ++i) {
    const uint2 h = held[i];
    r[i].x = pack_bf16x2(y[4 * i] + bf16_lo(h.x), y[4 * i + 1] + bf16_hi(h.x));
    r[i].y = pack_bf16x2(y[4 * i + 2] + bf16_lo(h.y), y[4 * i + 3] + bf16_hi(h.y));
  }
  if constexpr (N == 2)
    *reinterpret_cast<uint4*>(out + n0) = make_uint4(r[0].x, r[0].y, r[1].x, r[1].y);
  else
    *reinterpret_cast<uint2*>(out + n0) = r[0];
}

// 32 rows x 32 outputs.
__global__ __launch_bounds__(256) void gemm_small_kernel(const asrlayer_gemm_params p, int row_tiles, int col_tiles) {
  const int item = xcd_remap((int)blockIdx.x, (int)gridDim.x);
  const int n0 = item % col_tiles * 32;
  const int row0 = item / col_tiles % row_tiles * 32;
  const RowView v = row_view(p, item / col_tiles / row_tiles);
  if (row0 >= v.rows) return;  // uniform over the workgroup

  const int lane = threadIdx.x & 63, r32 = lane & 31, half = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int quarter = p.k / 4;
  const bf16_raw* xp = v.x + (int64_t)min(row0 + r32, v.rows - 1) * p.x_row_stride + wave * quarter + half * 8;
  const bf16_raw* wp = static_cast<const bf16_raw*>(p.w) + (int64_t)min(n0 + r32, p.n - 1) * p.k + wave * quarter + half * 8;
  const int steps = quarter / 16;
  constexpr int kAhead = 8;
  f32x16_t acc = f32x16_t{};
  for (int s0 = 0; s0 < steps; s0 += kAhead) {
    bf16x8_t a[kAhead], b[kAhead];
#pragma unroll
    for (int i = 0; i < kAhead; ++i) {
      const int s = min(s0 + i, steps - 1);  // past the last: repeated, unused
      a[i] = __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const uint4*>(wp + s * 16));
      b[i] = __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const uint4*>(xp + s * 16));
    }
#pragma unroll
    for (int i = 0; i < kAhead; ++i)
      if (s0 + i < steps) acc = mfma32(a[i], b[i], acc);
  }
  // Sum the quarters: accumulator r of a lane is output 8 (r / 4) + 4 half +
  // r % 4 of row r32.
  __shared__ float sm[4][32][36];
#pragma unroll
  for (int i = 0; i < 4; ++i)
    *reinterpret_cast<float4*>(&sm[wave][r32][8 * i + 4 * half]) =
        make_float4(acc[4 * i], acc[4 * i + 1], acc[4 * i + 2], acc[4 * i + 3]);
  __syncthreads();
  const int m = threadIdx.x / 8, c = threadIdx.x % 8 * 4;
  float y[4] = {};
#pragma unroll
  for (int w = 0; w < 4; ++w) {
    const float4 part = *reinterpret_cast<const float4*>(&sm[w][m][c]);
    y[0] += part.x;
    y[1] += part.y;
    y[2] += part.z;
    y[3] += part.w;
  }
  if (row0 + m < v.rows && n0 + c < p.n) finish<1>(p, y, v.out + (int64_t)(row0 + m) * p.out_row_stride, n0 + c);
}

// 128 rows x 64 NB outputs.
constexpr int kBM = 128, kBK = 64;

template <int NB>
__global__ __launch_bounds__(256, 2) void gemm_large_kernel(const asrlayer_gemm_params p, int row_tiles, int col_tiles) {
  constexpr int kBN = 64 * NB;
  constexpr int kTileBytes = kBM * kBK * 2;  // the X tile
  constexpr int kStageBytes = kTileBytes + kBN * kBK * 2;
  constexpr int kOutRow = 32 * NB + 4;  // staged floats per row of a wave's 32 rows
  __shared__ __attribute__((aligned(16))) unsigned char lds[2 * kStageBytes];
  static_assert(4 * 32 * kOutRow * 4 <= 2 * kStageBytes, "the staged outputs fit the ring");
  const int item = xcd_remap((int)blockIdx.x, (int)gridDim.x);
  const int n0 = item % col_tiles * kBN;
  const int row0 = item / col_tiles % row_tiles * kBM;
  const RowView v = row_view(p, item / col_tiles / row_tiles);
  if (row0 >= v.rows) return;  // uniform over the workgroup

  const int lane = threadIdx.x & 63, r32 = lane & 31, half = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int wm = wave & 1, wn = wave >> 1;
  const uint32_t lds_base = (uint32_t)(uintptr_t)lds;

  // Resources that end at the last computed row and the last output: tile rows
  // past them are zeros.
  const uint32_t xs = (uint32_t)p.x_row_stride * 2, ws = (uint32_t)p.k * 2;
  const __amdgpu_buffer_rsrc_t xrs =
      buffer_rsrc(v.x + (int64_t)row0 * p.x_row_stride, (uint32_t)(min(kBM, v.rows - row0) - 1) * xs + ws);
  const __amdgpu_buffer_rsrc_t wrs =
      buffer_rsrc(static_cast<const bf16_raw*>(p.w) + (int64_t)n0 * p.k, (uint32_t)min(kBN, p.n - n0) * ws);
  // A DMA instruction fills eight rows of eight chunks, the chunk order rotated
  // as the operand reads expect; wave w takes instructions 4 w .. of the X tile
  // and 2 NB w .. of the weights'.
  uint32_t xoff[4], woff[2 * NB];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int r = 8 * (4 * wave + i) + lane / 8;
    xoff[i] = (uint32_t)r * xs + (uint32_t)k_logical<64>(r, lane % 8) * 16;
  }
#pragma unroll
  for (int i = 0; i < 2 * NB; ++i) {
    const int r = 8 * (2 * NB * wave + i) + lane / 8;
    woff[i] = (uint32_t)r * ws + (uint32_t)k_logical<64>(r, lane % 8) * 16;
  }
  auto issue = [&](int t, int stage) {
    const uint32_t base = lds_base + (uint32_t)stage * kStageBytes;
#pragma unroll
    for (int i = 0; i < 4; ++i) dma16(xrs, base + (uint32_t)(4 * wave + i) * 1024, xoff[i] + (uint32_t)t * (kBK * 2));
#pragma unroll
    for (int i = 0; i < 2 * NB; ++i)
      dma16(wrs, base + kTileBytes + (uint32_t)(2 * NB * wave + i) * 1024, woff[i] + (uint32_t)t * (kBK * 2));
  };
  // Operand addresses in stage 0 (32-row blocks share the rotation).
  uint32_t xaddr[4], waddr[4];
#pragma unroll
  for (int kk = 0; kk < 4; ++kk) {
    const uint32_t c = (uint32_t)k_phys<64>(r32, 2 * kk + half) * 16;
    xaddr[kk] = (lds_base + (uint32_t)(64 * wm + r32) * (kBK * 2) + c) & 0x3ffffu;
    waddr[kk] = (lds_base + kTileBytes + (uint32_t)(32 * NB * wn + r32) * (kBK * 2) + c) & 0x3ffffu;
  }

  const bool idle = row0 + 64 * wm >= v.rows;  // none of this wave's rows: it moves tiles only
  f32x16_t acc[2][NB];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j) acc[i][j] = f32x16_t{};
  const int tiles = p.k / kBK;
  issue(0, 0);
  auto tile = [&](int t, int stage) {
    // Tile t has landed for every wave, and every wave is done with tile t - 1,
    // whose stage the next DMA takes.
    wait_vmcnt<0>();
    __syncthreads();
    if (t + 1 < tiles) issue(t + 1, stage ^ 1);
    if (idle) return;
    const uint32_t so = (uint32_t)stage * kStageBytes;
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) {
      bf16x8_t x[2], w[NB];
#pragma unroll
      for (int i = 0; i < 2; ++i) x[i] = lds_read16(xaddr[kk] + so + i * 32 * kBK * 2);
#pragma unroll
      for (int j = 0; j < NB; ++j) w[j] = lds_read16(waddr[kk] + so + j * 32 * kBK * 2);
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j) acc[i][j] = mfma32(w[j], x[i], acc[i][j]);
    }
  };
  for (int t = 0; t < tiles; t += 2) {
    tile(t, 0);
    if (t + 1 < tiles) tile(t + 1, 1);
  }
  __syncthreads();  // the ring is free for the outputs

  // 32 rows at a time, through LDS, for stores of 16 bytes a lane and 128 bytes
  // of a row and more.
  float* const stage = reinterpret_cast<float*>(lds) + wave * 32 * kOutRow;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
      for (int q = 0; q < 4; ++q)
        *reinterpret_cast<float4*>(stage + r32 * kOutRow + 32 * j + 8 * q + 4 * half) =
            make_float4(acc[i][j][4 * q], acc[i][j][4 * q + 1], acc[i][j][4 * q + 2], acc[i][j][4 * q + 3]);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
    for (int s = 0; s < 2 * NB; ++s) {
      const int ch = s * 64 + lane, m = ch / (4 * NB), c = ch % (4 * NB) * 8;
      const float4 lo = *reinterpret_cast<const float4*>(stage + m * kOutRow + c);
      const float4 hi = *reinterpret_cast<const float4*>(stage + m * kOutRow + c + 4);
      float y[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
      const int row = row0 + 64 * wm + 32 * i + m, n = n0 + 32 * NB * wn + c;
      if (row < v.rows && n < p.n) finish<2>(p, y, v.out + (int64_t)row * p.out_row_stride, n);
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  }
}

}  // namespace

hipError_t launch_gemm(const asrlayer_gemm_params& p, hipStream_t stream) {
  const auto tiles = [](long long count, int size) { return (count + size - 1) / size; };
  // Small tiles up to four workgroups per CU (300 rows of 512 to 1536 outputs,
  // 480 of them: 7.2 us against 9.2 in large tiles; 4 x 300 rows, 1920: 18.3
  // against 9.9).  Counted over all rows as one run, whatever part of them is
  // computed: the tilings sum in different orders, and a row's result does not
  // depend on how the batch is padded.
  const bool small = tiles((long long)p.batch * p.rows, 32) * tiles(p.n, 32) <= 1024;
  // 192 outputs a workgroup where they divide the outputs and leave at least a
  // round of workgroups (two per CU): five operand reads for six products
  // instead of four for four, and fewer rounds (16128 rows to 1536 outputs 45
  // -> 40 us).
  const bool wide = p.n % 192 == 0 && tiles((long long)p.batch * p.rows, kBM) * (p.n / 192) >= 512;
  const int row_tiles = (int)tiles(p.rows, small ? 32 : kBM);
  const int col_tiles = (int)tiles(p.n, small ? 32 : wide ? 192 : 128);
  const long long total = (long long)p.batch * row_tiles * col_tiles;
  if (total > 0x7fffffffLL) return hipErrorInvalidConfiguration;
  if (small)
    hipLaunchKernelGGL(gemm_small_kernel, dim3((unsigned)total), dim3(256), 0, stream, p, row_tiles, col_tiles);
  else if (wide)
    hipLaunchKernelGGL((gemm_large_kernel<3>), dim3((unsigned)total), dim3(256), 0, stream, p, row_tiles, col_tiles);
  else
    hipLaunchKernelGGL((gemm_large_kernel<2>), dim3((unsigned)total), dim3(256), 0, stream, p, row_tiles, col_tiles);
  return hipGetLastError();
}

}  // namespace asrattn
