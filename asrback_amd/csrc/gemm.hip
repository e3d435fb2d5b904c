// The projections around a module's attention over rows of bf16
// (asrlayer_gemm): x w^T, plus a bias or added to what the output holds.
//
// Two tilings, on v_mfma_f32_16x16x32_bf16 and v_mfma_f32_32x32x16_bf16, with
// the weight rows as the first operand, so that a lane's accumulators are
// consecutive outputs of one row:
//
//   * Few rows: a workgroup takes 16 or 32 rows x 16 or 32 outputs, each of its
//     four waves (eight from 768 inputs on) a part of the reduction, operands
//     straight from memory into registers, all of a wave's steps in flight up to
//     1280 inputs.  Bound by a round trip to memory and by what a CU loads (64 x 64
//     tiles in registers: 300 rows of 512 to 1536 outputs 6.6 -> 8.0 us).
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

typedef float f32x4_t __attribute__((ext_vector_type(4)));

// 16 RT rows x 16 CT outputs on v_mfma_f32_16x16x32_bf16; NW waves share the
// reduction, kAhead steps of 32 in flight.
template <int RT, int CT, int NW, int kAhead>
__global__ __launch_bounds__(64 * NW) void gemm_small_kernel(const asrlayer_gemm_params p, int row_tiles, int col_tiles) {
  const int item = xcd_remap((int)blockIdx.x, (int)gridDim.x);
  const int n0 = item % col_tiles * (16 * CT);
  const int row0 = item / col_tiles % row_tiles * (16 * RT);
  const RowView v = row_view(p, item / col_tiles / row_tiles);
  if (row0 >= v.rows) return;  // uniform over the workgroup

  const int lane = threadIdx.x & 63, r16 = lane & 15, quad = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int part = p.k / NW;
  const int64_t k0 = wave * part + quad * 8;
  const bf16_raw *xp[RT], *wp[CT];
#pragma unroll
  for (int i = 0; i < RT; ++i) xp[i] = v.x + (int64_t)min(row0 + 16 * i + r16, v.rows - 1) * p.x_row_stride + k0;
#pragma unroll
  for (int j = 0; j < CT; ++j)
    wp[j] = static_cast<const bf16_raw*>(p.w) + (int64_t)min(n0 + 16 * j + r16, p.n - 1) * p.k + k0;
  const int steps = part / 32;
  f32x4_t acc[RT][CT] = {};
  for (int s0 = 0; s0 < steps; s0 += kAhead) {
    bf16x8_t w[kAhead][CT], x[kAhead][RT];
#pragma unroll
    for (int a = 0; a < kAhead; ++a) {
      const int s = min(s0 + a, steps - 1);  // past the last: repeated, unused
#pragma unroll
      for (int j = 0; j < CT; ++j) w[a][j] = __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const uint4*>(wp[j] + s * 32));
#pragma unroll
      for (int i = 0; i < RT; ++i) x[a][i] = __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const uint4*>(xp[i] + s * 32));
    }
#pragma unroll
    for (int a = 0; a < kAhead; ++a)
      if (s0 + a < steps) {
#pragma unroll
        for (int i = 0; i < RT; ++i)
#pragma unroll
          for (int j = 0; j < CT; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[a][j], x[a][i], acc[i][j], 0, 0, 0);
      }
  }
  // Sum the waves' parts: accumulator r of a lane is output 16 j + 4 quad + r of
  // row 16 i + r16.
  __shared__ float sm[NW][16 * RT][16 * CT + 4];
#pragma unroll
  for (int i = 0; i < RT; ++i)
#pragma unroll
    for (int j = 0; j < CT; ++j)
      *reinterpret_cast<float4*>(&sm[wave][16 * i + r16][16 * j + 4 * quad]) =
          make_float4(acc[i][j][0], acc[i][j][1], acc[i][j][2], acc[i][j][3]);
  __syncthreads();
  for (int t = threadIdx.x; t < 64 * RT * CT; t += 64 * NW) {
    const int m = t / (4 * CT), c = t % (4 * CT) * 4;
    float y[4] = {};
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      const float4 one = *reinterpret_cast<const float4*>(&sm[w][m][c]);
      y[0] += one.x;
      y[1] += one.y;
      y[2] += one.z;
      y[3] += one.w;
    }
    if (row0 + m < v.rows && n0 + c < p.n) finish<1>(p, y, v.out + (int64_t)(row0 + m) * p.out_row_stride, n0 + c);
  }
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

namespace {

template <int RT, int CT, int NW, int kAhead>
hipError_t launch_waves(const asrlayer_gemm_params& p, hipStream_t stream) {
  const int row_tiles = (p.rows + 16 * RT - 1) / (16 * RT), col_tiles = (p.n + 16 * CT - 1) / (16 * CT);
  const long long total = (long long)p.batch * row_tiles * col_tiles;
  if (total > 0x7fffffffLL) return hipErrorInvalidConfiguration;
  hipLaunchKernelGGL((gemm_small_kernel<RT, CT, NW, kAhead>), dim3((unsigned)total), dim3(64 * NW), 0, stream, p,
                     row_tiles, col_tiles);
  return hipGetLastError();
}

// The waves a reduction takes, whole steps each, with all of a wave's steps in
// flight up to 1280.
template <int RT, int CT>
hipError_t launch_small(const asrlayer_gemm_params& p, hipStream_t stream) {
  if (p.k % 128 != 0) return launch_waves<RT, CT, 2, 8>(p, stream);
  if (p.k <= 512 || p.k % 256 != 0) return launch_waves<RT, CT, 4, 4>(p, stream);
  if (p.k <= 768) return launch_waves<RT, CT, 8, 3>(p, stream);
  return launch_waves<RT, CT, 8, 5>(p, stream);
}

template <int NB>
hipError_t launch_large(const asrlayer_gemm_params& p, hipStream_t stream) {
  const int row_tiles = (p.rows + kBM - 1) / kBM, col_tiles = (p.n + 64 * NB - 1) / (64 * NB);
  const long long total = (long long)p.batch * row_tiles * col_tiles;
  if (total > 0x7fffffffLL) return hipErrorInvalidConfiguration;
  hipLaunchKernelGGL((gemm_large_kernel<NB>), dim3((unsigned)total), dim3(256), 0, stream, p, row_tiles, col_tiles);
  return hipGetLastError();
}

}  // namespace

hipError_t launch_gemm(const asrlayer_gemm_params& p, hipStream_t stream) {
  // Counted over all rows as one run, whatever part of them is computed: the
  // tilings sum in different orders, and at one padded shape a row's result
  // does not depend on the counts.
  const auto tiles = [&](int rows, int outputs) {
    return (((long long)p.batch * p.rows + rows - 1) / rows) * ((p.n + outputs - 1) / outputs);
  };
  // The smallest workgroups that make at most one per CU, for these are bound by
  // what a CU loads (43 bytes a clock); 16 x 16, 32 x 16 and 32 x 32, us: 32 rows
  // of 768 to 768 outputs 4.2, 4.8, 5.4 (the library's product: 5.2), 128 rows 5.4,
  // 4.9, 5.5 (5.3), 32 of 1280 5.0, 6.1, 7.2 (5.5).  32 x 32 up to three or four
  // per CU: 300 rows of 512 to 1536 outputs (480 of them) 6.6 against 8.7 in large
  // tiles; within SAN-M's layer, whose operands the kernel before has just
  // written, 500 rows (768) 25.1 and 25.4 a layer, 600 (912) 26.3 and 24.8; added
  // to 512 outputs, 1200 rows (608) 27.3 and 30.7, 1800 (912) 29.2 and 31.2, 2048
  // (1024) 25.0 and 23.4.
  if (tiles(16, 16) <= 256) return launch_small<1, 1>(p, stream);
  if (tiles(32, 16) <= 256) return launch_small<2, 1>(p, stream);
  if (tiles(32, 32) <= (p.accumulate ? 1000 : 800)) return launch_small<2, 2>(p, stream);
  // 192 outputs a workgroup where they divide the outputs and leave at least a
  // round of workgroups (two per CU): five operand reads for six products
  // instead of four for four, and fewer rounds (16128 rows to 1536 outputs 45
  // -> 40 us).
  const bool wide = p.n % 192 == 0 && tiles(kBM, 192) >= 512;
  return wide ? launch_large<3>(p, stream) : launch_large<2>(p, stream);
}

}  // namespace asrattn
