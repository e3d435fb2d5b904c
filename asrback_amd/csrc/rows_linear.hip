// A decoder step's linear layers over at most 16 rows (asrlayer_rows_linear):
// up to three weight matrices over the same rows, with the layer norm before
// them and the activation or residual sum after them.
//
// Bound by launches and latency at the smallest models (float32, width 384,
// one row: 0.6 MB of weights a matrix), by reading the weights at larger
// ones.  As separate operations a Whisper decoder layer's step took 27
// launches of 4-5 us each (norm, bias copy, product, activation and sum apart);
// here it takes six of 3.3-3.8 us (a kernel that does nothing takes 1.8), besides
// its two attention launches.
//
// A wave takes two weight rows (output columns) and spreads the reduction over
// its lanes: a lane holds up to six 16-byte vectors of every input row and of
// each weight row, all loaded at once, so a launch is one round trip to memory,
// two sums over the lanes for the layer norm (statistics in two passes, in
// registers), and one for the products.  The weight rows are read in whole
// cache lines, once for each four input rows.  Longer reductions take a
// workgroup, a vector per thread, and sum over it.
#include "kernels.hpp"
#include "layers.hpp"
#include "row_ops.hpp"

namespace asrattn {
namespace {

constexpr int kMaxWaves = 16;

template <typename T>
__device__ __forceinline__ float dot_vec(const uint4& a, const uint4& b);

template <>
__device__ __forceinline__ float dot_vec<float>(const uint4& a, const uint4& b) {
  float acc = __uint_as_float(a.x) * __uint_as_float(b.x);
  acc = fmaf(__uint_as_float(a.y), __uint_as_float(b.y), acc);
  acc = fmaf(__uint_as_float(a.z), __uint_as_float(b.z), acc);
  return fmaf(__uint_as_float(a.w), __uint_as_float(b.w), acc);
}

template <>
__device__ __forceinline__ float dot_vec<bf16_raw>(const uint4& a, const uint4& b) {
  float x[8], y[8];
  unpack<bf16_raw>(a, x);
  unpack<bf16_raw>(b, y);
  float acc = x[0] * y[0];
#pragma unroll
  for (int e = 1; e < 8; ++e) acc = fmaf(x[e], y[e], acc);
  return acc;
}

// Sums each of a wave's R values over its lanes (R a power of two up to 32).
// While values remain, a step adds the partner lanes' values and leaves each
// lane half as many; the sum of value i ends in the lanes whose bits
// (5, 4, ...) spell i, value 0 of v.
template <int R, int OFF>
__device__ __forceinline__ void sum_lanes(float* v, int lane) {
  if constexpr (OFF == 0) {
    return;
  } else if constexpr (R > 1) {
#pragma unroll
    for (int i = 0; i < R / 2; ++i) {
      const float a = v[i], b = v[i + R / 2];
      if constexpr (OFF == 32) {
        const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
        v[i] = __uint_as_float(r[0]) + __uint_as_float(r[1]);
      } else if constexpr (OFF == 16) {
        const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
        v[i] = __uint_as_float(r[0]) + __uint_as_float(r[1]);
      } else {
        const bool upper = (lane & OFF) != 0;
        v[i] = (upper ? b : a) + __shfl_xor(upper ? a : b, OFF, 64);
      }
    }
    sum_lanes<R / 2, OFF / 2>(v, lane);
  } else {
    v[0] += __shfl_xor(v[0], OFF, 64);
    sum_lanes<1, OFF / 2>(v, lane);
  }
}

// The value sum_lanes<R> leaves in `lane`.
template <int R>
__device__ __forceinline__ int summed_value(int lane) {
  constexpr int kBits = R == 1 ? 0 : R == 2 ? 1 : R == 4 ? 2 : R == 8 ? 3 : R == 16 ? 4 : 5;
  return lane >> (6 - kBits);
}

// Output column `col` of the launch: the matrix it belongs to and its row.
struct Column {
  int matrix, n;
};
__device__ __forceinline__ Column column_of(const asrlayer_linear_params& p, int col) {
  const int n01 = p.n[0] + p.n[1];
  const int i = col < p.n[0] ? 0 : col < n01 ? 1 : 2;
  return {i, col - (i == 0 ? 0 : i == 1 ? p.n[0] : n01)};
}
template <typename P>
__device__ __forceinline__ P pick(P const* three, int i) {
  return i == 0 ? three[0] : i == 1 ? three[1] : three[2];
}

// Sums v[m] over the workgroup; every thread gets all the sums.
template <int R>
__device__ __forceinline__ void sum_workgroup(float* v, float (*sm)[R], int waves, int wave, int lane) {
  float u[R];
#pragma unroll
  for (int m = 0; m < R; ++m) u[m] = v[m];
  sum_lanes<R, 32>(u, lane);
  if (lane % (64 / R) == 0) sm[wave][summed_value<R>(lane)] = u[0];
  __syncthreads();
#pragma unroll
  for (int m = 0; m < R; ++m) v[m] = 0.f;
  for (int w = 0; w < waves; ++w)
#pragma unroll
    for (int m = 0; m < R; ++m) v[m] += sm[w][m];
}

__device__ __forceinline__ float gelu(float x) { return 0.5f * x * (1.f + erff(x * 0.70710678118654752f)); }

// Bias, activation and residual of one sum, rounded where the separate
// operations round, and its store.
template <typename T>
__device__ __forceinline__ void finish(const asrlayer_linear_params& p, Column c, int row, float y) {
  const T* bias = static_cast<const T*>(pick(p.b, c.matrix));
  T* out = static_cast<T*>(pick(p.out, c.matrix));
  if (bias != nullptr) y += Elem<T>::load1(bias + c.n);
  if (p.act == 1) y = gelu(round_to<T>(y));
  if (p.residual != nullptr)
    y = round_to<T>(y) + Elem<T>::load1(static_cast<const T*>(p.residual) + row * p.r_row_stride + c.n);
  Elem<T>::store1(out + (int64_t)row * pick(p.n, c.matrix) + c.n, y);
}

// A wave for kCols columns: every lane holds NV vectors of each row, the first
// kFull of which lie in the row whatever its length (the launch takes the
// smallest of 1, 2, 3 and 6 that holds it).
template <typename T, int R, int NV, int kCols>
__global__ __launch_bounds__(64) void rows_wave_kernel(const asrlayer_linear_params p) {
  constexpr int EPL = Elem<T>::kPerVec;
  constexpr int kFull = NV == 6 ? 3 : NV - 1;
  const int lane = threadIdx.x;
  const int vecs = p.k / EPL;
  const int columns = p.n[0] + p.n[1] + p.n[2];
  const int col0 = blockIdx.x * kCols, row0 = blockIdx.y * R;
  uint4 x[R][NV], w[kCols][NV], lw[NV], lb[NV];
  const bool norm = p.ln_weight != nullptr;
#pragma unroll
  for (int v = 0; v < NV; ++v) {
    const int at = min(v * 64 + lane, vecs - 1) * EPL;
#pragma unroll
    for (int m = 0; m < R; ++m)
      x[m][v] = *reinterpret_cast<const uint4*>(static_cast<const T*>(p.x) + min(row0 + m, p.rows - 1) * p.x_row_stride + at);
#pragma unroll
    for (int c = 0; c < kCols; ++c) {
      const Column k = column_of(p, min(col0 + c, columns - 1));
      w[c][v] = *reinterpret_cast<const uint4*>(static_cast<const T*>(pick(p.w, k.matrix)) + (int64_t)k.n * p.k + at);
    }
    // Without a norm these repeat a weight row (and are unused).
    const T* lwp = static_cast<const T*>(norm ? p.ln_weight : p.w[0]);
    const T* lbp = static_cast<const T*>(norm ? p.ln_bias : p.w[0]);
    lw[v] = *reinterpret_cast<const uint4*>(lwp + at);
    lb[v] = *reinterpret_cast<const uint4*>(lbp + at);
  }
#pragma unroll
  for (int v = kFull; v < NV; ++v)
    if (v * 64 + lane >= vecs) {
#pragma unroll
      for (int m = 0; m < R; ++m) x[m][v] = make_uint4(0u, 0u, 0u, 0u);
    }
  if (norm) {
    const float inv_k = 1.f / (float)p.k;
#pragma unroll
    for (int m = 0; m < R; ++m) {
      float sum = 0.f;
#pragma unroll
      for (int v = 0; v < NV; ++v) {
        float f[EPL];
        unpack<T>(x[m][v], f);
#pragma unroll
        for (int e = 0; e < EPL; ++e) sum += f[e];
      }
      const float mean = group_sum<64>(sum) * inv_k;
      float var = 0.f;
#pragma unroll
      for (int v = 0; v < NV; ++v) {
        float f[EPL];
        unpack<T>(x[m][v], f);
        float part = 0.f;
#pragma unroll
        for (int e = 0; e < EPL; ++e) part = fmaf(f[e] - mean, f[e] - mean, part);
        var += v < kFull || v * 64 + lane < vecs ? part : 0.f;
      }
      const float r = rsqrtf(group_sum<64>(var) * inv_k + p.ln_eps);
#pragma unroll
      for (int v = 0; v < NV; ++v) {
        float f[EPL], g[EPL], b[EPL];
        unpack<T>(x[m][v], f);
        unpack<T>(lw[v], g);
        unpack<T>(lb[v], b);
#pragma unroll
        for (int e = 0; e < EPL; ++e) f[e] = fmaf((f[e] - mean) * r, g[e], b[e]);
        const uint4 y = pack<T>(f);
        x[m][v] = v < kFull || v * 64 + lane < vecs ? y : make_uint4(0u, 0u, 0u, 0u);
      }
    }
  }
  float acc[kCols * R];
#pragma unroll
  for (int c = 0; c < kCols; ++c)
#pragma unroll
    for (int m = 0; m < R; ++m) {
      float y = 0.f;
#pragma unroll
      for (int v = 0; v < NV; ++v) {
        // Past the row the weights repeat its last vector: 0 times an infinite
        // one is not 0.
        float part = dot_vec<T>(x[m][v], w[c][v]);
        if (v >= kFull) part = v * 64 + lane < vecs ? part : 0.f;
        y = v == 0 ? part : y + part;
      }
      acc[c * R + m] = y;
    }
  sum_lanes<kCols * R, 32>(acc, lane);
  const int i = summed_value<kCols * R>(lane);
  const int col = col0 + i / R, row = row0 + i % R;
  if (lane % (64 / (kCols * R)) == 0 && col < columns && row < p.rows) finish<T>(p, column_of(p, col), row, acc[0]);
}

// A workgroup for kCols columns, a vector per thread.  R: rows of a workgroup, a
// power of two (rows past the last repeat it).
template <typename T, int R, int kCols>
__global__ __launch_bounds__(1024) void rows_linear_kernel(const asrlayer_linear_params p) {
  constexpr int EPL = Elem<T>::kPerVec;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int waves = blockDim.x >> 6;
  const int vecs = p.k / EPL;
  const bool mine = tid < vecs;
  const int at = (mine ? tid : 0) * EPL;

  __shared__ float sm_norm[2][kMaxWaves][R];
  __shared__ float sm_dot[kMaxWaves][kCols][R];

  // The column's weight row: matrices one after another.
  const int columns = p.n[0] + p.n[1] + p.n[2];
  const int col0 = blockIdx.x * kCols, row0 = blockIdx.y * R;
  uint4 x[R], w[kCols], lw = {}, lb = {};
#pragma unroll
  for (int m = 0; m < R; ++m)
    x[m] = *reinterpret_cast<const uint4*>(static_cast<const T*>(p.x) + min(row0 + m, p.rows - 1) * p.x_row_stride + at);
  const bool norm = p.ln_weight != nullptr;
  if (norm) {
    lw = *reinterpret_cast<const uint4*>(static_cast<const T*>(p.ln_weight) + at);
    lb = *reinterpret_cast<const uint4*>(static_cast<const T*>(p.ln_bias) + at);
  }
#pragma unroll
  for (int c = 0; c < kCols; ++c) {
    const int col = min(col0 + c, columns - 1);
    const Column k = column_of(p, col);
    w[c] = *reinterpret_cast<const uint4*>(static_cast<const T*>(pick(p.w, k.matrix)) + (int64_t)k.n * p.k + at);
  }
  if (!mine) {
#pragma unroll
    for (int m = 0; m < R; ++m) x[m] = make_uint4(0u, 0u, 0u, 0u);
  }

  if (norm) {
    // Rounded once to T, as torch's layer_norm does.
    float mean[R], var[R];
#pragma unroll
    for (int m = 0; m < R; ++m) {
      float f[EPL];
      unpack<T>(x[m], f);
      mean[m] = f[0];
#pragma unroll
      for (int e = 1; e < EPL; ++e) mean[m] += f[e];
    }
    sum_workgroup<R>(mean, sm_norm[0], waves, wave, lane);
    const float inv_k = 1.f / (float)p.k;
#pragma unroll
    for (int m = 0; m < R; ++m) {
      mean[m] *= inv_k;
      float f[EPL];
      unpack<T>(x[m], f);
      var[m] = 0.f;
#pragma unroll
      for (int e = 0; e < EPL; ++e) {
        const float d = f[e] - mean[m];
        var[m] = fmaf(d, d, var[m]);
      }
      var[m] = mine ? var[m] : 0.f;
    }
    sum_workgroup<R>(var, sm_norm[1], waves, wave, lane);
    float g[EPL], b[EPL];
    unpack<T>(lw, g);
    unpack<T>(lb, b);
#pragma unroll
    for (int m = 0; m < R; ++m) {
      const float r = rsqrtf(var[m] * inv_k + p.ln_eps);
      float f[EPL];
      unpack<T>(x[m], f);
#pragma unroll
      for (int e = 0; e < EPL; ++e) f[e] = fmaf((f[e] - mean[m]) * r, g[e], b[e]);
      const uint4 y = pack<T>(f);
      x[m] = mine ? y : make_uint4(0u, 0u, 0u, 0u);
    }
  }

#pragma unroll
  for (int c = 0; c < kCols; ++c) {
    float acc[R];
#pragma unroll
    for (int m = 0; m < R; ++m) acc[m] = mine ? dot_vec<T>(x[m], w[c]) : 0.f;
    sum_lanes<R, 32>(acc, lane);
    if (lane % (64 / R) == 0) sm_dot[wave][c][summed_value<R>(lane)] = acc[0];
  }
  __syncthreads();

  if (tid < kCols * R) {
    const int c = tid % kCols, m = tid / kCols, row = row0 + m;
    const int col = col0 + c;
    if (col < columns && row < p.rows) {
      float y = 0.f;
      for (int v = 0; v < waves; ++v) y += sm_dot[v][c][m];
      finish<T>(p, column_of(p, col), row, y);
    }
  }
}

template <typename T, int R, int NV, int kCols>
hipError_t launch_columns(const asrlayer_linear_params& p, hipStream_t stream) {
  const int columns = p.n[0] + p.n[1] + p.n[2];
  hipLaunchKernelGGL((rows_wave_kernel<T, R, NV, kCols>), dim3((columns + kCols - 1) / kCols, (p.rows + R - 1) / R),
                     dim3(64), 0, stream, p);
  return hipGetLastError();
}

template <typename T, int R, int NV>
hipError_t launch_wave(const asrlayer_linear_params& p, hipStream_t stream) {
  // A vocabulary's columns: eight a wave (four of long rows), more loads in
  // flight and fewer waves to start (one float32 row through 51865 x 384: 14.3
  // us, 5.6 TB/s; the library's product 20.7).
  constexpr int kMany = NV <= 3 ? 8 : 4;
  if (p.n[0] + p.n[1] + p.n[2] >= 16384) return launch_columns<T, R, NV, kMany>(p, stream);
  return launch_columns<T, R, NV, 2>(p, stream);
}

template <typename T, int NV>
hipError_t launch_wave_rows(const asrlayer_linear_params& p, hipStream_t stream) {
  if (p.rows <= 1) return launch_wave<T, 1, NV>(p, stream);
  if (p.rows <= 2) return launch_wave<T, 2, NV>(p, stream);
  return launch_wave<T, 4, NV>(p, stream);
}

template <typename T, int R>
hipError_t launch_rows(const asrlayer_linear_params& p, int threads, hipStream_t stream) {
  const int columns = p.n[0] + p.n[1] + p.n[2];
  constexpr int kCols = 4;
  static_assert(kCols * R <= 64, "an output per thread of one wave");
  hipLaunchKernelGGL((rows_linear_kernel<T, R, kCols>), dim3((columns + kCols - 1) / kCols, (p.rows + R - 1) / R),
                     dim3(threads), 0, stream, p);
  return hipGetLastError();
}

template <typename T>
hipError_t launch_typed(const asrlayer_linear_params& p, hipStream_t stream) {
  const int threads = (p.k / Elem<T>::kPerVec + 63) / 64 * 64;
  // A wave per column pair up to six vectors a lane (what its registers hold
  // for four rows): one row through 384 x 1152 float32 with the norm 4.7 -> 3.5
  // us against a workgroup per four columns, eight rows 6.0 -> 4.7; 1536 x 384
  // 4.1 -> 3.8, 1280 x 1280 bf16 with the norm 5.1 -> 4.0.
  if (threads <= 64) return launch_wave_rows<T, 1>(p, stream);
  if (threads <= 128) return launch_wave_rows<T, 2>(p, stream);
  if (threads <= 192) return launch_wave_rows<T, 3>(p, stream);
  if (threads <= 384) return launch_wave_rows<T, 6>(p, stream);
  if (p.rows <= 1) return launch_rows<T, 1>(p, threads, stream);
  if (p.rows <= 2) return launch_rows<T, 2>(p, threads, stream);
  return launch_rows<T, 4>(p, threads, stream);
}

// Sums of a token's and a position's embedding, a row per workgroup: launch and
// latency, one launch for three.
template <typename T>
__global__ __launch_bounds__(256) void embed_rows_kernel(const asrlayer_embed_params p) {
  constexpr int EPL = Elem<T>::kPerVec;
  const int row = blockIdx.x;
  const int64_t token = load_uniform(p.tokens + row * p.token_stride), pos = load_uniform(p.positions + row);
  const bool ok = token >= 0 && token < p.vocab && pos >= 0 && pos < p.length;
  const T* a = static_cast<const T*>(p.token_weight) + (ok ? token : 0) * p.width;
  const T* b = static_cast<const T*>(p.position_weight) + (ok ? pos : 0) * p.width;
  T* out = static_cast<T*>(p.out) + (int64_t)row * p.width;
  for (int at = threadIdx.x * EPL; at < p.width; at += 256 * EPL) {
    float x[EPL], y[EPL];
    unpack<T>(*reinterpret_cast<const uint4*>(a + at), x);
    unpack<T>(*reinterpret_cast<const uint4*>(b + at), y);
#pragma unroll
    for (int e = 0; e < EPL; ++e) x[e] = ok ? x[e] + y[e] : __builtin_nanf("");
    *reinterpret_cast<uint4*>(out + at) = pack<T>(x);
  }
}

}  // namespace

hipError_t launch_embed_rows(const asrlayer_embed_params& p, hipStream_t stream) {
  if (p.dtype == ASRATTN_BF16)
    hipLaunchKernelGGL((embed_rows_kernel<bf16_raw>), dim3(p.rows), dim3(256), 0, stream, p);
  else
    hipLaunchKernelGGL((embed_rows_kernel<float>), dim3(p.rows), dim3(256), 0, stream, p);
  return hipGetLastError();
}

hipError_t launch_rows_linear(const asrlayer_linear_params& p, hipStream_t stream) {
  return p.dtype == ASRATTN_BF16 ? launch_typed<bf16_raw>(p, stream) : launch_typed<float>(p, stream);
}

}  // namespace asrattn
