// Row reductions over the last axis of [rows, cols]: softmax and LayerNorm.
//
// A row is owned by 8, 16, 32, 64 or 256 lanes, whichever hold it as at most four (fp32 up to eight) 16-byte vectors
// each: it is read once, reduced with cross-lane shuffles (and LDS across four waves), and written once. Rows shorter
// than one vector take one element per lane; rows too long for registers fall back to one workgroup per row that
// streams the row through global memory in three passes.
//
// softmax (reference: src/backends/cpu/kernels/sequence.cpp:114-174): m = max, e = exp(x - m), s = sum(e),
// y = round(e / s). LayerNorm (reference: src/backends/cpu/kernels/sequence.cpp:182-279): two-pass mean and
// variance, r = 1 / sqrt(var + eps), y = round(gamma * ((x - mean) * r) + beta). All arithmetic in fp32;
// multiplies and adds are not contracted, division and sqrt are correctly rounded. For 16-bit rows of up to 2,048
// elements softmax evaluates e as 2^((x - m) log2 e) on v_exp_f32 and y as round(e * (1 / s)): the
// same d = x - m as the reference, an exponential within a few fp32 ulps of expf and a quotient within one, which
// changes a stored 8- or 11-bit probability only where it lies that close to a rounding boundary. expf and the
// correctly rounded division cost about 25 VALU instructions per element and made the [65536, 512] bf16 softmax
// instruction-bound (30.7 us for 134 MB); longer rows and fp32 keep them ([4096, 8192] f16 35.1 us, 23.9 without).
#include <hip/hip_runtime.h>

#include <string>
#include <type_traits>

#include "fh_common.h"

namespace fh {
namespace {

__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const float other = __shfl_xor(v, o, 64);
    v = (other > v) ? other : v;
  }
  return v;
}

__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}

constexpr int kRowsPerBlock = 4;  // 4 waves, one row each

// softmax's e = exp(d) for d = x - m: expf, or (FAST) 2^(d log2 e) on v_exp_f32
template <bool FAST>
__device__ __forceinline__ float softmax_exp(float d) {
  if constexpr (FAST) {
    return __builtin_amdgcn_exp2f(d * 1.44269504088896340736f);
  } else {
    return expf(d);
  }
}
// y = e / s: correctly rounded, or (FAST) e * (1 / s) (r passed in)
template <bool FAST>
__device__ __forceinline__ float softmax_div(float e, float s, float r) {
  if constexpr (FAST) {
    return e * r;
  } else {
    return e / s;
  }
}
// 16-bit rows of up to 2,048 elements take the fast forms; longer ones and fp32 do not.
template <typename T, int L>
constexpr bool softmax_fast() {
  return !std::is_same_v<T, float> && L <= 64;
}

// A row's 16-byte vectors over its L lanes (256 / L rows per workgroup): lane l holds the elements
// [V * (l + L * t), + V) for t < NV. Rows start wherever row * cols puts them, so the accesses are 16 bytes at element
// alignment (global memory takes them at any alignment). kRowFull: the row is exactly V * NV * L elements, no lane is
// idle. kRowVectors: whole vectors, the last lanes idle. kRowRagged: cols is no multiple of V, and the row's last vector
// is moved back to end at the row's end; the elements it then shares with the vector before it ("dup" of them) are
// left out of the sums, and both lanes store them with the same value.
// What bounds these kernels is HBM once the accesses are vectors (softmax bf16, us, one element per lane and access
// before): [32768, 1000] 53.0 -> 23.6 (5.6 TB/s), [32768, 1001] 53.7 -> 26.4, [65536, 47] f32 12.7 -> 6.9; rows of
// more than 2,048 elements, in three passes over memory before: [4096, 8192] f16 81 -> 35 (LayerNorm 64 -> 27).
enum RowMode { kRowFull, kRowVectors, kRowRagged };

template <int V, int NV, int L, int MODE>
struct RowVectors {
  int64_t at[NV];  // first element of each vector; -1 where the row has none
  int dup[NV];     // elements at its start that the vector before it holds as well
  __device__ RowVectors(int l, int64_t cols) {
#pragma unroll
    for (int t = 0; t < NV; ++t) {
      const int64_t j = static_cast<int64_t>(V) * (l + L * t);
      at[t] = j;
      dup[t] = 0;
      if constexpr (MODE != kRowFull) at[t] = j >= cols ? -1 : at[t];
      if constexpr (MODE == kRowRagged) {
        if (j < cols && j + V > cols) at[t] = cols - V, dup[t] = static_cast<int>(j - at[t]);
      }
    }
  }
  __device__ bool has(int t) const { return MODE == kRowFull || at[t] >= 0; }
  // whether element i of vector t is this lane's own
  __device__ bool own(int t, int i) const { return has(t) && (MODE != kRowRagged || i >= dup[t]); }
};

// One 16-byte vector at element alignment. Each row is read and written once, so whole rows go past the caches
// (non-temporal); a ragged row shares its first and last cache lines with its neighbours and does not.
typedef unsigned int u4_t __attribute__((ext_vector_type(4)));
typedef u4_t u4_any __attribute__((aligned(2)));
template <typename T, int MODE, int V>
__device__ __forceinline__ void row_load(const typename Io<T>::storage* p, float (&v)[V]) {
  const u4_any* q = reinterpret_cast<const u4_any*>(p);
  u4_t w;
  if constexpr (MODE == kRowRagged) w = *q;
  else w = __builtin_nontemporal_load(q);
  unpack_vec<T>(make_uint4(w.x, w.y, w.z, w.w), v);
}
template <typename T, int MODE, int V>
__device__ __forceinline__ void row_store(typename Io<T>::storage* p, const float (&v)[V]) {
  const uint4 w = pack_vec<T>(v);
  u4_any* q = reinterpret_cast<u4_any*>(p);
  if constexpr (MODE == kRowRagged) *q = u4_t{w.x, w.y, w.z, w.w};
  else __builtin_nontemporal_store(u4_t{w.x, w.y, w.z, w.w}, q);
}

// Reductions over the L lanes of a row (L = 256: all four waves of the workgroup, through `scratch`).
template <int L>
__device__ __forceinline__ float row_max(float v, float* scratch) {
#pragma unroll
  for (int o = (L < 64 ? L : 64) / 2; o > 0; o >>= 1) {
    const float other = __shfl_xor(v, o, 64);
    v = (other > v) ? other : v;
  }
  if constexpr (L == 256) {
    if ((threadIdx.x & 63) == 0) scratch[threadIdx.x >> 6] = v;
    __syncthreads();
    v = scratch[0];
#pragma unroll
    for (int k = 1; k < 4; ++k) v = (scratch[k] > v) ? scratch[k] : v;
  }
  return v;
}
template <int L>
__device__ __forceinline__ float row_sum(float v, float* scratch) {
#pragma unroll
  for (int o = (L < 64 ? L : 64) / 2; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  if constexpr (L == 256) {
    if ((threadIdx.x & 63) == 0) scratch[threadIdx.x >> 6] = v;
    __syncthreads();
    v = ((scratch[0] + scratch[1]) + scratch[2]) + scratch[3];
  }
  return v;
}

template <typename T, int NV, int L, int MODE>
__global__ __launch_bounds__(256) void softmax_row_kernel(const typename Io<T>::storage* __restrict__ x,
                                                          typename Io<T>::storage* __restrict__ y, int64_t rows,
                                                          int64_t cols) {
  constexpr int V = 16 / static_cast<int>(sizeof(typename Io<T>::storage));
  constexpr bool FAST = softmax_fast<T, L>();
  __shared__ float scratch[2][4];
  const int64_t row = static_cast<int64_t>(blockIdx.x) * (256 / L) + threadIdx.x / L;
  if (row >= rows) return;  // (whole row groups leave; with L = 256 every workgroup has its row)
  const RowVectors<V, NV, L, MODE> rv(threadIdx.x % L, cols);
  const auto* xr = x + row * cols;
  auto* yr = y + row * cols;
  float v[NV][V];
#pragma unroll
  for (int t = 0; t < NV; ++t) {
    if (rv.has(t)) {
      row_load<T, MODE>(xr + rv.at[t], v[t]);
    } else {
#pragma unroll
      for (int i = 0; i < V; ++i) v[t][i] = -__builtin_inff();
    }
  }
  float m = -__builtin_inff();
#pragma unroll
  for (int t = 0; t < NV; ++t)
#pragma unroll
    for (int i = 0; i < V; ++i) m = (v[t][i] > m) ? v[t][i] : m;
  m = row_max<L>(m, scratch[0]);
  float s = 0.0f;
#pragma unroll
  for (int t = 0; t < NV; ++t)
#pragma unroll
    for (int i = 0; i < V; ++i) {
      v[t][i] = softmax_exp<FAST>(v[t][i] - m);
      s += rv.own(t, i) ? v[t][i] : 0.0f;
    }
  s = row_sum<L>(s, scratch[1]);
  const float r = 1.0f / s;
#pragma unroll
  for (int t = 0; t < NV; ++t) {
    if (!rv.has(t)) continue;
    float o[V];
#pragma unroll
    for (int i = 0; i < V; ++i) o[i] = softmax_div<FAST>(v[t][i], s, r);
    row_store<T, MODE>(yr + rv.at[t], o);
  }
}

// Rows shorter than one vector: one element per lane, one wave per row.
template <typename T>
__global__ __launch_bounds__(256) void softmax_short_kernel(const typename Io<T>::storage* __restrict__ x,
                                                            typename Io<T>::storage* __restrict__ y, int64_t rows,
                                                            int64_t cols) {
  const int lane = threadIdx.x & 63;
  const int64_t row = static_cast<int64_t>(blockIdx.x) * kRowsPerBlock + (threadIdx.x >> 6);
  if (row >= rows) return;
  const float v = (lane < cols) ? Io<T>::load(x[row * cols + lane]) : -__builtin_inff();
  const float m = wave_max((v > -__builtin_inff()) ? v : -__builtin_inff());
  constexpr bool FAST = softmax_fast<T, 64>();
  const float e = (lane < cols) ? softmax_exp<FAST>(v - m) : 0.0f;
  const float s = wave_sum(e);
  if (lane < cols) y[row * cols + lane] = Io<T>::store(softmax_div<FAST>(e, s, 1.0f / s));
}

__device__ float block_reduce(float v, bool is_max, float* scratch) {
  v = is_max ? wave_max(v) : wave_sum(v);
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  if (lane == 0) scratch[w] = v;
  __syncthreads();
  float r = scratch[0];
  for (int k = 1; k < static_cast<int>(blockDim.x >> 6); ++k)
    r = is_max ? ((scratch[k] > r) ? scratch[k] : r) : r + scratch[k];
  __syncthreads();
  return r;
}

template <typename T>
__global__ __launch_bounds__(256) void softmax_block_kernel(const typename Io<T>::storage* __restrict__ x,
                                                            typename Io<T>::storage* __restrict__ y, int64_t cols) {
  __shared__ float scratch[4];
  const auto* xr = x + static_cast<int64_t>(blockIdx.x) * cols;
  auto* yr = y + static_cast<int64_t>(blockIdx.x) * cols;
  float m = -__builtin_inff();
  for (int64_t j = threadIdx.x; j < cols; j += blockDim.x) {
    const float v = Io<T>::load(xr[j]);
    m = (v > m) ? v : m;
  }
  m = block_reduce(m, true, scratch);
  float s = 0.0f;
  for (int64_t j = threadIdx.x; j < cols; j += blockDim.x) s += expf(Io<T>::load(xr[j]) - m);
  s = block_reduce(s, false, scratch);
  for (int64_t j = threadIdx.x; j < cols; j += blockDim.x) yr[j] = Io<T>::store(expf(Io<T>::load(xr[j]) - m) / s);
}

template <typename T, int NV, int L, int MODE>
__global__ __launch_bounds__(256) void layer_norm_row_kernel(const typename Io<T>::storage* __restrict__ x,
                                                             const typename Io<T>::storage* __restrict__ gamma,
                                                             const typename Io<T>::storage* __restrict__ beta,
                                                             typename Io<T>::storage* __restrict__ y, int64_t rows,
                                                             int64_t cols, float eps) {
  constexpr int V = 16 / static_cast<int>(sizeof(typename Io<T>::storage));
  __shared__ float scratch[2][4];
  const int64_t row = static_cast<int64_t>(blockIdx.x) * (256 / L) + threadIdx.x / L;
  if (row >= rows) return;
  const RowVectors<V, NV, L, MODE> rv(threadIdx.x % L, cols);
  const auto* xr = x + row * cols;
  auto* yr = y + row * cols;
  // every load (x, gamma, beta) is issued before the first reduction, so one memory latency covers the row
  float v[NV][V];
  uint4 gv[NV], bv[NV];
#pragma unroll
  for (int t = 0; t < NV; ++t) {
    if (rv.has(t)) {
      row_load<T, MODE>(xr + rv.at[t], v[t]);
      __builtin_memcpy(&gv[t], gamma + rv.at[t], 16);
      __builtin_memcpy(&bv[t], beta + rv.at[t], 16);
    } else {
#pragma unroll
      for (int i = 0; i < V; ++i) v[t][i] = 0.0f;
      gv[t] = bv[t] = make_uint4(0, 0, 0, 0);
    }
  }
  float sum = 0.0f;
#pragma unroll
  for (int t = 0; t < NV; ++t)
#pragma unroll
    for (int i = 0; i < V; ++i) sum += rv.own(t, i) ? v[t][i] : 0.0f;
  const float mean = row_sum<L>(sum, scratch[0]) / static_cast<float>(cols);
  float var_sum = 0.0f;
#pragma unroll
  for (int t = 0; t < NV; ++t)
#pragma unroll
    for (int i = 0; i < V; ++i) {
      v[t][i] -= mean;  // kept for the normalisation (the same fp32 value the reference computes twice)
      var_sum += rv.own(t, i) ? v[t][i] * v[t][i] : 0.0f;
    }
  const float variance = row_sum<L>(var_sum, scratch[1]) / static_cast<float>(cols);
  const float r = 1.0f / sqrtf(variance + eps);
#pragma unroll
  for (int t = 0; t < NV; ++t) {
    if (!rv.has(t)) continue;
    float g[V], b[V], o[V];
    unpack_vec<T>(gv[t], g);
    unpack_vec<T>(bv[t], b);
#pragma unroll
    for (int i = 0; i < V; ++i) o[i] = g[i] * (v[t][i] * r) + b[i];
    row_store<T, MODE>(yr + rv.at[t], o);
  }
}

// Rows shorter than one vector: one element per lane, one wave per row.
template <typename T>
__global__ __launch_bounds__(256) void layer_norm_short_kernel(const typename Io<T>::storage* __restrict__ x,
                                                               const typename Io<T>::storage* __restrict__ gamma,
                                                               const typename Io<T>::storage* __restrict__ beta,
                                                               typename Io<T>::storage* __restrict__ y, int64_t rows,
                                                               int64_t cols, float eps) {
  const int lane = threadIdx.x & 63;
  const int64_t row = static_cast<int64_t>(blockIdx.x) * kRowsPerBlock + (threadIdx.x >> 6);
  if (row >= rows) return;
  const float v = (lane < cols) ? Io<T>::load(x[row * cols + lane]) : 0.0f;
  const float c = v - wave_sum(v) / static_cast<float>(cols);
  const float r = 1.0f / sqrtf(wave_sum((lane < cols) ? c * c : 0.0f) / static_cast<float>(cols) + eps);
  if (lane < cols) y[row * cols + lane] = Io<T>::store(Io<T>::load(gamma[lane]) * (c * r) + Io<T>::load(beta[lane]));
}

template <typename T>
__global__ __launch_bounds__(256) void layer_norm_block_kernel(const typename Io<T>::storage* __restrict__ x,
                                                               const typename Io<T>::storage* __restrict__ gamma,
                                                               const typename Io<T>::storage* __restrict__ beta,
                                                               typename Io<T>::storage* __restrict__ y, int64_t cols,
                                                               float eps) {
  __shared__ float scratch[4];
  const auto* xr = x + static_cast<int64_t>(blockIdx.x) * cols;
  auto* yr = y + static_cast<int64_t>(blockIdx.x) * cols;
  float sum = 0.0f;
  for (int64_t j = threadIdx.x; j < cols; j += blockDim.x) sum += Io<T>::load(xr[j]);
  const float mean = block_reduce(sum, false, scratch) / static_cast<float>(cols);
  float var_sum = 0.0f;
  for (int64_t j = threadIdx.x; j < cols; j += blockDim.x) {
    const float c = Io<T>::load(xr[j]) - mean;
    var_sum += c * c;
  }
  const float variance = block_reduce(var_sum, false, scratch) / static_cast<float>(cols);
  const float r = 1.0f / sqrtf(variance + eps);
  for (int64_t j = threadIdx.x; j < cols; j += blockDim.x) {
    const float xhat = (Io<T>::load(xr[j]) - mean) * r;
    yr[j] = Io<T>::store(Io<T>::load(gamma[j]) * xhat + Io<T>::load(beta[j]));
  }
}

// Lanes and vectors per row, for rows of at least one vector. The fewest of 8, 16, 32 or 64 lanes that hold the row as
// one vector each, so that short rows share a wave; then 64 lanes of up to four vectors, then the whole workgroup of
// 256, up to 64 values in a lane's registers. fp32 rows of 1,025 to 2,048 elements in whole vectors stay with one wave at
// eight vectors, which needs no barrier ([4096, 2048] LayerNorm 9.1 us, 13.4 on 256 lanes; softmax 9.7 / 12.0); ragged ones do
// not ([4096, 1999] LayerNorm 13.5 / 11.6) until there are 2^24 of them, a workgroup each and more than a launch holds.
// go<NV, L, MODE>() launches; false when the row does not fit.
template <int V, typename Go>
bool by_row_width(int64_t rows, int64_t cols, Go&& go) {
  const int64_t vecs = (cols + V - 1) / V;
  const auto pick = [&]<int NV, int L>() {
    if (cols == int64_t{V} * NV * L) go.template operator()<NV, L, kRowFull>();
    else if (cols % V == 0) go.template operator()<NV, L, kRowVectors>();
    else go.template operator()<NV, L, kRowRagged>();
    return true;
  };
  if (cols < V) return false;
  if (vecs <= 8) return pick.template operator()<1, 8>();
  if (vecs <= 16) return pick.template operator()<1, 16>();
  if (vecs <= 32) return pick.template operator()<1, 32>();
  if (vecs <= 64) return pick.template operator()<1, 64>();
  if (vecs <= 128) return pick.template operator()<2, 64>();
  if (vecs <= 256) return pick.template operator()<4, 64>();
  if (V == 4 && vecs <= 512 && (cols % V == 0 || rows >= (int64_t{1} << 24))) return pick.template operator()<8, 64>();
  if (vecs <= 512) return pick.template operator()<2, 256>();
  if (vecs <= 1024) return pick.template operator()<4, 256>();
  if (vecs <= 2048) return pick.template operator()<8, 256>();
  return false;
}
uint32_t row_blocks(int64_t rows, int lanes) {
  const int64_t per = 256 / lanes;
  return static_cast<uint32_t>((rows + per - 1) / per);
}

template <typename T>
fh_status softmax_typed(const void* x, void* y, int64_t rows, int64_t cols, hipStream_t s) {
  using S = typename Io<T>::storage;
  constexpr int V = 16 / static_cast<int>(sizeof(S));
  const S* xs = static_cast<const S*>(x);
  S* ys = static_cast<S*>(y);
  const auto row_kernel = [&]<int NV, int L, int MODE>() {
    hipLaunchKernelGGL((softmax_row_kernel<T, NV, L, MODE>), dim3(row_blocks(rows, L)), dim3(256), 0, s, xs, ys, rows,
                       cols);
  };
  if (by_row_width<V>(rows, cols, row_kernel)) return launch_status("softmax_row_kernel launch");
  if (cols < V) {
    hipLaunchKernelGGL(softmax_short_kernel<T>, dim3(row_blocks(rows, 64)), dim3(256), 0, s, xs, ys, rows, cols);
    return launch_status("softmax_short_kernel launch");
  }
  hipLaunchKernelGGL(softmax_block_kernel<T>, dim3(static_cast<uint32_t>(rows)), dim3(256), 0, s,
                     static_cast<const S*>(x), static_cast<S*>(y), cols);
  return launch_status("softmax_block_kernel launch");
}

template <typename T>
fh_status layer_norm_typed(const void* x, const void* g, const void* b, void* y, int64_t rows, int64_t cols,
                           float eps, hipStream_t s) {
  using S = typename Io<T>::storage;
  const S *xs = static_cast<const S*>(x), *gs = static_cast<const S*>(g), *bs = static_cast<const S*>(b);
  S* ys = static_cast<S*>(y);
  constexpr int V = 16 / static_cast<int>(sizeof(S));
  const auto row_kernel = [&]<int NV, int L, int MODE>() {
    hipLaunchKernelGGL((layer_norm_row_kernel<T, NV, L, MODE>), dim3(row_blocks(rows, L)), dim3(256), 0, s, xs, gs, bs,
                       ys, rows, cols, eps);
  };
  if (by_row_width<V>(rows, cols, row_kernel)) return launch_status("layer_norm_row_kernel launch");
  if (cols < V) {
    hipLaunchKernelGGL(layer_norm_short_kernel<T>, dim3(row_blocks(rows, 64)), dim3(256), 0, s, xs, gs, bs, ys, rows,
                       cols, eps);
    return launch_status("layer_norm_short_kernel launch");
  }
  hipLaunchKernelGGL(layer_norm_block_kernel<T>, dim3(static_cast<uint32_t>(rows)), dim3(256), 0, s,
                     static_cast<const S*>(x), static_cast<const S*>(g), static_cast<const S*>(b), static_cast<S*>(y),
                     cols, eps);
  return launch_status("layer_norm_block_kernel launch");
}

}  // namespace
}  // namespace fh

using namespace fh;

extern "C" fh_status fh_softmax_rows(int32_t dtype, const void* x, void* y, int64_t rows, int64_t cols,
                                     void* stream) {
  if (!is_supported_float(dtype)) return fail(FH_UNIMPLEMENTED, "fh_softmax_rows: unsupported dtype");
  if (rows < 0 || cols < 0) return fail(FH_INVALID_ARGUMENT, "fh_softmax_rows: negative size");
  if (rows == 0 || cols == 0) return FH_OK;
  if (rows > 0x7fffffffLL) return fail(FH_INVALID_ARGUMENT, "fh_softmax_rows: too many rows");
  if (x == nullptr || y == nullptr) return fail(FH_INVALID_ARGUMENT, "fh_softmax_rows: null pointer");
  hipStream_t s = static_cast<hipStream_t>(stream);
  switch (dtype) {
    case FH_F32:
      return softmax_typed<float>(x, y, rows, cols, s);
    case FH_BF16:
      return softmax_typed<bf16_t>(x, y, rows, cols, s);
    default:
      return softmax_typed<f16_t>(x, y, rows, cols, s);
  }
}

extern "C" fh_status fh_layer_norm_rows(int32_t dtype, const void* x, const void* gamma, const void* beta, void* y,
                                        int64_t rows, int64_t cols, float eps, void* stream) {
  if (!is_supported_float(dtype)) return fail(FH_UNIMPLEMENTED, "fh_layer_norm_rows: unsupported dtype");
  if (rows < 0 || cols < 0) return fail(FH_INVALID_ARGUMENT, "fh_layer_norm_rows: negative size");
  if (rows == 0 || cols == 0) return FH_OK;
  if (rows > 0x7fffffffLL) return fail(FH_INVALID_ARGUMENT, "fh_layer_norm_rows: too many rows");
  if (x == nullptr || gamma == nullptr || beta == nullptr || y == nullptr)
    return fail(FH_INVALID_ARGUMENT, "fh_layer_norm_rows: null pointer");
  hipStream_t s = static_cast<hipStream_t>(stream);
  switch (dtype) {
    case FH_F32:
      return layer_norm_typed<float>(x, gamma, beta, y, rows, cols, eps, s);
    case FH_BF16:
      return layer_norm_typed<bf16_t>(x, gamma, beta, y, rows, cols, eps, s);
    default:
      return layer_norm_typed<f16_t>(x, gamma, beta, y, rows, cols, eps, s);
  }
}
