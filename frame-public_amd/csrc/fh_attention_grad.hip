// Gradients of the fused attention (fh_attention_grad), with the roundings of the per-(batch, head) gradient graph:
//   P = softmax(round(round(Q K^T) scale)), dP = dO V^T, s = sum_keys round(P dP),
//   dS = round(round(P round(dP - s)) scale), dQ = dS K, dK = dS^T Q, dV = P^T dO,
// every product and sum rounded to the storage type as the graph stores it.
//
// attention_scores_grad_kernel computes P and dS: one wave owns 16 queries and all keys, its scores in registers as 16x16
// MFMA tiles (a row's keys lie in the 16 lanes of a group, so the row sums are shuffles); Q, K, V and dO fragments are 16
// contiguous bytes of a head's row and are read from memory in the MFMA layout, with no LDS. P and dS go to a workspace,
// staged through LDS for 16-byte stores. dQ, dK and dV are then batched GEMMs over the heads in place (fh_gemm_any.h, the
// transposed operand read as it is stored). Four launches replace about 20 per head (1,250 -> 305 us for the training step of
// a 2 x 128-token block with 4 heads): what bounds it at that size is the latency of each, 5-8 us.
#include <hip/hip_runtime.h>

#include <string>

#include "fh_gemm_any.h"

namespace fh {
namespace {

using namespace mfma16;

__device__ __forceinline__ float group_max(float v) {  // over the 16 lanes of a group
#pragma unroll
  for (int o = 8; o > 0; o >>= 1) {
    const float other = __shfl_xor(v, o, 64);
    v = (other > v) ? other : v;
  }
  return v;
}
__device__ __forceinline__ float group_sum(float v) {
#pragma unroll
  for (int o = 8; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}

// NT: key tiles of 16. Grid: (seq / 16, heads, batch), one wave each.
template <typename T, int NT>
__global__ __launch_bounds__(64) void attention_scores_grad_kernel(const uint16_t* __restrict__ q,
                                                                   const uint16_t* __restrict__ k,
                                                                   const uint16_t* __restrict__ v,
                                                                   const uint16_t* __restrict__ dout,
                                                                   uint16_t* __restrict__ probs,
                                                                   uint16_t* __restrict__ dscores, int heads, float scale) {
  constexpr int SEQ = 16 * NT, PITCH = SEQ + 8;
  __shared__ __attribute__((aligned(16))) uint16_t rows[16 * PITCH];
  const int lane = threadIdx.x, r = lane & 15, g = lane >> 4;
  const int h = blockIdx.y, b = blockIdx.z;
  const int64_t ld = static_cast<int64_t>(heads) * 64;
  const int64_t head = static_cast<int64_t>(b) * SEQ * ld + h * 64;
  const int q0 = blockIdx.x * 16;

  // fragment s (dims 32 s .. + 31) of 16 rows from `row` on: lane l holds row l % 16, dims 32 s + 8 (l / 16) .. + 7
  auto fragment = [&](const uint16_t* base, int row, int s) {
    return *reinterpret_cast<const u32x4_t*>(base + head + (row + r) * ld + 32 * s + 8 * g);
  };
  auto tile = [&](const u32x4_t (&a)[2], const uint16_t* base, int n) {
    f32x4_t acc{0.0f, 0.0f, 0.0f, 0.0f};
    mfma16x<T>(a[0], fragment(base, 16 * n, 0), acc);
    mfma16x<T>(a[1], fragment(base, 16 * n, 1), acc);
    return acc;
  };
  const u32x4_t qf[2] = {fragment(q, q0, 0), fragment(q, q0, 1)};
  const u32x4_t of[2] = {fragment(dout, q0, 0), fragment(dout, q0, 1)};

  // scores, scaled; lane: queries 4 g + x, key 16 n + r
  f32x4_t s[NT];
#pragma unroll
  for (int n = 0; n < NT; ++n) {
    s[n] = tile(qf, k, n);
#pragma unroll
    for (int x = 0; x < 4; ++x) s[n][x] = Io<T>::round(Io<T>::round(s[n][x]) * scale);
  }
  float m[4], sum[4];
#pragma unroll
  for (int x = 0; x < 4; ++x) {
    m[x] = -__builtin_inff();
#pragma unroll
    for (int n = 0; n < NT; ++n) m[x] = (s[n][x] > m[x]) ? s[n][x] : m[x];
    m[x] = group_max(m[x]);
    sum[x] = 0.0f;
#pragma unroll
    for (int n = 0; n < NT; ++n) {
      s[n][x] = __builtin_amdgcn_exp2f((s[n][x] - m[x]) * 1.44269504088896340736f);
      sum[x] += s[n][x];
    }
    sum[x] = 1.0f / group_sum(sum[x]);
  }
  uint32_t p[NT][2];  // packed probabilities of queries (0, 1) and (2, 3)
#pragma unroll
  for (int n = 0; n < NT; ++n) {
    p[n][0] = store2<T>(s[n][0] * sum[0], s[n][1] * sum[1]);
    p[n][1] = store2<T>(s[n][2] * sum[2], s[n][3] * sum[3]);
  }
  auto prob = [&](int n, int x) { return x % 2 ? load_hi<T>(p[n][x / 2]) : load_lo<T>(p[n][x / 2]); };

  // the 16 x SEQ tile of `value(n, x)` bits to its place in a [batch, heads, SEQ, SEQ] tensor
  auto write = [&](uint16_t* out, auto&& value) {
#pragma unroll
    for (int n = 0; n < NT; ++n)
#pragma unroll
      for (int x = 0; x < 4; ++x) rows[(4 * g + x) * PITCH + 16 * n + r] = value(n, x);
    __syncthreads();
    uint16_t* dst = out + ((static_cast<int64_t>(b) * heads + h) * SEQ + q0) * SEQ;
#pragma unroll
    for (int i = lane; i < 16 * (SEQ / 8); i += 64) {
      const int row = i / (SEQ / 8), c = i % (SEQ / 8) * 8;
      *reinterpret_cast<u32x4_t*>(dst + row * SEQ + c) = *reinterpret_cast<const u32x4_t*>(rows + row * PITCH + c);
    }
    __syncthreads();
  };
  write(probs, [&](int n, int x) { return static_cast<uint16_t>(x % 2 ? p[n][x / 2] >> 16 : p[n][x / 2] & 0xffffu); });

  // dP in the scores' registers, then dS
  float dot[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int n = 0; n < NT; ++n) {
    s[n] = tile(of, v, n);
#pragma unroll
    for (int x = 0; x < 4; ++x) {
      s[n][x] = Io<T>::round(s[n][x]);
      dot[x] += Io<T>::round(prob(n, x) * s[n][x]);
    }
  }
#pragma unroll
  for (int x = 0; x < 4; ++x) dot[x] = Io<T>::round(group_sum(dot[x]));
  write(dscores, [&](int n, int x) {
    return Io<T>::store(Io<T>::round(prob(n, x) * Io<T>::round(s[n][x] - dot[x])) * scale);
  });
}

template <typename T>
fh_status launch_scores(const void* q, const void* k, const void* v, const void* dout, void* probs, void* ds, int64_t batch,
                        int64_t seq, int64_t heads, float scale, hipStream_t stream) {
  const dim3 grid(static_cast<uint32_t>(seq / 16), static_cast<uint32_t>(heads), static_cast<uint32_t>(batch));
  auto go = [&]<int NT>() {
    hipLaunchKernelGGL((attention_scores_grad_kernel<T, NT>), grid, dim3(64), 0, stream, static_cast<const uint16_t*>(q),
                       static_cast<const uint16_t*>(k), static_cast<const uint16_t*>(v), static_cast<const uint16_t*>(dout),
                       static_cast<uint16_t*>(probs), static_cast<uint16_t*>(ds), static_cast<int>(heads), scale);
    return launch_status("attention_scores_grad_kernel launch");
  };
  switch (seq / 64) {
    case 1: return go.template operator()<4>();
    case 2: return go.template operator()<8>();
    case 3: return go.template operator()<12>();
    case 4: return go.template operator()<16>();
    case 5: return go.template operator()<20>();
    case 6: return go.template operator()<24>();
    case 7: return go.template operator()<28>();
    default: return go.template operator()<32>();
  }
}

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

}  // namespace
}  // namespace fh

using namespace fh;

extern "C" int64_t fh_attention_grad_workspace(int64_t batch, int64_t seq, int64_t heads) {
  return 2 * 2 * batch * heads * seq * seq;
}

extern "C" fh_status fh_attention_grad(int32_t dtype, const void* q, const void* k, const void* v, const void* dout, void* dq,
                                       void* dk, void* dv, void* workspace, int64_t workspace_bytes, int64_t batch,
                                       int64_t seq, int64_t heads, int64_t dh, float scale, void* stream) {
  if (!fh_attention_supported(dtype, seq, dh))
    return fail(FH_UNIMPLEMENTED, "fh_attention_grad: needs bf16/f16, head dim 64, seq a multiple of 64 up to 512");
  if (batch < 0 || heads < 1 || batch > 65535 || heads > 65535 || batch * heads > 65535)
    return fail(FH_INVALID_ARGUMENT, "fh_attention_grad: bad batch/heads");
  if (batch == 0) return FH_OK;
  for (const void* p : {q, k, v, dout, static_cast<const void*>(dq), static_cast<const void*>(dk),
                        static_cast<const void*>(dv), static_cast<const void*>(workspace)})
    if (p == nullptr || !aligned16(p)) return fail(FH_INVALID_ARGUMENT, "fh_attention_grad: null or unaligned pointer");
  if (workspace_bytes < fh_attention_grad_workspace(batch, seq, heads))
    return fail(FH_INVALID_ARGUMENT, "fh_attention_grad: workspace too small");
  hipStream_t s = static_cast<hipStream_t>(stream);
  const int64_t plane = seq * seq;
  uint16_t* probs = static_cast<uint16_t*>(workspace);
  uint16_t* ds = probs + batch * heads * plane;
  fh_status st = dtype == FH_BF16 ? launch_scores<bf16_t>(q, k, v, dout, probs, ds, batch, seq, heads, scale, s)
                                  : launch_scores<f16_t>(q, k, v, dout, probs, ds, batch, seq, heads, scale, s);
  if (st != FH_OK) return st;
  // per head [seq, 64] = op([seq, seq]) [seq, 64], the heads' columns inside rows of heads * 64
  auto gemm = [&](const uint16_t* a, bool transposed, const void* b, void* c) {
    GemmArgs args{};
    args.A = a, args.B = b, args.C = c;
    args.M = seq, args.N = dh, args.K = seq;
    args.lda = seq, args.ldb = args.ldc = heads * dh;
    args.stride_a = heads * plane, args.stride_b = args.stride_c = seq * heads * dh;
    args.inner = heads, args.inner_a = plane, args.inner_b = args.inner_c = dh;
    args.trans_a = transposed;
    fh_status launched = FH_OK;
    if (!gemm_any16_try_launch(dtype, args, batch * heads, s, &launched))
      return fail(FH_INTERNAL, "fh_attention_grad: the GEMM kernel refused the shape");
    return launched;
  };
  if ((st = gemm(ds, false, k, dq)) != FH_OK) return st;
  if ((st = gemm(ds, true, q, dk)) != FH_OK) return st;
  return gemm(probs, true, dout, dv);
}
