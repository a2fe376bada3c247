// Dense GEMM for gfx950: C[M,N] = A[M,K] · B[K,N], row-major, fp32 accumulation: the dispatch between the MFMA kernels
// (fh_gemm16.hip, fh_gemm_any.hip, fh_gemm_f32.hip) and the kernels of small problems here.
//
// Semantics follow Frame's matmul (reference: src/backends/cpu/kernels/matmul.cpp:92-185): dtype in = out,
// products accumulated in fp32, one round-to-nearest-even store. The optional epilogue applies the
// elementwise segments Frame's graph would run next (bias add, ReLU, ...) on the rounded product before
// the single store, rounding between segments exactly like the unfused graph.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <string>
#include <type_traits>

#include "fh_common.h"
#include "fh_gemm.h"
#include "fh_gemm_any.h"

namespace fh {
namespace {

// Small GEMMs (few output tiles, or fewer columns than the tile kernels take): one thread per
// output of a 16 x 16 tile, its k loop strictly sequential like the reference CPU kernel (fp32 products and sums,
// no contraction, one rounding), so the result is bit-identical to it. K is staged through LDS in chunks of kKC as
// fp32, A row-major and B transposed, both k-contiguous so each step reads 4 k-values per operand with one
// 16-byte LDS read; the next chunk's global loads are in flight while the current one is consumed.
// WAYS > 1 (FH_GEMM_ANY_ORDER): WAYS such groups of 256 threads sum a WAYS-th of every chunk each, added in their order at
// the end. The chain of one sum, and the LDS latency before each 16 of its k, bound the kernel: 17 ns per k, 8 in four ways.
constexpr int kSeqT = 16;   // output tile edge
constexpr int kKC = 128;    // k per LDS chunk
constexpr int kKP = kKC + 4;  // padded row: 16 consecutive B rows hit distinct 16-byte bank groups

template <typename T, int WAYS>
__global__ __launch_bounds__(256 * WAYS) void gemm_seq_kernel(GemmArgs args) {
  using S = typename Io<T>::storage;
  __shared__ __attribute__((aligned(16))) float As[2][kSeqT * kKP];
  __shared__ __attribute__((aligned(16))) float Bt[2][kSeqT * kKP];
  const S* __restrict__ A = static_cast<const S*>(args.A) + blockIdx.z * args.stride_a;
  const S* __restrict__ B = static_cast<const S*>(args.B) + blockIdx.z * args.stride_b;
  S* __restrict__ C = static_cast<S*>(args.C) + blockIdx.z * args.stride_c;
  const int64_t m0 = static_cast<int64_t>(blockIdx.y) * kSeqT, n0 = static_cast<int64_t>(blockIdx.x) * kSeqT;
  const int64_t M = args.M, N = args.N, K = args.K;
  const int t = WAYS > 1 ? threadIdx.x & 255 : threadIdx.x;
  const int way = WAYS > 1 ? threadIdx.x >> 8 : 0;
  const int r = t >> 4, c = t & 15;

  // chunk loads: A[16][kKC] and B[kKC][16], each with consecutive lanes on the operand's contiguous index: k for
  // row-major A and transposed B (thread -> row / column t/16, k t%16 + 16 i), the row or column otherwise
  // (thread -> k t/16 + 16 i, row / column t%16)
  constexpr int U = 8 / WAYS;
  const int first = 16 * U * way;
  float la[U], lb[U];
  const bool ta = args.trans_a != 0, tb = args.trans_b != 0;
  auto load_chunk = [&](int64_t k0) {
#pragma unroll
    for (int i = 0; i < U; ++i) {
      const int64_t gm = m0 + (ta ? c : r), gk = k0 + first + (ta ? r : c) + 16 * i;
      la[i] = (gm < M && gk < K) ? Io<T>::load(A[ta ? gk * args.lda + gm : gm * args.lda + gk]) : 0.0f;
      const int64_t bk = k0 + first + (tb ? c : r) + 16 * i, bn = n0 + (tb ? r : c);
      lb[i] = (bk < K && bn < N) ? Io<T>::load(B[tb ? bn * args.ldb + bk : bk * args.ldb + bn]) : 0.0f;
    }
  };
  auto store_chunk = [&](int buf) {
#pragma unroll
    for (int i = 0; i < U; ++i) {
      const int k = first + 16 * i;
      As[buf][ta ? c * kKP + r + k : r * kKP + c + k] = la[i];
      Bt[buf][tb ? r * kKP + c + k : c * kKP + r + k] = lb[i];
    }
  };

  float acc = 0.0f;
  const int chunks = static_cast<int>((K + kKC - 1) / kKC);
  if (chunks > 0) {
    load_chunk(0);
    store_chunk(0);
  }
  __syncthreads();
  for (int ch = 0; ch < chunks; ++ch) {
    const int buf = ch & 1;
    if (ch + 1 < chunks) load_chunk(static_cast<int64_t>(ch + 1) * kKC);
    int kn = static_cast<int>(min<int64_t>(kKC, K - static_cast<int64_t>(ch) * kKC));
    if constexpr (WAYS > 1) kn = min(kn, (way + 1) * (kKC / WAYS));
    const float* ar = &As[buf][r * kKP];
    const float* br = &Bt[buf][c * kKP];
    int kk = way * (kKC / WAYS);
    // 16 k per step: the four LDS reads of each operand are issued before the sum uses them, so one LDS latency
    // covers 16 k instead of 4 (the sum itself is the same chain, in the same order)
    for (; kk + 16 <= kn; kk += 16) {
      float4 a[4], b[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        a[u] = *reinterpret_cast<const float4*>(ar + kk + 4 * u);
        b[u] = *reinterpret_cast<const float4*>(br + kk + 4 * u);
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        acc = acc + a[u].x * b[u].x;
        acc = acc + a[u].y * b[u].y;
        acc = acc + a[u].z * b[u].z;
        acc = acc + a[u].w * b[u].w;
      }
    }
    for (; kk + 4 <= kn; kk += 4) {
      const float4 a = *reinterpret_cast<const float4*>(ar + kk);
      const float4 b = *reinterpret_cast<const float4*>(br + kk);
      acc = acc + a.x * b.x;
      acc = acc + a.y * b.y;
      acc = acc + a.z * b.z;
      acc = acc + a.w * b.w;
    }
    for (; kk < kn; ++kk) acc = acc + ar[kk] * br[kk];
    if (ch + 1 < chunks) store_chunk(buf ^ 1);
    __syncthreads();
  }
  if constexpr (WAYS > 1) {  // (past the last chunk's barrier, or without a chunk, nothing else uses As)
    float* part = &As[0][0];
    static_assert((WAYS - 1) * 256 <= 2 * kSeqT * kKP, "the partial sums fit");
    if (way > 0) part[(way - 1) * 256 + t] = acc;
    __syncthreads();
    if (way > 0) return;
#pragma unroll
    for (int w = 0; w < WAYS - 1; ++w) acc = acc + part[w * 256 + t];
  }
  const int64_t row = m0 + r, col = n0 + c;
  if (row < M && col < N) {
    float v = Io<T>::round(acc);
    const int64_t idx = row * args.ldc + col;
    if (args.ep.nseg > 0) v = epilogue_one<T>(args.ep, v, idx);
    C[idx] = Io<T>::store(v);
  }
}

// Small GEMMs whose k-sum may be reassociated (FH_GEMM_ANY_ORDER): the sequential kernel's few 16 x 16 tiles leave
// most CUs idle, and each output's k loop is one long dependent chain. Here a workgroup of 16 waves owns a 4 x 16
// output tile (four times as many workgroups) and splits K 16 ways. K is staged through LDS as fp32 in chunks of
// up to kSplitKC = 1024 (A row-major, B transposed; every global load of a chunk in flight at once, so C1's layers
// pay one memory latency); within a chunk wave w sums its own contiguous sixteenth of the k, one output per lane,
// products and sums in fp32 without contraction like the sequential kernel. The 16 partial sums are then added in
// wave order: deterministic, and different from the sequential order by fp32 reassociation only. (Measured at
// C1's shapes on MI355X: 64x784x256 6.4 us and 64x256x10 3.4 us against 10.2 / 4.4 us with 4 waves and 16.3 /
// 6.1 us sequential; a launch of any kernel costs ~3 us there.)
// With row_softmax (N <= 16, so every output row lies in one workgroup), the rounded outputs of each row then
// go through softmax exactly as fh_softmax_rows computes it (m = max, e = exp(x - m), s = sum e, y = round(e / s);
// the sum taken over 16 lanes instead of 64).
constexpr int kSplitTM = 4, kSplitTN = 16, kSplitKC = 1024, kSplitKP = kSplitKC + 4, kSplitWaves = 16;

template <typename T>
__global__ __launch_bounds__(kSplitWaves * 64) void gemm_split_kernel(GemmArgs args) {
  using S = typename Io<T>::storage;
  __shared__ __attribute__((aligned(16))) float As[kSplitTM * kSplitKP];
  __shared__ __attribute__((aligned(16))) float Bt[kSplitTN * kSplitKP];
  __shared__ float part[kSplitWaves][kSplitTM * kSplitTN];
  constexpr int NT = kSplitWaves * 64;
  const S* __restrict__ A = static_cast<const S*>(args.A) + blockIdx.z * args.stride_a;
  const S* __restrict__ B = static_cast<const S*>(args.B) + blockIdx.z * args.stride_b;
  S* __restrict__ C = static_cast<S*>(args.C) + blockIdx.z * args.stride_c;
  const int64_t m0 = static_cast<int64_t>(blockIdx.y) * kSplitTM, n0 = static_cast<int64_t>(blockIdx.x) * kSplitTN;
  const int64_t M = args.M, N = args.N, K = args.K;
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int r = lane >> 4, c = lane & 15;  // this lane's output: (m0 + r, n0 + c)

  float acc = 0.0f;
  for (int64_t k0 = 0; k0 < K; k0 += kSplitKC) {
    const int kn = static_cast<int>(min<int64_t>(kSplitKC, K - k0));
    // every element of the chunk this thread stages is loaded into registers before the first is written to LDS,
    // so the loads overlap (a load-then-store loop waits for each load in turn)
    constexpr int AJ = kSplitTM * kSplitKC / NT, BJ = kSplitTN * kSplitKC / NT;
    static_assert(kSplitTM * kSplitKC % NT == 0 && kSplitTN * kSplitKC % NT == 0, "whole staging rounds");
    float av[AJ], bv[BJ];
#pragma unroll
    for (int j = 0; j < AJ; ++j) {
      const int i = t + j * NT, row = i / kSplitKC, kk = i - row * kSplitKC;
      av[j] = (kk < kn && m0 + row < M) ? Io<T>::load(A[(m0 + row) * args.lda + k0 + kk]) : 0.0f;
    }
#pragma unroll
    for (int j = 0; j < BJ; ++j) {
      const int i = t + j * NT, kk = i >> 4, cc = i & 15;
      bv[j] = (kk < kn && n0 + cc < N) ? Io<T>::load(B[(k0 + kk) * args.ldb + n0 + cc]) : 0.0f;
    }
    if (k0 > 0) __syncthreads();  // the previous chunk has been read
#pragma unroll
    for (int j = 0; j < AJ; ++j) {
      const int i = t + j * NT, row = i / kSplitKC, kk = i - row * kSplitKC;
      if (kk < kn) As[row * kSplitKP + kk] = av[j];
    }
#pragma unroll
    for (int j = 0; j < BJ; ++j) {
      const int i = t + j * NT, kk = i >> 4, cc = i & 15;
      if (kk < kn) Bt[cc * kSplitKP + kk] = bv[j];
    }
    __syncthreads();
    const int per = (kn + kSplitWaves - 1) / kSplitWaves;
    const int q0 = wave * per;
    const int qn = max(0, min(per, kn - q0));
    const float* ar = &As[r * kSplitKP + q0];
    const float* br = &Bt[c * kSplitKP + q0];
    for (int kk = 0; kk < qn; ++kk) acc = acc + ar[kk] * br[kk];
  }
  part[wave][lane] = acc;
  __syncthreads();
  if (t < kSplitTM * kSplitTN) {
    const int64_t row = m0 + (t >> 4), col = n0 + (t & 15);
    const bool live = row < M && col < N;
    float sum = part[0][t];
#pragma unroll
    for (int w = 1; w < kSplitWaves; ++w) sum = sum + part[w][t];
    float v = Io<T>::round(sum);
    const int64_t idx = row * args.ldc + col;
    if (live && args.ep.nseg > 0) v = epilogue_one<T>(args.ep, v, idx);
    if (args.row_softmax) {  // N <= 16: the row's outputs are the 16 lanes of this lane's group
      float m = live ? v : -__builtin_inff();
#pragma unroll
      for (int o = 8; o > 0; o >>= 1) {
        const float other = __shfl_xor(m, o, 16);
        m = (other > m) ? other : m;
      }
      const float e = live ? expf(v - m) : 0.0f;
      float s = e;
#pragma unroll
      for (int o = 8; o > 0; o >>= 1) s += __shfl_xor(s, o, 16);
      v = e / s;
    }
    if (live) C[idx] = Io<T>::store(v);
  }
}

template <typename T>
fh_status dispatch_gemm(GemmArgs args, int64_t batch, hipStream_t stream) {
  using S = typename Io<T>::storage;
  const int cus = device_cu_count();
  // Few 64 x 64 tiles: the sequential kernel, whose 16 x 16 tiles spread further and whose latency is a handful
  // of K chunks. fp32 below a quarter of the CUs; 16-bit only below 16 tiles (its MFMA kernel stays faster down
  // to there: the C4 classifier, 16 tiles, 7.8 us there against 22 us sequential).
  const int64_t tiles64 = ((args.M + 63) / 64) * ((args.N + 63) / 64) * batch;
  const bool small = (std::is_same_v<T, float> ? tiles64 * 4 < cus : tiles64 < 16) && args.K <= 16384;
  // A transposed operand in any order: the sequential kernel takes 3 us + 35 ns per k in 16 bits, the MFMA kernels 3.5 us +
  // 10 ns per k on few tiles (64x512x1000 bf16, B transposed: 40 us against 14). In fp32 it takes 17 ns per k, 8 in four
  // ways, while the planes' tiles take 23 with A transposed and 14 with B (256x1000x10 18.3 / 10.7 / 27.1 us, 17x3000x1000
  // 53 / 28 / 70). With more than two workgroups per CU the tiles are ahead for B transposed, with more than three for A and k
  // from 256 on (500x1000x400 32 us in four ways, 27 on tiles); till then two ways are (500x200x400 8.4 in order, 8.8, 9.5;
  // 40x384x3974 12.0, 11.5, 13.2). The sums in ways are closer to the exact ones than those in order: 500x128x400 1.5e-7
  // (2.1e-7), 256x3000x10 5.0e-7 (9.5e-7).
  const bool long_k = args.any_order && (args.trans_a || args.trans_b) && args.K >= 128;
  const double outputs16 = static_cast<double>((args.M + 15) / 16) * static_cast<double>((args.N + 15) / 16) * batch;
  const bool full = args.trans_b ? outputs16 > 2 * cus : outputs16 > 3 * cus && args.K >= 256;
  const bool planes = long_k && (!std::is_same_v<T, float> || full);
  // 16-bit operands that are not whole vectors and little work: the sequential kernel takes 3 us + 20 ns per k + (0.3 us + 5
  // ns per k) for every 65,536 outputs, an MFMA tile of any alignment 4.3-5 us at the least (bf16 2001x20x101 3.7 us against
  // 5.1, 4001x33x47 4.3 / 5.4, 600x33x333 4.2 / 4.7; past the line 1501x64x131 4.9 / 4.4, 511x63x513 7.2 / 5.0, 300x264x200
  // 9.6 / 5.5). fp32 stays on the planes, which are closer to the exact sum than fp32 sums in order are.
  const double outputs = static_cast<double>(args.M) * static_cast<double>((args.N + 15) / 16 * 16) * batch;
  const bool little = !std::is_same_v<T, float> && !args.trans_a && !args.trans_b && args.K <= 64 &&
                      outputs / 65536 * (0.3 + 0.005 * static_cast<double>(args.K)) <= 1.7;
  // everything else on the matrix cores: 16-bit operands of whole 16-byte vectors on the aligned pipeline, the rest on
  // the kernel of any alignment (8 columns or more, 8 rows of a transposed A)
  fh_status st = FH_OK;
  if ((!small || planes) && !args.row_softmax) {
    if constexpr (std::is_same_v<T, float>) {
      if (gemm_f32_try_launch(args, batch, stream, &st)) return st;
    } else {
      const int32_t dtype = std::is_same_v<T, bf16_t> ? FH_BF16 : FH_F16;
      if (!args.trans_a && !args.trans_b && gemm16_try_launch(dtype, args, batch, stream, &st)) return st;
      if (!little && gemm_any16_try_launch(dtype, args, batch, stream, &st)) return st;
    }
  }
  const bool split_ok = args.any_order && !args.trans_a && !args.trans_b &&
                        (args.M + kSplitTM - 1) / kSplitTM <= 65535 && batch <= 65535;
  if (args.row_softmax && (!split_ok || args.N > kSplitTN))
    return fail(FH_INVALID_ARGUMENT, "fh_gemm_ex: FH_GEMM_ROW_SOFTMAX needs FH_GEMM_ANY_ORDER, N <= 16 and at most "
                                     "262,140 rows");
  if ((small || args.row_softmax) && split_ok) {
    dim3 grid(static_cast<uint32_t>((args.N + kSplitTN - 1) / kSplitTN),
              static_cast<uint32_t>((args.M + kSplitTM - 1) / kSplitTM), static_cast<uint32_t>(batch));
    hipLaunchKernelGGL((gemm_split_kernel<T>), grid, dim3(kSplitWaves * 64), 0, stream, args);
    return launch_status("gemm_split_kernel launch");
  }
  // small problems, and the few that no MFMA kernel takes (N below 8, or a transposed A with M below 8), in launches of as
  // many rows as a grid's y holds. fp32 of 4 columns is faster here than on MFMA tiles of 64: 65536x512x4 57 us against 140.
  constexpr int64_t kRows = int64_t{65535} * kSeqT;
  for (int64_t m0 = 0; m0 < args.M; m0 += kRows) {
    GemmArgs part = args;
    part.M = std::min(kRows, args.M - m0);
    part.A = static_cast<const S*>(args.A) + m0 * (args.trans_a ? 1 : args.lda);
    part.C = static_cast<S*>(args.C) + m0 * args.ldc;
    for (int s = 0; s < args.ep.nseg; ++s)
      if (ew_is_binary(args.ep.ops[s])) part.ep.ins[s] = static_cast<const S*>(args.ep.ins[s]) + m0 * args.ldc;
    const dim3 grid(static_cast<uint32_t>((part.N + kSeqT - 1) / kSeqT),
                    static_cast<uint32_t>((part.M + kSeqT - 1) / kSeqT), static_cast<uint32_t>(batch));
    if constexpr (std::is_same_v<T, float>) {
      if (long_k && outputs16 <= 2 * cus) hipLaunchKernelGGL((gemm_seq_kernel<T, 4>), grid, dim3(1024), 0, stream, part);
      else if (long_k) hipLaunchKernelGGL((gemm_seq_kernel<T, 2>), grid, dim3(512), 0, stream, part);
      else hipLaunchKernelGGL((gemm_seq_kernel<T, 1>), grid, dim3(256), 0, stream, part);
    } else {
      hipLaunchKernelGGL((gemm_seq_kernel<T, 1>), grid, dim3(256), 0, stream, part);
    }
    st = launch_status("gemm_seq_kernel launch");
    if (st != FH_OK) break;
  }
  return st;
}

fh_status run_gemm(int32_t dtype, GemmArgs args, int64_t batch, hipStream_t stream) {
  switch (dtype) {
    case FH_F32:
      return dispatch_gemm<float>(args, batch, stream);
    case FH_BF16:
      return dispatch_gemm<bf16_t>(args, batch, stream);
    case FH_F16:
      return dispatch_gemm<f16_t>(args, batch, stream);
    default:
      return fail(FH_UNIMPLEMENTED, "fh_gemm: unsupported dtype code " + std::to_string(dtype));
  }
}

fh_status copy_epilogue(const fh_epilogue* in, EpilogueArgs& out) {
  out = EpilogueArgs{};
  if (in == nullptr) return FH_OK;
  if (in->nseg < 0 || in->nseg > FH_MAX_SEGMENTS)
    return fail(FH_INVALID_ARGUMENT, "epilogue: nseg out of range: " + std::to_string(in->nseg));
  out.nseg = in->nseg;
  out.round_between = in->round_between;
  for (int s = 0; s < in->nseg; ++s) {
    const uint8_t op = in->ops[s];
    if (!epilogue_op_ok(op))
      return fail(FH_INVALID_ARGUMENT, "epilogue: unknown op code " + std::to_string(op));
    if (ew_is_binary(op) && in->ins[s] == nullptr)
      return fail(FH_INVALID_ARGUMENT, "epilogue: binary segment " + std::to_string(s) + " has no operand");
    out.ops[s] = op;
    out.ins[s] = in->ins[s];
  }
  return FH_OK;
}

}  // namespace

fh_status gemm_with_epilogue_args(int32_t dtype, const void* A, const void* B, void* C, int64_t M, int64_t N,
                                  int64_t K, const fh_epilogue* epilogue, hipStream_t stream, int32_t flags,
                                  int32_t transposed = 0) {
  if ((flags & ~(FH_GEMM_ANY_ORDER | FH_GEMM_ROW_SOFTMAX)) != 0)
    return fail(FH_INVALID_ARGUMENT, "fh_gemm_ex: unknown flags " + std::to_string(flags));
  if (!is_supported_float(dtype)) return fail(FH_UNIMPLEMENTED, "fh_gemm: unsupported dtype");
  if (M < 0 || N < 0 || K < 0) return fail(FH_INVALID_ARGUMENT, "fh_gemm: negative dimension");
  if (M == 0 || N == 0) return FH_OK;
  if (A == nullptr || B == nullptr || C == nullptr) {
    if (K > 0 || C == nullptr) return fail(FH_INVALID_ARGUMENT, "fh_gemm: null operand");
  }
  GemmArgs args{};
  args.A = A;
  args.B = B;
  args.C = C;
  args.M = M;
  args.N = N;
  args.K = K;
  args.trans_a = transposed == 1;
  args.trans_b = transposed == 2;
  args.lda = args.trans_a ? M : K;
  args.ldb = args.trans_b ? K : N;
  args.ldc = N;
  args.any_order = (flags & FH_GEMM_ANY_ORDER) != 0;
  args.row_softmax = (flags & FH_GEMM_ROW_SOFTMAX) != 0;
  fh_status st = copy_epilogue(epilogue, args.ep);
  if (st != FH_OK) return st;
  return run_gemm(dtype, args, 1, stream);
}

}  // namespace fh

extern "C" fh_status fh_gemm_ex(int32_t dtype, const void* A, const void* B, void* C, int64_t M, int64_t N, int64_t K,
                                const fh_epilogue* epilogue, int32_t flags, void* stream) {
  return fh::gemm_with_epilogue_args(dtype, A, B, C, M, N, K, epilogue, static_cast<hipStream_t>(stream), flags);
}

extern "C" fh_status fh_gemm_transposed(int32_t dtype, int32_t transposed, const void* A, const void* B, void* C,
                                        int64_t M, int64_t N, int64_t K, const fh_epilogue* epilogue, int32_t flags,
                                        void* stream) {
  using namespace fh;
  if (transposed != 1 && transposed != 2)
    return fail(FH_INVALID_ARGUMENT, "fh_gemm_transposed: transposed must be 1 (A) or 2 (B)");
  if ((flags & FH_GEMM_ROW_SOFTMAX) != 0) return fail(FH_INVALID_ARGUMENT, "fh_gemm_transposed: no row softmax");
  return gemm_with_epilogue_args(dtype, A, B, C, M, N, K, epilogue, static_cast<hipStream_t>(stream), flags, transposed);
}

extern "C" fh_status fh_gemm_grouped(int32_t dtype, const void* A, int32_t groups, const void* const* B, void* const* C,
                                     int64_t M, int64_t N, int64_t K, const fh_epilogue* epilogues, int32_t flags,
                                     void* stream) {
  using namespace fh;
  if (groups < 1 || groups > kGemmMaxGroups)
    return fail(FH_INVALID_ARGUMENT, "fh_gemm_grouped: groups must be in [1, " + std::to_string(kGemmMaxGroups) + "]");
  if (B == nullptr || C == nullptr) return fail(FH_INVALID_ARGUMENT, "fh_gemm_grouped: null operand arrays");
  if ((flags & ~FH_GEMM_ANY_ORDER) != 0) return fail(FH_INVALID_ARGUMENT, "fh_gemm_grouped: unknown flags");
  // every group must carry the same epilogue program (one kernel instance serves them all)
  for (int g = 1; g < groups && epilogues != nullptr; ++g) {
    if (epilogues[g].nseg != epilogues[0].nseg || epilogues[g].round_between != epilogues[0].round_between)
      return fail(FH_INVALID_ARGUMENT, "fh_gemm_grouped: groups with different epilogue programs");
    for (int s = 0; s < epilogues[0].nseg && s < FH_MAX_SEGMENTS; ++s)
      if (epilogues[g].ops[s] != epilogues[0].ops[s])
        return fail(FH_INVALID_ARGUMENT, "fh_gemm_grouped: groups with different epilogue programs");
  }
  hipStream_t s = static_cast<hipStream_t>(stream);
  const bool sixteen = dtype == FH_BF16 || dtype == FH_F16;
  if (sixteen && M > 0 && N > 0 && K > 0 && A != nullptr) {
    GemmArgs args{};
    args.A = A;
    args.B = B[0];
    args.C = C[0];
    args.M = M;
    args.N = N;
    args.K = K;
    args.lda = K;
    args.ldb = N;
    args.ldc = N;
    args.any_order = (flags & FH_GEMM_ANY_ORDER) != 0;
    fh_status st = copy_epilogue(epilogues, args.ep);
    if (st != FH_OK) return st;
    args.groups = groups;
    for (int g = 0; g < groups; ++g) {
      if (B[g] == nullptr || C[g] == nullptr) return fail(FH_INVALID_ARGUMENT, "fh_gemm_grouped: null operand");
      args.group_b[g] = B[g];
      args.group_c[g] = C[g];
      EpilogueArgs eg{};
      if (epilogues != nullptr && (st = copy_epilogue(&epilogues[g], eg)) != FH_OK) return st;
      for (int sg = 0; sg < FH_MAX_SEGMENTS; ++sg) args.group_ins[g][sg] = eg.ins[sg];
    }
    // the MFMA kernel takes the groups as its second grid axis when the problem is one it accepts and is not small
    const int64_t tiles64 = ((M + 63) / 64) * ((N + 63) / 64) * groups;
    if (tiles64 >= 16 && gemm16_try_launch(dtype, args, groups, s, &st)) return st;
  }
  // otherwise: one GEMM per group
  for (int g = 0; g < groups; ++g) {
    const fh_status st = fh_gemm_ex(dtype, A, B[g], C[g], M, N, K, epilogues != nullptr ? &epilogues[g] : nullptr,
                                    flags, stream);
    if (st != FH_OK) return st;
  }
  return FH_OK;
}

extern "C" fh_status fh_gemm(int32_t dtype, const void* A, const void* B, void* C, int64_t M, int64_t N,
                             int64_t K, const fh_epilogue* epilogue, void* stream) {
  return fh::gemm_with_epilogue_args(dtype, A, B, C, M, N, K, epilogue, static_cast<hipStream_t>(stream), 0);
}

extern "C" fh_status fh_gemm_batched(int32_t dtype, const void* A, const void* B, void* C, int64_t M,
                                     int64_t N, int64_t K, int64_t lda, int64_t ldb, int64_t ldc,
                                     int64_t stride_a, int64_t stride_b, int64_t stride_c, int64_t batch,
                                     void* stream) {
  using namespace fh;
  if (!is_supported_float(dtype)) return fail(FH_UNIMPLEMENTED, "fh_gemm_batched: unsupported dtype");
  if (M < 0 || N < 0 || K < 0 || batch < 0)
    return fail(FH_INVALID_ARGUMENT, "fh_gemm_batched: negative dimension");
  if (M == 0 || N == 0 || batch == 0) return FH_OK;
  if (lda < K || ldb < N || ldc < N)
    return fail(FH_INVALID_ARGUMENT, "fh_gemm_batched: leading dimension smaller than the row width");
  if (batch > 65535) return fail(FH_INVALID_ARGUMENT, "fh_gemm_batched: batch above 65535");
  GemmArgs args{};
  args.A = A;
  args.B = B;
  args.C = C;
  args.M = M;
  args.N = N;
  args.K = K;
  args.lda = lda;
  args.ldb = ldb;
  args.ldc = ldc;
  args.stride_a = stride_a;
  args.stride_b = stride_b;
  args.stride_c = stride_c;
  return run_gemm(dtype, args, batch, static_cast<hipStream_t>(stream));
}

// matmul_grad_lhs_internal (rhs = 0): out [m,k] = gy [m,n] * b[k,n]^T; matmul_grad_rhs_internal (rhs = 1):
// out [k,n] = a[m,k]^T * gy [m,n]. The sequential kernel reads the transposed operand in place, so every output is
// one fp32 sum over the contraction index in ascending order (reference: src/backends/cpu/kernels/matmul.cpp:187-327).
extern "C" fh_status fh_matmul_grad(int32_t dtype, int32_t rhs, const void* p, const void* q, void* out, int64_t m,
                                    int64_t n, int64_t k, void* stream) {
  using namespace fh;
  if (!is_supported_float(dtype)) return fail(FH_UNIMPLEMENTED, "fh_matmul_grad: unsupported dtype");
  if (m < 0 || n < 0 || k < 0) return fail(FH_INVALID_ARGUMENT, "fh_matmul_grad: negative dimension");
  GemmArgs args{};
  if (rhs == 0) {  // A = gy [m,n] (contraction n), B(j, c) = b[c * n + j]
    args.A = p, args.B = q, args.M = m, args.N = k, args.K = n, args.lda = n, args.ldb = n, args.ldc = k;
    args.trans_b = 1;
  } else {  // A(c, i) = a[i * k + c], B = gy [m,n] (contraction m)
    args.A = p, args.B = q, args.M = k, args.N = n, args.K = m, args.lda = k, args.ldb = n, args.ldc = n;
    args.trans_a = 1;
  }
  args.C = out;
  if (args.M == 0 || args.N == 0) return FH_OK;
  if (p == nullptr || q == nullptr || out == nullptr) return fail(FH_INVALID_ARGUMENT, "fh_matmul_grad: null pointer");
  if ((args.M + kSeqT - 1) / kSeqT > 65535) return fail(FH_UNIMPLEMENTED, "fh_matmul_grad: more than 1,048,560 rows");
  const dim3 grid(static_cast<uint32_t>((args.N + kSeqT - 1) / kSeqT), static_cast<uint32_t>((args.M + kSeqT - 1) / kSeqT), 1);
  hipStream_t s = static_cast<hipStream_t>(stream);
  switch (dtype) {
    case FH_F32:
      hipLaunchKernelGGL((gemm_seq_kernel<float, 1>), grid, dim3(256), 0, s, args);
      break;
    case FH_BF16:
      hipLaunchKernelGGL((gemm_seq_kernel<bf16_t, 1>), grid, dim3(256), 0, s, args);
      break;
    default:
      hipLaunchKernelGGL((gemm_seq_kernel<f16_t, 1>), grid, dim3(256), 0, s, args);
      break;
  }
  return launch_status("fh_matmul_grad");
}
