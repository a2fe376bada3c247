// GEMM of any alignment, either operand transposed, for 16-bit and fp32 operands, of any size but the narrowest (an operand
// contiguous along m or n needs 8 of them, see accepts): C = op(A) · op(B) with fp32 accumulation on v_mfma_f32_16x16x32,
// one rounding per output, then the optional elementwise epilogue (semantics of Frame's matmul and its gradients: reference
// src/backends/cpu/kernels/matmul.cpp:92-327). The kernel template; its instances and their dispatch are in
// fh_gemm_any.hip (16-bit) and fh_gemm_f32.hip (fp32).
//
// Operands go global -> registers -> LDS in units of 8 elements along their contiguous index, so a unit needs element
// alignment only (global memory takes 16-byte accesses at any alignment) and edges are handled per unit: rows past the
// edge are clamped to the last valid one (their products land in discarded outputs), and in the last k tile the units past
// K are zeroed on their way to LDS; element by element goes only the unit that ends the operand, or a row's k, inside its 8
// (1024x40x1024 bf16 4.4 us, 6.0 with that tile loaded element by element throughout). Two register sets and two LDS
// buffers: the loads of tile k+2 and the LDS writes of tile k+1 are issued around the products of tile k, with one barrier
// per tile.
//
// An operand that is contiguous along k (A as stored, B transposed) lies in LDS as rows of 32 k and is read with
// ds_read_b128; one that is contiguous along m or n (A transposed, B as stored) lies as 32 k rows and is read with the
// LDS transpose read ds_read_b64_tr_b16: neither needs a transposed copy.
//
// fp32 operands are scaled by 2^24 and split on their way to LDS into three bf16 planes, 2^24 x = x1 + x2 + x3 (each the
// round-to-nearest bf16 of what the ones before it leave: all 24 bits of every |x| < 2^104, denormals included, in planes
// that are no denormals themselves); the sum is scaled back by 2^-48. A product is the eight plane products
// x1 y1 + x1 y2 + x2 y1 + x2 y2 + x1 y3 + x3 y1 + x2 y3 + x3 y2. With |x2| <= 2^-8 and |x3| <= 2^-17 of x's power of two,
// the one left out is at most 2^-34 of |x y|; without the last two it would be 2^-24, as much again as a product's own
// rounding (and of one sign where an operand repeats). The instruction does not round to nearest when it adds to its
// accumulator, so x1 y1, whose 16 bits rarely meet the end of the sum, has an accumulator of its own and the small terms
// another, added up once. Error against float64 (fp32 MFMA before; one accumulator and six products): N(0,1), K 4096
// 4.0e-7 (1.1e-6; 1.0e-6 with a bias of -2.7e-7), U(0,1), K 4096 3.0e-7 (8.5e-7; 5.3e-7), U(-1,1), K 1 2.5e-8 (2.5e-8;
// 3.1e-8), equal operands, K 4096 5.9e-8 (5.9e-8; 3.8e-6). The bf16 matrix rate is 16 times the fp32 one, so
// eight products take half of the time (2048^3: 109 us; 92 with six in one accumulator, 187 on fp32 MFMA). Infinities,
// NaN, operands of 2^104 or more and sums of 2^80 or more make the accumulators non-finite: those outputs, and no others, are
// taken again on fp32 MFMA after the loop (one NaN in an operand of 2048^3: 276 us).
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>
#include <utility>

#include "fh_common.h"
#include "fh_gemm.h"
#include "fh_mfma16.h"

namespace fh {
namespace gemm_any {

using namespace mfma16;

typedef u32x4_t u32x4_any __attribute__((aligned(2)));
typedef short s16x4_t __attribute__((ext_vector_type(4)));

template <typename T>
struct AnyTraits {
  static constexpr int P = 1;  // planes in LDS
  static constexpr int Q = 1;  // accumulators per output
  using mfma_t = T;
};
template <>
struct AnyTraits<float> {
  static constexpr int P = 3;
  static constexpr int Q = 2;  // x1 y1, and the small terms
  using mfma_t = bf16_t;
};

// Eight consecutive elements as loaded.
template <typename T>
struct Unit {
  static constexpr int R = sizeof(typename Io<T>::storage) / 2;  // 16-byte registers
  u32x4_t v[R];
};

template <typename T>
__device__ __forceinline__ Unit<T> load_unit(const typename Io<T>::storage* p) {
  Unit<T> u;
#pragma unroll
  for (int i = 0; i < Unit<T>::R; ++i) u.v[i] = *(reinterpret_cast<const u32x4_any*>(p) + i);
  return u;
}

// Element e of the unit at p when it is one of the first n, zero otherwise.
template <typename T>
__device__ __forceinline__ Unit<T> load_unit_partial(const typename Io<T>::storage* p, int n) {
  typename Io<T>::storage e[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) e[i] = 0;
#pragma unroll
  for (int i = 0; i < 8; ++i)
    if (i < n) e[i] = p[i];
  Unit<T> u;
  __builtin_memcpy(&u, e, sizeof(u));
  return u;
}

constexpr float kSplitScale = 0x1p24f, kSplitUnscale = 0x1p-48f;

// The unit's planes as packed 16-bit vectors.
template <typename T>
__device__ __forceinline__ void split_unit(const Unit<T>& u, u32x4_t (&plane)[AnyTraits<T>::P]) {
  if constexpr (std::is_same_v<T, float>) {
#pragma unroll
    for (int d = 0; d < 4; ++d) {
      float x0 = __uint_as_float(u.v[d / 2][2 * (d % 2)]) * kSplitScale;
      float x1 = __uint_as_float(u.v[d / 2][2 * (d % 2) + 1]) * kSplitScale;
#pragma unroll
      for (int p = 0; p < 3; ++p) {
        const uint32_t w = store2<bf16_t>(x0, x1);
        plane[p][d] = w;
        x0 -= __uint_as_float(w << 16);
        x1 -= __uint_as_float(w & 0xffff0000u);
      }
    }
  } else {
    plane[0] = u.v[0];
  }
}

// One operand of a tile: ROWS rows (of A) or columns (of B), BK k, held by NT threads as UNITS units each. KC: memory
// is contiguous along k.
template <typename T, int ROWS, int BK, int NT, bool KC>
struct Operand {
  using S = typename Io<T>::storage;
  static constexpr int P = AnyTraits<T>::P;
  static constexpr int UNITS = ROWS * BK / 8 / NT;
  static constexpr int CHUNKS = ROWS / 8;       // units per k row (MC)
  static constexpr int SUB = ROWS * 64;         // bytes of one plane's k32 block in LDS
  static constexpr int PLANE = SUB * (BK / 32);
  static constexpr int BYTES = PLANE * P;
  static_assert(ROWS * BK / 8 % NT == 0 && UNITS >= 1, "whole units per thread");
  static_assert(KC || CHUNKS >= 8, "the k rows' swizzle moves a chunk within eight");

  const S* src[UNITS];  // unit's address at k tile 0
  int dst[UNITS];       // its LDS offset
  int kk[UNITS];        // its k (KC: first of 8; MC: the row) within the tile
  int left[UNITS];      // MC: valid elements from its first (8 or more: all)
  Unit<T> reg[2][UNITS];
  uint32_t empty[2];    // bit u: unit u lies past K
  int64_t step;         // elements from one k tile to the next
  const S* whole_unit;  // any 8 elements of the operand; null where it has fewer

  __device__ void init(const S* base, int64_t ld, int64_t r0, int64_t rows, int64_t K, int tid) {
    step = KC ? BK : BK * ld;
    empty[0] = empty[1] = 0;
    whole_unit = (KC ? (rows - 1) * ld + K : (K - 1) * ld + rows) >= 8 ? base : nullptr;
#pragma unroll
    for (int u = 0; u < UNITS; ++u) {
      const int id = tid + NT * u;
      if constexpr (KC) {
        const int row = id / (BK / 8), c = id % (BK / 8);
        kk[u] = c * 8;
        left[u] = 8;
        src[u] = base + min(r0 + row, rows - 1) * ld + c * 8;
        dst[u] = (c / 4) * SUB + row * 64 + (((c % 4) ^ a_swizzle(row)) * 16);
      } else {
        const int row = id / CHUNKS, c = id % CHUNKS;
        kk[u] = row;
        // a unit past the edge reads the last whole unit's columns instead (discarded); one that straddles the edge
        // runs into the next k row, which exists in every tile but the last
        const int64_t col = r0 + c * 8 < rows ? r0 + c * 8 : rows - 8;
        left[u] = static_cast<int>(min<int64_t>(rows - col, 8));
        src[u] = base + static_cast<int64_t>(row) * ld + col;
        dst[u] = (row / 32) * SUB + (row % 32) * (ROWS * 2) + ((c ^ b_swizzle16<CHUNKS>(row % 32)) * 16);
      }
    }
  }
  template <int SET>
  __device__ void load(int64_t kt) {
#pragma unroll
    for (int u = 0; u < UNITS; ++u) reg[SET][u] = load_unit<T>(src[u] + kt * step);
  }
  // The last tile, k0 .. K - 1, with zeros for the rest. Units of 8 are loaded as ever, without a branch; those past K load
  // something else in their place and are zeroed on their way to LDS (store_any). Element by element goes only the unit
  // that K ends in (KC), or that runs past the end of the last k row (MC).
  template <int SET>
  __device__ void load_tail(int64_t kt, int64_t left_k) {
    int n[UNITS];
    bool some = false;
#pragma unroll
    for (int u = 0; u < UNITS; ++u) {
      const int64_t k = left_k - kk[u];  // valid k from this unit's first
      n[u] = KC ? static_cast<int>(min<int64_t>(max<int64_t>(k, 0), 8)) : k > 1 ? 8 : k == 1 ? left[u] : 0;
      empty[SET] |= n[u] == 0 ? 1u << u : 0u;
      some |= n[u] > 0 && n[u] < 8;
    }
    if (whole_unit != nullptr) {
#pragma unroll
      for (int u = 0; u < UNITS; ++u) reg[SET][u] = load_unit<T>(n[u] == 8 ? src[u] + kt * step : whole_unit);
    }
    if (whole_unit == nullptr || __any(some)) {
#pragma unroll
      for (int u = 0; u < UNITS; ++u)
        if (whole_unit == nullptr || (n[u] > 0 && n[u] < 8)) reg[SET][u] = load_unit_partial<T>(src[u] + kt * step, n[u]);
    }
  }
  template <int SET>
  __device__ void store(unsigned char* lds) {
#pragma unroll
    for (int u = 0; u < UNITS; ++u) {
      u32x4_t plane[P];
      split_unit<T>(reg[SET][u], plane);
#pragma unroll
      for (int p = 0; p < P; ++p) *reinterpret_cast<u32x4_t*>(lds + p * PLANE + dst[u]) = plane[p];
    }
  }
  // The same for a tile that may be the last.
  template <int SET>
  __device__ void store_any(unsigned char* lds) {
    if (empty[SET] != 0) {
#pragma unroll
      for (int u = 0; u < UNITS; ++u)
#pragma unroll
        for (int i = 0; i < Unit<T>::R; ++i)
#pragma unroll
          for (int d = 0; d < 4; ++d) reg[SET][u].v[i][d] = (empty[SET] >> u) & 1u ? 0u : reg[SET][u].v[i][d];
    }
    store<SET>(lds);
  }

  // Fragment of the 16 rows (columns) from w on, in the k32 block at `sub`: lane l holds row w + l % 16, k 8 (l / 16)..+7.
  __device__ static u32x4_t fragment(const unsigned char* sub, int w, int lane) {
    if constexpr (KC) {
      const int row = w + (lane & 15);
      return *reinterpret_cast<const u32x4_t*>(sub + row * 64 + (((lane >> 4) ^ a_swizzle(row)) * 16));
    } else {
      const int q = lane & 3, e = (lane >> 2) & 3;
      const int col = w + 4 * q, krow = 8 * (lane >> 4) + e;
      const unsigned char* p = sub + krow * (ROWS * 2) + (((col >> 3) ^ b_swizzle16<CHUNKS>(krow)) * 16) + (col & 7) * 2;
      const auto lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((FH_LDS s16x4_t*)(p));
      const auto hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((FH_LDS s16x4_t*)(p + 4 * ROWS * 2));
      const u32x2_t a = __builtin_bit_cast(u32x2_t, lo), b = __builtin_bit_cast(u32x2_t, hi);
      return u32x4_t{a[0], a[1], b[0], b[1]};
    }
  }
};

// Barrier over LDS traffic only: the register prefetch stays in flight across it.
__device__ __forceinline__ void lds_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

template <int Q, int TM, int TN>
__device__ __forceinline__ void clear(f32x4_t (&sums)[Q][TM][TN]) {
#pragma unroll
  for (int q = 0; q < Q; ++q)
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) sums[q][i][j] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
}
// The accumulators of each output added up, in the first of them.
template <int Q, int TM, int TN>
__device__ __forceinline__ auto total(f32x4_t (&sums)[Q][TM][TN]) -> f32x4_t (&)[TM][TN] {
#pragma unroll
  for (int q = 1; q < Q; ++q)
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) sums[0][i][j] += sums[q][i][j];
  return sums[0];
}

// The k loop of one tile: KT steps of BK. whole_load<SET>(kt) issues the loads of tile kt < whole into register set SET,
// any_load<SET>(kt) those of any tile (nothing from KT on). Step kt: loads of kt + 2 into the set that tile kt left,
// products of kt, LDS writes of kt + 1, barrier. The main loop has no branch: where a path might have left a load of the
// same registers in flight, the compiler waits for every load before issuing the next (4095^3 bf16: 278 us against 180).
// (Spreading the LDS writes between the products in fixed order was slower for fp32.)
template <typename T, typename OpA, typename OpB, int BK, int TM, int TN, typename Whole, typename Any>
__device__ __forceinline__ void k_loop(OpA& a, OpB& b, unsigned char* lds, int KT, int whole, int m_off, int n_off,
                                       int lane, Whole&& whole_load, Any&& any_load, f32x4_t (&acc)[AnyTraits<T>::Q][TM][TN]) {
  constexpr bool F32 = std::is_same_v<T, float>;
  constexpr int P = AnyTraits<T>::P;
  constexpr int BUF = OpA::BYTES + OpB::BYTES;
  using M16 = typename AnyTraits<T>::mfma_t;
  auto store = [&]<int SET>(unsigned char* buf) {
    a.template store<SET>(buf);
    b.template store<SET>(buf + OpA::BYTES);
  };
  auto store_any = [&]<int SET>(unsigned char* buf) {
    a.template store_any<SET>(buf);
    b.template store_any<SET>(buf + OpA::BYTES);
  };
  auto products = [&](const unsigned char* buf) {
#pragma unroll
    for (int s = 0; s < BK / 32; ++s) {
      u32x4_t fa[P][TM], fb[P][TN];
#pragma unroll
      for (int p = 0; p < P; ++p) {
#pragma unroll
        for (int i = 0; i < TM; ++i)
          fa[p][i] = OpA::fragment(buf + p * OpA::PLANE + s * OpA::SUB, m_off + i * 16, lane);
#pragma unroll
        for (int j = 0; j < TN; ++j)
          fb[p][j] = OpB::fragment(buf + OpA::BYTES + p * OpB::PLANE + s * OpB::SUB, n_off + j * 16, lane);
      }
      auto pair = [&]<int PA, int PB>() {
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int j = 0; j < TN; ++j) mfma16x<M16>(fa[PA][i], fb[PB][j], acc[PA + PB > 0][i][j]);
      };
      if constexpr (F32) {
        pair.template operator()<2, 1>();
        pair.template operator()<1, 2>();
        pair.template operator()<2, 0>();
        pair.template operator()<0, 2>();
        pair.template operator()<1, 1>();
        pair.template operator()<1, 0>();
        pair.template operator()<0, 1>();
      }
      pair.template operator()<0, 0>();
    }
  };
  auto whole_step = [&]<int SET>(int kt) {
    whole_load.template operator()<SET>(kt + 2);
    products(lds + SET * BUF);
    store.template operator()<1 - SET>(lds + (1 - SET) * BUF);
    lds_barrier();
  };
  auto any_step = [&]<int SET>(int kt) {
    any_load.template operator()<SET>(kt + 2);
    products(lds + SET * BUF);
    if (kt + 1 < KT) store_any.template operator()<1 - SET>(lds + (1 - SET) * BUF);
    lds_barrier();
  };
  if (KT <= 0) return;
  any_load.template operator()<0>(0);
  any_load.template operator()<1>(1);
  store_any.template operator()<0>(lds);
  lds_barrier();
  int kt = 0;
  for (; kt + 3 < whole; kt += 2) {
    whole_step.template operator()<0>(kt);
    whole_step.template operator()<1>(kt + 1);
  }
  for (; kt < KT; kt += 2) {
    any_step.template operator()<0>(kt);
    if (kt + 1 < KT) any_step.template operator()<1>(kt + 1);
  }
}

__device__ __forceinline__ bool finite(float v) { return __builtin_fabsf(v) <= 3.4028234663852886e38f; }
// Whether the wave's 16x16 tile holds a result that is not finite (the same answer on every lane).
__device__ __forceinline__ bool any_not_finite(const f32x4_t& acc) {
  return __any(!(finite(acc[0]) && finite(acc[1]) && finite(acc[2]) && finite(acc[3])));
}

// Waves per SIMD a kernel is compiled for: two workgroups of eight waves share a CU's 16-bit LDS buffers, which 128
// registers per lane allow and 130 (the compiler's own choice at 128x128x64) do not: 4095^3 bf16 181 us against 206.
// Three workgroups of four waves share its fp32 buffers at 64x64x32.
template <typename T, int WAVES, int LDS>
constexpr int min_waves() {
  if (std::is_same_v<T, float>) return WAVES < 8 && 3 * LDS <= 160 * 1024 ? 3 : 1;
  return WAVES < 8 ? 1 : 4;
}

template <typename T, int BM, int BN, int BK, int WAVES_M, int WAVES_N, bool TA, bool TB, int E>
__global__ __launch_bounds__(WAVES_M* WAVES_N * 64,
                             (min_waves<T, WAVES_M * WAVES_N, (BM + BN) * BK * 4 * AnyTraits<T>::P>())) void
gemm_any_kernel(GemmArgs args) {
  using S = typename Io<T>::storage;
  constexpr bool F32 = std::is_same_v<T, float>;
  constexpr int NT = WAVES_M * WAVES_N * 64;
  constexpr int WM = BM / WAVES_M, WN = BN / WAVES_N;
  constexpr int TM = WM / 16, TN = WN / 16;
  using OpA = Operand<T, BM, BK, NT, !TA>;
  using OpB = Operand<T, BN, BK, NT, TB>;
  constexpr int BUF = OpA::BYTES + OpB::BYTES;
  constexpr int STAGED = WAVES_M * WAVES_N * WM * WN * static_cast<int>(sizeof(S));
  static_assert(STAGED <= 2 * BUF, "the wave tiles fit in the buffers");
  __shared__ __attribute__((aligned(1024))) unsigned char lds[2 * BUF];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / WAVES_N, wn = wave % WAVES_N;

  // tile id: consecutive tiles on one XCD (any tile count), in groups of 8 tile rows
  const int tiles = args.tiles_m * args.tiles_n;
  const int block = static_cast<int>(blockIdx.z * gridDim.x + blockIdx.x);  // (see tile_grid)
  if (block >= tiles) return;
  const int xcd = block & 7;
  const int bid = xcd * (tiles >> 3) + min(xcd, tiles & 7) + (block >> 3);
  constexpr int GROUP_M = 8;
  const int group = bid / (GROUP_M * args.tiles_n);
  const int gsize = min(args.tiles_m - group * GROUP_M, GROUP_M);
  const int in_group = bid % (GROUP_M * args.tiles_n);
  const int64_t m0 = static_cast<int64_t>(group * GROUP_M + in_group % gsize) * BM;
  const int64_t n0 = static_cast<int64_t>(in_group / gsize) * BN;

  const int inner = args.inner > 1 ? static_cast<int>(args.inner) : 1;
  const int64_t outer_y = blockIdx.y / inner, inner_y = blockIdx.y % inner;
  const S* __restrict__ A = static_cast<const S*>(args.A) + outer_y * args.stride_a + inner_y * args.inner_a;
  const S* __restrict__ B = static_cast<const S*>(args.B) + outer_y * args.stride_b + inner_y * args.inner_b;
  S* __restrict__ C = static_cast<S*>(args.C) + outer_y * args.stride_c + inner_y * args.inner_c;
  const int64_t M = args.M, N = args.N, K = args.K;
  const int KT = static_cast<int>((K + BK - 1) / BK);
  const bool tail = K % BK != 0 || (TA && M % 8 != 0) || (!TB && N % 8 != 0);
  const int whole = tail ? KT - 1 : KT;  // tiles without a remainder

  OpA a;
  OpB b;
  a.init(A, args.lda, m0, M, K, tid);
  b.init(B, args.ldb, n0, N, K, tid);

  auto whole_load = [&]<int SET>(int kt) {
    a.template load<SET>(kt);
    b.template load<SET>(kt);
  };
  auto any_load = [&]<int SET>(int kt) {
    if (kt < whole) {
      whole_load.template operator()<SET>(kt);
    } else if (kt < KT) {
      a.template load_tail<SET>(kt, K - static_cast<int64_t>(kt) * BK);
      b.template load_tail<SET>(kt, K - static_cast<int64_t>(kt) * BK);
    }
  };
  f32x4_t sums[AnyTraits<T>::Q][TM][TN];
  clear(sums);

  k_loop<T, OpA, OpB, BK>(a, b, lds, KT, whole, wm * WM, wn * WN, lane, whole_load, any_load, sums);
  f32x4_t(&acc)[TM][TN] = total(sums);

  const int g = lane >> 4, r = lane & 15;
  if constexpr (F32) {
    // the sums scaled back; those that are not finite again, on fp32 operands from memory, a row of 16x16 tiles at a time
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      f32x4_t plain[TN];
      bool again = false;
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        plain[j] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
        again |= any_not_finite(acc[i][j]);
      }
      if (again) {
        constexpr int U = 4;  // k4 steps whose loads are in flight together
        const int64_t row = min(m0 + wm * WM + i * 16 + r, M - 1);
        for (int64_t k0 = 0; k0 < K; k0 += 4 * U) {
          float va[U], vb[U][TN];
#pragma unroll
          for (int u = 0; u < U; ++u) {
            const int64_t k = min(k0 + 4 * u + g, K - 1);
            va[u] = A[TA ? k * args.lda + row : row * args.lda + k];
#pragma unroll
            for (int j = 0; j < TN; ++j) {
              const int64_t col = min(n0 + wn * WN + j * 16 + r, N - 1);
              vb[u][j] = B[TB ? col * args.ldb + k : k * args.ldb + col];
            }
          }
#pragma unroll
          for (int u = 0; u < U; ++u) {
            const bool live = k0 + 4 * u + g < K;
#pragma unroll
            for (int j = 0; j < TN; ++j)
              plain[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(live ? va[u] : 0.0f, live ? vb[u][j] : 0.0f, plain[j], 0, 0, 0);
          }
        }
      }
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int x = 0; x < 4; ++x) acc[i][j][x] = finite(acc[i][j][x]) ? acc[i][j][x] * kSplitUnscale : plain[j][x];
    }
  }

  // epilogue: each wave stages its rounded tile in LDS (free: every wave is past its last read), then runs the program
  // on 8 or 4 outputs at a time; a row's last vector is moved back to end at the edge, and stores only the outputs that the
  // one before it does not. Fewer columns than a vector go one per lane. (4001x33x47 f16 with add;gelu 10.8 us while such
  // a vector went element by element, 5.6 now.)
  S* wl = reinterpret_cast<S*>(lds) + wave * (WM * WN);
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int x = 0; x < 4; ++x) wl[(i * 16 + 4 * g + x) * WN + j * 16 + r] = Io<T>::store(acc[i][j][x]);
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_wave_barrier();
  constexpr int V = 16 / static_cast<int>(sizeof(S));
  constexpr int LPR = WN / V, RPI = 64 / LPR;
  static_assert(64 % LPR == 0 && WM % RPI == 0, "epilogue access shape");
  const int lr = lane % LPR;
  const int64_t col0 = n0 + wn * WN;
  const int cols = static_cast<int>(min<int64_t>(N - col0, WN));  // this wave's, 0 or less when it has none
  const EpilogueArgs& ep = args.ep;
  for (int it = 0; it < WM / RPI; ++it) {
    const int rr = it * RPI + lane / LPR;
    const int64_t row = m0 + wm * WM + rr;
    if (row >= M) continue;
    const int64_t idx = row * args.ldc + col0;
    const S* wr = wl + rr * WN;
    if (cols >= V) {
      if (lr * V >= cols) continue;
      const int c = min(lr * V, cols - V);
      uint4 v;
      if (c == lr * V) v = *reinterpret_cast<const uint4*>(wr + c);
      else __builtin_memcpy(&v, wr + c, 16);
      const uint4 out = epi_vec<E, T>(ep, v, idx + c);
      if (c == lr * V) {
        *reinterpret_cast<u32x4_any*>(C + idx + c) = u32x4_t{out.x, out.y, out.z, out.w};
      } else {
        S e[V];
        __builtin_memcpy(e, &out, 16);
#pragma unroll
        for (int x = 1; x < V; ++x)
          if (c + x >= lr * V) C[idx + c + x] = e[x];
      }
    } else {
      for (int x = lr; x < cols; x += LPR) C[idx + x] = Io<T>::store(epi_one<E, T>(ep, Io<T>::load(wr[x]), idx + x));
    }
  }
}

// The grid of `tiles` workgroups: a launch holds fewer than 2^32 work items along x, so more than 2^22 workgroups (of up to
// 512) go along z as well.
inline dim3 tile_grid(int64_t tiles, int64_t batch) {
  const int64_t x = std::min<int64_t>(tiles, int64_t{1} << 22);
  return dim3(static_cast<uint32_t>(x), static_cast<uint32_t>(batch), static_cast<uint32_t>((tiles + x - 1) / x));
}

template <typename T, int BM, int BN, int BK, int WAVES_M, int WAVES_N, bool TA, bool TB>
fh_status launch(GemmArgs args, int64_t batch, hipStream_t stream) {
  args.tiles_m = static_cast<int32_t>((args.M + BM - 1) / BM);
  args.tiles_n = static_cast<int32_t>((args.N + BN - 1) / BN);
  const dim3 grid = tile_grid(static_cast<int64_t>(args.tiles_m) * args.tiles_n, batch);
  auto go = [&]<int E>() {
    hipLaunchKernelGGL((gemm_any_kernel<T, BM, BN, BK, WAVES_M, WAVES_N, TA, TB, E>), grid,
                       dim3(WAVES_M * WAVES_N * 64), 0, stream, args);
    return launch_status("gemm_any_kernel launch");
  };
  // the programs that Linear layers carry have kernels of their own, the rest takes the interpreter (see EpiKind);
  // gradients (a transposed operand) carry none
  if constexpr (!TA && !TB) {
    switch (epi_kind(args.ep)) {
      case kEpiNone: return go.template operator()<kEpiNone>();
      case kEpiAdd: return go.template operator()<kEpiAdd>();
      case kEpiAddRelu: return go.template operator()<kEpiAddRelu>();
      case kEpiAddGelu: return go.template operator()<kEpiAddGelu>();
      default: break;
    }
  } else {
    if (args.ep.nseg == 0) return go.template operator()<kEpiNone>();
  }
  return go.template operator()<kEpiAny>();
}

// What the kernel accepts: an operand contiguous along m or n needs 8 of them (its units are moved back to the edge)
// and a row stride of as many (a unit that straddles the edge runs into the next row).
inline bool accepts(const GemmArgs& args, int64_t batch) {
  if (args.K < 0 || args.groups > 0 || args.row_softmax || batch > 65535) return false;  // (K = 0: zeros)
  if (args.trans_a ? args.M < 8 : false) return false;
  if (args.trans_b ? false : args.N < 8) return false;
  const int64_t tiles = ((args.M + 31) / 32) * ((args.N + 63) / 64);
  return args.K <= (int64_t{1} << 30) && tiles <= (int64_t{1} << 30);
}

}  // namespace gemm_any

// Launches the kernel and returns true, with the launch's status in *status; false (and nothing launched) for a
// problem it does not accept.
bool gemm_any16_try_launch(int32_t dtype, const GemmArgs& args, int64_t batch, hipStream_t stream, fh_status* status);
bool gemm_f32_try_launch(const GemmArgs& args, int64_t batch, hipStream_t stream, fh_status* status);

}  // namespace fh
