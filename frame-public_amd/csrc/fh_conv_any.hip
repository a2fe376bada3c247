// Conv2d forward on the matrix cores for the geometries without a kernel of their own, NCHW in and out: the implicit GEMM
// y[cout, pixel] = w[cout, k] · x[k, pixel] with k = (ci, kh, kw) as the filter is stored and pixels numbered through the
// batch (reference semantics: src/backends/cpu/kernels/conv.cpp:223-314: the bias is added in fp32 before the one
// rounding, then the epilogue program). 16-bit operands as they are, fp32 as three bf16 planes; tile loop, split and
// its range as in fh_gemm_any.h.
//
// No operand is copied or repacked: the filter is the k-contiguous operand, and 8 consecutive output pixels of one k are
// 8 consecutive inputs of a row (stride 1 along the row, output rows of at least 8: one vector load at element alignment,
// two where the pixels run over a row's end; else one load per pixel), with the padding masked in registers.
// What bounds it is the operand's way to LDS: every input is loaded and (fp32) split once per filter tap and tile of
// output channels.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <string>

#include "fh_conv_any.h"
#include "fh_gemm_any.h"

namespace fh {
namespace {

using namespace gemm_any;

struct ConvAnyArgs {
  const void *x, *w, *bias;
  void* y;
  int32_t cin, h, wd, cout, kh, kw, sh, sw, ph, pw, oh, ow;
  int32_t k, p;         // Cin * KH * KW, N * OH * OW
  int64_t total;        // elements of x
  uint32_t m_taps, m_kw;  // ceil(2^32 / (KH * KW)), ceil(2^32 / KW); 0 for a divisor of 1
  int32_t tiles_m, tiles_n;
  EpilogueArgs ep;
};

__device__ __forceinline__ int div_by(int v, uint32_t magic) {
  return magic == 0 ? v : static_cast<int>(__umulhi(static_cast<uint32_t>(v), magic));
}

struct Tap {
  int a, b, delta;  // filter row and column, offset of (ci, a, b) from a pixel's first input
};
__device__ __forceinline__ Tap tap_of(const ConvAnyArgs& g, int k) {
  const int ci = div_by(k, g.m_taps), r = k - ci * (g.kh * g.kw);
  const int a = div_by(r, g.m_kw), b = r - a * g.kw;
  return {a, b, (ci * g.h + a) * g.wd + b};
}

// First input of an output pixel: its offset in x and its row and column in the plane (negative in the padding).
struct Pixel {
  int base, ih, iw;
};
__device__ __forceinline__ Pixel pixel_of(const ConvAnyArgs& g, int p) {
  const int ohw = g.oh * g.ow;
  const int img = p / ohw, r = p - img * ohw, oh = r / g.ow, ow = r - oh * g.ow;
  const int ih = oh * g.sh - g.ph, iw = ow * g.sw - g.pw;
  return {(img * g.cin * g.h + ih) * g.wd + iw, ih, iw};
}

// The elements of u that `mask` (bit e: element e) keeps, zero elsewhere.
template <typename T>
__device__ __forceinline__ Unit<T> keep(const Unit<T>& u, uint32_t mask) {
  Unit<T> o;
#pragma unroll
  for (int i = 0; i < Unit<T>::R; ++i)
#pragma unroll
    for (int d = 0; d < 4; ++d) {
      uint32_t m;
      if constexpr (std::is_same_v<T, float>) {
        m = 0u - ((mask >> (4 * i + d)) & 1u);
      } else {
        m = (0u - ((mask >> (2 * d)) & 1u)) & 0xffffu;
        m |= (0u - ((mask >> (2 * d + 1)) & 1u)) & 0xffff0000u;
      }
      o.v[i][d] = u.v[i][d] & m;
    }
  return o;
}

// How a thread's 8 consecutive output pixels lie in x.
enum PixelRuns {
  kOneRun,   // one run of consecutive inputs (stride 1, output rows of whole units)
  kTwoRuns,  // at most two (stride 1, output rows of at least 8)
  kGather,   // anything
};

// The im2col operand of a tile. Thread t holds the 8 pixels n0 + 8 (t % CHUNKS) .. + 7 for the k rows t / CHUNKS + ...
// Loads are unconditional, from addresses clamped into x, and what they bring is masked on its way to LDS: a load whose
// result is masked at once, or that is skipped on a branch, would be waited for before the next one is issued.
template <typename T, int BN, int BK, int NT, int RUNS>
struct Im2col : Operand<T, BN, BK, NT, false> {
  using Base = Operand<T, BN, BK, NT, false>;
  using S = typename Io<T>::storage;
  static constexpr int U = Base::UNITS;
  static constexpr int PIX = RUNS == kGather ? 8 : RUNS == kTwoRuns ? 2 : 1;
  static_assert(NT % Base::CHUNKS == 0, "a thread's units are the same pixels");

  const S* x;
  Pixel px[PIX];
  int run;                                          // pixels of the first run
  Unit<T> raw[2][U][RUNS == kTwoRuns ? 2 : 1];      // (kGather: gathered instead)
  S gathered[2][U][RUNS == kGather ? 8 : 1];
  uint32_t mask[2][U];                              // elements to keep: bits 0-7, of the second run bits 8-15

  __device__ void init(const ConvAnyArgs& g, int n0, int tid) {
    x = static_cast<const S*>(g.x);
    const int c = tid % Base::CHUNKS, p0 = n0 + 8 * c;
    if constexpr (RUNS != kGather) {
      const int first = min(p0, g.p - 1);
      px[0] = pixel_of(g, first);
      run = 8;
      if constexpr (RUNS == kTwoRuns) {
        run = min(8, g.ow - (px[0].iw + g.pw));
        px[1] = pixel_of(g, min(first + run, g.p - 1));
        px[1].base -= run;  // element e of the unit is at base + e in either run
        px[1].iw -= run;
      }
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e) px[e] = pixel_of(g, min(p0 + e, g.p - 1));
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int row = tid / Base::CHUNKS + u * (NT / Base::CHUNKS);
      this->kk[u] = row;
      this->dst[u] = (row / 32) * Base::SUB + (row % 32) * (BN * 2) + ((c ^ b_swizzle16<Base::CHUNKS>(row % 32)) * 16);
    }
  }

  // Mask of the elements in [from, to) of a run at pixel q that tap t finds inside the plane; the run's 8 elements in u.
  __device__ uint32_t load_run(const ConvAnyArgs& g, const Pixel& q, const Tap& t, bool live, int from, int to,
                               Unit<T>& u) const {
    const int iw = q.iw + t.b;
    const int lo = max(from, -iw), hi = min(to, g.wd - iw);
    const bool in = live && static_cast<unsigned>(q.ih + t.a) < static_cast<unsigned>(g.h) && lo < hi;
    const uint32_t m = in ? ((1u << (hi & 31)) - 1u) & ~((1u << (lo & 31)) - 1u) : 0u;
    const int off = q.base + t.delta;
    const int last = static_cast<int>(g.total) - 8;
    const int at = in ? min(max(off, 0), last) : 0;
    u = load_unit<T>(x + at);
    if (__any(in && at != off)) {  // the run would leave the tensor: its very first and last pixels
      if (in && at != off) {
        S e[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) e[i] = 0;
#pragma unroll
        for (int i = 0; i < 8; ++i)
          if ((m >> i) & 1u) e[i] = x[off + i];
        __builtin_memcpy(&u, e, sizeof(u));
      }
    }
    return m;
  }

  template <int SET>
  __device__ void load(const ConvAnyArgs& g, int kt) {
#pragma unroll
    for (int n = 0; n < U; ++n) {
      const int k = kt * BK + this->kk[n];
      const bool live = k < g.k;
      const Tap t = tap_of(g, live ? k : 0);
      if constexpr (RUNS != kGather) {
        uint32_t m = load_run(g, px[0], t, live, 0, run, raw[SET][n][0]);
        if constexpr (RUNS == kTwoRuns) m |= load_run(g, px[1], t, live && run < 8, run, 8, raw[SET][n][1]) << 8;
        mask[SET][n] = m;
      } else {
        uint32_t m = 0;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const bool in = live && static_cast<unsigned>(px[i].ih + t.a) < static_cast<unsigned>(g.h) &&
                          static_cast<unsigned>(px[i].iw + t.b) < static_cast<unsigned>(g.wd);
          gathered[SET][n][i] = x[in ? px[i].base + t.delta : 0];
          m |= in ? 1u << i : 0u;
        }
        mask[SET][n] = m;
      }
    }
  }
  template <int SET>
  __device__ void store(unsigned char* lds) {
#pragma unroll
    for (int n = 0; n < U; ++n) {
      Unit<T> u;
      if constexpr (RUNS == kGather) {
        __builtin_memcpy(&u, gathered[SET][n], sizeof(u));
        u = keep<T>(u, mask[SET][n]);
      } else {
        u = keep<T>(raw[SET][n][0], mask[SET][n]);
        if constexpr (RUNS == kTwoRuns) {
          const Unit<T> v = keep<T>(raw[SET][n][1], mask[SET][n] >> 8);
#pragma unroll
          for (int i = 0; i < Unit<T>::R; ++i) u.v[i] |= v.v[i];
        }
      }
      u32x4_t plane[Base::P];
      split_unit<T>(u, plane);
#pragma unroll
      for (int p = 0; p < Base::P; ++p) *reinterpret_cast<u32x4_t*>(lds + p * Base::PLANE + this->dst[n]) = plane[p];
    }
  }
  template <int SET>
  __device__ void store_any(unsigned char* lds) { store<SET>(lds); }
};

// Waves per SIMD, as min_waves; a gather of fp32 pixels needs more registers than three leave (stride 2, [32,64,56,56] to
// 128 channels: 80 us with them, 57 without).
template <typename T, int WAVES, int LDS, int RUNS>
constexpr int conv_waves() {
  return RUNS == kGather ? 1 : min_waves<T, WAVES, LDS>();
}

template <typename T, int BM, int BN, int BK, int WAVES_M, int WAVES_N, int RUNS, int E>
__global__ __launch_bounds__(WAVES_M* WAVES_N * 64,
                             (conv_waves<T, WAVES_M * WAVES_N, (BM + BN) * BK * 4 * AnyTraits<T>::P, RUNS>())) void
conv_any_kernel(ConvAnyArgs g) {
  using S = typename Io<T>::storage;
  constexpr int NT = WAVES_M * WAVES_N * 64;
  constexpr int WM = BM / WAVES_M, WN = BN / WAVES_N;
  constexpr int TM = WM / 16, TN = WN / 16;
  using OpA = Operand<T, BM, BK, NT, true>;
  using OpB = Im2col<T, BN, BK, NT, RUNS>;
  constexpr int BUF = OpA::BYTES + OpB::BYTES;
  static_assert(WAVES_M * WAVES_N * WM * WN * static_cast<int>(sizeof(S)) <= 2 * BUF, "the wave tiles fit in the buffers");
  __shared__ __attribute__((aligned(1024))) unsigned char lds[2 * BUF];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / WAVES_N, wn = wave % WAVES_N;

  // consecutive tiles on one XCD; the channel tiles of one pixel tile are neighbours, so its inputs are shared in L2
  const int tiles = g.tiles_m * g.tiles_n;
  const int block = static_cast<int>(blockIdx.z * gridDim.x + blockIdx.x);  // (see tile_grid)
  if (block >= tiles) return;
  const int xcd = block & 7;
  const int bid = xcd * (tiles >> 3) + min(xcd, tiles & 7) + (block >> 3);
  const int m0 = (bid % g.tiles_m) * BM, n0 = (bid / g.tiles_m) * BN;

  OpA a;
  OpB b;
  a.init(static_cast<const S*>(g.w), g.k, m0, g.cout, g.k, tid);
  b.init(g, n0, tid);
  const int KT = (g.k + BK - 1) / BK;
  const int whole = g.k % BK != 0 ? KT - 1 : KT;
  auto whole_load = [&]<int SET>(int kt) {
    a.template load<SET>(kt);
    b.template load<SET>(g, kt);
  };
  auto any_load = [&]<int SET>(int kt) {
    if (kt < whole) {
      whole_load.template operator()<SET>(kt);
    } else if (kt < KT) {
      a.template load_tail<SET>(kt, g.k - kt * BK);
      b.template load<SET>(g, kt);
    }
  };
  f32x4_t sums[AnyTraits<T>::Q][TM][TN];
  clear(sums);
  k_loop<T, OpA, OpB, BK>(a, b, lds, KT, whole, wm * WM, wn * WN, lane, whole_load, any_load, sums);
  f32x4_t(&acc)[TM][TN] = total(sums);

  const int q = lane >> 4, r = lane & 15;
  // Results that are not finite are taken again one product at a time, in the reference's order: it skips the taps in the
  // padding, where a matrix product would add zero times the filter's value, NaN for an infinite one. 16-bit operands
  // without padding need no second pass (their sums hold the same infinities and NaN), fp32 planes always do. The loads of
  // several taps are in flight together: with one infinite value in the filter [32,64,56,56] x [64,64,3,3] f32 takes 560 us
  // (73 without; 813 one tap at a time), in the input 223; bf16 [16,16,35,35] x [100,16,5,5] 160 (19; 214).
  constexpr bool F32 = std::is_same_v<T, float>;
  if (F32 || g.ph > 0 || g.pw > 0) {
    const S* x = static_cast<const S*>(g.x);
    const S* w = static_cast<const S*>(g.w);
#pragma unroll
    for (int j = 0; j < TN; ++j) {
#pragma unroll
      for (int i = 0; i < TM; ++i) {
        f32x4_t plain{0.0f, 0.0f, 0.0f, 0.0f};
        if (any_not_finite(acc[i][j])) {
          constexpr int U = 8;  // taps whose loads are in flight together
          const Pixel px = pixel_of(g, min(n0 + wn * WN + j * 16 + r, g.p - 1));
          for (int k0 = 0; k0 < g.k; k0 += U) {
            S xv[U], wv[U][4];
            bool in[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
              const int k = min(k0 + u, g.k - 1);
              const Tap t = tap_of(g, k);
              in[u] = k0 + u < g.k && static_cast<unsigned>(px.ih + t.a) < static_cast<unsigned>(g.h) &&
                      static_cast<unsigned>(px.iw + t.b) < static_cast<unsigned>(g.wd);
              xv[u] = x[in[u] ? px.base + t.delta : 0];
#pragma unroll
              for (int e = 0; e < 4; ++e)
                wv[u][e] = w[static_cast<int64_t>(min(m0 + wm * WM + i * 16 + 4 * q + e, g.cout - 1)) * g.k + k];
            }
#pragma unroll
            for (int u = 0; u < U; ++u)
#pragma unroll
              for (int e = 0; e < 4; ++e)
                plain[e] = in[u] ? plain[e] + Io<T>::load(xv[u]) * Io<T>::load(wv[u][e]) : plain[e];
          }
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float v = acc[i][j][e];
          acc[i][j][e] = finite(v) ? (F32 ? v * kSplitUnscale : v) : plain[e];
        }
      }
    }
  }

  // bias and the one rounding, the wave's tile through LDS, then the program on 16-byte vectors of a channel's pixels; a
  // vector that runs over an image's end or the last pixel is stored element by element (the program before the branch, and
  // no division: a launch this short waits for its instructions, f16 [55,24,2,13] 1x1 to 100 with relu 12.7 us, 8.6 so)
  const S* bias = static_cast<const S*>(g.bias);
  S* wl = reinterpret_cast<S*>(lds) + wave * (WM * WN);
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int x = 0; x < 4; ++x) {
      const int row = i * 16 + 4 * q + x;
      float add = 0.0f;
      if (bias != nullptr) add = Io<T>::load(bias[min(m0 + wm * WM + row, g.cout - 1)]);
#pragma unroll
      for (int j = 0; j < TN; ++j) wl[row * WN + j * 16 + r] = Io<T>::store(acc[i][j][x] + add);
    }
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_wave_barrier();
  constexpr int V = 16 / static_cast<int>(sizeof(S));
  constexpr int LPR = WN / V, RPI = 64 / LPR;
  static_assert(64 % LPR == 0 && WM % RPI == 0, "epilogue access shape");
  S* y = static_cast<S*>(g.y);
  const int c = (lane % LPR) * V;
  const int p = n0 + wn * WN + c;
  const int ohw = g.oh * g.ow;
  const int img = p / ohw, at = p - img * ohw;
  for (int it = 0; it < WM / RPI; ++it) {
    const int rr = it * RPI + lane / LPR;
    const int row = m0 + wm * WM + rr;
    if (row >= g.cout || p >= g.p) continue;
    const int64_t idx = (static_cast<int64_t>(img) * g.cout + row) * ohw + at;
    const bool whole = at + V <= ohw && p + V <= g.p;
    // (of the instances here only the interpreter, kEpiAny, has operands to load)
    uint4 out = *reinterpret_cast<const uint4*>(wl + rr * WN + c);
    if (E != kEpiAny || whole) out = epi_vec<E, T>(g.ep, out, idx);
    if (whole) {
      *reinterpret_cast<u32x4_any*>(y + idx) = u32x4_t{out.x, out.y, out.z, out.w};
    } else {
      S e[V];
      __builtin_memcpy(e, &out, 16);
      const int64_t hop = static_cast<int64_t>(g.cout - 1) * ohw;  // from an image's end to the same channel's next pixel
#pragma unroll
      for (int x = 0; x < V; ++x) {
        if (p + x >= g.p) continue;
        const int over = ohw >= V ? (at + x >= ohw ? 1 : 0) : (at + x) / ohw;
        const int64_t ix = idx + x + over * hop;
        if constexpr (E == kEpiAny) e[x] = Io<T>::store(epi_one<E, T>(g.ep, Io<T>::load(e[x]), ix));
        y[ix] = e[x];
      }
    }
  }
}

template <typename T, int BM, int BN, int BK, int WAVES_M, int WAVES_N>
fh_status launch_conv(ConvAnyArgs g, int runs, hipStream_t stream) {
  g.tiles_m = (g.cout + BM - 1) / BM;
  g.tiles_n = (g.p + BN - 1) / BN;
  const dim3 grid = tile_grid(static_cast<int64_t>(g.tiles_m) * g.tiles_n, 1);
  auto go = [&]<int RUNS, int E>() {
    hipLaunchKernelGGL((conv_any_kernel<T, BM, BN, BK, WAVES_M, WAVES_N, RUNS, E>), grid, dim3(WAVES_M * WAVES_N * 64), 0,
                       stream, g);
    return launch_status("conv_any_kernel launch");
  };
  auto by_program = [&]<int RUNS>() {
    switch (epi_kind(g.ep)) {
      case kEpiNone: return go.template operator()<RUNS, kEpiNone>();
      case kEpiRelu: return go.template operator()<RUNS, kEpiRelu>();
      default: return go.template operator()<RUNS, kEpiAny>();
    }
  };
  return runs == kOneRun    ? by_program.template operator()<kOneRun>()
         : runs == kTwoRuns ? by_program.template operator()<kTwoRuns>()
                            : by_program.template operator()<kGather>();
}

// 64 x 64 tiles throughout: the steps are bound by the latency and the vector instructions of the operands' way to LDS, and
// three to five such workgroups per CU overlap it best (us on 64x64 / 64x128 / 128x128 tiles, fp32 of six products:
// [32,64,56,56] x [64,64,3,3] 67 / 80 / 129, [8,128,28,28] x [128,128,3,3] 37 / 62 / 61, stride 2 to 256 channels 43 / 68 / 70; bf16 27 /
// 35 / 54, 21 / 113 / 28, 27 / 303 / 47).
template <typename T>
fh_status dispatch_conv(const ConvAnyArgs& g, int runs, hipStream_t stream) {
  // fp32 with a tile per CU or less waits for its loads, splits and barriers in turn: half of the channels and twice the k
  // between barriers take 0.6-0.75 us per k32 against 0.75-0.9 (one image of 512 channels, 14 x 14, 3x3 to 64: 130 us,
  // 108 so; 106 channels-last on fp32 MFMA)
  const int64_t tiles32 = ((g.cout + 31) / 32) * ((static_cast<int64_t>(g.p) + 63) / 64);
  if constexpr (std::is_same_v<T, float>) {
    if (tiles32 <= device_cu_count()) return launch_conv<T, 32, 64, 64, 2, 2>(g, runs, stream);
  }
  return launch_conv<T, 64, 64, std::is_same_v<T, float> ? 32 : 64, 2, 2>(g, runs, stream);
}

// Whether one thread per output (conv2d_direct_kernel, in the reference's order) is done first: with few output channels most
// of a tile's 64 are idle, and in planes lower than the filter the tiles multiply the rows of padding that it skips. us,
// measured on MI355X over 1 to 512 channels, 1 to 2^22 pixels and K from 1 to 2000: a tile costs 2.8 ns and 1.8 per step, and
// 0.9 us per step where it waits for each; 64 outputs of the direct kernel 0.3 ns and 0.05 (16-bit 0.042) per k, its sum in
// order 0.12 us per k and 0.03 per skipped row, whichever is longer and a part of the other.
// 3x3 of one channel to one, [16,1,512,512] f32 54 us against 306, to four 185 / 309, to eight 374 / 309; three to one,
// [16,3,224,224] bf16 20 / 59; 16 to one, [16,16,128,128] f32 35 / 51; 64 to one 1x1, [16,64,64,64] f32 18 / 9; one 8x8 plane
// 3.7 / 5.1; 7x7 stride 2, [9,3,1,14] to 512 f32 7.6 / 11.8, [4,24,1,100] to 64 31 / 43.
bool direct_first(const ConvGeom& c, int64_t pixels, bool f32) {
  const double rows = static_cast<double>((pixels + 63) / 64), cin = static_cast<double>(c.cin);
  const double inside = static_cast<double>(std::min(c.kh, c.h)), k = cin * inside * static_cast<double>(c.kw);
  const double steps = std::ceil(cin * static_cast<double>(c.kh * c.kw) / (f32 ? 32 : 64));
  const double sum = 0.12 * k + 0.03 * cin * (static_cast<double>(c.kh) - inside);
  const double all = 1e-3 * rows * static_cast<double>(c.cout) * (0.3 + (f32 ? 0.05 : 0.042) * k);
  const double direct = 3.1 + std::max(sum, all) + 0.3 * std::min(sum, all);
  const double tiles = 4.4 + std::max(0.9 * steps, 1e-3 * rows * static_cast<double>((c.cout + 63) / 64) * (2.8 + 1.8 * steps));
  return direct < tiles;
}

}  // namespace

bool conv_any_try_launch(int32_t dtype, const void* x, const void* w, const void* bias, void* y, const ConvGeom& c,
                         const ConvEpilogue& ep, hipStream_t stream, fh_status* status) {
  constexpr int64_t kMax = int64_t{1} << 30;  // offsets and pixel numbers are 32-bit
  const int64_t total = c.n * c.cin * c.h * c.w, pixels = c.n * c.oh * c.ow, k = c.cin * c.kh * c.kw;
  if (c.groups != 1 || total <= 0 || total > kMax || pixels > kMax || k > kMax || c.kh * c.kw > 4096 ||
      k * c.kh * c.kw >= (int64_t{1} << 32) || c.cout > kMax || c.ph > 32767 || c.pw > 32767 || c.sh > 32767 ||
      c.sw > 32767 || (c.oh * c.sh + c.ph + c.kh) * (c.w + c.pw + c.kw) > kMax)
    return false;
  const int64_t tiles = ((c.cout + 63) / 64) * ((pixels + 63) / 64);
  if (tiles > (int64_t{1} << 30) || direct_first(c, pixels, dtype == FH_F32)) return false;
  auto magic = [](int64_t d) { return d == 1 ? 0u : static_cast<uint32_t>(((int64_t{1} << 32) + d - 1) / d); };
  auto i32 = [](int64_t v) { return static_cast<int32_t>(v); };
  ConvAnyArgs g{x,        w,        bias,     y,        i32(c.cin), i32(c.h),  i32(c.w),  i32(c.cout), i32(c.kh),
                i32(c.kw), i32(c.sh), i32(c.sw), i32(c.ph), i32(c.pw), i32(c.oh), i32(c.ow), i32(k),      i32(pixels),
                total,    magic(c.kh * c.kw), magic(c.kw), 0, 0, {}};
  g.ep.nseg = ep.nseg;
  g.ep.round_between = ep.round_between;
  for (int s = 0; s < FH_MAX_SEGMENTS; ++s) g.ep.ops[s] = ep.ops[s], g.ep.ins[s] = ep.ins[s];
  // (vector loads need a whole unit in x)
  const int runs = c.sw != 1 || c.ow < 8 || total < 8 ? kGather : c.ow % 8 == 0 ? kOneRun : kTwoRuns;
  *status = dtype == FH_F32    ? dispatch_conv<float>(g, runs, stream)
            : dtype == FH_BF16 ? dispatch_conv<bf16_t>(g, runs, stream)
                               : dispatch_conv<f16_t>(g, runs, stream);
  return true;
}

}  // namespace fh
