// conv2d_grad_filter_internal on MFMA (bf16 / f16): the filter gradient as a GEMM over the batch-spatial positions,
//   dW[co][(a,b,ci)] = sum over p = (n, oh, ow) of dy[p][co] * x[n][oh*sh - ph + a][ow*sw - pw + b][ci],
// M = Cout, N = KH*KW*Cin, K = N*Ho*Wo, with both operands channels-last (dy [P][Cout], x [N][H][W][Cin]). K is
// the long dimension (batch times the output plane) and M*N is small, so K is split across workgroups: each
// writes an fp32 partial tile into a workspace, and a second kernel sums the partials in split order and writes
// dW in the reference's [Cout][Cin][KH][KW] layout with one rounding.
//
// Both operands are k-major (rows of p), so both MFMA fragments come from ds_read_b64_tr_b16 transpose reads of
// [BK][cols] LDS tiles; the k loop is the one of the GEMMs of any alignment (fh_gemm_any.h: v_mfma_f32_16x16x32, two LDS
// buffers of 64 p-rows, two register sets, loads two tiles ahead, no branch). Loads are unconditional: rows past the split
// and taps in the padding read the operand's first vector and are zeroed on their way to LDS, because a load behind a
// branch is waited for before the next one is issued. Tiles: WM (co) x 128 (a,b,ci) per workgroup of 4 waves, WM = 128 when
// Cout >= 128 and 64 otherwise; two workgroups per CU. What bounds it is the operands' way from L2, as x is read once per
// filter tap: ResNet-18's layers move 230-385 MB through it per gradient, 6-7.7 TB/s. us per gradient at batch 64, bf16
// (before: conditional loads one tile ahead, 32x32x16 tiles): WM 64 72.0 -> 64.4, WM 128 30.8 -> 30.5.
#include <algorithm>
#include <mutex>
#include <string>

#include "fh_gemm_any.h"
#include "fh_mfma16.h"

namespace fh {
namespace {

using namespace mfma16;

constexpr int kWN = 128, kWK = 64;  // workgroup tile columns and rows per stage (WM is a template argument)
constexpr int kWThreads = 256;

struct WgradArgs {
  const void* x;   // [N][H][W][Cin] (Cin % 8 == 0)
  const void* dy;  // [P][Cout] (Cout % 8 == 0)
  float* part;     // [splits][Cout][NC]
  int32_t h, w, cin, cout, kw, sh, sw, ph, pw, oh, ow, nc, tiles_n;
  int64_t p, rows_per_split;
  uint64_t plane_m, ow_m;  // multiply-shift dividers for Ho*Wo and Wo (make_divider)
  uint32_t plane_s, ow_s;
};

// Division of 0 <= n < 2^31 by a fixed d >= 1 as floor(n * m / 2^s) (Granlund and Montgomery, "Division by
// invariant integers using multiplication", 1994, theorem 4.2 with N = 31): l = ceil(log2 d), s = 31 + l,
// m = floor(2^s / d) + 1, so 2^s < m d <= 2^s + 2^l and the quotient is exact. m <= 2^32, so n * m < 2^63.
inline void make_divider(int64_t d, uint64_t& m, uint32_t& s) {
  int l = 0;
  while ((int64_t{1} << l) < d) ++l;
  s = static_cast<uint32_t>(31 + l);
  m = (uint64_t{1} << s) / static_cast<uint64_t>(d) + 1;
}
__device__ __forceinline__ int32_t div_by(int32_t n, uint64_t m, uint32_t s) {
  return static_cast<int32_t>((static_cast<uint64_t>(static_cast<uint32_t>(n)) * m) >> s);
}

// Workgroup tile rows for a filter of cout output channels (the host's and the kernel's choice must agree).
inline int wgrad_wm(int64_t cout) { return cout >= 128 ? 128 : 64; }

// One operand of a tile, COLS columns of rows p: thread t holds the column vector t % CHUNKS of the p-rows
// t / CHUNKS + u * NT / CHUNKS.
template <typename T, int COLS>
struct RowsOperand : gemm_any::Operand<T, COLS, kWK, kWThreads, false> {
  using Base = gemm_any::Operand<T, COLS, kWK, kWThreads, false>;
  using S = typename Io<T>::storage;
  static constexpr int U = Base::UNITS, STEP = kWThreads / Base::CHUNKS;
  static_assert(kWThreads % Base::CHUNKS == 0, "a thread's units are the same columns");
  uint32_t live[2];  // bit u: unit u holds values (zero otherwise)

  __device__ void init(int tid) {
    const int c = tid % Base::CHUNKS;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int row = tid / Base::CHUNKS + u * STEP;
      this->kk[u] = row;
      this->dst[u] = (row / 32) * Base::SUB + (row % 32) * (COLS * 2) + ((c ^ b_swizzle16<Base::CHUNKS>(row % 32)) * 16);
    }
  }
  // address(p): the unit's vector in row p, or null where it is zero
  template <int SET, typename Address>
  __device__ void load(int32_t p0, const S* base, Address&& address) {
    uint32_t m = 0;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const S* at = address(p0 + this->kk[u]);
      m |= at != nullptr ? 1u << u : 0u;
      this->reg[SET][u].v[0] = *reinterpret_cast<const u32x4_t*>(at != nullptr ? at : base);
    }
    live[SET] = m;
  }
  template <int SET>
  __device__ void store(unsigned char* lds) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const bool on = (live[SET] >> u) & 1u;
      u32x4_t v = this->reg[SET][u].v[0];
#pragma unroll
      for (int d = 0; d < 4; ++d) v[d] = on ? v[d] : 0u;
      *reinterpret_cast<u32x4_t*>(lds + this->dst[u]) = v;
    }
  }
  template <int SET>
  __device__ void store_any(unsigned char* lds) { store<SET>(lds); }
};

template <typename T, int kWM>
__global__ __launch_bounds__(kWThreads) void conv_wgrad_kernel(WgradArgs a) {
  static_assert(kWM == 64 || kWM == 128, "tile rows");
  using S = typename Io<T>::storage;
  using OpA = RowsOperand<T, kWM>;
  using OpB = RowsOperand<T, kWN>;
  constexpr int WM = kWM / 2, WN = kWN / 2, TM = WM / 16, TN = WN / 16;
  __shared__ __attribute__((aligned(1024))) unsigned char lds[2 * (OpA::BYTES + OpB::BYTES)];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave >> 1, wn = wave & 1;
  const int tm = blockIdx.x / a.tiles_n, tn = blockIdx.x % a.tiles_n;
  const int m0 = tm * kWM, n0 = tn * kWN;
  // p fits 32 bits (checked by the host)
  const int32_t p_begin = static_cast<int32_t>(static_cast<int64_t>(blockIdx.y) * a.rows_per_split);
  const int32_t p_end = static_cast<int32_t>(min(a.p, static_cast<int64_t>(p_begin) + a.rows_per_split));
  const S* __restrict__ X = static_cast<const S*>(a.x);
  const S* __restrict__ DY = static_cast<const S*>(a.dy);

  OpA oa;
  OpB ob;
  oa.init(tid);
  ob.init(tid);
  // this thread's columns: 8 output channels of dy, 8 input channels of one filter tap of x
  const int mcol = m0 + 8 * (tid % OpA::CHUNKS);
  const bool a_ok = mcol < a.cout;
  const int ncol = n0 + 8 * (tid % OpB::CHUNKS);
  const bool b_ok = ncol < a.nc;
  const int tap = b_ok ? ncol / a.cin : 0;
  const int ci = b_ok ? ncol - tap * a.cin : 0;
  const int ta = tap / a.kw, tb = tap - ta * a.kw;
  const int32_t plane = a.oh * a.ow;
  auto dy_at = [&](int32_t p) -> const S* {
    return p < p_end && a_ok ? DY + static_cast<int64_t>(p) * a.cout + mcol : nullptr;
  };
  auto x_at = [&](int32_t p) -> const S* {
    const int32_t n = div_by(p, a.plane_m, a.plane_s);
    const int32_t rem = p - n * plane;
    const int32_t oh = div_by(rem, a.ow_m, a.ow_s), ow = rem - oh * a.ow;
    const int32_t ih = oh * a.sh - a.ph + ta, iw = ow * a.sw - a.pw + tb;
    const bool in = p < p_end && b_ok && ih >= 0 && ih < a.h && iw >= 0 && iw < a.w;
    return in ? X + ((static_cast<int64_t>(n) * a.h + ih) * a.w + iw) * a.cin + ci : nullptr;
  };
  auto load = [&]<int SET>(int kt) {  // (rows past the split are zero, so any tile number will do)
    const int32_t p0 = p_begin + kt * kWK;
    oa.template load<SET>(p0, DY, dy_at);
    ob.template load<SET>(p0, X, x_at);
  };

  f32x4_t sums[1][TM][TN];
  gemm_any::clear(sums);
  const int32_t steps = (p_end - p_begin + kWK - 1) / kWK;
  gemm_any::k_loop<T, OpA, OpB, kWK>(oa, ob, lds, steps, steps, wm * WM, wn * WN, lane, load, load, sums);
  const f32x4_t(&acc)[TM][TN] = sums[0];

  // fp32 partial tile
  float* out = a.part + static_cast<int64_t>(blockIdx.y) * a.cout * a.nc;
  const int g = lane >> 4, r = lane & 15;
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const int col = n0 + wn * WN + j * 16 + r;
      if (col >= a.nc) continue;
#pragma unroll
      for (int x = 0; x < 4; ++x) {
        const int row = m0 + wm * WM + i * 16 + 4 * g + x;
        if (row < a.cout) out[static_cast<int64_t>(row) * a.nc + col] = acc[i][j][x];
      }
    }
}

// dw[co][ci][kh][kw] = round(sum over splits, in order, of part[s][co][(kh*KW + kw)*cin_pad + ci]), ci < cin. One
// thread per workspace column in its natural (co, tap, ci) order, so the split-strided reads of a wave are
// contiguous; the scattered 2-byte writes are the small side.
template <typename T>
__global__ __launch_bounds__(64) void wgrad_reduce_kernel(const float* __restrict__ part, typename Io<T>::storage* __restrict__ dw,
                                                           int32_t splits, int32_t cout, int32_t cin, int32_t cin_pad,
                                                           int32_t taps, int64_t nc, int64_t total) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * 64 + threadIdx.x;
  if (i >= total) return;
  const int32_t ci = static_cast<int32_t>(i % cin_pad);
  const int64_t r = i / cin_pad;
  const int32_t tap = static_cast<int32_t>(r % taps);
  const int32_t co = static_cast<int32_t>(r / taps);
  if (ci >= cin) return;
  const int64_t stride = static_cast<int64_t>(cout) * nc;
  // Sixteen partials in flight per batch, summed in split order (the order does not depend on the batching).
  constexpr int32_t kB = 16;
  float s = 0.0f;
  int32_t k = 0;
  for (; k + kB <= splits; k += kB) {
    float t[kB];
#pragma unroll
    for (int32_t u = 0; u < kB; ++u) t[u] = part[(k + u) * stride + i];
#pragma unroll
    for (int32_t u = 0; u < kB; ++u) s += t[u];
  }
  for (; k < splits; ++k) s += part[k * stride + i];
  dw[(static_cast<int64_t>(co) * cin + ci) * taps + tap] = Io<T>::store(s);
}

template <typename T>
fh_status run_wgrad(const WgradArgs& args, int32_t splits, int32_t cin_real, int32_t kh, void* dw, hipStream_t s) {
  const int wm = wgrad_wm(args.cout);
  const int tiles = ((args.cout + wm - 1) / wm) * args.tiles_n;
  const dim3 grid(static_cast<uint32_t>(tiles), static_cast<uint32_t>(splits));
  if (wm == 128)
    hipLaunchKernelGGL((conv_wgrad_kernel<T, 128>), grid, dim3(kWThreads), 0, s, args);
  else
    hipLaunchKernelGGL((conv_wgrad_kernel<T, 64>), grid, dim3(kWThreads), 0, s, args);
  if (fh_status st = launch_status("conv_wgrad_kernel"); st != FH_OK) return st;
  const int64_t total = static_cast<int64_t>(args.cout) * args.nc;  // every workspace column (co, tap, ci_pad)
  // 64-lane workgroups: the small layers' few thousand columns still spread over every CU
  hipLaunchKernelGGL((wgrad_reduce_kernel<T>), dim3(static_cast<uint32_t>((total + 63) / 64)), dim3(64), 0, s,
                     args.part, static_cast<typename Io<T>::storage*>(dw), splits, args.cout, cin_real, args.cin,
                     kh * args.kw, static_cast<int64_t>(args.nc), total);
  return launch_status("wgrad_reduce_kernel");
}

// ---- no-allocation variant -----------------------------------------------------------------------------------
// The split-K partials of fh_conv2d_wgrad_nhwc_noalloc live in this file-scope device array. Each device the
// library runs on holds its own copy until the process ends. In host code the name `scratch` is only a host-side
// stand-in: its device address is looked up once per device (hipGetSymbolAddress with that device current) and
// only that address is handed to kernels. Nothing in it needs to start at zero: the main kernel writes every
// partial of every split before the reduction reads it.
constexpr int64_t kWgradScratchBytes = int64_t{64} << 20;
constexpr int kScratchMaxDevices = 64;
static __device__ __align__(256) unsigned char scratch[kWgradScratchBytes];

// Calls on one device are ordered through the array: each call's stream first waits for the event the previous
// call recorded after its kernels (on whatever stream that was), and the call records it again after its own.
// g_scratch_mu is held from the wait to the record, so the order is the order in which the host made the calls.
std::mutex g_scratch_mu;
void* g_scratch_ptr[kScratchMaxDevices] = {};
hipEvent_t g_scratch_done[kScratchMaxDevices] = {};

// Set-up, once per device with that device current (g_scratch_mu held): the array's device address and the
// ordering event. No device memory is allocated.
fh_status scratch_of_current_device_locked(int* dev_out, void** out) {
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess) return fail(FH_DEVICE_ERROR, "fh_conv2d_wgrad_nhwc_noalloc: hipGetDevice failed");
  if (dev < 0 || dev >= kScratchMaxDevices)
    return fail(FH_UNIMPLEMENTED, "fh_conv2d_wgrad_nhwc_noalloc: device index above 63");
  if (g_scratch_ptr[dev] == nullptr) {
    void* p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || p == nullptr)
      return fail(FH_DEVICE_ERROR, std::string("fh_conv2d_wgrad_nhwc_noalloc: hipGetSymbolAddress(scratch): ") +
                                       hipGetErrorString(e));
    hipEvent_t ev = nullptr;
    const hipError_t ee = hipEventCreateWithFlags(&ev, hipEventDisableTiming);
    if (ee != hipSuccess)
      return fail(FH_DEVICE_ERROR, std::string("fh_conv2d_wgrad_nhwc_noalloc: hipEventCreateWithFlags: ") +
                                       hipGetErrorString(ee));
    g_scratch_done[dev] = ev;
    g_scratch_ptr[dev] = p;
  }
  *dev_out = dev;
  *out = g_scratch_ptr[dev];
  return FH_OK;
}

}  // namespace
}  // namespace fh

using namespace fh;

extern "C" int64_t fh_conv2d_wgrad_workspace(int32_t dtype, const int64_t geom[12], int32_t cin_pad, int32_t* splits) {
  if (dtype != FH_BF16 && dtype != FH_F16) return -1;
  if (geom == nullptr || geom[11] != 1 || cin_pad % 8 != 0 || cin_pad < geom[1] || geom[4] % 8 != 0) return -1;
  // every extent positive, strides positive, padding non-negative, each 31-bit; the padded input covers the filter
  for (int k = 0; k < 11; ++k)
    if (geom[k] < (k >= 9 ? 0 : 1) || geom[k] > 0x7fffffffLL) return -1;
  if (geom[2] + 2 * geom[9] < geom[5] || geom[3] + 2 * geom[10] < geom[6]) return -1;
  const int64_t oh = (geom[2] + 2 * geom[9] - geom[5]) / geom[7] + 1, ow = (geom[3] + 2 * geom[10] - geom[6]) / geom[8] + 1;
  const int64_t p = geom[0] * oh * ow, nc = geom[5] * geom[6] * cin_pad;
  if (p <= 0 || nc <= 0 || p >= (int64_t{1} << 31) - (int64_t{1} << 23) || nc > (1 << 30)) return -1;  // rows fit int32
  const int64_t wm = wgrad_wm(geom[4]);
  const int64_t tiles = ((geom[4] + wm - 1) / wm) * ((nc + kWN - 1) / kWN);
  // enough workgroups to fill the device twice over, each at least 512 p-rows, the workspace within 256 MiB
  int64_t sp = (2 * 256 + tiles - 1) / tiles;
  sp = std::min<int64_t>(sp, std::max<int64_t>(1, p / 512));
  sp = std::min<int64_t>(sp, std::max<int64_t>(1, (int64_t{256} << 20) / (4 * geom[4] * nc)));
  sp = std::max<int64_t>(1, std::min<int64_t>(sp, 65535));
  if (splits != nullptr) *splits = static_cast<int32_t>(sp);
  return sp * geom[4] * nc * 4;
}

extern "C" fh_status fh_conv2d_wgrad_nhwc(int32_t dtype, const void* x, const void* dy, void* dw, void* workspace,
                                          int64_t workspace_bytes, const int64_t geom[12], int32_t cin_pad, void* stream) {
  int32_t splits = 0;
  const int64_t need = fh_conv2d_wgrad_workspace(dtype, geom, cin_pad, &splits);
  if (need < 0) return fail(FH_UNIMPLEMENTED, "fh_conv2d_wgrad_nhwc: unsupported dtype or geometry");
  if (workspace_bytes < need) return fail(FH_INVALID_ARGUMENT, "fh_conv2d_wgrad_nhwc: workspace too small");
  for (int k = 0; k < 12; ++k)
    if (geom[k] < 0 || geom[k] > 0x7fffffffLL) return fail(FH_INVALID_ARGUMENT, "fh_conv2d_wgrad_nhwc: geometry out of range");
  if (x == nullptr || dy == nullptr || dw == nullptr || workspace == nullptr)
    return fail(FH_INVALID_ARGUMENT, "fh_conv2d_wgrad_nhwc: null pointer");
  WgradArgs a{};
  a.x = x, a.dy = dy, a.part = static_cast<float*>(workspace);
  a.h = static_cast<int32_t>(geom[2]), a.w = static_cast<int32_t>(geom[3]), a.cin = cin_pad;
  a.cout = static_cast<int32_t>(geom[4]), a.kw = static_cast<int32_t>(geom[6]);
  a.sh = static_cast<int32_t>(geom[7]), a.sw = static_cast<int32_t>(geom[8]);
  a.ph = static_cast<int32_t>(geom[9]), a.pw = static_cast<int32_t>(geom[10]);
  a.oh = static_cast<int32_t>((geom[2] + 2 * geom[9] - geom[5]) / geom[7] + 1);
  a.ow = static_cast<int32_t>((geom[3] + 2 * geom[10] - geom[6]) / geom[8] + 1);
  a.nc = static_cast<int32_t>(geom[5] * geom[6] * cin_pad);
  a.tiles_n = (a.nc + kWN - 1) / kWN;
  a.p = geom[0] * a.oh * a.ow;
  a.rows_per_split = ((a.p + splits - 1) / splits + kWK - 1) / kWK * kWK;
  if (a.oh <= 0 || a.ow <= 0) return fail(FH_INVALID_ARGUMENT, "fh_conv2d_wgrad_nhwc: empty output plane");
  make_divider(static_cast<int64_t>(a.oh) * a.ow, a.plane_m, a.plane_s);
  make_divider(a.ow, a.ow_m, a.ow_s);
  if (!(reinterpret_cast<uintptr_t>(x) % 16 == 0 && reinterpret_cast<uintptr_t>(dy) % 16 == 0))
    return fail(FH_INVALID_ARGUMENT, "fh_conv2d_wgrad_nhwc: operands must be 16-byte aligned");
  if ((geom[4] * static_cast<int64_t>(a.nc) + 63) / 64 > 0xffffffffLL ||
      (geom[4] + wgrad_wm(geom[4]) - 1) / wgrad_wm(geom[4]) * static_cast<int64_t>(a.tiles_n) > 0xffffffffLL)
    return fail(FH_INVALID_ARGUMENT, "fh_conv2d_wgrad_nhwc: filter too large for one launch");
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (dtype == FH_BF16) return run_wgrad<bf16_t>(a, splits, static_cast<int32_t>(geom[1]), static_cast<int32_t>(geom[5]), dw, s);
  return run_wgrad<f16_t>(a, splits, static_cast<int32_t>(geom[1]), static_cast<int32_t>(geom[5]), dw, s);
}

extern "C" fh_status fh_conv2d_wgrad_nhwc_noalloc(int32_t dtype, const void* x, const void* dy, void* dw,
                                                  const int64_t geom[12], int32_t cin_pad, void* stream) {
  const int64_t need = fh_conv2d_wgrad_workspace(dtype, geom, cin_pad, nullptr);
  if (need < 0) return fail(FH_UNIMPLEMENTED, "fh_conv2d_wgrad_nhwc_noalloc: unsupported dtype or geometry");
  if (need > kWgradScratchBytes)
    return fail(FH_INVALID_ARGUMENT, "fh_conv2d_wgrad_nhwc_noalloc: the split-K partials need " + std::to_string(need) +
                                         " bytes, above the " + std::to_string(kWgradScratchBytes) +
                                         "-byte no-allocation scratch (use fh_conv2d_wgrad_nhwc with a workspace)");
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  void* ws = nullptr;
  int dev = -1;
  if (fh_status st = scratch_of_current_device_locked(&dev, &ws); st != FH_OK) return st;
  // Under graph capture the graph's own dependencies order the work (an event recorded outside the capture is not
  // waited on there): overlapping replays of such graphs on one device race.
  hipStream_t s = static_cast<hipStream_t>(stream);
  hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
  FH_HIP_CHECK(hipStreamIsCapturing(s, &cap));
  const bool order = cap == hipStreamCaptureStatusNone;
  if (order) FH_HIP_CHECK(hipStreamWaitEvent(s, g_scratch_done[dev], 0));
  if (fh_status st = fh_conv2d_wgrad_nhwc(dtype, x, dy, dw, ws, need, geom, cin_pad, stream); st != FH_OK) return st;
  if (order) FH_HIP_CHECK(hipEventRecord(g_scratch_done[dev], s));
  return FH_OK;
}
