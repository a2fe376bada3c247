// 16-bit GEMMs that the aligned pipeline of fh_gemm16.hip does not take: any K, N and alignment, and either operand
// transposed (see fh_gemm_any.h).
#include <algorithm>
#include <cmath>

#include "fh_gemm_any.h"

namespace fh {
namespace {

template <typename T, bool TA, bool TB>
fh_status dispatch(const GemmArgs& args, int64_t batch, hipStream_t stream) {
  const double cus = device_cu_count();
  const auto tiles = [&](int64_t bm, int64_t bn) {
    return static_cast<double>(((args.M + bm - 1) / bm) * ((args.N + bn - 1) / bn) * batch);
  };
  // The tile of the least estimated time, in us per k64 measured on MI355X (bf16, M, K, N from 64 to 4096): a CU takes a
  // 128x128 tile's step every 0.71 with two of them at hand and 1.2 alone, a 64x64 one's every 0.52 and 0.65 alone, a
  // 32x64 one's every 0.35 and 0.5 alone. us at 4095^3: 189 / 349 / 509; 2049^3: 47 / 65 / 76; 1111x777x1000: 15.4 /
  // 12.5 / 11.8; 513x1001x513: 18.7 / 13.3 / 11.2 (one output per thread, in order, before: 13,100 / 1,450 / 127 / -).
  const double c128 = std::max(1.2, 0.71 * std::ceil(tiles(128, 128) / cus));
  const double c64 = std::max(0.65, 0.52 * tiles(64, 64) / cus);
  const double c32 = TA ? HUGE_VAL : std::max(0.5, 0.35 * tiles(32, 64) / cus);  // (32 rows are no whole k row in LDS)
  if constexpr (!TA) {
    if (c32 <= std::min(c64, c128)) return gemm_any::launch<T, 32, 64, 64, 2, 2, TA, TB>(args, batch, stream);
  }
  if (c64 <= c128) return gemm_any::launch<T, 64, 64, 64, 2, 2, TA, TB>(args, batch, stream);
  // a short K is one to four steps of 32: 2718x64x3180 18.5 us against 20.7 with 64
  if (args.K <= 128) return gemm_any::launch<T, 128, 128, 32, 2, 4, TA, TB>(args, batch, stream);
  return gemm_any::launch<T, 128, 128, 64, 2, 4, TA, TB>(args, batch, stream);
}

template <typename T>
fh_status dispatch(const GemmArgs& args, int64_t batch, hipStream_t stream) {
  if (args.trans_a) return dispatch<T, true, false>(args, batch, stream);
  if (args.trans_b) return dispatch<T, false, true>(args, batch, stream);
  return dispatch<T, false, false>(args, batch, stream);
}

}  // namespace

bool gemm_any16_try_launch(int32_t dtype, const GemmArgs& args, int64_t batch, hipStream_t stream, fh_status* status) {
  if ((dtype != FH_BF16 && dtype != FH_F16) || !gemm_any::accepts(args, batch)) return false;
  if (args.trans_a && args.trans_b) return false;
  *status = dtype == FH_BF16 ? dispatch<bf16_t>(args, batch, stream) : dispatch<f16_t>(args, batch, stream);
  return true;
}

}  // namespace fh
