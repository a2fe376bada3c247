// fp32 GEMMs on the bf16 matrix cores: three-plane split operands, eight products (see fh_gemm_any.h).
#include <algorithm>
#include <cmath>

#include "fh_gemm_any.h"

namespace fh {
namespace {

template <bool TA, bool TB>
fh_status dispatch(const GemmArgs& args, int64_t batch, hipStream_t stream) {
  const double cus = device_cu_count();
  // The tile of the least estimated time. Costs are us per k32 of one round of tiles over the CUs, measured on MI355X over M,
  // N, K from 64 to 4096: a 128x128 tile costs 1.7 (2048^3: 109 us, 137 on 64x64 and 180 on 32x64), a 64x64 one 0.53, and
  // 0.82 where there is one per CU, whose loads, conversions and barriers then lie bare (1024^3: 26.2 us, 51.6 on 128x128);
  // 32x64 tiles fill a CU count that 64x64 ones leave idle (512^3: 10.0 us against 14.4; 64x4096x4096: 59 against 92) but
  // convert each operand more often. (256x128 tiles spill: 4096^3 1,004 us against 833.) Up to two k32 steps the epilogue is
  // most of the time, and smaller tiles overlap theirs better: 4096x8x4096 25.1 us on 64x64 against 27.7 on 128x128.
  const auto rounds = [&](int64_t bm, int64_t bn) {
    return std::ceil(static_cast<double>(((args.M + bm - 1) / bm) * ((args.N + bn - 1) / bn) * batch) / cus);
  };
  const double c128 = args.K <= 64 ? HUGE_VAL : 1.7 * rounds(128, 128), c64 = std::max(0.82, 0.53 * rounds(64, 64));
  const double c32 = TA ? HUGE_VAL : std::max(0.5, 0.42 * rounds(32, 64));  // (32 rows are no whole k row in LDS)
  if constexpr (!TA) {
    if (c32 <= std::min(c64, c128)) return gemm_any::launch<float, 32, 64, 64, 2, 2, TA, TB>(args, batch, stream);
  }
  if (c64 <= c128) return gemm_any::launch<float, 64, 64, 32, 2, 2, TA, TB>(args, batch, stream);
  return gemm_any::launch<float, 128, 128, 32, 2, 4, TA, TB>(args, batch, stream);
}

}  // namespace

bool gemm_f32_try_launch(const GemmArgs& args, int64_t batch, hipStream_t stream, fh_status* status) {
  if (!gemm_any::accepts(args, batch) || (args.trans_a && args.trans_b)) return false;
  *status = args.trans_a   ? dispatch<true, false>(args, batch, stream)
            : args.trans_b ? dispatch<false, true>(args, batch, stream)
                           : dispatch<false, false>(args, batch, stream);
  return true;
}

}  // namespace fh
