// fp32 GEMMs on the bf16 matrix cores: three-plane split operands, six products (see fh_gemm_any.h).
#include <algorithm>
#include <cmath>

#include "fh_gemm_any.h"

namespace fh {
namespace {

template <bool TA, bool TB>
fh_status dispatch(const GemmArgs& args, int64_t batch, hipStream_t stream) {
  const double cus = device_cu_count();
  // The tile of the least estimated time. Costs are us per k32 of one round (all CUs holding what they can), measured on
  // MI355X over M, N, K from 64 to 4096: a 256x128 tile costs 2.4 (4096^3: 626 us against 692 on 128x128 tiles), a
  // 128x128 one 1.42 (2048^3: 94 us, 147 on 256x128 and 129 on 64x64); several 64x64 tiles share a CU at 0.5 each, and
  // where there is at most one per CU the latency of its loads, conversions and barriers sets 0.85 (0.78 with 64 k
  // between barriers: 1024^3 25.8 us against 28.0); 32x64 tiles fill a CU count that 64x64 ones leave idle
  // (512^3: 10.8 us against 14.3; 2366x1473x192: 28.3 against 36.7) but convert each operand more often.
  const auto tiles = [&](int64_t bm, int64_t bn) {
    return static_cast<double>(((args.M + bm - 1) / bm) * ((args.N + bn - 1) / bn) * batch);
  };
  const double t64 = tiles(64, 64), t32 = tiles(32, 64);
  const double c256 = 2.4 * std::ceil(tiles(256, 128) / cus), c128 = 1.42 * std::ceil(tiles(128, 128) / cus);
  const double c64 = t64 <= cus ? 0.78 : std::max(0.85, 0.5 * t64 / cus);
  const double c32 = TA ? HUGE_VAL : std::max(0.5, 0.45 * t32 / cus);  // (32 rows are no whole k row in LDS)
  const double best = std::min(std::min(c256, c128), std::min(c64, c32));
  if constexpr (!TA) {
    if (c32 == best) return gemm_any::launch<float, 32, 64, 64, 2, 2, TA, TB>(args, batch, stream);
  }
  if (c64 == best) {
    if (t64 <= cus) return gemm_any::launch<float, 64, 64, 64, 2, 2, TA, TB>(args, batch, stream);
    return gemm_any::launch<float, 64, 64, 32, 2, 2, TA, TB>(args, batch, stream);
  }
  if (c128 == best) return gemm_any::launch<float, 128, 128, 32, 2, 4, TA, TB>(args, batch, stream);
  return gemm_any::launch<float, 256, 128, 32, 4, 2, TA, TB>(args, batch, stream);
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
