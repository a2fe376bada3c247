// Conv2d forward on MFMA for any ungrouped geometry, NCHW (fh_conv_any.hip).
#pragma once

#include "fh_conv_direct.h"

namespace fh {

// Launches the kernel and returns true, with the launch's status in *status; false (and nothing launched) for a geometry
// it does not accept (groups, or sizes past 2^30 elements) or that one thread per output is faster for (few output channels).
bool conv_any_try_launch(int32_t dtype, const void* x, const void* w, const void* bias, void* y, const ConvGeom& geom,
                         const ConvEpilogue& epilogue, hipStream_t stream, fh_status* status);

}  // namespace fh
