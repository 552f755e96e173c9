// Matrix-vector launches shared between their translation units.
#pragma once

#include "si_internal.hpp"

namespace si {

constexpr int MAX_SEGS = 8;   // products of one launch

// The streaming kernel (si_gemv_stream.hip) over n <= MAX_SEGS products of
// one format: any whole number of blocks per row, at least 32 columns,
// weights at even addresses, no input transform.
hipError_t launch_gemv_stream(const GemvOp* ops, int n, hipStream_t s);

}  // namespace si
