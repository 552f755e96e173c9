// Prefill launches shared between their translation units.
#pragma once

#include "si_internal.hpp"

namespace si {

// The skinny form (si_prefill_skinny.hip): 16-row tiles of W, up to 64 tokens
// a workgroup, K split over its waves.  Same operands as launch_prefill.
hipError_t launch_prefill_skinny(int fmt, const void* w, const void* x_bf16, float* y, int64_t m, int64_t rows,
                                 int64_t cols, hipStream_t s);

}  // namespace si
