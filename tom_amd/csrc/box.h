// The template box's reference weighting (host side of box.hip).
#pragma once
#include <hip/hip_runtime.h>

#include "fft_kernels.h"

namespace tomhip {

// Makes the twiddle lists (an allocation: before a capture).
void box_prepare(Twiddles& tw, int nx, int ny, int nz);

// t <- M .* ifftn(fftn(t) .* wsh) of count boxes of nx x ny x nz (edges up to
// 64, supported lengths); work: as many complex boxes.
void box_filter(Twiddles& tw, hipStream_t s, int count, float* t, c32* work, const float* wsh, const float* mask,
                int nx, int ny, int nz);

}  // namespace tomhip
