// The two-kernel inverse of the exhaustive search (host side of fused.hip).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "fft_kernels.h"

namespace tomhip {

// Whether a batch of ka angles over X x Y x Z runs fused_a / fused_bc: lengths
// that have the kernels, and a batch that gains.
bool fused_supported(int X, int Y, int Z, int ka);

// Makes the twiddle lists (an allocation: before a capture).
void fused_prepare(Twiddles& tw, int X, int Y, int Z);

// Ty (kx-tiled: fused_ty_index), Tyn [a][uz][Y], Pn [a][kz][Y] (workspace),
// FI [kz][ky][X/2], FIn [ky][kz] -> Q in the layout that fused_bc reads.
void fused_a(Twiddles& tw, hipStream_t s, const c32* Ty, const c32* Tyn, c32* Pn, const c32* FI, const c32* FIn,
             c32* Q, int X, int Y, int Z, int nz, int ka);
// Angle groups of a batch in fused_bc.
int fused_bc_groups(int X, int Y, int Z, int ka);
// Q -> the running maximum of the ka correlations and its first angle index.
// With pv and pi: of each group of apb angles by itself, the index within the
// batch, [group][N].
void fused_bc(Twiddles& tw, hipStream_t s, const c32* Q, float* maxc, int32_t* argm, int X, int Y, int Z, int ka,
              int first_index, const long* desc, int apb, float* pv, uint8_t* pi);

// Columns of kx that a block of fused_a holds: 64 lines over the first radix
// of the y transform.
__host__ __device__ constexpr int fused_tile(int Y) { return 64 / plan_radix(Y, 0); }
// Position of (ky, kx) in a plane of Ty: the 64 lines of one block of fused_a
// (kx tile, ky = j + r Y / R0 for one j) lie together.
__host__ __device__ constexpr long fused_ty_index(int Y, int ky, int kx) {
  const int R0 = plan_radix(Y, 0), T = 64 / R0, NJ = Y / R0;
  return ((long)(kx / T) * NJ + ky % NJ) * 64 + (ky / NJ) * T + kx % T;
}

}  // namespace tomhip
