// 16-point DFT in registers (two radix-4 steps), for transforms of 256 = 16 x 16.
#pragma once
#include "fft.h"

namespace tomhip {

template <int DIR>
__device__ __forceinline__ c32 w16(int m) {
  // exp(DIR 2 pi i m / 16) for m in [0, 16)
  constexpr float c1 = 0.92387953251128675613f, s1 = 0.38268343236508977173f, h = 0.70710678118654752440f;
  const float cs[5] = {1.f, c1, h, s1, 0.f};  // cos(2 pi m / 16), m = 0..4
  const int q = m & 3, o = m >> 2;            // m = q + 4 o: rotate by o quarter turns
  c32 w = mk(cs[q], cs[4 - q]);
  for (int k = 0; k < o; ++k) w = mk(-w.y, w.x);
  if (DIR < 0) w.y = -w.y;
  return w;
}

template <int DIR>
__device__ __forceinline__ void dft16(c32* v) {
  // n = a + 4 b, k = kb + 4 ka: 4-point DFTs over b (in place: (a, kb) at
  // a + 4 kb), twiddles, 4-point DFTs over a (in place: (kb, ka) at a + 4 kb
  // with a -> ka), then the register renaming to natural order
#pragma unroll
  for (int a = 0; a < 4; ++a) {
    c32 q[4] = {v[a], v[a + 4], v[a + 8], v[a + 12]};
    Bfly<float, 4, DIR>::run(q);
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) v[a + 4 * kb] = (a == 0 || kb == 0) ? q[kb] : cmul(q[kb], w16<DIR>(a * kb));
  }
#pragma unroll
  for (int kb = 0; kb < 4; ++kb) {
    c32 q[4] = {v[4 * kb], v[4 * kb + 1], v[4 * kb + 2], v[4 * kb + 3]};
    Bfly<float, 4, DIR>::run(q);
#pragma unroll
    for (int ka = 0; ka < 4; ++ka) v[4 * kb + ka] = q[ka];
  }
  // X[kb + 4 ka] sits at v[4 kb + ka]: transpose the 4 x 4 register block
#pragma unroll
  for (int kb = 0; kb < 4; ++kb)
#pragma unroll
    for (int ka = kb + 1; ka < 4; ++ka) {
      const c32 t = v[4 * kb + ka];
      v[4 * kb + ka] = v[4 * ka + kb];
      v[4 * ka + kb] = t;
    }
}

// dft16<-1> of v whose elements 2 .. 13 are zero: in the first step every
// 4-point DFT has one nonzero input, so its outputs are that input times
// powers of i (exact), and the rest is as above.
__device__ __forceinline__ void dft16_ends(c32* v) {
#pragma unroll
  for (int a = 0; a < 4; ++a) {
    c32 q[4];
    if (a < 2) {
      q[0] = q[1] = q[2] = q[3] = v[a];
    } else {  // input 3 of 4
      const c32 y = v[a + 12];
      q[0] = y;
      q[1] = mk(-y.y, y.x);
      q[2] = mk(-y.x, -y.y);
      q[3] = mk(y.y, -y.x);
    }
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) v[a + 4 * kb] = (a == 0 || kb == 0) ? q[kb] : cmul(q[kb], w16<-1>(a * kb));
  }
#pragma unroll
  for (int kb = 0; kb < 4; ++kb) Bfly<float, 4, -1>::run(v + 4 * kb);
#pragma unroll
  for (int kb = 0; kb < 4; ++kb)
#pragma unroll
    for (int ka = kb + 1; ka < 4; ++ka) {
      const c32 t = v[4 * kb + ka];
      v[4 * kb + ka] = v[4 * ka + kb];
      v[4 * ka + kb] = t;
    }
}

}  // namespace tomhip
