// Float-exact trilinear sample of rot3d (Sptrans/tom_rotatec.c:293-398) for
// one output voxel, gathering from global memory. Contraction is off inside
// so products and sums round like the reference C.
#pragma once
#include <hip/hip_runtime.h>

namespace tomhip {

__device__ __forceinline__ float rot3d_voxel(const float* __restrict__ img, int sx, int sy, int sz,
                                             const float* rm, float px, float py, float pz, int i, int j, int k) {
#pragma clang fp contract(off)
  const float pi = (float)(int)((float)i - px);
  const float pj = (float)(int)((float)j - py);
  const float pk = (float)(int)((float)k - pz);
  const float rx = px + rm[0] * pi + rm[1] * pj + rm[2] * pk;
  if (rx < 0 || rx > (float)(sx - 1)) return 0.f;
  const float ry = py + rm[3] * pi + rm[4] * pj + rm[5] * pk;
  if (ry < 0 || ry > (float)(sy - 1)) return 0.f;
  const float rz = pz + rm[6] * pi + rm[7] * pj + rm[8] * pk;
  if (rz < 0 || rz > (float)(sz - 1)) return 0.f;
  const int fx = (int)rx, fy = (int)ry, fz = (int)rz;
  const float vx2 = rx - (float)fx, vx1 = 1 - vx2;
  const float vy2 = ry - (float)fy, vy1 = 1 - vy2;
  const float vz2 = rz - (float)fz, vz1 = 1 - vz2;
  const int ex = (fx == sx - 1), ey = (fy == sy - 1), ez = (fz == sz - 1);
  const long sxy = (long)sx * sy;
  const long b = fx + (long)fy * sx + (long)fz * sxy;
  const float i0 = ex ? 0.f : img[b + 1];
  const float i1 = ey ? 0.f : img[b + sx];
  const float i2 = (ex || ey) ? 0.f : img[b + sx + 1];
  const float i3 = ez ? 0.f : img[b + sxy];
  const float i4 = (ex || ez) ? 0.f : img[b + sxy + 1];
  const float i5 = (ey || ez) ? 0.f : img[b + sx + sxy];
  const float i6 = (ex || ey || ez) ? 0.f : img[b + sx + sxy + 1];
  const float a = img[b];
  const float AA = a + (i0 - a) * vx2;
  const float BB = i1 * vx1 + i2 * vx2;
  const float CC = i3 * vx1 + i4 * vx2;
  const float DD = i5 * vx1 + i6 * vx2;
  return (AA * vy1 + BB * vy2) * vz1 + (CC * vy1 + DD * vy2) * vz2;
}

// The same sample of a cube of edge B about the centre (B + 1) / 2, from an
// image of finite values followed by B^2 + B + 1 zeros: a corner past the last
// column, row or plane has weight 0 exactly, so whatever finite value it reads
// the sample is the same, and the eight corners are four unconditional 8-byte
// gathers (of x neighbours) from one 32-bit offset. 0 where not wanted.
template <int B>
__device__ __forceinline__ float rot3d_voxel_cube(const float* __restrict__ img, const float* rm, int i, int j,
                                                  int k, bool want) {
#pragma clang fp contract(off)
  typedef float pair __attribute__((ext_vector_type(2), aligned(4)));
  const float c = (float)((B + 1) / 2);
  const float pi = (float)i - c, pj = (float)j - c, pk = (float)k - c;  // whole numbers
  const float rx = c + rm[0] * pi + rm[1] * pj + rm[2] * pk;
  const float ry = c + rm[3] * pi + rm[4] * pj + rm[5] * pk;
  const float rz = c + rm[6] * pi + rm[7] * pj + rm[8] * pk;
  const float last = (float)(B - 1);
  const bool in = want & !((rx < 0) | (rx > last) | (ry < 0) | (ry > last) | (rz < 0) | (rz > last));
  const unsigned fx = (unsigned)(int)rx, fy = (unsigned)(int)ry, fz = (unsigned)(int)rz;
  const float vx2 = __builtin_amdgcn_fractf(rx), vx1 = 1 - vx2;
  const float vy2 = __builtin_amdgcn_fractf(ry), vy1 = 1 - vy2;
  const float vz2 = __builtin_amdgcn_fractf(rz), vz1 = 1 - vz2;
  const unsigned b = in ? fx + B * (fy + B * fz) : 0u;
  const pair p0 = *(const pair*)(img + b), p1 = *(const pair*)(img + (b + B));
  const pair p2 = *(const pair*)(img + (b + B * B)), p3 = *(const pair*)(img + (b + B * B + B));
  const float AA = p0.x + (p0.y - p0.x) * vx2;
  const float BB = p1.x * vx1 + p1.y * vx2;
  const float CC = p2.x * vx1 + p2.y * vx2;
  const float DD = p3.x * vx1 + p3.y * vx2;
  return in ? (AA * vy1 + BB * vy2) * vz1 + (CC * vy1 + DD * vy2) * vz2 : 0.f;
}

}  // namespace tomhip
