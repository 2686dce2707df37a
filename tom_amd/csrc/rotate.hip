// Trilinear ZXZ rotation (tom_rotatec semantics) on gfx950.
//
// Reference: Sptrans/tom_rotatec.c rot3d:146-401 (identical arithmetic to
// Oscar3/c++Picker/src/tom/core/rotate.c rot3dlin:719-843). The per-voxel
// arithmetic below follows the reference's float evaluation order exactly and
// is compiled with FP contraction off, so results are bit-identical to it.
//
// Design: each output voxel gathers its eight taps from the source volume,
// which for templates (up to 64^3) stays resident in L2; a wavefront owns a
// small patch, so its taps fall in a few cache lines. A batch of rotations of
// the same volume runs in one launch (grid.z strides over rotations); an
// optional mask multiplies the result (t = rot(T) .* M of the
// template-matching loop).
#include <algorithm>
#include <type_traits>

#include "common.h"
#include "rotate.h"

#pragma clang fp contract(off)

namespace tomhip {

namespace {

constexpr int NT_ROT = 256;

struct RotParams {
  const float* src;
  float* dst;
  const float* rm;      // [nrot][9]: rm00 rm10 rm20 rm01 rm11 rm21 rm02 rm12 rm22
  const float* mask;    // optional, same size as src
  int sx, sy, sz;
  float px, py, pz;
  long dst_stride;      // elements between consecutive rotations in dst
  const long* desc;     // optional graph batch descriptor {batch, first}: rm += batch*rm_step
  long rm_step;
  int nrot;
  const float2* pairs;  // optional x-neighbour pairs of src (src[b], src[b + 1] or 0 in the last column)
};

__global__ void k_pairs_x(const float* src, int sx, long n, float2* pairs) {
  for (long b = (long)blockIdx.x * blockDim.x + threadIdx.x; b < n; b += (long)gridDim.x * blockDim.x)
    pairs[b] = make_float2(src[b], (b % sx) == sx - 1 ? 0.f : src[b + 1]);
}

// A thread takes rz planes of one column of one rotation, a block 16 x 16
// columns (grid: tiles, plane groups, rotations) or, with FLAT, 256 of the
// columns of all plane groups numbered through (grid.x): of a source
// coordinate, px + rm00 i + rm10 j + rm20 k summed in this order, only the last
// sum changes with the plane, and the gathers of RU planes (4, or rz = 1) are
// in flight together. They are unconditional: a tap past the last row or plane
// is read at the row or plane itself and then replaced by 0, and a voxel
// outside reads element 0. A tile's wave, a patch of 16 x 4, keeps its gathers
// near each other whichever way the volume is turned.
// 1,728 rotations of 48^3 with pairs and mask, with a voxel per thread (64-bit
// index divisions, branches per axis) and this: 1.03 and 0.80 ms, bound by the
// gathers. Single 4-byte-aligned loads of the source in place of the pairs,
// and 8 x 8 patches: 0.78 and 0.84 ms.
template <bool PAIRS, int RU, bool FLAT>
__global__ __launch_bounds__(NT_ROT) void k_rotate_direct(RotParams P, int rz_) {
  const int sx = P.sx, sy = P.sy, sz = P.sz, sxy = sx * sy;
  const float px = P.px, py = P.py, pz = P.pz;
  int i, j, k0;
  if constexpr (FLAT) {
    const unsigned q = blockIdx.x * NT_ROT + threadIdx.x, c = q % (unsigned)sxy;
    i = c % (unsigned)sx;
    j = c / (unsigned)sx;
    k0 = (int)(q / (unsigned)sxy) * rz_;
    if (k0 >= sz) return;
  } else {
    const int nbx = (sx + 15) / 16;
    i = blockIdx.x % nbx * 16 + threadIdx.x % 16;
    j = blockIdx.x / nbx * 16 + threadIdx.x / 16;
    k0 = blockIdx.y * rz_;
    if (i >= sx || j >= sy) return;
  }
  const float* img = P.src;
  const float2* pr = P.pairs;
  const float pi = (float)(int)((float)i - px);
  const float pj = (float)(int)((float)j - py);
  const float lx = (float)(sx - 1), ly = (float)(sy - 1), lz = (float)(sz - 1);
  for (int rot = blockIdx.z; rot < P.nrot; rot += gridDim.z) {
    const float* rmp = P.rm + (long)rot * 9 + (P.desc ? P.desc[0] * P.rm_step : 0);
    const float ax = px + rmp[0] * pi + rmp[1] * pj;
    const float ay = py + rmp[3] * pi + rmp[4] * pj;
    const float az = pz + rmp[6] * pi + rmp[7] * pj;
    const float rm20 = rmp[2], rm21 = rmp[5], rm22 = rmp[8];
    float* out = P.dst + (long)rot * P.dst_stride + (long)j * sx + i;
    const float* mask = P.mask ? P.mask + (long)j * sx + i : nullptr;
    for (int kb = k0; kb < min(k0 + rz_, sz); kb += RU) {
      float v[RU];
#pragma unroll
      for (int u = 0; u < RU; ++u) {
        const float pk = (float)(int)((float)(kb + u) - pz);
        const float rx = ax + rm20 * pk, ry = ay + rm21 * pk, rz = az + rm22 * pk;
        const bool in =
            !((rx < 0) | (rx > lx)) & !((ry < 0) | (ry > ly)) & !((rz < 0) | (rz > lz)) & (kb + u < sz);
        const int fx = in ? (int)rx : 0, fy = in ? (int)ry : 0, fz = in ? (int)rz : 0;
        const float vx2 = rx - (float)fx, vx1 = 1 - vx2;
        const float vy2 = ry - (float)fy, vy1 = 1 - vy2;
        const float vz2 = rz - (float)fz, vz1 = 1 - vz2;
        const bool ey = fy == sy - 1, ez = fz == sz - 1;
        const int b = fx + fy * sx + fz * sxy;
        const int b1 = ey ? b : b + sx, b2 = ez ? b : b + sxy, b3 = ez ? b1 : b1 + sxy;
        float2 p0, p1, p2, p3;
        if constexpr (PAIRS) {
          p0 = pr[b];
          p1 = pr[b1];
          p2 = pr[b2];
          p3 = pr[b3];
        } else {
          const int e = fx == sx - 1 ? 0 : 1;
          p0 = make_float2(img[b], img[b + e]);
          p1 = make_float2(img[b1], img[b1 + e]);
          p2 = make_float2(img[b2], img[b2 + e]);
          p3 = make_float2(img[b3], img[b3 + e]);
          p0.y = e ? p0.y : 0.f;
          p1.y = e ? p1.y : 0.f;
          p2.y = e ? p2.y : 0.f;
          p3.y = e ? p3.y : 0.f;
        }
        p1.x = ey ? 0.f : p1.x;
        p1.y = ey ? 0.f : p1.y;
        p2.x = ez ? 0.f : p2.x;
        p2.y = ez ? 0.f : p2.y;
        p3.x = (ey | ez) ? 0.f : p3.x;
        p3.y = (ey | ez) ? 0.f : p3.y;
        const float AA = p0.x + (p0.y - p0.x) * vx2;
        const float BB = p1.x * vx1 + p1.y * vx2;
        const float CC = p2.x * vx1 + p2.y * vx2;
        const float DD = p3.x * vx1 + p3.y * vx2;
        v[u] = in ? (AA * vy1 + BB * vy2) * vz1 + (CC * vy1 + DD * vy2) * vz2 : 0.f;
      }
#pragma unroll
      for (int u = 0; u < RU; ++u) {
        if (kb + u < sz) {
          const long o = (long)(kb + u) * sxy;
          out[o] = mask ? v[u] * mask[o] : v[u];
        }
      }
    }
  }
}

}  // namespace

// Rotation matrix exactly as rot3d builds it (tom_rotatec.c:146-291): exact
// cos/sin for the 16 table angles, else cos/sin in double of the float-rounded
// radian value; products in float.
static void cossin_ref(float deg, float* c, float* s) {
  static const float tab[16] = {0, 30, 45, 60, 90, 120, 135, 150, 180, 210, 225, 240, 270, 300, 315, 330};
  const float tc[16] = {1.0f, (float)(sqrt(3.0) / 2), (float)(sqrt(2.0) / 2), 0.5f, 0.0f, -0.5f,
                        (float)(-sqrt(2.0) / 2), (float)(-sqrt(3.0) / 2), -1.0f, (float)(-sqrt(3.0) / 2),
                        (float)(-sqrt(2.0) / 2), -0.5f, 0.0f, 0.5f, (float)(sqrt(2.0) / 2), (float)(sqrt(3.0) / 2)};
  const float ts[16] = {0.0f, 0.5f, (float)(sqrt(2.0) / 2), (float)(sqrt(3.0) / 2), 1.0f, (float)(sqrt(3.0) / 2),
                        (float)(sqrt(2.0) / 2), 0.5f, 0.0f, -0.5f, (float)(-sqrt(2.0) / 2),
                        (float)(-sqrt(3.0) / 2), -1.0f, (float)(-sqrt(3.0) / 2), (float)(-sqrt(2.0) / 2), -0.5f};
  for (int i = 0; i < 16; ++i)
    if (tab[i] == deg) {
      *c = tc[i];
      *s = ts[i];
      return;
    }
  const double kPi = 3.14159265358979323846264338327950288419716939937510;
  const float rad = (float)(deg * kPi / 180);
  *c = (float)cos((double)rad);
  *s = (float)sin((double)rad);
}

void rotmat_ref(const float* euler, int neuler, float* rm) {
  if (neuler != 3) {
    for (int i = 0; i < 9; ++i) rm[i] = euler[i];
    return;
  }
  float cphi, sphi, cpsi, spsi, cthe, sthe;
  cossin_ref(euler[0], &cphi, &sphi);
  cossin_ref(euler[1], &cpsi, &spsi);
  cossin_ref(euler[2], &cthe, &sthe);
  // volatile temporaries pin the float rounding of every product
  volatile float t;
  t = cpsi * cphi; float a = t; t = cthe * spsi; t = t * sphi; rm[0] = a - t;
  t = spsi * cphi; a = t; t = cthe * cpsi; t = t * sphi; rm[1] = a + t;
  t = sthe * sphi; rm[2] = t;
  t = -cpsi * sphi; a = t; t = cthe * spsi; t = t * cphi; rm[3] = a - t;
  t = -spsi * sphi; a = t; t = cthe * cpsi; t = t * cphi; rm[4] = a + t;
  t = sthe * cphi; rm[5] = t;
  t = sthe * spsi; rm[6] = t;
  t = -sthe * cpsi; rm[7] = t;
  rm[8] = cthe;
}

namespace {

// rot2d of Sptrans/tom_rotatec.c:49-142 (the gateway's 2D branch): bilinear,
// inverse-mapped, in the reference's float order. The pixel coordinates
// pi, pj come from host tables because the reference accumulates them by
// repeated float increments from -px, -py.
__global__ __launch_bounds__(NT_ROT) void k_rotate2d(const float* __restrict__ img, float* __restrict__ out,
                                                     long sx, long sy, const float* __restrict__ tab,
                                                     float rm00, float rm01, float rm10, float rm11, float px,
                                                     float py) {
  const long n = sx * sy;
  for (long idx = (long)blockIdx.x * NT_ROT + threadIdx.x; idx < n; idx += (long)gridDim.x * NT_ROT) {
    const long i = idx % sx, j = idx / sx;
    const float pi = tab[i], pj = tab[sx + j];
    const long sx_1 = sx - 1, sy_1 = sy - 1;
    const float r_x = px + rm00 * pi + rm10 * pj;
    if (r_x < 0 || r_x > (float)sx_1) {
      out[idx] = 0.f;
      continue;
    }
    const float r_y = py + rm01 * pi + rm11 * pj;
    if (r_y < 0 || r_y > (float)sy_1) {
      out[idx] = 0.f;
      continue;
    }
    const long floorx = (long)r_x;
    const float vx2 = r_x - (float)floorx;
    const long floory = (long)r_y;
    const float vy2 = r_y - (float)floory;
    const float* p = img + floorx + sx * floory;
    const bool inx = r_x < (float)(sx - 1);
    const float a0 = p[0];
    const float AA = inx ? a0 + (p[1] - a0) * vx2 : a0;
    float BB = 0.f;
    if (r_y < (float)(sy - 1)) {
      const float b0 = p[sx];
      BB = inx ? b0 + (p[sx + 1] - b0) * vx2 : b0;
    }
    out[idx] = AA + (BB - AA) * vy2;
  }
}

}  // namespace

void rotmat2d_ref(const float* phi_or_R, int n, float* rm) {
  if (n == 4) {  // rm00 rm10 rm01 rm11, as the gateway reads a 2x2 matrix
    rm[0] = phi_or_R[0];
    rm[1] = phi_or_R[1];
    rm[2] = phi_or_R[2];
    rm[3] = phi_or_R[3];
    return;
  }
  const double kPi = 3.14159265358979323846264338327950288419716939937510;
  const float phi = (float)((double)phi_or_R[0] * kPi / 180);
  rm[0] = (float)cos((double)phi);   // rm00
  rm[1] = (float)sin((double)phi);   // rm10
  rm[2] = (float)-sin((double)phi);  // rm01
  rm[3] = (float)cos((double)phi);   // rm11
}

void launch_rotate2d(const float* src, float* dst, long sx, long sy, const float* tab_dev, const float rm[4],
                     float px, float py, hipStream_t stream) {
  const long n = sx * sy;
  const long bx = std::min((n + NT_ROT - 1) / NT_ROT, 65535L * 16);
  hipLaunchKernelGGL(k_rotate2d, dim3((unsigned)bx), dim3(NT_ROT), 0, stream, src, dst, sx, sy, tab_dev, rm[0],
                     rm[2], rm[1], rm[3], px, py);
  TOMHIP_CHECK(hipGetLastError());
}

void make_x_pairs(const float* src, int sx, long n, float2* pairs, hipStream_t stream) {
  hipLaunchKernelGGL(k_pairs_x, dim3((unsigned)std::min((n + NT_ROT - 1) / NT_ROT, 65535L)), dim3(NT_ROT), 0, stream,
                     src, sx, n, pairs);
  TOMHIP_CHECK(hipGetLastError());
}

void launch_rotate(const float* src, float* dst, const float* rm_dev, int nrot, const float* mask, int sx,
                   int sy, int sz, float px, float py, float pz, long dst_stride, hipStream_t stream,
                   const long* desc, long rm_step, const float2* pairs) {
  RotParams P;
  P.src = src;
  P.dst = dst;
  P.rm = rm_dev;
  P.mask = mask;
  P.sx = sx;
  P.sy = sy;
  P.sz = sz;
  P.px = px;
  P.py = py;
  P.pz = pz;
  P.dst_stride = dst_stride;
  P.desc = desc;
  P.rm_step = rm_step;
  P.nrot = nrot;
  P.pairs = pairs;
  // Tiles of 16 x 16 columns where the tiles are full, and for volumes that an
  // XCD's L2 does not hold (there the patch matters more than idle lanes);
  // otherwise the columns numbered through, so that no lane is idle. 6 million
  // voxels with pairs, in us, a voxel per thread / tiles / numbered: 17^3 36 /
  // 74 / 34, 24^3 36 / 44 / 28, 40^3 35 / 33 / 33, 44^3 34 / 31 / 33, 48^3 34 /
  // 31 / 34, 50^3 36 / 50 / 35, 60^3 32 / 35 / 31, 64^3 34 / 30 / 33; 10 million
  // without: 100^3 241 / 200 / 198, 112^3 379 / 264 / 284.
  const long sxy = (long)sx * sy, plane = (long)((sx + 15) / 16) * ((sy + 15) / 16);
  const double full = sxy / (256.0 * plane);
  const bool flat = full < 0.95 && (full < 0.5 || sxy * sz <= (1L << 20)) && sxy * sz < (1L << 31);
  auto blocks = [&](int rz) {
    const long groups = (sz + rz - 1) / rz;
    return flat ? (sxy * groups + NT_ROT - 1) / NT_ROT : plane * groups;
  };
  // 8 planes a thread, one where the blocks are few (batches of 16, 4 planes
  // and one, in us: 24^3 7.7 and 6.9, 16^3 7.1 and 6.1), the planes, or, of
  // numbered columns, the share of threads that have a whole column (12^3 41
  // and 33, 17^3 41 and 34, 20^3 30 and 34) or where a wave's columns leave
  // its plane's neighbourhood (60^3 36 and 31)
  int rz = sz >= 3 && blocks(8) * nrot >= 2048 ? 8 : 1;
  if (flat && (sxy * sz < 0.75 * 8 * NT_ROT * blocks(8) || (sxy > 1400 && sz > 8))) rz = 1;
  while (!flat && (sz + rz - 1) / rz > 65535) rz *= 2;
  const dim3 grid((unsigned)(flat ? blocks(rz) : plane), flat ? 1u : (unsigned)((sz + rz - 1) / rz),
                  (unsigned)std::min(nrot, 65535));
  auto go = [&](auto pairs_c, auto ru, auto flat_c) {
    hipLaunchKernelGGL((k_rotate_direct<decltype(pairs_c)::value, decltype(ru)::value, decltype(flat_c)::value>), grid,
                       dim3(NT_ROT), 0, stream, P, rz);
  };
  auto with = [&](auto pairs_c, auto flat_c) {
    rz > 1 ? go(pairs_c, std::integral_constant<int, 4>{}, flat_c) : go(pairs_c, std::integral_constant<int, 1>{}, flat_c);
  };
  auto on = [&](auto pairs_c) { flat ? with(pairs_c, std::true_type{}) : with(pairs_c, std::false_type{}); };
  pairs ? on(std::true_type{}) : on(std::false_type{});
  TOMHIP_CHECK(hipGetLastError());
}

}  // namespace tomhip
