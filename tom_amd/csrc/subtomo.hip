// Batched subtomogram scoring (gfx950).
//
// Reference semantics: tom_mex_corr3d 'peak' -> tom::corr3d_batch ->
// tom::corr3d_single with reapply_mask_after_wedge = true ->
// CorrelationHandlerPeaks::process
// (Oscar3/c++Picker/src/mex/tom_mex_corr3d.cpp:639,
//  src/tom/corr/corr.cpp:969-1210, 1217-1400,
//  src/tom/corr/correlation_handler.cpp:96-120), with a per-particle angle
// list (the local search of av3/alignment/av3_tomomatch.m:173-224).
//
// Per particle p (box B) and orientation a:
//   t  = rot(T_B, a)                        (rot3d arithmetic)
//   t' = norm_mask(t, M)                    (volume_fcn.cpp:168-247, non-boolean)
//   Tf = FFT(t'), DC = 0; Tw = Tf . W_p, DC = 0       (SimpleWedge, cutoff (B-1)/2)
//   tw = c2r(Tw) (unnormalised); tw' = norm_mask_bool(tw, M) -> var_t; Tw = FFT(tw')
//   template wedge W_T of box B, turned with the template (corr.cpp:1086-1111):
//   Pw = P_p . W_T(a), DC = 0; pw = c2r(Pw); pw' = norm_mask_bool(pw, M) -> var_p;
//   Pw = FFT(pw')
//   C  = conj(Tw) . Pw, DC = 0;  c = c2r(C) / (sqrt(var_p var_t) B^6)
//   peak of c over mask_cc != 0, first in x-fastest order; keep strictly better
// Without a particle wedge Tw = Tf and var_t is norm_mask's variance of t';
// without a template wedge Pw = P_p and var_p is the particle's norm_mask variance.
//
// Design. Items are (particle, orientation) pairs, grouped by box and cut
// into chunks of whole particles. Each step is one launch over the chunk with
// one z plane (x and y transforms) or 64 half-spectrum columns (z transform)
// of one item per block, so every launch has thousands of blocks and the
// items' half spectra stream through the memory-side cache; the spectral products, wedges and
// mean removals sit between the forward and inverse z transforms, the re-mask
// between the inverse and forward transforms of its plane. The mask's mean
// subtraction of norm_mask is linear, so it is applied in Fourier space with
// precomputed FFT(M) and FFT(M != 0) instead of an extra real-space pass.
//
// Transforms. A length B = 8 RB (RB = 8, 6, 4) takes two steps with the data
// in registers and one exchange through LDS; what one transform leaves in a
// thread is what the next one takes from it. Real planes are transformed two
// rows at a time (row l + i row l + B/2), the kx = 0 and kx = B/2 columns as
// one. 3,321 items of 64^3 (1.08 MB of half spectrum each), in ms, in chunks
// of 2 GiB with whole complex lines through LDS stages, and now: template load
// 4.8 and 2.9, z with the particle wedge 3.0 and 1.25, re-mask 5.8 and 1.95, z
// to the correlation 3.3 and 1.63, peak 3.6 and 1.01. The z steps run at 5.8
// and 4.4 TB/s, the re-mask at 3.7; the load is held by its instructions (85 a
// voxel, the vector units 66% busy) and gathers (address units 70% busy).
#include <cfloat>
#include <cmath>
#include <vector>

#include "fused_dev.h"
#include "rotate.h"
#include "rotate_dev.h"
#include "pool.h"
#include "subtomo.h"

namespace tomhip {

namespace {

// Spectra of a chunk: as many as the 256 MB memory-side cache holds, since
// each step reads what the one before wrote. 384 particles of 32^3 to 64^3, 16
// orientations each, sum of kernels: 2 GiB 17.3 ms, 256 MB 14.9, 192 MB 15.1,
// 128 MB 15.6 (more launches, each with its last blocks alone).
constexpr long kChunkBytes = 256L << 20;

// SimpleWedge turned with the template (src/tom/core/wedge.cpp:149-224,
// cutoff branch): the reference evaluates its r2c half (z index <= B/2) at
// grid index (x, y, z) -> (xs, ys, zs) = ((x + B/2) mod B, ...) through the
// float affine map P (3 x 4, row-major, rotation and -P.centre), in this
// order of float operations. This layout stores kx <= B/2 for every kz, so an
// entry with kz > B/2 takes the value of its Hermitian partner, as the
// reference's half spectrum implies.
template <int B>
__device__ __forceinline__ bool wedge_keep_rot(int kx, int ky, int kz, const float* P, float tan_a) {
  int x = kx, y = ky, z = kz;
  if (kz > B / 2) {
    x = (B - kx) % B;
    y = (B - ky) % B;
    z = B - kz;
  }
  const float xs = (float)((x + B / 2) % B), ys = (float)((y + B / 2) % B), zs = (float)((z + B / 2) % B);
  float xt = P[2] * zs + P[3];
  float yt = P[6] * zs + P[7];
  float zt = P[10] * zs + P[11];
  xt = P[1] * ys + xt;
  yt = P[5] * ys + yt;
  zt = P[9] * ys + zt;
  const float x_ = P[0] * xs + xt;
  const float y_ = P[4] * xs + yt;
  const float z_ = fabsf(P[8] * xs + zt);
  const float cutoff = (float)((B - 1) / 2);
  const float r = sqrtf((x_ * x_ + y_ * y_) + z_ * z_);
  return (r <= cutoff) && ((z_ < 1e-4f) || (tan_a <= fabsf(x_) / z_));
}

// SimpleWedge (cutoff branch) at unshifted frequency index (kx<=B/2, ky, kz),
// float arithmetic as src/tom/core/wedge.cpp:188-196.
template <int B>
__device__ __forceinline__ bool wedge_keep(int kx, int ky, int kz, float tan_a) {
  const float fx = (float)kx;
  const float fy = (float)(ky <= B / 2 ? ky : ky - B);
  const float fz = fabsf((float)(kz <= B / 2 ? kz : kz - B));
  const float cutoff = (float)((B - 1) / 2);
  const float r = sqrtf(fx * fx + fy * fy + fz * fz);
  return (r <= cutoff) && ((fz < 1e-4f) || (tan_a <= fabsf(fx) / fz));
}

// ---------------------------------------------------------------- transforms
template <int B>
struct Geo {
  static constexpr int RB = B / 8, LN = B / 2;  // second factor; packed lines of a plane, packed columns
  static constexpr int XH1 = B / 2 + 1;
  static constexpr long N3 = (long)B * B * B;
  static constexpr long PL = (long)B * XH1;  // one kz plane of the half spectrum
  static constexpr long NH = PL * B;
  static constexpr int TP = 4 * B;           // threads of a plane: 8 per line
  };

template <int R, int DIR>
__device__ __forceinline__ void dft(c32* v) {
  if constexpr (R == 6) {  // 2 x 3: k = k1 + 2 k2
    c32 e[3], o[3];
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      e[j] = v[j] + v[j + 3];
      o[j] = v[j] - v[j + 3];
    }
    const float h = 0.86602540378443864676f;  // exp(DIR 2 pi i / 6) = 1/2 + DIR i h
    o[1] = cmul(o[1], mk(0.5f, DIR * h));
    o[2] = cmul(o[2], mk(-0.5f, DIR * h));
    Bfly<float, 3, DIR>::run(e);
    Bfly<float, 3, DIR>::run(o);
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      v[2 * k] = e[k];
      v[2 * k + 1] = o[k];
    }
  } else {
    Bfly<float, R, DIR>::run(v);
  }
}

// Transforms of length B = 8 RB of the line that the threads (line, q), q < 8,
// share; t: exp(2 pi i q k / B), k < 8; row(k): LDS place of exchange row k
// (B rows) of this line; sync(): before the rows are read.
// split8: threads q < RB hold x[q + RB r] in u, r < 8; on return every thread
// holds X[q + 8 k] in v, k < RB.
// splitR: every thread holds x[q + 8 r] in u, r < RB; on return the threads
// q < RB hold X[q + RB k] in v, k < 8.
// Exchange rows: split8 writes 8 q + k and reads 8 j + q; splitR writes
// 8 k + q, the rows that this thread's split8 read, and reads 8 q + j.
template <int B, int DIR, class ROW, class SYNC>
__device__ __forceinline__ void split8(c32* u, c32* v, const c32* t, int q, const ROW& row, const SYNC& sync) {
  constexpr int RB = B / 8;
  if (q < RB) {
    dft<8, DIR>(u);
    row(8 * q) = u[0];
#pragma unroll
    for (int k = 1; k < 8; ++k) row(8 * q + k) = DIR < 0 ? cmulc(u[k], t[k]) : cmul(u[k], t[k]);
  }
  sync();
#pragma unroll
  for (int j = 0; j < RB; ++j) v[j] = row(8 * j + q);
  dft<RB, DIR>(v);
}
template <int B, int DIR, class ROW, class SYNC>
__device__ __forceinline__ void splitR(c32* u, c32* v, const c32* t, int q, const ROW& row, const SYNC& sync) {
  constexpr int RB = B / 8;
  dft<RB, DIR>(u);
  row(q) = u[0];
#pragma unroll
  for (int k = 1; k < RB; ++k) row(8 * k + q) = DIR < 0 ? cmulc(u[k], t[k]) : cmul(u[k], t[k]);
  sync();
  if (q < RB) {
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = row(8 * q + j);
    dft<8, DIR>(v);
  }
}
__device__ __forceinline__ void block_sync() { __syncthreads(); }
// orders the LDS accesses of one wave (the hardware runs them in order)
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// A plane's threads: lines of x are (lx, qx) with q fastest (neighbouring
// threads take neighbouring voxels; a line's threads are of one wave), columns
// of y (iy, qy) with the column fastest (they take neighbouring entries of a
// half-spectrum row). One LDS area of B rows (an x position or a y one) of LN
// lines or columns, pitch 32, the column XORed with a permutation of the row:
// its upper two bits differ over 4 rows 8 apart and over 4 consecutive rows
// (8 q's by 8 lines of a wave: x), its five bits over 32 consecutive rows (the
// transpose), so that no access takes more turns than its bytes do. A wave's x
// exchanges stay in its own lines' columns: no block barrier.
template <int B>
struct Plane {
  using G = Geo<B>;
  static constexpr int RB = G::RB, LN = G::LN;
  static constexpr int kLds = B * 32 + B;
  int lx, qx, iy, qy;
  const c32* twq;
  c32 *a, *pk;  // the area; the packed column

  __device__ __forceinline__ Plane(c32* lds, const c32* twq_) : twq(twq_), a(lds), pk(lds + B * 32) {
    const int t = threadIdx.x;
    qx = t % 8;
    lx = t / 8;
    iy = t % LN;
    qy = t / LN;
  }
  static __device__ __forceinline__ int at(int r, int c) {
    return r * 32 + (c ^ ((((r ^ (r >> 3)) & 3) << 3) | ((r >> 3) & 3) | (r & 4)));
  }
  // the 8 twiddles of a q
  __device__ __forceinline__ void row_tw(int q, c32* t) const {
    const float4* p = (const float4*)(twq + q * 8);
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const float4 f = p[k];
      t[2 * k] = mk(f.x, f.y);
      t[2 * k + 1] = mk(f.z, f.w);
    }
  }

  // half-spectrum plane -> v[k] = (row lx, row lx + LN) at x = qx + 8 k,
  // unnormalised. SEP: the columns kx = 0 and B/2 by themselves, their real
  // parts kept (a spectrum that is not Hermitian there); otherwise as one.
  template <bool SEP>
  __device__ __forceinline__ void inverse(const c32* Hz, c32* v) {
    auto rowy = [&](int k) -> c32& { return a[at(k, iy)]; };
    c32 t[8], u[8], h[8], w[RB], n[RB];
    row_tw(qy, t);
    if (qy < RB) {
#pragma unroll
      for (int r = 0; r < 8; ++r) {
        u[r] = Hz[(qy + RB * r) * G::XH1 + iy];
        h[r] = Hz[(qy + RB * r) * G::XH1 + (SEP || iy ? iy : LN)];
      }
#pragma unroll
      for (int r = 0; r < 8; ++r)
        if (!SEP && iy == 0) u[r] = mk(u[r].x - h[r].y, u[r].y + h[r].x);
    }
    split8<B, 1>(u, w, t, qy, rowy, block_sync);
    if constexpr (SEP) {
      __syncthreads();
      if (qy < RB && iy == 0) {
#pragma unroll
        for (int r = 0; r < 8; ++r) u[r] = Hz[(qy + RB * r) * G::XH1 + LN];
      }
      split8<B, 1>(u, n, t, qy, rowy, block_sync);
    }
    __syncthreads();
    // line l of the two-row form: P_l + i P_(l + LN) at every kx
#pragma unroll
    for (int k = 0; k < RB / 2; ++k) {
      const int l = qy + 8 * k;
      const c32 p = w[k], s = w[k + RB / 2];
      if (iy == 0) {
        a[at(0, l)] = mk(p.x, s.x);
        a[at(LN, l)] = SEP ? mk(n[k].x, n[k + RB / 2].x) : mk(p.y, s.y);
      } else {
        a[at(iy, l)] = mk(p.x - s.y, p.y + s.x);
        a[at(B - iy, l)] = mk(p.x + s.y, s.x - p.y);
      }
    }
    row_tw(qx, t);
    __syncthreads();
    if (qx < RB) {
#pragma unroll
      for (int r = 0; r < 8; ++r) u[r] = a[at(qx + RB * r, lx)];
    }
    wave_sync();
    split8<B, 1>(u, v, t, qx, [&](int k) -> c32& { return a[at(k, lx)]; }, wave_sync);
  }

  // v[r] = (row lx, row lx + LN) at x = qx + 8 r -> half-spectrum plane. The
  // area's columns lx were last read by this wave, or not at all.
  __device__ __forceinline__ void forward(c32* v, c32* Hz) {
    c32 t[8], u[8], y[RB];
    row_tw(qx, t);
    splitR<B, -1>(v, u, t, qx, [&](int k) -> c32& { return a[at(k, lx)]; }, wave_sync);
    wave_sync();
    if (qx < RB) {
#pragma unroll
      for (int k = 0; k < 8; ++k) a[at(qx + RB * k, lx)] = u[k];
    }
    row_tw(qy, t);
    __syncthreads();
#pragma unroll
    for (int r = 0; r < RB / 2; ++r) {
      const int l = qy + 8 * r;
      if (iy == 0) {
        const c32 A = a[at(0, l)], D = a[at(LN, l)];
        y[r] = mk(A.x, D.x);
        y[r + RB / 2] = mk(A.y, D.y);
      } else {
        const c32 A = a[at(iy, l)], C = a[at(B - iy, l)];
        y[r] = mk(0.5f * (A.x + C.x), 0.5f * (A.y - C.y));
        y[r + RB / 2] = mk(0.5f * (A.y + C.y), 0.5f * (C.x - A.x));
      }
    }
    __syncthreads();
    splitR<B, -1>(y, u, t, qy, [&](int k) -> c32& { return a[at(k, iy)]; }, block_sync);
    if (qy < RB) {
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        const int ky = qy + RB * k;
        if (iy == 0)
          pk[ky] = u[k];
        else
          Hz[ky * G::XH1 + iy] = u[k];
      }
    }
    __syncthreads();
    if (threadIdx.x < B) {  // the packed column back into kx = 0 and kx = B/2
      const int ky = threadIdx.x;
      const c32 g = pk[ky], m = pk[(B - ky) % B];
      Hz[ky * G::XH1] = mk(0.5f * (g.x + m.x), 0.5f * (g.y - m.y));
      Hz[ky * G::XH1 + LN] = mk(0.5f * (g.y + m.y), 0.5f * (m.x - g.x));
    }
  }
};

// ---------------------------------------------------------------- pipeline
//   boxes: FFT(M), FFT(M != 0): load + r2c -> z forward
//   particles: load (V.M, sums) + r2c -> z forward (mean removal) -> Pp
//   template wedge (per item): z inverse of Pp . W_T(a) -> c2r, re-mask, sums,
//       r2c of one plane -> z forward (mean removal) -> Pw
//   per item: load (rot(T).M, sums) + r2c -> [particle wedge: z forward . W_p,
//       z inverse -> c2r, re-mask, sums, r2c] -> z forward, mean removal,
//       conj(Tw) . P, z inverse -> c2r, masked peak per plane -> best
// Per-plane partial sums (FP64) and peaks are reduced over an item's planes by
// one wave, so the results do not depend on scheduling.
struct Chunk {
  SubtomoBox bx;
  int np, A;
  const int32_t* pid;       // [np] particle ids
  const float* particles;   // packed
  const long* poff;         // [P]
  const float* tanw;        // [P] tan of the particle wedge (< 0: none)
  float tan_r;              // tan of the box template's wedge (< 0: none)
  const float* rms;         // [P][A][9]
  const float* wmap;        // [P][A][12]
  c32* H;                   // [max(np A, np)][NH]
  c32* Pp;                  // [np][NH]
  c32* Pw;                  // [np A][NH] (template wedge only)
  double* S;                // [max(np A, np)][B][4] per-plane sums of the step before
  // per particle / item: what the z step subtracts (two factors) and the
  // variance, of the particle, the template, the re-masked particle and template
  float2 *fp, *ft, *fpw, *ftw;
  double *vp, *vt, *vpw, *vtw;
  float* pkv;               // [np A][B]
  int* pki;                 // [np A][B]
  float* sc;                // [np A] score of an item's peak (of all items of the box,
  int* at;                  // [np A] its voxel, INT_MAX: none   from this chunk's first on)
  const c32* twq;           // [8][8] exp(2 pi i q k / B)
  int32_t* best_idx;
  int32_t* best_pos;
  float* best_val;
};

// Block sums of K doubles; the result is valid in thread 0.
template <int K, int NT>
__device__ __forceinline__ void blk_sum(double* v, double* red) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
#pragma unroll
  for (int k = 0; k < K; ++k) {
    double x = v[k];
    for (int o = 32; o > 0; o >>= 1) x += __shfl_xor(x, o, 64);
    if (lane == 0) red[k * (NT / 64) + w] = x;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
#pragma unroll
    for (int k = 0; k < K; ++k) {
      double t = 0;
      for (int i = 0; i < NT / 64; ++i) t += red[k * (NT / 64) + i];
      v[k] = t;
    }
  }
}

// grid (B, count). What a plane is loaded from: particle i of the chunk (v =
// V M), item it = i A + a (v = rot(T, a) M), or the mask of the box (item 0: M,
// item 1: M != 0). Writes the plane's norm_mask sums (not for the mask) and
// its half spectrum H[item].
enum Source { S_PART, S_TMPL, S_MASK };
template <int B, int SRC>
__global__ __launch_bounds__(Geo<B>::TP) void k_b_load(Chunk C) {
  using G = Geo<B>;
  __shared__ c32 lds[Plane<B>::kLds];
  __shared__ double red[4 * (G::TP / 64)];
  const int z = blockIdx.x, item = blockIdx.y;
  Plane<B> pl(lds, C.twq);
  const float* M = C.bx.M + (long)z * B * B;
  double s[4] = {0, 0, 0, 0};
  const float* V = nullptr;
  float rmr[9];
  if (SRC == S_PART) {
    V = C.particles + C.poff[C.pid[item]] + (long)z * B * B;
  } else if (SRC == S_TMPL) {
    const int p = C.pid[item / C.A], a = item % C.A;
    const float* rm = C.rms + ((long)p * C.A + a) * 9;
#pragma unroll
    for (int k = 0; k < 9; ++k) rmr[k] = rm[k];
  }
  float m[2][G::RB];
#pragma unroll
  for (int r = 0; r < G::RB; ++r)
#pragma unroll
    for (int h = 0; h < 2; ++h) m[h][r] = M[(pl.lx + h * G::LN) * B + pl.qx + 8 * r];
  // the norm_mask sums of one voxel over M != 0; its value in the transform
  auto masked = [&](float v, float mk) -> float {
    const double dv = mk != 0.f ? v : 0.f, dm = mk, p = dv * dm;
    s[0] += dv;
    s[1] += p;
    s[2] = fma(p, p, s[2]);
    s[3] = fma(p, dm, s[3]);
    return v * mk;
  };
  c32 v[G::RB];
  if constexpr (SRC == S_TMPL) {
    // two x positions of the two rows at a time: 16 gathers in flight. The
    // rotated template is finite, so outside the mask it need not be known.
#pragma unroll
    for (int r = 0; r < G::RB; r += 2) {
      if (!__any(m[0][r] != 0.f || m[1][r] != 0.f || m[0][r + 1] != 0.f || m[1][r + 1] != 0.f)) {
        v[r] = v[r + 1] = mk(0.f, 0.f);
        continue;
      }
      float w[4];
#pragma unroll
      for (int k = 0; k < 4; ++k)
        w[k] = rot3d_voxel_cube<B>(C.bx.Tc, rmr, pl.qx + 8 * (r + k / 2), pl.lx + (k & 1) * G::LN, z,
                                   m[k & 1][r + k / 2] != 0.f);
#pragma unroll
      for (int k = 0; k < 2; ++k) v[r + k] = mk(masked(w[2 * k], m[0][r + k]), masked(w[2 * k + 1], m[1][r + k]));
    }
  } else {
#pragma unroll
    for (int r = 0; r < G::RB; ++r) {
      if (SRC == S_PART) {
        const int i = pl.lx * B + pl.qx + 8 * r;
        v[r] = mk(masked(V[i], m[0][r]), masked(V[i + G::LN * B], m[1][r]));
      } else {
        v[r] = item == 0 ? mk(m[0][r], m[1][r]) : mk(m[0][r] != 0.f ? 1.f : 0.f, m[1][r] != 0.f ? 1.f : 0.f);
      }
    }
  }
  if (SRC != S_MASK) {
    blk_sum<4, G::TP>(s, red);
    if (threadIdx.x == 0) {
      double* S = C.S + ((long)item * B + z) * 4;
#pragma unroll
      for (int k = 0; k < 4; ++k) S[k] = s[k];
    }
  }
  pl.forward(v, C.H + (long)item * G::NH + (long)z * G::PL);
}

// One wave per item: norm_mask statistics (volume_fcn.cpp:168-247) from the
// per-plane sums {sum v, sum v M, sum v^2 M^2, sum v M^2} over M != 0: mean
// mu1, mean of the masked volume mu2, variance.
__global__ __launch_bounds__(64) void k_b_norm4(const double* S, int B, SubtomoBox bx, float2* f, double* var) {
  const int item = blockIdx.x, lane = threadIdx.x;
  double s[4] = {0, 0, 0, 0};
  if (lane < B) {
#pragma unroll
    for (int k = 0; k < 4; ++k) s[k] = S[((long)item * B + lane) * 4 + k];
  }
#pragma unroll
  for (int k = 0; k < 4; ++k)
    for (int o = 32; o > 0; o >>= 1) s[k] += __shfl_xor(s[k], o, 64);
  if (lane) return;
  const double n = (double)bx.n, numel = (double)B * B * B;
  const double mu1 = s[0] / n, mu2 = (s[1] - mu1 * bx.SM) / n;
  const double q = s[2] - 2.0 * mu1 * s[3] + mu1 * mu1 * bx.SM2;
  f[item] = make_float2((float)mu1, (float)mu2);
  var[item] = (q - n * mu2 * mu2) / numel;
}
// boolean re-mask statistics {sum v, sum v^2} over M != 0: mean, variance
__global__ __launch_bounds__(64) void k_b_norm2(const double* S, int B, SubtomoBox bx, float2* f, double* var) {
  const int item = blockIdx.x, lane = threadIdx.x;
  double t0 = 0, t1 = 0;
  if (lane < B) {
    t0 = S[((long)item * B + lane) * 4];
    t1 = S[((long)item * B + lane) * 4 + 1];
  }
  for (int o = 32; o > 0; o >>= 1) {
    t0 += __shfl_xor(t0, o, 64);
    t1 += __shfl_xor(t1, o, 64);
  }
  if (lane) return;
  const double n = (double)bx.n, numel = (double)B * B * B;
  const double mb = t0 / n;
  f[item] = make_float2((float)mb, 0.f);
  var[item] = (t1 - n * mb * mb) / numel;
}

enum ZMode { Z_MASK, Z_PART, Z_WEDGE, Z_FINAL, Z_WREF };

// grid (ceil(PL / 64), count), 512 threads: 64 half-spectrum columns of one
// item, a column per lane; z forward transform, the mode's product, then
// (Z_WEDGE, Z_FINAL) the z inverse back to H or (Z_MASK, Z_PART, Z_WREF) the
// forward result to dst.
template <int B, int MODE>
__global__ __launch_bounds__(512) void k_b_z(Chunk C, c32* dst) {
  using G = Geo<B>;
  constexpr int RB = G::RB, XH1 = G::XH1;
  __shared__ c32 buf[B * 64];
  const int lane = threadIdx.x & 63, q = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int item = blockIdx.y, col = blockIdx.x * 64 + lane;
  const bool in = col < (int)G::PL;
  const int ci = (MODE == Z_PART) ? item : item / C.A;  // chunk particle index
  const float tan_a = MODE == Z_MASK ? -1.f : C.tanw[C.pid[ci]];
  const bool wedge = tan_a >= 0.f;
  if (MODE == Z_WEDGE && !wedge) return;  // items of particles without a wedge skip this step
  c32 t[8], u[8], v[RB];
  tw_load<8>(C.twq + q * 8, t);
  c32* Hi = C.H + (long)item * G::NH + col;
  if (q < RB) {
#pragma unroll
    for (int r = 0; r < 8; ++r) u[r] = in ? Hi[(q + RB * r) * G::PL] : mk(0.f, 0.f);
  }
  auto row = [&](int k) -> c32& { return buf[k * 64 + lane]; };
  split8<B, -1>(u, v, t, q, row, block_sync);
  if (MODE != Z_MASK) {
    const bool both = MODE == Z_PART || MODE == Z_WEDGE || (MODE == Z_FINAL && !wedge);
    const float2 f = MODE == Z_PART ? C.fp[item] : MODE == Z_WREF ? C.fpw[item] : both ? C.ft[item] : C.ftw[item];
    const c32* Pa = (MODE == Z_FINAL) ? ((C.tan_r >= 0.f) ? C.Pw + (long)item * G::NH : C.Pp + (long)ci * G::NH)
                                      : nullptr;
    const int kx = col % XH1, ky = col / XH1;
    if (in) {
#pragma unroll
      for (int k = 0; k < RB; ++k) {
        const int kz = q + 8 * k;
        const long idx = kz * G::PL + col;
        c32 r = v[k];
        if ((col == 0 && kz == 0) || (MODE == Z_WEDGE && !wedge_keep<B>(kx, ky, kz, tan_a))) {
          r = mk(0.f, 0.f);
        } else {
          const c32 fb = C.bx.FB[idx];
          if (both) {
            const c32 fm = C.bx.FM[idx];
            r = mk(r.x - f.x * fm.x - f.y * fb.x, r.y - f.x * fm.y - f.y * fb.y);
          } else {  // boolean-mask mean
            r = mk(r.x - f.x * fb.x, r.y - f.x * fb.y);
          }
          if (MODE == Z_FINAL) r = cmulc(Pa[idx], r);  // conj(Tw) . P
        }
        v[k] = r;
      }
    }
  }
  if (MODE == Z_WEDGE || MODE == Z_FINAL) {
    splitR<B, 1>(v, u, t, q, row, block_sync);
    if (q < RB && in) {
#pragma unroll
      for (int r = 0; r < 8; ++r) Hi[(q + RB * r) * G::PL] = u[r];
    }
  } else if (in) {
    c32* d = dst + (long)item * G::NH + col;
#pragma unroll
    for (int k = 0; k < RB; ++k) d[(q + 8 * k) * G::PL] = v[k];
  }
}

// grid (ceil(PL / 64), np A): the particle spectrum times the template's wedge
// turned by the item's orientation (DC 0), z inverse -> H[item]
template <int B>
__global__ __launch_bounds__(512) void k_b_wref(Chunk C) {
  using G = Geo<B>;
  constexpr int RB = G::RB, XH1 = G::XH1;
  __shared__ c32 buf[B * 64];
  const int lane = threadIdx.x & 63, q = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int item = blockIdx.y, col = blockIdx.x * 64 + lane;
  const bool in = col < (int)G::PL;
  const int ci = item / C.A, a = item % C.A, p = C.pid[ci];
  float Pr[12];
#pragma unroll
  for (int k = 0; k < 12; ++k) Pr[k] = C.wmap[((long)p * C.A + a) * 12 + k];
  c32 t[8], u[8], v[RB];
  tw_load<8>(C.twq + q * 8, t);
  const c32* src = C.Pp + (long)ci * G::NH + col;
  if (q < RB) {
#pragma unroll
    for (int r = 0; r < 8; ++r) {
      const int kz = q + RB * r;
      const bool keep = in && !(col == 0 && kz == 0) && wedge_keep_rot<B>(col % XH1, col / XH1, kz, Pr, C.tan_r);
      u[r] = keep ? src[kz * G::PL] : mk(0.f, 0.f);
    }
  }
  split8<B, 1>(u, v, t, q, [&](int k) -> c32& { return buf[k * 64 + lane]; }, block_sync);
  if (!in) return;
  c32* d = C.H + (long)item * G::NH + col;
#pragma unroll
  for (int k = 0; k < RB; ++k) d[(q + 8 * k) * G::PL] = v[k];
}

// grid (B, np A): plane z of H[item] back to real space, boolean re-mask
// (M != 0) with its two sums, and forward again into the same plane. PART: of
// the particle under the template's wedge (every item), else of the template
// under the particle's.
template <int B, bool PART>
__global__ __launch_bounds__(Geo<B>::TP) void k_b_remask(Chunk C) {
  using G = Geo<B>;
  __shared__ c32 lds[Plane<B>::kLds];
  __shared__ double red[2 * (G::TP / 64)];
  const int z = blockIdx.x, item = blockIdx.y;
  if (!PART && C.tanw[C.pid[item / C.A]] < 0.f) return;  // no particle wedge: nothing to re-mask
  Plane<B> pl(lds, C.twq);
  c32* Hz = C.H + (long)item * G::NH + (long)z * G::PL;
  c32 v[G::RB];
  // the turned wedge decides at its cutoff by rounding, not always alike for
  // (0, ky, kz) and its Hermitian partner
  pl.template inverse<PART>(Hz, v);
  const float* M = C.bx.M + (long)z * B * B;
  double t[2] = {0, 0};
#pragma unroll
  for (int r = 0; r < G::RB; ++r) {
    const int x = pl.qx + 8 * r;
    const bool i0 = M[pl.lx * B + x] != 0.f, i1 = M[(pl.lx + G::LN) * B + x] != 0.f;
    v[r] = mk(i0 ? v[r].x : 0.f, i1 ? v[r].y : 0.f);
    t[0] += (double)v[r].x + (double)v[r].y;
    t[1] += (double)v[r].x * (double)v[r].x + (double)v[r].y * (double)v[r].y;
  }
  blk_sum<2, G::TP>(t, red);
  if (threadIdx.x == 0) {
    double* S = C.S + ((long)item * B + z) * 4;
    S[0] = t[0];
    S[1] = t[1];
  }
  pl.forward(v, Hz);
}

// the larger value, the lower voxel among equals
__device__ __forceinline__ void take(float& pv, int& pi, float v, int i) {
  const bool up = (v > pv) | ((v == pv) & (i < pi));
  pv = up ? v : pv;
  pi = up ? i : pi;
}

// grid (B, np A): plane z of the correlation back to real space; its maximum
// over mask_cc != 0 (first in x-fastest order) -> pkv / pki[item][z]
template <int B>
__global__ __launch_bounds__(Geo<B>::TP) void k_b_peak(Chunk C) {
  using G = Geo<B>;
  __shared__ c32 lds[Plane<B>::kLds];
  __shared__ float rv[G::TP / 64];
  __shared__ int ri[G::TP / 64];
  const int z = blockIdx.x, item = blockIdx.y;
  Plane<B> pl(lds, C.twq);
  const float* Mcc = C.bx.Mcc ? C.bx.Mcc + (long)z * B * B : nullptr;
  unsigned keep = ~0u;
  if (Mcc) {
    keep = 0;
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int r = 0; r < G::RB; ++r)
        keep |= (Mcc[(pl.lx + h * G::LN) * B + pl.qx + 8 * r] != 0.f ? 1u : 0u) << (h * 8 + r);
  }
  c32 v[G::RB];
  pl.template inverse<false>(C.H + (long)item * G::NH + (long)z * G::PL, v);
  // a thread's voxels in x-fastest order: the first among equals stays
  float pv = -FLT_MAX;
  int pi = 0x7fffffff;
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int r = 0; r < G::RB; ++r) {
      const float x = h ? v[r].y : v[r].x;
      const bool up = (keep >> (h * 8 + r) & 1u) && (x > pv || (x == pv && pi == 0x7fffffff));
      pv = up ? x : pv;
      pi = up ? z * B * B + (pl.lx + h * G::LN) * B + pl.qx + 8 * r : pi;
    }
  for (int o = 32; o > 0; o >>= 1) {
    const float ov = __shfl_xor(pv, o, 64);
    const int oi = __shfl_xor(pi, o, 64);
    take(pv, pi, ov, oi);
  }
  if ((threadIdx.x & 63) == 0) {
    rv[threadIdx.x >> 6] = pv;
    ri[threadIdx.x >> 6] = pi;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int k = 1; k < G::TP / 64; ++k) take(pv, pi, rv[k], ri[k]);
    C.pkv[(long)item * B + z] = pv;
    C.pki[(long)item * B + z] = pi;
  }
}

// One wave per item: its peak over the planes and the score
// peak / (sqrt(var_p var_t) B^6).
__global__ __launch_bounds__(64) void k_b_score(Chunk C, int B) {
  const int item = blockIdx.x, lane = threadIdx.x, ci = item / C.A;
  float pv = -FLT_MAX;
  int pi = 0x7fffffff;
  if (lane < B) {
    pv = C.pkv[(long)item * B + lane];
    pi = C.pki[(long)item * B + lane];
  }
  for (int o = 32; o > 0; o >>= 1) {
    const float ov = __shfl_xor(pv, o, 64);
    const int oi = __shfl_xor(pi, o, 64);
    take(pv, pi, ov, oi);
  }
  if (lane) return;
  const double numel = (double)B * B * B;
  const double var_p = C.tan_r >= 0.f ? C.vpw[item] : C.vp[ci];
  const double var_t = C.tanw[C.pid[ci]] >= 0.f ? C.vtw[item] : C.vt[item];
  const double den = sqrt(var_p * var_t) * numel * numel;
  const bool ok = pi != 0x7fffffff && den > 0;
  C.sc[item] = ok ? (float)((double)pv / den) : 0.f;
  C.at[item] = ok ? pi : 0x7fffffff;
}

// one thread per particle of the box: the first best orientation
__global__ void k_b_best(Chunk C, int B) {
  const int ci = blockIdx.x * blockDim.x + threadIdx.x;
  if (ci >= C.np) return;
  const int p = C.pid[ci];
  int best = -1, bpos = 0;
  float bestv = 0.f;
  for (int a = 0; a < C.A; ++a) {
    const long item = (long)ci * C.A + a;
    const float val = C.sc[item];
    const int pi = C.at[item];
    if (pi != 0x7fffffff && (best < 0 || val > bestv)) {
      best = a;
      bestv = val;
      bpos = pi;
    }
  }
  C.best_idx[p] = best;
  C.best_val[p] = best >= 0 ? bestv : NAN;
  C.best_pos[3 * p + 0] = best >= 0 ? bpos % B : 0;
  C.best_pos[3 * p + 1] = best >= 0 ? (bpos / B) % B : 0;
  C.best_pos[3 * p + 2] = best >= 0 ? bpos / (B * B) : 0;
}

// template minus its mean (over the whole box, corr.cpp:1283-1289), followed
// by the B^2 + B + 1 zeros that rot3d_voxel_cube reads past its end. part:
// kMeanBlocks partial sums.
constexpr int kMeanBlocks = 64;
__global__ __launch_bounds__(256) void k_mean_part(const float* T, long n, double* part) {
  __shared__ double red[4];
  double s[1] = {0};
  for (long i = (long)blockIdx.x * 256 + threadIdx.x; i < n; i += kMeanBlocks * 256) s[0] += T[i];
  blk_sum<1, 256>(s, red);
  if (threadIdx.x == 0) part[blockIdx.x] = s[0];
}
__global__ __launch_bounds__(256) void k_center(const float* T, long n, long npad, const double* part, float* out) {
  double s = part[threadIdx.x & 63];
  for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
  const float mean = (float)(s / (double)n);
  const long b = (long)blockIdx.x * 256 + threadIdx.x;
  if (b < npad) out[b] = b < n ? T[b] - mean : 0.f;
}

}  // namespace

void simple_wedge_map(const float euler_deg[3], int B, float out[12]) {
  // tom_mex_corr3d converts degrees with a * (PI / 180.) (tom_mex_corr3d.cpp:247-249)
  const double kPi = 3.141592653589793238512808959406186204433;
  const double ang[3] = {(double)euler_deg[0] * (kPi / 180.), (double)euler_deg[2] * (kPi / 180.),
                         (double)euler_deg[1] * (kPi / 180.)};  // {phi, theta, psi}
  const int axes[3] = {2, 0, 2};
  double P[3][3] = {{1, 0, 0}, {0, 1, 0}, {0, 0, 1}};
  for (int k = 0; k < 3; ++k) {
    if (ang[k] - floor(ang[k] / (kPi / 2.)) * (2. * kPi) == 0.) continue;
    const double sa = sin(ang[k]), ca = cos(ang[k]);
    const int i0 = axes[k] == 0 ? 1 : 0, i1 = axes[k] == 2 ? 1 : 2;
    for (int r = 0; r < 3; ++r) {
      const double p0 = P[r][i0], p1 = P[r][i1];
      if (axes[k] == 1) {
        P[r][i0] = p0 * ca + p1 * sa;
        P[r][i1] = -p0 * sa + p1 * ca;
      } else {
        P[r][i0] = p0 * ca - p1 * sa;
        P[r][i1] = p0 * sa + p1 * ca;
      }
    }
  }
  const double c = (double)(float)ceil((B - 1) / 2.);
  for (int r = 0; r < 3; ++r) {
    out[4 * r + 0] = (float)P[r][0];
    out[4 * r + 1] = (float)P[r][1];
    out[4 * r + 2] = (float)P[r][2];
    out[4 * r + 3] = (float)(-(P[r][0] * c + P[r][1] * c + P[r][2] * c));
  }
}

// the [8][8] list exp(2 pi i q k / B)
static const c32* square_list(Twiddles& tw, int B) {
  return tw.list(-(long)B, [&](std::vector<c32>& h) {
    for (int q = 0; q < 8; ++q)
      for (int k = 0; k < 8; ++k) h.push_back(Twiddles::root<float>(B, q * k % B));
  });
}

// whole particles per chunk: their items' spectra within the budget, and at
// most 65,535 items (grid y)
static long chunk_particles(int B, int A, bool wref, long budget) {
  const long nh = (long)B * B * (B / 2 + 1);
  const long per_item = nh * 8L * (wref ? 2 : 1), per_part = nh * 8L;
  return std::max(1L, std::min(budget / (A * per_item + per_part), 65535L / A));
}

template <int B>
static void run_box_chunks(hipStream_t s, Chunk C, const int32_t* d_ids, long nids, bool wref, long budget) {
  using G = Geo<B>;
  const int A = C.A;
  const dim3 pt(G::TP), zt(512), wv(64);
  const unsigned ncolb = (unsigned)((G::PL + 63) / 64);
  // FFT(M), FFT(M != 0), next to each other
  hipLaunchKernelGGL((k_b_load<B, S_MASK>), dim3(B, 2), pt, 0, s, C);
  hipLaunchKernelGGL((k_b_z<B, Z_MASK>), dim3(ncolb, 2), zt, 0, s, C, const_cast<c32*>(C.bx.FM));
  const long npc = chunk_particles(B, A, wref, budget);
  for (long c0 = 0; c0 < nids; c0 += npc) {
    C.np = (int)std::min(npc, nids - c0);
    C.pid = d_ids + c0;
    const unsigned np = (unsigned)C.np, ni = (unsigned)(C.np * A);
    hipLaunchKernelGGL((k_b_load<B, S_PART>), dim3(B, np), pt, 0, s, C);
    hipLaunchKernelGGL(k_b_norm4, dim3(np), wv, 0, s, (const double*)C.S, B, C.bx, C.fp, C.vp);
    hipLaunchKernelGGL((k_b_z<B, Z_PART>), dim3(ncolb, np), zt, 0, s, C, C.Pp);
    if (wref) {
      hipLaunchKernelGGL(k_b_wref<B>, dim3(ncolb, ni), zt, 0, s, C);
      hipLaunchKernelGGL((k_b_remask<B, true>), dim3(B, ni), pt, 0, s, C);
      hipLaunchKernelGGL(k_b_norm2, dim3(ni), wv, 0, s, (const double*)C.S, B, C.bx, C.fpw, C.vpw);
      hipLaunchKernelGGL((k_b_z<B, Z_WREF>), dim3(ncolb, ni), zt, 0, s, C, C.Pw);
    }
    hipLaunchKernelGGL((k_b_load<B, S_TMPL>), dim3(B, ni), pt, 0, s, C);
    hipLaunchKernelGGL(k_b_norm4, dim3(ni), wv, 0, s, (const double*)C.S, B, C.bx, C.ft, C.vt);
    hipLaunchKernelGGL((k_b_z<B, Z_WEDGE>), dim3(ncolb, ni), zt, 0, s, C, (c32*)nullptr);
    hipLaunchKernelGGL((k_b_remask<B, false>), dim3(B, ni), pt, 0, s, C);
    hipLaunchKernelGGL(k_b_norm2, dim3(ni), wv, 0, s, (const double*)C.S, B, C.bx, C.ftw, C.vtw);
    hipLaunchKernelGGL((k_b_z<B, Z_FINAL>), dim3(ncolb, ni), zt, 0, s, C, (c32*)nullptr);
    hipLaunchKernelGGL(k_b_peak<B>, dim3(B, ni), pt, 0, s, C);
    hipLaunchKernelGGL(k_b_score, dim3(ni), wv, 0, s, C, B);
    TOMHIP_CHECK(hipGetLastError());
    C.sc += ni;
    C.at += ni;
  }
  C.sc -= nids * A;
  C.at -= nids * A;
  C.np = (int)nids;
  C.pid = d_ids;
  hipLaunchKernelGGL(k_b_best, dim3((unsigned)((nids + 63) / 64)), wv, 0, s, C, B);
  TOMHIP_CHECK(hipGetLastError());
}

void subtomo_run(Twiddles& tws, hipStream_t s, std::vector<SubtomoBox>& boxes_h, const float* templates_dev,
                 const long* tmpl_off, int64_t P, const std::vector<int32_t>& pbox_h, const float* particles_dev,
                 const long* poff_dev, const float* tan_dev, const float* rms_dev, const std::vector<float>& tanr_h,
                 const float* wref_P_dev, int64_t A, int32_t* best_idx, int32_t* best_pos, float* best_val) {
  const int nbox = (int)boxes_h.size();
  std::vector<void*> owned;
  auto alloc = [&](size_t bytes) {
    void* p = nullptr;
    work_get(&p, bytes, s);
    owned.push_back(p);
    return p;
  };
  try {
    // per box: the centred template; room for FFT(M), FFT(M != 0)
    double* part = (double*)alloc(sizeof(double) * kMeanBlocks);
    for (int k = 0; k < nbox; ++k) {
      SubtomoBox& b = boxes_h[k];
      const long n3 = (long)b.B * b.B * b.B, nh = (long)b.B * b.B * (b.B / 2 + 1);
      const long npad = n3 + (long)b.B * b.B + b.B + 1;
      float* Tc = (float*)alloc(sizeof(float) * npad);
      const float* T = templates_dev + tmpl_off[k];
      hipLaunchKernelGGL(k_mean_part, dim3(kMeanBlocks), dim3(256), 0, s, T, n3, part);
      hipLaunchKernelGGL(k_center, dim3((unsigned)((npad + 255) / 256)), dim3(256), 0, s, T, n3, npad,
                         (const double*)part, Tc);
      TOMHIP_CHECK(hipGetLastError());
      b.Tc = Tc;
      c32* F = (c32*)alloc(sizeof(c32) * 2 * nh);
      b.FM = F;
      b.FB = F + nh;
    }
    // particles of each box, in input order
    std::vector<std::vector<int32_t>> ids(nbox);
    for (int64_t i = 0; i < P; ++i) ids[pbox_h[i]].push_back((int32_t)i);
    std::vector<int32_t> all;
    std::vector<long> first(nbox + 1, 0);
    for (int k = 0; k < nbox; ++k) {
      first[k] = (long)all.size();
      all.insert(all.end(), ids[k].begin(), ids[k].end());
    }
    first[nbox] = (long)all.size();
    int32_t* d_ids = (int32_t*)alloc(sizeof(int32_t) * all.size());
    TOMHIP_CHECK(hipMemcpyAsync(d_ids, all.data(), sizeof(int32_t) * all.size(), hipMemcpyHostToDevice, s));
    // chunk buffers sized once for the largest box of this call
    const long budget = kChunkBytes;
    long maxH = 0, maxPp = 0, maxPw = 0, maxS = 0, maxIt = 0, maxNp = 0, maxAll = 0;
    for (int k = 0; k < nbox; ++k) {
      if (ids[k].empty()) continue;
      const int B = boxes_h[k].B;
      const long nh = (long)B * B * (B / 2 + 1);
      const bool wref = tanr_h[k] >= 0.f;
      const long npc = std::min(chunk_particles(B, (int)A, wref, budget), (long)ids[k].size());
      maxH = std::max(maxH, std::max(npc * A, 2L) * nh);
      maxPp = std::max(maxPp, npc * nh);
      if (wref) maxPw = std::max(maxPw, npc * A * nh);
      maxS = std::max(maxS, npc * A * (long)B);
      maxIt = std::max(maxIt, npc * A);
      maxNp = std::max(maxNp, npc);
      maxAll = std::max(maxAll, (long)ids[k].size() * A);
    }
    Chunk C{};
    C.A = (int)A;
    C.particles = particles_dev;
    C.poff = poff_dev;
    C.tanw = tan_dev;
    C.rms = rms_dev;
    C.wmap = wref_P_dev;
    C.H = (c32*)alloc(sizeof(c32) * maxH);
    C.Pp = (c32*)alloc(sizeof(c32) * maxPp);
    C.Pw = maxPw ? (c32*)alloc(sizeof(c32) * maxPw) : nullptr;
    C.S = (double*)alloc(sizeof(double) * 4 * maxS);
    C.fp = (float2*)alloc(sizeof(float2) * maxNp);
    C.vp = (double*)alloc(sizeof(double) * maxNp);
    float2* f = (float2*)alloc(sizeof(float2) * 3 * maxIt);
    double* d = (double*)alloc(sizeof(double) * 3 * maxIt);
    C.ft = f;
    C.fpw = f + maxIt;
    C.ftw = f + 2 * maxIt;
    C.vt = d;
    C.vpw = d + maxIt;
    C.vtw = d + 2 * maxIt;
    C.pkv = (float*)alloc(sizeof(float) * maxS);
    C.pki = (int*)alloc(sizeof(int) * maxS);
    C.sc = (float*)alloc(sizeof(float) * maxAll);
    C.at = (int*)alloc(sizeof(int) * maxAll);
    C.best_idx = best_idx;
    C.best_pos = best_pos;
    C.best_val = best_val;
    // largest boxes first
    std::vector<int> korder(nbox);
    for (int k = 0; k < nbox; ++k) korder[k] = k;
    std::stable_sort(korder.begin(), korder.end(), [&](int a, int b) { return boxes_h[a].B > boxes_h[b].B; });
    for (int k : korder) {
      if (ids[k].empty()) continue;
      C.bx = boxes_h[k];
      C.tan_r = tanr_h[k];
      const bool wref = tanr_h[k] >= 0.f;
      const long nids = first[k + 1] - first[k];
      C.twq = square_list(tws, C.bx.B);
      if (C.bx.B == 32)
        run_box_chunks<32>(s, C, d_ids + first[k], nids, wref, budget);
      else if (C.bx.B == 48)
        run_box_chunks<48>(s, C, d_ids + first[k], nids, wref, budget);
      else
        run_box_chunks<64>(s, C, d_ids + first[k], nids, wref, budget);
    }
    TOMHIP_CHECK(hipStreamSynchronize(s));
  } catch (...) {
    for (void* p : owned) work_put(p, s);
    throw;
  }
  for (void* p : owned) work_put(p, s);
}

}  // namespace tomhip
