// Reference weighting of template boxes: M .* ifftn(fftn(t) .* W) of a batch
// of them (tom_os3_findTemplate.m:264-267 followed by the masking inside
// tom_os3_corr), as complex transforms of edges up to 64.
//
// A line is a lane, wave w takes the butterflies w (mod NW) of all lines of
// the block (fused_dev.h): the stages after the first run on the elements that
// the wave holds in registers, so a transform is one exchange through LDS, and
// its twiddles are scalar loads.
#include "box.h"
#include "fft_io.h"
#include "fused_dev.h"

namespace tomhip {

namespace {

// ---------------------------------------------------------------- uneven planes
// Lines of a block: with 16 a batch of 4 boxes of 40 x 32 x 24 is 192 blocks,
// forward 4.8 us and inverse 4.9; with 102 (32 KB of LDS) 32 blocks, 9.2 and
// 14.9.
constexpr int kBoxLines = 16;
// real lines of L -> complex, forward FFT along x
// Blocks never straddle two templates: every template's line j sits at the
// same place in its block whatever the template's position in the batch, so a
// template's filtered result does not depend on how the batch is grouped.
__device__ __forceinline__ void box_block_lines(long lines_per_vol, int NL, long& l0, long& nl) {
  const long nbt = (lines_per_vol + NL - 1) / NL;
  const long a = blockIdx.x / nbt, b = blockIdx.x % nbt;
  l0 = a * lines_per_vol + b * NL;
  nl = (lines_per_vol - b * NL < NL) ? (lines_per_vol - b * NL) : NL;
}

template <int L>
__global__ __launch_bounds__(NT) void k_box_x_fwd(const float* t, c32* out, long lines_per_vol, const c32* twg) {
  constexpr int NL = kBoxLines;
  __shared__ c32 buf[NL * L];
  __shared__ c32 tw[L];
  load_table<float, L, NT>(tw, twg);
  long l0, nl;
  box_block_lines(lines_per_vol, NL, l0, nl);
  const int nval = (int)(nl * L);
  for (int i = threadIdx.x; i < NL * L; i += NT) buf[i] = mk((i < nval) ? t[l0 * L + i] : 0.f, 0.f);
  __syncthreads();
  lds_fft<float, L, NL, NT, -1, Contig<L>>(buf, tw);
  for (int i = threadIdx.x; i < nval; i += NT) out[l0 * L + i] = buf[i];
}

// inverse FFT along x, real part / n3, times mask -> float
template <int L>
__global__ __launch_bounds__(NT) void k_box_x_inv(const c32* in, float* t, const float* M, long lines_per_vol,
                                                  float inv_n3, const c32* twg) {
  constexpr int NL = kBoxLines;
  __shared__ c32 buf[NL * L];
  __shared__ c32 tw[L];
  load_table<float, L, NT>(tw, twg);
  long l0, nl;
  box_block_lines(lines_per_vol, NL, l0, nl);
  const int nval = (int)(nl * L);
  for (int i = threadIdx.x; i < NL * L; i += NT) buf[i] = (i < nval) ? in[l0 * L + i] : mk(0.f, 0.f);
  __syncthreads();
  lds_fft<float, L, NL, NT, 1, Contig<L>>(buf, tw);
  for (int i = threadIdx.x; i < nval; i += NT) {
    const long g = l0 * L + i;
    const long vox = ((g / L) % lines_per_vol) * L + (g % L);
    t[g] = buf[i].x * inv_n3 * M[vox];
  }
}

// ---------------------------------------------------------------- square planes, z
// One transform of length L of this lane's line, in place between stage 0 and
// the rest: slot(e) is the LDS place of element e. NW waves share a line.
constexpr int NW = 4;
template <int L, int DIR>
struct BoxLine {
  static constexpr int R0 = plan_radix(L, 0), NJ0 = L / R0, P0 = (NJ0 + NW - 1) / NW, EPT = L / NW;
  // stage 0 of a wave takes the elements w (mod NW), those that rest() made
  static constexpr bool kOwn = NJ0 % NW == 0;
  using T = Tail<L, NW>;
  // stage 0; its outputs go to the slots of its inputs, ld(k, e): element e,
  // k = (e - w) / NW where that is whole
  template <class LD, class SLOT>
  static __device__ __forceinline__ void first(int w, const LD& ld, const SLOT& slot) {
    c32 u[P0][R0];
#pragma unroll
    for (int p = 0; p < P0; ++p)
      if (kOwn || w + NW * p < NJ0) {
#pragma unroll
        for (int r = 0; r < R0; ++r) u[p][r] = ld(p + P0 * r, w + NW * p + r * NJ0);
      }
#pragma unroll
    for (int p = 0; p < P0; ++p)
      if (kOwn || w + NW * p < NJ0) {
        Bfly<float, R0, DIR>::run(u[p]);
#pragma unroll
        for (int r = 0; r < R0; ++r) slot(w + NW * p + r * NJ0) = u[p][r];
      }
  }
  // the other stages: x[k] = the transform's element w + NW k
  template <class SLOT>
  static __device__ __forceinline__ void rest(int w, const c32* tw, const SLOT& slot, c32* x) {
    T::template run<DIR>(
        w, tw, [&](int e) { return slot(e / R0 + NJ0 * (e % R0)); }, [&](int k, c32 v) { x[k] = v; });
  }
};

// Both in-plane transforms of one xy plane per block: the plane sits in LDS
// with row pitch L + 1, x lines are rows, y lines are columns. grid: planes of
// all boxes. 1,728 boxes of 48^3, in us, with every stage through LDS and
// this: forward 640 and 524, inverse 730 and 457 (4.4 and 5.0 TB/s). In slabs
// that stay in the memory-side cache between the passes, the three gain 25 us
// and the rotation before them loses 87.
template <int L>
__global__ __launch_bounds__(64 * NW) void k_box_xy_fwd(const float* __restrict__ t, c32* __restrict__ out,
                                                                  const c32* tw) {
  using B = BoxLine<L, -1>;
  constexpr int P = L + 1;
  __shared__ c32 buf[L * P];
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const long base = (long)blockIdx.x * L * L;
  for (int i = threadIdx.x; i < L * L; i += 64 * NW) buf[i / L * P + i % L] = mk(t[base + i], 0.f);
  __syncthreads();
  const bool in = L == 64 || lane < L;
  auto xs = [&](int e) -> c32& { return buf[lane * P + e]; };
  auto ys = [&](int e) -> c32& { return buf[e * P + lane]; };
  c32 v[B::EPT];
  if (in) B::first(w, [&](int, int e) { return xs(e); }, xs);
  __syncthreads();
  if (in) B::rest(w, tw, xs, v);
  __syncthreads();
  if (in) {
#pragma unroll
    for (int k = 0; k < B::EPT; ++k) xs(w + NW * k) = v[k];
  }
  __syncthreads();
  if (in) B::first(w, [&](int, int e) { return ys(e); }, ys);
  __syncthreads();
  if (in) {
    B::rest(w, tw, ys, v);
#pragma unroll
    for (int k = 0; k < B::EPT; ++k) out[base + (w + NW * k) * L + lane] = v[k];
  }
}

// inverse of the above, real part / n3, times mask -> float
template <int L>
__global__ __launch_bounds__(64 * NW) void k_box_xy_inv(const c32* __restrict__ in_, float* __restrict__ t,
                                                                  const float* __restrict__ M, int nz, float inv_n3,
                                                                  const c32* tw) {
  using B = BoxLine<L, 1>;
  constexpr int P = L + 1;
  __shared__ c32 buf[L * P];
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const long base = (long)blockIdx.x * L * L;
  const float* m = M + (long)(blockIdx.x % nz) * L * L;
  const bool in = L == 64 || lane < L;
  auto xs = [&](int e) -> c32& { return buf[lane * P + e]; };
  auto ys = [&](int e) -> c32& { return buf[e * P + lane]; };
  c32 v[B::EPT];
  if (in) B::first(w, [&](int, int e) { return in_[base + e * L + lane]; }, ys);
  __syncthreads();
  if (in) B::rest(w, tw, ys, v);
  __syncthreads();
  if (in) {
#pragma unroll
    for (int k = 0; k < B::EPT; ++k) ys(w + NW * k) = v[k];
  }
  __syncthreads();
  if (in) B::first(w, [&](int, int e) { return xs(e); }, xs);
  __syncthreads();
  if (in) B::rest(w, tw, xs, v);
  __syncthreads();
  float* re = reinterpret_cast<float*>(buf);
  if (in) {
#pragma unroll
    for (int k = 0; k < B::EPT; ++k) re[lane * P + w + NW * k] = v[k].x;
  }
  __syncthreads();
  for (int i = threadIdx.x; i < L * L; i += 64 * NW) t[base + i] = re[i / L * P + i % L] * inv_n3 * m[i];
}

// z: forward, times the weight, inverse, in place. grid (ceil(XY / 64),
// boxes): 64 columns of one box. The inverse's stage 0 takes the elements that
// the wave holds after the product, where its butterflies divide that way. 1,728 boxes of 48^3, in us, with every
// stage through LDS and this: 930 and 538 (5.7 TB/s).
template <int L>
__global__ __launch_bounds__(64 * NW) void k_box_z(c32* __restrict__ data, const float* __restrict__ wsh,
                                                             int XY, const c32* tw) {
  using F = BoxLine<L, -1>;
  using I = BoxLine<L, 1>;
  __shared__ c32 buf[L * 64];
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int col = blockIdx.x * 64 + lane;
  const bool in = col < XY;
  c32* d = data + (long)blockIdx.y * XY * L + col;
  auto slot = [&](int e) -> c32& { return buf[e * 64 + lane]; };
  c32 v[F::EPT];
  F::first(w, [&](int, int e) { return in ? d[(long)e * XY] : mk(0.f, 0.f); }, slot);
  __syncthreads();
  F::rest(w, tw, slot, v);
#pragma unroll
  for (int k = 0; k < F::EPT; ++k) v[k] = scale(v[k], in ? wsh[(w + NW * k) * XY + col] : 0.f);
  __syncthreads();
  if constexpr (I::kOwn) {
    I::first(w, [&](int k, int) { return v[k]; }, slot);
  } else {
#pragma unroll
    for (int k = 0; k < F::EPT; ++k) slot(w + NW * k) = v[k];
    __syncthreads();
    I::first(w, [&](int, int e) { return slot(e); }, slot);
  }
  __syncthreads();
  I::rest(w, tw, slot, v);
  if (!in) return;
#pragma unroll
  for (int k = 0; k < F::EPT; ++k) d[(long)(w + NW * k) * XY] = v[k];
}

// the supported lengths up to 64
template <class F>
void dispatch_box(int L, F&& f) {
  switch (L) {
#define TOMHIP_BOX(n) \
  case n:             \
    f(std::integral_constant<int, n>{}); \
    break;
    TOMHIP_BOX(16)
    TOMHIP_BOX(24)
    TOMHIP_BOX(32)
    TOMHIP_BOX(40)
    TOMHIP_BOX(48)
    TOMHIP_BOX(64)
#undef TOMHIP_BOX
    default: throw Error(ERR_UNSUPPORTED, "unsupported box edge " + std::to_string(L));
  }
}

}  // namespace

void box_prepare(Twiddles& tw, int nx, int ny, int nz) {
  for (int L : {nx, ny, nz}) (void)line_list(tw, L);
}

// count up to 65,535: a grid dimension
static void box_filter_slab(Twiddles& tw, hipStream_t s, int count, float* t, c32* work, const float* wsh,
                            const float* mask, int nx, int ny, int nz) {
  const long n3 = (long)nx * ny * nz;
  const long lpv = (long)ny * nz;  // x lines per box
  const long XY = (long)nx * ny;
  const bool plane = nx == ny;
  if (plane) {
    dispatch_box(nx, [&](auto Lc) {
      constexpr int L = decltype(Lc)::value;
      hipLaunchKernelGGL(k_box_xy_fwd<L>, dim3((unsigned)(count * nz)), dim3(64 * NW), 0, s,
                         (const float*)t, work, line_list(tw, L));
    });
  } else {
    dispatch_box(nx, [&](auto Lc) {
      constexpr int L = decltype(Lc)::value;
      constexpr int NL = kBoxLines;
      hipLaunchKernelGGL(k_box_x_fwd<L>, dim3((unsigned)(count * ((lpv + NL - 1) / NL))), dim3(NT), 0, s,
                         (const float*)t, work, lpv, tw.f32(L));
    });
    TOMHIP_CHECK(hipGetLastError());
    dispatch_box(ny, [&](auto Lc) {
      constexpr int L = decltype(Lc)::value;
      constexpr int TW = strided_tw<float, L>();
      hipLaunchKernelGGL((k_c2c_strided<float, L, -1>), dim3((nx + TW - 1) / TW, nz, count), dim3(NT), 0, s, work, nx,
                         (long)nx, XY, n3, tw.f32(L));
    });
  }
  TOMHIP_CHECK(hipGetLastError());
  dispatch_box(nz, [&](auto Lc) {
    constexpr int L = decltype(Lc)::value;
    hipLaunchKernelGGL(k_box_z<L>, dim3((unsigned)((XY + 63) / 64), (unsigned)count), dim3(64 * NW), 0, s, work, wsh,
                       (int)XY, line_list(tw, L));
  });
  TOMHIP_CHECK(hipGetLastError());
  if (plane) {
    dispatch_box(nx, [&](auto Lc) {
      constexpr int L = decltype(Lc)::value;
      hipLaunchKernelGGL(k_box_xy_inv<L>, dim3((unsigned)(count * nz)), dim3(64 * NW), 0, s,
                         (const c32*)work, t, mask, nz, (float)(1.0 / (double)n3), line_list(tw, L));
    });
    TOMHIP_CHECK(hipGetLastError());
    return;
  }
  dispatch_box(ny, [&](auto Lc) {
    constexpr int L = decltype(Lc)::value;
    constexpr int TW = strided_tw<float, L>();
    hipLaunchKernelGGL((k_c2c_strided<float, L, 1>), dim3((nx + TW - 1) / TW, nz, count), dim3(NT), 0, s, work, nx,
                       (long)nx, XY, n3, tw.f32(L));
  });
  TOMHIP_CHECK(hipGetLastError());
  dispatch_box(nx, [&](auto Lc) {
    constexpr int L = decltype(Lc)::value;
    constexpr int NL = kBoxLines;
    hipLaunchKernelGGL(k_box_x_inv<L>, dim3((unsigned)(count * ((lpv + NL - 1) / NL))), dim3(NT), 0, s,
                       (const c32*)work, t, mask, lpv, (float)(1.0 / (double)n3), tw.f32(L));
  });
  TOMHIP_CHECK(hipGetLastError());
}

void box_filter(Twiddles& tw, hipStream_t s, int count, float* t, c32* work, const float* wsh, const float* mask,
                int nx, int ny, int nz) {
  const long n3 = (long)nx * ny * nz;
  for (int b = 0; b < count; b += 65535)
    box_filter_slab(tw, s, std::min(count - b, 65535), t + b * n3, work + b * n3, wsh, mask, nx, ny, nz);
}

}  // namespace tomhip
