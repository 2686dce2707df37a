// FFT stages with one line per lane, the butterfly index uniform over a wave.
//
// A block transforms up to 64 lines of length L, a line per lane; wave w of
// NW takes the butterflies j = w (mod NW), so a stage's twiddles are the same
// for all lanes and come through scalar loads, and its element addresses are
// one lane offset plus scalars. The plan, twiddles, butterflies and their
// order of operations are those of fft_io.h, so the values are the same bits.
#pragma once
#include "fft_kernels.h"

namespace tomhip {

// N consecutive twiddles at a wave-uniform address, as one scalar load.
// Through the constant address space: the load then is scalar whatever the
// kernel stores elsewhere (a vector load behind a kernel's stores waits for
// them). One load for all of a butterfly's twiddles matters: every scalar
// load is waited for by itself.
template <int N>
struct TwVec {
  typedef uint32_t type __attribute__((ext_vector_type(2 * N)));
};
template <int N>
__device__ __forceinline__ void tw_load(const c32* p, c32* t) {
  typedef typename TwVec<N>::type V;
  typedef const __attribute__((address_space(4))) V* cptr;
  const V u = *(cptr)(uintptr_t)p;
#pragma unroll
  for (int i = 0; i < N; ++i) t[i] = mk(__uint_as_float(u[2 * i]), __uint_as_float(u[2 * i + 1]));
}
// entries kept for the R - 1 twiddles of a butterfly (entry 0 is 1)
__host__ __device__ constexpr int tw_slots(int R) { return R <= 2 ? 2 : R <= 4 ? 4 : 8; }

// The same value, unknown to the compiler: addresses derived from it are made
// again in every pass of a loop instead of being held in registers over it.
__device__ __forceinline__ int fresh(int x) {
  asm volatile("" : "+v"(x));
  return x;
}
// the same for a wave-uniform value
__device__ __forceinline__ int fresh_uniform(int x) {
  asm volatile("" : "+s"(x));
  return x;
}

// Twiddles of the stages 1 .. of length L in the order in which waves read
// them: stage, k = j mod NS, the butterfly's entries.
__host__ __device__ constexpr int line_tw_at(int L, int S) {
  int at = 0;
  for (int s = 1; s < S; ++s) at += plan_ns(L, s) * tw_slots(plan_radix(L, s));
  return at;
}
inline void line_tw_list(int L, std::vector<c32>& out) {
  for (int s = 1; s < plan_nstages(L); ++s) {
    const int R = plan_radix(L, s), NS = plan_ns(L, s);
    for (int k = 0; k < NS; ++k)
      for (int r = 0; r < tw_slots(R); ++r)
        out.push_back(r < R ? Twiddles::root<float>(L, r * k * (L / (NS * R))) : mk(0.f, 0.f));
  }
}
inline const c32* line_list(Twiddles& tw, int L) {
  return tw.list(L, [&](std::vector<c32>& h) {
    line_tw_list(L, h);
    if (h.empty()) h.push_back(mk(1.f, 0.f));
  });
}
// the twiddles of a butterfly of stage S (k = j mod NS) on its inputs
template <int L, int S, int DIR>
__device__ __forceinline__ void line_twiddle(const c32* tw, int k, c32* t) {
  constexpr int RP = tw_slots(plan_radix(L, S));
  tw_load<RP>(tw + line_tw_at(L, S) + k * RP, t);
#pragma unroll
  for (int r = 1; r < RP; ++r)
    if (DIR < 0) t[r] = conjg(t[r]);
}

// Everything after stage 0 of a length of two or three stages. With three,
// the last two run on the R1 R2 elements of a group in registers: group
// m (< NS1) holds the butterflies m + NS1 s of stage 1, whose outputs are the
// inputs of the butterflies m + NS1 s of stage 2. Wave w takes the groups
// m = w + NW g. All it reads and all it makes are elements e = w (mod NW):
// rd(e) reads stage 0's result e, out(k, v) takes the transform's element
// e = w + NW k.
template <int L, int NW>
struct Tail {
  static constexpr int S = plan_nstages(L);
  static_assert(S == 2 || S == 3, "two or three stages");
  static constexpr bool kMerged = S == 3;
  static constexpr int RA = kMerged ? plan_radix(L, 1) : 1, NSA = plan_ns(L, kMerged ? 1 : S - 1);
  static constexpr int RB = plan_radix(L, S - 1), NSB = plan_ns(L, S - 1);
  static constexpr int NG = NSA / NW, EPT = L / NW;
  static_assert(NSA % NW == 0 && (L / RA) % NW == 0 && NSB % NW == 0, "groups per wave");

  template <int DIR, class RD, class OUT>
  static __device__ __forceinline__ void run(int w, const c32* tw, const RD& rd, const OUT& out) {
    c32 u[NG][RB][RA];
#pragma unroll
    for (int g = 0; g < NG; ++g)
#pragma unroll
      for (int q = 0; q < RB; ++q)
#pragma unroll
        for (int t = 0; t < RA; ++t)
          u[g][q][t] = rd(w + NW * g + (kMerged ? NSA * q + L / RA * t : L / RB * q));
#pragma unroll
    for (int g = 0; g < NG; ++g) {
      const int m = w + NW * g;
      if constexpr (kMerged) {
        c32 t1[tw_slots(RA)];
        line_twiddle<L, 1, DIR>(tw, m, t1);
#pragma unroll
        for (int q = 0; q < RB; ++q) {
#pragma unroll
          for (int t = 1; t < RA; ++t) u[g][q][t] = cmul(u[g][q][t], t1[t]);
          Bfly<float, RA, DIR>::run(u[g][q]);
        }
      }
#pragma unroll
      for (int s = 0; s < RA; ++s) {
        c32 t2[tw_slots(RB)], x[RB];
        line_twiddle<L, S - 1, DIR>(tw, m + (kMerged ? NSA * s : 0), t2);
        x[0] = u[g][0][s];
#pragma unroll
        for (int q = 1; q < RB; ++q) x[q] = cmul(u[g][q][s], t2[q]);
        Bfly<float, RB, DIR>::run(x);
#pragma unroll
        for (int r = 0; r < RB; ++r) out(g + (kMerged ? NSA / NW * s : 0) + NSB / NW * r, x[r]);
      }
    }
  }
};

// LDS written by this wave is read back by other lanes of the same wave
__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

}  // namespace tomhip
