// The inverse transform of the exhaustive search in two kernels.
//
// The y transform (length Y) begins with a radix-R0 stage that combines the
// rows ky = j + r Y/R0 and from then on works within the R0 classes
// y = r (mod R0). So that stage can run where the z transform's results are
// still on the chip, and the rest of it where the x transform needs them:
//   fused_a   per (kx tile of 64 / R0 columns, j): z forward of the template,
//             product with F_I, z inverse, radix-R0 stage of y -> Q
//   fused_bc  per (z, class r): the remaining y stages and the x c2r of the
//             class's Y / R0 rows, running maximum over the batch
// Q is written once and read once, where three kernels (z; y in place; x)
// move it four times. Every value passes through the same butterflies,
// twiddles and products in the same order as there, so the maps are the same
// bits.
//
// Q[a][z mod Z/2][r][kx / 8][p][kx % 8][z / (Z/2)], p = the row within the
// class: the 128 bytes of eight columns and two planes are written by one
// store instruction, 16 bytes a lane. What a block of fused_a holds of one
// (z, r, p) is 64 / R0 columns, 64 bytes for R0 = 8: stored as such, 8 bytes a
// lane, the same traffic runs at half the rate (4.3 GB: 1.75 ms against 0.88).
#include <type_traits>

#include "common.h"
#include "dft16.h"
#include "fused.h"
#include "fused_dev.h"

namespace tomhip {

namespace {

// Waves of fused_a: every wave holds the elements z = w (mod NW) of its
// lines in registers.
constexpr int waves_a(int Z) {
  return Z == 256 ? 16 : Z >= 128 ? 8 : Z >= 64 ? 4 : Z >= 32 ? 2 : 1;
}
// LDS of fused_a: rows of 64 lines at this pitch, 16 banks apart (the y stage
// reads several rows at once).
constexpr int kRow = 72;
constexpr int kRows(int Z) { return Z * kRow; }
__device__ __forceinline__ int row_at(int row) { return row * kRow; }

// Which radix-R0 inputs j + r NJ of a transform of length Z can hold a
// template plane: the planes lie within 32 of the origin, wrapped.
template <int Z>
constexpr bool may_hold(int lo, int hi) {
  return lo < 32 || hi >= Z - 32;
}

// Row p of a class (of Lp) is kept at row p + class_turn, wrapped: what a
// block of fused_a writes at one time (one row of many z and classes r, a
// power of two apart) then spreads over the memory channels.
__device__ __forceinline__ int class_turn(int z, int r, int Lp) {
  return (((z ^ (z >> 4)) + 2 * r) & 15) * (Lp >> 4);
}

// ---------------------------------------------------------------- z transforms
// Forward z transform of the template planes, the product with F_I, the
// inverse, for the line of this lane; wave w holds kz = w + NW k and then
// z = w + NW k in registers. Z = 256 runs as 16 x 16, the others as the radix
// plan of fft.h. Stage 0 of the inverse takes the elements that the wave
// holds, so there are two exchanges through LDS, and what a wave writes goes
// where it alone has read before: a barrier after each write, and one before
// the forward write.
template <int Z>
struct ZOps {
  static constexpr int NW = waves_a(Z), EPT = Z / NW;
  static constexpr int R0 = plan_radix(Z, 0), NJ0 = Z / R0, P0 = NJ0 / NW;
  using T = Tail<Z, NW>;
  static_assert(NJ0 % NW == 0, "stage 0 within a wave");
  c32 f[EPT];  // F_I of this lane's outputs

  // stage 0 leaves its output e = j R0 + r with the wave j mod NW as number
  // i = j / NW R0 + r: the row of e where wave w keeps its i-th at w + NW i
  static __device__ __forceinline__ int own_row(int e) {
    const int j = e / R0;
    return j % NW + NW * (j / NW * R0 + e % R0);
  }
  // row that holds plane z after inverse()
  static __device__ __forceinline__ int row(int z) { return own_row(z); }

  // The template planes of the first stage. They are loaded for the next
  // angle before this one's results are stored: loads and stores return in
  // order, so a load behind the stores would wait for all of them.
  struct In {
    c32 u[P0][R0];
  };
  // ld(z): the template's value at wrapped plane z
  template <class LD>
  static __device__ __forceinline__ void load(In& in, int w, const LD& ld) {
#pragma unroll
    for (int p = 0; p < P0; ++p)
#pragma unroll
      for (int r = 0; r < R0; ++r)
        in.u[p][r] = may_hold<Z>(r * NJ0, r * NJ0 + NJ0 - 1) ? ld(w + NW * p + r * NJ0) : mk(0.f, 0.f);
  }
  // next(): loads the next angle's planes; hook(k, v): the product's last word
  template <class NEXT, class HOOK>
  __device__ __forceinline__ void forward(c32* buf, const c32* tw, int w, int lane, In& in, const NEXT& next,
                                          const HOOK& hook, c32* v) const {
    c32 u[P0][R0];
#pragma unroll
    for (int p = 0; p < P0; ++p) {
#pragma unroll
      for (int r = 0; r < R0; ++r) u[p][r] = in.u[p][r];
      Bfly<float, R0, -1>::run(u[p]);
    }
    next();
    __syncthreads();  // the previous angle's rows have been read
#pragma unroll
    for (int p = 0; p < P0; ++p)
#pragma unroll
      for (int r = 0; r < R0; ++r) buf[row_at((w + NW * p) * R0 + r) + lane] = u[p][r];
    __syncthreads();
    T::template run<-1>(w, tw, [&](int e) { return buf[row_at(e) + lane]; },
                        [&](int k, c32 q) { v[k] = hook(k, cmulc(f[k], q)); });
  }
  __device__ __forceinline__ void inverse(c32* buf, const c32* tw, int w, int lane, c32* v) const {
#pragma unroll
    for (int p = 0; p < P0; ++p) {
      c32 u[R0];
#pragma unroll
      for (int r = 0; r < R0; ++r) u[r] = v[p + P0 * r];
      Bfly<float, R0, 1>::run(u);
#pragma unroll
      for (int r = 0; r < R0; ++r) buf[row_at(w + NW * (p * R0 + r)) + lane] = u[r];
    }
    __syncthreads();
    T::template run<1>(w, tw, [&](int e) { return buf[row_at(own_row(e)) + lane]; }, [&](int k, c32 q) { v[k] = q; });
#pragma unroll
    for (int k = 0; k < EPT; ++k) buf[row_at(row(w + NW * k)) + lane] = v[k];
  }
};

// twiddles: list of exp(2 pi i w k / 256), k = 0 .. 15, of every wave w
template <>
struct ZOps<256> {
  static constexpr int NW = 16, EPT = 16;
  c32 f[16];

  static __device__ __forceinline__ int row(int z) { return z; }

  struct In {
    c32 u[4];
  };
  // planes lie in z < 32 or z >= 224: n2 = 0, 1, 14, 15
  template <class LD>
  static __device__ __forceinline__ void load(In& in, int w, const LD& ld) {
    in.u[0] = ld(w);
    in.u[1] = ld(w + 16);
    in.u[2] = ld(w + 224);
    in.u[3] = ld(w + 240);
  }
  template <class NEXT, class HOOK>
  __device__ __forceinline__ void forward(c32* buf, const c32* tw, int w, int lane, In& in, const NEXT& next,
                                          const HOOK& hook, c32* v) const {
    v[0] = in.u[0];
    v[1] = in.u[1];
    v[14] = in.u[2];
    v[15] = in.u[3];
    dft16_ends(v);
    next();
    c32 t[16];
    tw_load<8>(tw + w * 16, t);
    tw_load<8>(tw + w * 16 + 8, t + 8);
#pragma unroll
    for (int k2 = 1; k2 < 16; ++k2) v[k2] = cmul(v[k2], conjg(t[k2]));
    // rows k2 * 16 + w are this wave's alone here and in the y stage that
    // read them last: no barrier before the write
#pragma unroll
    for (int k2 = 0; k2 < 16; ++k2) buf[row_at(k2 * 16 + w) + lane] = v[k2];
    __syncthreads();
#pragma unroll
    for (int n1 = 0; n1 < 16; ++n1) v[n1] = buf[row_at(w * 16 + n1) + lane];
    dft16<-1>(v);
#pragma unroll
    for (int k1 = 0; k1 < 16; ++k1) v[k1] = hook(k1, cmulc(f[k1], v[k1]));
  }

  __device__ __forceinline__ void inverse(c32* buf, const c32* tw, int w, int lane, c32* v) const {
    dft16<1>(v);
    c32 t[16];
    tw_load<8>(tw + w * 16, t);
    tw_load<8>(tw + w * 16 + 8, t + 8);
#pragma unroll
    for (int m1 = 1; m1 < 16; ++m1) v[m1] = cmul(v[m1], t[m1]);
    // rows w * 16 + m1 were read by this wave alone: no barrier before the write
#pragma unroll
    for (int m1 = 0; m1 < 16; ++m1) buf[row_at(w * 16 + m1) + lane] = v[m1];
    __syncthreads();
#pragma unroll
    for (int k2 = 0; k2 < 16; ++k2) v[k2] = buf[row_at(k2 * 16 + w) + lane];
    dft16<1>(v);  // q[w + 16 m2]
    // rows k2 * 16 + w, k2 = 0 .. 15, were read by this wave alone
#pragma unroll
    for (int m2 = 0; m2 < 16; ++m2) buf[row_at(m2 * 16 + w) + lane] = v[m2];
  }
};

// ---------------------------------------------------------------- kernels
// Product of the kx = X/2 column: Pn[a][kz][ky]. grid (ceil(Y / 64), ka).
template <int Z>
__global__ __launch_bounds__(64 * waves_a(Z)) void k_fused_nyq(const c32* __restrict__ Tyn,
                                                               const c32* __restrict__ FIn, c32* __restrict__ Pn,
                                                               const c32* tw, int Y, int nz) {
  using O = ZOps<Z>;
  __shared__ c32 buf[kRows(Z)];
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int ky = blockIdx.x * 64 + lane, a = blockIdx.y;
  const bool ok = ky < Y;
  O zo;
#pragma unroll
  for (int k = 0; k < O::EPT; ++k) zo.f[k] = ok ? FIn[(long)ky * Z + w + O::NW * k] : mk(0.f, 0.f);
  const int hz = nz / 2;
  const c32* src = Tyn + (long)a * nz * Y + ky;
  c32 v[O::EPT];
  typename O::In in;
  O::load(in, w, [&](int z) {
    int uz = z + hz;
    if (uz >= Z) uz -= Z;
    return (uz < nz && ok) ? src[(long)uz * Y] : mk(0.f, 0.f);
  });
  zo.forward(
      buf, tw, w, lane, in, [] {}, [](int, c32 q) { return q; }, v);
  if (!ok) return;
  c32* dst = Pn + (long)a * Z * Y + ky;
#pragma unroll
  for (int k = 0; k < O::EPT; ++k) dst[(long)(w + O::NW * k) * Y] = v[k];
}

// grid (Xh / T * NJ, angle groups of apb). 512x512x256, 16 angles: 1.45 ms
// for 5.4 GB; with its loads and stores taken out 1.17 ms, the vector
// instructions alone 0.9 (66 a complex element). What it took: 16 bytes a
// lane and 128 a line in the stores (2.7 -> 1.45 ms), twiddles as one scalar
// load per butterfly, next-angle loads ahead of the stores.
template <int Z, int R0>
__global__ __launch_bounds__(64 * waves_a(Z), Z / waves_a(Z) > 16 ? 2 : 4) void k_fused_a(const c32* __restrict__ Ty, const c32* __restrict__ Pn,
                                                             const c32* __restrict__ FI, c32* __restrict__ Q,
                                                             const c32* tw, int Y, int Xh, int nz, int ka, int apb) {
  using O = ZOps<Z>;
  constexpr int T = 64 / R0, NW = O::NW;
  __shared__ c32 buf[kRows(Z)];
  const int lane_ = threadIdx.x & 63, w_ = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int NJ = Y / R0;
  const int j = blockIdx.x % NJ, tile = blockIdx.x / NJ;
  O zo;
#pragma unroll
  for (int k = 0; k < O::EPT; ++k)
    zo.f[k] = FI[((long)(w_ + NW * k) * Y + j + lane_ / T * NJ) * Xh + tile * T + lane_ % T];
  const int hz = nz / 2;
  const long su = (long)Y * Xh;
  const int a0 = blockIdx.y * apb, a1 = min(a0 + apb, ka);
  typename O::In in;
  auto load = [&](int a, int w, int lane) {
    const c32* src = Ty + (long)a * nz * su + ((long)tile * NJ + j) * 64 + lane;
    O::load(in, w, [&](int z) {
      int uz = z + hz;
      if (uz >= Z) uz -= Z;
      return (uz < nz) ? src[(long)uz * su] : mk(0.f, 0.f);
    });
  };
  load(a0, w_, lane_);
  for (int a = a0; a < a1; ++a) {
    const int w = fresh_uniform(w_);
    const int lane = fresh(lane_), c = lane % T, ky = j + lane / T * NJ;
    const c32* pn = Pn + (long)a * Z * Y + ky;
    c32 v[O::EPT];
    zo.forward(
        buf, tw, w, lane, in,
        [&] {
          if (a + 1 < a1) load(a + 1, fresh_uniform(w), fresh(lane));
        },
        [&](int k, c32 q) {
          if (tile == 0 && c == 0) {  // P(0) + i P(X/2)
            const c32 n = pn[(long)(w + NW * k) * Y];
            q = mk(q.x - n.y, q.y + n.x);
          }
          return q;
        },
        v);
    zo.inverse(buf, tw, w, lane, v);
    // radix-R0 stage of y: lane = (pair of planes, column), its R0 lines from
    // the rows of this wave
    wave_lds_sync();
    constexpr int NP = 64 / T, Zh = Z / 2, PAIRS = O::EPT / 2;
    c32* qa = Q + (long)a * Z * su + (long)tile * (T / 8) * NJ * 16 + c / 8 * (NJ * 16) + c % 8 * 2;
#pragma unroll
    for (int s = 0; s < (PAIRS + NP - 1) / NP; ++s) {
      const int i = s * NP + lane / T, zp = w + NW * i;
      if (PAIRS % NP == 0 || i < PAIRS) {
        c32 u0[R0], u1[R0];
        const int r0 = row_at(O::row(zp)) + c, r1 = row_at(O::row(zp + Zh)) + c;
#pragma unroll
        for (int q = 0; q < R0; ++q) {
          u0[q] = buf[r0 + q * T];
          u1[q] = buf[r1 + q * T];
        }
        Bfly<float, R0, 1>::run(u0);
        Bfly<float, R0, 1>::run(u1);
        c32* qz = qa + (long)zp * 2 * su;
#pragma unroll
        for (int q = 0; q < R0; ++q) {
          int at = j + class_turn(zp, q, NJ);
          if (at >= NJ) at -= NJ;
          *reinterpret_cast<float4*>(qz + (q * (Xh / 8) * NJ + at) * 16) = make_float4(u0[q].x, u0[q].y, u1[q].x, u1[q].y);
        }
      }
    }
    wave_lds_sync();
  }
}

// ---------------------------------------------------------------- y rest, x, maximum
constexpr int waves_bc(int XH) { return XH >= 160 ? 8 : XH >= 80 ? 4 : 2; }
// z planes per block of fused_bc: as many as 64 lines hold. An even number is
// taken as pairs (z, z + Z/2), whose 16 bytes of a column one lane loads; an
// odd number as planes of one half, the block of the other half next to it on
// the same XCD (the second one reads the lines from the L2).
constexpr int z_group(int Y) { return 64 / (Y / plan_radix(Y, 0)); }
constexpr bool z_paired(int Y) { return z_group(Y) % 2 == 0; }

// Twiddle list of k_fused_bc: y stages 1 .. by class and butterfly, then the
// pre-twiddles and stages of x.
__host__ __device__ constexpr int class_tw_at(int Y, int S) {
  int at = 0;
  for (int s = 1; s < S; ++s) at += plan_ns(Y, s) * tw_slots(plan_radix(Y, s));
  return at;
}
void bc_tw_list(int XH, int Y, std::vector<c32>& out) {
  const int R0 = plan_radix(Y, 0);
  for (int s = 1; s < plan_nstages(Y); ++s) {
    const int R = plan_radix(Y, s), NS = plan_ns(Y, s), NSC = NS / R0;
    for (int rc = 0; rc < R0; ++rc)
      for (int q = 0; q < NSC; ++q)
        for (int r = 0; r < tw_slots(R); ++r)
          out.push_back(r < R ? Twiddles::root<float>(Y, r * (R0 * q + rc) * (Y / (NS * R))) : mk(0.f, 0.f));
  }
  // butterfly j with its mirror: entries j + r NJ0; for j = 0 those of 0 and
  // then those of NJ0 / 2, half as many each
  const int RX = plan_radix(XH, 0), NJ0 = XH / RX;
  for (int j = 0; j < NJ0 / 2; ++j)
    for (int r = 0; r < RX; ++r)
      out.push_back(Twiddles::root<float>(
          2 * XH, j ? j + r * NJ0 : r < RX / 2 ? r * NJ0 : NJ0 / 2 + (r - RX / 2) * NJ0));
  line_tw_list(XH, out);
}

// The y stages after the first within one class of rows, as tasks of a wave:
// (butterfly q of the class, 64 of the ZB * XH (z, column) items).
template <int XH, int Y, int S>
struct ClassStage {
  static constexpr int R0 = plan_radix(Y, 0), Lp = Y / R0, ZB = z_group(Y), NW = waves_bc(XH);
  static constexpr int R = plan_radix(Y, S), NS = plan_ns(Y, S);  // NS counts R0
  static constexpr int NSC = NS / R0;                             // within the class
  static constexpr int NQ = Lp / R, TWS = Y / (NS * R);
  static constexpr int NCH = (ZB * XH + 63) / 64;
  static constexpr int M = (NQ * NCH + NW - 1) / NW;
  static __device__ __forceinline__ void task(int t, int w, int& q, int& ch) {
    const int k = w + NW * t;
    q = k % NQ;
    ch = k / NQ;
  }
  static __device__ __forceinline__ bool valid(int t, int w) { return (NQ * NCH) % NW == 0 || w + NW * t < NQ * NCH; }
  // (z, column) of item ch * 64 + lane; false beyond the block's planes
  static __device__ __forceinline__ bool item(int ch, int lane, int nzb, int& zb, int& col) {
    if constexpr (XH % 64 == 0) {
      zb = ch / (XH / 64);
      col = (ch % (XH / 64)) * 64 + lane;
    } else {
      const int i = ch * 64 + lane;
      zb = i / XH;
      col = i % XH;
    }
    return zb < nzb;
  }
  static constexpr int RP = tw_slots(R);
  // twiddles of class rc, butterfly, stage inputs v -> outputs v
  static __device__ __forceinline__ void run(c32* v, int q, int rc, const c32* tw) {
    c32 t[RP];
    tw_load<RP>(tw + class_tw_at(Y, S) + (rc * NSC + q % NSC) * RP, t);
#pragma unroll
    for (int r = 1; r < R; ++r) v[r] = cmul(v[r], t[r]);
    Bfly<float, R, 1>::run(v);
  }
  static __device__ __forceinline__ int out_row(int q) { return (q / NSC) * NSC * R + q % NSC; }
};

template <int XH, int Y, int S, int P>
__device__ __forceinline__ void class_stages(c32* buf, const c32* tw, int w, int lane, int rc, int nzb) {
  if constexpr (S < plan_nstages(Y)) {
    using I = ClassStage<XH, Y, S>;
    c32 v[I::M][I::R];
#pragma unroll
    for (int t = 0; t < I::M; ++t) {
      int q, ch, zb, col;
      I::task(t, w, q, ch);
      if (I::valid(t, w) && I::item(ch, lane, nzb, zb, col)) {
#pragma unroll
        for (int r = 0; r < I::R; ++r) v[t][r] = buf[(zb * I::Lp + q + r * I::NQ) * P + col];
        I::run(v[t], q, rc, tw);
      }
    }
    // the last stage puts its results where their inputs were
    if constexpr (S < plan_nstages(Y) - 1) __syncthreads();
#pragma unroll
    for (int t = 0; t < I::M; ++t) {
      int q, ch, zb, col;
      I::task(t, w, q, ch);
      if (I::valid(t, w) && I::item(ch, lane, nzb, zb, col)) {
#pragma unroll
        for (int r = 0; r < I::R; ++r) buf[(zb * I::Lp + I::out_row(q) + r * I::NSC) * P + col] = v[t][r];
      }
    }
    __syncthreads();
    class_stages<XH, Y, S + 1, P>(buf, tw, fresh_uniform(w), fresh(lane), rc, nzb);
  }
}

// Class rc of ZB planes, all angles of the batch, one line per lane in the x
// part. 512x512x256, 16 angles: 1.65 ms for 4.6 GB (1.53 without the loads;
// vector instructions 0.9): with 128 KB of LDS a CU holds one block, whose
// eight waves have 256 registers each for the maxima (72), the next angle's
// inputs (64) and the 32 elements at work; 16 waves of 128 registers spill
// (2.35 ms). An angle has three exchanges through LDS and four barriers.
// GROUPS: the angles in groups of apb (grid.y), each one's maxima for the merge
// to pv and pi (a kernel of its own: with the choice made at run time the
// undivided batch takes 1.63 for 1.61 ms here, 204 for 196 us at 256x256x128).
template <int XH, int Y, bool GROUPS>
__global__ __launch_bounds__(64 * waves_bc(XH)) void k_fused_bc(const c32* __restrict__ Q, float* __restrict__ maxc,
                                                                int32_t* __restrict__ argm,
                                                                const c32* tw, int Z, int ka, int first_index,
                                                                const long* desc, int apb, float* __restrict__ pv,
                                                                uint8_t* __restrict__ pi, long n) {
  const int a0 = GROUPS ? blockIdx.y * apb : 0, a1 = GROUPS ? min(a0 + apb, ka) : ka;
  if (desc) first_index = (int)(desc[1] + desc[0] * ka);
  using I1 = ClassStage<XH, Y, 1>;
  constexpr int NW = waves_bc(XH), NT_ = 64 * NW, R0 = I1::R0, Lp = I1::Lp, ZB = I1::ZB;
  constexpr int P = XH + 1;
  constexpr int RX = plan_radix(XH, 0), NJ0 = XH / RX, NPAIR = NJ0 / 2;
  constexpr int TPW = (NPAIR + NW - 1) / NW;  // stage-0 butterfly pairs per wave
  constexpr int TW0 = class_tw_at(Y, plan_nstages(Y)), TWH = TW0 + NPAIR * RX;
  static_assert(NJ0 % 2 == 0 && RX % 2 == 0, "c2r pairing");
  using TX = Tail<XH, NW>;
  constexpr int EPT = TX::EPT;
  __shared__ c32 buf[64 * P];
  const int lane_ = threadIdx.x & 63, w_ = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  constexpr bool PAIR = z_paired(Y);
  int b = blockIdx.x;
  const int nb = gridDim.x;
  if ((nb & 7) == 0) b = (b & 7) * (nb >> 3) + (b >> 3);
  const int Zh = Z / 2;
  const int bit = PAIR ? 0 : b % 2;
  if (!PAIR) b /= 2;
  const int rc = b % R0, z0 = (b / R0) * (PAIR ? ZB / 2 : ZB);
  const int nzb = min(ZB, (Zh - z0) * (PAIR ? 2 : 1));
  // plane zb of the block
  auto plane = [&](int zb) { return PAIR ? z0 + zb / 2 + zb % 2 * Zh : z0 + zb + bit * Zh; };
  constexpr long SU = (long)Y * XH;
  // first remaining y stage: inputs from Q, the next angle's while this one
  // runs its LDS stages. Items are the columns of ZL planes (of pairs).
  constexpr int ZL = PAIR ? ZB / 2 : ZB, NCH1 = (ZL * XH + 63) / 64, M1 = (I1::NQ * NCH1 + NW - 1) / NW;
  using In = std::conditional_t<PAIR, float4, c32>;
  In pf[M1][I1::R];
  auto task1 = [&](int t, int w, int lane, int& q, int& zl, int& col) {
    const int k = w + NW * t, i = k / I1::NQ * 64 + lane;
    q = k % I1::NQ;
    zl = i / XH;
    col = i % XH;
    if constexpr (XH % 64 == 0) {
      const int ch = k / I1::NQ;
      zl = ch / (XH / 64);
      col = ch % (XH / 64) * 64 + lane;
    }
    return ((I1::NQ * NCH1) % NW == 0 || k < I1::NQ * NCH1) && zl < (PAIR ? nzb / 2 : nzb);
  };
  const c32* qp = Q + (GROUPS ? a0 * Z * SU : 0) + (long)z0 * 2 * SU + (long)rc * Lp * XH * 2 + bit;
  // quarter part of the loads of one angle (all of them: part < 0)
  auto fetch = [&](const c32* qa, int part, int w, int lane) {
#pragma unroll
    for (int t = 0; t < M1; ++t) {
      int q, zl, col;
      if (task1(t, w, lane, q, zl, col)) {
        const c32* src = qa + (zl * 2 * SU + col / 8 * (Lp * 16) + col % 8 * 2);
        const int turn = class_turn(z0 + zl, rc, Lp);
#pragma unroll
        for (int r = 0; r < I1::R; ++r) {
          if (part >= 0 && (t * I1::R + r) * 4 / (M1 * I1::R) != part) continue;
          int at = q + r * I1::NQ + turn;
          if (at >= Lp) at -= Lp;
          pf[t][r] = *reinterpret_cast<const In*>(src + at * 16);
        }
      }
    }
  };
  // the next angle's loads are issued a quarter at a time between the stages
  auto ahead = [&](int a, int part, int w, int lane) {
    if (a + 1 < a1) fetch(qp, part, fresh_uniform(w), fresh(lane));
  };
  float bx[EPT], by[EPT];
  constexpr int NI = (EPT + 7) / 8;
  uint32_t ix[NI], iy[NI];  // batch indices, 4 bits each
#pragma unroll
  for (int p = 0; p < NI; ++p) ix[p] = iy[p] = 0u;
#pragma unroll
  for (int k = 0; k < EPT; ++k) bx[k] = by[k] = GROUPS ? -INFINITY : 0.f;
  fetch(qp, -1, w_, lane_);
  for (int a = a0; a < a1; ++a) {
    const int lane = fresh(lane_), w = fresh_uniform(w_);
    if (a > a0) __syncthreads();  // the previous angle's lines have been read
#pragma unroll
    for (int t = 0; t < M1; ++t) {
      int q, zl, col;
      if (task1(t, w, lane, q, zl, col)) {
#pragma unroll
        for (int h = 0; h < (PAIR ? 2 : 1); ++h) {
          c32 v[I1::R];
#pragma unroll
          for (int r = 0; r < I1::R; ++r) {
            if constexpr (PAIR)
              v[r] = h ? mk(pf[t][r].z, pf[t][r].w) : mk(pf[t][r].x, pf[t][r].y);
            else
              v[r] = pf[t][r];
          }
          I1::run(v, q, rc, tw);
          const int zb = PAIR ? 2 * zl + h : zl;
#pragma unroll
          for (int r = 0; r < I1::R; ++r) buf[(zb * Lp + I1::out_row(q) + r * I1::NSC) * P + col] = v[r];
        }
      }
    }
    qp += (long)Z * SU;
    ahead(a, 0, w, lane);
    __syncthreads();
    class_stages<XH, Y, 2, P>(buf, tw, fresh_uniform(w), fresh(lane), rc, nzb);
    ahead(a, 1, w, lane);
    // x: complex-to-real pre-twiddle and stage 0, line = lane, each butterfly
    // j with its mirror NJ0 - j (0 with NJ0 / 2); output J RX + r goes to
    // column J + NJ0 r, which this wave has just read
    {
      c32* g = buf + fresh(lane) * P;
#pragma unroll
      for (int t = 0; t < TPW; ++t) {
        const int j = w + NW * t;
        if (NPAIR % NW != 0 && j >= NPAIR) continue;
        c32 va[RX], vb[RX], z1[RX], z2[RX];
        const int jb = j == 0 ? NPAIR : NJ0 - j;
        c32 tx[RX];
        tw_load<RX>(tw + TW0 + j * RX, tx);
#pragma unroll
        for (int r = 0; r < RX; ++r) va[r] = g[j + r * NJ0];
#pragma unroll
        for (int r = 0; r < RX; ++r) vb[r] = g[jb + r * NJ0];
        if (j == 0) {
          z1[0] = mk(va[0].x + va[0].y, va[0].x - va[0].y);
#pragma unroll
          for (int r = 1; r < RX / 2; ++r) {
            const c32 gk = va[r], gm = va[RX - r];
            const c32 A = mk(gk.x + gm.x, gk.y - gm.y);
            const c32 B = cmul(mk(gk.x - gm.x, gk.y + gm.y), tx[r]);
            z1[r] = mk(A.x - B.y, A.y + B.x);
            z1[RX - r] = mk(A.x + B.y, B.x - A.y);
          }
          z1[RX / 2] = mk(2.f * va[RX / 2].x, -2.f * va[RX / 2].y);
#pragma unroll
          for (int r = 0; r < RX / 2; ++r) {
            const c32 gk = vb[r], gm = vb[RX - 1 - r];
            const c32 A = mk(gk.x + gm.x, gk.y - gm.y);
            const c32 B = cmul(mk(gk.x - gm.x, gk.y + gm.y), tx[RX / 2 + r]);
            z2[r] = mk(A.x - B.y, A.y + B.x);
            z2[RX - 1 - r] = mk(A.x + B.y, B.x - A.y);
          }
        } else {
#pragma unroll
          for (int r = 0; r < RX; ++r) {
            const c32 gk = va[r], gm = vb[RX - 1 - r];
            const c32 A = mk(gk.x + gm.x, gk.y - gm.y);
            const c32 B = cmul(mk(gk.x - gm.x, gk.y + gm.y), tx[r]);
            z1[r] = mk(A.x - B.y, A.y + B.x);
            z2[RX - 1 - r] = mk(A.x + B.y, B.x - A.y);
          }
        }
        Bfly<float, RX, 1>::run(z1);
        Bfly<float, RX, 1>::run(z2);
#pragma unroll
        for (int r = 0; r < RX; ++r) {
          g[j + r * NJ0] = z1[r];
          g[jb + r * NJ0] = z2[r];
        }
      }
      __syncthreads();
    }
    ahead(a, 2, w, lane);
    // x: the other stages, into the running maximum
    const c32* g = buf + fresh(lane) * P;
    // the batch's first angle is taken whatever it is, as a mask rather than a
    // branch: a branch would hold every output in registers on both sides
    const bool first = fresh_uniform(a) == 0;
    TX::template run<1>(
        fresh_uniform(w), tw + TWH, [&](int e) { return g[e / RX + NJ0 * (e % RX)]; },
        [&](int k, c32 v) {
          const uint32_t sh = 4u * (k % 8), msk = ~(15u << sh), av = (uint32_t)a << sh;
          if ((int)first | (int)(v.x > bx[k])) {
            bx[k] = v.x;
            ix[k / 8] = (ix[k / 8] & msk) | av;
          }
          if ((int)first | (int)(v.y > by[k])) {
            by[k] = v.y;
            iy[k / 8] = (iy[k / 8] & msk) | av;
          }
        });
    ahead(a, 3, w, lane);
  }
  const int first = GROUPS ? 0 : first_index;
  // the batch's maximum against the resident maps, a quarter of every line at
  // a time through LDS so that the maps are read and written in rows
  constexpr int KC = EPT / 4, NS = NW * KC, FP = NS + 1;
  static_assert(EPT % 4 == 0 && 64 * FP * 2 <= 64 * P, "staging area");
  float2* sval = reinterpret_cast<float2*>(buf);
  int2* sidx = reinterpret_cast<int2*>(buf + 64 * FP);
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    __syncthreads();
#pragma unroll
    for (int i = 0; i < KC; ++i) {
      const int k = r * KC + i, e = lane_ * FP + w_ + NW * i;
      sval[e] = make_float2(bx[k], by[k]);
      sidx[e] = make_int2(first + (int)((ix[k / 8] >> (4 * (k % 8))) & 15u),
                          first + (int)((iy[k / 8] >> (4 * (k % 8))) & 15u));
    }
    __syncthreads();
    for (int i = threadIdx.x; i < nzb * Lp * NS; i += NT_) {
      const int l = i / NS, e = i % NS;
      const long line = (long)plane(l / Lp) * Y + (l % Lp) * R0 + rc;
      const long vx = (line * XH + r * NS + e) * 2;
      const float2 nv = sval[l * FP + e];
      const int2 ni = sidx[l * FP + e];
      if constexpr (GROUPS) {
        *reinterpret_cast<float2*>(pv + blockIdx.y * n + vx) = nv;
        *reinterpret_cast<uchar2*>(pi + blockIdx.y * n + vx) = make_uchar2(ni.x, ni.y);
        continue;
      }
      const float2 cur = *reinterpret_cast<const float2*>(maxc + vx);
      if (nv.x > cur.x) {
        maxc[vx] = nv.x;
        argm[vx] = ni.x;
      }
      if (nv.y > cur.y) {
        maxc[vx + 1] = nv.y;
        argm[vx + 1] = ni.y;
      }
    }
  }
}

// The lengths that have the fused kernels. Z: 16 elements a lane (24 at 192).
// 48, 80 and 96 leave waves or lanes idle and measured slower than the separate
// passes (batches of 16, fused / separate in us: 512x192x48 560 / 445,
// 320x320x80 772 / 697, 256x96x96 292 / 236); 120, 160, 200 and 240 fit LDS and
// have not been measured. Y: first radix 8 or 4, at most 64 rows in a class,
// the next radix 8 or 4.
#define TOMHIP_CASE(n)                   \
  case n:                                \
    f(std::integral_constant<int, n>{}); \
    return true;
template <class F>
bool dispatch_z(int Z, F&& f) {
  switch (Z) {
    TOMHIP_CASE(32)
    TOMHIP_CASE(64)
    TOMHIP_CASE(128)
    TOMHIP_CASE(192)
    TOMHIP_CASE(256)
    default: return false;
  }
}
template <class F>
bool dispatch_x(int Xh, F&& f) {
  switch (Xh) {
    TOMHIP_CASE(64)
    TOMHIP_CASE(96)
    TOMHIP_CASE(128)
    TOMHIP_CASE(160)
    TOMHIP_CASE(192)
    TOMHIP_CASE(256)
    default: return false;
  }
}
template <class F>
bool dispatch_y(int Y, F&& f) {
  switch (Y) {
    TOMHIP_CASE(64)
    TOMHIP_CASE(96)
    TOMHIP_CASE(128)
    TOMHIP_CASE(160)
    TOMHIP_CASE(192)
    TOMHIP_CASE(240)
    TOMHIP_CASE(256)
    TOMHIP_CASE(320)
    TOMHIP_CASE(384)
    TOMHIP_CASE(480)
    TOMHIP_CASE(512)
    default: return false;
  }
}
#undef TOMHIP_CASE

}  // namespace

namespace {
const c32* z_list(Twiddles& tw, int Z) {
  if (Z != 256) return line_list(tw, Z);
  return tw.list(Z, [&](std::vector<c32>& h) {
    for (int w = 0; w < 16; ++w)
      for (int k = 0; k < 16; ++k) h.push_back(Twiddles::root<float>(256, w * k));
  });
}
const c32* bc_list(Twiddles& tw, int X, int Y) {
  return tw.list((long)X * 4096 + Y, [&](std::vector<c32>& h) { bc_tw_list(X / 2, Y, h); });
}
}  // namespace

void fused_prepare(Twiddles& tw, int X, int Y, int Z) {
  (void)z_list(tw, Z);
  (void)bc_list(tw, X, Y);
}

// Angles per block of k_fused_a. Few blocks: the batch's angles over more of
// them, to twice what the CUs hold at once by their LDS at Z = 32 and 64
// (batches of 16, us, to 1,024 blocks and to this: 512x192x32 187 and 98,
// 512x160x64 214 and 127), 1,024 from 128 on (more read F_I more often:
// 512x96x128 ka 8 83 and, to 2,048, 95).
static int a_angles(int X, int Y, int Z, int ka) {
  const int R0 = plan_radix(Y, 0), blocks = X / 2 / (64 / R0) * (Y / R0);
  const int groups = std::min(ka, std::max(1, std::max(1024, 131072 / Z) / blocks));
  return (ka + groups - 1) / groups;
}
// Blocks of k_fused_bc for one group of angles, and how many the CUs hold at
// once by their LDS.
static int bc_blocks(int Y, int Z) {
  const int ZB = z_group(Y), half = z_paired(Y) ? ZB / 2 : ZB, sides = z_paired(Y) ? 1 : 2;
  return (Z / 2 + half - 1) / half * sides * plan_radix(Y, 0);
}
static int bc_places(int X) { return 256 * (160 * 1024 / (64 * (X / 2 + 1) * (int)sizeof(c32))); }

int fused_bc_groups(int X, int Y, int Z, int ka) {
  // half a chip of blocks or less: two groups, merged by one more launch.
  // Batches of 16, us, one group and two with the merge: 512x192x32 173 and
  // 103, 128x240x128 216 and 128, 256x256x64 161 and 115; where the blocks
  // fill more: 512x192x64 177 and 205. Three and four groups take longer.
  return ka >= 4 && 2 * bc_blocks(Y, Z) <= bc_places(X) ? 2 : 1;
}

bool fused_supported(int X, int Y, int Z, int ka) {
  // The saved traffic pays once a batch's Q does not fit in the memory-side
  // cache (256 MB); below, the separate passes have more blocks to fill the
  // chip with. Batches, fused / separate in us: 134 MB 128x128x128 216 / 207,
  // 512x64x64 242 / 235; 4.3 GB 512x512x256 3218 / 4500.
  if (8L * ka * Z * Y * (X / 2) < (192L << 20)) return false;
  if (!(dispatch_z(Z, [](auto) {}) && dispatch_x(X / 2, [](auto) {}) && dispatch_y(Y, [](auto) {}))) return false;
  // 1,402 batches of all these lengths, 192 MB to 3 GB, whole runs, separate
  // passes over fused kernels: Z = 32 and 64 1.03 to 1.46; from 128 on 0.81 to
  // 1.57, slower with the fused ones at Z = 192 (one block of 8 waves a CU),
  // with few angles to a block of fused_a, and where the last of fused_bc's
  // blocks leave most CUs empty. The sum below is a fit to the difference, in ns
  // per 10^6 bytes of Q (the separate passes take 1,000 to 1,400). Where it is
  // positive the ratio is 0.94 to 1.57, below 0.98 in 28 of 910; where it is
  // not, 0.81 to 1.14 in 255.
  if (Z < 128) return true;
  const int nb = bc_blocks(Y, Z) * fused_bc_groups(X, Y, Z, ka);
  const int y = (Y & (Y - 1)) == 0 ? 250 : Y < 200 ? 320 : 390;  // fused_bc's own time
  int gain = Z == 128 ? 480 : Z == 192 ? 390 : 580 - 500 / ka;
  if ((X & (X - 1)) == 0 && X > 128) gain += 50;
  return gain > y * ((nb + 255) / 256 * 256) / nb + 250 / a_angles(X, Y, Z, ka);
}

void fused_a(Twiddles& tw, hipStream_t s, const c32* Ty, const c32* Tyn, c32* Pn, const c32* FI, const c32* FIn,
             c32* Q, int X, int Y, int Z, int nz, int ka) {
  const int Xh = X / 2, R0 = plan_radix(Y, 0), T = 64 / R0;
  const int blocks = Xh / T * (Y / R0), apb = a_angles(X, Y, Z, ka);
  dispatch_z(Z, [&](auto Zc) {
    constexpr int L = decltype(Zc)::value;
    const dim3 bt(64 * waves_a(L));
    hipLaunchKernelGGL(k_fused_nyq<L>, dim3((Y + 63) / 64, ka), bt, 0, s, Tyn, FIn, Pn, z_list(tw, L), Y, nz);
    const dim3 g(blocks, (ka + apb - 1) / apb);
    if (R0 == 8)
      hipLaunchKernelGGL((k_fused_a<L, 8>), g, bt, 0, s, Ty, (const c32*)Pn, FI, Q, z_list(tw, L), Y, Xh, nz, ka, apb);
    else
      hipLaunchKernelGGL((k_fused_a<L, 4>), g, bt, 0, s, Ty, (const c32*)Pn, FI, Q, z_list(tw, L), Y, Xh, nz, ka, apb);
  });
  TOMHIP_CHECK(hipGetLastError());
}

void fused_bc(Twiddles& tw, hipStream_t s, const c32* Q, float* maxc, int32_t* argm, int X, int Y, int Z, int ka,
              int first_index, const long* desc, int apb, float* pv, uint8_t* pi) {
  dispatch_x(X / 2, [&](auto Xc) {
    dispatch_y(Y, [&](auto Yc) {
      constexpr int XH = decltype(Xc)::value, YL = decltype(Yc)::value;
      auto go = [&](auto kern) {
        hipLaunchKernelGGL(kern, dim3((unsigned)bc_blocks(YL, Z), (unsigned)((ka + apb - 1) / apb)),
                           dim3(64 * waves_bc(XH)), 0, s, Q, maxc, argm, bc_list(tw, X, YL), Z, ka, first_index, desc,
                           apb, pv, pi, (long)X * Y * Z);
      };
      if (pv)
        go(k_fused_bc<XH, YL, true>);
      else
        go(k_fused_bc<XH, YL, false>);
    });
  });
  TOMHIP_CHECK(hipGetLastError());
}

}  // namespace tomhip
