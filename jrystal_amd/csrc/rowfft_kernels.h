// Kernels of the row-buffer path (rowfft.hip): row passes, one set per length
// N of the z axis, and z-plane passes, one set per side N of the square (x, y)
// planes; each with the mask's window PR along the axes it transforms:
//   PR 1: every mask point has |m| <= N / 4 (a density box that is free of
//         aliasing); PR 2: |m| <= N / 4 - 1; PR 3: |m| <= 3 N / 8 - 1 (N = 64
//         only); PR 0: any mask (z-plane passes: of at most 64 x-planes;
//         N = 64 and 128 only).
// With a window, the first radix stage of an inverse transform has about half
// of its inputs and the last one of a forward transform about half of its
// outputs: the loads, stores and additions of the rest are not there.
#pragma once
#include "fft_kernels.h"
#include "regfft.h"

namespace jrx {

// Host launchers of one (N, PR); defined below, instantiated in
// rowfft_*.hip.
template <int N, int PR>
struct RowPass {
  static int ifft(const double2* q, double2* R, int64_t state0, int nstates,
                  const BoxGeom& geo, const double2* tw, hipStream_t s);
  static int gather(const double2* R, const double2* q, double2* qbar,
                    double* kin_partial, int64_t state0, int nstates,
                    const BoxGeom& geo, const double2* tw,
                    const GatherParams& gp, hipStream_t s);
};
template <int N, int PR>
struct ZPass {
  static int density(const double2* R, double* rho_part, int groups,
                     const double* occ, int64_t state0, int nstates,
                     double inv_vol, const BoxGeom& geo, const double2* tw,
                     bool store, hipStream_t s);
  static int vpsi(double2* R, const double* v, int groups, int nstates,
                  const BoxGeom& geo, const double2* tw, hipStream_t s);
};

// Rows per block of the row passes: four waves of 64 / L rows each, so that
// a block writes whole cache lines of every z-slice of R.
template <int N>
struct RowBlock {
  static constexpr int NW = 4;
  static constexpr int RPB = NW * RegLine<N>::LPW;
};

#ifdef JRX_ROWFFT_KERNELS

// Launch shape of the z-plane passes: NW and NWD, waves per block of the
// v(r) psi and the density pass (whole passes over the lines where they come
// out even, two or four waves where the last pass does not lose more); VR,
// whether v(r) of the lane's points stays in registers; PFV and PFD, whether
// the next state's inputs are prefetched into registers.  Each row is the
// fastest of the sets measured at 432 states of an alias-free cubic box
// (time per state and box point, density / v psi: 2.9 / 4.0 ps at 32, 2.9 /
// 5.1 at 45, 2.5 / 3.8 at 48, 1.9 / 3.1 at 64, 2.7 / 4.9 at 75); a set that
// spills many registers loses up to a factor of two.  Kernels that spill a few
// and are still the fastest measured: v psi of 42 points (4 registers; 1984
// states 639 us, without the prefetch and the spill 674) and the 128-point
// kernels without a window (density 24, v psi 4; 512 states of |m| <= 40:
// 2530 and 4500 us, and 4030 and 4490 with the y lines split over two blocks
// and LDS exchange).
template <int N>
struct ZShape;
#define JRX_ZSHAPE(NN, NW_, NWD_, VR_, PFV_, PFD_)                       \
  template <>                                                            \
  struct ZShape<NN> {                                                    \
    static constexpr int NW = NW_, NWD = NWD_;                           \
    static constexpr bool VR = VR_, PFV = PFV_, PFD = PFD_;              \
  };
JRX_ZSHAPE(32, 2, 2, 1, 1, 1)
JRX_ZSHAPE(35, 4, 4, 1, 1, 1)
JRX_ZSHAPE(36, 4, 4, 1, 1, 1)
JRX_ZSHAPE(40, 2, 2, 0, 0, 0)
JRX_ZSHAPE(42, 2, 2, 1, 1, 1)
JRX_ZSHAPE(45, 4, 4, 1, 0, 1)
JRX_ZSHAPE(48, 2, 3, 0, 0, 0)
JRX_ZSHAPE(49, 3, 3, 1, 1, 1)
JRX_ZSHAPE(50, 4, 4, 0, 0, 0)
JRX_ZSHAPE(54, 3, 3, 0, 1, 1)
JRX_ZSHAPE(56, 4, 4, 1, 1, 1)
JRX_ZSHAPE(60, 2, 2, 0, 1, 0)
JRX_ZSHAPE(63, 4, 4, 0, 1, 1)
JRX_ZSHAPE(64, 4, 4, 1, 1, 1)
JRX_ZSHAPE(70, 4, 4, 0, 1, 1)
JRX_ZSHAPE(72, 4, 4, 0, 1, 1)
JRX_ZSHAPE(75, 4, 4, 0, 0, 0)
JRX_ZSHAPE(80, 4, 6, 0, 0, 1)
JRX_ZSHAPE(128, 8, 8, 0, 0, 0)

// The window of the mask: lane j holds the nonzero inputs x = j + L m at
// m = 0 .. LO-1 and V-HI .. V-1; index i = 0 .. M-1 runs over those m.
template <int N, int PR>
struct Window {
  static constexpr int V = RegLine<N>::V, L = RegLine<N>::L;
  static constexpr int Q = PR == 3   ? 3 * N / 8 - 1
                           : PR == 2 ? N / 4 - 1
                                     : N / 4;
  static constexpr int LO = PR ? (Q + L) / L : V;  // ceil((Q + 1) / L)
  static constexpr int HI = PR ? (Q + L - 1) / L : 0;
  static constexpr int M = LO + HI;
  static_assert(M <= V, "window");
  __device__ static constexpr int m(int i) {
    return i < LO ? i : V - HI + (i - LO);
  }
  // slot j + L i of point z of the window
  __device__ __forceinline__ static int slot(int z) {
    return (PR == 0 || z < LO * L) ? z : z - (N - M * L);
  }
  static constexpr int WS = (M * L) | 1;  // LDS stride of a row's window
};

// ---------------------------------------------------------- row passes --
// LDS of a row pass: the windows of the block's rows, or (sizes that
// exchange through LDS) the rows' exchange slots, whichever is larger; the
// same space serves one after the other.
template <int N, int PR>
constexpr int row_lds_doubles() {
  constexpr int RPB = RowBlock<N>::RPB;
  constexpr int a = RPB * Window<N, PR>::WS * 2, b = RPB * RegLine<N>::XS;
  return a > b ? a : b;
}

// ------------------------------------------------------------ row_ifft --
// Block = RPB rows of one state: the mask points are scattered into zeroed
// LDS windows, each row is transformed along z by its L lanes, and the
// result goes to R[c][z][r0 .. r0 + RPB) straight from registers (the lanes
// of 64 / L neighbouring rows store 64 / L * 16 contiguous bytes; plain
// stores, whose partial lines the L2 merges).  Bound by HBM.
template <int N, int PR>
__global__ __launch_bounds__(RowBlock<N>::NW * 64) void row_ifft_kernel(
    const double2* __restrict__ q, double2* __restrict__ R, int64_t state0,
    BoxGeom geo, const double2* __restrict__ tab) {
  using F = RegLine<N>;
  using Wn = Window<N, PR>;
  constexpr int RPB = RowBlock<N>::RPB, NT = RowBlock<N>::NW * 64;
  constexpr int V = F::V, L = F::L, W = F::W, WS = Wn::WS;
  extern __shared__ double2 sm[];
  const LaneMap<N> lm;
  const int tid = threadIdx.x, j = lm.j, rl = lm.line();
  const int r0 = blockIdx.x * RPB;
  const int nr = min(RPB, geo.nrows - r0);
  const int c = blockIdx.y;
  const int64_t st = state0 + c;
  double2* row = sm + rl * WS;
  typename F::Tw tw;
  tw.init(tab, j);
  if (lm.on)
#pragma unroll
    for (int i = 0; i < Wn::M; ++i) row[j + L * i] = czero();
  __syncthreads();
  const int g0 = geo.row_g0[r0], g1 = geo.row_g0[r0 + nr];
  const double2* qs = q + st * geo.ng;
  for (int g = g0 + tid; g < g1; g += NT)
    sm[(geo.g_row[g] - r0) * WS + Wn::slot(geo.g_yz[g] % N)] = nt_load(qs + g);
  __syncthreads();
  double2 v[F::VP];
#pragma unroll
  for (int m = 0; m < V; ++m) v[m] = czero();
  if (lm.on)
#pragma unroll
    for (int i = 0; i < Wn::M; ++i) v[Wn::m(i)] = row[j + L * i];
  if constexpr (!F::kReg) __syncthreads();  // the windows become slots
  if (lm.on) {
    F::inverse(v, reinterpret_cast<double*>(sm) + rl * F::XS, j, tw);
    if (rl < nr) {
      double2* dst = R + (int64_t)c * N * geo.rstride + r0 + rl;
#pragma unroll
      for (int u = 0; u < W; ++u)
        if (F::alive(j, u))
#pragma unroll
          for (int b = 0; b < L; ++b)
            dst[(int64_t)(j + L * u + V * b) * geo.rstride] = v[u * L + b];
    }
  }
}

// ------------------------------------------------------- row_fft_gather --
// Block = RPB rows of one state: the rows of R[c][z][.] straight into
// registers, forward z transform, window to LDS, then qbar at the block's
// mask points and the block's partials of sum |G+k|^2 |q|^2 (and, with BE,
// of Re conj(q) h).  Bound by HBM.
template <int N, int PR, bool BE>
__global__ __launch_bounds__(RowBlock<N>::NW * 64) void row_fft_gather_kernel(
    const double2* __restrict__ R, const double2* __restrict__ q,
    double2* __restrict__ qbar, double* __restrict__ kin_partial,
    int64_t state0, BoxGeom geo, const double2* __restrict__ tab,
    GatherParams gp) {
  using F = RegLine<N>;
  using Wn = Window<N, PR>;
  constexpr int RPB = RowBlock<N>::RPB, NT = RowBlock<N>::NW * 64;
  constexpr int V = F::V, L = F::L, W = F::W, WS = Wn::WS;
  extern __shared__ double2 sm[];
  __shared__ double red[2 * (NT / 64)];
  const LaneMap<N> lm;
  const int tid = threadIdx.x, j = lm.j, rl = lm.line();
  const int r0 = blockIdx.x * RPB;
  const int nr = min(RPB, geo.nrows - r0);
  const int c = blockIdx.y;
  const int64_t st = state0 + c;
  double2 v[F::VP];
  if (lm.on) {
    // (rows past the end read the block's first row; nothing uses them)
    const double2* src =
        R + (int64_t)c * N * geo.rstride + r0 + (rl < nr ? rl : 0);
#pragma unroll
    for (int u = 0; u < W; ++u)
#pragma unroll
      for (int b = 0; b < L; ++b)
        v[u * L + b] =
            nt_load(src + (int64_t)(F::acol(j, u) + V * b) * geo.rstride);
    typename F::Tw tw;
    tw.init(tab, j);
    F::forward(v, reinterpret_cast<double*>(sm) + rl * F::XS, j, tw);
  }
  if constexpr (!F::kReg) __syncthreads();  // the slots become windows
  if (lm.on)
#pragma unroll
    for (int i = 0; i < Wn::M; ++i) sm[rl * WS + j + L * i] = v[Wn::m(i)];
  __syncthreads();
  const int g0 = geo.row_g0[r0], g1 = geo.row_g0[r0 + nr];
  const int k = (int)((st / gp.nb) % gp.nk);
  const double f = gp.occ[st];
  const double kx = gp.kpts[3 * k], ky = gp.kpts[3 * k + 1],
               kz = gp.kpts[3 * k + 2];
  const double2* qs = q + st * geo.ng;
  double2* qb = qbar + st * geo.ng;
  double kin = 0.0, pe = 0.0;
  for (int g = g0 + tid; g < g1; g += NT) {
    const int mx = gp.g_m[3 * g], my = gp.g_m[3 * g + 1],
              mz = gp.g_m[3 * g + 2];
    const double gx = mx * gp.B[0] + my * gp.B[3] + mz * gp.B[6] + kx;
    const double gy = mx * gp.B[1] + my * gp.B[4] + mz * gp.B[7] + ky;
    const double gz = mx * gp.B[2] + my * gp.B[5] + mz * gp.B[8] + kz;
    const double gk2 = gx * gx + gy * gy + gz * gz;
    const double2 cv = nt_load(qs + g);
    const double2 hv =
        sm[(geo.g_row[g] - r0) * WS + Wn::slot(geo.g_yz[g] % N)];
    nt_store(qb + g, make_double2(f * (gp.two_over_vol * hv.x + gk2 * cv.x),
                                  f * (gp.two_over_vol * hv.y + gk2 * cv.y)));
    kin += gk2 * (cv.x * cv.x + cv.y * cv.y);
    if constexpr (BE) pe += cv.x * hv.x + cv.y * hv.y;
  }
  const double wk = wave_sum(kin);
  const double wp = BE ? wave_sum(pe) : 0.0;
  if ((tid & 63) == 0) {
    red[lm.wave] = wk;
    if constexpr (BE) red[NT / 64 + lm.wave] = wp;
  }
  __syncthreads();
  if (tid == 0) {
    double a = 0.0, b = 0.0;
#pragma unroll
    for (int w = 0; w < NT / 64; ++w) {
      a += red[w];
      if constexpr (BE) b += red[NT / 64 + w];
    }
    kin_partial[st * gridDim.x + blockIdx.x] = a;
    if constexpr (BE) gp.pot_partial[st * gridDim.x + blockIdx.x] = b;
  }
}

// ------------------------------------------------------ z-plane passes --
// Block (z, state group).  LDS holds one z-plane P[y][xa] of the state in
// hand: the active x columns (compact), an odd row stride (lanes on 16
// neighbouring rows then hit distinct banks; those on neighbouring columns
// always do).  Lanes (column xa, j) own column xa in the y transforms,
// lanes (line y, j) row y in the x transforms.  With the exchanges in
// registers, LDS carries only the turn between the two directions.
template <int N, int PR, int NW_>
struct ZPlane {
  using F = RegLine<N>;
  using Wn = Window<N, PR>;
  static constexpr int V = F::V, L = F::L, W = F::W, VP = F::VP, M = Wn::M;
  static constexpr int NW = NW_, NT = NW * 64, LPP = NW * F::LPW;
  static constexpr int YP = (N + LPP - 1) / LPP;  // line passes
  // most active columns (at 128 points the path takes at most 64 x-planes)
  static constexpr int NXM = PR && 2 * Wn::Q + 1 < 64 ? 2 * Wn::Q + 1 : 64;
  static constexpr int CP = (NXM + LPP - 1) / LPP;
  static constexpr int RS = NXM | 1;
  static constexpr size_t kLds =
      (size_t)N * RS * sizeof(double2) +
      (size_t)NW * F::LPW * F::XS * sizeof(double);

  // Pairs of 16-bit signed indices per register, -1 = off the mask.
  struct Packed {
    unsigned w[(M + 1) / 2];
    __device__ __forceinline__ int operator[](int i) const {
      return (int)(short)(w[i >> 1] >> (16 * (i & 1)));
    }
    __device__ __forceinline__ void set(int i, int v) {
      const unsigned h = (unsigned)(v & 0xffff) << (16 * (i & 1));
      w[i >> 1] = (i & 1) ? ((w[i >> 1] & 0xffffu) | h) : h;
    }
  };

  double2* sm;   // P [N][RS]
  double* xch;   // this lane's line of exchange slots (LDS exchange only)
  LaneMap<N> lm;
  int cw;        // wave index of the column phases
  typename F::Tw tw;
  Packed ri[CP], xo;

  // The columns need fewer waves than the lines; which waves take them
  // turns with the block, so that the SIMDs of a CU share the work.
  __device__ __forceinline__ ZPlane(double2* lds, const BoxGeom& geo,
                                    const double2* __restrict__ tab)
      : sm(lds) {
    xch = reinterpret_cast<double*>(lds + N * RS) + lm.line() * F::XS;
    cw = lm.wave + (int)((blockIdx.x >> 3) + blockIdx.x + blockIdx.y) % NW;
    if (cw >= NW) cw -= NW;
    tw.init(tab, lm.j);
#pragma unroll
    for (int p = 0; p < CP; ++p) {
      const int xa = column(p);
#pragma unroll
      for (int i = 0; i < M; ++i)
        ri[p].set(i, lm.on && xa < geo.nxa
                         ? geo.rowidx[xa * N + lm.j + L * Wn::m(i)]
                         : -1);
    }
#pragma unroll
    for (int i = 0; i < M; ++i) xo.set(i, geo.xmap[lm.j + L * Wn::m(i)]);
  }
  __device__ __forceinline__ int column(int p) const {
    return cw * F::LPW + lm.l + p * LPP;
  }
  __device__ __forceinline__ int line(int p) const {
    return lm.line() + p * LPP;
  }
  __device__ __forceinline__ void load(double2 (&pre)[CP][M],
                                       const double2* src) const {
#pragma unroll
    for (int p = 0; p < CP; ++p)
#pragma unroll
      for (int i = 0; i < M; ++i) {
        const int r = ri[p][i];
        pre[p][i] = r >= 0 ? src[r] : czero();
      }
  }
  // Inverse y transform of the active columns (inputs in pre) into P.
  __device__ __forceinline__ void y_inverse(const double2 (&pre)[CP][M],
                                            int nxa) const {
#pragma unroll
    for (int p = 0; p < CP; ++p) {
      const int xa = column(p);
      if (lm.on && xa < nxa) {
        double2 v[VP];
#pragma unroll
        for (int m = 0; m < V; ++m) v[m] = czero();
#pragma unroll
        for (int i = 0; i < M; ++i) v[Wn::m(i)] = pre[p][i];
        F::inverse(v, xch, lm.j, tw);
        double2* col = sm + xa;
#pragma unroll
        for (int u = 0; u < W; ++u)
          if (F::alive(lm.j, u))
#pragma unroll
            for (int b = 0; b < L; ++b)
              col[(lm.j + L * u + V * b) * RS] = v[u * L + b];
      }
    }
  }
  // x transform of row y of P: v[u L + b] = psi(x = a + V b).
  __device__ __forceinline__ void x_inverse(double2 (&v)[VP], int y) const {
    const double2* row = sm + y * RS;
#pragma unroll
    for (int m = 0; m < V; ++m) v[m] = czero();
#pragma unroll
    for (int i = 0; i < M; ++i) {
      const int x = xo[i];
      v[Wn::m(i)] = x >= 0 ? row[x] : czero();
    }
    F::inverse(v, xch, lm.j, tw);
  }
};

// (two waves per SIMD: the register budget of the transforms)
template <int N, int PR, int NW, bool PF>
__global__ __launch_bounds__(NW * 64, 2) void zplane_density_kernel(
    const double2* __restrict__ R, double* __restrict__ rho_part,
    const double* __restrict__ occ, int64_t state0, int nstates,
    double inv_vol, BoxGeom geo, const double2* __restrict__ tab, int store) {
  using Z = ZPlane<N, PR, NW>;
  using F = RegLine<N>;
  constexpr int V = Z::V, L = Z::L, W = Z::W, YP = Z::YP;
  extern __shared__ double2 sm[];
  const int z = blockIdx.x;
  const int G = gridDim.y, gi = blockIdx.y;
  const int per = (nstates + G - 1) / G;
  const int cb = gi * per, ce = min(nstates, cb + per);
  double* part = rho_part + ((int64_t)gi * geo.nz + z) * N * N;  // [x][y]
  if (cb >= ce) {  // uniform over the block: an empty group
    if (store)
      for (int i = threadIdx.x; i < N * N; i += Z::NT) part[i] = 0.0;
    return;
  }
  const Z zp(sm, geo, tab);
  const int j = zp.lm.j;
  double acc[YP][Z::VP];
#pragma unroll
  for (int p = 0; p < YP; ++p)
#pragma unroll
    for (int t = 0; t < Z::VP; ++t) acc[p][t] = 0.0;
  const int64_t sstride = (int64_t)geo.nz * geo.rstride;
  const double2* src0 = R + (int64_t)z * geo.rstride;
  double2 pre[Z::CP][Z::M];
  if constexpr (PF) zp.load(pre, src0 + (int64_t)cb * sstride);
  for (int c = cb; c < ce; ++c) {
    if constexpr (!PF) zp.load(pre, src0 + (int64_t)c * sstride);
    zp.y_inverse(pre, geo.nxa);
    // the next state's column inputs fly during the line passes
    if constexpr (PF)
      if (c + 1 < ce) zp.load(pre, src0 + (int64_t)(c + 1) * sstride);
    __syncthreads();
    const double f = occ[state0 + c];
#pragma unroll
    for (int p = 0; p < YP; ++p) {
      const int y = zp.line(p);
      if (zp.lm.on && y < N) {
        double2 v[Z::VP];
        zp.x_inverse(v, y);
#pragma unroll
        for (int t = 0; t < Z::VP; ++t)
          acc[p][t] += f * (v[t].x * v[t].x + v[t].y * v[t].y);
      }
    }
    __syncthreads();
  }
  // the group's plane: stored by the first sweep chunk, added to after
#pragma unroll
  for (int p = 0; p < YP; ++p) {
    const int y = zp.line(p);
    if (zp.lm.on && y < N)
#pragma unroll
      for (int u = 0; u < W; ++u)
        if (F::alive(j, u))
#pragma unroll
          for (int b = 0; b < L; ++b) {
            double* dst = part + (j + L * u + V * b) * N + y;
            const double a = acc[p][u * L + b] * inv_vol;
            *dst = store ? a : *dst + a;
          }
  }
}

template <int N, int PR, int NW, bool VR, bool PF>
__global__ __launch_bounds__(NW * 64, 2) void zplane_vpsi_kernel(
    double2* __restrict__ R, const double* __restrict__ vpot, int nstates,
    BoxGeom geo, const double2* __restrict__ tab) {
  using Z = ZPlane<N, PR, NW>;
  using F = RegLine<N>;
  using Wn = Window<N, PR>;
  constexpr int V = Z::V, L = Z::L, W = Z::W, YP = Z::YP;
  extern __shared__ double2 sm[];
  const int z = blockIdx.x;
  const int G = gridDim.y, gi = blockIdx.y;
  const int per = (nstates + G - 1) / G;
  const int cb = gi * per, ce = min(nstates, cb + per);
  if (cb >= ce) return;  // uniform over the block
  const Z zp(sm, geo, tab);
  const int j = zp.lm.j;
  const double* vz = vpot + (int64_t)z * N * N;  // [x][y]
  // v(r) of the lane's points in registers, or read again for every state
  // (the lanes of neighbouring lines read neighbouring values)
  double vr[VR ? YP : 1][Z::VP];
  auto load_v = [&](double (&w)[Z::VP], int y) {
#pragma unroll
    for (int u = 0; u < W; ++u)
#pragma unroll
      for (int b = 0; b < L; ++b)
        w[u * L + b] = vz[(F::acol(j, u) + V * b) * N + y];
  };
  if constexpr (VR) {
#pragma unroll
    for (int p = 0; p < YP; ++p) load_v(vr[p], min(zp.line(p), N - 1));
  }
  const int64_t sstride = (int64_t)geo.nz * geo.rstride;
  double2* buf0 = R + (int64_t)z * geo.rstride;
  double2 pre[Z::CP][Z::M];
  if constexpr (PF) zp.load(pre, buf0 + (int64_t)cb * sstride);
  for (int c = cb; c < ce; ++c) {
    double2* buf = buf0 + (int64_t)c * sstride;
    if constexpr (!PF) zp.load(pre, buf);
    zp.y_inverse(pre, geo.nxa);
    if constexpr (PF)
      if (c + 1 < ce) zp.load(pre, buf + sstride);
    __syncthreads();
    auto line_pass = [&](int p) {
      const int y = zp.line(p);
      if (zp.lm.on && y < N) {
        double2 v[Z::VP];
        if constexpr (!VR) load_v(vr[0], y);
        zp.x_inverse(v, y);
#pragma unroll
        for (int t = 0; t < Z::VP; ++t) v[t] = cscale(v[t], vr[VR ? p : 0][t]);
        F::forward(v, zp.xch, j, zp.tw);
        double2* row = sm + y * Z::RS;
#pragma unroll
        for (int i = 0; i < Z::M; ++i) {
          const int x = zp.xo[i];
          if (x >= 0) row[x] = v[Wn::m(i)];
        }
      }
    };
    // v(r) in registers needs compile-time pass indices; otherwise the pass
    // loop stays rolled (code size)
    if constexpr (VR) {
#pragma unroll
      for (int p = 0; p < YP; ++p) line_pass(p);
    } else {
#pragma unroll 1
      for (int p = 0; p < YP; ++p) line_pass(p);
    }
    __syncthreads();
    // forward y transform of the active columns, back to the rows of R
    // (the lanes of a column are those that own it in y_inverse, so the
    // next state's y_inverse needs no barrier after this)
#pragma unroll
    for (int p = 0; p < Z::CP; ++p) {
      const int xa = zp.column(p);
      if (zp.lm.on && xa < geo.nxa) {
        const double2* col = sm + xa;
        double2 v[Z::VP];
#pragma unroll
        for (int u = 0; u < W; ++u)
#pragma unroll
          for (int b = 0; b < L; ++b)
            v[u * L + b] = col[(F::acol(j, u) + V * b) * Z::RS];
        F::forward(v, zp.xch, j, zp.tw);
        // Plain stores: the lanes of a column fill a cache line in several
        // stores, which the L2 merges (nontemporal stores wrote the parts
        // back separately: +50% writes).
#pragma unroll
        for (int i = 0; i < Z::M; ++i) {
          const int r = zp.ri[p][i];
          if (r >= 0) buf[r] = v[Wn::m(i)];
        }
      }
    }
  }
}

// ------------------------------------------------------------ launchers --
template <int N, int PR>
int RowPass<N, PR>::ifft(const double2* q, double2* R, int64_t state0,
                         int nstates, const BoxGeom& geo, const double2* tw,
                         hipStream_t s) {
  constexpr int RPB = RowBlock<N>::RPB;
  const size_t shm = row_lds_doubles<N, PR>() * sizeof(double);
  hipLaunchKernelGGL((row_ifft_kernel<N, PR>),
                     dim3((geo.nrows + RPB - 1) / RPB, nstates),
                     dim3(RowBlock<N>::NW * 64), shm, s, q, R, state0, geo,
                     tw);
  JRX_LAUNCH_CHECK();
  return JRX_OK;
}

template <int N, int PR>
int RowPass<N, PR>::gather(const double2* R, const double2* q, double2* qbar,
                           double* kin_partial, int64_t state0, int nstates,
                           const BoxGeom& geo, const double2* tw,
                           const GatherParams& gp, hipStream_t s) {
  constexpr int RPB = RowBlock<N>::RPB;
  const size_t shm = row_lds_doubles<N, PR>() * sizeof(double);
  const dim3 grid((geo.nrows + RPB - 1) / RPB, nstates),
      block(RowBlock<N>::NW * 64);
  if (gp.pot_partial)
    hipLaunchKernelGGL((row_fft_gather_kernel<N, PR, true>), grid, block, shm,
                       s, R, q, qbar, kin_partial, state0, geo, tw, gp);
  else
    hipLaunchKernelGGL((row_fft_gather_kernel<N, PR, false>), grid, block,
                       shm, s, R, q, qbar, kin_partial, state0, geo, tw, gp);
  JRX_LAUNCH_CHECK();
  return JRX_OK;
}

// 64-point masks of 33 or more x-planes: 512 threads, so that one column
// pass is enough.  With a window v psi then fits 128 registers without the
// prefetch, and two blocks share a CU; any mask takes 132 without it, so
// the next state's inputs are prefetched instead (180).  v psi of 2048
// states: |m| <= 17, PR 0 without prefetch 2650 us, with it 2310, PR 3 1900
// (with prefetch 2310); |m| <= 28, PR 0 without prefetch 3400, with it 2650.
template <int N, int PR>
struct ZWide {
  static constexpr bool value = N == 64 && PR != 2;
};

template <int N, int PR>
int ZPass<N, PR>::density(const double2* R, double* rho_part, int groups,
                            const double* occ, int64_t state0, int nstates,
                            double inv_vol, const BoxGeom& geo,
                            const double2* tw, bool store, hipStream_t s) {
  using S = ZShape<N>;
  constexpr int NW = ZWide<N, PR>::value ? 8 : S::NWD;
  constexpr bool PF = PR != 0 && PR != 3 && S::PFD;
  hipLaunchKernelGGL((zplane_density_kernel<N, PR, NW, PF>),
                     dim3(geo.nz, groups), dim3(NW * 64),
                     (ZPlane<N, PR, NW>::kLds), s, R, rho_part, occ, state0,
                     nstates, inv_vol, geo, tw, store ? 1 : 0);
  JRX_LAUNCH_CHECK();
  return JRX_OK;
}

template <int N, int PR>
int ZPass<N, PR>::vpsi(double2* R, const double* v, int groups, int nstates,
                         const BoxGeom& geo, const double2* tw,
                         hipStream_t s) {
  using S = ZShape<N>;
  constexpr bool wide = ZWide<N, PR>::value;
  constexpr int NW = wide ? 8 : S::NW;
  constexpr bool VR = S::VR, PF = wide ? PR == 0 : PR != 0 && S::PFV;
  hipLaunchKernelGGL((zplane_vpsi_kernel<N, PR, NW, VR, PF>),
                     dim3(geo.nz, groups), dim3(NW * 64),
                     (ZPlane<N, PR, NW>::kLds), s, R, v, nstates, geo, tw);
  JRX_LAUNCH_CHECK();
  return JRX_OK;
}
#endif  // JRX_ROWFFT_KERNELS

}  // namespace jrx
