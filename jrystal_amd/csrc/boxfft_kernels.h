// Full-box transforms by register lines: one-axis passes, (y, x) planes in one
// pass, and the potential stage's fused passes (boxfft.hip).
#pragma once
#include "energy_kernels.h"
#include "fft_kernels.h"
#include "regfft.h"

namespace jrx {

// Host launchers; defined below, instantiated in boxfft_*.hip.
template <int N>
struct BoxLine {
  // lines (o, q) at o os + q qs (q < Q), element stride es
  static int run(const double2* in, double2* out, int64_t nouter, int64_t os,
                 int64_t Q, int64_t qs, int64_t es, bool inverse,
                 double scale, const double2* tw, hipStream_t s);
  // forward, potential_rec, inverse along axis 0 of one box
  static int potential(double2* box, double* eh_part, double* ee_part,
                       const CellParams& cp, const double2* sterm,
                       double scale, const double2* tw, int* nparts,
                       hipStream_t s);
};
template <int N>
struct BoxPlane {
  // both axes of B planes of N x N; rin: the planes of sum_s rin[s] instead
  static int run(const double2* in, double2* out, int64_t B, bool inverse,
                 double scale, const double2* tw, hipStream_t s,
                 const double* rin, int ns);
  // inverse, then v = Re + v_x of rho (LDA exchange), exchange partials
  static int potential(const double2* box, const double* rho, double* v,
                       double* exc_part, int ns, int planes, double vol,
                       double cx, bool ks, const double2* tw,
                       hipStream_t s);
};

#ifdef JRX_BOXFFT_KERNELS

// ------------------------------------------------------------ one axis --
// One wave = 64 / L lines, straight from and to memory (lanes of
// neighbouring lines are adjacent on the strided axes; on the contiguous one
// a load instruction covers L neighbouring elements of each line and the
// rest of the cache line hits in the next ones).  No barrier, no LDS beyond
// the exchange of the sizes that need it.  Bound by HBM for a batch of
// boxes, by launch and latency for one.
template <int N, bool INV>
__global__ __launch_bounds__(256) void box_line_kernel(
    const double2* in, double2* out, int64_t lines, int64_t os, int64_t Q,
    int64_t qs, int64_t es, double scale, const double2* __restrict__ tab) {
  using F = RegLine<N>;
  constexpr int V = F::V, L = F::L, W = F::W;
  extern __shared__ double xsm[];
  const LaneMap<N> lm;
  const int j = lm.j;
  const int nw = blockDim.x >> 6;
  const int64_t line =
      ((int64_t)blockIdx.x * nw + lm.wave) * F::LPW + lm.l;
  if (!lm.on || line >= lines) return;
  typename F::Tw tw;
  tw.init(tab, j);
  const int64_t o = line / Q, q = line - o * Q;
  const int64_t off = o * os + q * qs;
  const double2* src = in + off;
  double2 v[F::VP];
#pragma unroll
  for (int m = 0; m < V; ++m) v[m] = src[(j + L * m) * es];
  F::template to_ab<INV>(v, xsm + lm.line() * F::XS, j, tw);
  double2* dst = out + off;
#pragma unroll
  for (int u = 0; u < W; ++u)
    if (F::alive(j, u))
#pragma unroll
      for (int b = 0; b < L; ++b)
        dst[(j + L * u + V * b) * es] = cscale(v[u * L + b], scale);
}

// Axis 0 of the potential box (n0 = N planes of NN points): forward, the
// Hartree and external terms at the line's G vectors (launch_potential_rec),
// inverse.  One wave per block, whose energy partials it writes.
template <int N>
__global__ __launch_bounds__(64) void box_potential_kernel(
    double2* box, double* __restrict__ eh_part, double* __restrict__ ee_part,
    CellParams cp, const double2* __restrict__ sterm, double scale,
    const double2* __restrict__ tab) {
  using F = RegLine<N>;
  constexpr int V = F::V, L = F::L, W = F::W;
  extern __shared__ double xsm[];
  const LaneMap<N> lm;
  const int j = lm.j;
  const int NN = cp.ny * cp.nz;
  const int p = blockIdx.x * F::LPW + lm.l;
  double eh = 0.0, ee = 0.0;
  if (lm.on && p < NN) {
    typename F::Tw tw;
    tw.init(tab, j);
    double2* col = box + p;
    double* x = xsm + lm.l * F::XS;
    double2 v[F::VP];
#pragma unroll
    for (int m = 0; m < V; ++m) v[m] = col[(int64_t)(j + L * m) * NN];
    F::template to_ab<false>(v, x, j, tw);
    auto fq = [](int i, int n) { return i < (n + 1) / 2 ? i : i - n; };
    const int iy = p / cp.nz, iz = p - iy * cp.nz;
    const int my = fq(iy, cp.ny), mz = fq(iz, cp.nz);
    const double dN = (double)NN * N;
    const double fh = 2.0 * M_PI * cp.vol / (dN * dN);
    const double fe = 4.0 * M_PI / dN;
#pragma unroll
    for (int u = 0; u < W; ++u)
      if (F::alive(j, u))
#pragma unroll
        for (int b = 0; b < L; ++b) {
          const int k = j + L * u + V * b;
          const int mx = fq(k, N);
          double g2 = 0.0;
#pragma unroll
          for (int d = 0; d < 3; ++d) {
            const double g =
                mx * cp.B[d] + my * cp.B[3 + d] + mz * cp.B[6 + d];
            g2 += g * g;
          }
          const double2 r = v[u * L + b];
          double2 w = czero();
          if (k != 0 || p != 0) {
            const double2 t = sterm[(int64_t)k * NN + p];
            const double inv_g2 = 1.0 / g2;
            eh += fh * (r.x * r.x + r.y * r.y) * inv_g2;
            ee -= fe * (t.x * r.x - t.y * r.y);
            const double ch = 4.0 * M_PI * cp.vol / dN * inv_g2;
            w = make_double2((ch * r.x - 4.0 * M_PI * t.x) * scale,
                             (ch * r.y + 4.0 * M_PI * t.y) * scale);
          }
          v[u * L + b] = w;
        }
    F::template from_ab<true>(v, x, j, tw);
#pragma unroll
    for (int m = 0; m < V; ++m) col[(int64_t)(j + L * m) * NN] = v[m];
  }
  eh = wave_sum(eh);
  ee = wave_sum(ee);
  if (threadIdx.x == 0) {
    eh_part[blockIdx.x] = eh;
    ee_part[blockIdx.x] = ee;
  }
}

// -------------------------------------------------------------- planes --
// Block = one N x N plane in LDS: contiguous axis first (rows from memory
// into registers), the other axis from LDS to memory, where neighbouring
// lanes hold neighbouring columns.  One pass over memory and one launch
// instead of two.
template <int N>
struct PlaneShape {
  using F = RegLine<N>;
  static constexpr int WV = (N + F::LPW - 1) / F::LPW;
  static constexpr int NW = WV < 8 ? WV : 8;  // waves per block
  static constexpr int LPP = NW * F::LPW, PASS = (N + LPP - 1) / LPP;
  static constexpr int PS = N | 1;
  static constexpr size_t kLds = (size_t)N * PS * sizeof(double2) +
                                 (size_t)LPP * F::XS * sizeof(double);
  static_assert(kLds <= 160 * 1024, "LDS");
};

// Rows of the plane at src (element e = row N + col through load(e)) into P.
template <int N, bool INV, class Load>
__device__ __forceinline__ void plane_rows(double2* sm, const LaneMap<N>& lm,
                                           double* x,
                                           const typename RegLine<N>::Tw& tw,
                                           Load load) {
  using S = PlaneShape<N>;
  using F = RegLine<N>;
  constexpr int V = F::V, L = F::L, W = F::W;
#pragma unroll 1
  for (int p = 0; p < S::PASS; ++p) {
    const int r = lm.line() + p * S::LPP;
    if (lm.on && r < N) {
      double2 v[F::VP];
#pragma unroll
      for (int m = 0; m < V; ++m) v[m] = load(r * N + lm.j + L * m);
      F::template to_ab<INV>(v, x, lm.j, tw);
#pragma unroll
      for (int u = 0; u < W; ++u)
        if (F::alive(lm.j, u))
#pragma unroll
          for (int b = 0; b < L; ++b)
            sm[r * S::PS + lm.j + L * u + V * b] = v[u * L + b];
    }
  }
}
// Columns of P; out(row, col, value) of every element of the result.
template <int N, bool INV, class Out>
__device__ __forceinline__ void plane_cols(const double2* sm,
                                           const LaneMap<N>& lm, double* x,
                                           const typename RegLine<N>::Tw& tw,
                                           Out out) {
  using S = PlaneShape<N>;
  using F = RegLine<N>;
  constexpr int V = F::V, L = F::L, W = F::W;
#pragma unroll 1
  for (int p = 0; p < S::PASS; ++p) {
    const int c = lm.line() + p * S::LPP;
    if (lm.on && c < N) {
      double2 v[F::VP];
#pragma unroll
      for (int m = 0; m < V; ++m) v[m] = sm[(lm.j + L * m) * S::PS + c];
      F::template to_ab<INV>(v, x, lm.j, tw);
#pragma unroll
      for (int u = 0; u < W; ++u)
        if (F::alive(lm.j, u))
#pragma unroll
          for (int b = 0; b < L; ++b)
            out(lm.j + L * u + V * b, c, v[u * L + b]);
    }
  }
}

template <int N, bool INV, bool REAL>
__global__ __launch_bounds__(PlaneShape<N>::NW * 64) void box_plane_kernel(
    const double2* in, double2* out, double scale,
    const double2* __restrict__ tab, const double* __restrict__ rin, int ns) {
  using F = RegLine<N>;
  extern __shared__ double2 sm[];
  const LaneMap<N> lm;
  double* x = reinterpret_cast<double*>(sm + N * PlaneShape<N>::PS) +
              lm.line() * F::XS;
  typename F::Tw tw;
  tw.init(tab, lm.j);
  const int64_t off = (int64_t)blockIdx.x * N * N;
  if constexpr (REAL) {
    const int64_t rn = (int64_t)gridDim.x * N * N;
    plane_rows<N, INV>(sm, lm, x, tw, [&](int e) {
      double r = 0.0;
      for (int c = 0; c < ns; ++c) r += rin[c * rn + off + e];
      return make_double2(r, 0.0);
    });
  } else {
    const double2* src = in + off;
    plane_rows<N, INV>(sm, lm, x, tw, [&](int e) { return src[e]; });
  }
  __syncthreads();
  double2* dst = out + off;
  plane_cols<N, INV>(sm, lm, x, tw, [&](int r, int c, double2 v) {
    dst[r * N + c] = cscale(v, scale);
  });
}

// The inverse planes of the potential box with the point kernel of
// launch_potential_real folded into the stores.
template <int N>
__global__ __launch_bounds__(PlaneShape<N>::NW * 64)
void box_plane_potential_kernel(
    const double2* __restrict__ box, const double* __restrict__ rho,
    double* __restrict__ vout, double* __restrict__ exc_part, int ns,
    double vol, double cx, int ks, const double2* __restrict__ tab) {
  using F = RegLine<N>;
  extern __shared__ double2 sm[];
  __shared__ double red[16];
  const LaneMap<N> lm;
  double* x = reinterpret_cast<double*>(sm + N * PlaneShape<N>::PS) +
              lm.line() * F::XS;
  typename F::Tw tw;
  tw.init(tab, lm.j);
  const int64_t off = (int64_t)blockIdx.x * N * N;
  const int64_t NT = (int64_t)gridDim.x * N * N;
  const double2* src = box + off;
  plane_rows<N, true>(sm, lm, x, tw, [&](int e) { return src[e]; });
  __syncthreads();
  double exc = 0.0;
  const double w = vol / (double)NT;
  plane_cols<N, true>(sm, lm, x, tw, [&](int r, int c, double2 a) {
    exc += lda_x_point(a.x, rho, vout, off + r * N + c, NT, ns, w, cx, ks);
  });
  const double t = block_sum(exc, red);
  if (threadIdx.x == 0) exc_part[blockIdx.x] = t;
}

// ------------------------------------------------------------ launchers --
template <int N>
int BoxLine<N>::run(const double2* in, double2* out, int64_t nouter,
                    int64_t os, int64_t Q, int64_t qs, int64_t es,
                    bool inverse, double scale, const double2* tw,
                    hipStream_t s) {
  using F = RegLine<N>;
  const int64_t lines = nouter * Q;
  const int64_t waves = (lines + F::LPW - 1) / F::LPW;
  // four waves a block, fewer where that leaves CUs without one
  const int nw = waves >= 1024 ? 4 : waves >= 512 ? 2 : 1;
  const int64_t blocks = (waves + nw - 1) / nw;
  if (blocks <= 0) return JRX_OK;
  if (blocks > 0x7fffffff) {
    set_error("FFT batch too large");
    return JRX_ERR_UNSUPPORTED;
  }
  const size_t shm = (size_t)nw * F::LPW * F::XS * sizeof(double);
  if (inverse)
    hipLaunchKernelGGL((box_line_kernel<N, true>), dim3((unsigned)blocks),
                       dim3(nw * 64), shm, s, in, out, lines, os, Q, qs, es,
                       scale, tw);
  else
    hipLaunchKernelGGL((box_line_kernel<N, false>), dim3((unsigned)blocks),
                       dim3(nw * 64), shm, s, in, out, lines, os, Q, qs, es,
                       scale, tw);
  JRX_LAUNCH_CHECK();
  return JRX_OK;
}

template <int N>
int BoxLine<N>::potential(double2* box, double* eh_part, double* ee_part,
                          const CellParams& cp, const double2* sterm,
                          double scale, const double2* tw, int* nparts,
                          hipStream_t s) {
  using F = RegLine<N>;
  const int blocks = (cp.ny * cp.nz + F::LPW - 1) / F::LPW;
  hipLaunchKernelGGL((box_potential_kernel<N>), dim3(blocks), dim3(64),
                     (size_t)F::LPW * F::XS * sizeof(double), s, box, eh_part,
                     ee_part, cp, sterm, scale, tw);
  JRX_LAUNCH_CHECK();
  *nparts = blocks;
  return JRX_OK;
}

template <int N>
int BoxPlane<N>::run(const double2* in, double2* out, int64_t B, bool inverse,
                     double scale, const double2* tw, hipStream_t s,
                     const double* rin, int ns) {
  using S = PlaneShape<N>;
  const dim3 grid((unsigned)B), block(S::NW * 64);
  if (rin)
    hipLaunchKernelGGL((box_plane_kernel<N, false, true>), grid, block,
                       S::kLds, s, in, out, scale, tw, rin, ns);
  else if (inverse)
    hipLaunchKernelGGL((box_plane_kernel<N, true, false>), grid, block,
                       S::kLds, s, in, out, scale, tw, rin, ns);
  else
    hipLaunchKernelGGL((box_plane_kernel<N, false, false>), grid, block,
                       S::kLds, s, in, out, scale, tw, rin, ns);
  JRX_LAUNCH_CHECK();
  return JRX_OK;
}

template <int N>
int BoxPlane<N>::potential(const double2* box, const double* rho, double* v,
                           double* exc_part, int ns, int planes, double vol,
                           double cx, bool ks, const double2* tw,
                           hipStream_t s) {
  using S = PlaneShape<N>;
  hipLaunchKernelGGL((box_plane_potential_kernel<N>), dim3(planes),
                     dim3(S::NW * 64), S::kLds, s, box, rho, v, exc_part, ns,
                     vol, cx, ks ? 1 : 0, tw);
  JRX_LAUNCH_CHECK();
  return JRX_OK;
}
#endif  // JRX_BOXFFT_KERNELS

}  // namespace jrx
