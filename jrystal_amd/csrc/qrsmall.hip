// The small (nb x nb) matrices of the QR and its adjoint: Cholesky factor and
// inverse of the Gram matrices, and the factors of the adjoint, on 16 x 16
// tiles with FP64 MFMA.
#include "qr_kernels.h"
#include "qr_mfma.h"

namespace jrx {

// 1 / sqrt(a): the hardware estimate y with the first two terms of the series
// of (1 - r)^-1/2 in r = 1 - a y^2; NaN for a <= 0 (or NaN), so that a
// non-positive pivot poisons the factor as the IEEE sqrt does.
// Largest relative error over 2^20 values of 1 to 4 and of e^-100 to e^100:
// the estimate 5.2e-8, with the first term only (a Newton step) 4.1e-15 and
// 1.6e-16 low on average, with both 1.4e-16 (IEEE 1 / sqrt(a): 1.7e-16).
__device__ __forceinline__ double rsqrt_series(double a) {
  const double y = __builtin_amdgcn_rsq(a);
  const double r = fma(-a * y, y, 1.0);
  return a > 0.0 ? fma(y * r, fma(0.375, r, 0.5), y) : __builtin_nan("");
}

// ------------------------------------------------------------- tiles --
// A tile is 256 complex values, element (i, k) at i * 16 + (k ^ i): rows and
// columns are both free of bank conflicts for 16 lanes.
__device__ __forceinline__ int tile_at(int i, int k) {
  return i * 16 + (k ^ i);
}
// Complex accumulator of one tile: lane l holds rows 4 r + l / 16 (r < 4) of
// column l % 16.
struct TileAcc {
  d4 re, im;
  __device__ __forceinline__ TileAcc() : re(d4zero()), im(d4zero()) {}
  // += a b for one step of four in k: a = A[i = li][k], b = B[k][j = li]
  __device__ __forceinline__ void step(double2 a, double2 b) {
    re = mfma4(a.x, b.x, re);
    re = mfma4(-a.y, b.y, re);
    im = mfma4(a.x, b.y, im);
    im = mfma4(a.y, b.x, im);
  }
  // += A B (or A^H B) of two tiles in LDS
  template <bool AH>
  __device__ __forceinline__ void mul(const double2* A, const double2* B,
                                      int li, int lk) {
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const int k = 4 * s + lk;
      step(AH ? cconj(A[tile_at(k, li)]) : A[tile_at(li, k)],
           B[tile_at(k, li)]);
    }
  }
  __device__ __forceinline__ double2 at(int r) const {
    return make_double2(re[r], im[r]);
  }
  __device__ __forceinline__ void store(double2* C, int li, int lk) const {
#pragma unroll
    for (int r = 0; r < 4; ++r) C[tile_at(4 * r + lk, li)] = at(r);
  }
};

// Value of lane S of the lane's row of 16, in every lane of that row.
template <int S>
__device__ __forceinline__ double row_bcast(double v) {
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), 0x150 + S,
                                             0xf, 0xf, true);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), 0x150 + S,
                                             0xf, 0xf, true);
  return __hiloint2double(hi, lo);
}
// Values of the K-th row of 16 lanes, in all four rows.
template <int K>
__device__ __forceinline__ double rows_bcast(double v) {
  auto one = [](unsigned x) {
    const auto a = __builtin_amdgcn_permlane32_swap(x, x, false, false);
    const unsigned y = a[K >> 1];
    const auto b = __builtin_amdgcn_permlane16_swap(y, y, false, false);
    return b[K & 1];
  };
  return __hiloint2double((int)one((unsigned)__double2hiint(v)),
                          (int)one((unsigned)__double2loint(v)));
}
template <int LANE>
__device__ __forceinline__ double lane_value(double v) {
  return __hiloint2double(
      __builtin_amdgcn_readlane(__double2hiint(v), LANE),
      __builtin_amdgcn_readlane(__double2loint(v), LANE));
}

// Step S of the elimination of a 16 x 16 Hermitian positive tile on one
// wave: lane l holds row r = l % 16, columns 4 (l / 16) + q of A and of
// E = (product of the elimination steps).  f_r = A[r][S] / A[S][S] for the
// rows below; the rows' 1 / sqrt(pivot) collect in ysr.  n: rows of the tile
// inside the matrix (from row n on it is the identity, which no step changes:
// jrx_qr, 8 problems of 2000 rows, 1 band: 26.7 us with all 16 steps, 21.5).
template <int S>
__device__ __forceinline__ void chol_step(double2 (&a)[4], double2 (&e)[4],
                                          double& ysr, int r, int n) {
  constexpr int K = S >> 2, Q = S & 3;
  const double piv = lane_value<S + 16 * K>(a[Q].x);
  const double ys = rsqrt_series(piv);
  if (r == S) ysr = ys;
  if constexpr (S < 15) {
    if (S + 1 >= n) return;
    const double y = r > S ? ys : 0.0;
    const double2 f = make_double2(rows_bcast<K>(a[Q].x) * y * y,
                                   rows_bcast<K>(a[Q].y) * y * y);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const double2 pa =
          make_double2(row_bcast<S>(a[q].x), row_bcast<S>(a[q].y));
      const double2 pe =
          make_double2(row_bcast<S>(e[q].x), row_bcast<S>(e[q].y));
      a[q] = csub(a[q], cmul(f, pa));
      e[q] = csub(e[q], cmul(f, pe));
    }
    chol_step<S + 1>(a, e, ysr, r, n);
  }
}
// The tile (its factor R_dd aside) becomes X = R_dd^{-1} = E^H.
__device__ __forceinline__ void chol_tile(double2* C, int lane,
                                          int n) {
  const int r = lane & 15, g = lane >> 4;
  double2 a[4], e[4];
  double ysr = 1.0;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    a[q] = C[tile_at(r, 4 * g + q)];
    e[q] = make_double2(r == 4 * g + q ? 1.0 : 0.0, 0.0);
  }
  chol_step<0>(a, e, ysr, r, n);
#pragma unroll
  for (int q = 0; q < 4; ++q)
    C[tile_at(4 * g + q, r)] = make_double2(ysr * e[q].x, -ysr * e[q].y);
}

// One block per problem: S = R^H R (R upper) and X = R^{-1}, by 16-wide
// panels of the upper triangle's tiles in LDS.  Panel d:
//   tile (d, d) -> X_dd = R_dd^{-1} on one wave (16 elimination steps in
//   registers; lane broadcasts instead of LDS and barriers);
//   R_dJ = X_dd^H A_dJ, one tile per wave;
//   A_IJ -= R_dI^H R_dJ (d < I <= J), the first wave taking tile
//   (d+1, d+1) and factoring it while the others update the rest.
// Then X_IJ = -(sum_{I<=K<J} X_IK R_KJ) X_JJ column by column, in place.
// Two barriers a panel and two a column: the former kernels swept one column
// per barrier and measured 22 us at 28 bands, 370 us at 128; these chains
// are what bounds them (one block per problem).
// flag_out[p] = S is close to diagonal; flag_in[p] != 0: X = I; with L
// (upper triangular) the output is L X.
template <int T>
__global__ __launch_bounds__(T <= 2 ? 256 : T <= 4 ? 512 : 1024)
void chol_inv_kernel(const double2* __restrict__ S,
                     double2* __restrict__ rinv, int nb,
                     int* __restrict__ flag_out,
                     const int* __restrict__ flag_in,
                     const double2* __restrict__ lmul) {
  constexpr int NT = T <= 2 ? 256 : T <= 4 ? 512 : 1024, NW = NT / 64;
  extern __shared__ double2 sm[];  // upper tiles, row by row
  __shared__ double red[NW];
  const int64_t p = blockIdx.x;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int li = lane & 15, lk = lane >> 4;
  double2* out = rinv + p * nb * nb;
  const double2* Lp = lmul ? lmul + p * nb * nb : nullptr;
  if (flag_in && flag_in[p]) {  // uniform over the block: X = I
    for (int e = tid; e < nb * nb; e += NT) {
      const int i = e / nb, j = e - i * nb;
      out[e] = Lp ? Lp[e] : make_double2(i == j ? 1.0 : 0.0, 0.0);
    }
    return;
  }
  auto tile = [&](int I, int J) {
    return sm + 256 * (I * T - I * (I - 1) / 2 + (J - I));
  };
  const double2* Sp = S + p * nb * nb;
  double dist = 0.0;  // of the scaled Gram matrix from I
#pragma unroll 1
  for (int I = 0; I < T; ++I)
#pragma unroll 1
    for (int e = tid; e < 256 * (T - I); e += NT) {
      const int J = I + (e >> 8), i = (e >> 4) & 15, k = e & 15;
      const int r = 16 * I + i, c = 16 * J + k;
      // the lower half of a diagonal tile mirrors the upper one; beyond nb
      // the matrix continues as the identity
      double2 v = make_double2(r == c ? 1.0 : 0.0, 0.0);
      if (r < nb && c < nb) {
        v = r <= c ? Sp[r * nb + c] : cconj(Sp[c * nb + r]);
        if (flag_out && r < c)  // (r, c) and (c, r)
          dist += 2.0 * (v.x * v.x + v.y * v.y) /
                  (Sp[r * nb + r].x * Sp[c * nb + c].x);
      }
      tile(I, J)[tile_at(i, k)] = v;
    }
  if (flag_out) {
    const double d2 = block_sum(dist, red);
    if (tid == 0)  // NaN or a non-positive diagonal compares false
      flag_out[p] = (d2 < kQrOnePass * kQrOnePass) ? 1 : 0;
  }
  __syncthreads();
  if (wave == 0) chol_tile(tile(0, 0), lane, nb);
  __syncthreads();
#pragma unroll 1
  for (int d = 0; d + 1 < T; ++d) {
    for (int J = d + 1 + wave; J < T; J += NW) {
      TileAcc c;
      c.mul<true>(tile(d, d), tile(d, J), li, lk);
      wave_order();
      c.store(tile(d, J), li, lk);
    }
    __syncthreads();
    auto update = [&](int I, int J) {
      TileAcc c;
      c.mul<true>(tile(d, I), tile(d, J), li, lk);
      double2* C = tile(I, J);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        double2& x = C[tile_at(4 * r + lk, li)];
        x = csub(x, c.at(r));
      }
    };
    if (wave == 0) {
      update(d + 1, d + 1);
      wave_order();
      chol_tile(tile(d + 1, d + 1), lane, nb - 16 * (d + 1));
    } else {
      int n = 0;  // the other tiles, dealt to the other waves
      for (int I = d + 1; I < T; ++I)
        for (int J = I == d + 1 ? I + 1 : I; J < T; ++J, ++n)
          if (n % (NW - 1) == wave - 1) update(I, J);
    }
    __syncthreads();
  }
#pragma unroll 1
  for (int J = 1; J < T; ++J) {
    // (T <= NW: one row of tiles per wave)
    TileAcc c;
    if (wave < J) {
      for (int K = wave; K < J; ++K)
        c.mul<false>(tile(wave, K), tile(K, J), li, lk);
    }
    __syncthreads();  // column J of R is dead
    if (wave < J) {
      double2* C = tile(wave, J);
      c.store(C, li, lk);
      wave_order();
      TileAcc x;
      x.mul<false>(C, tile(J, J), li, lk);
      wave_order();
#pragma unroll
      for (int r = 0; r < 4; ++r)
        C[tile_at(4 * r + lk, li)] = make_double2(-x.re[r], -x.im[r]);
    }
    __syncthreads();
  }
  if (!Lp) {
    for (int e = tid; e < nb * nb; e += NT) {
      const int r = e / nb, c = e - r * nb;
      out[e] = c >= r ? tile(r >> 4, c >> 4)[tile_at(r & 15, c & 15)]
                      : czero();
    }
    return;
  }
  for (int t = wave; t < T * T; t += NW) {
    const int I = t / T, J = t - I * T;
    TileAcc c;
    for (int K = I; K <= J; ++K)
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        const int r = 16 * I + li, k = 16 * K + 4 * s + lk;
        c.step(r <= k && k < nb ? Lp[r * nb + k] : czero(),
               tile(K, J)[tile_at(4 * s + lk, li)]);
      }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int i = 16 * I + 4 * r + lk, j = 16 * J + li;
      if (i < nb && j < nb) out[i * nb + j] = j >= i ? c.at(r) : czero();
    }
  }
}

size_t chol_inv_lds_bytes(int nb) {
  const size_t T = (nb + 15) / 16;
  return T * (T + 1) / 2 * 256 * sizeof(double2) + 16 * sizeof(double);
}

int launch_chol_inv(const double2* S, double2* rinv, int64_t P, int nb,
                    hipStream_t s, int* flag_out, const int* flag_in,
                    const double2* lmul) {
  const int T = (nb + 15) / 16;
  const size_t shm = (size_t)T * (T + 1) / 2 * 256 * sizeof(double2);
#define JRX_CHOL(TT)                                                        \
  case TT:                                                                  \
    hipLaunchKernelGGL((chol_inv_kernel<TT>), dim3((unsigned)P),            \
                       dim3(TT <= 2 ? 256 : TT <= 4 ? 512 : 1024), shm, s,  \
                       S, rinv, nb, flag_out, flag_in, lmul);               \
    break;
  switch (T) {
    JRX_CHOL(1) JRX_CHOL(2) JRX_CHOL(3) JRX_CHOL(4)
    JRX_CHOL(5) JRX_CHOL(6) JRX_CHOL(7) JRX_CHOL(8)
    default:
      set_error("nb above 128 is not supported by this build");
      return JRX_ERR_UNSUPPORTED;
  }
#undef JRX_CHOL
  JRX_LAUNCH_CHECK();
  return JRX_OK;
}

// A = R^{-H} and B = copyltu(triu(-G)) R^{-H}, operands from global memory
// (L2): B_IJ = sum_{K >= J} M_IK (Ri_JK)^H, with M[i][k] = -G[i][k] above the
// diagonal, its mirror image below and -Re G[i][i] on it.  A_IJ = (Ri_JI)^H
// is the operand of K = I.
// Step s (of four in k) of the tiles (I, K) of M and (J, K) of Ri^H.
__device__ __forceinline__ void adjoint_step(const double2* Gp,
                                             const double2* Rp, int nb, int i,
                                             int j, int k, double2& a,
                                             double2& b) {
  a = b = czero();
  if (i < nb && k < nb) {
    const double2 g = i <= k ? Gp[i * nb + k] : Gp[k * nb + i];
    a = make_double2(-g.x, i < k ? -g.y : i > k ? g.y : 0.0);
  }
  if (j <= k && k < nb) b = cconj(Rp[j * nb + k]);
}

// One 16 x 16 tile per wave.
__global__ __launch_bounds__(256) void qr_bwd_small_kernel(
    const double2* __restrict__ G, const double2* __restrict__ rinv,
    double2* __restrict__ A, double2* __restrict__ Bm, int nb, int T) {
  const int64_t p = blockIdx.y;
  const int lane = threadIdx.x & 63, li = lane & 15, lk = lane >> 4;
  const int t =
      blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (t >= T * T) return;
  const int I = t / T, J = t - I * T;
  const double2* Gp = G + p * nb * nb;
  const double2* Rp = rinv + p * nb * nb;
  TileAcc c;
  double2 aij[4] = {czero(), czero(), czero(), czero()};
  const int i = 16 * I + li, j = 16 * J + li;
  for (int K = J; K < T; ++K) {
    double2 a[4], b[4];
#pragma unroll
    for (int s = 0; s < 4; ++s)
      adjoint_step(Gp, Rp, nb, i, j, 16 * K + 4 * s + lk, a[s], b[s]);
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      c.step(a[s], b[s]);
      if (K == I) aij[s] = b[s];
    }
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int ii = 16 * I + 4 * r + lk;
    if (ii < nb && j < nb) {
      const int64_t o = p * nb * nb + ii * nb + j;
      Bm[o] = c.at(r);
      A[o] = aij[r];
    }
  }
}

// The same for a single tile (nb <= 16): one step of four in k per wave, the
// four partial products added through LDS.  A wave alone takes its 16 matrix
// instructions one after another and was slower than a plain sum per entry
// (64 problems of 3000 rows, 16 bands, whole adjoint: 54.4 us with such sums,
// 56.2 with one wave, 53.4 so).
__global__ __launch_bounds__(256) void qr_bwd_tile_kernel(
    const double2* __restrict__ G, const double2* __restrict__ rinv,
    double2* __restrict__ A, double2* __restrict__ Bm, int nb) {
  __shared__ double2 part[3][4][64];
  const int64_t o = (int64_t)blockIdx.x * nb * nb;
  const int lane = threadIdx.x & 63, li = lane & 15, lk = lane >> 4;
  const int s = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int ii = 4 * s + lk;
  TileAcc c;
  double2 a, b;
  adjoint_step(G + o, rinv + o, nb, li, li, ii, a, b);
  c.step(a, b);
  if (ii < nb && li < nb) A[o + ii * nb + li] = b;
  if (s > 0)
#pragma unroll
    for (int r = 0; r < 4; ++r) part[s - 1][r][lane] = c.at(r);
  __syncthreads();
  if (s > 0) return;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const double2 v = cadd(cadd(c.at(r), part[0][r][lane]),
                           cadd(part[1][r][lane], part[2][r][lane]));
    if (4 * r + lk < nb && li < nb) Bm[o + (4 * r + lk) * nb + li] = v;
  }
}

int launch_qr_bwd_small(const double2* G, const double2* rinv, double2* A,
                        double2* Bm, int64_t P, int nb, hipStream_t s) {
  const int T = (nb + 15) / 16;
  if (T == 1)
    hipLaunchKernelGGL(qr_bwd_tile_kernel, dim3((unsigned)P), dim3(256), 0, s,
                       G, rinv, A, Bm, nb);
  else
    hipLaunchKernelGGL(qr_bwd_small_kernel,
                       dim3((T * T + 3) / 4, (unsigned)P), dim3(256), 0, s, G,
                       rinv, A, Bm, nb, T);
  JRX_LAUNCH_CHECK();
  return JRX_OK;
}

}  // namespace jrx
