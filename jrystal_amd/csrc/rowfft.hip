// Row-buffer path of the fused evaluation, for cubic boxes (sides of
// JRX_ROW_SIZES, and 128).
//
// A state's 3D transform runs through a row buffer R[state][z][row], where
// the rows are the (x, y) lines along z that hold mask points (numbered in
// C order, so the mask points of a row are a contiguous range of g):
//   row_ifft        sphere -> inverse z transform of every row -> R
//   zplane_density  per z-plane: inverse y transform of the active x
//                   columns, inverse x transform of every y line,
//                   occupation-weighted |psi|^2 accumulated per state group
//   zplane_vpsi     the same inverse transforms, times v(r), forward x and
//                   y transforms back to the rows of R (in place)
//   row_fft_gather  forward z transform of every row, gather at the mask,
//                   qbar and the kinetic / band-energy partials
// R holds N * rows points per state (0.81 MB at 64^3 with 793 rows),
// against N * N * active planes (2.0 MB) for a buffer of y,z-transformed
// planes, and it is crossed four times per evaluation.  Densities and
// potentials on this path are z-major: [z][x][y].
#include "rowfft_kernels.h"

namespace jrx {

// Sides with an alias-free window only; 64 and 128 also take wider masks.
#define JRX_ROW_SIZES(X)                                                    \
  X(35) X(36) X(40) X(42) X(45) X(48) X(49) X(50) X(54) X(56) X(60) X(63)   \
  X(70) X(72) X(75) X(80)

// Mask window of the box: 2 or 1 (see rowfft_kernels.h), 0 for any mask of
// 64^3 and 128^3 boxes with at most 64 x-planes, -1 = no row path.
static int row_window(const BoxGeom& geo) {
  const int n = geo.nx;
  if (geo.ny != n || geo.nz != n || geo.nxa > 64 || geo.nrows <= 0 ||
      geo.nrows > 32767)
    return -1;
  const bool tight = geo.mmax <= n / 4 - 1, fits = geo.mmax <= n / 4;
  switch (n) {
    case 32:
      return tight ? 2 : fits ? 1 : -1;
    case 64:
    case 128:
      return tight ? 2 : (fits && n == 64) ? 1 : 0;
#define JRX_X(NN) case NN:
    JRX_ROW_SIZES(JRX_X)
#undef JRX_X
      return fits ? 1 : -1;
    default:
      return -1;
  }
}

bool use_rowpath(const BoxGeom& geo) { return row_window(geo) >= 0; }

// CALL(N, PR) of the box's kernels.
#define JRX_ROW_DISPATCH(CALL)                                              \
  switch (geo.nx * 4 + row_window(geo)) {                                   \
    case 32 * 4 + 1: return CALL(32, 1);                                    \
    case 32 * 4 + 2: return CALL(32, 2);                                    \
    case 64 * 4 + 0: return CALL(64, 0);                                    \
    case 64 * 4 + 1: return CALL(64, 1);                                    \
    case 64 * 4 + 2: return CALL(64, 2);                                    \
    case 128 * 4 + 0: return CALL(128, 0);                                  \
    case 128 * 4 + 2: return CALL(128, 2);                                  \
    JRX_ROW_SIZES(JRX_X)                                                    \
    default:                                                                \
      set_error("row path: unsupported box");                               \
      return JRX_ERR_UNSUPPORTED;                                           \
  }

int row_chunks(const BoxGeom& geo) {
  int rpb = 0;
  switch (geo.nx) {
#define JRX_X(NN) case NN: rpb = RowBlock<NN>::RPB; break;
    JRX_ROW_SIZES(JRX_X)
    JRX_X(32)
    JRX_X(64)
    JRX_X(128)
#undef JRX_X
    default: return 0;
  }
  return (geo.nrows + rpb - 1) / rpb;
}

int zplane_groups(const BoxGeom& geo, int nstates) {
  // about 2048 blocks (z-planes x groups) when every group gets 16 states
  // or more; with fewer states, fewer groups down to about 512 blocks, each
  // group then taking several states (one state per block repeats the
  // block's set-up for little work)
  const int hi = (2048 + geo.nz - 1) / geo.nz, lo = (512 + geo.nz - 1) / geo.nz;
  int G = nstates / 16;
  if (G > hi) G = hi;
  if (G < lo) G = lo;
  if (G > nstates) G = nstates;
  return G < 1 ? 1 : G;
}

int launch_row_ifft(const double2* q, double2* R, int64_t state0, int nstates,
                    const BoxGeom& geo, const double2* tw, hipStream_t s) {
#define JRX_CALL(NN, PR) RowPath<NN, PR>::ifft(q, R, state0, nstates, geo, tw, s)
#define JRX_X(NN) case NN * 4 + 1: return JRX_CALL(NN, 1);
  JRX_ROW_DISPATCH(JRX_CALL)
#undef JRX_X
#undef JRX_CALL
}

int launch_row_fft_gather(const double2* R, const double2* q, double2* qbar,
                          double* kin_partial, int64_t state0, int nstates,
                          const BoxGeom& geo, const double2* tw,
                          const GatherParams& gp, hipStream_t s) {
#define JRX_CALL(NN, PR)                                                    \
  RowPath<NN, PR>::gather(R, q, qbar, kin_partial, state0, nstates, geo, tw, \
                          gp, s)
#define JRX_X(NN) case NN * 4 + 1: return JRX_CALL(NN, 1);
  JRX_ROW_DISPATCH(JRX_CALL)
#undef JRX_X
#undef JRX_CALL
}

int launch_zplane_density(const double2* R, double* rho_part, int groups,
                          const double* occ, int64_t state0, int nstates,
                          double inv_vol, const BoxGeom& geo,
                          const double2* tw, bool store, hipStream_t s) {
#define JRX_CALL(NN, PR)                                                    \
  RowPath<NN, PR>::density(R, rho_part, groups, occ, state0, nstates,       \
                           inv_vol, geo, tw, store, s)
#define JRX_X(NN) case NN * 4 + 1: return JRX_CALL(NN, 1);
  JRX_ROW_DISPATCH(JRX_CALL)
#undef JRX_X
#undef JRX_CALL
}

int launch_zplane_vpsi(double2* R, const double* v, int groups, int nstates,
                       const BoxGeom& geo, const double2* tw, hipStream_t s) {
#define JRX_CALL(NN, PR) RowPath<NN, PR>::vpsi(R, v, groups, nstates, geo, tw, s)
#define JRX_X(NN) case NN * 4 + 1: return JRX_CALL(NN, 1);
  JRX_ROW_DISPATCH(JRX_CALL)
#undef JRX_X
#undef JRX_CALL
}

// out[s][c][r] = in[s][r][c] (32 x 32 tiles).
__global__ __launch_bounds__(256) void rotate_axes_kernel(
    const double* __restrict__ in, double* __restrict__ out, int nr, int nc) {
  __shared__ double tile[32][33];
  const int64_t base = (int64_t)blockIdx.z * nr * nc;
  const int c0 = blockIdx.x * 32, r0 = blockIdx.y * 32;
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;  // 32 x 8
  for (int k = ty; k < 32; k += 8) {
    const int r = r0 + k, c = c0 + tx;
    tile[k][tx] = (r < nr && c < nc) ? in[base + (int64_t)r * nc + c] : 0.0;
  }
  __syncthreads();
  for (int k = ty; k < 32; k += 8) {
    const int c = c0 + k, r = r0 + tx;
    if (r < nr && c < nc) out[base + (int64_t)c * nr + r] = tile[tx][k];
  }
}

int launch_rotate_axes(const double* in, double* out, int ns, int nr, int nc,
                       hipStream_t s) {
  hipLaunchKernelGGL(rotate_axes_kernel,
                     dim3((nc + 31) / 32, (nr + 31) / 32, ns), dim3(256), 0, s,
                     in, out, nr, nc);
  JRX_LAUNCH_CHECK();
  return JRX_OK;
}

}  // namespace jrx
