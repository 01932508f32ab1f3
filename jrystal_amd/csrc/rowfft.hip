// Row-buffer path of the fused evaluation, for boxes with square (x, y)
// planes (sides of JRX_Z_SIZES, 32, 64 and 128) and any of the JRX_ROW_SIZES
// along z.
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

// Lengths with an alias-free window (PR 1) only; 32, 64 and 128 also have the
// tighter one (PR 2), 64 the wider one (PR 3), 64 and 128 kernels for any
// mask (PR 0).
#define JRX_Z_SIZES(X)                                                      \
  X(35) X(36) X(40) X(42) X(45) X(48) X(49) X(50) X(54) X(56) X(60) X(63)   \
  X(70) X(72) X(75) X(80)
#define JRX_ROW_SIZES(X)                                                    \
  JRX_Z_SIZES(X)                                                            \
  X(81) X(84) X(90) X(96) X(98) X(100) X(105) X(108) X(112) X(120) X(126)

// Window of the largest |frequency| m along axes of n points (PR), -1 = none.
static int window_of(int n, int m, bool row) {
  const bool tight = m <= n / 4 - 1, fits = m <= n / 4;
  switch (n) {
    case 32:
      return tight ? 2 : fits ? 1 : -1;
    case 64:
      return tight ? 2 : fits ? 1 : m <= 3 * n / 8 - 1 ? 3 : 0;
    case 128:
      return tight ? 2 : 0;
#define JRX_X(NN) case NN:
    JRX_Z_SIZES(JRX_X)
      return fits ? 1 : -1;
    default:
      break;
  }
  switch (row ? n : 0) {
    JRX_ROW_SIZES(JRX_X)
#undef JRX_X
      return fits ? 1 : -1;
    default:
      return -1;
  }
}
static int row_window(const BoxGeom& geo) {
  return window_of(geo.nz, geo.mmax_z, true);
}
static int z_window(const BoxGeom& geo) {
  return window_of(geo.nx, geo.mmax_xy, false);
}

// Square planes, a window along every axis, and not beyond what the plane
// path takes unless cubic.  (The z-plane passes hold the active columns of a
// plane in LDS and row indices in 16 bits.)
bool use_rowpath(const BoxGeom& geo) {
  return geo.nx == geo.ny && geo.nxa <= 64 && geo.nrows > 0 &&
         geo.nrows <= 32767 &&
         (geo.nz == geo.nx || geo.ny * geo.nz <= kPlaneCap) &&
         row_window(geo) >= 0 && z_window(geo) >= 0;
}

static int unsupported_box() {
  set_error("row path: unsupported box");
  return JRX_ERR_UNSUPPORTED;
}

// CALL(N, PR) of the box: z-plane passes, row passes.
#define JRX_DISPATCH_COMMON(CALL)                                           \
  case 32 * 4 + 1: return CALL(32, 1);                                      \
  case 32 * 4 + 2: return CALL(32, 2);                                      \
  case 64 * 4 + 0: return CALL(64, 0);                                      \
  case 64 * 4 + 1: return CALL(64, 1);                                      \
  case 64 * 4 + 2: return CALL(64, 2);                                      \
  case 64 * 4 + 3: return CALL(64, 3);                                      \
  case 128 * 4 + 0: return CALL(128, 0);                                    \
  case 128 * 4 + 2: return CALL(128, 2);
#define JRX_Z_DISPATCH(CALL)                                                \
  switch (geo.nx * 4 + z_window(geo)) {                                     \
    JRX_DISPATCH_COMMON(CALL)                                               \
    JRX_Z_SIZES(JRX_X)                                                      \
    default: return unsupported_box();                                      \
  }
#define JRX_ROW_DISPATCH(CALL)                                              \
  switch (geo.nz * 4 + row_window(geo)) {                                   \
    JRX_DISPATCH_COMMON(CALL)                                               \
    JRX_ROW_SIZES(JRX_X)                                                    \
    default: return unsupported_box();                                      \
  }

int row_chunks(const BoxGeom& geo) {
  int rpb = 0;
  switch (geo.nz) {
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

// State groups of a z-plane pass: nz x G blocks, each with a run of states.
// The G of the least expected time,
//   blocks run by the busiest CU x states of the fullest group
//     x (1 + tail / blocks per CU) x (1 + setup / states per block),
// over at most max_blocks blocks: a number of blocks just below a multiple
// of the 256 CUs and a G that divides the states well, more and shorter
// blocks to even out the end of the pass, fewer to set up less (twiddles,
// row indices; density: a partial plane written per block).  A CU is not
// taken to be done faster with fewer blocks than `resident`.  Against fixed
// targets of 512 .. 2048 blocks with 16 states each (us, density + vpsi,
// before -> with this rule): 48^3, 112 states 127 -> 94; 60^3, 128 states
// 269 -> 168; 75^3, 1984 states 6180 -> 5750; 64^3, 2048 states 2350 -> 2230;
// 128^3, 128 states 1570 -> 1480.
struct GroupWeights {
  int max_blocks, resident;
  double tail, setup;
};
static int zplane_groups(const BoxGeom& geo, int nstates,
                         const GroupWeights& w) {
  constexpr int kCUs = 256;
  int most = w.max_blocks / geo.nz, best = 1;
  if (most > nstates) most = nstates;
  double least = 0;
  for (int G = 1; G <= most; ++G) {
    int rounds = (geo.nz * G + kCUs - 1) / kCUs;
    if (rounds < w.resident) rounds = w.resident;
    const int per = (nstates + G - 1) / G;
    const double cost =
        (double)rounds * per * (1 + w.tail / rounds) * (1 + w.setup / per);
    if (G == 1 || cost < least) {
      least = cost;
      best = G;
    }
  }
  return best;
}

// Passes of up to 4 waves a block (several blocks a CU): weights fitted to
// the times at 22 sizes of 32 to 80 points and 64 to 1984 states, every G up
// to 2304 blocks; on average within 2.2 % (density) and 1.4 % (vpsi) of the
// best G.  8 waves a block (128 points, wide masks of 64) fill a CU by one
// block; then as few blocks as keep the CUs full are best (128^3, 128 states,
// density: 545 us with 2 groups, 575 with 8, 621 with 16), and no tail shows.
// Two such blocks share a CU in the density pass of 64 points and in its v psi
// pass with a window: at 2048 states of |m| <= 17 the latter takes 2650 us
// with one block a CU (4 groups), 2040 with 8, 1970 with 16 and 1900 with 32.
static bool wide_blocks(const BoxGeom& geo) {
  return geo.nx == 128 || (geo.nx == 64 && z_window(geo) != 2);
}
// The partial planes are part of the workspace.  64 and 128 points gain
// nothing from more groups than one per 16 states above 512 blocks (64^3, 64
// states: 8 groups 41 us, 16 groups 44 us), so they stay within that.
int zplane_density_groups(const BoxGeom& geo, int nstates) {
  const bool wide = wide_blocks(geo);
  int most = 2048;
  if (geo.nx == 64 || geo.nx == 128) {
    const int few = (512 + geo.nz - 1) / geo.nz;
    most = geo.nz * (nstates / 16 > few ? nstates / 16 : few);
    if (most > 2048) most = 2048;
  }
  return zplane_groups(geo, nstates,
                       wide ? GroupWeights{most, geo.nx == 64 ? 2 : 1, 0.0, 2.0}
                            : GroupWeights{most, 1, 0.25, 0.4});
}
int zplane_vpsi_groups(const BoxGeom& geo, int nstates) {
  if (!wide_blocks(geo))
    return zplane_groups(geo, nstates, GroupWeights{3072, 1, 1.5, 0.4});
  const bool two = geo.nx == 64 && z_window(geo) != 0;
  return zplane_groups(geo, nstates,
                       two ? GroupWeights{2048, 2, 0.3, 0.4}
                           : GroupWeights{2048, 1, 0.0, 0.3});
}

int launch_row_ifft(const double2* q, double2* R, int64_t state0, int nstates,
                    const BoxGeom& geo, const double2* tw, hipStream_t s) {
#define JRX_CALL(NN, PR) RowPass<NN, PR>::ifft(q, R, state0, nstates, geo, tw, s)
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
  RowPass<NN, PR>::gather(R, q, qbar, kin_partial, state0, nstates, geo, tw, \
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
  ZPass<NN, PR>::density(R, rho_part, groups, occ, state0, nstates,       \
                           inv_vol, geo, tw, store, s)
#define JRX_X(NN) case NN * 4 + 1: return JRX_CALL(NN, 1);
  JRX_Z_DISPATCH(JRX_CALL)
#undef JRX_X
#undef JRX_CALL
}

int launch_zplane_vpsi(double2* R, const double* v, int groups, int nstates,
                       const BoxGeom& geo, const double2* tw, hipStream_t s) {
#define JRX_CALL(NN, PR) ZPass<NN, PR>::vpsi(R, v, groups, nstates, geo, tw, s)
#define JRX_X(NN) case NN * 4 + 1: return JRX_CALL(NN, 1);
  JRX_Z_DISPATCH(JRX_CALL)
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
