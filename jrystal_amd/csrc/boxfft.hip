// Which full-box transforms run as register lines and planes, and the
// potential stage's fused passes.
#include "boxfft_kernels.h"

namespace jrx {

#define JRX_PLANE_SIZES(X)                                                  \
  X(32) X(35) X(36) X(40) X(42) X(45) X(48) X(49) X(50) X(54) X(56) X(60)   \
  X(63) X(64) X(70) X(72) X(75) X(80)
#define JRX_LINE_SIZES(X)                                                   \
  JRX_PLANE_SIZES(X)                                                        \
  X(81) X(84) X(90) X(96) X(98) X(100) X(105) X(108) X(112) X(120) X(126)   \
  X(128)

bool box_line_size(int n) {
  switch (n) {
#define JRX_X(NN) case NN:
    JRX_LINE_SIZES(JRX_X)
#undef JRX_X
      return true;
    default:
      return false;
  }
}
bool box_plane_size(int n) { return n <= 80 && box_line_size(n); }

static int unsupported_size() {
  set_error("full-box transform: unsupported size");
  return JRX_ERR_UNSUPPORTED;
}

int box_line(const double2* in, double2* out, int64_t nouter, int64_t os,
             int64_t Q, int64_t qs, int64_t es, bool inverse, double scale,
             const FftLen& L, hipStream_t s) {
  switch (L.n) {
#define JRX_X(NN)                                                           \
  case NN:                                                                  \
    return BoxLine<NN>::run(in, out, nouter, os, Q, qs, es, inverse, scale, \
                            L.tw, s);
    JRX_LINE_SIZES(JRX_X)
#undef JRX_X
    default:
      return unsupported_size();
  }
}

int box_planes(const double2* in, double2* out, int64_t B, bool inverse,
               double scale, const FftLen& L, hipStream_t s,
               const double* rin, int ns) {
  if (B > 0x7fffffff) {
    set_error("FFT batch too large");
    return JRX_ERR_UNSUPPORTED;
  }
  switch (L.n) {
#define JRX_X(NN)                                                           \
  case NN:                                                                  \
    return BoxPlane<NN>::run(in, out, B, inverse, scale, L.tw, s, rin, ns);
    JRX_PLANE_SIZES(JRX_X)
#undef JRX_X
    default:
      return unsupported_size();
  }
}

bool box_potential_size(const CellParams& cp) {
  return cp.ny == cp.nz && box_plane_size(cp.ny) && box_line_size(cp.nx);
}

int box_potential_lda(const double* rho, double2* box, double* v, double* eh,
                      double* ee, double* exc, int ns, double cx, bool ks,
                      const CellParams& cp, const double2* sterm,
                      const FftLen& L0, const FftLen& L12, int* nrec,
                      int* nexc, hipStream_t s) {
  int rc = box_planes(nullptr, box, cp.nx, false, 1.0, L12, s, rho, ns);
  if (rc) return rc;
  const double scale = 1.0 / ((double)cp.nx * cp.ny * cp.nz);
  switch (cp.nx) {
#define JRX_X(NN)                                                           \
  case NN:                                                                  \
    rc = BoxLine<NN>::potential(box, eh, ee, cp, sterm, scale, L0.tw, nrec, \
                                s);                                         \
    break;
    JRX_LINE_SIZES(JRX_X)
#undef JRX_X
    default:
      rc = unsupported_size();
  }
  if (rc) return rc;
  *nexc = cp.nx;
  switch (cp.ny) {
#define JRX_X(NN)                                                           \
  case NN:                                                                  \
    return BoxPlane<NN>::potential(box, rho, v, exc, ns, cp.nx, cp.vol, cx, \
                                   ks, L12.tw, s);
    JRX_PLANE_SIZES(JRX_X)
#undef JRX_X
    default:
      return unsupported_size();
  }
}

}  // namespace jrx
