// Host-side launchers of the reciprocal/real-space energy kernels.
#pragma once
#include "common.h"

namespace jrx {

constexpr int kRedBlock = 256;

struct CellParams {
  int nx, ny, nz;
  double B[9];       // reciprocal basis rows, B = 2 pi A^{-T}
  double vol;
  int natom;
  const double* pos;     // device [natom*3]
  const double* charge;  // device [natom]
};

// out[i] = (sum_s rho[s*N + i], 0)
int launch_rho_to_complex(const double* rho, double2* out, int ns, int64_t N,
                          hipStream_t s);

// From rho_rec = fftn(rho_tot) build the reciprocal potential
//   vrec(G) = (4 pi vol / N) rho_rec / |G|^2 - 4 pi conj(S(G)) / (|G|^2+1e-10)
// (zero at G = 0; S(G) = sum_a Z_a e^{i G.R_a}) and per-block partials of
//   E_H   = (2 pi vol / N^2) sum_{G!=0} |rho_rec|^2 / |G|^2
//   E_ext = -(4 pi / N) sum_{G!=0} Re(S rho_rec) / (|G|^2 + 1e-10).
// vrec may alias rho_rec.  Returns the number of partials written.
// sterm (optional): S(G) / (|G|^2 + 1e-10) per box point, as
// launch_structure_term writes it; without it S(G) is formed per point.
int launch_potential_rec(const double2* rho_rec, double2* vrec,
                         double* eh_part, double* ee_part,
                         const CellParams& cp, int* nparts, hipStream_t s,
                         const double2* sterm = nullptr);

// out[i] = S(G_i) / (|G_i|^2 + 1e-10) (0 at G = 0) over cp's box: the
// geometry-only factor of the external term, formed once per plan.
int launch_structure_term(const CellParams& cp, double2* out, hipStream_t s);

// v_s(r) = Re(vbox(r)) + v_xc,s(r) and partials of E_xc (LDA exchange);
// ks: the spin-polarised v_xc in the Kohn-Sham form of the band driver
// (eps + rho_s d eps / d rho_s instead of d E_xc / d rho_s).
int launch_potential_real(const double2* vbox, const double* rho, double* v,
                          double* exc_part, int ns, int64_t N, double vol,
                          double cx, int* nparts, hipStream_t s,
                          bool ks = false);

// Partials of |G+k|^2 |q|^2, *nper per state (at most ceil(ng / kRedBlock)),
// band-major q.
int launch_kinetic(const double2* q, const double* kpts, const short* g_m,
                   const CellParams& cp, int64_t nstates, int ng, int nk,
                   int nb, double* kin_part, int* nper, hipStream_t s);

// tb[st] = sum_j part[st * nper + j]: sum_G |G+k|^2 |q|^2 of each state
// (twice the band kinetic energy).
int launch_state_sums(const double* part, int nper, int64_t S, double* tb,
                      hipStream_t s);

// energies[0..4] = kinetic (1/2 sum occ tb), hartree, external, xc, total
// from the partials (fixed summation order).  With kin, tb is first formed
// from its nper partials per state in the same launch; finalize_sums_states
// says where that one block is quicker than launch_state_sums (up to 256
// states of 128 partials, four passes of 64 states).
bool finalize_sums_states(int64_t S, int nper);
int launch_finalize_energies(const double* kin, int nper, double* tb,
                             const double* occ, int64_t S, const double* eh,
                             const double* ee, int nrec, const double* exc,
                             int nexc, double* energies, hipStream_t s);
// energies of the band mode: {1/2 sum occ tb, sum occ pot / vol, 0, 0, sum}
// (kin and pot_part as kin above, both or neither).
int launch_band_trace(const double* kin, const double* pot_part, int nper,
                      double* tb, double* pot, const double* occ, int64_t S,
                      double vol, double* energies, hipStream_t s);

int launch_fill(double* p, double v, int64_t n, hipStream_t s);

struct FftLen;
// The whole potential stage of LDA exchange in three launches (boxfft.hip),
// for boxes box_potential_size covers (two equal inner axes): (y, z) planes
// of the real density; x lines forward, potential_rec, inverse; planes back
// with potential_real at the points.  box is scratch; arguments and partials
// as in the separate launchers (L12: the length of both inner axes).
bool box_potential_size(const CellParams& cp);
int box_potential_lda(const double* rho, double2* box, double* v, double* eh,
                      double* ee, double* exc, int ns, double cx, bool ks,
                      const CellParams& cp, const double2* sterm,
                      const FftLen& L0, const FftLen& L12, int* nrec,
                      int* nexc, hipStream_t s);

// Exchange-correlation stage beyond LDA exchange (xc.hip), unpolarised.
bool xc_is_gga(int flags);
// gb[3][N] = ifftn(i G_d rho_rec) (the density gradient boxes; cp's box)
// (gvec, optional: the G grid [N][3] to use instead of cp's basis)
int xc_stage_gradients(const double2* rho_rec, double2* gb,
                       const CellParams& cp, const FftLen& L0,
                       const FftLen& L1, const FftLen& L2, hipStream_t s,
                       const double* gvec = nullptr);
// v = Re(vbox) (vbox may be NULL) + dE_xc/drho and partials of E_xc for
// the JRX_XC_* terms in flags; for GGA terms gb holds the gradient boxes on
// entry and is used as scratch.
int xc_stage_potential(const double2* vbox, const double* rho, double* v,
                       double2* gb, double* exc_part, int* nparts,
                       const CellParams& cp, int flags, const FftLen& L0,
                       const FftLen& L1, const FftLen& L2, hipStream_t s,
                       const double* gvec = nullptr);

// eps_x(n) = -cx n^(1/3) above the density threshold, else 0.
__device__ __forceinline__ double lda_x_eps(double n, double cx) {
  return n > 1e-15 ? -cx * cbrt(n) : 0.0;
}
__device__ __forceinline__ double lda_x_deps(double n, double cx) {
  if (!(n > 1e-15)) return 0.0;
  const double c = cbrt(n);
  return -cx / (3.0 * c * c);
}
// v at point i of N (all ns channels) from the Hartree + external potential
// vhe there, and the point's exchange energy; w = vol / N.
__device__ __forceinline__ double lda_x_point(
    double vhe, const double* __restrict__ rho, double* __restrict__ v,
    int64_t i, int64_t N, int ns, double w, double cx, int ks) {
  if (ns == 1) {
    const double r = rho[i];
    const double e = lda_x_eps(r, cx);
    v[i] = vhe + w * (4.0 / 3.0) * e;
    return w * e * r;
  }
  // Spin-polarised exchange as in xc.py:56-59: eps = (e(2ru)+e(2rd))/2
  // multiplies the total density.  v_s = d E / d rho_s = eps + rt
  // d eps / d rho_s; the Kohn-Sham form (ks) of the band driver is
  // vxc_lda (xc.py:109-124), eps + rho_s d eps / d rho_s.
  const double ru = rho[i], rd = rho[N + i];
  const double e = 0.5 * (lda_x_eps(2.0 * ru, cx) + lda_x_eps(2.0 * rd, cx));
  const double rt = ru + rd;
  v[i] = vhe + w * (e + (ks ? ru : rt) * lda_x_deps(2.0 * ru, cx));
  v[N + i] = vhe + w * (e + (ks ? rd : rt) * lda_x_deps(2.0 * rd, cx));
  return w * e * rt;
}

// Twiddle tables of the plan-less FFT entry points (a per-device cache).
int cached_fftlen(int n, FftLen* L);

}  // namespace jrx
