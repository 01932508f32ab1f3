// Batched CholeskyQR2 and the QR adjoint (FP64).
//
// The reference orthonormalises W = w_re + i w_im with a Householder QR
// (jrystal/_src/unitary_module.py:74-75).  The total energy is invariant
// under Q -> Q D (D diagonal unitary) and W -> W T (T invertible upper
// triangular), so any QR of W gives the same energy and gradient.
// CholeskyQR2 (Fukaya et al. 2014) maps the work onto Gram and small
// triangular products:
//   S1 = W^H W = R1^H R1,  S2 = (W R1^-1)^H (W R1^-1) = R2^H R2,
//   Q = W (R2 R1)^-1 = W R1^-1 R2^-1.
// Adjoint (PyTorch's form of Walter & Lehmann 2018 for a loss of Q only):
//   Wbar = (Qbar + Q copyltu(X)) R^-H,  X = triu(-Q^H Qbar),
//   copyltu(X) = X + X^H - Re diag(X).
#include "qr_kernels.h"
#include "qr_mfma.h"

#include <algorithm>

namespace jrx {

GramSplit gram_split(int64_t P, int ng, int nb, int unit) {
  const int tiles = (ng + kQrRows - 1) / kQrRows;
  // about 2048 blocks in all; the wide kernels do four to sixteen times
  // the work per row, and each chunk adds an nb x nb partial to reduce
  const int64_t target = nb > kNarrowBands ? 256 : 2048;
  int64_t want = (target + P - 1) / P;  // chunks per problem
  if (want < 1) want = 1;
  if (want > tiles) want = tiles;
  // whole 64-row tiles; for the wide kernels whole 16-row slabs, so that one
  // block a CU leaves no CU without (137 059 rows: 252 blocks instead of 238)
  if (unit <= 0) unit = nb > kNarrowBands ? 16 : kQrRows;
  const int units = (ng + unit - 1) / unit;
  GramSplit sp;
  sp.rows_per_chunk = (int)((units + want - 1) / want) * unit;
  sp.nchunk = (ng + sp.rows_per_chunk - 1) / sp.rows_per_chunk;
  return sp;
}


// Small nb x nb matrix into LDS, zero-padded to NBP x NBP.
__device__ __forceinline__ void load_small(double2* dst, const double2* src,
                                           int nb, int NBP) {
  for (int e = threadIdx.x; e < NBP * NBP; e += kQrBlock) {
    const int i = e / NBP, j = e - i * NBP;
    dst[e] = (i < nb && j < nb) ? src[i * nb + j] : czero();
  }
}

// ------------------------------------------------- wide kernels (nb > 64) --
// Threads of the wide Gram kernel: 512 at 8 tiles (128 bands: 36 or 64
// pairs over 8 waves, 5 or 8 per wave); below, 256 (the compiler keeps the
// accumulators in AGPRs there and spills at 512).
constexpr int gram_wide_block(int T) { return T == 8 ? 512 : 256; }

// Tile pairs (I, J) of the wide Gram kernels: HERM takes I <= J (row-major
// over the upper triangle; the result is Hermitian), otherwise all T x T.
// NZ blocks share one chunk's pairs, PW pairs to a wave (at most 9).
template <int T, bool HERM>
struct WidePairs {
  static constexpr int NW = gram_wide_block(T) / 64;
  static constexpr int NPAIR = HERM ? T * (T + 1) / 2 : T * T;
  static constexpr int NZ = (NPAIR + 9 * NW - 1) / (9 * NW);
  static constexpr int PW = (NPAIR + NW * NZ - 1) / (NW * NZ);
};

__device__ inline void decode_pair(int q, int T, bool herm, int* I, int* J) {
  if (!herm) {
    *I = q / T;
    *J = q - *I * T;
    return;
  }
  int i = 0;
  while (q >= T - i) {
    q -= T - i;
    ++i;
  }
  *I = i;
  *J = i + q;
}

// Rows per LDS slab of the wide Gram kernel: 16 for a Hermitian result
// (one staged matrix), 8 for Q^H Qbar (two), so that the two slab buffers
// fit twice per CU.
template <bool HERM>
constexpr int wide_slab() { return HERM ? 16 : 8; }

// Partial Gram sums over a chunk's rows, one partial per chunk:
//   GMAJOR: S = W^H W (W planar g-major, the Hermitian pairs only);
//   else:   G = A^H B (A, B band-major complex; HERM when B is A).
// Row slabs are staged in LDS ([row][NBP + 1]), double-buffered: the next
// slab's global loads are in flight in registers while the MFMAs run on
// the current one, one barrier per slab.  Each wave accumulates its own
// tile pairs and writes them (and, for HERM, their mirror images).
template <int T, bool GMAJOR, bool HERM>
__global__ __launch_bounds__(gram_wide_block(T)) void gram_wide_kernel(
    const double* __restrict__ wr, const double* __restrict__ wi,
    const double2* __restrict__ qa, const double2* __restrict__ qb,
    double2* __restrict__ partial, int ng, int nb, int rows_per_chunk,
    int nchunk, const int* __restrict__ skip) {
  using PL = WidePairs<T, HERM>;
  constexpr int NBP = 16 * T, LD = NBP + 1, PW = PL::PW;
  constexpr int SR = wide_slab<HERM>();
  constexpr int NS = SR * NBP;                        // elements per slab
  constexpr int BLK = gram_wide_block(T);
  constexpr int NE = (NS + BLK - 1) / BLK;  // elements per thread
  constexpr int BUF = (HERM ? 1 : 2) * SR * LD;       // one slab buffer
  extern __shared__ double2 sm[];
  // (the wave index through readfirstlane: the pair tables are scalars)
  const int lane = threadIdx.x & 63,
            wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int li = lane & 15, lk = lane >> 4;
  const int64_t p = blockIdx.y;
  const int chunk = blockIdx.x;
  if (skip && skip[p]) return;  // uniform over the block
  int pI[PW], pJ[PW];
  bool live[PW];
#pragma unroll
  for (int t = 0; t < PW; ++t) {
    // dealt round: waves w and w + 4 share a SIMD, 9 of 36 pairs to each
    const int q = (t * PL::NZ + (int)blockIdx.z) * PL::NW + wave;
    live[t] = q < PL::NPAIR;  // uniform over the wave
    decode_pair(live[t] ? q : 0, T, HERM, &pI[t], &pJ[t]);
  }
  d4 re[PW], im[PW];
#pragma unroll
  for (int t = 0; t < PW; ++t) { re[t] = d4zero(); im[t] = d4zero(); }
  const int gb = chunk * rows_per_chunk;
  const int ge = min(ng, gb + rows_per_chunk);
  const double* Wr = wr + p * ng * nb;
  const double* Wi = wi + p * ng * nb;
  const double2* A = qa + p * nb * ng;
  const double2* B = qb + p * nb * ng;
  double2 ra[NE], rb[HERM ? 1 : NE];
  // slab element e: GMAJOR row e / NBP, band e % NBP (consecutive threads
  // read consecutive bands of a row); band-major band e / SR, row e % SR
  // (consecutive threads read consecutive rows of a band)
  auto fetch = [&](int g0) {
#pragma unroll
    for (int i = 0; i < NE; ++i) {
      const int e = threadIdx.x + i * BLK;
      const int r = GMAJOR ? e / NBP : e % SR;
      const int c = GMAJOR ? e % NBP : e / SR;
      const int g = g0 + r;
      const bool ok = e < NS && g < ge && c < nb;
      if (GMAJOR) {
        ra[i] = ok ? make_double2(Wr[(int64_t)g * nb + c], Wi[(int64_t)g * nb + c])
                   : czero();
      } else {
        ra[i] = ok ? A[(int64_t)c * ng + g] : czero();
        if (!HERM) rb[i] = ok ? B[(int64_t)c * ng + g] : czero();
      }
    }
  };
  auto store = [&](int buf) {
    double2* sa = sm + buf * BUF;
#pragma unroll
    for (int i = 0; i < NE; ++i) {
      const int e = threadIdx.x + i * BLK;
      if (e < NS) {
        const int r = GMAJOR ? e / NBP : e % SR;
        const int c = GMAJOR ? e % NBP : e / SR;
        sa[r * LD + c] = ra[i];
        if (!HERM) sa[SR * LD + r * LD + c] = rb[i];
      }
    }
  };
  if (gb < ge) {
    fetch(gb);
    store(0);
  }
  __syncthreads();
  int buf = 0;
  for (int g0 = gb; g0 < ge; g0 += SR) {
    const bool more = g0 + SR < ge;  // uniform over the block
    if (more) fetch(g0 + SR);
    const double2* sa = sm + buf * BUF;
    const double2* sb = HERM ? sa : sa + SR * LD;
#pragma unroll
    for (int r = 0; r < SR / 4; ++r) {
      const double2* ra4 = sa + (4 * r + lk) * LD + li;
      const double2* rb4 = sb + (4 * r + lk) * LD + li;
#pragma unroll
      for (int t = 0; t < PW; ++t) {
        if (!live[t]) continue;
        const double2 a = ra4[16 * pI[t]], b = rb4[16 * pJ[t]];
        // conj(a) b
        re[t] = mfma4(a.x, b.x, re[t]);
        re[t] = mfma4(a.y, b.y, re[t]);
        im[t] = mfma4(a.x, b.y, im[t]);
        im[t] = mfma4(-a.y, b.x, im[t]);
      }
    }
    // the other buffer was last read before the previous barrier
    if (more) store(buf ^ 1);
    __syncthreads();
    buf ^= 1;
  }
  double2* out = partial + (p * nchunk + chunk) * nb * nb;
#pragma unroll
  for (int t = 0; t < PW; ++t) {
    if (!live[t]) continue;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int i = 16 * pI[t] + 4 * r + lk, j = 16 * pJ[t] + li;
      if (i < nb && j < nb) {
        const double2 v = make_double2(re[t][r], im[t][r]);
        out[i * nb + j] = v;
        if (HERM && pI[t] < pJ[t]) out[j * nb + i] = cconj(v);
      }
    }
  }
}

// GMAJOR when wr is given (qa, qb unused), else band-major qa, qb (HERM when
// qa == qb).
int launch_gram_wide(const double* wr, const double* wi, const double2* qa,
                     const double2* qb, double2* partial, int64_t P, int ng,
                     int nb, const GramSplit& sp, hipStream_t s,
                     const int* skip) {
  const int T = (nb + 15) / 16;
  const bool gmajor = wr != nullptr, herm = gmajor || qa == qb;
  // two slab buffers of one (HERM) or two staged matrices
  const size_t shm = 2 * (herm ? 1 : 2) *
                     (size_t)(herm ? wide_slab<true>() : wide_slab<false>()) *
                     (16 * T + 1) * sizeof(double2);
#define JRX_GRAM_WIDE(TT, GM, HM)                                            \
  hipLaunchKernelGGL((gram_wide_kernel<TT, GM, HM>),                         \
                     dim3(sp.nchunk, (unsigned)P, WidePairs<TT, HM>::NZ),    \
                     dim3(gram_wide_block(TT)), shm, s, wr, wi, qa, qb,     \
                     partial, ng, nb,                                        \
                     sp.rows_per_chunk, sp.nchunk, skip)
#define JRX_GRAM_WIDE_T(TT)                              \
  if (gmajor) JRX_GRAM_WIDE(TT, true, true);             \
  else if (herm) JRX_GRAM_WIDE(TT, false, true);         \
  else JRX_GRAM_WIDE(TT, false, false);
  switch (T) {
    case 5: JRX_GRAM_WIDE_T(5) break;
    case 6: JRX_GRAM_WIDE_T(6) break;
    case 7: JRX_GRAM_WIDE_T(7) break;
    case 8: JRX_GRAM_WIDE_T(8) break;
    default:
      set_error("nb above 128 is not supported by this build");
      return JRX_ERR_UNSUPPORTED;
  }
#undef JRX_GRAM_WIDE_T
#undef JRX_GRAM_WIDE
  JRX_LAUNCH_CHECK();
  return JRX_OK;
}

constexpr int kWideRows = 64;  // g rows per block of the wide apply kernels

// apply_fwd_kernel for nb > 64.  One 16-row slab of W per wave; rinv is
// staged in LDS by chunks of 16 rows (the tiles on and right of the
// diagonal), double-buffered: the next chunk of rinv and of the wave's W
// is in flight in registers while the MFMAs run on the current one.  The
// chunks are unrolled, so that the triangular tile loop has no branch (a
// branch costs copies of the accumulators, which wait for the matrix unit).
// k of an MFMA step is 16 c + 4 lk + m: a lane's four W values are adjacent.
// FP64 MFMA bound: 137 059 x 128: 340 us before (43 % MFMA
// busy), 210 now (67 %).
template <int T>
__global__ __launch_bounds__(kQrBlock) void apply_fwd_wide_kernel(
    const double* __restrict__ wr, const double* __restrict__ wi,
    const double2* __restrict__ rinv, double2* __restrict__ q, int ng, int nb,
    const int* __restrict__ skip) {
  extern __shared__ double2 sm[];  // [2][16][NBP]
  constexpr int NBP = 16 * T;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int li = lane & 15, lk = lane >> 4;
  const int sk = threadIdx.x >> 4, sj = threadIdx.x & 15;  // staged element
  const int64_t p = blockIdx.y;
  if (skip && skip[p]) return;  // uniform over the block
  const double2* Rp = rinv + p * nb * nb;
  const int g0 = blockIdx.x * kWideRows + wave * 16;
  const int row = g0 + li;
  const double* Wr = wr + (p * ng + row) * nb;
  const double* Wi = wi + (p * ng + row) * nb;
  double2* Q = q + p * nb * ng;
  double2 st[T];
  double ar[2][4], ai[2][4];
  auto fetch = [&](int c, double (&xr)[4], double (&xi)[4]) {
    const int k = 16 * c + sk;
#pragma unroll
    for (int J = c; J < T; ++J) {
      const int b = 16 * J + sj;
      st[J] = (k < nb && b < nb) ? Rp[k * nb + b] : czero();
    }
#pragma unroll
    for (int m = 0; m < 4; ++m) {
      const int col = 16 * c + 4 * lk + m;
      const bool ok = row < ng && (c < T - 1 || col < nb);
      xr[m] = ok ? Wr[col] : 0.0;
      xi[m] = ok ? Wi[col] : 0.0;
    }
  };
  d4 qre[T], qim[T];
#pragma unroll
  for (int J = 0; J < T; ++J) { qre[J] = d4zero(); qim[J] = d4zero(); }
  fetch(0, ar[0], ai[0]);
#pragma unroll
  for (int c = 0; c < T; ++c) {
    double2* buf = sm + (c & 1) * 16 * NBP;
    // (buffer c & 1 was last read before the barrier of chunk c - 1)
#pragma unroll
    for (int J = c; J < T; ++J) buf[sk * NBP + 16 * J + sj] = st[J];
    __syncthreads();
    if (c + 1 < T) fetch(c + 1, ar[(c + 1) & 1], ai[(c + 1) & 1]);
#pragma unroll
    for (int m = 0; m < 4; ++m) {
      const double a_r = ar[c & 1][m], a_i = ai[c & 1][m];
#pragma unroll
      for (int J = c; J < T; ++J) {  // rinv[k][b] = 0 for k > b
        const double2 rv = buf[(4 * lk + m) * NBP + 16 * J + li];
        qre[J] = mfma4(rv.x, a_r, qre[J]);
        qim[J] = mfma4(rv.x, a_i, qim[J]);
        qre[J] = mfma4(-rv.y, a_i, qre[J]);
        qim[J] = mfma4(rv.y, a_r, qim[J]);
      }
    }
  }
  if (row >= ng) return;
#pragma unroll
  for (int J = 0; J < T; ++J)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int b = 16 * J + 4 * r + lk;
      if (J < T - 1 || b < nb)
        Q[(int64_t)b * ng + row] = make_double2(qre[J][r], qim[J][r]);
    }
}

// apply_bwd_kernel for nb > 64.  As apply_fwd_wide_kernel, with A (lower
// triangular: the tiles left of and on the diagonal) and Bm staged side by
// side; two waves share a 16-row slab, one the even and one the odd column
// tiles (an even and an odd wave to each SIMD), so that a block of eight
// waves, whose LDS fills a CU, still takes only 64 rows (137 059 rows are
// 8.4 such blocks a CU).
// FP64 MFMA bound: 137 059 x 128: 678 us before (57 % MFMA
// busy), 535 now (73 %).
constexpr int kWideBwdBlock = 512;
template <int T>
__global__ __launch_bounds__(kWideBwdBlock) void apply_bwd_wide_kernel(
    const double2* __restrict__ qbar, const double2* __restrict__ q,
    const double2* __restrict__ A, const double2* __restrict__ Bm,
    double* __restrict__ dwr, double* __restrict__ dwi, int ng, int nb) {
  extern __shared__ double2 sm[];  // [2][2][16][NBP]
  constexpr int NBP = 16 * T, TH = (T + 1) / 2;
  // (the wave index through readfirstlane: branches on it are scalar)
  const int lane = threadIdx.x & 63,
            wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int li = lane & 15, lk = lane >> 4, odd = (wave ^ (wave >> 2)) & 1;
  const int sk = (threadIdx.x >> 4) & 15, sj = threadIdx.x & 15;
  const int mat = wave >> 2;  // staged matrix: 0 = A, 1 = Bm
  const int64_t p = blockIdx.y;
  const double2* Sp = (mat ? Bm : A) + p * nb * nb;
  const int g0 = blockIdx.x * kWideRows + (wave >> 1) * 16;
  const int g = g0 + li;
  const double2* Qb = qbar + p * nb * ng + g;
  const double2* Q = q + p * nb * ng + g;
  double* Dr = dwr + p * ng * nb;
  double* Di = dwi + p * ng * nb;
  double2 st[T], vb[2][4], vq[2][4];
  auto fetch = [&](int c, double2 (&xb)[4], double2 (&xq)[4]) {
    const int k = 16 * c + sk;
#pragma unroll
    for (int J = 0; J < T; ++J) {
      const int b = 16 * J + sj;
      st[J] = (k < nb && b < nb && (J <= c || mat)) ? Sp[k * nb + b] : czero();
    }
#pragma unroll
    for (int m = 0; m < 4; ++m) {
      const int band = 16 * c + 4 * m + lk;
      const bool ok = g < ng && (c < T - 1 || band < nb);
      xb[m] = ok ? Qb[(int64_t)band * ng] : czero();
      xq[m] = ok ? Q[(int64_t)band * ng] : czero();
    }
  };
  d4 re[TH], im[TH];
#pragma unroll
  for (int h = 0; h < TH; ++h) { re[h] = d4zero(); im[h] = d4zero(); }
  fetch(0, vb[0], vq[0]);
#pragma unroll
  for (int c = 0; c < T; ++c) {
    double2* buf = sm + (c & 1) * 2 * 16 * NBP;
    // (buffer c & 1 was last read before the barrier of chunk c - 1)
#pragma unroll
    for (int J = 0; J < T; ++J)
      if (J <= c || mat) buf[(mat * 16 + sk) * NBP + 16 * J + sj] = st[J];
    __syncthreads();
    if (c + 1 < T) fetch(c + 1, vb[(c + 1) & 1], vq[(c + 1) & 1]);
#pragma unroll
    for (int m = 0; m < 4; ++m) {
      const double2 xb = vb[c & 1][m], xq = vq[c & 1][m];
      const double2* sa = buf + (4 * m + lk) * NBP + 16 * odd + li;
      const double2* sb = sa + 16 * NBP;
#pragma unroll
      for (int h = 0; h < TH; ++h) {  // column tile 2 h + odd
        if (2 * h + 1 <= c || (2 * h <= c && !odd)) {  // A[i][j] = 0 for j > i
          const double2 a = sa[32 * h];
          re[h] = mfma4(xb.x, a.x, re[h]);
          im[h] = mfma4(xb.x, a.y, im[h]);
          re[h] = mfma4(-xb.y, a.y, re[h]);
          im[h] = mfma4(xb.y, a.x, im[h]);
        }
        if (2 * h + 1 < T || !odd) {
          const double2 b = sb[32 * h];
          re[h] = mfma4(xq.x, b.x, re[h]);
          im[h] = mfma4(xq.x, b.y, im[h]);
          re[h] = mfma4(-xq.y, b.y, re[h]);
          im[h] = mfma4(xq.y, b.x, im[h]);
        }
      }
    }
  }
#pragma unroll
  for (int h = 0; h < TH; ++h) {
    const int col = 16 * (2 * h + odd) + li;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int row = g0 + 4 * r + lk;
      if (row < ng && col < nb) {
        Dr[(int64_t)row * nb + col] = re[h][r];
        Di[(int64_t)row * nb + col] = im[h][r];
      }
    }
  }
}

// Partial Gram sums over the chunk's rows (one per block):
//   S = A^H A with A = W (PRE = false) or A = W pre (PRE = true).
// Waves take 16-row slabs in turn; only tile pairs I <= J are accumulated
// and the full Hermitian matrix is written.
template <int T, bool PRE>
__global__ __launch_bounds__(kQrBlock) void gram_w_kernel(
    const double* __restrict__ wr, const double* __restrict__ wi,
    const double2* __restrict__ pre, double2* __restrict__ partial, int ng,
    int nb, int rows_per_chunk, int nchunk, const int* __restrict__ skip) {
  extern __shared__ double2 sm[];
  constexpr int NBP = 16 * T;
  constexpr int NP = T * (T + 1) / 2;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int li = lane & 15, lk = lane >> 4;
  const int64_t p = blockIdx.y;
  const int chunk = blockIdx.x;
  if (skip && skip[p]) return;  // uniform over the block
  if (PRE) load_small(sm, pre + p * nb * nb, nb, NBP);
  __syncthreads();
  d4 sre[NP], sim[NP];
#pragma unroll
  for (int i = 0; i < NP; ++i) { sre[i] = d4zero(); sim[i] = d4zero(); }
  const int gb = chunk * rows_per_chunk;
  const int ge = min(ng, gb + rows_per_chunk);
  const double* Wr = wr + p * ng * nb;
  const double* Wi = wi + p * ng * nb;
  const int nm = (nb + 3) / 4;
  for (int g0 = gb + wave * 16; g0 < ge; g0 += 64) {
    double xr[T][4], xi[T][4];
    if (PRE) {
      d4 are[T], aim[T];
#pragma unroll
      for (int J = 0; J < T; ++J) { are[J] = d4zero(); aim[J] = d4zero(); }
      const int row = g0 + li;
      for (int m = 0; m < nm; ++m) {
        const int col = 4 * m + lk;
        const bool ok = row < ge && col < nb;
        const double a_r = ok ? Wr[(int64_t)row * nb + col] : 0.0;
        const double a_i = ok ? Wi[(int64_t)row * nb + col] : 0.0;
#pragma unroll
        for (int J = 0; J < T; ++J) {
          const double2 rv = sm[(4 * m + lk) * NBP + 16 * J + li];
          are[J] = mfma4(a_r, rv.x, are[J]);
          are[J] = mfma4(-a_i, rv.y, are[J]);
          aim[J] = mfma4(a_r, rv.y, aim[J]);
          aim[J] = mfma4(a_i, rv.x, aim[J]);
        }
      }
#pragma unroll
      for (int J = 0; J < T; ++J)
#pragma unroll
        for (int r = 0; r < 4; ++r) { xr[J][r] = are[J][r]; xi[J][r] = aim[J][r]; }
    } else {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = g0 + 4 * r + lk;
#pragma unroll
        for (int J = 0; J < T; ++J) {
          const int col = 16 * J + li;
          const bool ok = row < ge && col < nb;
          xr[J][r] = ok ? Wr[(int64_t)row * nb + col] : 0.0;
          xi[J][r] = ok ? Wi[(int64_t)row * nb + col] : 0.0;
        }
      }
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      int pi = 0;
#pragma unroll
      for (int I = 0; I < T; ++I)
#pragma unroll
        for (int J = I; J < T; ++J, ++pi) {
          sre[pi] = mfma4(xr[I][r], xr[J][r], sre[pi]);
          sre[pi] = mfma4(xi[I][r], xi[J][r], sre[pi]);
          sim[pi] = mfma4(xr[I][r], xi[J][r], sim[pi]);
          sim[pi] = mfma4(-xi[I][r], xr[J][r], sim[pi]);
        }
    }
  }
  // Sum the four waves' tiles in LDS (wave order 0..3), one partial per
  // block.
  double2* red = sm + (PRE ? NBP * NBP : 0);
  for (int w = 0; w < 4; ++w) {
    if (wave == w) {
      int pi = 0;
#pragma unroll
      for (int I = 0; I < T; ++I)
#pragma unroll
        for (int J = I; J < T; ++J, ++pi)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int i = 16 * I + 4 * r + lk, j = 16 * J + li;
            const double2 v = make_double2(sre[pi][r], sim[pi][r]);
            if (w == 0) {
              red[i * NBP + j] = v;
              if (I < J) red[j * NBP + i] = cconj(v);
            } else {
              red[i * NBP + j] = cadd(red[i * NBP + j], v);
              if (I < J) red[j * NBP + i] = cadd(red[j * NBP + i], cconj(v));
            }
          }
    }
    __syncthreads();
  }
  double2* out = partial + (p * nchunk + chunk) * nb * nb;
  for (int e = threadIdx.x; e < nb * nb; e += kQrBlock) {
    const int i = e / nb, j = e - i * nb;
    out[e] = red[i * NBP + j];
  }
}

int launch_gram_gmajor(const double* wr, const double* wi, const double2* pre,
                       double2* partial, int64_t P, int ng, int nb,
                       const GramSplit& sp, hipStream_t s, const int* skip,
                       double2* q1) {
  const int T = (nb + 15) / 16;
  if (nb > kNarrowBands) {
    if (!pre) return launch_gram_wide(wr, wi, nullptr, nullptr, partial, P, ng,
                                      nb, sp, s, skip);
    if (!q1) {
      set_error("the wide Gram pass with a preconditioner needs q1");
      return JRX_ERR_INVALID;
    }
    const int rc = launch_apply_fwd(wr, wi, pre, q1, P, ng, nb, s, skip);
    if (rc) return rc;
    return launch_gram_wide(nullptr, nullptr, q1, q1, partial, P, ng, nb, sp,
                            s, skip);
  }
  size_t shm = (pre ? 2 : 1) * (size_t)(16 * T) * (16 * T) * sizeof(double2);
  dim3 grid(sp.nchunk, (unsigned)P), block(kQrBlock);
#define JRX_GRAM_W(TT)                                                        \
  if (pre)                                                                    \
    hipLaunchKernelGGL((gram_w_kernel<TT, true>), grid, block, shm, s, wr, wi, \
                       pre, partial, ng, nb, sp.rows_per_chunk, sp.nchunk,    \
                       skip);                                                 \
  else                                                                        \
    hipLaunchKernelGGL((gram_w_kernel<TT, false>), grid, block, shm, s, wr,   \
                       wi, pre, partial, ng, nb, sp.rows_per_chunk,           \
                       sp.nchunk, skip);
  switch (T) {
    case 1: JRX_GRAM_W(1) break;
    case 2: JRX_GRAM_W(2) break;
    case 3: JRX_GRAM_W(3) break;
    case 4: JRX_GRAM_W(4) break;
    default:
      set_error("nb above 64 is not supported by this build");
      return JRX_ERR_UNSUPPORTED;
  }
#undef JRX_GRAM_W
  JRX_LAUNCH_CHECK();
  return JRX_OK;
}

// Partial sums of G = Q^H Qbar over the chunk (band-major inputs), one per
// block.  A wave takes 16-row slabs in turn, 4 rows at a time (row
// g0 + 4 r + lk, bands 16 I + li).
template <int T>
__global__ __launch_bounds__(kQrBlock) void gram_q_kernel(
    const double2* __restrict__ q, const double2* __restrict__ qb,
    double2* __restrict__ partial, int ng, int nb, int rows_per_chunk,
    int nchunk) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int li = lane & 15, lk = lane >> 4;
  const int64_t p = blockIdx.y;
  const int chunk = blockIdx.x;
  d4 gre[T][T], gim[T][T];
#pragma unroll
  for (int I = 0; I < T; ++I)
#pragma unroll
    for (int J = 0; J < T; ++J) { gre[I][J] = d4zero(); gim[I][J] = d4zero(); }
  const int gb = chunk * rows_per_chunk;
  const int ge = min(ng, gb + rows_per_chunk);
  const double2* Q = q + p * nb * ng;
  const double2* B = qb + p * nb * ng;
  auto accum = [&](const double2* a, const double2* b) {
#pragma unroll
    for (int I = 0; I < T; ++I)
#pragma unroll
      for (int J = 0; J < T; ++J) {
        gre[I][J] = mfma4(a[I].x, b[J].x, gre[I][J]);
        gre[I][J] = mfma4(a[I].y, b[J].y, gre[I][J]);
        gim[I][J] = mfma4(a[I].x, b[J].y, gim[I][J]);
        gim[I][J] = mfma4(-a[I].y, b[J].x, gim[I][J]);
      }
  };
  if constexpr (T <= 2) {
    // units of 4 rows; the loads of the next unit are issued before the
    // MFMAs of the current one
    const int gw = gb + wave * 16;  // first slab of this wave
    const int nunit = gw < ge ? ((ge - gw + 63) / 64) * 4 : 0;
    double2 ca[T], cb[T];
    auto load = [&](int u, double2* a, double2* b) {
      const int g = gw + 64 * (u >> 2) + 4 * (u & 3) + lk;
#pragma unroll
      for (int I = 0; I < T; ++I) {
        const int band = 16 * I + li;
        const bool ok = u < nunit && g < ge && band < nb;
        a[I] = ok ? Q[(int64_t)band * ng + g] : czero();
        b[I] = ok ? B[(int64_t)band * ng + g] : czero();
      }
    };
    load(0, ca, cb);
    for (int u = 0; u < nunit; ++u) {
      double2 na[T], nbv[T];
      load(u + 1, na, nbv);
      accum(ca, cb);
#pragma unroll
      for (int I = 0; I < T; ++I) { ca[I] = na[I]; cb[I] = nbv[I]; }
    }
  } else {
    // whole slabs (more registers per unit than a second buffer allows)
    for (int g0 = gb + wave * 16; g0 < ge; g0 += 64) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int g = g0 + 4 * r + lk;
        double2 a[T], b[T];
#pragma unroll
        for (int I = 0; I < T; ++I) {
          const int band = 16 * I + li;
          const bool ok = g < ge && band < nb;
          a[I] = ok ? Q[(int64_t)band * ng + g] : czero();
          b[I] = ok ? B[(int64_t)band * ng + g] : czero();
        }
        accum(a, b);
      }
    }
  }
  // Sum the four waves' tiles in LDS (wave order 0..3), one partial per
  // block.
  extern __shared__ double2 red[];
  constexpr int NBP = 16 * T;
  for (int w = 0; w < 4; ++w) {
    if (wave == w) {
#pragma unroll
      for (int I = 0; I < T; ++I)
#pragma unroll
        for (int J = 0; J < T; ++J)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int i = 16 * I + 4 * r + lk, j = 16 * J + li;
            const double2 v = make_double2(gre[I][J][r], gim[I][J][r]);
            red[i * NBP + j] = w == 0 ? v : cadd(red[i * NBP + j], v);
          }
    }
    __syncthreads();
  }
  double2* out = partial + (p * nchunk + chunk) * nb * nb;
  for (int e = threadIdx.x; e < nb * nb; e += kQrBlock) {
    const int i = e / nb, j = e - i * nb;
    out[e] = red[i * NBP + j];
  }
}

int launch_gram_bmajor(const double2* q, const double2* qb, double2* partial,
                       int64_t P, int ng, int nb, const GramSplit& sp,
                       hipStream_t s) {
  const int T = (nb + 15) / 16;
  if (nb > kNarrowBands)
    return launch_gram_wide(nullptr, nullptr, q, qb, partial, P, ng, nb, sp, s,
                            nullptr);
  const size_t shm = (size_t)(16 * T) * (16 * T) * sizeof(double2);
  dim3 grid(sp.nchunk, (unsigned)P), block(kQrBlock);
  switch (T) {
    case 1: hipLaunchKernelGGL((gram_q_kernel<1>), grid, block, shm, s, q, qb, partial, ng, nb, sp.rows_per_chunk, sp.nchunk); break;
    case 2: hipLaunchKernelGGL((gram_q_kernel<2>), grid, block, shm, s, q, qb, partial, ng, nb, sp.rows_per_chunk, sp.nchunk); break;
    case 3: hipLaunchKernelGGL((gram_q_kernel<3>), grid, block, shm, s, q, qb, partial, ng, nb, sp.rows_per_chunk, sp.nchunk); break;
    case 4: hipLaunchKernelGGL((gram_q_kernel<4>), grid, block, shm, s, q, qb, partial, ng, nb, sp.rows_per_chunk, sp.nchunk); break;
    default:
      set_error("nb above 64 is not supported by this build");
      return JRX_ERR_UNSUPPORTED;
  }
  JRX_LAUNCH_CHECK();
  return JRX_OK;
}

// A block sums kRedOut consecutive outputs: its kRedGroups thread groups
// take chunks c = g, g + kRedGroups, ... in order, then the group sums are
// added in group order (a fixed order for every launch).
constexpr int kRedOut = 32, kRedGroups = kQrBlock / kRedOut;

__global__ __launch_bounds__(kQrBlock) void reduce_partials_kernel(
    const double2* __restrict__ partial, double2* __restrict__ out,
    int nchunk, int nout, const int* __restrict__ skip) {
  __shared__ double2 acc[kRedGroups][kRedOut];
  const int64_t p = blockIdx.y;
  if (skip && skip[p]) return;  // uniform over the block
  const int ol = threadIdx.x % kRedOut, grp = threadIdx.x / kRedOut;
  const int o = blockIdx.x * kRedOut + ol;
  // four independent sums in flight, added in a fixed order
  double2 a = czero(), b = czero(), c2 = czero(), d = czero();
  if (o < nout) {
    const double2* src = partial + p * nchunk * nout + o;
    int c = grp;
    for (; c + 3 * kRedGroups < nchunk; c += 4 * kRedGroups) {
      a = cadd(a, src[(int64_t)c * nout]);
      b = cadd(b, src[(int64_t)(c + kRedGroups) * nout]);
      c2 = cadd(c2, src[(int64_t)(c + 2 * kRedGroups) * nout]);
      d = cadd(d, src[(int64_t)(c + 3 * kRedGroups) * nout]);
    }
    for (; c < nchunk; c += kRedGroups) a = cadd(a, src[(int64_t)c * nout]);
  }
  a = cadd(cadd(a, b), cadd(c2, d));
  acc[grp][ol] = a;
  __syncthreads();
  if (grp == 0 && o < nout) {
    for (int g = 1; g < kRedGroups; ++g) a = cadd(a, acc[g][ol]);
    out[p * nout + o] = a;
  }
}

int launch_reduce_partials(const double2* partial, double2* out, int64_t P,
                           int nchunk, int nb, hipStream_t s,
                           const int* skip) {
  const int nout = nb * nb;
  dim3 grid(ceil_div(nout, kRedOut), (unsigned)P), block(kQrBlock);
  hipLaunchKernelGGL(reduce_partials_kernel, grid, block, 0, s, partial, out,
                     nchunk, nout, skip);
  JRX_LAUNCH_CHECK();
  return JRX_OK;
}

// Rows per block of the narrow apply kernels: 256, halved (down to 64)
// while the grid would hold fewer than 2048 blocks, so that problems with
// few k-points still spread over the chip.
inline int apply_rows(int ng, int64_t P) {
  int rows = 256;
  while (rows > 64 && (int64_t)ceil_div(ng, rows) * P < 2048) rows >>= 1;
  return rows;
}

// Q[p][b][g] = sum_i W[p][g][i] rinv[p][i][b], computed as Q^T = R^T W^T so
// that each accumulator row is 16 consecutive g of one band.  rinv is upper
// triangular (as the Cholesky inverses and their products are), so up to
// 48 bands the (column group, band tile) pairs below the diagonal are
// skipped.  A wave takes 16-row slabs in turn.
template <int T>
__global__ __launch_bounds__(kQrBlock) void apply_fwd_kernel(
    const double* __restrict__ wr, const double* __restrict__ wi,
    const double2* __restrict__ rinv, double2* __restrict__ q, int ng,
    int nb, int rows) {
  extern __shared__ double2 sm[];
  constexpr int NBP = 16 * T;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int li = lane & 15, lk = lane >> 4;
  const int64_t p = blockIdx.y;
  load_small(sm, rinv + p * nb * nb, nb, NBP);
  __syncthreads();
  const double* Wr = wr + p * ng * nb;
  const double* Wi = wi + p * ng * nb;
  double2* Q = q + p * nb * ng;
  const int gb = blockIdx.x * rows;
  const int ge = min(ng, gb + rows);
  const int gw = gb + wave * 16;  // first slab of this wave
  if constexpr (T <= 3) {
    // units of 16 columns; the loads of the next unit are issued before
    // the MFMAs of the current one
    const int nunit = gw < ge ? ((ge - gw + 63) / 64) * T : 0;
    double ar[4], ai[4];
    auto load = [&](int u, double* xr, double* xi) {
      const int row = gw + 64 * (u / T) + li, mg = u % T;
#pragma unroll
      for (int mm = 0; mm < 4; ++mm) {
        const int col = 16 * mg + 4 * mm + lk;
        const bool ok = u < nunit && row < ge && col < nb;
        xr[mm] = ok ? Wr[(int64_t)row * nb + col] : 0.0;
        xi[mm] = ok ? Wi[(int64_t)row * nb + col] : 0.0;
      }
    };
    load(0, ar, ai);
    d4 qre[T], qim[T];
#pragma unroll
    for (int J = 0; J < T; ++J) { qre[J] = d4zero(); qim[J] = d4zero(); }
    for (int u = 0; u < nunit; ++u) {
      double nr[4], ni[4];
      load(u + 1, nr, ni);
      const int mg = u % T;
#pragma unroll
      for (int mm = 0; mm < 4; ++mm) {
        const int k = 16 * mg + 4 * mm + lk;
#pragma unroll
        for (int J = 0; J < T; ++J) {
          if (mg > J) continue;  // rinv[i][b] = 0 for i > b
          const double2 rv = sm[k * NBP + 16 * J + li];
          qre[J] = mfma4(rv.x, ar[mm], qre[J]);
          qre[J] = mfma4(-rv.y, ai[mm], qre[J]);
          qim[J] = mfma4(rv.x, ai[mm], qim[J]);
          qim[J] = mfma4(rv.y, ar[mm], qim[J]);
        }
      }
      if (mg == T - 1) {
        const int g = gw + 64 * (u / T) + li;
#pragma unroll
        for (int J = 0; J < T; ++J) {
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int b = 16 * J + 4 * r + lk;
            if (b < nb && g < ge)
              Q[(int64_t)b * ng + g] = make_double2(qre[J][r], qim[J][r]);
          }
          qre[J] = d4zero();
          qim[J] = d4zero();
        }
      }
#pragma unroll
      for (int mm = 0; mm < 4; ++mm) { ar[mm] = nr[mm]; ai[mm] = ni[mm]; }
    }
  } else {
    // one column group of 4 at a time (more registers per unit than a
    // second buffer allows)
    const int nm = (nb + 3) / 4;
    for (int g0 = gw; g0 < ge; g0 += 64) {
      d4 qre[T], qim[T];
#pragma unroll
      for (int J = 0; J < T; ++J) { qre[J] = d4zero(); qim[J] = d4zero(); }
      const int row = g0 + li;
      for (int m = 0; m < nm; ++m) {
        const int col = 4 * m + lk;
        const bool ok = row < ge && col < nb;
        const double a_r = ok ? Wr[(int64_t)row * nb + col] : 0.0;
        const double a_i = ok ? Wi[(int64_t)row * nb + col] : 0.0;
#pragma unroll
        for (int J = 0; J < T; ++J) {
          const double2 rv = sm[(4 * m + lk) * NBP + 16 * J + li];
          qre[J] = mfma4(rv.x, a_r, qre[J]);
          qre[J] = mfma4(-rv.y, a_i, qre[J]);
          qim[J] = mfma4(rv.x, a_i, qim[J]);
          qim[J] = mfma4(rv.y, a_r, qim[J]);
        }
      }
      const int g = g0 + li;
#pragma unroll
      for (int J = 0; J < T; ++J)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int b = 16 * J + 4 * r + lk;
          if (b < nb && g < ge)
            Q[(int64_t)b * ng + g] = make_double2(qre[J][r], qim[J][r]);
        }
    }
  }
}

int launch_apply_fwd(const double* wr, const double* wi, const double2* rinv,
                     double2* q, int64_t P, int ng, int nb, hipStream_t s,
                     const int* skip) {
  const int T = (nb + 15) / 16;
  if (nb > kNarrowBands) {
    const size_t shm = 2 * (size_t)16 * 16 * T * sizeof(double2);
    dim3 grid(ceil_div(ng, kWideRows), (unsigned)P), block(kQrBlock);
    switch (T) {
      case 5: hipLaunchKernelGGL((apply_fwd_wide_kernel<5>), grid, block, shm, s, wr, wi, rinv, q, ng, nb, skip); break;
      case 6: hipLaunchKernelGGL((apply_fwd_wide_kernel<6>), grid, block, shm, s, wr, wi, rinv, q, ng, nb, skip); break;
      case 7: hipLaunchKernelGGL((apply_fwd_wide_kernel<7>), grid, block, shm, s, wr, wi, rinv, q, ng, nb, skip); break;
      case 8: hipLaunchKernelGGL((apply_fwd_wide_kernel<8>), grid, block, shm, s, wr, wi, rinv, q, ng, nb, skip); break;
      default:
        set_error("nb above 128 is not supported by this build");
        return JRX_ERR_UNSUPPORTED;
    }
    JRX_LAUNCH_CHECK();
    return JRX_OK;
  }
  if (skip) {
    set_error("launch_apply_fwd: skip is for the wide kernels");
    return JRX_ERR_INVALID;
  }
  size_t shm = (size_t)(16 * T) * (16 * T) * sizeof(double2);
  const int rows = apply_rows(ng, P);
  dim3 grid(ceil_div(ng, rows), (unsigned)P), block(kQrBlock);
  switch (T) {
    case 1: hipLaunchKernelGGL((apply_fwd_kernel<1>), grid, block, shm, s, wr, wi, rinv, q, ng, nb, rows); break;
    case 2: hipLaunchKernelGGL((apply_fwd_kernel<2>), grid, block, shm, s, wr, wi, rinv, q, ng, nb, rows); break;
    case 3: hipLaunchKernelGGL((apply_fwd_kernel<3>), grid, block, shm, s, wr, wi, rinv, q, ng, nb, rows); break;
    case 4: hipLaunchKernelGGL((apply_fwd_kernel<4>), grid, block, shm, s, wr, wi, rinv, q, ng, nb, rows); break;
    default:
      set_error("nb above 64 is not supported by this build");
      return JRX_ERR_UNSUPPORTED;
  }
  JRX_LAUNCH_CHECK();
  return JRX_OK;
}

// Wbar[p][g][j] = sum_i Qbar[p][i][g] A[i][j] + Q[p][i][g] Bm[i][j], planar
// g-major outputs.  A = R^{-H} is lower triangular, so its (band group,
// column tile) pairs above the diagonal are skipped.  A wave takes 16-row
// slabs in turn and reads each slab in T units of 16 bands; the loads of the
// next unit are issued before the MFMAs of the current one.
template <int T>
__global__ __launch_bounds__(kQrBlock) void apply_bwd_kernel(
    const double2* __restrict__ qbar, const double2* __restrict__ q,
    const double2* __restrict__ A, const double2* __restrict__ Bm,
    double* __restrict__ dwr, double* __restrict__ dwi, int ng, int nb,
    int rows) {
  extern __shared__ double2 sm[];
  constexpr int NBP = 16 * T;
  double2* sa = sm;
  double2* sb = sm + NBP * NBP;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int li = lane & 15, lk = lane >> 4;
  const int64_t p = blockIdx.y;
  load_small(sa, A + p * nb * nb, nb, NBP);
  load_small(sb, Bm + p * nb * nb, nb, NBP);
  __syncthreads();
  const double2* Qb = qbar + p * nb * ng;
  const double2* Q = q + p * nb * ng;
  double* Dr = dwr + p * ng * nb;
  double* Di = dwi + p * ng * nb;
  const int gb = blockIdx.x * rows;
  const int ge = min(ng, gb + rows);
  const int gw = gb + wave * 16;  // first slab of this wave
  const int nunit = gw < ge ? ((ge - gw + 63) / 64) * T : 0;
  double2 cb[4], cq[4];
  auto load = [&](int u, double2* vb, double2* vq) {
    const int g = gw + 64 * (u / T) + li, mg = u % T;
#pragma unroll
    for (int mm = 0; mm < 4; ++mm) {
      const int band = 16 * mg + 4 * mm + lk;
      const bool ok = u < nunit && g < ge && band < nb;
      vb[mm] = ok ? Qb[(int64_t)band * ng + g] : czero();
      vq[mm] = ok ? Q[(int64_t)band * ng + g] : czero();
    }
  };
  load(0, cb, cq);
  d4 re[T], im[T];
#pragma unroll
  for (int J = 0; J < T; ++J) { re[J] = d4zero(); im[J] = d4zero(); }
  for (int u = 0; u < nunit; ++u) {
    double2 nbv[4], nqv[4];
    load(u + 1, nbv, nqv);
    const int mg = u % T;
#pragma unroll
    for (int mm = 0; mm < 4; ++mm) {
      const int k = 16 * mg + 4 * mm + lk;
      const double2 vb = cb[mm], vq = cq[mm];
#pragma unroll
      for (int J = 0; J < T; ++J) {
        if (J <= mg) {  // A[i][j] = 0 for j > i
          const double2 a = sa[k * NBP + 16 * J + li];
          re[J] = mfma4(vb.x, a.x, re[J]);
          re[J] = mfma4(-vb.y, a.y, re[J]);
          im[J] = mfma4(vb.x, a.y, im[J]);
          im[J] = mfma4(vb.y, a.x, im[J]);
        }
        const double2 b = sb[k * NBP + 16 * J + li];
        re[J] = mfma4(vq.x, b.x, re[J]);
        re[J] = mfma4(-vq.y, b.y, re[J]);
        im[J] = mfma4(vq.x, b.y, im[J]);
        im[J] = mfma4(vq.y, b.x, im[J]);
      }
    }
    if (mg == T - 1) {
      const int g0 = gw + 64 * (u / T);
#pragma unroll
      for (int J = 0; J < T; ++J) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int row = g0 + 4 * r + lk, col = 16 * J + li;
          if (row < ge && col < nb) {
            Dr[(int64_t)row * nb + col] = re[J][r];
            Di[(int64_t)row * nb + col] = im[J][r];
          }
        }
        re[J] = d4zero();
        im[J] = d4zero();
      }
    }
#pragma unroll
    for (int mm = 0; mm < 4; ++mm) { cb[mm] = nbv[mm]; cq[mm] = nqv[mm]; }
  }
}

size_t qr_lds_bytes(int nb) {
  const size_t nbp = 16 * (size_t)((nb + 15) / 16), z = sizeof(double2);
  const size_t chol = chol_inv_lds_bytes(nb);
  if (nb <= kNarrowBands)  // Gram (pre + sums), apply_bwd
    return std::max(2 * nbp * nbp * z, chol);
  const size_t gram = 2 * 2 * (size_t)wide_slab<false>() * (nbp + 1) * z;
  const size_t fwd = 2 * (size_t)16 * nbp * z;
  const size_t bwd = 2 * fwd;
  return std::max(std::max(gram, fwd), std::max(bwd, chol));
}

int launch_apply_bwd(const double2* qbar, const double2* q, const double2* A,
                     const double2* Bm, double* dwr, double* dwi, int64_t P,
                     int ng, int nb, hipStream_t s) {
  const int T = (nb + 15) / 16;
  if (nb > kNarrowBands) {
    const size_t shm = 2 * 2 * (size_t)16 * 16 * T * sizeof(double2);
    dim3 grid(ceil_div(ng, kWideRows), (unsigned)P), block(kWideBwdBlock);
    switch (T) {
      case 5: hipLaunchKernelGGL((apply_bwd_wide_kernel<5>), grid, block, shm, s, qbar, q, A, Bm, dwr, dwi, ng, nb); break;
      case 6: hipLaunchKernelGGL((apply_bwd_wide_kernel<6>), grid, block, shm, s, qbar, q, A, Bm, dwr, dwi, ng, nb); break;
      case 7: hipLaunchKernelGGL((apply_bwd_wide_kernel<7>), grid, block, shm, s, qbar, q, A, Bm, dwr, dwi, ng, nb); break;
      case 8: hipLaunchKernelGGL((apply_bwd_wide_kernel<8>), grid, block, shm, s, qbar, q, A, Bm, dwr, dwi, ng, nb); break;
      default:
        set_error("nb above 128 is not supported by this build");
        return JRX_ERR_UNSUPPORTED;
    }
    JRX_LAUNCH_CHECK();
    return JRX_OK;
  }
  size_t shm = 2 * (size_t)(16 * T) * (16 * T) * sizeof(double2);
  const int rows = apply_rows(ng, P);
  dim3 grid(ceil_div(ng, rows), (unsigned)P), block(kQrBlock);
  switch (T) {
    case 1: hipLaunchKernelGGL((apply_bwd_kernel<1>), grid, block, shm, s, qbar, q, A, Bm, dwr, dwi, ng, nb, rows); break;
    case 2: hipLaunchKernelGGL((apply_bwd_kernel<2>), grid, block, shm, s, qbar, q, A, Bm, dwr, dwi, ng, nb, rows); break;
    case 3: hipLaunchKernelGGL((apply_bwd_kernel<3>), grid, block, shm, s, qbar, q, A, Bm, dwr, dwi, ng, nb, rows); break;
    case 4: hipLaunchKernelGGL((apply_bwd_kernel<4>), grid, block, shm, s, qbar, q, A, Bm, dwr, dwi, ng, nb, rows); break;
    default:
      set_error("nb above 64 is not supported by this build");
      return JRX_ERR_UNSUPPORTED;
  }
  JRX_LAUNCH_CHECK();
  return JRX_OK;
}

}  // namespace jrx
