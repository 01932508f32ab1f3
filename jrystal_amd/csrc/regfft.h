// Register transforms of one line of N points on L lanes of a wavefront.
//
// N = V * L.  Lane j of a line holds x[j + L m] in v[m] (m < V).  to_ab runs a
// V-point DFT over m in registers, multiplies by w_N^{ja}, transposes blocks
// of L registers over the L lanes, and runs W = ceil(V / L) L-point DFTs: lane
// i ends with X[a + V b] in v[u L + b], a = i + L u (u < W; where a >= V the
// lane holds nothing of use).  The forward transform is its mirror image, so a
// product with v(r) between the two needs no further exchange.  64 / L lines
// share a wave and never leave it: no block barrier inside.
//
// The transposition is what such a transform costs beside its arithmetic.
// Measured on gfx950 (cycles of a CU per wave access, conflict-free): a
// 16-byte LDS write 13.6, a 16-byte read 5.3, a pair of 8-byte reads 8.9; so
// eight values exchanged through LDS take 150 to 180, about what their
// arithmetic takes on the four SIMDs.  With L = 4, the lanes of a line 16
// apart, it is two v_permlane*_swap per register pair instead (32 VALU
// instructions for eight values, no LDS); with L = 8, lanes 8 apart, a third
// stage by row rotation.  The other L exchange through LDS.
//
// The small DFTs are written with compile-time constants: powers of two by
// radix 2 / 4 / 8, odd primes by the symmetric sums u_k +- u_{p-k} (half the
// products of the direct sum), coprime products by index maps without
// twiddles (Good 1958), 9 and 16 by one Cooley-Tukey step.  Inputs that are
// literal zeros (the part of the box outside the mask's window) and outputs
// that nobody reads fold away; the files of the row-path kernels
// (rowfft_*.hip) are built with -fno-signed-zeros, without which x + 0 stays
// an addition.  (The full-box kernels have no zero inputs.)
#pragma once
#include "fft_core.h"

namespace jrx {

template <int R, bool INV>
struct RDft;  // in place on u[R], u[k] <- sum_n u[n] exp(-+ 2 pi i n k / R)

template <bool INV>
struct RDft<1, INV> {
  __device__ __forceinline__ static void run(double2*) {}
};
template <bool INV>
struct RDft<2, INV> {
  __device__ __forceinline__ static void run(double2* u) {
    Dft<2, INV>::run(u, nullptr, 0);
  }
};
template <bool INV>
struct RDft<4, INV> {
  __device__ __forceinline__ static void run(double2* u) {
    Dft<4, INV>::run(u, nullptr, 0);
  }
};
template <bool INV>
struct RDft<8, INV> {
  __device__ __forceinline__ static void run(double2* u) {
    Dft<8, INV>::run(u, nullptr, 0);
  }
};

// cos and sin of 2 pi k / p, k = 1 .. (p - 1) / 2.
template <int P>
struct Roots;
template <>
struct Roots<3> {
  static constexpr double c[1] = {-0.5};
  static constexpr double s[1] = {0.8660254037844386467637};
};
template <>
struct Roots<5> {
  static constexpr double c[2] = {0.3090169943749474241023,
                                  -0.8090169943749474241023};
  static constexpr double s[2] = {0.9510565162951535721164,
                                  0.5877852522924731291687};
};
template <>
struct Roots<7> {
  static constexpr double c[3] = {0.6234898018587335305251,
                                  -0.2225209339563144042889,
                                  -0.9009688679024191262361};
  static constexpr double s[3] = {0.7818314824680298087084,
                                  0.9749279121818236070181,
                                  0.4338837391175581204758};
};

template <int P, bool INV>
struct RDftOdd {
  __device__ __forceinline__ static void run(double2* u) {
    constexpr int H = (P - 1) / 2;
    double2 t[H], d[H];
#pragma unroll
    for (int k = 0; k < H; ++k) {
      t[k] = cadd(u[k + 1], u[P - 1 - k]);
      d[k] = csub(u[k + 1], u[P - 1 - k]);
    }
    double2 y0 = u[0];
#pragma unroll
    for (int k = 0; k < H; ++k) y0 = cadd(y0, t[k]);
#pragma unroll
    for (int q = 1; q <= H; ++q) {
      double2 a = u[0], b = czero();
#pragma unroll
      for (int k = 1; k <= H; ++k) {
        const int r = (q * k) % P;
        const double c = r <= H ? Roots<P>::c[r - 1] : Roots<P>::c[P - r - 1];
        const double s = r <= H ? Roots<P>::s[r - 1] : -Roots<P>::s[P - r - 1];
        a.x += c * t[k - 1].x;
        a.y += c * t[k - 1].y;
        b.x += s * d[k - 1].x;
        b.y += s * d[k - 1].y;
      }
      // y_q = a -+ i b, y_{p-q} = a +- i b
      const double2 lo = make_double2(a.x + b.y, a.y - b.x);
      const double2 hi = make_double2(a.x - b.y, a.y + b.x);
      u[q] = INV ? hi : lo;
      u[P - q] = INV ? lo : hi;
    }
    u[0] = y0;
  }
};
template <bool INV>
struct RDft<3, INV> : RDftOdd<3, INV> {};
template <bool INV>
struct RDft<5, INV> : RDftOdd<5, INV> {};
template <bool INV>
struct RDft<7, INV> : RDftOdd<7, INV> {};

// A * B points, A and B coprime: n = (n1 B + n2 A) mod N turns the DFT into
// an A x B one without twiddles, k = k1 mod A = k2 mod B.
template <int A, int B, bool INV>
struct RDftPfa {
  static constexpr int N = A * B;
  static constexpr int crt(int k1, int k2) {
    int k = k1;
    while (k % B != k2) k += A;
    return k;
  }
  __device__ __forceinline__ static void run(double2* u) {
    double2 t[A][B];
#pragma unroll
    for (int n1 = 0; n1 < A; ++n1) {
#pragma unroll
      for (int n2 = 0; n2 < B; ++n2) t[n1][n2] = u[(n1 * B + n2 * A) % N];
      RDft<B, INV>::run(t[n1]);
    }
#pragma unroll
    for (int k2 = 0; k2 < B; ++k2) {
      double2 c[A];
#pragma unroll
      for (int n1 = 0; n1 < A; ++n1) c[n1] = t[n1][k2];
      RDft<A, INV>::run(c);
#pragma unroll
      for (int k1 = 0; k1 < A; ++k1) u[crt(k1, k2)] = c[k1];
    }
  }
};
template <bool INV>
struct RDft<6, INV> : RDftPfa<2, 3, INV> {};
template <bool INV>
struct RDft<10, INV> : RDftPfa<2, 5, INV> {};
template <bool INV>
struct RDft<12, INV> : RDftPfa<4, 3, INV> {};
template <bool INV>
struct RDft<14, INV> : RDftPfa<2, 7, INV> {};
template <bool INV>
struct RDft<15, INV> : RDftPfa<3, 5, INV> {};

// Multiply by w (forward) or conj(w) (inverse), w = (c, -s).
template <bool INV>
__device__ __forceinline__ double2 rot(double2 a, double c, double s) {
  return INV ? make_double2(a.x * c - a.y * s, a.y * c + a.x * s)
             : make_double2(a.x * c + a.y * s, a.y * c - a.x * s);
}

// R * R points, one Cooley-Tukey step: n = R n1 + n2, k = k1 + R k2.
template <bool INV>
struct RDft<9, INV> {
  __device__ __forceinline__ static void run(double2* u) {
    constexpr double c1 = 0.7660444431189780352024, s1 = 0.6427876096865393263227;
    constexpr double c2 = 0.1736481776669303488517, s2 = 0.9848077530122080593667;
    constexpr double c4 = -0.9396926207859083840541, s4 = 0.3420201433256687330441;
    double2 t[3][3];
#pragma unroll
    for (int n2 = 0; n2 < 3; ++n2) {
#pragma unroll
      for (int n1 = 0; n1 < 3; ++n1) t[n2][n1] = u[3 * n1 + n2];
      RDft<3, INV>::run(t[n2]);
    }
    t[1][1] = rot<INV>(t[1][1], c1, s1);
    t[1][2] = rot<INV>(t[1][2], c2, s2);
    t[2][1] = rot<INV>(t[2][1], c2, s2);
    t[2][2] = rot<INV>(t[2][2], c4, s4);
#pragma unroll
    for (int k1 = 0; k1 < 3; ++k1) {
      double2 c[3] = {t[0][k1], t[1][k1], t[2][k1]};
      RDft<3, INV>::run(c);
#pragma unroll
      for (int k2 = 0; k2 < 3; ++k2) u[k1 + 3 * k2] = c[k2];
    }
  }
};
template <bool INV>
struct RDft<16, INV> {
  __device__ __forceinline__ static void run(double2* u) {
    constexpr double c1 = 0.9238795325112867561282, s1 = 0.3826834323650897717285;
    constexpr double h = 0.7071067811865475244008;
    double2 t[4][4];
#pragma unroll
    for (int n2 = 0; n2 < 4; ++n2) {
#pragma unroll
      for (int n1 = 0; n1 < 4; ++n1) t[n2][n1] = u[4 * n1 + n2];
      RDft<4, INV>::run(t[n2]);
    }
    t[1][1] = rot<INV>(t[1][1], c1, s1);
    t[1][2] = rot<INV>(t[1][2], h, h);
    t[1][3] = rot<INV>(t[1][3], s1, c1);
    t[2][1] = rot<INV>(t[2][1], h, h);
    t[2][2] = mul_mi<INV>(t[2][2]);
    t[2][3] = rot<INV>(t[2][3], -h, h);
    t[3][1] = rot<INV>(t[3][1], s1, c1);
    t[3][2] = rot<INV>(t[3][2], -h, h);
    t[3][3] = rot<INV>(t[3][3], -c1, -s1);
#pragma unroll
    for (int k1 = 0; k1 < 4; ++k1) {
      double2 c[4] = {t[0][k1], t[1][k1], t[2][k1], t[3][k1]};
      RDft<4, INV>::run(c);
#pragma unroll
      for (int k2 = 0; k2 < 4; ++k2) u[k1 + 4 * k2] = c[k2];
    }
  }
};


// Split of a line length: V values per lane, L lanes.  L = 4 or 8 (exchange
// in registers) where that divides N without many idle registers in the
// second stage or a V that leaves fewer than two waves per SIMD; else an L
// that divides V where a split has one, or wastes little of the second
// stage.  XS, A, B: exchange slots through LDS, value (a, j) of a line at
// a A + j B of the line's XS doubles, the layout with the fewest bank
// conflicts of the transform's writes and reads (16 lanes per cycle on 32
// banks, counted over all A, B and XS up to 1.35 N + 8; at 75 points 45 extra
// cycles for 120, against 90 with a L + j).
template <int N>
struct LineSplit;
#define JRX_LINE_SPLIT(NN, VV, LL, XX, AA, BB)                           \
  template <>                                                            \
  struct LineSplit<NN> {                                                 \
    static constexpr int V = VV, L = LL, XS = XX, A = AA, B = BB;        \
  };
JRX_LINE_SPLIT(32, 8, 4, 0, 0, 0)
JRX_LINE_SPLIT(35, 5, 7, 45, 2, 5)
JRX_LINE_SPLIT(36, 6, 6, 53, 2, 7)
JRX_LINE_SPLIT(40, 10, 4, 0, 0, 0)
JRX_LINE_SPLIT(42, 14, 3, 61, 1, 17)
JRX_LINE_SPLIT(45, 9, 5, 57, 1, 12)
JRX_LINE_SPLIT(48, 12, 4, 0, 0, 0)
JRX_LINE_SPLIT(49, 7, 7, 73, 1, 10)
JRX_LINE_SPLIT(50, 10, 5, 61, 1, 12)
JRX_LINE_SPLIT(54, 9, 6, 69, 7, 2)
JRX_LINE_SPLIT(56, 7, 8, 0, 0, 0)
JRX_LINE_SPLIT(60, 15, 4, 0, 0, 0)
JRX_LINE_SPLIT(63, 9, 7, 73, 1, 10)
JRX_LINE_SPLIT(64, 8, 8, 0, 0, 0)
JRX_LINE_SPLIT(70, 10, 7, 101, 2, 13)
JRX_LINE_SPLIT(72, 12, 6, 83, 1, 14)
JRX_LINE_SPLIT(75, 15, 5, 87, 5, 4)
JRX_LINE_SPLIT(80, 10, 8, 0, 0, 0)
JRX_LINE_SPLIT(128, 16, 8, 0, 0, 0)
// (z axes only: the row passes)
JRX_LINE_SPLIT(81, 9, 9, 87, 1, 9)
JRX_LINE_SPLIT(84, 12, 7, 101, 2, 13)
JRX_LINE_SPLIT(90, 15, 6, 117, 7, 2)
JRX_LINE_SPLIT(96, 12, 8, 0, 0, 0)
JRX_LINE_SPLIT(98, 14, 7, 121, 1, 17)
JRX_LINE_SPLIT(100, 10, 10, 103, 1, 10)
JRX_LINE_SPLIT(105, 15, 7, 121, 1, 17)
JRX_LINE_SPLIT(108, 12, 9, 151, 1, 17)
JRX_LINE_SPLIT(112, 14, 8, 0, 0, 0)
JRX_LINE_SPLIT(120, 15, 8, 0, 0, 0)
JRX_LINE_SPLIT(126, 14, 9, 151, 1, 17)
#undef JRX_LINE_SPLIT

// Lane-bit swaps of two registers: after it, a lane with the bit set holds
// in x what its partner (bit clear) had in y, and the other way round.
// BIT 5 and 4: the halves of the wave, the rows of 16 of each half; BIT 3:
// the halves of each row (rotation by 8, written under a bank mask).
template <int BIT>
__device__ __forceinline__ void lane_swap(unsigned& x, unsigned& y) {
  if constexpr (BIT == 5) {
    const auto r = __builtin_amdgcn_permlane32_swap(x, y, false, false);
    x = r[0];
    y = r[1];
  } else if constexpr (BIT == 4) {
    const auto r = __builtin_amdgcn_permlane16_swap(x, y, false, false);
    x = r[0];
    y = r[1];
  } else {
    constexpr int kRor8 = 0x128;
    const unsigned t = x;
    x = __builtin_amdgcn_update_dpp(x, y, kRor8, 0xf, 0xc, false);
    y = __builtin_amdgcn_update_dpp(y, t, kRor8, 0xf, 0x3, false);
  }
}
template <int BIT>
__device__ __forceinline__ void lane_swap(double2& a, double2& b) {
  auto one = [](double& p, double& q) {
    unsigned pl = (unsigned)__double2loint(p), ph = (unsigned)__double2hiint(p);
    unsigned ql = (unsigned)__double2loint(q), qh = (unsigned)__double2hiint(q);
    lane_swap<BIT>(pl, ql);
    lane_swap<BIT>(ph, qh);
    p = __hiloint2double((int)ph, (int)pl);
    q = __hiloint2double((int)qh, (int)ql);
  };
  one(a.x, b.x);
  one(a.y, b.y);
}

template <int N>
struct RegLine {
  static constexpr int V = LineSplit<N>::V, L = LineSplit<N>::L;
  static constexpr int W = (V + L - 1) / L;
  static constexpr int VP = W * L;    // registers of a line's lane
  static constexpr int LPW = 64 / L;  // lines of one wave
  // the exchange stays in registers, else it takes XS doubles of LDS a line
  static constexpr bool kReg = L == 4 || L == 8;
  static constexpr int XS = kReg ? 0 : LineSplit<N>::XS;
  static constexpr int A = LineSplit<N>::A, B = LineSplit<N>::B;
  static_assert(kReg || (V - 1) * A + (L - 1) * B < XS, "exchange slots");
  static_assert(V * L == N, "line split");

  // Lane of a wave -> line (fastest) and lane of the line.
  __device__ __forceinline__ static int line_of(int lane) {
    return lane % LPW;
  }
  __device__ __forceinline__ static int j_of(int lane) { return lane / LPW; }
  static constexpr int kLanes = LPW * L;  // lanes in use

  // Lane twiddles w_N^{ja} (forward sign); j a < N.
  struct Tw {
    double2 w[V];
    __device__ __forceinline__ void init(const double2* __restrict__ tab,
                                         int j) {
#pragma unroll
      for (int a = 1; a < V; ++a) w[a] = tab[j * a];
    }
  };

  // a of register block u on lane j (V - 1 past the end).
  __device__ __forceinline__ static int acol(int j, int u) {
    const int a = j + L * u;
    return (V % L == 0 || u < W - 1) ? a : (a < V ? a : V - 1);
  }
  __device__ __forceinline__ static bool alive(int j, int u) {
    return (V % L == 0 || u < W - 1) ? true : j + L * u < V;
  }

  // Transposes every block of L registers over the L lanes of the line.
  __device__ __forceinline__ static void transpose_regs(double2 (&v)[VP]) {
#pragma unroll
    for (int u = 0; u < W; ++u) {
      double2* r = v + u * L;
      if constexpr (L == 4) {  // j bits: lane bits 4, 5
        lane_swap<5>(r[0], r[2]);
        lane_swap<5>(r[1], r[3]);
        lane_swap<4>(r[0], r[1]);
        lane_swap<4>(r[2], r[3]);
      } else if constexpr (L == 8) {  // j bits: lane bits 3, 4, 5
#pragma unroll
        for (int b = 0; b < 4; ++b) lane_swap<5>(r[b], r[b + 4]);
#pragma unroll
        for (int b = 0; b < 8; ++b)
          if (!(b & 2)) lane_swap<4>(r[b], r[b + 2]);
#pragma unroll
        for (int b = 0; b < 8; b += 2) lane_swap<3>(r[b], r[b + 1]);
      }
    }
  }

  // v <- the line transformed (natural order in, X[a + V b] in v[u L + b]
  // out); x: the line's exchange slots (unused in registers).
  template <bool INV>
  __device__ __forceinline__ static void to_ab(double2 (&v)[VP], double* x,
                                               int j, const Tw& tw) {
    RDft<V, INV>::run(v);
#pragma unroll
    for (int a = 1; a < V; ++a)
      v[a] = INV ? cmulc(tw.w[a], v[a]) : cmul(tw.w[a], v[a]);
    if constexpr (kReg) {
#pragma unroll
      for (int a = V; a < VP; ++a) v[a] = czero();
      transpose_regs(v);
    } else {
      double t[V];
      wave_sync();
#pragma unroll
      for (int a = 0; a < V; ++a) {
        x[a * A + j * B] = v[a].x;
        t[a] = v[a].y;
      }
      wave_sync();
#pragma unroll
      for (int u = 0; u < W; ++u)
#pragma unroll
        for (int b = 0; b < L; ++b) v[u * L + b].x = x[acol(j, u) * A + b * B];
      wave_sync();
#pragma unroll
      for (int a = 0; a < V; ++a) x[a * A + j * B] = t[a];
      wave_sync();
#pragma unroll
      for (int u = 0; u < W; ++u)
#pragma unroll
        for (int b = 0; b < L; ++b) v[u * L + b].y = x[acol(j, u) * A + b * B];
      wave_sync();
    }
#pragma unroll
    for (int u = 0; u < W; ++u) RDft<L, INV>::run(v + u * L);
  }

  // The mirror image: X[a + V b] in v[u L + b] in, natural order out
  // (v[0 .. V-1]).
  template <bool INV>
  __device__ __forceinline__ static void from_ab(double2 (&v)[VP], double* x,
                                                 int j, const Tw& tw) {
#pragma unroll
    for (int u = 0; u < W; ++u) RDft<L, INV>::run(v + u * L);
    if constexpr (kReg) {
      transpose_regs(v);
    } else {
      double t[VP];
      wave_sync();
#pragma unroll
      for (int u = 0; u < W; ++u)
#pragma unroll
        for (int b = 0; b < L; ++b) {
          if (alive(j, u)) x[(j + L * u) * A + b * B] = v[u * L + b].x;
          t[u * L + b] = v[u * L + b].y;
        }
      wave_sync();
#pragma unroll
      for (int a = 0; a < V; ++a) v[a].x = x[a * A + j * B];
      wave_sync();
#pragma unroll
      for (int u = 0; u < W; ++u)
#pragma unroll
        for (int b = 0; b < L; ++b)
          if (alive(j, u)) x[(j + L * u) * A + b * B] = t[u * L + b];
      wave_sync();
#pragma unroll
      for (int a = 0; a < V; ++a) v[a].y = x[a * A + j * B];
      wave_sync();
    }
#pragma unroll
    for (int a = 1; a < V; ++a)
      v[a] = INV ? cmulc(tw.w[a], v[a]) : cmul(tw.w[a], v[a]);
    RDft<V, INV>::run(v);
  }
  __device__ __forceinline__ static void inverse(double2 (&v)[VP], double* x,
                                                 int j, const Tw& tw) {
    to_ab<true>(v, x, j, tw);
  }
  __device__ __forceinline__ static void forward(double2 (&v)[VP], double* x,
                                                 int j, const Tw& tw) {
    from_ab<false>(v, x, j, tw);
  }
};

// Lane of a wave -> (line of the block, lane of the line).
template <int N>
struct LaneMap {
  int j, l, wave;
  bool on;
  __device__ __forceinline__ LaneMap() {
    using F = RegLine<N>;
    const int lane = threadIdx.x & 63;
    wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    on = F::kLanes == 64 || lane < F::kLanes;
    l = F::line_of(lane);
    j = on ? F::j_of(lane) : 0;
  }
  __device__ __forceinline__ int line() const {
    return wave * RegLine<N>::LPW + l;
  }
};

}  // namespace jrx
