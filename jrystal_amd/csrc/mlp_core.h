// Small FP32 multilayer perceptron of the learned preconditioner:
//   x (kMlpIn features, normalised (x - mu) * inv_sd)
//   -> tanh(W1 x + b1) (64) -> tanh(W2 h1 + b2) (64) -> W3 h2 + b3 (2).
// Output 0 is the log of the per-coefficient preconditioner factor, output
// 1 the log amplitude of the warm-start coefficients.  Parameters live in
// one flat FP32 vector (offsets below).
#pragma once
#include <hip/hip_runtime.h>
#include "fft_core.h"

namespace jrx {

constexpr int kMlpIn = 8;  // feature slots; unused slots are zero
constexpr int kMlpHidden = 64;
constexpr int kMlpOut = 2;
constexpr int kMlpW1 = 0;  // [hidden][in]
constexpr int kMlpB1 = kMlpW1 + kMlpHidden * kMlpIn;
constexpr int kMlpW2 = kMlpB1 + kMlpHidden;  // [hidden][hidden]
constexpr int kMlpB2 = kMlpW2 + kMlpHidden * kMlpHidden;
constexpr int kMlpW3 = kMlpB2 + kMlpHidden;  // [out][hidden]
constexpr int kMlpB3 = kMlpW3 + kMlpOut * kMlpHidden;
constexpr int kMlpParams = kMlpB3 + kMlpOut;  // 4866

// Feature normalisation: norm[0..7] = mu, norm[8..15] = 1 / sd.
constexpr int kMlpNorm = 2 * kMlpIn;

__device__ inline void mlp_stage(const float* __restrict__ params,
                                 float* __restrict__ lds) {
  for (int i = threadIdx.x; i < kMlpParams; i += blockDim.x) lds[i] = params[i];
}

__device__ inline void mlp_normalise(const float* __restrict__ norm,
                                     float x[kMlpIn]) {
#pragma unroll
  for (int i = 0; i < kMlpIn; ++i) x[i] = (x[i] - norm[i]) * norm[kMlpIn + i];
}

// Forward pass of a wave on the FP32 matrix unit, 16 samples at a time.
// v_mfma_f32_16x16x4_f32: lane (li = lane % 16, lk = lane / 16) gives
// A[li][k = lk] and B[lk][li] of a step and holds D[4 lk + r][li],
// r = 0 .. 3.  A layer is z[unit][sample] = W h with the units in tiles of
// 16; the four values that a lane holds of tile I are the B operands of the
// next layer's four steps with k = 16 I + 4 lk + r, so no value changes
// lanes between the layers.  The sums stay in FP32, started from the bias.
// The weights of the hidden layer are read from LDS as the lanes' A operands
// of four steps (one b128), which leaves the registers for four waves a SIMD
// (held in registers with two waves: 6 % slower).
// 2.2 million coefficients: 508 us with a sample a lane and its 4736
// multiply-adds on the vector unit (bound there), 350 us now, of which the
// matrix unit is busy for 140 and the vector unit (tanh, features) for 190;
// the counters show the two adding up.
typedef float f4 __attribute__((ext_vector_type(4)));

// tanh without a branch (with the library's, whose two sides most waves take
// one after the other, the kernel needs 60 us more), errors below 1.6 ulp plus those of the
// exponential and the reciprocal: below 5/8 x + x^3 P(x^2) (P: the minimax
// polynomial of degree 4 in the relative error, 4.4e-9, fitted by reweighted
// least squares), above 1 - 2 / (1 + e^{2x}), where the error of e^{2x} is
// damped by 2 e^{2x} / (1 + e^{2x})^2.
__device__ __forceinline__ float mlp_tanh(float x) {
  const float a = __builtin_fabsf(x), s = x * x;
  const float e = __builtin_amdgcn_exp2f(2.8853900817779268f * a);
  const float big = 1.f - 2.f * __builtin_amdgcn_rcpf(1.f + e);
  float p = -0.0057049864f;
  p = __builtin_fmaf(p, s, 0.020639086f);
  p = __builtin_fmaf(p, s, -0.053739715f);
  p = __builtin_fmaf(p, s, 0.13331442f);
  p = __builtin_fmaf(p, s, -0.3333328f);
  const float small = __builtin_fmaf(p, s * x, x);
  return a < 0.625f ? small : __builtin_copysignf(big, x);
}

struct MlpWave {
  static constexpr int T = kMlpHidden / 16;
  static constexpr int kRow = kMlpIn + 1;  // LDS stride of a sample
  // float4 blocks in LDS: w2 [J][I][lane], then per lk: b1 [I][lk],
  // b2 [J][lk], w3 [o][J][lk]
  static constexpr int kW2 = 0, kB1 = kW2 + T * T * 64, kB2 = kB1 + 4 * T;
  static constexpr int kW3 = kB2 + 4 * T, kF4 = kW3 + kMlpOut * 4 * T;
  const f4* w;
  float w1[T][2], b3[kMlpOut];

  // The parameters into LDS (all threads of the block) and registers; the
  // caller synchronises the block before eval.
  __device__ __forceinline__ void load(const float* __restrict__ p, f4* lds,
                                       int lane) {
    w = lds;
    const int li = lane & 15, lk = lane >> 4;
    for (int e = threadIdx.x; e < kF4; e += blockDim.x) {
      const float* src;
      if (e < kB1) {
        const int l = e & 63, I = (e >> 6) % T, J = (e >> 6) / T;
        src = p + kMlpW2 + (16 * J + (l & 15)) * kMlpHidden + 16 * I +
              4 * (l >> 4);
      } else if (e < kB2) {
        src = p + kMlpB1 + 4 * (e - kB1);
      } else if (e < kW3) {
        src = p + kMlpB2 + 4 * (e - kB2);
      } else {
        src = p + kMlpW3 + 4 * (e - kW3);
      }
      lds[e] = f4{src[0], src[1], src[2], src[3]};
    }
#pragma unroll
    for (int I = 0; I < T; ++I)
#pragma unroll
      for (int m = 0; m < 2; ++m)
        w1[I][m] = p[kMlpW1 + (16 * I + li) * kMlpIn + 4 * m + lk];
#pragma unroll
    for (int o = 0; o < kMlpOut; ++o) b3[o] = p[kMlpB3 + o];
  }

  // y of the wave's 64 samples (lane = sample) with normalised features f;
  // x: 64 * kRow floats of LDS of this wave.
  __device__ __forceinline__ void eval(const float (&f)[kMlpIn], float* x,
                                       int lane, float (&y)[kMlpOut]) const {
    const int li = lane & 15, lk = lane >> 4;
    wave_sync();  // the previous samples are read
#pragma unroll
    for (int k = 0; k < kMlpIn; ++k) x[lane * kRow + k] = f[k];
    wave_sync();
#pragma unroll 1
    for (int t = 0; t < 4; ++t) {  // samples 16 t .. 16 t + 15
      // keeps the weights in LDS (hoisted out of the loop, they spill)
      asm volatile("" ::: "memory");
      const float* xs = x + (16 * t + li) * kRow + lk;
      const float x0 = xs[0], x1 = xs[4];
      f4 h[T];
#pragma unroll
      for (int I = 0; I < T; ++I) {
        f4 z = w[kB1 + 4 * I + lk];
        z = __builtin_amdgcn_mfma_f32_16x16x4f32(w1[I][0], x0, z, 0, 0, 0);
        h[I] = __builtin_amdgcn_mfma_f32_16x16x4f32(w1[I][1], x1, z, 0, 0, 0);
      }
#pragma unroll
      for (int I = 0; I < T; ++I)
#pragma unroll
        for (int r = 0; r < 4; ++r) h[I][r] = mlp_tanh(h[I][r]);
      f4 z[T];
#pragma unroll
      for (int J = 0; J < T; ++J) z[J] = w[kB2 + 4 * J + lk];
#pragma unroll
      for (int I = 0; I < T; ++I) {
        f4 a[T];
#pragma unroll
        for (int J = 0; J < T; ++J) a[J] = w[kW2 + (J * T + I) * 64 + lane];
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
          for (int J = 0; J < T; ++J)
            z[J] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[J][r], h[I][r], z[J],
                                                        0, 0, 0);
      }
      float s[kMlpOut] = {};
#pragma unroll
      for (int J = 0; J < T; ++J) {
        f4 v;
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] = mlp_tanh(z[J][r]);
#pragma unroll
        for (int o = 0; o < kMlpOut; ++o) {
          const f4 w3 = w[kW3 + 4 * (o * T + J) + lk];
#pragma unroll
          for (int r = 0; r < 4; ++r) s[o] += w3[r] * v[r];
        }
      }
#pragma unroll
      for (int o = 0; o < kMlpOut; ++o) {  // over lk, the same on all lanes
        s[o] += __shfl_xor(s[o], 16);
        s[o] += __shfl_xor(s[o], 32);
        if (lk == t) y[o] = s[o] + b3[o];
      }
    }
  }
};

// Blocks of 4 waves for n samples, at most 4 a CU; a wave takes runs of 64
// samples one after another (mlp_run: the first and the end of its part).
constexpr int kMlpBlock = 256, kMlpMaxBlocks = 1024;
inline unsigned mlp_blocks(int64_t n) {
  const int64_t b = (n + kMlpBlock - 1) / kMlpBlock;
  return (unsigned)(b < kMlpMaxBlocks ? b : kMlpMaxBlocks);
}
__device__ __forceinline__ int64_t mlp_run(int64_t n, int64_t* end) {
  const int64_t waves = (int64_t)gridDim.x * (kMlpBlock / 64);
  const int64_t runs = (n + 63) / 64;
  const int64_t w = (int64_t)blockIdx.x * (kMlpBlock / 64) +
                    __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  *end = (w + 1) * runs / waves * 64;
  return w * runs / waves * 64;
}

// Raw features of one coefficient: |G+k|^2, the band's tb (twice its
// kinetic energy), its energy gap below the highest occupied band of its
// (s,k) block (Rayleigh quotients; 0 for empty bands) and the density mean /
// variance of the current iterate.
__device__ inline double mlp_band_energy(double tb) {
  return tb > 1e-300 ? tb : 1e-300;
}
__device__ inline void mlp_density_features(double rho_mean, double rho_var,
                                            float x[kMlpIn]) {
  const double m = rho_mean > 1e-300 ? rho_mean : 1e-300;
  x[3] = (float)log(m);
  x[4] = (float)log1p((rho_var > 0.0 ? rho_var : 0.0) / (m * m));
}
__device__ inline void mlp_state_features(double tb, double gap,
                                          float x[kMlpIn]) {
  x[2] = (float)log(mlp_band_energy(tb));
  x[5] = (float)log1p(gap > 0.0 ? gap : 0.0);
}
__device__ inline void mlp_plane_wave_features(double gk2, double tb,
                                               float x[kMlpIn]) {
  x[0] = (float)log1p(gk2);
  x[1] = (float)log1p(gk2 / mlp_band_energy(tb));
}
__device__ inline void mlp_features(double gk2, double tb, double gap,
                                    double rho_mean, double rho_var,
                                    float x[kMlpIn]) {
  mlp_plane_wave_features(gk2, tb, x);
  mlp_state_features(tb, gap, x);
  mlp_density_features(rho_mean, rho_var, x);
  x[6] = 0.f;
  x[7] = 0.f;
}

// Clamp ranges of the two outputs before exponentiation.
constexpr float kLogFactorMin = -8.f, kLogFactorMax = 8.f;
constexpr float kLogAmpMin = -30.f, kLogAmpMax = 8.f;

}  // namespace jrx
