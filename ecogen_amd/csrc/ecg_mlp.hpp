// Learned Newton warm start of the infinite pressure relaxation (gfx950).
//
// The reference relaxation (RelaxationPInfinite::relaxation +
// RelaxationP::NewtonRaphson, RelaxationPInfinite.cpp:43-98,
// RelaxationP.cpp:43-93) starts Newton from the cold guess
// p_cold = sum_k alpha_k p_k.  Here a 12 -> 64 -> 64 -> 1 GELU network
// predicts the relaxed pressure instead; Newton then runs to the reference
// tolerance from that guess, and the cold-start Newton stays the fallback.
//
// Scale-free inputs, per phase slot k (3 slots, unused slots zero), from the
// pre-relaxation phase state (alpha_k, rho_k, p_k, e_k) through the EOS:
//   x_k0 = alpha_k
//   x_k1 = (p_k - p_cold) / s,          s = max_k |p_k - p_cold|
//   x_k2 = (alpha_k / Z_k) / sum_j (alpha_j / Z_j),   Z_k = rho_k c_k^2 = gamma_k (p_k + pinf_k)
//   x_k3 = s / (s + Z_k)
// x_k2 are the weights of the linearised relaxation, so t_lin = sum_k x_k2 x_k1
// is its normalised root.  The remainder t - t_lin is second order in the
// phase pressure spread; it is measured in units of
//   sigma = max(|sum_k x_k2 (t_lin - x_k1)^2 s / Z_k|, 1e-9)
// (computed in FP64) and the network predicts it in those units, clipped to
// +-4 in training:  p_guess = p_cold + s * (t_lin + sigma * y).  Where the
// relaxation is nearly linear sigma is tiny, so the network's BF16-limited
// error cannot spoil the linearised guess.
//
// Inference: BF16 weights and activations, FP32 accumulation on MFMA: the 12
// inputs (padded to 16) on v_mfma_f32_16x16x16_bf16, the two 64-wide layers on
// gfx950's v_mfma_f32_16x16x32_bf16.  Cells are the N dimension of every product,
// out^T[64 x 16 cells] = W^T[64 x K] in^T[K x 16 cells], so the accumulator
// fragment of one layer (lane l: rows 4*(l/16)+j, column l%16) is, after bias,
// GELU and BF16 rounding, a B fragment of the next: for a 32-deep product lane
// l's eight values are the four rows it holds of two consecutive 16-row tiles,
// and the weight fragments are packed with the same order of the K index, so no
// data moves between layers.
#pragma once

#include "ecg_physics.hpp"

namespace ecg {

constexpr int MLP_SLOTS = 3;
constexpr int MLP_IN = 12;
constexpr int MLP_H = 64;
// FP32 parameter vector: W1[IN][H], b1[H], W2[H][H], b2[H], w3[H], b3.
constexpr int MLP_OFF_W1 = 0;
constexpr int MLP_OFF_B1 = MLP_OFF_W1 + MLP_IN * MLP_H;
constexpr int MLP_OFF_W2 = MLP_OFF_B1 + MLP_H;
constexpr int MLP_OFF_B2 = MLP_OFF_W2 + MLP_H * MLP_H;
constexpr int MLP_OFF_W3 = MLP_OFF_B2 + MLP_H;
constexpr int MLP_OFF_B3 = MLP_OFF_W3 + MLP_H;
constexpr int MLP_NPARAM = MLP_OFF_B3 + 1;
// BF16 A fragments in units of 64 lanes x 4 values: W1 tiles mt = 0..3 (4 values a
// lane); W2 tiles (mt, q), q = 0..1 (8 values a lane, two units each); w3 tiles q.
constexpr int MLP_FRAG_W1 = 0;
constexpr int MLP_FRAG_W2 = 4;
constexpr int MLP_FRAG_W3 = 20;
constexpr int MLP_NFRAG = 24;
// Hidden unit that K slot j (0..7) of lane group g (= lane / 16) carries in the
// 32-deep block q of a 64-wide layer: the rows the previous layer's accumulator
// leaves in that lane, tile 2q then tile 2q + 1.
__host__ __device__ constexpr int mlp_k32_unit(int q, int g, int j) {
  return (j < 4) ? 32 * q + 4 * g + j : 32 * q + 16 + 4 * g + (j - 4);
}
// FP32 biases next to the fragments: b1[64], b2[64], b3.
constexpr int MLP_NBIAS = 2 * MLP_H + 1;
// Cells whose linearised residual exceeds this are sampled while a sample buffer is
// attached: every relaxation that needs more than the cold guess's first evaluation,
// a wider set than the cells the network is consulted for (WARM_MIN_RESIDUAL).
constexpr double CAPTURE_MIN_RESIDUAL = 1e-10;
// Relaxation sample record: features[12], t = (p* - p_cold)/s, cold-start
// iterations, u = (t - t_lin)/sigma (FP64-computed training target), sigma.
constexpr float MLP_TARGET_CLIP = 4.f;
constexpr int SAMPLE_FLOATS = 16;
// Newton evaluations allowed from the learned guess before the reference procedure
// continues from its first evaluation.
constexpr int WARM_MAX_IT = 30;
// The network is consulted only where the linearised residual at the cold
// guess, sum_k alpha_k (p_k - p_cold) / Z_k, exceeds this (and the linearised
// move exceeds its second-order scale, relax_features).  Below it the cold
// Newton reaches the 1e-10 tolerance in one or two evaluations, fewer than an
// inference is worth: on the 512^3 two-phase case a gate at 1e-11 warm-started
// ten times more cells, saved 2.6 times more evaluations and ran 2.4 % slower.
constexpr double WARM_MIN_RESIDUAL = 1e-6;

struct MlpDev {
  const uint2* frag;     // MLP_NFRAG * 64 entries of 4 packed BF16
  const float* bias;     // MLP_NBIAS
};

__device__ __forceinline__ float gelu_f(float x) {
  const float u = 0.7978845608f * (x + 0.044715f * x * x * x);
  const float th = 1.f - 2.f * __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(2.885390082f * u));
  return 0.5f * x * (1.f + th);
}
// d gelu / dx of the same tanh form.
__device__ __forceinline__ float gelu_grad_f(float x) {
  const float u = 0.7978845608f * (x + 0.044715f * x * x * x);
  const float th = 1.f - 2.f * __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(2.885390082f * u));
  return 0.5f * (1.f + th) + 0.5f * x * (1.f - th * th) * 0.7978845608f * (1.f + 0.134145f * x * x);
}

// FP32 -> BF16, round to nearest even (finite inputs).
__device__ __host__ __forceinline__ unsigned short bf16_bits(float f) {
  unsigned int u = __builtin_bit_cast(unsigned int, f);
  u += 0x7FFFu + ((u >> 16) & 1u);
  return (unsigned short)(u >> 16);
}
__device__ __forceinline__ unsigned int pack_bf16x2(float a, float b) {
  return (unsigned int)bf16_bits(a) | ((unsigned int)bf16_bits(b) << 16);
}

// Features of one cell before relaxation (double state); false when the linearised
// residual at the cold guess is at most `gate` (WARM_MIN_RESIDUAL for the warm start,
// CAPTURE_MIN_RESIDUAL for sampling) or, for the warm start (`warm`), when the
// linearised move |t_lin| is within the second-order scale sigma.
template <int N>
__device__ __forceinline__ bool relax_features(const Params& P, const Cell<N>& s, double gate, bool warm, double& p_cold,
                                               double& spread, float* x, float& t_lin, double& t_lin_d,
                                               double& sigma) {
  double pc = 0.;
#pragma unroll
  for (int k = 0; k < N; k++) pc += s.a[k] * s.p[k];
  double sp = 0.;
#pragma unroll
  for (int k = 0; k < N; k++) sp = fmax(sp, fabs(s.p[k] - pc));
  p_cold = pc;
  spread = sp;
#pragma unroll
  for (int i = 0; i < MLP_IN; i++) x[i] = 0.f;
  t_lin = 0.f;
  t_lin_d = 0.;
  sigma = 1e-9;
  if (!(sp > 0.)) return false;
  // The quotients by Z_k, sp and wsum share one reciprocal each (div_ieee: the
  // IEEE quotients bit for bit).
  double w[N], wsum = 0., Z[N], iZ[N], flin = 0.;
#pragma unroll
  for (int k = 0; k < N; k++) {
    Z[k] = fmax(P.eos[k].g * (s.p[k] + P.eos[k].pinf), 1.e-300);
    iZ[k] = rcp_ieee(Z[k]);
    w[k] = div_ieee(s.a[k], Z[k], iZ[k]);
    wsum += w[k];
    flin += w[k] * (s.p[k] - pc);
  }
  if (!(fabs(flin) > gate)) return false;
  const double isp = rcp_ieee(sp), iws = rcp_ieee(wsum);
  double tl = 0., dp[N], wk[N];
#pragma unroll
  for (int k = 0; k < N; k++) {
    dp[k] = div_ieee(s.p[k] - pc, sp, isp);
    wk[k] = div_ieee(w[k], wsum, iws);
    x[4 * k + 0] = (float)s.a[k];
    x[4 * k + 1] = (float)dp[k];
    x[4 * k + 2] = (float)wk[k];
    x[4 * k + 3] = (float)div1(sp, sp + Z[k]);
    tl += wk[k] * dp[k];
  }
  double r2 = 0.;
#pragma unroll
  for (int k = 0; k < N; k++) {
    const double d = tl - dp[k];
    r2 += wk[k] * d * d * div_ieee(sp, Z[k], iZ[k]);
  }
  sigma = fmax(fabs(r2), 1e-9);
  t_lin = (float)tl;
  t_lin_d = tl;
  // The warm start also needs the linearised move from the cold guess to exceed the
  // second-order scale: where |t_lin| <= sigma the cold guess is already that close
  // to the root (a nearly pure cell with trace phases far from its pressure), the
  // cold Newton ends in two evaluations, and a guess from the network, whose error
  // is a fraction of sigma, cannot do better.
  return !warm || fabs(tl) > sigma;
}

typedef short v4i16 __attribute__((ext_vector_type(4)));
typedef float v4f32 __attribute__((ext_vector_type(4)));
typedef __bf16 v8bf16 __attribute__((ext_vector_type(8)));

// Eight BF16 values: a 16x16x32 fragment.
__device__ __forceinline__ v8bf16 as_v8bf16(uint4 v) { return __builtin_bit_cast(v8bf16, v); }
__device__ __forceinline__ v8bf16 join_frags(v4i16 lo, v4i16 hi) {
  const uint2 a = __builtin_bit_cast(uint2, lo), b = __builtin_bit_cast(uint2, hi);
  return as_v8bf16(make_uint4(a.x, a.y, b.x, b.y));
}

__device__ __forceinline__ v4i16 as_v4i16(uint2 v) {
  v4i16 r;
  r[0] = (short)(v.x & 0xFFFFu); r[1] = (short)(v.x >> 16);
  r[2] = (short)(v.y & 0xFFFFu); r[3] = (short)(v.y >> 16);
  return r;
}

// Bias + GELU on an accumulator fragment (rows 4*(l/16)+j of tile mt) -> BF16 B fragment.
__device__ __forceinline__ v4i16 act_frag(const v4f32& acc, const float* __restrict__ bias, int mt, int lane) {
  const int r0 = mt * 16 + 4 * (lane >> 4);
  uint2 o;
  o.x = pack_bf16x2(gelu_f(acc[0] + bias[r0 + 0]), gelu_f(acc[1] + bias[r0 + 1]));
  o.y = pack_bf16x2(gelu_f(acc[2] + bias[r0 + 2]), gelu_f(acc[3] + bias[r0 + 3]));
  return as_v4i16(o);
}

// LDS one wave needs for mlp_wave_infer: 64 rows of 16 BF16 features, then 64
// FP32 outputs; a 256-thread block needs four of them.
constexpr int MLP_WAVE_LDS = 64 * 16 * 2 + 64 * 4;
constexpr int MLP_BLOCK_LDS = 4 * MLP_WAVE_LDS;

// Network output for one tile of 16 staged rows (rows nt*16 .. nt*16+15);
// one wave, wave-uniform control flow.
__device__ __forceinline__ void mlp_infer_tile(const MlpDev& M, const unsigned short* fstage, float* ystage, int nt) {
  const int lane = threadIdx.x & 63;
  // B fragment of the inputs: features 4*(l/16)..+3 of row nt*16 + l%16.
  const uint2 xin = *reinterpret_cast<const uint2*>(fstage + (nt * 16 + (lane & 15)) * 16 + 4 * (lane >> 4));
  const v4i16 bx = as_v4i16(xin);
  const float* b1 = M.bias;
  const float* b2 = M.bias + MLP_H;
  v4i16 h1[4];
#pragma unroll
  for (int mt = 0; mt < 4; mt++) {
    v4f32 acc = {0.f, 0.f, 0.f, 0.f};
    acc = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(as_v4i16(M.frag[(MLP_FRAG_W1 + mt) * 64 + lane]), bx, acc, 0, 0, 0);
    h1[mt] = act_frag(acc, b1, mt, lane);
  }
  const v8bf16 x2[2] = {join_frags(h1[0], h1[1]), join_frags(h1[2], h1[3])};
  const uint4* w2 = reinterpret_cast<const uint4*>(M.frag + MLP_FRAG_W2 * 64);
  const uint4* w3 = reinterpret_cast<const uint4*>(M.frag + MLP_FRAG_W3 * 64);
  // Layer 3 consumes the 16-row tiles of layer 2 in pairs, as soon as they are
  // activated.  The loop stays rolled: unrolled, the compiler interleaves all the
  // GELUs and the inference alone needs far more VGPRs, which costs the fused step
  // kernel a wave per SIMD.
  v4f32 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
  for (int q = 0; q < 2; q++) {
    asm volatile("" ::: "memory");
    v4i16 h2[2];
#pragma unroll
    for (int half = 0; half < 2; half++) {
      const int mt = 2 * q + half;
      v4f32 a2 = {0.f, 0.f, 0.f, 0.f};
      a2 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_v8bf16(w2[(mt * 2 + 0) * 64 + lane]), x2[0], a2, 0, 0, 0);
      a2 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_v8bf16(w2[(mt * 2 + 1) * 64 + lane]), x2[1], a2, 0, 0, 0);
      h2[half] = act_frag(a2, b2, mt, lane);
    }
    acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_v8bf16(w3[q * 64 + lane]), join_frags(h2[0], h2[1]), acc, 0, 0, 0);
  }
  // Row 0 of the output tile: lanes 0..15, element 0.
  if (lane < 16) ystage[nt * 16 + lane] = acc[0] + M.bias[2 * MLP_H];
}

// Network output y for every lane of the calling wave whose `need` is set (others
// get 0).  The wave's candidates are compacted into LDS rows of its own region
// (MLP_WAVE_LDS bytes at lds), and it runs as many 16-row tiles as they fill: a
// wave without a candidate does nothing, and no other wave is waited for.  The
// region must be free of other use: the step kernel calls it after its last flux
// pass, whose closing barrier has released the staging LDS.
__device__ __forceinline__ float mlp_wave_infer(const MlpDev& M, bool need, const float* x, unsigned char* lds) {
  const int lane = threadIdx.x & 63;
  const unsigned long long m = __ballot(need);
  if (m == 0ull) return 0.f;   // wave-uniform
  const int total = __popcll(m);
  const int rank = __popcll(m & ((1ull << lane) - 1ull));
  unsigned short* fstage = reinterpret_cast<unsigned short*>(lds);
  float* ystage = reinterpret_cast<float*>(lds + 64 * 16 * 2);
  if (need) {
    uint4 a, b;
    a.x = pack_bf16x2(x[0], x[1]);  a.y = pack_bf16x2(x[2], x[3]);
    a.z = pack_bf16x2(x[4], x[5]);  a.w = pack_bf16x2(x[6], x[7]);
    b.x = pack_bf16x2(x[8], x[9]);  b.y = pack_bf16x2(x[10], x[11]);
    b.z = 0u; b.w = 0u;
    uint4* dst = reinterpret_cast<uint4*>(fstage + rank * 16);
    dst[0] = a;
    dst[1] = b;
  }
  // The rows become visible to the whole wave.
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  const int ntiles = (total + 15) >> 4;
  // Keeps the weight fragments in L1/L2 rather than in registers for the whole kernel.
#pragma unroll 1
  for (int nt = 0; nt < ntiles; nt++) {
    asm volatile("" ::: "memory");
    mlp_infer_tile(M, fstage, ystage, nt);
  }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  return need ? ystage[rank] : 0.f;
}

}  // namespace ecg
