// Learned Newton warm start: relaxation sample buffers, training kernels
// (FP32 forward/backward with deterministic block partials, Adam) and the
// BF16 fragment packing used by the fused MFMA inference in the step kernel.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <numeric>
#include <vector>

#include "ecg_learn.hpp"

namespace ecg {

// Training sums run in a fixed order: chunks of TBS samples of a batch, samples in order
// within a chunk, chunks in order.  A batch is worked off in segments of at most
// SEG_CHUNKS chunks (35 MB of activations), the running sums carried between them.
constexpr int TBS = 64;
constexpr int SEG_CHUNKS = 512;
constexpr int FB_SAMPLES = 16;             // samples of a k_mlp_fwd_bwd block, of 16 different chunks
constexpr int LDU = MLP_H + 4;             // padded row of the block's per-sample rows (16-byte aligned)
// Rows of the activation workspace: row u, sample r of its chunk and chunk c lie at
// (u * TBS + r) * ld + c, so that a wave whose lanes are chunks reads consecutive words.
constexpr int ACT_H1 = 0, ACT_DZ2 = MLP_H, ACT_DZ1 = 2 * MLP_H, ACT_P3 = 3 * MLP_H, ACT_X = 4 * MLP_H;
constexpr int ACT_DY = ACT_X + MLP_IN, ACT_LS = ACT_DY + 1, ACT_ROWS = ACT_LS + 1;

// Orders of the three phase slots; training sees every order of every sample.
__constant__ int k_slot_perm[6][3] = {{0, 1, 2}, {0, 2, 1}, {1, 0, 2}, {1, 2, 0}, {2, 0, 1}, {2, 1, 0}};

__device__ __forceinline__ unsigned long long mix64(unsigned long long z) {
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  return z ^ (z >> 31);
}

// Forward and backward pass of the mean squared error of the clipped remainder
// r = clip(u), samples idx = (mult * (q0 + b) + offs) mod n of a batch of `count`; every
// factor of the parameter gradients goes to the activation workspace (rows above).
// Sixteen threads share a sample, four hidden units each, so that a 4096-record batch
// fills the chip's 256 CUs with a block each; a thread's sum over the 64 units of a layer
// stays one chain in the units' order.  Bound by LDS: per unit a 16-byte weight read and a
// broadcast feed four multiply-adds.  With one thread per sample (64 blocks of one wave,
// the weight gradients from the same block) a batch took 110 us here and 25 us in the
// reduction, loss and optimiser kernels behind it; now 12 us and 8 us (k_mlp_grad).
__global__ __launch_bounds__(256) void k_mlp_fwd_bwd(const float* __restrict__ prm_g, const float* __restrict__ smp,
                                                     long long n, long long q0, long long count,
                                                     unsigned long long mult, unsigned long long offs,
                                                     unsigned long long perm_seed, float inv_batch, long long c0,
                                                     int nchunk, int ld, float* __restrict__ act) {
  __shared__ __align__(16) float prm[(MLP_NPARAM + 3) & ~3];
  __shared__ __align__(16) float W2T[MLP_H * LDU];
  __shared__ __align__(16) float H1[FB_SAMPLES * LDU], PW[FB_SAMPLES * LDU], D2[FB_SAMPLES * LDU], P3[FB_SAMPLES * LDU];
  __shared__ __align__(16) float X[FB_SAMPLES * MLP_IN];
  __shared__ float DY[FB_SAMPLES], LS[FB_SAMPLES];
  const int t = threadIdx.x;
  const int s = t >> 4, tj = t & 15;
  const int r = blockIdx.x & (TBS - 1), cb = (blockIdx.x / TBS) * FB_SAMPLES;

  // The sample's record: thread tj < 12 holds input tj, every thread the target.
  float xin = 0.f, tgt = 0.f, msk = 0.f;
  const long long b = (c0 + cb + s) * TBS + r;
  if (cb + s < nchunk && b < count) {
    const unsigned long long q = (unsigned long long)(q0 + b);
    const long long idx = (long long)((mult * q + offs) % (unsigned long long)n);
    const float* rec = smp + idx * SAMPLE_FLOATS;
    const int pm = perm_seed ? (int)(mix64(perm_seed ^ (unsigned long long)idx * 0x9E3779B97F4A7C15ull) % 6ull) : 0;
    if (tj < MLP_IN) xin = rec[4 * k_slot_perm[pm][tj >> 2] + (tj & 3)];
    tgt = fminf(fmaxf(rec[14], -MLP_TARGET_CLIP), MLP_TARGET_CLIP);
    msk = 1.f;
  }
  for (int i = t; i < MLP_NPARAM / 4; i += 256)
    reinterpret_cast<float4*>(prm)[i] = reinterpret_cast<const float4*>(prm_g)[i];
  if (t < (MLP_NPARAM & 3)) prm[(MLP_NPARAM & ~3) + t] = prm_g[(MLP_NPARAM & ~3) + t];
  for (int e = t; e < MLP_H * MLP_H; e += 256) W2T[(e & 63) * LDU + (e >> 6)] = prm_g[MLP_OFF_W2 + e];
  if (tj < MLP_IN) X[s * MLP_IN + tj] = xin;
  __syncthreads();

  const float4* W1 = reinterpret_cast<const float4*>(prm + MLP_OFF_W1) + tj;   // row i: + i * 16
  const float4* W2 = reinterpret_cast<const float4*>(prm + MLP_OFF_W2) + tj;
  const float4* WT = reinterpret_cast<const float4*>(W2T) + tj;                // row j: + j * LDU / 4
  auto unit4 = [&](int off) { return *reinterpret_cast<const float4*>(prm + off + 4 * tj); };
  auto row4 = [&](float* A) { return reinterpret_cast<float4*>(A + s * LDU); };
  auto mac = [](float4& a, float x, const float4& w) {
    a.x += x * w.x; a.y += x * w.y; a.z += x * w.z; a.w += x * w.w;
  };
  // A layer's 64 inputs (row in of the sample) against rows w, stride ws, of 64 units.
  auto layer = [&](float4 acc, const float4* in, const float4* w, int ws) {
#pragma unroll 8
    for (int i = 0; i < MLP_H / 4; i++) {
      const float4 h = in[i];
      mac(acc, h.x, w[(4 * i + 0) * ws]);
      mac(acc, h.y, w[(4 * i + 1) * ws]);
      mac(acc, h.z, w[(4 * i + 2) * ws]);
      mac(acc, h.w, w[(4 * i + 3) * ws]);
    }
    return acc;
  };
  const float4 w3 = unit4(MLP_OFF_W3);

  float4 z1 = unit4(MLP_OFF_B1);
#pragma unroll
  for (int i = 0; i < MLP_IN; i++) mac(z1, X[s * MLP_IN + i], W1[i * (MLP_H / 4)]);
  row4(H1)[tj] = make_float4(gelu_f(z1.x), gelu_f(z1.y), gelu_f(z1.z), gelu_f(z1.w));
  __syncthreads();
  const float4 z2 = layer(unit4(MLP_OFF_B2), row4(H1), W2, MLP_H / 4);
  const float4 g2 = make_float4(gelu_f(z2.x), gelu_f(z2.y), gelu_f(z2.z), gelu_f(z2.w));
  row4(PW)[tj] = make_float4(w3.x * g2.x, w3.y * g2.y, w3.z * g2.z, w3.w * g2.w);
  __syncthreads();
  float y = prm[MLP_OFF_B3];
  float4 pw[MLP_H / 4];
#pragma unroll
  for (int i = 0; i < MLP_H / 4; i++) pw[i] = row4(PW)[i];
  __builtin_amdgcn_sched_barrier(0);   // the reads together, then the chain of additions
#pragma unroll
  for (int i = 0; i < MLP_H / 4; i++) { y += pw[i].x; y += pw[i].y; y += pw[i].z; y += pw[i].w; }
  const float d = y - tgt;
  const float dy = msk * 2.f * d * inv_batch;
  if (tj == 0) { DY[s] = dy; LS[s] = msk * d * d; }
  row4(D2)[tj] = make_float4(dy * w3.x * gelu_grad_f(z2.x), dy * w3.y * gelu_grad_f(z2.y), dy * w3.z * gelu_grad_f(z2.z),
                             dy * w3.w * gelu_grad_f(z2.w));
  row4(P3)[tj] = make_float4(dy * g2.x, dy * g2.y, dy * g2.z, dy * g2.w);
  __syncthreads();
  // dL/dz1 = (W2 dz2) * gelu'(z1), into the output products' rows.
  const float4 a1 = layer(make_float4(0.f, 0.f, 0.f, 0.f), row4(D2), WT, LDU / 4);
  row4(PW)[tj] = make_float4(a1.x * gelu_grad_f(z1.x), a1.y * gelu_grad_f(z1.y), a1.z * gelu_grad_f(z1.z),
                             a1.w * gelu_grad_f(z1.w));
  __syncthreads();

  // To the workspace, the block's 16 chunks (64 bytes) of one row per four threads.
  const int u = t >> 2, q4 = 4 * (t & 3);
  auto put = [&](int row, const float* A, int lda, int col) {
    *reinterpret_cast<float4*>(act + ((size_t)row * TBS + r) * ld + cb + q4) =
        make_float4(A[q4 * lda + col], A[(q4 + 1) * lda + col], A[(q4 + 2) * lda + col], A[(q4 + 3) * lda + col]);
  };
  put(ACT_H1 + u, H1, LDU, u);
  put(ACT_DZ2 + u, D2, LDU, u);
  put(ACT_DZ1 + u, PW, LDU, u);
  put(ACT_P3 + u, P3, LDU, u);
  if (u < MLP_IN) put(ACT_X + u, X, MLP_IN, u);
  else if (u == MLP_IN) put(ACT_DY, DY, 1, 0);
  else if (u == MLP_IN + 1) put(ACT_LS, LS, 1, 0);
}

// Parameter gradients of a segment of nchunk chunks from the activation workspace, and
// with last and adam_m the optimiser step: one wave for eight parameters, a 2 x 4 tile of
// a weight matrix or eight column sums (and one wave for b3 and the loss).  Lanes are chunks
// and sum their 64 samples in order; eight threads then add the chunks in order.  633 waves
// over the chip; a 2 x 4 tile reads six rows for eight products, which keeps a CU's loads
// (48 cycles of L1 a sample for its two or three waves) below their arithmetic (64 cycles a
// SIMD).  The eight XCDs take eight rows of W2 each, so that each L2 holds an eighth of h1.
constexpr int GR_W2 = (MLP_H / 2) * (MLP_H / 4), GR_W1 = (MLP_IN / 2) * (MLP_H / 4), GR_SUM = 3 * MLP_H / 8;
constexpr int GR_BLOCKS = GR_W2 + GR_W1 + GR_SUM + 1;
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(1, 1))) void k_mlp_grad(const float* __restrict__ act, int nchunk, int ld, int first, int last,
                                                 float* __restrict__ grad, float* __restrict__ adam_m,
                                                 float* __restrict__ adam_v, float* __restrict__ prm, float lr_t,
                                                 double* __restrict__ loss_part, double* __restrict__ loss, int loss_first) {
  constexpr int LDG = 68, RB = 16;
  __shared__ __align__(16) float part[8 * LDG];
  const int t = threadIdx.x, blk = blockIdx.x;
  int ra, rb, kind, p = -1;   // first rows; 0: tile, 1: column sums, 2: b3 and the loss; the thread's parameter
  if (blk < GR_W2) {
    const int i = 2 * ((blk & 7) * 4 + ((blk >> 3) & 3)), j = 4 * (blk >> 5);
    kind = 0; ra = ACT_H1 + i; rb = ACT_DZ2 + j;
    p = MLP_OFF_W2 + (i + (t >> 2)) * MLP_H + j + (t & 3);
  } else if (blk < GR_W2 + GR_W1) {
    const int e = blk - GR_W2, i = 2 * (e >> 4), j = 4 * (e & 15);
    kind = 0; ra = ACT_X + i; rb = ACT_DZ1 + j;
    p = MLP_OFF_W1 + (i + (t >> 2)) * MLP_H + j + (t & 3);
  } else if (blk < GR_W2 + GR_W1 + GR_SUM) {
    const int e = blk - GR_W2 - GR_W1, j = 8 * (e & 7);
    kind = 1; ra = rb = ((e >> 3) == 0 ? ACT_DZ1 : (e >> 3) == 1 ? ACT_DZ2 : ACT_P3) + j;
    p = ((e >> 3) == 0 ? MLP_OFF_B1 : (e >> 3) == 1 ? MLP_OFF_B2 : MLP_OFF_W3) + j + t;
  } else {
    kind = 2; ra = rb = ACT_DY;   // and the losses, the row behind it
    p = MLP_OFF_B3;
  }
  const bool owner = t < ((kind == 2) ? 1 : 8);
  const bool step = owner && last && adam_m != nullptr;
  float g = (owner && !first) ? grad[p] : 0.f;
  float m = 0.f, v = 0.f, w = 0.f;
  if (step) { m = adam_m[p]; v = adam_v[p]; w = prm[p]; }
  double lsum = (kind == 2 && t == 1 && !first) ? *loss_part : 0.;

  const size_t rs = (size_t)TBS * ld;
  for (int c0 = 0; c0 < nchunk; c0 += 64) {
    const int nc = (nchunk - c0 < 64) ? nchunk - c0 : 64;
    const float* A = act + ra * rs + c0 + (t < nc ? t : nc - 1);
    const float* B = act + rb * rs + c0 + (t < nc ? t : nc - 1);
    float a[8];
#pragma unroll
    for (int k = 0; k < 8; k++) a[k] = 0.f;
    // Loads of RB samples are issued together, ahead of the sums (the workspace comes from the
    // other XCDs' writes; the compiler's own order waited for every load, 24 us).
    if (kind == 0) {
      for (int r0 = 0; r0 < TBS; r0 += RB) {
        float f[RB][6];
#pragma unroll
        for (int r = 0; r < RB; r++) {
          const int o = (r0 + r) * ld;
          f[r][0] = A[o]; f[r][1] = A[rs + o];
#pragma unroll
          for (int k = 0; k < 4; k++) f[r][2 + k] = B[k * rs + o];
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int r = 0; r < RB; r++)
#pragma unroll
          for (int k = 0; k < 8; k++) a[k] += f[r][k >> 2] * f[r][2 + (k & 3)];
      }
    } else {
      const int rows = (kind == 1) ? 8 : 2;
      for (int r0 = 0; r0 < TBS; r0 += RB) {
        float f[RB][8];
#pragma unroll
        for (int r = 0; r < RB; r++)
#pragma unroll
          for (int k = 0; k < 8; k++) f[r][k] = A[(k < rows ? k : 0) * rs + (r0 + r) * ld];
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int r = 0; r < RB; r++)
#pragma unroll
          for (int k = 0; k < 8; k++) a[k] += f[r][k];
      }
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 8; k++) part[k * LDG + t] = a[k];
    __syncthreads();
    if (owner) {
      const float* q = part + t * LDG;
      int c = 0;
      if (nc == 64) {
        float4 f[16];
#pragma unroll
        for (int k = 0; k < 16; k++) f[k] = reinterpret_cast<const float4*>(q)[k];
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int k = 0; k < 16; k++) { g += f[k].x; g += f[k].y; g += f[k].z; g += f[k].w; }
        c = 64;
      }
      for (; c < nc; c++) g += q[c];
    } else if (kind == 2 && t == 1) {
      for (int c = 0; c < nc; c++) lsum += (double)part[LDG + c];
    }
  }
  if (kind == 2 && t == 1) {
    if (!last) *loss_part = lsum;
    else if (loss_first) *loss = lsum;
    else *loss += lsum;
  }
  if (step) {
    m = 0.9f * m + 0.1f * g;
    v = 0.999f * v + 0.001f * g * g;
    adam_m[p] = m;
    adam_v[p] = v;
    prm[p] = w - lr_t * m / (sqrtf(v) + 1e-8f);
  } else if (owner) {
    grad[p] = g;
  }
}

// BF16 A fragments of v_mfma_f32_16x16x16bf16_1k (lane l holds A[l%16][4*(l/16)+j])
// of W^T for every (output tile, input tile), plus the FP32 biases.
__global__ __launch_bounds__(256) void k_mlp_pack(const float* __restrict__ prm, uint2* __restrict__ frag,
                                                  float* __restrict__ bias) {
  const int e = blockIdx.x * 256 + threadIdx.x;
  if (e < MLP_NBIAS) {
    bias[e] = (e < MLP_H) ? prm[MLP_OFF_B1 + e] : (e < 2 * MLP_H) ? prm[MLP_OFF_B2 + e - MLP_H] : prm[MLP_OFF_B3];
  }
  if (e >= MLP_NFRAG * 64) return;
  const int f = e >> 6, l = e & 63;
  const int i = l & 15, g = l >> 4;
  float v[4];
  if (f < MLP_FRAG_W2) {
    // 16x16x16 fragment of W1^T: lane (g, i) holds output unit 16 mt + i, inputs 4 g + j.
    const int mt = f - MLP_FRAG_W1;
    for (int j = 0; j < 4; j++) {
      const int k = 4 * g + j;
      v[j] = (k < MLP_IN) ? prm[MLP_OFF_W1 + k * MLP_H + mt * 16 + i] : 0.f;
    }
  } else {
    // 16x16x32 fragments, two 4-value units each (unit u = f - MLP_FRAG_W2): lane (g, i)
    // holds output unit i of its tile and the hidden units mlp_k32_unit(q, g, .).
    const int u = f - MLP_FRAG_W2;
    const bool w3 = u >= 16;
    const int t = (w3 ? u - 16 : u) >> 1, part = u & 1;        // fragment index, half of its 8 values
    const int q = w3 ? t : (t & 1), mt = w3 ? 0 : (t >> 1);
    // A uint4 fragment of lane l spans units 2 t (lanes 0..31 as uint2 pairs) ... : the
    // uint2 slot e of the unit region is (fragment t, lane e / 2, half e % 2).
    const int lane4 = (part * 64 + l) >> 1, half = (part * 64 + l) & 1;
    const int ii = lane4 & 15, gg = lane4 >> 4;
    for (int j = 0; j < 4; j++) {
      const int h = mlp_k32_unit(q, gg, 4 * half + j);
      v[j] = w3 ? ((ii == 0) ? prm[MLP_OFF_W3 + h] : 0.f) : prm[MLP_OFF_W2 + h * MLP_H + mt * 16 + ii];
    }
  }
  frag[e] = make_uint2(pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]));
}

// Stand-alone inference over sample records with the device function the step
// kernel fuses into the relaxation: out = the network output y (the warm start
// uses t_lin + sigma * y).
__global__ __launch_bounds__(256) void k_mlp_predict(MlpDev M, const float* __restrict__ smp, long long n,
                                                     float* __restrict__ out) {
  __shared__ __align__(16) unsigned char stage[MLP_BLOCK_LDS];
  const long long g = (long long)blockIdx.x * 256 + threadIdx.x;
  float x[MLP_IN];
#pragma unroll
  for (int i = 0; i < MLP_IN; i++) x[i] = 0.f;
  if (g < n) {
    const float* rec = smp + g * SAMPLE_FLOATS;
#pragma unroll
    for (int i = 0; i < MLP_IN; i++) x[i] = rec[i];
  }
  const float y = mlp_wave_infer(M, g < n, x, stage + (threadIdx.x >> 6) * MLP_WAVE_LDS);
  if (g < n) out[g] = y;
}

int api_fail(int code, const std::string& msg);

long long samples_count(ecg_samples* s) {
  if (s->uploaded >= 0) return s->uploaded;
  unsigned long long seen = 0;
  if (hipDeviceSynchronize() != hipSuccess) return -1;
  if (hipMemcpy(&seen, s->seen, sizeof(seen), hipMemcpyDeviceToHost) != hipSuccess) return -1;
  const unsigned long long st = (unsigned long long)(s->stride > 0 ? s->stride : 1);
  const unsigned long long used = (unsigned long long)s->base + (seen + st - 1) / st;
  return (long long)(used < (unsigned long long)s->cap ? used : (unsigned long long)s->cap);
}

}  // namespace ecg

using namespace ecg;

#define HIPCHK(expr)                                                                                     \
  do {                                                                                                   \
    hipError_t e_ = (expr);                                                                              \
    if (e_ != hipSuccess) return api_fail(ECG_E_HIP, std::string(#expr) + ": " + hipGetErrorString(e_)); \
  } while (0)

extern "C" {

ecg_samples* ecg_samples_create(int64_t capacity) {
  if (capacity <= 0) { api_fail(ECG_E_ARG, "sample capacity must be positive"); return nullptr; }
  ecg_samples* s = new ecg_samples();
  s->cap = capacity;
  if (hipMalloc(&s->buf, (size_t)capacity * SAMPLE_FLOATS * sizeof(float)) != hipSuccess ||
      hipMalloc(&s->seen, sizeof(unsigned long long)) != hipSuccess ||
      hipMemset(s->seen, 0, sizeof(unsigned long long)) != hipSuccess) {
    api_fail(ECG_E_HIP, "device allocation of the sample buffer failed");
    if (s->buf) hipFree(s->buf);
    if (s->seen) hipFree(s->seen);
    delete s;
    return nullptr;
  }
  return s;
}

int ecg_samples_destroy(ecg_samples* s) {
  if (!s) return ECG_OK;
  if (s->attached > 0) return api_fail(ECG_E_ARG, "the sample buffer is attached to a solver context (detach it first)");
  hipDeviceSynchronize();
  hipFree(s->buf);
  hipFree(s->seen);
  delete s;
  return ECG_OK;
}

int ecg_samples_reset(ecg_samples* s) {
  if (!s) return api_fail(ECG_E_ARG, "null sample buffer");
  HIPCHK(hipDeviceSynchronize());
  HIPCHK(hipMemset(s->seen, 0, sizeof(unsigned long long)));
  s->uploaded = -1;
  s->base = 0;
  s->stride = 1;
  return ECG_OK;
}

int64_t ecg_samples_count(ecg_samples* s) {
  if (!s) return api_fail(ECG_E_ARG, "null sample buffer");
  const long long n = samples_count(s);
  if (n < 0) return api_fail(ECG_E_HIP, "reading the sample counter failed");
  return n;
}

int64_t ecg_samples_seen(ecg_samples* s) {
  if (!s) return api_fail(ECG_E_ARG, "null sample buffer");
  unsigned long long seen = 0;
  HIPCHK(hipDeviceSynchronize());
  HIPCHK(hipMemcpy(&seen, s->seen, sizeof(seen), hipMemcpyDeviceToHost));
  return (int64_t)seen;
}

int ecg_samples_download(ecg_samples* s, float* host, int64_t n) {
  if (!s || !host || n < 0) return api_fail(ECG_E_ARG, "invalid sample download arguments");
  const long long have = samples_count(s);
  if (have < 0) return api_fail(ECG_E_HIP, "reading the sample counter failed");
  if (n > have) return api_fail(ECG_E_ARG, "more records requested than the buffer holds");
  HIPCHK(hipMemcpy(host, s->buf, (size_t)n * SAMPLE_FLOATS * sizeof(float), hipMemcpyDeviceToHost));
  return ECG_OK;
}

int ecg_samples_upload(ecg_samples* s, const float* host, int64_t n) {
  if (!s || !host || n < 0 || n > s->cap) return api_fail(ECG_E_ARG, "invalid sample upload arguments");
  HIPCHK(hipDeviceSynchronize());
  HIPCHK(hipMemcpy(s->buf, host, (size_t)n * SAMPLE_FLOATS * sizeof(float), hipMemcpyHostToDevice));
  HIPCHK(hipMemset(s->seen, 0, sizeof(unsigned long long)));
  s->uploaded = n;
  return ECG_OK;
}

ecg_mlp* ecg_mlp_create(uint64_t seed) {
  ecg_mlp* M = new ecg_mlp();
  bool ok = hipStreamCreateWithFlags(&M->stream, hipStreamNonBlocking) == hipSuccess;
  ok = ok && hipMalloc(&M->prm, MLP_NPARAM * sizeof(float)) == hipSuccess;
  ok = ok && hipMalloc(&M->adam_m, MLP_NPARAM * sizeof(float)) == hipSuccess;
  ok = ok && hipMalloc(&M->adam_v, MLP_NPARAM * sizeof(float)) == hipSuccess;
  ok = ok && hipMalloc(&M->grad, MLP_NPARAM * sizeof(float)) == hipSuccess;
  ok = ok && hipMalloc(&M->frag, MLP_NFRAG * 64 * sizeof(uint2)) == hipSuccess;
  ok = ok && hipMalloc(&M->bias, MLP_NBIAS * sizeof(float)) == hipSuccess;
  if (!ok) {
    api_fail(ECG_E_HIP, "device allocation of the network failed");
    ecg_mlp_destroy(M);
    return nullptr;
  }
  // He-scaled normal weights (xorshift64* + Box-Muller), zero biases, small output layer
  // so that the untrained network returns the linearised guess.
  std::vector<float> h(MLP_NPARAM, 0.f);
  unsigned long long st = seed * 0x9E3779B97F4A7C15ull + 0x2545F4914F6CDD1Dull;
  auto uni = [&]() {
    st ^= st >> 12; st ^= st << 25; st ^= st >> 27;
    return ((st * 0x2545F4914F6CDD1Dull) >> 11) * (1.0 / 9007199254740992.0);
  };
  auto normal = [&]() {
    double u1 = uni(), u2 = uni();
    if (u1 < 1e-300) u1 = 1e-300;
    return std::sqrt(-2. * std::log(u1)) * std::cos(6.283185307179586 * u2);
  };
  for (int i = 0; i < MLP_IN * MLP_H; i++) h[MLP_OFF_W1 + i] = (float)(normal() * std::sqrt(2. / MLP_IN));
  for (int i = 0; i < MLP_H * MLP_H; i++) h[MLP_OFF_W2 + i] = (float)(normal() * std::sqrt(2. / MLP_H));
  for (int i = 0; i < MLP_H; i++) h[MLP_OFF_W3 + i] = (float)(normal() * 0.01);
  if (ecg_mlp_set_params(M, h.data()) != ECG_OK) {
    ecg_mlp_destroy(M);
    return nullptr;
  }
  return M;
}

int ecg_mlp_destroy(ecg_mlp* M) {
  if (!M) return ECG_OK;
  if (M->attached > 0) return api_fail(ECG_E_ARG, "the network is the warm start of a solver context (detach it first)");
  if (M->stream) hipStreamSynchronize(M->stream);
  hipFree(M->prm); hipFree(M->adam_m); hipFree(M->adam_v); hipFree(M->grad);
  hipFree(M->act); hipFree(M->loss_acc); hipFree(M->frag); hipFree(M->bias);
  if (M->stream) hipStreamDestroy(M->stream);
  delete M;
  return ECG_OK;
}

static int mlp_pack(ecg_mlp* M) {
  hipLaunchKernelGGL(k_mlp_pack, dim3((MLP_NFRAG * 64 + 255) / 256), dim3(256), 0, M->stream, M->prm, M->frag, M->bias);
  HIPCHK(hipGetLastError());
  HIPCHK(hipStreamSynchronize(M->stream));
  return ECG_OK;
}

int ecg_mlp_set_params(ecg_mlp* M, const float* host) {
  if (!M || !host) return api_fail(ECG_E_ARG, "null network or parameters");
  // Step kernels of attached contexts may still read the inference fragments.
  if (M->attached > 0) HIPCHK(hipDeviceSynchronize());
  for (int i = 0; i < MLP_NPARAM; i++)
    if (!std::isfinite(host[i])) return api_fail(ECG_E_ARG, "non-finite network parameter");
  HIPCHK(hipMemcpy(M->prm, host, MLP_NPARAM * sizeof(float), hipMemcpyHostToDevice));
  HIPCHK(hipMemset(M->adam_m, 0, MLP_NPARAM * sizeof(float)));
  HIPCHK(hipMemset(M->adam_v, 0, MLP_NPARAM * sizeof(float)));
  M->adam_t = 0;
  return mlp_pack(M);
}

int ecg_mlp_get_params(ecg_mlp* M, float* host) {
  if (!M || !host) return api_fail(ECG_E_ARG, "null network or parameters");
  HIPCHK(hipStreamSynchronize(M->stream));
  HIPCHK(hipMemcpy(host, M->prm, MLP_NPARAM * sizeof(float), hipMemcpyDeviceToHost));
  return ECG_OK;
}

// Workspace of a batch of nblk chunks and of nloss loss sums.
static int ensure_workspace(ecg_mlp* M, long long nblk, int nloss) {
  const int ld = (int)((std::min<long long>(nblk, SEG_CHUNKS) + FB_SAMPLES - 1) / FB_SAMPLES * FB_SAMPLES);
  if (ld > M->act_ld) {
    HIPCHK(hipStreamSynchronize(M->stream));
    hipFree(M->act);
    M->act = nullptr;
    M->act_ld = 0;
    HIPCHK(hipMalloc(&M->act, (size_t)ACT_ROWS * TBS * ld * sizeof(float)));
    M->act_ld = ld;
  }
  if (nloss > M->loss_cap) {
    HIPCHK(hipStreamSynchronize(M->stream));
    hipFree(M->loss_acc);
    M->loss_acc = nullptr;
    M->loss_cap = 0;
    HIPCHK(hipMalloc(&M->loss_acc, (size_t)(nloss + 1) * sizeof(double)));   // the last one: a batch's running sum
    M->loss_cap = nloss;
  }
  return ECG_OK;
}

// Gradient of one batch (nblk chunks) into M->grad, or with adam the optimiser step on it;
// the batch's loss sum is added to loss sum `e` (set, when loss_first).
static int launch_batch(ecg_mlp* M, const ecg_samples* S, long long n, long long q0, long long count,
                        unsigned long long mult, unsigned long long offs, unsigned long long perm_seed,
                        float inv_batch, long long nblk, bool adam, float lr_t, int e, bool loss_first) {
  for (long long c0 = 0; c0 < nblk; c0 += SEG_CHUNKS) {
    const int nc = (int)std::min<long long>(nblk - c0, SEG_CHUNKS);
    hipLaunchKernelGGL(k_mlp_fwd_bwd, dim3(TBS * ((nc + FB_SAMPLES - 1) / FB_SAMPLES)), dim3(256), 0, M->stream, M->prm,
                       S->buf, n, q0, count, mult, offs, perm_seed, inv_batch, c0, nc, M->act_ld, M->act);
    hipLaunchKernelGGL(k_mlp_grad, dim3(GR_BLOCKS), dim3(64), 0, M->stream, M->act, nc, M->act_ld, c0 == 0 ? 1 : 0,
                       c0 + nc >= nblk ? 1 : 0, M->grad, adam ? M->adam_m : (float*)nullptr, M->adam_v, M->prm, lr_t,
                       M->loss_acc + M->loss_cap, M->loss_acc + e, loss_first ? 1 : 0);
  }
  HIPCHK(hipGetLastError());
  return ECG_OK;
}

int ecg_mlp_gradient(ecg_mlp* M, ecg_samples* S, int64_t n, float* grad, double* loss) {
  if (!M || !S || !grad || n <= 0) return api_fail(ECG_E_ARG, "invalid gradient arguments");
  const long long have = samples_count(S);
  if (have < 0) return api_fail(ECG_E_HIP, "reading the sample counter failed");
  if (n > have) return api_fail(ECG_E_ARG, "more records requested than the buffer holds");
  const long long nblk = (n + TBS - 1) / TBS;
  int rc = ensure_workspace(M, nblk, 1);
  if (rc != ECG_OK) return rc;
  rc = launch_batch(M, S, n, 0, n, 1ull, 0ull, 0ull, 1.f / (float)n, nblk, false, 0.f, 0, true);
  if (rc != ECG_OK) return rc;
  double acc = 0.;
  HIPCHK(hipMemcpyAsync(grad, M->grad, MLP_NPARAM * sizeof(float), hipMemcpyDeviceToHost, M->stream));
  HIPCHK(hipMemcpyAsync(&acc, M->loss_acc, sizeof(double), hipMemcpyDeviceToHost, M->stream));
  HIPCHK(hipStreamSynchronize(M->stream));
  if (loss) *loss = acc / (double)n;
  return ECG_OK;
}

static unsigned long long gcd_u(unsigned long long a, unsigned long long b) {
  while (b) { const unsigned long long t = a % b; a = b; b = t; }
  return a;
}

int ecg_mlp_train(ecg_mlp* M, ecg_samples* S, int epochs, int batch, float lr, uint64_t seed, double* epoch_loss) {
  if (!M || !S || epochs <= 0 || batch < TBS || !(lr > 0.f)) return api_fail(ECG_E_ARG, "invalid training arguments");
  batch = batch / TBS * TBS;
  const long long n = samples_count(S);
  if (n < 0) return api_fail(ECG_E_HIP, "reading the sample counter failed");
  if (n < batch) return api_fail(ECG_E_ARG, "fewer samples than one batch");
  if (n >= (1ll << 31)) return api_fail(ECG_E_ARG, "at most 2^31 samples per training call");
  if (M->attached > 0) HIPCHK(hipDeviceSynchronize());
  const int nblk = batch / TBS;
  int rc = ensure_workspace(M, nblk, epochs);
  if (rc != ECG_OK) return rc;
  const long long nb = n / batch;
  // Multipliers of the per-epoch affine permutation of the sample order (coprime with n).
  static const unsigned long long primes[] = {1000003ull, 2000003ull, 3000017ull, 4000037ull, 5000011ull,
                                              6000011ull, 7000003ull, 8000009ull, 9000011ull, 10000019ull};
  for (int e = 0; e < epochs; e++) {
    unsigned long long mult = 1ull;
    for (int q = 0; q < 10; q++) {
      const unsigned long long cand = primes[(q + e + seed) % 10];
      if (gcd_u(cand, (unsigned long long)n) == 1ull) { mult = cand; break; }
    }
    unsigned long long z = seed * 0x9E3779B97F4A7C15ull + (unsigned long long)e * 0xD1B54A32D192ED03ull + 1ull;
    z = (z ^ (z >> 31)) * 0xBF58476D1CE4E5B9ull;
    const unsigned long long offs = (z ^ (z >> 29)) % (unsigned long long)n;
    for (long long b = 0; b < nb; b++) {
      M->adam_t++;
      const double bc1 = 1. - std::pow(0.9, (double)M->adam_t);
      const double bc2 = 1. - std::pow(0.999, (double)M->adam_t);
      const float lr_t = (float)(lr * std::sqrt(bc2) / bc1);
      rc = launch_batch(M, S, n, b * batch, batch, mult, offs, z | 1ull, 1.f / (float)batch, nblk, true, lr_t, e, b == 0);
      if (rc != ECG_OK) return rc;
    }
  }
  std::vector<double> acc((size_t)epochs);
  HIPCHK(hipMemcpyAsync(acc.data(), M->loss_acc, sizeof(double) * epochs, hipMemcpyDeviceToHost, M->stream));
  HIPCHK(hipStreamSynchronize(M->stream));
  for (int e = 0; e < epochs && epoch_loss; e++) epoch_loss[e] = acc[e] / (double)(nb * batch);
  return mlp_pack(M);
}

int ecg_mlp_predict(ecg_mlp* M, ecg_samples* S, int64_t n, float* out) {
  if (!M || !S || !out || n <= 0) return api_fail(ECG_E_ARG, "invalid prediction arguments");
  const long long have = samples_count(S);
  if (have < 0) return api_fail(ECG_E_HIP, "reading the sample counter failed");
  if (n > have) return api_fail(ECG_E_ARG, "more records requested than the buffer holds");
  float* d = nullptr;
  HIPCHK(hipMalloc(&d, (size_t)n * sizeof(float)));
  MlpDev md;
  md.frag = M->frag;
  md.bias = M->bias;
  hipLaunchKernelGGL(k_mlp_predict, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, M->stream, md, S->buf, (long long)n, d);
  hipError_t e1 = hipGetLastError();
  hipError_t e2 = hipMemcpyAsync(out, d, (size_t)n * sizeof(float), hipMemcpyDeviceToHost, M->stream);
  hipError_t e3 = hipStreamSynchronize(M->stream);
  hipFree(d);
  if (e1 != hipSuccess || e2 != hipSuccess || e3 != hipSuccess) return api_fail(ECG_E_HIP, "network inference failed");
  return ECG_OK;
}

}  // extern "C"
