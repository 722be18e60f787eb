// MLP building blocks on CDNA4 matrix cores (v_mfma_f32_32x32x16_bf16), shared by the surrogate training kernels
// and the batched material kernels.
//
// Layout ("transposed" formulation): an MFMA tile is 32 samples wide. A layer computes Z = W H + b with the weights as the MFMA
// A operand (32 output features x 16 inputs per instruction) and the activations as the B operand (16 inputs x 32 samples).
// Measured operand layouts on gfx950 (lane l, element i; h = l / 32):
//   A[m = l % 32][k = 8 h + i],  B[k = 8 h + i][n = l % 32],  D register j: [m = 8 (j / 4) + 4 h + j % 4][n = l % 32].
// A 32-feature output tile in D layout is, after bias + GELU + conversion to BF16, already the B operand of the next
// layer for two 16-input blocks, provided the next layer's weight columns are stored in the matching order: input block
// kb = 2 t + s, lane half h, element i holds hidden feature
//   perm(kb, h, i) = 32 t + 16 s + 8 (i / 4) + 4 h + i % 4.
// So a wavefront's inference runs in registers, with no LDS traffic between layers (one or two tiles, mlp_hidden). Training
// gives each wavefront 32 features of a hidden layer and hands these operands round through LDS, backwards too, with W^T packed
// in the same permuted order (mlp.hip). The weight-gradient GEMM (sum over samples) uses the same instruction with samples as
// the reduction dimension.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "../../include/fecx.h"

namespace fecx {

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8;
typedef __attribute__((__vector_size__(16 * sizeof(float)))) float f32x16;

// Network shapes. D: true widths; P: padded widths (inputs to a 16-multiple, outputs to a 32-multiple).
template <int ARCH>
struct Arch;
template <>
struct Arch<FECX_MLP_J2> {
  static constexpr int NL = 4;
  static constexpr int D[5] = {13, 128, 128, 128, 13};
  static constexpr int P[5] = {16, 128, 128, 128, 32};
};
template <>
struct Arch<FECX_MLP_NH> {
  static constexpr int NL = 3;
  static constexpr int D[4] = {9, 256, 256, 15};
  static constexpr int P[4] = {16, 256, 256, 32};
};

// widest hidden layer (register arrays are sized by it)
template <class A>
constexpr int max_hidden() {
  int w = 32;
  for (int l = 1; l < A::NL; ++l) w = A::P[l] > w ? A::P[l] : w;
  return w;
}

template <class A>
struct Offs {
  // packed forward weights of layer l, in bf16x8 units: (P[l+1] / 32) x (P[l] / 16) x 64 lanes
  static constexpr int64_t wf(int l) {
    int64_t o = 0;
    for (int k = 0; k < l; ++k) o += (int64_t)(A::P[k + 1] / 32) * (A::P[k] / 16) * 64;
    return o;
  }
  // packed backward weights W_l^T (l >= 1): (P[l] / 32) x (P[l+1] / 16) x 64 lanes
  static constexpr int64_t wb(int l) {
    int64_t o = 0;
    for (int k = 1; k < l; ++k) o += (int64_t)(A::P[k] / 32) * (A::P[k + 1] / 16) * 64;
    return o;
  }
  static constexpr int bias(int l) {
    int o = 0;
    for (int k = 0; k < l; ++k) o += A::P[k + 1];
    return o;
  }
  // canonical parameters: per layer W (D[l+1] x D[l], row-major) then b (D[l+1])
  static constexpr int64_t param(int l) {
    int64_t o = 0;
    for (int k = 0; k < l; ++k) o += (int64_t)A::D[k + 1] * A::D[k] + A::D[k + 1];
    return o;
  }
  static constexpr int64_t wf_total() { return wf(A::NL); }
  static constexpr int64_t wb_total() { return wb(A::NL); }
  static constexpr int bias_total() { return bias(A::NL); }
  static constexpr int64_t params() { return param(A::NL); }
  // activation rows stored for the weight gradient: h_l for l < NL (h_0 padded to 32 rows), dz_l for 1 <= l <= NL
  static constexpr int hrows(int l) { return l == 0 ? 32 : A::P[l]; }
};

// feature held by D-layout register j of output tile mt in lane half h
__host__ __device__ constexpr int dreg_feature(int mt, int h, int j) { return 32 * mt + 8 * (j / 4) + 4 * h + j % 4; }

struct MlpDev {
  const bf16x8* wf;        // packed forward weights
  const bf16x8* wb;        // packed W^T for the backward pass
  const float* bias;       // padded biases
  const float* in_shift;   // D[0]
  const float* in_scale;
  const float* out_shift;  // D[NL]
  const float* out_scale;
};

// GELU in its tanh form, 0.5 z (1 + tanh(sqrt(2/pi) (z + 0.044715 z^3))) = z sigma(u), u = 2 sqrt(2/pi) (z + 0.044715 z^3)
// (Hendrycks & Gimpel, "Gaussian Error Linear Units"), evaluated with the hardware exp2 and reciprocal: five VALU
// operations and two transcendental ones per activation (the erf form costs several times that, and the network's
// hidden activations dominate its VALU work). exp2 overflow gives sigma = 0, the correct limit.
constexpr float GELU_U = 1.5957691216057308f;   // 2 sqrt(2 / pi)
constexpr float GELU_C = 0.044715f;
constexpr float LOG2E = 1.4426950408889634f;
// sigma(u) = 1 / (1 + 2^(-log2(e) u)) with the constants folded: -log2(e) u = z (GA + GB z^2)
constexpr float GELU_A = -LOG2E * GELU_U, GELU_B = GELU_A * GELU_C;
__device__ __forceinline__ float gelu_sigma(float z) {
  return __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(z * fmaf(GELU_B, z * z, GELU_A)));
}
__device__ __forceinline__ float gelu(float z) { return z * gelu_sigma(z); }
__device__ __forceinline__ float gelu_prime(float z) {
  const float s = gelu_sigma(z);
  const float du = GELU_U * fmaf(3.0f * GELU_C * z, z, 1.0f);
  return fmaf(z * s * (1.0f - s), du, s);
}

// Z = W_l H + b for one hidden layer and T tiles of 32 samples, with the bias, GELU and BF16 packing applied one 32-feature D
// tile at a time straight into the next layer's B operands: T D tiles (16 registers each) are live instead of P[l+1] / 2
// registers per tile of samples. Every weight operand is loaded once for the T tiles: the weights of a wavefront come from L2
// (76 KB for the J2 network, 144 KB for the neo-Hookean one, against 32 KB of L1).
template <class A, int L, int T>
__device__ __forceinline__ void mlp_layer_gelu(const MlpDev& m, const bf16x8 (&hb)[T][A::P[L] / 16],
                                               bf16x8 (&hn)[T][A::P[L + 1] / 16], int lane) {
  constexpr int IN = A::P[L], OUT = A::P[L + 1];
  const bf16x8* w = m.wf + Offs<A>::wf(L);
  const float* b = m.bias + Offs<A>::bias(L);
  const int h = lane >> 5;
#pragma unroll
  for (int mt = 0; mt < OUT / 32; ++mt) {
    f32x16 c[T];
#pragma unroll
    for (int j = 0; j < 16; ++j) {
      const float bj = b[dreg_feature(mt, h, j)];
#pragma unroll
      for (int t = 0; t < T; ++t) c[t][j] = bj;
    }
#pragma unroll
    for (int kb = 0; kb < IN / 16; ++kb) {
      const bf16x8 wv = w[(mt * (IN / 16) + kb) * 64 + lane];
#pragma unroll
      for (int t = 0; t < T; ++t) c[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wv, hb[t][kb], c[t], 0, 0, 0);
    }
#pragma unroll
    for (int t = 0; t < T; ++t)
#pragma unroll
      for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int i = 0; i < 8; ++i) hn[t][2 * mt + s][i] = (__bf16)gelu(c[t][8 * s + i]);
  }
}
// the output layer of T tiles (one D tile each)
template <class A, int T>
__device__ __forceinline__ void mlp_layer_out(const MlpDev& m, const bf16x8 (&hb)[T][A::P[A::NL - 1] / 16], f32x16 (&out)[T],
                                              int lane) {
  constexpr int L = A::NL - 1, IN = A::P[L];
  const bf16x8* w = m.wf + Offs<A>::wf(L);
  const float* b = m.bias + Offs<A>::bias(L);
  const int h = lane >> 5;
#pragma unroll
  for (int j = 0; j < 16; ++j) {
    const float bj = b[dreg_feature(0, h, j)];
#pragma unroll
    for (int t = 0; t < T; ++t) out[t][j] = bj;
  }
#pragma unroll
  for (int kb = 0; kb < IN / 16; ++kb) {
    const bf16x8 wv = w[kb * 64 + lane];
#pragma unroll
    for (int t = 0; t < T; ++t) out[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wv, hb[t][kb], out[t], 0, 0, 0);
  }
}

// all layers of T tiles, from their input operands to the output layer's D tiles
template <class A, int T>
__device__ __forceinline__ void mlp_hidden(const MlpDev& m, const bf16x8 (&h0)[T][1], f32x16 (&out)[T], int lane) {
  static_assert(A::NL == 3 || A::NL == 4, "three or four layers");
  bf16x8 h1[T][A::P[1] / 16], h2[T][A::P[2] / 16];
  mlp_layer_gelu<A, 0, T>(m, h0, h1, lane);
  mlp_layer_gelu<A, 1, T>(m, h1, h2, lane);
  if constexpr (A::NL == 3) {
    mlp_layer_out<A, T>(m, h2, out, lane);
  } else {
    bf16x8 h3[T][A::P[3] / 16];
    mlp_layer_gelu<A, 2, T>(m, h2, h3, lane);
    mlp_layer_out<A, T>(m, h3, out, lane);
  }
}

// Exchanges the upper 32 lanes of a with the lower 32 of b: {a.low, b.low} and {a.high, b.high} (v_permlane32_swap_b32).
__device__ __forceinline__ void swap_halves(uint32_t& a, uint32_t& b) {
  const auto r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
  a = r[0];
  b = r[1];
}

// Forward pass of one wavefront over 64 samples, lane = sample, as two 32-sample tiles (samples 0-31 and 32-63). xin: this
// lane's sample features, already normalized (the first D[0] of them); on return y[0 .. 16) holds this lane's normalized
// outputs. One lane per sample outside the network, so nothing around it (features, the check of the outputs, the plain
// fallback) runs twice, as it did with each sample on both lane halves of a 32-sample wavefront.
template <class A>
__device__ __forceinline__ void mlp_forward_wave(const MlpDev& m, const float* xin, float* y, int lane) {
  static_assert(A::P[0] == 16 && A::P[A::NL] == 32 && A::D[0] <= 16 && A::D[A::NL] <= 16, "one input block, half an output tile");
  // a tile's operand holds features 0-7 of its samples in the lower lanes and 8-15 in the upper ones
  union Block {
    bf16x8 v;
    uint32_t w[4];
  } t0, t1;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    t0.v[i] = (__bf16)(i < A::D[0] ? xin[i] : 0.0f);
    t1.v[i] = (__bf16)(8 + i < A::D[0] ? xin[(8 + i) % A::D[0]] : 0.0f);
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) swap_halves(t0.w[i], t1.w[i]);
  const bf16x8 h0[2][1] = {{t0.v}, {t1.v}};
  f32x16 out[2];
  mlp_hidden<A, 2>(m, h0, out, lane);
#pragma unroll
  for (int j = 0; j < 8; ++j) {  // features 0-15: lane halves 0 and 1 of the tiles' D registers
    uint32_t a = __float_as_uint(out[0][j]), b = __float_as_uint(out[1][j]);
    swap_halves(a, b);
    y[dreg_feature(0, 0, j)] = __uint_as_float(a);
    y[dreg_feature(0, 1, j)] = __uint_as_float(b);
  }
}

}  // namespace fecx
