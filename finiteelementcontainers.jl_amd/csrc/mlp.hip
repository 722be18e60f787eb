// Learned constitutive surrogate: training and batched inference kernels (BF16 MFMA, FP32 accumulation), the batched
// plain material updates they are trained on and fall back to, and training-sample generation.
//
// The reference has no surrogate and no batched material pass; its materials are evaluated inside the element loop
// (test/mechanics/TestMechanicsCommon.jl:140-222). The plain models here are the same FP32 material functions the
// element kernels use (fem_device.h), so a surrogate is checked against exactly what the plain assembly computes.
#include "fem_device.h"
#include "mlp_device.h"
#include "surrogate.h"

namespace fecx {

// ------------------------------------------------------------------ per-material feature maps
// J2: raw input {H (9, row-major displacement gradient), state (7)}, features {eps (6), plastic strain (6), eqps},
//     raw output {sigma (6), plastic strain increment (6), eqps increment}; symmetric tensors in the state order
//     (11, 21, 31, 22, 32, 33).
// NH: raw input H (9), features H, raw output {P (9, row-major), C^-1 - I (6)}.
template <int ARCH>
struct Feat;
template <>
struct Feat<FECX_MLP_J2> {
  static constexpr int IN_W = 16, NF = 13, OUT_W = 13;
  __device__ static void features(const float* raw, float* x) {
    x[0] = raw[0]; x[1] = 0.5f * (raw[3] + raw[1]); x[2] = 0.5f * (raw[6] + raw[2]);
    x[3] = raw[4]; x[4] = 0.5f * (raw[7] + raw[5]); x[5] = raw[8];
#pragma unroll
    for (int i = 0; i < 7; ++i) x[6 + i] = raw[9 + i];
  }
};
template <>
struct Feat<FECX_MLP_NH> {
  static constexpr int IN_W = 9, NF = 9, OUT_W = 15;
  __device__ static void features(const float* raw, float* x) {
#pragma unroll
    for (int i = 0; i < 9; ++i) x[i] = raw[i];
  }
};

template <int ARCH>
__device__ __forceinline__ void normalized_features(const MlpDev& m, const float* raw, float* x) {
  Feat<ARCH>::features(raw, x);
#pragma unroll
  for (int f = 0; f < Feat<ARCH>::NF; ++f) x[f] = (x[f] - m.in_shift[f]) / m.in_scale[f];
}

// ------------------------------------------------------------------ training: fused forward + backward
// One work-group per 32 TT samples, one wavefront per 32 features of the hidden layers: wavefront w computes D tile w of every
// layer for the TT sample tiles, and the activations go round through LDS as the next layer's B operands (two buffers, one
// barrier per layer). The output layer, the loss and its gradient are one wavefront's work per sample tile. Every sum has
// the order it has with one wavefront per tile.
// The weight gradients want the same numbers with the samples as the reduction index: ds_read_tr turns the 32 x 32 tiles round
// on their way out of LDS, so h and dz are stored as ready MFMA operands, one kilobyte per store.
// Bound by latency on small batches (a chain of 2 NL - 1 layers) and by the write of h and dz (2.2 KB per neo-Hookean sample) on
// large ones. With one wavefront per 32 samples doing all layers (512 wavefronts for 16,384 samples, 1.4 KB of scratch each,
// 2-byte stores, GELU' through memory) the neo-Hookean kernel took 183 us at 16,384 samples, now 17; 97 us at 100,000.
typedef short s16x4 __attribute__((__vector_size__(4 * sizeof(short))));

template <class A>
constexpr int train_waves() {
  static_assert(A::P[1] == max_hidden<A>() && A::P[2] == max_hidden<A>() && A::P[A::NL - 1] == max_hidden<A>(),
                "hidden layers of one width: one D tile per wavefront");
  return max_hidden<A>() / 32;
}

// Operand u (samples 16 u .. 16 u + 15) of one 32-feature x 32-sample tile with k = sample: lane l, element i = feature l % 32 of
// sample 16 u + 8 (l / 32) + i. `b` holds the tile's two B operands (k = feature). ds_read_tr16_b64, measured: in a group of 16
// lanes, lane p element e = element p % 4 of the 8 bytes that lane 4 e + p / 4 points at; so lane c points at sample c / 4 and
// the four features 4 (c % 4) of its group's 16. In the hidden layers' order (PERM) four features lie at block f / 16, lane
// half f / 4 % 2, half-operand f / 8 % 2; the network's inputs are in plain order and fill one block.
template <bool PERM>
__device__ __forceinline__ bf16x8 transposed_operand(const bf16x8 (*b)[64], int u, int lane) {
  union {
    bf16x8 v;
    s16x4 q[2];
  } o;
  const int c4 = lane % 4, fh = lane / 16 % 2;
  const int kb = PERM ? fh : 0, hh = PERM ? c4 % 2 : c4 / 2, half = PERM ? c4 / 2 : c4 % 2;
#pragma unroll
  for (int r = 0; r < 2; ++r) {
    const int smp = 16 * u + 8 * (lane / 32) + 4 * r + lane % 16 / 4;
    const __bf16* p = reinterpret_cast<const __bf16*>(&b[kb][hh * 32 + smp]) + 4 * half;
    o.q[r] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)p);
  }
  return o.v;
}

template <int ARCH, int TT>
__global__ __launch_bounds__(train_waves<Arch<ARCH>>() * 64) void mlp_train_kernel(TrainArgs a) {
  using A = Arch<ARCH>;
  using O = Offs<A>;
  constexpr int NL = A::NL, DOUT = A::D[NL], W = max_hidden<A>(), NW = train_waves<A>();
  static_assert(TT <= NW, "one wavefront per sample tile at the ends");
  __shared__ bf16x8 act[2][TT][W / 16][64];
  const int lane = threadIdx.x % 64, h = lane >> 5;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
  const int64_t tile0 = (int64_t)blockIdx.x * TT;
  const int64_t nsb = a.npad / 16;  // operands (16 samples each) per 32 features
  const int64_t s = (tile0 + wv) * 32 + lane % 32;  // this wavefront's samples at the ends (wv < TT)
  const bool valid = wv < TT && s < a.n;
  const int64_t row = valid ? (a.idx ? (int64_t)a.idx[s] : s) : 0;
  bf16x8* hbuf = reinterpret_cast<bf16x8*>(a.hbuf);
  bf16x8* dzbuf = reinterpret_cast<bf16x8*>(a.dzbuf);
  if (wv < TT) {
    float raw[Feat<ARCH>::IN_W], x[16];
#pragma unroll
    for (int i = 0; i < Feat<ARCH>::IN_W; ++i) raw[i] = valid ? a.X[row * Feat<ARCH>::IN_W + i] : 0.0f;
    normalized_features<ARCH>(a.m, raw, x);
    bf16x8 v;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float v0 = i < A::D[0] ? x[i] : 0.0f;
      const float v1 = 8 + i < A::D[0] ? x[(8 + i) % A::D[0]] : 0.0f;
      v[i] = (__bf16)(valid ? (h ? v1 : v0) : 0.0f);
    }
    act[0][wv][0][lane] = v;
  }
  f32x16 acc[TT];
  bf16x8 gp[NL - 1][TT][2];  // GELU'(z) of this wavefront's features
  int p = 0;                 // buffer of the current layer's inputs
  int64_t ho = 0;            // operands of the layers before
  // the inputs of layer L, from buffer p; the weights are on their way before the barrier
  auto layer = [&](auto LC) {
    constexpr int L = decltype(LC)::value, IN = A::P[L];
    const int mt = L == NL - 1 ? 0 : wv;
    const bf16x8* w = a.m.wf + O::wf(L) + (int64_t)mt * (IN / 16) * 64 + lane;
    const float* b = a.m.bias + O::bias(L);
    bf16x8 wr[IN / 16];
    if (L < NL - 1 || wv < TT) {
#pragma unroll
      for (int kb = 0; kb < IN / 16; ++kb) wr[kb] = w[kb * 64];
    }
    __syncthreads();
    if constexpr (L == 0) {  // h_0: rows 16 .. 31 are zero
      if (wv < TT) {
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          const bf16x8 v = transposed_operand<false>(act[0][wv], u, lane), z = {};
          hbuf[((tile0 + wv) * 2 + u) * 64 + lane] = lane / 16 % 2 ? z : v;
        }
      }
      ho += nsb * 64;
    } else {
#pragma unroll
      for (int t = 0; t < TT; ++t)
#pragma unroll
        for (int u = 0; u < 2; ++u)
          hbuf[ho + (wv * nsb + (tile0 + t) * 2 + u) * 64 + lane] = transposed_operand<true>(&act[p][t][2 * wv], u, lane);
      ho += NW * nsb * 64;
    }
    if constexpr (L < NL - 1) {
#pragma unroll
      for (int j = 0; j < 16; ++j) {
        const float bj = b[dreg_feature(mt, h, j)];
#pragma unroll
        for (int t = 0; t < TT; ++t) acc[t][j] = bj;
      }
#pragma unroll
      for (int kb = 0; kb < IN / 16; ++kb)
#pragma unroll
        for (int t = 0; t < TT; ++t)
          acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wr[kb], act[p][t][kb][lane], acc[t], 0, 0, 0);
      p ^= 1;
#pragma unroll
      for (int t = 0; t < TT; ++t)
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          bf16x8 v;
#pragma unroll
          for (int i = 0; i < 8; ++i) {
            const float z = acc[t][8 * u + i];
            gp[L][t][u][i] = (__bf16)gelu_prime(z);
            v[i] = (__bf16)gelu(z);
          }
          act[p][t][2 * wv + u][lane] = v;
        }
    } else if (wv < TT) {
#pragma unroll
      for (int j = 0; j < 16; ++j) acc[0][j] = b[dreg_feature(0, h, j)];
#pragma unroll
      for (int kb = 0; kb < IN / 16; ++kb)
        acc[0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wr[kb], act[p][wv][kb][lane], acc[0], 0, 0, 0);
    }
  };
  layer(std::integral_constant<int, 0>());
  layer(std::integral_constant<int, 1>());
  if constexpr (NL >= 3) layer(std::integral_constant<int, 2>());
  if constexpr (NL >= 4) layer(std::integral_constant<int, 3>());
  // loss and output gradient, dz_NL = 2 (y - t) / (n * DOUT)
  int64_t dzo = (int64_t)(NL - 1) * NW * nsb * 64;
  p ^= 1;
  if (wv < TT) {
    const float gscale = 2.0f / (float)((double)a.n * DOUT);
    double lsum = 0.0;
#pragma unroll
    for (int j = 0; j < 16; ++j) {
      const int o = dreg_feature(0, h, j);
      float dy = 0.0f;
      if (valid && o < DOUT) {
        const float t = (a.T[row * DOUT + o] - a.m.out_shift[o]) / a.m.out_scale[o];
        const float d = acc[0][j] - t;
        lsum += (double)d * d;
        dy = gscale * d;
      }
      act[p][wv][j / 8][lane][j % 8] = (__bf16)dy;
    }
    // wave sum of the loss, in a fixed order
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) lsum += __shfl_xor(lsum, off);
    if (lane == 0) a.loss_part[tile0 + wv] = lsum / ((double)a.n * DOUT);
  }
  // dh_L = W_L^T dz_{L+1}; dz_L = dh_L * GELU'(z_L)
  auto back = [&](auto LC) {
    constexpr int L = decltype(LC)::value, IN = A::P[L + 1];
    const bf16x8* w = a.m.wb + O::wb(L) + (int64_t)wv * (IN / 16) * 64 + lane;
    bf16x8 wr[IN / 16];
#pragma unroll
    for (int kb = 0; kb < IN / 16; ++kb) wr[kb] = w[kb * 64];
    __syncthreads();
    if constexpr (L == NL - 1) {
      if (wv < TT) {
#pragma unroll
        for (int u = 0; u < 2; ++u)
          dzbuf[dzo + ((tile0 + wv) * 2 + u) * 64 + lane] = transposed_operand<true>(&act[p][wv][0], u, lane);
      }
    }
#pragma unroll
    for (int t = 0; t < TT; ++t) acc[t] = f32x16{};
#pragma unroll
    for (int kb = 0; kb < IN / 16; ++kb)
#pragma unroll
      for (int t = 0; t < TT; ++t)
        acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wr[kb], act[p][t][kb][lane], acc[t], 0, 0, 0);
    p ^= 1;
#pragma unroll
    for (int t = 0; t < TT; ++t)
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        bf16x8 v;
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = (__bf16)(acc[t][8 * u + i] * (float)gp[L - 1][t][u][i]);
        act[p][t][2 * wv + u][lane] = v;
      }
    dzo -= (int64_t)NW * nsb * 64;
#pragma unroll
    for (int t = 0; t < TT; ++t)
#pragma unroll
      for (int u = 0; u < 2; ++u)  // this wavefront's own part of the buffer
        dzbuf[dzo + (wv * nsb + (tile0 + t) * 2 + u) * 64 + lane] = transposed_operand<true>(&act[p][t][2 * wv], u, lane);
  };
  if constexpr (NL >= 4) back(std::integral_constant<int, 3>());
  if constexpr (NL >= 3) back(std::integral_constant<int, 2>());
  back(std::integral_constant<int, 1>());
}

// ------------------------------------------------------------------ training: weight gradients (MFMA over samples)
// One wavefront per (layer, up to 2 x 2 weight tiles of 32 x 32, chunk of samples): dW[o][i] = sum_s dz_{l+1}[o][s] h_l[i][s] with
// samples as the MFMA reduction dimension and the operands as the training kernel stored them; the blocks of the first inputs
// also sum dz rows for the bias gradient. Partial sums per chunk go to part[chunk][param]; the reduction over chunks runs in a
// fixed order (mlp_update_kernel). The blocks of one chunk are launched eight apart, so that one XCD's L2 serves all of them.
// Bound by the read of h and dz: neo-Hookean 16,384 samples 31 us with single tiles and 32-byte pieces of feature-major rows,
// now 11; 100,000 (218 MB) 60 us.
template <class A, int L>
struct WGradShape {
  static constexpr int NOT = A::P[L + 1] / 32, NIT = Offs<A>::hrows(L) / 32;
  static constexpr int MB = NOT > 1 ? 2 : 1, NB = NIT > 1 ? 2 : 1;
  static constexpr int BLOCKS = (NOT / MB) * (NIT / NB);
};
template <int ARCH>
__global__ __launch_bounds__(64) void mlp_wgrad_kernel(WGradArgs a) {
  using A = Arch<ARCH>;
  using O = Offs<A>;
  constexpr int NL = A::NL;
  const int lane = threadIdx.x, h = lane >> 5;
  int t = blockIdx.x / 8 % a.nblocks;
  const int chunk = blockIdx.x / (8 * a.nblocks) * 8 + blockIdx.x % 8;
  if (chunk >= a.nchunk) return;
  const int64_t nsb = a.npad / 16;
  const int64_t k0 = (int64_t)chunk * (a.chunk_len / 16), k1 = min(k0 + a.chunk_len / 16, nsb);
  int64_t ho = 0, dzo = 0;
  auto tile = [&](auto LC) {
    constexpr int L = decltype(LC)::value;
    using S = WGradShape<A, L>;
    constexpr int MB = S::MB, NB = S::NB;
    if (t < 0) return;
    if (t >= S::BLOCKS) {
      t -= S::BLOCKS;
      ho += (int64_t)S::NIT * nsb * 64;
      dzo += (int64_t)S::NOT * nsb * 64;
      return;
    }
    const int ot = t / (S::NIT / NB) * MB, it = t % (S::NIT / NB) * NB;
    t = -1;
    const bf16x8* dz = reinterpret_cast<const bf16x8*>(a.dzbuf) + dzo + ot * nsb * 64 + lane;
    const bf16x8* hl = reinterpret_cast<const bf16x8*>(a.hbuf) + ho + it * nsb * 64 + lane;
    f32x16 c[MB][NB] = {};
    float bsum[MB] = {};
    for (int64_t k = k0; k < k1; k += 4) {  // samples are padded to 64
      bf16x8 av[4][MB], bv[4][NB];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
#pragma unroll
        for (int m = 0; m < MB; ++m) av[u][m] = dz[(m * nsb + k + u) * 64];
#pragma unroll
        for (int n = 0; n < NB; ++n) bv[u][n] = hl[(n * nsb + k + u) * 64];
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) {
#pragma unroll
        for (int m = 0; m < MB; ++m)
#pragma unroll
          for (int n = 0; n < NB; ++n) c[m][n] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(av[u][m], bv[u][n], c[m][n], 0, 0, 0);
        if (it == 0) {
#pragma unroll
          for (int m = 0; m < MB; ++m)
#pragma unroll
            for (int e = 0; e < 8; ++e) bsum[m] += (float)av[u][m][e];
        }
      }
    }
    float* part = a.part + (int64_t)chunk * O::params() + O::param(L);
#pragma unroll
    for (int m = 0; m < MB; ++m)
#pragma unroll
      for (int n = 0; n < NB; ++n) {
        const int i = (it + n) * 32 + lane % 32;
#pragma unroll
        for (int j = 0; j < 16; ++j) {
          const int o = dreg_feature(ot + m, h, j);
          if (o < A::D[L + 1] && i < A::D[L]) part[(int64_t)o * A::D[L] + i] = c[m][n][j];
        }
      }
    if (it == 0) {
#pragma unroll
      for (int m = 0; m < MB; ++m) {
        bsum[m] += __shfl_xor(bsum[m], 32);
        const int o = (ot + m) * 32 + lane % 32;
        if (h == 0 && o < A::D[L + 1]) part[(int64_t)A::D[L + 1] * A::D[L] + o] = bsum[m];
      }
    }
  };
  tile(std::integral_constant<int, 0>());
  tile(std::integral_constant<int, 1>());
  if constexpr (NL >= 3) tile(std::integral_constant<int, 2>());
  if constexpr (NL >= 4) tile(std::integral_constant<int, 3>());
}

template <int ARCH>
int wgrad_blocks() {
  using A = Arch<ARCH>;
  int n = WGradShape<A, 0>::BLOCKS + WGradShape<A, 1>::BLOCKS + WGradShape<A, 2>::BLOCKS;
  if constexpr (A::NL >= 4) n += WGradShape<A, 3>::BLOCKS;
  return n;
}

// ------------------------------------------------------------------ parameter update and repacking
// Writes canonical parameter p into the packed forward / backward weights or the padded biases.
template <int ARCH>
__device__ void repack_param(const MlpPack& pk, int64_t p, float w) {
  using A = Arch<ARCH>;
  using O = Offs<A>;
  int L = 0;
  while (L + 1 < A::NL && p >= O::param(L + 1)) ++L;
  int64_t q = p - O::param(L);
  const int din = A::D[L], dout = A::D[L + 1];
  __bf16* wf = reinterpret_cast<__bf16*>(pk.wf);
  __bf16* wb = reinterpret_cast<__bf16*>(pk.wb);
  if (q < (int64_t)dout * din) {
    const int o = (int)(q / din), i = (int)(q % din);
    // forward: A operand row o, input i
    int kb, hh, e;
    if (L == 0) { kb = i / 16; hh = (i % 16) / 8; e = i % 8; }
    else { const int t = i / 32, r = i % 32, sgn = r / 16, rem = r % 16; kb = 2 * t + sgn; e = 4 * (rem / 8) + rem % 4; hh = (rem % 8) / 4; }
    const int64_t vf = O::wf(L) + ((int64_t)(o / 32) * (A::P[L] / 16) + kb) * 64 + hh * 32 + o % 32;
    wf[vf * 8 + e] = (__bf16)w;
    if (L >= 1) {  // backward: W^T row i, input o (permuted order of layer L's outputs)
      const int t = o / 32, r = o % 32, sgn = r / 16, rem = r % 16;
      const int kb2 = 2 * t + sgn, e2 = 4 * (rem / 8) + rem % 4, h2 = (rem % 8) / 4;
      const int64_t vb = O::wb(L) + ((int64_t)(i / 32) * (A::P[L + 1] / 16) + kb2) * 64 + h2 * 32 + i % 32;
      wb[vb * 8 + e2] = (__bf16)w;
    }
  } else {
    pk.bias[O::bias(L) + (q - (int64_t)dout * din)] = w;
  }
}

// The last work-group sums the n loss partials by one wavefront in a fixed order (lane l takes partials l, l + 64, ..., then a
// fixed xor tree across lanes), so every run gives the same bits. The chunks of a parameter are added in a fixed order too, by
// eights whose loads are on their way together (64 chunks of the neo-Hookean network: 14 us one load at a time, now 5) and
// whose sum is a tree: 64 rounded additions one after the other are 1.2e-7 off the exact sum, these 4.9e-8 (4,096 samples,
// relative 2-norm; 16 chunks of 256 samples one after the other were 6.8e-8 off).
template <int ARCH>
__global__ void mlp_update_kernel(UpdateArgs a) {
  if (a.loss && blockIdx.x == gridDim.x - 1) {
    if (threadIdx.x >= 64) return;
    double s = 0.0;
    for (int64_t i = threadIdx.x; i < a.nloss; i += 64) s += a.loss_part[i];
    for (int off = 32; off >= 1; off >>= 1) s += __shfl_xor(s, off);
    if (threadIdx.x == 0) a.loss[0] = s;
    return;
  }
  const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= a.np) return;
  float w = a.w[p];
  if (a.part) {
    float g = 0.0f;
    int c = 0;
    for (; c + 8 <= a.nchunk; c += 8) {
      float v[8];
#pragma unroll
      for (int k = 0; k < 8; ++k) v[k] = a.part[(int64_t)(c + k) * a.np + p];
      g += ((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7]));
    }
    for (; c < a.nchunk; ++c) g += a.part[(int64_t)c * a.np + p];
    if (a.grad) a.grad[p] = g;
    if (a.adam) {
      const float m1 = a.b1 * a.m1[p] + (1.0f - a.b1) * g;
      const float m2 = a.b2 * a.m2[p] + (1.0f - a.b2) * g * g;
      a.m1[p] = m1;
      a.m2[p] = m2;
      w -= a.lr * (m1 * a.c1) / (sqrtf(m2 * a.c2) + a.eps);
      a.w[p] = w;
    }
  }
  if (a.repack) repack_param<ARCH>(a.pk, p, w);
}

__global__ void gather_rows_kernel(int64_t n, int w, const int32_t* idx, const float* src, float* dst) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n * w) dst[i] = src[(int64_t)idx[i / w] * w + i % w];
}

// ------------------------------------------------------------------ plain material models on one sample
// J2 raw in {H (9), state (7)} -> raw out {sigma (6), dplastic (6), deqps}, plus P (9), state_new (7), C (9)
__device__ __forceinline__ void j2_plain(const MatParams& mp, const float* H, const float* so, float* y, float* P,
                                         float* sn, float* C) {
  j2_update(mp.p, H, so, sn, P, C);
  y[0] = P[0]; y[1] = P[3]; y[2] = P[6]; y[3] = P[4]; y[4] = P[7]; y[5] = P[8];
#pragma unroll
  for (int i = 0; i < 7; ++i) y[6 + i] = sn[i] - so[i];
}

// NH raw in H (9) -> raw out {P (9), C^-1 - I (6)}, plus C = {F^-T (9), mu - lambda ln J}
__device__ __forceinline__ void nh_plain(const MatParams& mp, const float* H, float* y, float* P, float* C, bool& bad) {
  Mat<FECX_NEOHOOKEAN>::eval<3>(mp, H, nullptr, nullptr, P, C, bad);
#pragma unroll
  for (int i = 0; i < 9; ++i) y[i] = P[i];
  // C^-1 = F^-1 F^-T, F^-T row-major in C[0..9)
  float Ci[9];
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int j = 0; j < 3; ++j) Ci[i * 3 + j] = C[0 * 3 + i] * C[0 * 3 + j] + C[1 * 3 + i] * C[1 * 3 + j] + C[2 * 3 + i] * C[2 * 3 + j];
  y[9] = Ci[0] - 1.0f; y[10] = Ci[3]; y[11] = Ci[6]; y[12] = Ci[4] - 1.0f; y[13] = Ci[7]; y[14] = Ci[8] - 1.0f;
}

// ------------------------------------------------------------------ surrogate decode + residual check
// Whether all N outputs are finite: a maximum drops NaN, so the deviations below cannot tell. 0 y is NaN unless y is finite.
template <int N>
__device__ __forceinline__ bool all_finite(const float* y) {
  float z = 0.0f;
#pragma unroll
  for (int o = 0; o < N; ++o) z = fmaf(y[o], 0.0f, z);
  return z == 0.0f;
}

// J2: the network's {sigma, dplastic, deqps} is accepted when it satisfies the return-mapping equations to `tol`:
//   elastic law   |sigma - (kappa tr(eps - ep_new) I + 2 mu dev(eps - ep_new))| <= tol sigma_y
//   yield         |f| <= tol sigma_y when deqps > 0 (on the yield surface), f <= tol sigma_y otherwise
//   flow          |dplastic - sqrt(3/2) deqps n| <= tol sigma_y / (2 mu), deqps >= -tol sigma_y / (2 mu)
// and all of it is finite. The tangent data follow from the closed-form consistent tangent at the network's plastic multiplier.
__device__ __forceinline__ bool j2_surrogate(const MatParams& mp, const float* H, const float* so, const float* y,
                                             float tol, float* P, float* sn, float* C) {
  const float E = mp.p[0], nu = mp.p[1], sy = mp.p[2], Hh = mp.p[3];
  const float mu = E / (2 * (1 + nu)), kap = E / (3 * (1 - 2 * nu));
  const float r23 = 0.81649658092772603f, r32 = 1.2247448713915890f;
  const float eref = sy / (2 * mu);
  auto sym = [](const float* v, float* M) {  // state order -> row-major
    M[0] = v[0]; M[1] = v[1]; M[2] = v[2]; M[3] = v[1]; M[4] = v[3]; M[5] = v[4]; M[6] = v[2]; M[7] = v[4]; M[8] = v[5];
  };
  float sig[9], dep[9], epo[9], eps[9];
  sym(y, sig);
  sym(y + 6, dep);
  sym(so, epo);
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int j = 0; j < 3; ++j) eps[i * 3 + j] = 0.5f * (H[i * 3 + j] + H[j * 3 + i]);
  const float dal = y[12];
  // elastic law
  float ee[9];
#pragma unroll
  for (int i = 0; i < 9; ++i) ee[i] = eps[i] - epo[i] - dep[i];
  const float tre = ee[0] + ee[4] + ee[8];
  float r = 0.0f;  // the largest deviation, divided once (division by a positive number keeps the order, rounding included)
#pragma unroll
  for (int i = 0; i < 9; ++i) {
    const float se = 2 * mu * ee[i] + ((i % 4 == 0) ? (kap - 2 * mu / 3) * tre : 0.0f);
    r = fmaxf(r, fabsf(sig[i] - se));
  }
  // yield
  const float trs = (sig[0] + sig[4] + sig[8]) / 3;
  float s[9], sn2 = 0.0f;
#pragma unroll
  for (int i = 0; i < 9; ++i) { s[i] = sig[i] - ((i % 4 == 0) ? trs : 0.0f); sn2 += s[i] * s[i]; }
  const float snorm = sqrtf(sn2);
  const float f = snorm - r23 * (sy + Hh * (so[6] + dal));
  const bool plastic = dal > tol * eref;
  r = fmaxf(0.0f, fmaxf(r, plastic ? fabsf(f) : fmaxf(f, 0.0f)) / sy);
  // flow rule
  const float inv = snorm > 0.0f ? 1.0f / snorm : 0.0f;
  float rf = fmaxf(-dal, 0.0f);
#pragma unroll
  for (int i = 0; i < 9; ++i) rf = fmaxf(rf, fabsf(dep[i] - r32 * fmaxf(dal, 0.0f) * s[i] * inv));
  r = fmaxf(r, rf / eref);
  if (!(r <= tol) || !all_finite<13>(y)) return false;
#pragma unroll
  for (int i = 0; i < 9; ++i) P[i] = sig[i];
#pragma unroll
  for (int i = 0; i < 6; ++i) sn[i] = so[i] + y[6 + i];
  sn[6] = so[6] + y[12];
  // tangent from the trial state and the network's multiplier
  float st[9], stn2 = 0.0f;
  const float trt = (eps[0] - epo[0]) + (eps[4] - epo[4]) + (eps[8] - epo[8]);
#pragma unroll
  for (int i = 0; i < 9; ++i) { st[i] = 2 * mu * (eps[i] - epo[i] - ((i % 4 == 0) ? trt / 3 : 0.0f)); stn2 += st[i] * st[i]; }
  const float stn = sqrtf(stn2);
  const float dg = plastic ? r32 * dal : 0.0f;
  const float th = (plastic && stn > 0.0f) ? 1.0f - 2 * mu * dg / stn : 1.0f;
  const float thb = plastic ? 1.0f / (1.0f + Hh / (3 * mu)) - (1.0f - th) : 0.0f;
  const float ti = stn > 0.0f ? 1.0f / stn : 0.0f;
  C[0] = st[0] * ti; C[1] = st[4] * ti; C[2] = st[8] * ti; C[3] = st[1] * ti; C[4] = st[5] * ti; C[5] = st[2] * ti;
  C[6] = kap - 2 * mu * th / 3; C[7] = mu * th; C[8] = 2 * mu * thb;
  return true;
}

// NH: the network's {P, C^-1 - I} is accepted when C C^-1 = I to `tol` and P agrees to `tol` with the stress the
// predicted C^-1 implies, P(F, C^-1) = mu (F - F C^-1) + lambda ln J F C^-1 (F^-T = F C^-1), relative to the stress
// scale (mu + lambda) max(|H|, 0.01), and all of it is finite.
__device__ __forceinline__ bool nh_surrogate(const MatParams& mp, const float* H, const float* y, float tol, float* P,
                                             float* C) {
  const float lam = mp.p[0], mu = mp.p[1];
  const float F[9] = {1 + H[0], H[1], H[2], H[3], 1 + H[4], H[5], H[6], H[7], 1 + H[8]};
  const float Ci[9] = {1 + y[9], y[10], y[11], y[10], 1 + y[12], y[13], y[11], y[13], 1 + y[14]};
  float r = 0.0f, hmax = 0.01f;
#pragma unroll
  for (int i = 0; i < 9; ++i) hmax = fmaxf(hmax, fabsf(H[i]));
  // C C^-1 - I with C = F^T F
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      float v = 0.0f;
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        const float Cik = F[0 * 3 + i] * F[0 * 3 + k] + F[1 * 3 + i] * F[1 * 3 + k] + F[2 * 3 + i] * F[2 * 3 + k];
        v += Cik * Ci[k * 3 + j];
      }
      r = fmaxf(r, fabsf(v - (i == j ? 1.0f : 0.0f)));
    }
  const float tr = H[0] + H[4] + H[8];
  const float trH2 = H[0] * H[0] + H[4] * H[4] + H[8] * H[8] + 2.0f * (H[1] * H[3] + H[2] * H[6] + H[5] * H[7]);
  const float detH = H[0] * (H[4] * H[8] - H[5] * H[7]) - H[1] * (H[3] * H[8] - H[5] * H[6]) + H[2] * (H[3] * H[7] - H[4] * H[6]);
  const float Jm1 = tr + 0.5f * (tr * tr - trH2) + detH;
  if (!(Jm1 > -1.0f)) return false;
  const float lnJ = log1pf(Jm1);
  float FiT[9];
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int j = 0; j < 3; ++j) FiT[i * 3 + j] = F[i * 3 + 0] * Ci[0 * 3 + j] + F[i * 3 + 1] * Ci[1 * 3 + j] + F[i * 3 + 2] * Ci[2 * 3 + j];
  const float ps = (mu + lam) * hmax;
  float rp = 0.0f;
#pragma unroll
  for (int i = 0; i < 9; ++i) {
    const float pp = mu * (F[i] - FiT[i]) + lam * lnJ * FiT[i];
    rp = fmaxf(rp, fabsf(y[i] - pp));
  }
  r = fmaxf(r, rp / ps);
  if (!(r <= tol) || !all_finite<15>(y)) return false;
#pragma unroll
  for (int i = 0; i < 9; ++i) { P[i] = y[i]; C[i] = FiT[i]; }
  C[9] = mu - lam * lnJ;
  return true;
}

// ------------------------------------------------------------------ batched material update
// One wavefront per 64 samples, lane = sample: features, residual check, decode and stores are done once per sample, and the
// network runs two 32-sample tiles at a time (mlp_forward_wave). Bound by VALU: a hidden activation costs five VALU operations,
// two transcendental ones (quarter rate) and half a conversion, so 2,097,152 J2 samples with 384 each need about 0.4 ms, and
// their 245 MB in and out 0.06 ms. With one 32-sample tile per wavefront, both lane halves doing the same check and every weight
// operand loaded per tile: J2 2,097,152 samples 888 us, now 457; neo-Hookean 2,000,000 873 -> 533, 70,000 85 -> 72; J2 5,000
// 46 -> 41. Sources and sinks:
//   batch mode    : in (n x IN_W raw) -> out (n x OUT_W raw)
//   assembly mode : hq (n x 9 quadrature-point gradients, n = ne x nq in element storage order) and the element's
//                   state (via eperm) -> qpmat (n x (9 + NC): P, compact tangent) and state_new
template <int ARCH, bool SURR>
__global__ __launch_bounds__(256) void material_kernel(MatBatchArgs a) {
  using A = Arch<ARCH>;
  using FT = Feat<ARCH>;
  constexpr bool J2 = ARCH == FECX_MLP_J2;
  constexpr int NC = J2 ? Mat<FECX_J2>::NC : Mat<FECX_NEOHOOKEAN>::NC;
  const int lane = threadIdx.x % 64;
  const int64_t tile = (int64_t)blockIdx.x * 4 + threadIdx.x / 64;
  const int64_t i = tile * 64 + lane;
  if (tile * 64 >= a.n) return;  // wave-uniform
  const bool valid = i < a.n;
  float H[9] = {}, so[7] = {};
  int64_t sidx = 0;
  if (valid) {
    if (a.hq) {
#pragma unroll
      for (int c = 0; c < 9; ++c) H[c] = a.hq[i * 9 + c];
      if (J2) {
        sidx = ((int64_t)a.eperm[i / a.nq] * a.nq + i % a.nq) * 7;
#pragma unroll
        for (int c = 0; c < 7; ++c) so[c] = a.st_old[sidx + c];
      }
    } else {
#pragma unroll
      for (int c = 0; c < 9; ++c) H[c] = a.in[i * FT::IN_W + c];
      if (J2) {
#pragma unroll
        for (int c = 0; c < 7; ++c) so[c] = a.in[i * FT::IN_W + 9 + c];
      }
    }
  }
  float P[9], C[10], sn[7], y[16];
  bool ok = false, bad = false;
  if constexpr (SURR) {
    float raw[16], x[16];
#pragma unroll
    for (int c = 0; c < 9; ++c) raw[c] = H[c];
#pragma unroll
    for (int c = 0; c < 7; ++c) raw[9 + c] = so[c];
    normalized_features<ARCH>(a.m, raw, x);
    float yn[16];
    mlp_forward_wave<A>(a.m, x, yn, lane);
#pragma unroll
    for (int o = 0; o < FT::OUT_W; ++o) y[o] = yn[o] * a.m.out_scale[o] + a.m.out_shift[o];
    if (valid) {
      // frozen decisions: a point that passed keeps the network's output (checked with an infinite tolerance, which
      // only assembles P and the tangent data), a point that fell back stays on the plain model
      const bool frozen = a.freeze && a.accept;
      const bool use = frozen ? a.accept[i] != 0 : true;
      const float tol = frozen ? 3.0e38f : a.tol;
      if (use) {
        if constexpr (J2) ok = j2_surrogate(a.mp, H, so, y, tol, P, sn, C);
        else ok = nh_surrogate(a.mp, H, y, tol, P, C);
      }
      if (a.accept && !frozen) a.accept[i] = ok ? 1 : 0;
    }
    const uint64_t fb = __ballot(valid && !ok);
    if (lane == 0 && fb && a.nfallback) atomicAdd(a.nfallback, (unsigned long long)__popcll(fb));
  }
  if (valid && !ok) {  // the plain model: the fallback, or the whole update when SURR is off
    if constexpr (J2) j2_plain(a.mp, H, so, y, P, sn, C);
    else nh_plain(a.mp, H, y, P, C, bad);
  } else if (valid && SURR && !a.hq) {
    // batch output of an accepted surrogate sample: report what the assembly would use
    if constexpr (J2) {
      y[0] = P[0]; y[1] = P[3]; y[2] = P[6]; y[3] = P[4]; y[4] = P[7]; y[5] = P[8];
#pragma unroll
      for (int c = 0; c < 7; ++c) y[6 + c] = sn[c] - so[c];
    }
  }
  if (!valid) return;
  if (bad && a.flag) raise_flag(a.flag);
  if (a.hq) {
    float* q = a.qpmat + i * (9 + NC);
#pragma unroll
    for (int c = 0; c < 9; ++c) q[c] = P[c];
#pragma unroll
    for (int c = 0; c < NC; ++c) q[9 + c] = C[c];
    if (J2 && a.st_new) {
#pragma unroll
      for (int c = 0; c < 7; ++c) a.st_new[sidx + c] = sn[c];
    }
  } else {
#pragma unroll
    for (int c = 0; c < FT::OUT_W; ++c) a.out[i * FT::OUT_W + c] = y[c];
  }
}

// ------------------------------------------------------------------ network-only forward (raw units)
// TT = 2: 64 samples per wavefront, lane = sample, as in the update. TT = 1: 32, on both lane halves; the lower
// stores. One tile is the shorter chain, two load every weight once for both and go further
// where there is work for them; the J2 network's two tiles at 3 wavefronts per SIMD (40 bytes of scratch) beat 2. One tile | two
// without | with that cap: J2 3,000 samples 25.0 | 28.0 | 35.6 us, 100,000 44.1 | 43.3 | 45.4, 2,000,000 422 | 445 | 360;
// neo-Hookean (no cap: it spills) 3,000 40.2 | 31.7, 100,000 69.6 | 50.9, 2,000,000 669 | 566.
template <int ARCH, int TT>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(ARCH == FECX_MLP_J2 && TT == 2 ? 3 : 1, 8)))
void mlp_forward_kernel(MatBatchArgs a) {
  using A = Arch<ARCH>;
  using FT = Feat<ARCH>;
  constexpr int SPW = 32 * TT;  // samples per wavefront
  const int lane = threadIdx.x % 64;
  const int64_t tile = (int64_t)blockIdx.x * 4 + threadIdx.x / 64;
  const int64_t i = tile * SPW + lane % SPW;
  if (tile * SPW >= a.n) return;
  const bool valid = i < a.n;
  float raw[16] = {}, x[16];
#pragma unroll
  for (int c = 0; c < FT::IN_W; ++c) raw[c] = valid ? a.in[i * FT::IN_W + c] : 0.0f;
  normalized_features<ARCH>(a.m, raw, x);
  if constexpr (TT == 2) {
    float yn[16];
    mlp_forward_wave<A>(a.m, x, yn, lane);
    if (valid) {
#pragma unroll
      for (int o = 0; o < FT::OUT_W; ++o) a.out[i * FT::OUT_W + o] = yn[o] * a.m.out_scale[o] + a.m.out_shift[o];
    }
  } else {
    const int h = lane >> 5;
    bf16x8 h0[1][1];
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const float lo = k < A::D[0] ? x[k] : 0.0f, hi = 8 + k < A::D[0] ? x[(8 + k) % A::D[0]] : 0.0f;
      h0[0][0][k] = (__bf16)(h ? hi : lo);
    }
    f32x16 out[1];
    mlp_hidden<A, 1>(a.m, h0, out, lane);
    float yn[16];
#pragma unroll
    for (int j = 0; j < 8; ++j) {  // the halves' D registers to both
      uint32_t lo = __float_as_uint(out[0][j]), hi = lo;
      swap_halves(lo, hi);
      yn[dreg_feature(0, 0, j)] = __uint_as_float(lo);
      yn[dreg_feature(0, 1, j)] = __uint_as_float(hi);
    }
    if (valid && h == 0) {
#pragma unroll
      for (int o = 0; o < FT::OUT_W; ++o) a.out[i * FT::OUT_W + o] = yn[o] * a.m.out_scale[o] + a.m.out_shift[o];
    }
  }
}

// ------------------------------------------------------------------ J2 training samples: random strain paths
// Thread p follows one macroscopic strain path from zero through 4 random waypoints (symmetric directions, norm
// max_norm * U(0.2, 1.1)), piecewise linear over `steps` steps, updating the plain model; every step emits the raw
// input {H = eps, state} and the raw output {sigma, dplastic, deqps}.
__device__ __forceinline__ uint64_t smix(uint64_t& s) {
  uint64_t z = (s += 0x9E3779B97F4A7C15ULL);
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ULL;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBULL;
  return z ^ (z >> 31);
}
__device__ __forceinline__ float urand(uint64_t& s) { return (float)((smix(s) >> 40) * (1.0 / 16777216.0)); }
__device__ __forceinline__ float nrand(uint64_t& s) {
  const float u1 = fmaxf(urand(s), 1e-7f), u2 = urand(s);
  return sqrtf(-2.0f * logf(u1)) * cospif(2.0f * u2);
}

__global__ void j2_paths_kernel(int64_t npaths, int steps, float max_norm, uint64_t seed, MatParams mp, float* X,
                                float* T) {
  const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= npaths) return;
  uint64_t st = seed ^ ((uint64_t)p * 0xD1B54A32D192ED03ULL);
  float W[5][9];
#pragma unroll
  for (int c = 0; c < 9; ++c) W[0][c] = 0.0f;
  for (int k = 1; k < 5; ++k) {
    float g[6], nn = 0.0f;
    for (int c = 0; c < 6; ++c) g[c] = nrand(st);
    float S[9] = {g[0], g[3], g[5], g[3], g[1], g[4], g[5], g[4], g[2]};
    for (int c = 0; c < 9; ++c) nn += S[c] * S[c];
    const float amp = max_norm * (0.2f + 0.9f * urand(st)) / sqrtf(nn);
    for (int c = 0; c < 9; ++c) W[k][c] = amp * S[c];
  }
  const int per = steps / 4 > 0 ? steps / 4 : 1;
  float so[7] = {}, sn[7], P[9], C[9], y[13];
  for (int n = 1; n <= steps; ++n) {
    const int seg = min((n - 1) / per, 3);
    const float t = (float)(n - seg * per) / (float)per;
    float Hs[9];
    for (int c = 0; c < 9; ++c) Hs[c] = (1 - t) * W[seg][c] + t * W[seg + 1][c];
    j2_plain(mp, Hs, so, y, P, sn, C);
    const int64_t r = p * steps + (n - 1);
    for (int c = 0; c < 9; ++c) X[r * 16 + c] = Hs[c];
    for (int c = 0; c < 7; ++c) X[r * 16 + 9 + c] = so[c];
    for (int c = 0; c < 13; ++c) T[r * 13 + c] = y[c];
    for (int c = 0; c < 7; ++c) so[c] = sn[c];
  }
}

// ------------------------------------------------------------------ column mean / standard deviation (FP64 sums)
__global__ void column_stats_kernel(const float* X, int64_t n, int w, int ncol, float* shift, float* scale) {
  const int c = blockIdx.x;  // one work-group per column
  if (c >= ncol) return;
  __shared__ double s1[256], s2[256];
  double a = 0.0, b = 0.0;
  for (int64_t i = threadIdx.x; i < n; i += blockDim.x) {
    const double v = X[i * w + c];
    a += v;
    b += v * v;
  }
  s1[threadIdx.x] = a;
  s2[threadIdx.x] = b;
  __syncthreads();
  for (int off = 128; off >= 1; off >>= 1) {
    if ((int)threadIdx.x < off) { s1[threadIdx.x] += s1[threadIdx.x + off]; s2[threadIdx.x] += s2[threadIdx.x + off]; }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    const double m = s1[0] / (double)n, var = fmax(s2[0] / (double)n - m * m, 0.0);
    const double sd = sqrt(var);
    shift[c] = (float)m;
    scale[c] = (float)(sd > 1e-12 * fmax(1.0, fabs(m)) ? sd : 1.0);
  }
}

// J2 features from raw inputs, for the column statistics of the inputs
__global__ void j2_feature_rows_kernel(const float* in, int64_t n, float* x) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  float raw[16], f[13];
  for (int c = 0; c < 16; ++c) raw[c] = in[i * 16 + c];
  Feat<FECX_MLP_J2>::features(raw, f);
  for (int c = 0; c < 13; ++c) x[i * 13 + c] = f[c];
}

// ------------------------------------------------------------------ host launchers
template <int ARCH, int TT>
static void launch_train_tiles(const TrainArgs& a, hipStream_t s) {
  static_assert(TRAIN_PAD % (32 * TT) == 0, "whole work-groups");
  mlp_train_kernel<ARCH, TT><<<(unsigned)(a.npad / (32 * TT)), train_waves<Arch<ARCH>>() * 64, 0, s>>>(a);
}
// Sample tiles of one work-group: two share every weight operand, one is the shorter chain and leaves the 128-wide network,
// with three hidden layers' GELU' in registers, two work-groups on a CU. Measured, one | two tiles, whole gradient: neo-Hookean
// 1,500 samples 35.5 | 38.0 us, 16,384 51.6 | 47.1, 100,000 202 | 183; J2 1,500 32.8 | 36.7, 16,384 42.0 | 45.0, 100,000
// 141 | 165. So the 256-wide network takes two once every CU (256 of them) has a work-group of one.
template <int ARCH>
static void launch_train(const TrainArgs& a, hipStream_t s) {
  constexpr int MOST = max_hidden<Arch<ARCH>>() > 128 ? 2 : 1;
  if (a.npad > 32 * 256) launch_train_tiles<ARCH, MOST>(a, s);
  else launch_train_tiles<ARCH, 1>(a, s);
}
template <int ARCH>
static void launch_wgrad(WGradArgs a, hipStream_t s) {
  a.nblocks = wgrad_blocks<ARCH>();
  mlp_wgrad_kernel<ARCH><<<(unsigned)((a.nchunk + 7) / 8 * 8 * a.nblocks), 64, 0, s>>>(a);
}

void mlp_launch_train(int arch, const TrainArgs& a, hipStream_t s) {
  if (arch == FECX_MLP_J2) launch_train<FECX_MLP_J2>(a, s);
  else launch_train<FECX_MLP_NH>(a, s);
}
void mlp_launch_wgrad(int arch, const WGradArgs& a, hipStream_t s) {
  if (arch == FECX_MLP_J2) launch_wgrad<FECX_MLP_J2>(a, s);
  else launch_wgrad<FECX_MLP_NH>(a, s);
}
void mlp_launch_update(int arch, const UpdateArgs& a, hipStream_t s) {
  const unsigned g = (unsigned)((a.np + 255) / 256) + (a.loss ? 1u : 0u);
  if (arch == FECX_MLP_J2) mlp_update_kernel<FECX_MLP_J2><<<g, 256, 0, s>>>(a);
  else mlp_update_kernel<FECX_MLP_NH><<<g, 256, 0, s>>>(a);
}
void mlp_launch_gather(int64_t n, int w, const int32_t* idx, const float* src, float* dst, hipStream_t s) {
  if (n > 0) gather_rows_kernel<<<(unsigned)((n * w + 255) / 256), 256, 0, s>>>(n, w, idx, src, dst);
}
void mlp_launch_forward(int arch, const MatBatchArgs& a, hipStream_t s) {
  if (a.n == 0) return;
  const bool one = arch == FECX_MLP_J2 && a.n <= (1 << 18);  // 140,000 samples 51 | 55 us, 280,000 77.6 | 77.4
  const unsigned g = one ? (unsigned)((a.n + 127) / 128) : (unsigned)((a.n + 255) / 256);
  if (one) mlp_forward_kernel<FECX_MLP_J2, 1><<<g, 256, 0, s>>>(a);
  else if (arch == FECX_MLP_J2) mlp_forward_kernel<FECX_MLP_J2, 2><<<g, 256, 0, s>>>(a);
  else mlp_forward_kernel<FECX_MLP_NH, 2><<<g, 256, 0, s>>>(a);
}
void mlp_launch_material(int arch, bool surrogate, const MatBatchArgs& a, hipStream_t s) {
  const unsigned g = (unsigned)((a.n + 255) / 256);
  if (a.n == 0) return;
  if (arch == FECX_MLP_J2) {
    if (surrogate) material_kernel<FECX_MLP_J2, true><<<g, 256, 0, s>>>(a);
    else material_kernel<FECX_MLP_J2, false><<<g, 256, 0, s>>>(a);
  } else {
    if (surrogate) material_kernel<FECX_MLP_NH, true><<<g, 256, 0, s>>>(a);
    else material_kernel<FECX_MLP_NH, false><<<g, 256, 0, s>>>(a);
  }
}
void mlp_launch_j2_paths(int64_t npaths, int steps, float max_norm, uint64_t seed, const MatParams& mp, float* X,
                         float* T, hipStream_t s) {
  if (npaths > 0) j2_paths_kernel<<<(unsigned)((npaths + 127) / 128), 128, 0, s>>>(npaths, steps, max_norm, seed, mp, X, T);
}
void mlp_launch_column_stats(const float* X, int64_t n, int w, int ncol, float* shift, float* scale, hipStream_t s) {
  column_stats_kernel<<<(unsigned)ncol, 256, 0, s>>>(X, n, w, ncol, shift, scale);
}
void mlp_launch_j2_features(const float* in, int64_t n, float* x, hipStream_t s) {
  if (n > 0) j2_feature_rows_kernel<<<(unsigned)((n + 255) / 256), 256, 0, s>>>(in, n, x);
}

template <int ARCH>
static ArchInfo make_info() {
  using A = Arch<ARCH>;
  using O = Offs<A>;
  ArchInfo r{};
  r.nl = A::NL;
  for (int l = 0; l <= A::NL; ++l) { r.d[l] = A::D[l]; r.p[l] = A::P[l]; }
  r.in_w = Feat<ARCH>::IN_W;
  r.nfeat = Feat<ARCH>::NF;
  r.out_w = Feat<ARCH>::OUT_W;
  r.nparams = O::params();
  r.wf_vecs = O::wf_total();
  r.wb_vecs = O::wb_total();
  r.nbias = O::bias_total();
  return r;
}

ArchInfo arch_info(int arch) { return arch == FECX_MLP_J2 ? make_info<FECX_MLP_J2>() : make_info<FECX_MLP_NH>(); }

}  // namespace fecx
