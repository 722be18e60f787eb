// Residuals and matrix-free actions of tet10 elements, one lane per element (launch_lane_element).
//
// element_kernel (element.hip) gives a tet10 element 16 lanes, four per quadrature point, each of which inverts the Jacobian and
// evaluates the material at its point: four times the work, which the element blocks' node phase (where there is one) dwarfs.
// Without element blocks it is the larger part. One lane per element does it once, the points one after the other with their
// shape functions as literals and the zero ones left out, and holds the element's rows in registers. The sums over nodes and
// points keep element_kernel's order, so both give the same bits.
// Bound by the gather (10 scattered nodes of 48 bytes per lane) and by VALU issue at 2 wavefronts per SIMD. Neo-Hookean, whole
// calls, 16 lanes per element against one: residual 33 x 39 x 35 x 6 elements 92.4 against 75 us (kernel 52, now 31), action
// 39^3 x 6 139 against 117, action 25^3 x 6 57 against 53.5; Poisson residual 39^3 x 6 82.7 against 59. A cap of 3 wavefronts
// per SIMD spills (94 and 190 us). hex8, whose 8 lanes share nothing but the node inputs, lost by it (neo-Hookean action 83 x 67 x
// 71 97 against 138 us) and keeps its lanes.
#include "fem_device.h"

namespace fecx {

constexpr int LE_THREADS = 64;  // one wavefront: 64 elements

template <int NF, int PHYS, bool MF>
__global__ __launch_bounds__(LE_THREADS) __attribute__((amdgpu_waves_per_eu(2, 8))) void lane_element_kernel(ElementArgs args) {
  constexpr int KIND = FECX_TET10;
  using T = ET<KIND>;
  using M = Mat<PHYS>;
  constexpr int ND = 3, NNPE = T::NNPE, NQ = T::NQ, D = NF * ND, NDOF = NNPE * NF;
  const int64_t e = args.ebeg + xcd_chunk(blockIdx.x, gridDim.x) * LE_THREADS + threadIdx.x;
  if (e >= args.ne) return;
  bool bad = false;
  float X[NNPE][ND], U[NNPE][NF], V[MF ? NNPE : 1][NF], x0[ND];
  {
    int64_t nd[NNPE];
#pragma unroll
    for (int a = 0; a < NNPE; ++a) nd[a] = args.conn[e * NNPE + a];
    float hi[NNPE][ND], lo[NNPE][ND];
    double u[NNPE][NF];
#pragma unroll
    for (int a = 0; a < NNPE; ++a) {
#pragma unroll
      for (int d = 0; d < ND; ++d) { hi[a][d] = args.xhi[nd[a] * ND + d]; lo[a][d] = args.xlo[nd[a] * ND + d]; }
#pragma unroll
      for (int i = 0; i < NF; ++i) u[a][i] = args.U[nd[a] * NF + i];
    }
#pragma unroll
    for (int a = 0; a < NNPE; ++a) {
#pragma unroll
      for (int d = 0; d < ND; ++d) X[a][d] = (hi[a][d] - hi[0][d]) + (lo[a][d] - lo[0][d]);
#pragma unroll
      for (int i = 0; i < NF; ++i) U[a][i] = (float)(u[a][i] - u[0][i]);
    }
#pragma unroll
    for (int d = 0; d < ND; ++d) x0[d] = hi[0][d] + lo[0][d];
    if constexpr (MF) {
#pragma unroll
      for (int a = 0; a < NNPE; ++a)
#pragma unroll
        for (int i = 0; i < NF; ++i) u[a][i] = args.V[nd[a] * NF + i];
#pragma unroll
      for (int a = 0; a < NNPE; ++a)
#pragma unroll
        for (int i = 0; i < NF; ++i) V[a][i] = (float)(u[a][i] - u[0][i]);
    }
  }
  // the sum over the nodes of term(a, sum so far) in element_kernel's order: the nodes r, r + 4, r + 8 on lane r of a point's
  // four, then the lanes in pairs
  auto node_sum = [](auto term) {
    float p[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      p[r] = 0.0f;
#pragma unroll
      for (int a = r; a < NNPE; a += 4) p[r] = term(a, p[r]);
    }
    return (p[0] + p[1]) + (p[2] + p[3]);
  };
  float R[NDOF] = {};
#pragma unroll
  for (int q = 0; q < NQ; ++q) {
    float xi[ND], N[NNPE], dN[NNPE][ND];
    qpoint<KIND>(q, xi);
#pragma unroll
    for (int a = 0; a < NNPE; ++a) shape_node<KIND>(a, xi, N[a], dN[a]);
    float J[ND][ND];
#pragma unroll
    for (int i = 0; i < ND; ++i)
#pragma unroll
      for (int j = 0; j < ND; ++j)
        J[i][j] = node_sum([&](int a, float s) { return dN[a][j] != 0.0f ? fmaf(X[a][i], dN[a][j], s) : s; });
    const float c00 = J[1][1] * J[2][2] - J[1][2] * J[2][1], c01 = J[1][2] * J[2][0] - J[1][0] * J[2][2],
                c02 = J[1][0] * J[2][1] - J[1][1] * J[2][0];
    const float det = J[0][0] * c00 + J[0][1] * c01 + J[0][2] * c02;
    const float id = 1.0f / det;
    float Ji[ND][ND];
    Ji[0][0] = c00 * id; Ji[0][1] = (J[0][2] * J[2][1] - J[0][1] * J[2][2]) * id;
    Ji[0][2] = (J[0][1] * J[1][2] - J[0][2] * J[1][1]) * id;
    Ji[1][0] = c01 * id; Ji[1][1] = (J[0][0] * J[2][2] - J[0][2] * J[2][0]) * id;
    Ji[1][2] = (J[0][2] * J[1][0] - J[0][0] * J[1][2]) * id;
    Ji[2][0] = c02 * id; Ji[2][1] = (J[0][1] * J[2][0] - J[0][0] * J[2][1]) * id;
    Ji[2][2] = (J[0][0] * J[1][1] - J[0][1] * J[1][0]) * id;
    if (!(det > 0.0f)) bad = true;
    float g[NNPE][ND];
#pragma unroll
    for (int a = 0; a < NNPE; ++a)
#pragma unroll
      for (int j = 0; j < ND; ++j) {
        float t = 0.0f;
#pragma unroll
        for (int i = 0; i < ND; ++i)
          if (dN[a][i] != 0.0f) t = fmaf(dN[a][i], Ji[i][j], t);
        g[a][j] = t;
      }
    const float w = det * qweight<KIND, float>();
    float H[D], P[D], C[M::NC];
#pragma unroll
    for (int i = 0; i < NF; ++i)
#pragma unroll
      for (int j = 0; j < ND; ++j) H[i * ND + j] = node_sum([&](int a, float s) { return fmaf(U[a][i], g[a][j], s); });
    float so[7] = {}, sn[7];
    M::template eval<ND>(args.mp, H, so, sn, P, C, bad);
#pragma unroll
    for (int c = 0; c < D; ++c)
      if (!(P[c] == P[c])) bad = true;
    float f = 0.0f;  // Poisson source at the point
    if constexpr (!MF && PHYS == FECX_POISSON) {
      f = args.mp.p[1];
      if (args.mp.source_kind == 1) {
        f *= (float)ND * 9.8696044010893586f;
#pragma unroll
        for (int d = 0; d < ND; ++d)
          f *= sinpif(x0[d] + node_sum([&](int a, float s) { return fmaf(N[a], X[a][d], s); }));
      }
    }
    if constexpr (MF) {
      float Gv[D];
#pragma unroll
      for (int i = 0; i < NF; ++i)
#pragma unroll
        for (int j = 0; j < ND; ++j) Gv[i * ND + j] = node_sum([&](int a, float s) { return fmaf(V[a][i], g[a][j], s); });
      M::template dP<ND>(args.mp, C, Gv, P);
    }
#pragma unroll
    for (int a = 0; a < NNPE; ++a)
#pragma unroll
      for (int i = 0; i < NF; ++i) {
        float s = 0.0f;
#pragma unroll
        for (int j = 0; j < ND; ++j) s = fmaf(P[i * ND + j], g[a][j], s);
        if constexpr (!MF && PHYS == FECX_POISSON) s = fmaf(-N[a], f, s);
        R[a * NF + i] = fmaf(w, s, R[a * NF + i]);
      }
  }
  typedef float vec2 __attribute__((ext_vector_type(2)));
  float* out = args.Rel + e * NDOF;  // 8-byte aligned: an even number of words per element
  static_assert(NDOF % 2 == 0, "pairs");
#pragma unroll
  for (int c = 0; c < NDOF; c += 2) *reinterpret_cast<vec2*>(out + c) = vec2{R[c], R[c + 1]};
  if (bad) raise_flag(args.flag);
}

template <int NF, int PHYS>
static int launch_one(int mode, const ElementArgs& a, hipStream_t s) {
  const unsigned g = (unsigned)(((a.ne - a.ebeg + LE_THREADS - 1) / LE_THREADS + 7) / 8 * 8);
  if (mode == MODE_R) lane_element_kernel<NF, PHYS, false><<<g, LE_THREADS, 0, s>>>(a);
  else lane_element_kernel<NF, PHYS, true><<<g, LE_THREADS, 0, s>>>(a);
  return 0;
}

int launch_lane_element(int kind, int nf, int mode, const ElementArgs& a, hipStream_t s) {
  if (kind != FECX_TET10 || a.fp64_geometry || (mode != MODE_R && mode != MODE_ACTION_MF)) return -1;
  // One lane per element has to fill the chip: half a wavefront per SIMD. Neo-Hookean, 16 lanes against one: 12^3 x 6 (10,368
  // elements) residual 33.4 against 35.1 us, action 35.1 against 38.6; 20^3 x 6 (48,000) 42.1 against 40.3 and 45.4 against 44.6.
  if (a.ne - a.ebeg <= (1 << 15)) return -1;
  const int phys = a.mp.phys;
  if (nf == 1 && phys == FECX_POISSON) return launch_one<1, FECX_POISSON>(mode, a, s);
  if (nf == 3 && phys == FECX_LINEAR_ELASTIC) return launch_one<3, FECX_LINEAR_ELASTIC>(mode, a, s);
  if (nf == 3 && phys == FECX_NEOHOOKEAN) return launch_one<3, FECX_NEOHOOKEAN>(mode, a, s);
  return -1;
}

}  // namespace fecx
