// Poisson residual and Jacobian of a structured hex8 mesh, one lane per element and one lane per row (launch_poisson_hex8_*).
//
// The element kernel of element.hip gives an element 8 lanes, one quadrature point and then one node each, and hands the shape
// gradients over through LDS: for a scalar field that is about 700 VALU instructions per wavefront of 8 elements, a third of
// them addresses, lane shuffles and shape functions. With one lane per element the quadrature points are unrolled, their shape
// functions are literals, nothing leaves the registers, and 64 elements take about 3,000 instructions. The sums have the
// order of element.hip and reduce.hip, so both paths give the same bits.
#include "fem_device.h"

namespace fecx {

constexpr int PH_PAIRS = 36;  // words of a symmetric 8 x 8 element matrix
// word of the pair {a, b}
__host__ __device__ constexpr int ph_pair(int a, int b) { return a <= b ? a * 8 - a * (a - 1) / 2 + b - a : ph_pair(b, a); }
// local node at corner (ox, oy, oz)
__host__ __device__ constexpr int ph_local(int ox, int oy, int oz) { return 4 * oz + (oy ? 3 - ox : ox); }

// Where an element's NW words are stored: 64 elements' words together, word by word (word k is 64 k further on), so that a
// wavefront stores and loads whole lines. (One plane per word instead: 36 streams, and with planes a power of two apart the
// rows of 128^3 elements took 510 us where they now take 185.) Elements are numbered with x fastest here, like the nodes.
template <int NW>
__device__ __forceinline__ int64_t ph_store(uint32_t e) {
  return (int64_t)(e / 64) * (64 * NW) + e % 64;
}

// Inputs of one element's nodes, in local order
struct PhNode {
  float hi[3], lo[3];
  double u;
};

// The element: 36 words of K (K[ph_pair(a, b)]) and 8 of R, the sums in the order of element_eval (element.hip), whose 8 lanes
// per element hold one quadrature point each.
template <bool DO_R>
__device__ __forceinline__ void ph_element(const MatParams& mp, const PhNode (&nd)[8], float (&K)[PH_PAIRS], float (&R)[8],
                                           bool& bad) {
  float X[8][3], U[8];
#pragma unroll
  for (int a = 0; a < 8; ++a) {
#pragma unroll
    for (int d = 0; d < 3; ++d) X[a][d] = (nd[a].hi[d] - nd[0].hi[d]) + (nd[a].lo[d] - nd[0].lo[d]);
    U[a] = (float)(nd[a].u - nd[0].u);
  }
  // node 0's differences are zero, or NaN where its inputs are not finite: they enter the sums below as that check only
  if (!(X[0][0] == 0.0f && X[0][1] == 0.0f && X[0][2] == 0.0f && U[0] == 0.0f)) bad = true;
  float T[4][8];  // residual: sums over the points q and 7 - q
#pragma unroll
  for (int k = 0; k < PH_PAIRS; ++k) K[k] = 0.0f;
#pragma unroll
  for (int q = 0; q < 8; ++q) {
    float xi[3], N[8], dN[8][3];
    qpoint<FECX_HEX8>(q, xi);
#pragma unroll
    for (int a = 0; a < 8; ++a) shape_node<FECX_HEX8>(a, xi, N[a], dN[a]);
    float J[3][3] = {};
#pragma unroll
    for (int a = 1; a < 8; ++a)
#pragma unroll
      for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j) J[i][j] = a == 1 ? X[a][i] * dN[a][j] : fmaf(X[a][i], dN[a][j], J[i][j]);
    const float c00 = J[1][1] * J[2][2] - J[1][2] * J[2][1], c01 = J[1][2] * J[2][0] - J[1][0] * J[2][2],
                c02 = J[1][0] * J[2][1] - J[1][1] * J[2][0];
    const float det = J[0][0] * c00 + J[0][1] * c01 + J[0][2] * c02;
    const float id = 1.0f / det;
    float Ji[3][3];
    Ji[0][0] = c00 * id; Ji[0][1] = (J[0][2] * J[2][1] - J[0][1] * J[2][2]) * id;
    Ji[0][2] = (J[0][1] * J[1][2] - J[0][2] * J[1][1]) * id;
    Ji[1][0] = c01 * id; Ji[1][1] = (J[0][0] * J[2][2] - J[0][2] * J[2][0]) * id;
    Ji[1][2] = (J[0][2] * J[1][0] - J[0][0] * J[1][2]) * id;
    Ji[2][0] = c02 * id; Ji[2][1] = (J[0][1] * J[2][0] - J[0][0] * J[2][1]) * id;
    Ji[2][2] = (J[0][0] * J[1][1] - J[0][1] * J[1][0]) * id;
    if (!(det > 0.0f)) bad = true;
    float g[8][3];
#pragma unroll
    for (int a = 0; a < 8; ++a)
#pragma unroll
      for (int j = 0; j < 3; ++j) g[a][j] = fmaf(dN[a][2], Ji[2][j], fmaf(dN[a][1], Ji[1][j], dN[a][0] * Ji[0][j]));
    const float w = det;
    float H[3];
#pragma unroll
    for (int a = 1; a < 8; ++a)
#pragma unroll
      for (int j = 0; j < 3; ++j) H[j] = a == 1 ? U[a] * g[a][j] : fmaf(U[a], g[a][j], H[j]);
    if (!(H[0] == H[0] && H[1] == H[1] && H[2] == H[2])) bad = true;
    if constexpr (DO_R) {
      float wP[3];
#pragma unroll
      for (int j = 0; j < 3; ++j) wP[j] = w * H[j];
      float f = mp.p[1];
      if (mp.source_kind == 1) {
        f *= 3.0f * 9.8696044010893586f;
#pragma unroll
        for (int d = 0; d < 3; ++d) {
          float t = N[1] * X[1][d];
#pragma unroll
          for (int a = 2; a < 8; ++a) t = fmaf(N[a], X[a][d], t);
          f *= sinpif((nd[0].hi[d] + nd[0].lo[d]) + t);
        }
      }
      const float wf = w * f;
#pragma unroll
      for (int a = 0; a < 8; ++a) {
        const float s = fmaf(-N[a], wf, fmaf(wP[2], g[a][2], fmaf(wP[1], g[a][1], wP[0] * g[a][0])));
        if (q < 4) T[q][a] = s;
        else T[7 - q][a] = s + T[7 - q][a];
      }
    }
    const float sw = sqrtf(w);
#pragma unroll
    for (int a = 0; a < 8; ++a)
#pragma unroll
      for (int j = 0; j < 3; ++j) g[a][j] *= sw;
#pragma unroll
    for (int a = 0; a < 8; ++a)
#pragma unroll
      for (int b = a; b < 8; ++b)
#pragma unroll
        for (int j = 0; j < 3; ++j) K[ph_pair(a, b)] = fmaf(g[a][j], g[b][j], K[ph_pair(a, b)]);
  }
  if constexpr (DO_R) {
#pragma unroll
    for (int a = 0; a < 8; ++a) R[a] = (T[0][a] + T[2][a]) + (T[1][a] + T[3][a]);
  }
}

constexpr int PH_ELEMS = 256;  // elements of one work-group
// Bound by VALU issue, some 3,000 instructions per element: 128^3 elements 164 us (8 lanes per element: 295). STREAM: nontemporal
// stores, where the words of the mesh do not fit the 256 MB Infinity Cache anyway (128^3 step 357 against 382 us, 121 x 117 x 128
// 307 against 332; below, the rows read them from there: 64^3 62 against 69 us).
template <bool DO_R, bool STREAM>
__global__ __launch_bounds__(PH_ELEMS) void ph_element_kernel(ElementArgs a, FusedArgs f) {
  const uint32_t nex = f.nx - 1, ney = f.ny - 1;
  const int64_t e = xcd_chunk(blockIdx.x, gridDim.x) * PH_ELEMS + threadIdx.x;
  if (e >= a.ne) return;
  const uint32_t ex = (uint32_t)e % nex, r = (uint32_t)e / nex, ey = r % ney, ez = r / ney;
  const int64_t n0 = ex + (int64_t)f.nx * (ey + (int64_t)f.ny * ez);
  PhNode nd[8];
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    const int64_t n = n0 + ((k & 3) == 1 || (k & 3) == 2 ? 1 : 0) + ((k & 2) ? f.nx : 0) + ((k & 4) ? (int64_t)f.nx * f.ny : 0);
#pragma unroll
    for (int d = 0; d < 3; ++d) { nd[k].hi[d] = a.xhi[n * 3 + d]; nd[k].lo[d] = a.xlo[n * 3 + d]; }
    nd[k].u = a.U[n];
  }
  float K[PH_PAIRS], R[8];
  bool bad = false;
  ph_element<DO_R>(a.mp, nd, K, R, bad);
  auto store = [](float* p, float v) {
    if constexpr (STREAM) __builtin_nontemporal_store(v, p);
    else *p = v;
  };
#pragma unroll
  for (int k = 0; k < PH_PAIRS; ++k) store(a.Kel + ph_store<PH_PAIRS>((uint32_t)e) + 64 * k, K[k]);
  if constexpr (DO_R) {
#pragma unroll
    for (int k = 0; k < 8; ++k) store(a.Rel + ph_store<8>((uint32_t)e) + 64 * k, R[k]);
  }
  if (bad) raise_flag(a.flag);
}

// One lane per row: its 8 elements' words are loaded straight from their places (neighbouring lanes, neighbouring words) and added
// in FP64 in ascending order of the element ids, each into the accumulator of a fixed neighbour; the rows of a wavefront are
// consecutive in the CSR, so they are packed in LDS and stored as one range, in whole 128-byte lines but for its ends. Bound by
// that traffic: 128^3 elements, 369 MB read and 464 MB written in about 185 us (reduce_scalar_hex8_kernel, 8 lanes per row with
// an LDS read-add-write per word: 347). ROWS per work-group: 64 fills the chip sooner, 256 walks the words in longer
// pieces: 64^3 step 61.5 against 64.2 us, 101 x 83 x 127 205 against 194. (Backwards, from the elements stored last: as fast
// on large meshes, 32^3 37.0 against 34.8 us.)
template <bool DO_R, int ROWS>
__global__ __launch_bounds__(ROWS) void ph_row_kernel(ElementArgs a, FusedArgs f) {
  __shared__ __attribute__((aligned(16))) double all_rows[ROWS / 64][64 * 27 + 2];
  double* rows = all_rows[threadIdx.x / 64];
  const uint32_t nx = f.nx, ny = f.ny, nz = f.nz, nex = nx - 1, ney = ny - 1, nez = nz - 1;
  const int64_t nn = (int64_t)nx * ny * nz;
  const int lane = threadIdx.x % 64;
  const int64_t n = xcd_chunk(blockIdx.x, gridDim.x) * ROWS + threadIdx.x;
  const bool valid = n < nn;
  const int2 info = valid ? f.nodeinfo[n] : make_int2(0, 0);
  const uint32_t mask = (uint32_t)info.y;
  const uint32_t i = (uint32_t)n % nx, r = (uint32_t)n / nx, j = r % ny, k = r / ny;
  double acc[27], racc = 0.0;
#pragma unroll
  for (int d = 0; d < 27; ++d) acc[d] = 0.0;
  // the node's elements in ascending order of their ids: x slowest, z fastest (StructuredMesh.jl:116-123)
  float kv[8][8], rw[8];
  bool in[8];
#pragma unroll
  for (int t = 0; t < 8; ++t) {
    const int sx = t >> 2, sy = (t >> 1) & 1, sz = t & 1;  // element (i - 1 + sx, j - 1 + sy, k - 1 + sz)
    in[t] = valid && i + sx >= 1 && i + sx <= nex && j + sy >= 1 && j + sy <= ney && k + sz >= 1 && k + sz <= nez;
    const int la = ph_local(1 - sx, 1 - sy, 1 - sz);
    const uint32_t e = in[t] ? (i + sx - 1) + nex * ((j + sy - 1) + ney * (k + sz - 1)) : 0;
    if constexpr (DO_R) rw[t] = a.Rel[ph_store<8>(e) + 64 * la];
    const float* kw = a.Kel + ph_store<PH_PAIRS>(e);
#pragma unroll
    for (int b = 0; b < 8; ++b) kv[t][b] = kw[64 * ph_pair(la, b)];
  }
#pragma unroll
  for (int t = 0; t < 8; ++t) {
    const int sx = t >> 2, sy = (t >> 1) & 1, sz = t & 1;
    if constexpr (DO_R) racc += in[t] ? (double)rw[t] : 0.0;
#pragma unroll
    for (int b = 0; b < 8; ++b) {
      const int bx = (b & 3) == 1 || (b & 3) == 2, by = (b >> 1) & 1, bz = b >> 2;
      const int d = (bx + sx) + 3 * (by + sy) + 9 * (bz + sz);
      acc[d] += in[t] ? (double)kv[t][b] : 0.0;
    }
  }
  if (DO_R && valid) f.R[n] = racc;
  // the rows of consecutive nodes are consecutive in the CSR: packed in LDS, then stored as one range
  const uint64_t free_rows = __ballot(mask != 0);
  if (free_rows == 0) return;
  const int deg = __builtin_popcount(mask);
  const int first = __builtin_ctzll(free_rows), last = 63 - __builtin_clzll(free_rows);
  const int32_t base = __builtin_amdgcn_readlane(info.x, first);
  const int total = __builtin_amdgcn_readlane(info.x, last) + __builtin_amdgcn_readlane(deg, last) - base;
  double* out = f.vals + base;
  const int lead = (int)((reinterpret_cast<uintptr_t>(out) >> 3) & 15);  // words past a 128-byte line
  const int shift = lead & 1;
  if (__all(mask == 0x7FFFFFFu)) {
    double* row = rows + shift + (info.x - base);
#pragma unroll
    for (int d = 0; d < 27; ++d) row[d] = acc[d];
  } else if (mask) {
    double* row = rows + shift + (info.x - base);
#pragma unroll
    for (int d = 0; d < 27; ++d)
      if ((mask >> d) & 1u) row[__builtin_popcount(mask & ((1u << d) - 1u))] = acc[d];
  }
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
  __builtin_amdgcn_wave_barrier();
  // whole wavefronts store from 128-byte line to line, 16 bytes per lane
  const int head = min((16 - lead) & 15, total);
  if (lane < head) out[lane] = rows[shift + lane];
  typedef double f64x2 __attribute__((__vector_size__(16)));
  int w = head + 2 * lane;
  const int body = head + ((total - head) & ~1);
  for (; w < body; w += 128)
    __builtin_nontemporal_store(*reinterpret_cast<const f64x2*>(rows + shift + w), reinterpret_cast<f64x2*>(out + w));
  if (lane == 0 && body < total) out[body] = rows[shift + body];
}

bool poisson_hex8_applies(int64_t ne) {
  // One lane per element has to fill the chip: half a wavefront per SIMD. Steps, 8 lanes per element against one: 24^3 elements 31.7
  // against 33.9 us, 32^3 36.5 against 35-37, 43 x 37 x 51 49.9 against 42.7, 64^3 102 against 64, 128^3 637 against 353. Indexes are 32-bit.
  return ne > (1 << 15) && ne < (int64_t(1) << 31);
}
int64_t poisson_hex8_words(int64_t ne, int nw) { return (ne + 63) / 64 * 64 * nw; }

void launch_poisson_hex8_elements(int mode, const ElementArgs& a, const FusedArgs& f, hipStream_t s) {
  const unsigned g = (unsigned)(((a.ne + PH_ELEMS - 1) / PH_ELEMS + 7) / 8 * 8);
  const bool r = (mode & MODE_R) != 0;
  const bool stream = sizeof(float) * (poisson_hex8_words(a.ne, PH_PAIRS) + (r ? poisson_hex8_words(a.ne, 8) : 0)) > (256u << 20);
  if (r && stream) ph_element_kernel<true, true><<<g, PH_ELEMS, 0, s>>>(a, f);
  else if (r) ph_element_kernel<true, false><<<g, PH_ELEMS, 0, s>>>(a, f);
  else if (stream) ph_element_kernel<false, true><<<g, PH_ELEMS, 0, s>>>(a, f);
  else ph_element_kernel<false, false><<<g, PH_ELEMS, 0, s>>>(a, f);
}

template <int ROWS>
static void launch_rows(int mode, const ElementArgs& a, const FusedArgs& f, hipStream_t s) {
  const int64_t nn = (int64_t)f.nx * f.ny * f.nz;
  const unsigned g = (unsigned)(((nn + ROWS - 1) / ROWS + 7) / 8 * 8);
  if (mode & MODE_R) ph_row_kernel<true, ROWS><<<g, ROWS, 0, s>>>(a, f);
  else ph_row_kernel<false, ROWS><<<g, ROWS, 0, s>>>(a, f);
}
void launch_poisson_hex8_rows(int mode, const ElementArgs& a, const FusedArgs& f, hipStream_t s) {
  const int64_t nn = (int64_t)f.nx * f.ny * f.nz;
  if (nn < (1 << 19)) launch_rows<64>(mode, a, f, s);  // below eight work-groups of 256 rows per CU
  else launch_rows<256>(mode, a, f, s);
}

}  // namespace fecx
