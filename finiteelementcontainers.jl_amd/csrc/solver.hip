// Linear algebra on the assembled CSR Jacobian: SpMV, diagonal, and Jacobi-preconditioned conjugate gradients in FP64.
//
// The reference solves each Newton step with Krylov.jl's CG on stiffness(asm) (src/Solvers.jl:128-153) on the CPU. Here
// the CSR values stay in HBM where the assembly wrote them. The SpMV reads the column indices from the block-CSR view
// (one column index per NF x NF block, NF consecutive columns per block), so the CSR colval array is never
// materialised on the device. All reductions are two-stage in a fixed order: deterministic and bit-reproducible.
//
// A CG iteration is two kernels. cg_product_kernel forms p = z + beta p while it gathers it, A p and the partials of
// p.Ap; cg_update_kernel moves x, r and z and leaves the partials of r.z and r.r. Each kernel's work-groups sum the other
// one's partials themselves (at most CG_PARTS of them, in one fixed order, so all get the same bits), so no scalar kernel
// sits between them. The host enqueues CG_BATCH iterations ahead of the batch whose end it waits for, and learns of
// convergence from a pinned word, so the device never idles on the host; the iterations past convergence return at once.
#include "api_util.h"

namespace fecx {

constexpr int SV_THREADS = 256;
constexpr int CG_PARTS = 1024;  // work-groups (and partials) of a CG kernel, at most: 4 per CU, the product's occupancy
constexpr int CG_BATCH = 8;  // iterations enqueued per look at the convergence word

struct CsrView {
  int64_t nrows;            // unknowns = NF x free nodes
  const int64_t* bptr;      // free nodes + 1
  const int32_t* bcol;      // nnzb
  const double* vals;       // nnz
  const int64_t* rptr;      // dof-level CSR (a Dirichlet set that splits nodes): nrows + 1, or null
  const int32_t* rcol;      // its column indices
};

// A lane permutation of both halves of a double, folded into the adds below (no LDS round trip).
template <int CTRL>
__device__ __forceinline__ double dpp64(double x) {
  const int64_t b = __double_as_longlong(x);
  const int lo = __builtin_amdgcn_mov_dpp((int)(b & 0xffffffff), CTRL, 0xF, 0xF, true);
  const int hi = __builtin_amdgcn_mov_dpp((int)(b >> 32), CTRL, 0xF, 0xF, true);
  return __longlong_as_double(((int64_t)hi << 32) | (uint32_t)lo);
}
// Sum over aligned groups of L lanes, left on every lane of the group: quad_perm (xor 1, xor 2), then row_half_mirror
// and row_mirror, which exchange halves that are uniform by then, then across rows of 16 lanes.
template <int L>
__device__ __forceinline__ double group_sum(double v) {
  static_assert(L == 8 || L == 16 || L == 32, "lane groups");
  v += dpp64<0xB1>(v);
  v += dpp64<0x4E>(v);
  v += dpp64<0x141>(v);
  if constexpr (L >= 16) v += dpp64<0x140>(v);
  if constexpr (L >= 32) v += __shfl_xor(v, 16);
  return v;
}
__device__ __forceinline__ double wave_sum(double v) {
  v = group_sum<16>(v);
  v += __shfl_xor(v, 16);
  v += __shfl_xor(v, 32);
  return v;
}

// work-group sum of one double per thread (fixed order), on every thread; sh holds one double per wavefront
__device__ __forceinline__ double block_sum(double v, double* sh) {
  static_assert(SV_THREADS == 256, "four wavefronts");
  v = wave_sum(v);
  if (threadIdx.x % 64 == 0) sh[threadIdx.x / 64] = v;
  __syncthreads();
  v = (sh[0] + sh[1]) + (sh[2] + sh[3]);
  __syncthreads();  // sh may be written again
  return v;
}
// fixed-order sum of n partials by every work-group that needs it
__device__ __forceinline__ double sum_partials(const double* p, int n, double* sh) {
  double a = 0.0;
  for (int k = threadIdx.x; k < n; k += SV_THREADS) a += p[k];
  return block_sum(a, sh);
}
// the same of two arrays, their loads in flight together; sh holds two doubles per wavefront
__device__ __forceinline__ void sum_partials2(const double* p, const double* q, int n, double* sh, double& sp, double& sq) {
  double a = 0.0, b = 0.0;
  for (int k = threadIdx.x; k < n; k += SV_THREADS) {
    a += p[k];
    b += q[k];
  }
  a = wave_sum(a);
  b = wave_sum(b);
  if (threadIdx.x % 64 == 0) {
    sh[threadIdx.x / 64] = a;
    sh[4 + threadIdx.x / 64] = b;
  }
  __syncthreads();
  sp = (sh[0] + sh[1]) + (sh[2] + sh[3]);
  sq = (sh[4] + sh[5]) + (sh[6] + sh[7]);
  __syncthreads();  // sh may be written again
}

// ------------------------------------------------------------------ products with the matrix
// A "line" is what one lane group multiplies: the NF rows of a free node (NF columns per block share one column index and
// one gather of the vector across the NF rows), or (DOF_ROWS) one row of a dof-level CSR. L lanes per line, lane l taking
// columns l, l + L, ..., U of them in flight together: L U covers the rows of a structured mesh (hex8: 27 columns of one
// field, 81 of three; quad4: 18 of two), so such a line costs one chain of loads (pointer, column, vector), and the next
// line's pointer and columns are fetched under the current one's (cg_product_kernel). Wider rows (tet10: up to 195) loop.
// Lanes for 81 columns, whole solve of an elastic hex8 40 x 32 x 36 block (1,187 iterations): 16 lanes x 6 columns 37.0 ms
// (spills at 4 waves per SIMD), 32 x 3 31.4 ms; for 27 columns (Poisson hex8 36^3, 155 iterations): 8 lanes x 4 2.13 ms,
// 16 x 2 2.36 ms, 32 x 1 2.62 ms; for the 18 of a dof-level row of two fields (300 x 401 nodes on rollers, 100 iterations): 8 lanes
// x 3 2.64 ms, 32 x 3 6.50 (SpMV 26.9 against 48.6 us).
constexpr int DOF_ROWS = 0, DOF_ROWS_2 = -2;  // a row of a dof-level CSR, of 3 fields and of 2
template <int NF>
struct LineShape {
  static constexpr bool DOF = NF <= 0;
  static constexpr int L = NF == 1 || NF == DOF_ROWS_2 ? 8 : (NF == 2 ? 16 : 32);
  static constexpr int U = NF == 1 ? 4 : (NF == 2 ? 2 : 3);
  static constexpr int R = DOF ? 1 : NF, B = R;  // rows and columns per block
  static constexpr int GPW = SV_THREADS / L;         // lines per work-group
};
template <int NF>
struct LinePtr {
  int64_t rb;  // first block of the line (0 where it has none)
  int n;       // its columns (0: past the last line, or a node that no element touches)
};
template <int NF>
__device__ __forceinline__ LinePtr<NF> line_ptr(const CsrView& A, uint32_t g, uint32_t lines) {
  LinePtr<NF> p{0, 0};
  if (g < lines) {
    const int64_t* q = (LineShape<NF>::DOF ? A.rptr : A.bptr) + g;
    const int64_t rb = q[0];
    p.n = (int)(q[1] - rb) * LineShape<NF>::B;
    p.rb = p.n > 0 ? rb : 0;  // the last rows, empty, start where the matrix ends
  }
  return p;
}
// this lane's columns j0 + u L of the line; a column past the line repeats one of its own (an empty line: the matrix's entry
// 0, which csr_view makes sure exists)
template <int NF>
__device__ __forceinline__ int line_col(const LinePtr<NF>& p, int j) { return j < p.n ? j : (p.n > 0 ? p.n - 1 : 0); }
template <int NF>
__device__ __forceinline__ void line_index(const CsrView& A, const LinePtr<NF>& p, int j0, uint32_t (&idx)[LineShape<NF>::U]) {
  using S = LineShape<NF>;
  const int32_t* col = (S::DOF ? A.rcol : A.bcol) + p.rb;
#pragma unroll
  for (int u = 0; u < S::U; ++u) {
    const int j = line_col<NF>(p, j0 + u * S::L);
    idx[u] = (uint32_t)S::B * (uint32_t)col[j / S::B] + (uint32_t)(j % S::B);
  }
}
template <int NF>
__device__ __forceinline__ void line_vals(const CsrView& A, const LinePtr<NF>& p, int j0,
                                          double (&a)[LineShape<NF>::U][LineShape<NF>::R]) {
  using S = LineShape<NF>;
  const double* v = A.vals + (int64_t)(S::B * S::B) * p.rb;
#pragma unroll
  for (int u = 0; u < S::U; ++u) {
    const int j = line_col<NF>(p, j0 + u * S::L);
#pragma unroll
    for (int i = 0; i < S::R; ++i) a[u][i] = v[i * p.n + j];
  }
}
template <int NF>
__device__ __forceinline__ void line_add(const LinePtr<NF>& p, int j0, const double (&a)[LineShape<NF>::U][LineShape<NF>::R],
                                         const double (&x)[LineShape<NF>::U], double (&acc)[LineShape<NF>::R]) {
  using S = LineShape<NF>;
#pragma unroll
  for (int u = 0; u < S::U; ++u)
    if (j0 + u * S::L < p.n)
#pragma unroll
      for (int i = 0; i < S::R; ++i) acc[i] = fma(a[u][i], x[u], acc[i]);
}
// columns L U and on of a wide line
template <int NF, class GET>
__device__ __forceinline__ void line_rest(const CsrView& A, const LinePtr<NF>& p, int lane, GET get,
                                          double (&acc)[LineShape<NF>::R]) {
  using S = LineShape<NF>;
  for (int j0 = lane + S::L * S::U; j0 < p.n; j0 += S::L * S::U) {
    uint32_t idx[S::U];
    double a[S::U][S::R], x[S::U];
    line_index<NF>(A, p, j0, idx);
    line_vals<NF>(A, p, j0, a);
#pragma unroll
    for (int u = 0; u < S::U; ++u) x[u] = get(idx[u]);
    line_add<NF>(p, j0, a, x, acc);
  }
}
// the line's row products, row `lane` on lane `lane`
template <int NF>
__device__ __forceinline__ double line_rows(double (&acc)[LineShape<NF>::R], int lane) {
  using S = LineShape<NF>;
#pragma unroll
  for (int i = 0; i < S::R; ++i) acc[i] = group_sum<S::L>(acc[i]);
  double y = acc[0];
#pragma unroll
  for (int i = 1; i < S::R; ++i)
    if (lane == i) y = acc[i];
  return y;
}

// y = A x
template <int NF>
__global__ __launch_bounds__(SV_THREADS) void spmv_kernel(CsrView A, uint32_t lines, const double* x, double* y) {
  using S = LineShape<NF>;
  const int lane = threadIdx.x % S::L;
  const uint32_t g = blockIdx.x * S::GPW + threadIdx.x / S::L;
  if (g >= lines) return;  // whole lane groups
  const LinePtr<NF> p = line_ptr<NF>(A, g, lines);
  uint32_t idx[S::U];
  double a[S::U][S::R], v[S::U], acc[S::R] = {};
  line_index<NF>(A, p, lane, idx);
  line_vals<NF>(A, p, lane, a);
#pragma unroll
  for (int u = 0; u < S::U; ++u) v[u] = x[idx[u]];
  line_add<NF>(p, lane, a, v, acc);
  line_rest<NF>(A, p, lane, [&](uint32_t c) { return x[c]; }, acc);
  const double s = line_rows<NF>(acc, lane);
  if (lane < S::R) y[(int64_t)g * S::R + lane] = s;
}

// dinv[row] = 1 / A[row][row]; the diagonal block of free rank r is the slot s with bcol[rb + s] == r
template <int NF>
__global__ void diag_inv_kernel(CsrView A, double* dinv) {
  const int64_t row = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (row >= A.nrows) return;
  if (A.rptr) {  // dof-level CSR: binary search for the diagonal column
    int64_t lo = A.rptr[row], hi = A.rptr[row + 1] - 1;
    while (lo < hi) {
      const int64_t mid = (lo + hi) / 2;
      if (A.rcol[mid] < row) lo = mid + 1;
      else hi = mid;
    }
    const double d = (lo < A.rptr[row + 1] && A.rcol[lo] == row) ? A.vals[lo] : 0.0;
    dinv[row] = d != 0.0 ? 1.0 / d : 1.0;
    return;
  }
  const int64_t r = row / NF;
  const int i = (int)(row - r * NF);
  const int64_t rb = A.bptr[r];
  const int deg = (int)(A.bptr[r + 1] - rb);
  if (deg == 0) {  // a node that no element touches: no entry to read
    dinv[row] = 1.0;
    return;
  }
  int lo = 0, hi = deg - 1;
  while (lo < hi) {
    const int mid = (lo + hi) / 2;
    if (A.bcol[rb + mid] < r) lo = mid + 1;
    else hi = mid;
  }
  const double d = A.vals[NF * NF * rb + (int64_t)i * NF * deg + NF * lo + i];
  dinv[row] = d != 0.0 ? 1.0 / d : 1.0;
}

// ------------------------------------------------------------------ CG
// scalars: [0], [1] r.z of even and odd iterations, [4] r.r, [5] tol^2, [6] iterations (as double)
struct CgState {
  int64_t n;
  double* x;
  double* r;
  double* z;
  double* p[2];            // direction of odd and even iterations: each is formed from the other
  double* Ap;
  const double* dinv;
  double* sc;
  int* done;               // set by the iteration that finds r.r <= tol^2
  int* done_host;          // the same word in pinned host memory
  double *pap, *rz, *rr;   // partials
  int npap, nvec;          // their counts
  uint32_t lines, per;     // line groups of the matrix, and how many work-groups' worth one product work-group takes
};

// r holds A x; r = b - r, z = dinv r; partials of r.z, r.r and (in pap) b.b
__global__ __launch_bounds__(SV_THREADS) void cg_init_kernel(CgState c, const double* b) {
  __shared__ double sh[SV_THREADS / 64];
  double rz = 0.0, rr = 0.0, bb = 0.0;
  for (int64_t i = (int64_t)blockIdx.x * SV_THREADS + threadIdx.x; i < c.n; i += (int64_t)gridDim.x * SV_THREADS) {
    const double bi = b[i], r = bi - c.r[i], z = c.dinv ? c.dinv[i] * r : r;
    c.r[i] = r;
    c.z[i] = z;
    rz += r * z;
    rr += r * r;
    bb += bi * bi;
  }
  rz = block_sum(rz, sh);
  rr = block_sum(rr, sh);
  bb = block_sum(bb, sh);
  if (threadIdx.x == 0) {
    c.rz[blockIdx.x] = rz;
    c.rr[blockIdx.x] = rr;
    c.pap[blockIdx.x] = bb;
  }
}
__global__ __launch_bounds__(SV_THREADS) void cg_tolerance_kernel(CgState c, double rtol, double atol) {
  __shared__ double sh[SV_THREADS / 64];
  const double tol = atol + rtol * sqrt(sum_partials(c.pap, c.nvec, sh));
  if (threadIdx.x == 0) {
    c.sc[5] = tol * tol;
    *c.done = 0;
  }
}

// Iteration k: stops where r.r <= tol^2, else p = z + beta p (k = 0: p = z), Ap = A p, partials of p.Ap. Work-groups
// take equal contiguous ranges of lines, an XCD's one after the other, so that the gathers of z and p of neighbouring
// rows meet in its L2. The first line's loads are issued before the sums of the other kernel's partials, which they do
// not need, and each line's pointers and columns under the line before it. Bound by the matrix: on the elastic block above
// (12 million values, 98 MB with the columns) 20.9 us, 4.7 TB/s, where a plain read of a buffer of that size reaches
// 6.2 TB/s; the five kernels per iteration that this pair replaces took 56 us, 31.7 of them the product.
template <int NF>
__global__ __launch_bounds__(SV_THREADS) __attribute__((amdgpu_waves_per_eu(4, 8))) void cg_product_kernel(CsrView A,
                                                                                                          CgState c, int k) {
  using S = LineShape<NF>;
  __shared__ double sh[2 * SV_THREADS / 64];
  const int lane = threadIdx.x % S::L;
  const uint32_t g0 = (uint32_t)xcd_chunk(blockIdx.x, gridDim.x) * c.per * S::GPW + threadIdx.x / S::L;
  const double* z = c.z;
  const double* po = k > 0 ? c.p[(k + 1) & 1] : c.z;  // k = 0: beta = 0, and z is finite where p has not been written
  double* pn = c.p[k & 1];
  LinePtr<NF> cur = line_ptr<NF>(A, g0, c.lines), nxt = line_ptr<NF>(A, c.per > 1 ? g0 + S::GPW : c.lines, c.lines);
  uint32_t idx[S::U];
  double a[S::U][S::R], zc[S::U], pc[S::U], zr, pr;
  line_index<NF>(A, cur, lane, idx);
  auto issue = [&](uint32_t g) {  // the loads of the line at g with pointers `cur` and columns idx
    line_vals<NF>(A, cur, lane, a);
#pragma unroll
    for (int u = 0; u < S::U; ++u) { zc[u] = z[idx[u]]; pc[u] = po[idx[u]]; }
    const int64_t row = g < c.lines ? (int64_t)g * S::R + (lane < S::R ? lane : 0) : 0;
    zr = z[row];
    pr = po[row];
  };
  issue(g0);
  const double tol2 = c.sc[5], rz_old = k > 0 ? c.sc[(k - 1) & 1] : 0.0;
  double rr, rz;
  sum_partials2(c.rr, c.rz, c.nvec, sh, rr, rz);
  const bool stop = rr <= tol2;
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    if (!stop) c.sc[k & 1] = rz;
    else if (!*c.done) {
      c.sc[4] = rr;
      c.sc[6] = (double)k;
      *c.done = 1;
      *(volatile int*)c.done_host = 1;
    }
  }
  if (stop) return;
  const double beta = rz_old != 0.0 ? rz / rz_old : 0.0;
  double pap = 0.0;
  for (uint32_t t = 0; t < c.per; ++t) {
    const uint32_t g = g0 + t * S::GPW;
    if (t > 0) issue(g);
    const LinePtr<NF> now = cur;
    if (t + 1 < c.per) {  // the next line's columns, and the pointers of the one after
      cur = nxt;
      line_index<NF>(A, cur, lane, idx);
      nxt = line_ptr<NF>(A, t + 2 < c.per ? g + 2 * S::GPW : c.lines, c.lines);
    }
    double x[S::U], acc[S::R] = {};
#pragma unroll
    for (int u = 0; u < S::U; ++u) x[u] = fma(beta, pc[u], zc[u]);
    const double p = fma(beta, pr, zr);
    line_add<NF>(now, lane, a, x, acc);
    line_rest<NF>(A, now, lane, [&](uint32_t i) { return fma(beta, po[i], z[i]); }, acc);
    const double y = line_rows<NF>(acc, lane);
    if (g < c.lines && lane < S::R) {
      const int64_t row = (int64_t)g * S::R + lane;
      pn[row] = p;
      c.Ap[row] = y;
      pap = fma(p, y, pap);
    }
  }
  pap = block_sum(pap, sh);
  if (threadIdx.x == 0) c.pap[blockIdx.x] = pap;
}

// x += alpha p; r -= alpha Ap; z = dinv r; partials of r.z and r.r. The first entries' loads are issued before the sum
// of the partials of p.Ap.
__global__ __launch_bounds__(SV_THREADS) void cg_update_kernel(CgState c, int k) {
  __shared__ double sh[2 * SV_THREADS / 64];
  const double* p = c.p[k & 1];
  const int64_t i0 = (int64_t)blockIdx.x * SV_THREADS + threadIdx.x, step = (int64_t)gridDim.x * SV_THREADS;
  double x = 0.0, pi = 0.0, r = 0.0, ap = 0.0, di = 1.0;
  auto fetch = [&](int64_t i) {
    if (i < c.n) {
      x = c.x[i];
      pi = p[i];
      r = c.r[i];
      ap = c.Ap[i];
      if (c.dinv) di = c.dinv[i];
    }
  };
  fetch(i0);
  const int done = *c.done;
  const double rz_k = c.sc[k & 1];
  const double pap = sum_partials(c.pap, c.npap, sh);
  if (done) return;
  const double alpha = pap != 0.0 ? rz_k / pap : 0.0;
  double rz = 0.0, rr = 0.0;
  for (int64_t i = i0; i < c.n; i += step) {
    c.x[i] = x + alpha * pi;
    r -= alpha * ap;
    const double zi = c.dinv ? di * r : r;
    c.r[i] = r;
    c.z[i] = zi;
    rz += r * zi;
    rr += r * r;
    fetch(i + step);
  }
  rz = wave_sum(rz);
  rr = wave_sum(rr);
  if (threadIdx.x % 64 == 0) {
    sh[threadIdx.x / 64] = rz;
    sh[4 + threadIdx.x / 64] = rr;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    c.rz[blockIdx.x] = (sh[0] + sh[1]) + (sh[2] + sh[3]);
    c.rr[blockIdx.x] = (sh[4] + sh[5]) + (sh[6] + sh[7]);
  }
}

// after the last iteration: r.r and the iteration count, unless an iteration has stopped the solve
__global__ __launch_bounds__(SV_THREADS) void cg_finish_kernel(CgState c, int iterations) {
  __shared__ double sh[SV_THREADS / 64];
  if (*c.done) return;
  const double rr = sum_partials(c.rr, c.nvec, sh);
  if (threadIdx.x == 0) {
    c.sc[4] = rr;
    c.sc[6] = (double)iterations;
  }
}

__global__ __launch_bounds__(SV_THREADS) void sumsq_kernel(int64_t n, const double* v, double* partial) {
  __shared__ double sh[SV_THREADS / 64];
  double a = 0.0;
  for (int64_t i = (int64_t)blockIdx.x * SV_THREADS + threadIdx.x; i < n; i += (int64_t)gridDim.x * SV_THREADS)
    a += v[i] * v[i];
  const double s = block_sum(a, sh);
  if (threadIdx.x == 0) partial[blockIdx.x] = s;
}
__global__ __launch_bounds__(SV_THREADS) void sum_kernel(const double* partial, int n, double* out) {
  __shared__ double sh[SV_THREADS / 64];
  const double s = sum_partials(partial, n, sh);
  if (threadIdx.x == 0) *out = s;
}
__global__ void axpy_kernel(int64_t n, double a, const double* x, double* y) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) y[i] += a * x[i];
}

// work-groups of an elementwise kernel over n entries that leaves one partial each
static int vec_groups(int64_t n) { return (int)std::min<int64_t>((n + SV_THREADS - 1) / SV_THREADS, CG_PARTS); }

template <class F>
static void by_line(int nf, const CsrView& A, F f) {  // f(integral constant NF)
  if (A.rptr && nf == 2) f(std::integral_constant<int, DOF_ROWS_2>());
  else if (A.rptr) f(std::integral_constant<int, DOF_ROWS>());
  else if (nf == 1) f(std::integral_constant<int, 1>());
  else if (nf == 2) f(std::integral_constant<int, 2>());
  else f(std::integral_constant<int, 3>());
}

static void spmv(int nf, const CsrView& A, const double* x, double* y, hipStream_t s) {
  by_line(nf, A, [&](auto NFC) {
    using S = LineShape<decltype(NFC)::value>;
    const int64_t lines = A.nrows / S::R;
    spmv_kernel<decltype(NFC)::value><<<(unsigned)((lines + S::GPW - 1) / S::GPW), SV_THREADS, 0, s>>>(A, (uint32_t)lines, x, y);
  });
}

// work-groups of the product kernel: a multiple of 8 (XCD ranges), at most CG_PARTS, as few as give every one the same
// number of units
static void product_split(int nf, const CsrView& A, CgState& c) {
  int64_t units = 0;
  by_line(nf, A, [&](auto NFC) {
    using S = LineShape<decltype(NFC)::value>;
    c.lines = (uint32_t)(A.nrows / S::R);
    units = (c.lines + S::GPW - 1) / S::GPW;
  });
  const int64_t per = std::max<int64_t>((units + CG_PARTS - 1) / CG_PARTS, 1);
  c.per = (uint32_t)per;
  c.npap = (int)(((units + per - 1) / per + 7) / 8 * 8);
}

}  // namespace fecx

using namespace fecx_api;

namespace {

fecx::CsrView csr_view(fecx_ctx* ctx, const double* vals) {
  fecx::CsrView A{};
  A.nrows = (int64_t)ctx->hp.nfree * ctx->nf;
  A.bptr = get<int64_t>(ctx, "bptr");
  A.bcol = get<int32_t>(ctx, "bcol");
  A.vals = vals;
  if (ctx->partial) {
    A.nrows = (int64_t)ctx->unknown_dofs.size();
    A.rptr = get<int64_t>(ctx, "rptr");
    A.rcol = get<int32_t>(ctx, "rcol");
  }
  if (ctx->nnz == 0) {  // every free node is loose: what the empty lines load in place of their columns is one zero
    double* zero = get<double>(ctx, "sv_zero");
    if (!zero) zero = upload(ctx, "sv_zero", std::vector<double>(1, 0.0));
    A.vals = zero;
    A.bcol = A.rcol = (const int32_t*)zero;
  }
  return A;
}

void check_solver_ready(fecx_ctx* ctx) {
  check_device_ctx(ctx);
  require(ctx->has_pattern, FECX_ERR_STATE, "fecx_build_pattern has not been called");
  require(ctx->nf >= 1 && ctx->nf <= 3, FECX_ERR_UNSUPPORTED, "nf must be 1, 2 or 3");
}

}  // namespace

extern "C" {

int fecx_csr_spmv(fecx_ctx* ctx, const double* vals, const double* x, double* y) {
  return guard(ctx, [&] {
    check_solver_ready(ctx);
    require(vals && x && y, FECX_ERR_ARG, "null array");
    const fecx::CsrView A = csr_view(ctx, vals);
    fecx::spmv(ctx->nf, A, x, y, ctx->stream);
    HIPCHK(hipGetLastError());
    HIPCHK(hipStreamSynchronize(ctx->stream));
  });
}

int fecx_csr_diagonal_inverse(fecx_ctx* ctx, const double* vals, double* dinv) {
  return guard(ctx, [&] {
    check_solver_ready(ctx);
    require(vals && dinv, FECX_ERR_ARG, "null array");
    const fecx::CsrView A = csr_view(ctx, vals);
    if (A.nrows > 0) {
      const unsigned g = (unsigned)((A.nrows + 255) / 256);
      if (ctx->nf == 1) fecx::diag_inv_kernel<1><<<g, 256, 0, ctx->stream>>>(A, dinv);
      else if (ctx->nf == 2) fecx::diag_inv_kernel<2><<<g, 256, 0, ctx->stream>>>(A, dinv);
      else fecx::diag_inv_kernel<3><<<g, 256, 0, ctx->stream>>>(A, dinv);
    }
    HIPCHK(hipGetLastError());
    HIPCHK(hipStreamSynchronize(ctx->stream));
  });
}

int fecx_cg_solve(fecx_ctx* ctx, const double* vals, const double* b, double* x, double rtol, double atol, int maxit,
                  int precond, int* iters, double* resnorm) {
  return guard(ctx, [&] {
    check_solver_ready(ctx);
    require(vals && b && x && maxit >= 0 && rtol >= 0 && atol >= 0, FECX_ERR_ARG, "bad arguments");
    const fecx::CsrView A = csr_view(ctx, vals);
    const int64_t n = A.nrows;
    hipStream_t s = ctx->stream;
    fecx::CgState c{};
    c.n = n;
    c.x = x;
    c.r = (double*)dev_atleast(ctx, "cg_r", sizeof(double) * (n + 1));
    c.z = (double*)dev_atleast(ctx, "cg_z", sizeof(double) * (n + 1));
    c.p[0] = (double*)dev_atleast(ctx, "cg_p", sizeof(double) * (n + 1));
    c.p[1] = (double*)dev_atleast(ctx, "cg_q", sizeof(double) * (n + 1));
    c.Ap = (double*)dev_atleast(ctx, "cg_ap", sizeof(double) * (n + 1));
    c.sc = (double*)dev_atleast(ctx, "cg_sc", sizeof(double) * 8);
    c.done = (int*)dev_atleast(ctx, "cg_done", sizeof(int));
    c.done_host = ctx->cg_done_host;
    require(c.done_host != nullptr, FECX_ERR_STATE, "no host word");
    fecx::product_split(ctx->nf, A, c);
    c.nvec = fecx::vec_groups(n);
    c.pap = (double*)dev_atleast(ctx, "cg_pap", sizeof(double) * (fecx::CG_PARTS + 8));
    c.rz = (double*)dev_atleast(ctx, "cg_rz", sizeof(double) * fecx::CG_PARTS);
    c.rr = (double*)dev_atleast(ctx, "cg_rr", sizeof(double) * fecx::CG_PARTS);
    double* dinv = nullptr;
    if (precond) {
      dinv = (double*)dev_atleast(ctx, "cg_dinv", sizeof(double) * (n + 1));
      const unsigned g = (unsigned)((n + 255) / 256);
      if (n > 0) {
        if (ctx->nf == 1) fecx::diag_inv_kernel<1><<<g, 256, 0, s>>>(A, dinv);
        else if (ctx->nf == 2) fecx::diag_inv_kernel<2><<<g, 256, 0, s>>>(A, dinv);
        else fecx::diag_inv_kernel<3><<<g, 256, 0, s>>>(A, dinv);
      }
    }
    c.dinv = dinv;
    // r = b - A x; the stopping rule is ||r|| <= atol + rtol ||b|| (Krylov.jl's cg)
    *(volatile int*)c.done_host = 0;
    fecx::spmv(ctx->nf, A, x, c.r, s);
    fecx::cg_init_kernel<<<(unsigned)c.nvec, fecx::SV_THREADS, 0, s>>>(c, b);
    fecx::cg_tolerance_kernel<<<1, fecx::SV_THREADS, 0, s>>>(c, rtol, atol);
    HIPCHK(hipGetLastError());
    while (ctx->cg_events.size() < 2) {
      hipEvent_t e;
      HIPCHK(hipEventCreateWithFlags(&e, hipEventDisableTiming));
      ctx->cg_events.push_back(e);
    }
    int it = 0;
    for (int b0 = 0; it < maxit; ++b0) {
      const int end = std::min(it + fecx::CG_BATCH, maxit);
      for (; it < end; ++it) {
        fecx::by_line(ctx->nf, A, [&](auto NFC) {
          fecx::cg_product_kernel<decltype(NFC)::value><<<(unsigned)c.npap, fecx::SV_THREADS, 0, s>>>(A, c, it);
        });
        fecx::cg_update_kernel<<<(unsigned)c.nvec, fecx::SV_THREADS, 0, s>>>(c, it);
      }
      HIPCHK(hipGetLastError());
      HIPCHK(hipEventRecord(ctx->cg_events[b0 & 1], s));
      if (b0 == 0) continue;
      HIPCHK(hipEventSynchronize(ctx->cg_events[(b0 - 1) & 1]));  // the batch before the one just enqueued
      if (*(volatile int*)c.done_host) break;
    }
    fecx::cg_finish_kernel<<<1, fecx::SV_THREADS, 0, s>>>(c, it);
    HIPCHK(hipGetLastError());
    double sc[8];
    HIPCHK(hipMemcpyAsync(sc, c.sc, sizeof(sc), hipMemcpyDeviceToHost, s));
    HIPCHK(hipStreamSynchronize(s));
    if (iters) *iters = (int)sc[6];
    if (resnorm) *resnorm = std::sqrt(sc[4]);
  });
}

int fecx_vector_norm(fecx_ctx* ctx, const double* v, int64_t n, double* out) {
  return guard(ctx, [&] {
    check_device_ctx(ctx);
    require(n >= 0 && (n == 0 || v) && out, FECX_ERR_ARG, "bad arguments");
    const int np = std::max(fecx::vec_groups(n), 1);
    double* part = (double*)dev_atleast(ctx, "vn_part", sizeof(double) * fecx::CG_PARTS);
    double* res = (double*)dev_atleast(ctx, "vn_res", sizeof(double));
    fecx::sumsq_kernel<<<(unsigned)np, fecx::SV_THREADS, 0, ctx->stream>>>(n, v, part);
    fecx::sum_kernel<<<1, fecx::SV_THREADS, 0, ctx->stream>>>(part, np, res);
    HIPCHK(hipGetLastError());
    double h = 0.0;
    HIPCHK(hipMemcpyAsync(&h, res, sizeof(double), hipMemcpyDeviceToHost, ctx->stream));
    HIPCHK(hipStreamSynchronize(ctx->stream));
    *out = std::sqrt(h);
  });
}

int fecx_vector_axpy(fecx_ctx* ctx, int64_t n, double a, const double* x, double* y) {
  return guard(ctx, [&] {
    check_device_ctx(ctx);
    require(n >= 0 && (n == 0 || (x && y)), FECX_ERR_ARG, "bad arguments");
    if (n > 0) fecx::axpy_kernel<<<(unsigned)((n + 255) / 256), 256, 0, ctx->stream>>>(n, a, x, y);
    HIPCHK(hipGetLastError());
    HIPCHK(hipStreamSynchronize(ctx->stream));
  });
}

}  // extern "C"
