// Kernels of the device linear solve (GMRES preconditioned by aggregation
// multigrid or by node block-Jacobi) that stands in for goal's Belos/MueLu
// solve (src/goal_linear_solve.cpp:22-90).  FP64; every reduction has a fixed
// order, so a solve is bitwise reproducible.

#include "goal_kernels.hpp"

namespace goal {
namespace {

constexpr int kSolveThreads = 256;

// ------------------------------------------------- products with a matrix
// What a product is for: y = A x, y = b - A x, or a Chebyshev step of the
// block-Jacobi smoother, r = b - A x, d = c1 d + c2 Binv r, y = x + d (y other
// than x: other rows still read x; with c1 = 0 d is not read).
enum ProductKind { PRODUCT, RESIDUAL, SMOOTH };
struct ProductArgs {
  const double *x, *b, *binv;
  double c1, c2;
  double *d, *y;
};

// What a lane that ends row i of a node needs beside the sums; loaded before
// them, so that the loads' latency is not added to the matrix's (SMOOTH on the
// P2 24^3 cube: 96 -> 91 us).
template <int KIND>
struct RowEnd {
  double b = 0.0, x = 0.0, d = 0.0, B[4] = {0.0, 0.0, 0.0, 0.0};
  __device__ inline void load(const ProductArgs& a, int64_t node, int i) {
    const int64_t k = 4 * node + i;
    if constexpr (KIND != PRODUCT) b = a.b[k];
    if constexpr (KIND == SMOOTH) {
      x = a.x[k];
      if (a.c1 != 0.0) d = a.d[k];
      for (int j = 0; j < 4; ++j) B[j] = a.binv[4 * k + j];
    }
  }
  // r: A x, b - A x or, of all four rows, the residual
  __device__ inline void store(const ProductArgs& a, int64_t node, int i, const double* r) const {
    const int64_t k = 4 * node + i;
    if constexpr (KIND == SMOOTH) {
      const double z = B[0] * r[0] + B[1] * r[1] + B[2] * r[2] + B[3] * r[3];
      const double dn = a.c1 * d + a.c2 * z;
      a.d[k] = dn;
      a.y[k] = x + dn;
    } else {
      a.y[k] = r[0];
    }
  }
};

// The finest level: scalar CSR whose rows come four to a node with the same
// columns, four to a neighbour.  L lanes take a node: each reads two columns of
// all four rows (four 16-byte loads in flight, every one coalesced) and two
// values of x; the neighbour's id comes from the node adjacency (4 bytes per
// 4 x 4 block).  Bound by HBM: the matrix is read once.  One wavefront per
// scalar row with the columns of every row took 230 us per product of the
// P2 24^3 cube (51 M values) against 75.
template <int L, int KIND>
__global__ __launch_bounds__(kSolveThreads) void node_product_kernel(int64_t nn, const int64_t* rp,
                                                                     const int32_t* adj, const double* vals,
                                                                     ProductArgs a) {
  const int l = threadIdx.x % L;
  const int64_t node = (int64_t)blockIdx.x * (kSolveThreads / L) + threadIdx.x / L;
  if (node >= nn) return;  // uniform per group of L lanes
  const int64_t base = rp[4 * node];
  const int len = (int)(rp[4 * node + 1] - base);
  const double* v = vals + base;
  const int32_t* nb = adj + base / 16;
  const int i = l / (L / 4);  // the row this lane holds in the end
  RowEnd<KIND> end;
  if (l % (L / 4) == 0) end.load(a, node, i);
  double s0 = 0.0, s1 = 0.0, s2 = 0.0, s3 = 0.0;
  for (int p = l; p < len / 2; p += L) {
    const double2 xc = *reinterpret_cast<const double2*>(a.x + 4 * (int64_t)nb[p >> 1] + 2 * (p & 1));
    const double2 v0 = *reinterpret_cast<const double2*>(v + 2 * p);
    const double2 v1 = *reinterpret_cast<const double2*>(v + len + 2 * p);
    const double2 v2 = *reinterpret_cast<const double2*>(v + 2 * len + 2 * p);
    const double2 v3 = *reinterpret_cast<const double2*>(v + 3 * (int64_t)len + 2 * p);
    s0 += v0.x * xc.x + v0.y * xc.y;
    s1 += v1.x * xc.x + v1.y * xc.y;
    s2 += v2.x * xc.x + v2.y * xc.y;
    s3 += v3.x * xc.x + v3.y * xc.y;
  }
  // four sums over L lanes: halve the rows a lane holds twice, then the lanes
  const bool h = l & (L / 2), q = l & (L / 4);
  double t0 = h ? s2 : s0, t1 = h ? s3 : s1;
  t0 += __shfl_xor(h ? s0 : s2, L / 2, 64);
  t1 += __shfl_xor(h ? s1 : s3, L / 2, 64);
  double t = q ? t1 : t0;
  t += __shfl_xor(q ? t0 : t1, L / 4, 64);
  for (int off = L / 8; off > 0; off >>= 1) t += __shfl_xor(t, off, 64);
  double r[4] = {t, 0.0, 0.0, 0.0};
  if constexpr (KIND != PRODUCT) r[0] = t = end.b - t;
  if constexpr (KIND == SMOOTH)
    for (int j = 0; j < 4; ++j) r[j] = __shfl(t, (threadIdx.x & 63) / L * L + j * (L / 4), 64);
  if (l % (L / 4) == 0) end.store(a, node, i, r);
}

// Gauss-Jordan inverse with partial pivoting of the 4x4 block in M[:, 0:4]
// (M[:, 4:8] holds the identity); writes it to out, or the identity and
// status bit 0 for a zero pivot.
__device__ inline void invert4(double (&M)[4][8], double* out, int* status) {
  bool ok = true;
  for (int c = 0; c < 4; ++c) {
    int p = c;
    for (int r = c + 1; r < 4; ++r)
      if (fabs(M[r][c]) > fabs(M[p][c])) p = r;
    if (M[p][c] == 0.0) {
      ok = false;
      break;
    }
    if (p != c)
      for (int j = 0; j < 8; ++j) {
        const double t = M[c][j];
        M[c][j] = M[p][j];
        M[p][j] = t;
      }
    const double inv = 1.0 / M[c][c];
    for (int j = 0; j < 8; ++j) M[c][j] *= inv;
    for (int r = 0; r < 4; ++r)
      if (r != c) {
        const double f = M[r][c];
        for (int j = 0; j < 8; ++j) M[r][j] -= f * M[c][j];
      }
  }
  for (int i = 0; i < 4; ++i)
    for (int j = 0; j < 4; ++j) out[4 * i + j] = ok ? M[i][4 + j] : (i == j ? 1.0 : 0.0);
  if (!ok) atomicOr(status, 1);
}

// Inverse of each node's 4x4 diagonal block.  The block's columns 4a..4a+3
// sit contiguously in each of the node's rows.
__global__ __launch_bounds__(kSolveThreads) void block_inverse_kernel(int64_t nn, const int64_t* rp,
                                                                      const int32_t* cols, const double* vals,
                                                                      double* binv, int* status) {
  const int64_t a = (int64_t)blockIdx.x * kSolveThreads + threadIdx.x;
  if (a >= nn) return;
  double M[4][8];
  for (int i = 0; i < 4; ++i) {
    const int64_t row = 4 * a + i;
    int64_t lo = rp[row], hi = rp[row + 1];
    const int32_t c0 = (int32_t)(4 * a);
    while (lo < hi) {  // first column >= 4a
      const int64_t mid = (lo + hi) >> 1;
      if (cols[mid] < c0) lo = mid + 1;
      else hi = mid;
    }
    for (int j = 0; j < 4; ++j) {
      const int64_t k = lo + j;
      M[i][j] = (k < rp[row + 1] && cols[k] == c0 + j) ? vals[k] : 0.0;
      M[i][4 + j] = (i == j) ? 1.0 : 0.0;
    }
  }
  invert4(M, binv + 16 * a, status);
}

// ---------------------------------------------------- aggregation multigrid
// Coarse levels are node-block CSR (BSR) matrices: block k (row node a,
// column node bcol[k]) holds its 4x4 values row-major at bval[16 k].

// Inverse of each diagonal block of a BSR matrix (missing: identity, status 1).
__global__ __launch_bounds__(kSolveThreads) void bsr_block_inverse_kernel(int64_t nb, const int64_t* bptr,
                                                                          const int32_t* bcol, const double* bval,
                                                                          double* binv, int* status) {
  const int64_t a = (int64_t)blockIdx.x * kSolveThreads + threadIdx.x;
  if (a >= nb) return;
  int64_t lo = bptr[a], hi = bptr[a + 1];
  while (lo < hi) {
    const int64_t mid = (lo + hi) >> 1;
    if (bcol[mid] < a) lo = mid + 1;
    else hi = mid;
  }
  const bool has = lo < bptr[a + 1] && bcol[lo] == a;
  double M[4][8];
  for (int i = 0; i < 4; ++i)
    for (int j = 0; j < 4; ++j) {
      M[i][j] = has ? bval[16 * lo + 4 * i + j] : 0.0;
      M[i][4 + j] = (i == j) ? 1.0 : 0.0;
    }
  invert4(M, binv + 16 * a, status);
}

// Coarse levels: 16 lanes take a block row, lane 4 k + i the row i of every
// fourth block.
template <int KIND>
__global__ __launch_bounds__(kSolveThreads) void bsr_product_kernel(int64_t nb, const int64_t* bptr,
                                                                    const int32_t* bcol, const double* bval,
                                                                    ProductArgs a) {
  const int l = threadIdx.x & 15, i = l & 3;
  const int64_t node = (int64_t)blockIdx.x * (kSolveThreads / 16) + threadIdx.x / 16;
  if (node >= nb) return;  // uniform per group of 16 lanes
  RowEnd<KIND> end;
  if (l < 4) end.load(a, node, i);
  double t = 0.0;
  for (int64_t k = bptr[node] + (l >> 2); k < bptr[node + 1]; k += 4) {
    const double2* v = reinterpret_cast<const double2*>(bval + 16 * k + 4 * i);
    const double2* xc = reinterpret_cast<const double2*>(a.x + 4 * (int64_t)bcol[k]);
    const double2 v0 = v[0], v1 = v[1], x0 = xc[0], x1 = xc[1];
    t += v0.x * x0.x + v0.y * x0.y + v1.x * x1.x + v1.y * x1.y;
  }
  t += __shfl_xor(t, 4, 64);
  t += __shfl_xor(t, 8, 64);
  double r[4] = {t, 0.0, 0.0, 0.0};
  if constexpr (KIND != PRODUCT) r[0] = t = end.b - t;
  if constexpr (KIND == SMOOTH)
    for (int j = 0; j < 4; ++j) r[j] = __shfl(t, (threadIdx.x & 48) + j, 64);
  if (l < 4) end.store(a, node, i, r);
}

// Galerkin sum P^T A P of the plain-aggregation prolongator: coarse block s,
// entry e, is the sum of entry e of the fine blocks gidx[gptr[s]..gptr[s+1])
// in list order.  Fine blocks of the finest level live in the scalar CSR
// (brow: each block's row node; its 4 rows start at rp[4 a] and are 4 deg(a)
// long, block k is columns 4 (k - rp[4 a] / 16) ..); others are BSR.
__global__ __launch_bounds__(kSolveThreads) void galerkin_kernel(int64_t ncb, const int64_t* gptr,
                                                                 const int64_t* gidx, const int32_t* brow,
                                                                 const int64_t* rp, const double* fvals,
                                                                 double* cvals) {
  const int64_t t = (int64_t)blockIdx.x * kSolveThreads + threadIdx.x;
  if (t >= 16 * ncb) return;
  const int64_t sidx = t >> 4;
  const int e = (int)(t & 15), i = e >> 2, j = e & 3;
  double sum = 0.0;
  for (int64_t p = gptr[sidx]; p < gptr[sidx + 1]; ++p) {
    const int64_t k = gidx[p];
    if (brow) {
      const int64_t a = brow[k];
      const int64_t base = rp[4 * a], len = rp[4 * a + 1] - base;  // 4 deg(a)
      sum += fvals[base + i * len + 4 * (k - base / 16) + j];
    } else {
      sum += fvals[16 * k + e];
    }
  }
  cvals[16 * sidx + e] = sum;
}

// bc[A] = sum of r over the aggregate's nodes (P^T r): 16 lanes per aggregate,
// lane 4 k + i entry i of every fourth node.
__global__ __launch_bounds__(kSolveThreads) void restrict_kernel(int64_t nc, const int64_t* aptr,
                                                                 const int32_t* amem, const double* r,
                                                                 double* bc) {
  const int l = threadIdx.x & 15, i = l & 3;
  const int64_t A = (int64_t)blockIdx.x * (kSolveThreads / 16) + threadIdx.x / 16;
  if (A >= nc) return;  // uniform per group of 16 lanes
  double s = 0.0;
  for (int64_t m = aptr[A] + (l >> 2); m < aptr[A + 1]; m += 4) s += r[4 * (int64_t)amem[m] + i];
  s += __shfl_xor(s, 4, 64);
  s += __shfl_xor(s, 8, 64);
  if (l < 4) bc[4 * A + i] = s;
}

// x += P xc: each node takes its aggregate's correction.
__global__ __launch_bounds__(kSolveThreads) void prolong_kernel(int64_t nf, const int32_t* agg, const double* xc,
                                                                double* x) {
  const int64_t t = (int64_t)blockIdx.x * kSolveThreads + threadIdx.x;
  if (t >= 4 * nf) return;
  x[t] += xc[4 * (int64_t)agg[t >> 2] + (t & 3)];
}

// The first Chebyshev step from x = 0: d = x = c2 Binv b.
__global__ __launch_bounds__(kSolveThreads) void smooth_start_kernel(int64_t nn, const double* binv, const double* b,
                                                                     double c2, double* d, double* x) {
  const int64_t k = (int64_t)blockIdx.x * kSolveThreads + threadIdx.x;
  if (k >= 4 * nn) return;
  const double* B = binv + 4 * k;
  const double* r = b + k / 4 * 4;
  const double v = c2 * (B[0] * r[0] + B[1] * r[1] + B[2] * r[2] + B[3] * r[3]);
  d[k] = v;
  x[k] = v;
}

// y = M x for a dense row-major n x n matrix (the coarsest level's inverse),
// one wavefront per row.
__global__ __launch_bounds__(kSolveThreads) void dense_matvec_kernel(int n, const double* M, const double* x,
                                                                     double* y) {
  const int lane = threadIdx.x & 63, i = blockIdx.x * (kSolveThreads / 64) + (threadIdx.x >> 6);
  if (i >= n) return;  // uniform per wave
  double s = 0.0;
  for (int j = lane; j < n; j += 64) s += M[(int64_t)i * n + j] * x[j];
  for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off, 64);
  if (lane == 0) y[i] = s;
}

// y = Binv x, node by node.
__global__ __launch_bounds__(kSolveThreads) void block_apply_kernel(int64_t nn, const double* binv,
                                                                    const double* x, double* y) {
  const int64_t a = (int64_t)blockIdx.x * kSolveThreads + threadIdx.x;
  if (a >= nn) return;
  const double* B = binv + 16 * a;
  const double x0 = x[4 * a], x1 = x[4 * a + 1], x2 = x[4 * a + 2], x3 = x[4 * a + 3];
  for (int i = 0; i < 4; ++i) y[4 * a + i] = B[4 * i] * x0 + B[4 * i + 1] * x1 + B[4 * i + 2] * x2 + B[4 * i + 3] * x3;
}

// partial[j][block] = sum over the block's slice of V_j . w, j < k.  The
// vectors go eight at a time, one group of eight per grid row: each row's w is
// read once per eight vectors, the eight loads of a row are independent, and
// the groups run beside each other.
constexpr int kDotGroup = 8;

__global__ __launch_bounds__(kSolveThreads) void multi_dot_partial_kernel(int64_t n, int k, const double* V,
                                                                          int64_t ldv, const double* w,
                                                                          double* partial, DgksTest test) {
  if (!test.again()) return;
  __shared__ double red[kSolveThreads / 64][kDotGroup];
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const int64_t stride = (int64_t)gridDim.x * kSolveThreads;
  const int j0 = blockIdx.y * kDotGroup, nj = min(kDotGroup, k - j0);
  double s[kDotGroup];
#pragma unroll
  for (int jj = 0; jj < kDotGroup; ++jj) s[jj] = 0.0;
  for (int64_t i = (int64_t)blockIdx.x * kSolveThreads + tid; i < n; i += stride) {
    const double wi = w[i];
#pragma unroll
    for (int jj = 0; jj < kDotGroup; ++jj)
      if (jj < nj) s[jj] += V[(int64_t)(j0 + jj) * ldv + i] * wi;
  }
#pragma unroll
  for (int jj = 0; jj < kDotGroup; ++jj) {
    double t = s[jj];
    for (int off = 32; off > 0; off >>= 1) t += __shfl_down(t, off, 64);
    if (lane == 0) red[wv][jj] = t;
  }
  __syncthreads();
  if (tid < nj) {
    double t = 0.0;
    for (int q = 0; q < kSolveThreads / 64; ++q) t += red[q][tid];
    partial[(int64_t)(j0 + tid) * gridDim.x + blockIdx.x] = t;
  }
}

// out[j] = sum_b partial[j][b], one block per j.
__global__ __launch_bounds__(kSolveThreads) void multi_dot_final_kernel(int nb, const double* partial, double* out,
                                                                        DgksTest test) {
  if (!test.again()) return;
  __shared__ double red[kSolveThreads / 64];
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, j = blockIdx.x;
  double s = 0.0;
  for (int b = tid; b < nb; b += kSolveThreads) s += partial[(int64_t)j * nb + b];
  for (int off = 32; off > 0; off >>= 1) s += __shfl_down(s, off, 64);
  if (lane == 0) red[wv] = s;
  __syncthreads();
  if (tid == 0) {
    double t = 0.0;
    for (int q = 0; q < kSolveThreads / 64; ++q) t += red[q];
    out[j] = t;
  }
}

// w += sign * sum_j c_j V_j, j < k.
__global__ __launch_bounds__(kSolveThreads) void multi_axpy_kernel(int64_t n, int k, const double* V, int64_t ldv,
                                                                   const double* c, double sign, double* w,
                                                                   DgksTest test) {
  const int64_t i = (int64_t)blockIdx.x * kSolveThreads + threadIdx.x;
  if (i >= n || !test.again()) return;
  double s = 0.0;
  for (int j = 0; j < k; ++j) s += c[j] * V[(int64_t)j * ldv + i];
  w[i] += sign * s;
}

// w /= |w| (as it is where |w| = 0), with |w|^2 already on the device, so the
// next step can be queued before the host has seen the norm.  Block 0 hands
// what the host needs (k1 + k2 coefficients, both squared norms) to its
// pinned memory.
__global__ __launch_bounds__(kSolveThreads) void arnoldi_end_kernel(int64_t n, double* w, const double* norms,
                                                                    const double* h1, int k1, const double* h2, int k2,
                                                                    double* host) {
  const double hn = sqrt(norms[1]);
  if (blockIdx.x == 0 && host) {
    for (int j = threadIdx.x; j < k1; j += kSolveThreads) host[2 + j] = h1[j];
    for (int j = threadIdx.x; j < k2; j += kSolveThreads) host[2 + k1 + j] = h2[j];
    if (threadIdx.x < 2) host[threadIdx.x] = norms[threadIdx.x];
    __threadfence_system();
  }
  const int64_t i = (int64_t)blockIdx.x * kSolveThreads + threadIdx.x;
  if (i < n && hn > 0.0) w[i] = (1.0 / hn) * w[i];
}

// splitmix64 (goal_mesh.hpp), on the device
__device__ inline uint64_t device_splitmix64(uint64_t x) {
  x += 0x9E3779B97F4A7C15ull;
  x = (x ^ (x >> 30)) * 0xBF58476D1CE4E5B9ull;
  x = (x ^ (x >> 27)) * 0x94D049BB133111EBull;
  return x ^ (x >> 31);
}

// The start vector of the smoother's Arnoldi steps: fixed noise in [-1/2, 1/2).
__global__ __launch_bounds__(kSolveThreads) void arnoldi_start_kernel(int64_t n, double* q) {
  const int64_t i = (int64_t)blockIdx.x * kSolveThreads + threadIdx.x;
  if (i < n) q[i] = (double)(device_splitmix64(0xA3C5u + (uint64_t)i) >> 11) * (1.0 / 9007199254740992.0) - 0.5;
}

// y = a * x  (y may alias x)
__global__ __launch_bounds__(kSolveThreads) void scale_kernel(int64_t n, double a, const double* x, double* y) {
  const int64_t i = (int64_t)blockIdx.x * kSolveThreads + threadIdx.x;
  if (i < n) y[i] = a * x[i];
}

dim3 grid_for(int64_t n) { return dim3((unsigned)((n + kSolveThreads - 1) / kSolveThreads)); }

}  // namespace

int multi_dot_blocks(int64_t n) {
  const int64_t b = (n + 4 * kSolveThreads - 1) / (4 * kSolveThreads);  // four rows a thread and more
  return (int)std::min<int64_t>(std::max<int64_t>(b, 1), 1024);
}

namespace {
// Lanes per node: a node's row pairs fit the group for most nodes (P1: 15
// neighbours, 30 pairs; P2: 28 on average, 57).
template <int KIND>
hipError_t node_product(int64_t nn, int64_t nnz, const int64_t* rp, const int32_t* adj, const double* vals,
                        const ProductArgs& a, hipStream_t s) {
  if (nn == 0) return hipSuccess;
  if (nnz / (8 * nn) <= 40) {
    hipLaunchKernelGGL((node_product_kernel<32, KIND>), dim3((unsigned)((nn + kSolveThreads / 32 - 1) / (kSolveThreads / 32))),
                       dim3(kSolveThreads), 0, s, nn, rp, adj, vals, a);
  } else {
    hipLaunchKernelGGL((node_product_kernel<64, KIND>), dim3((unsigned)((nn + kSolveThreads / 64 - 1) / (kSolveThreads / 64))),
                       dim3(kSolveThreads), 0, s, nn, rp, adj, vals, a);
  }
  return hipGetLastError();
}
template <int KIND>
hipError_t bsr_product(int64_t nb, const int64_t* bptr, const int32_t* bcol, const double* bval, const ProductArgs& a,
                       hipStream_t s) {
  if (nb == 0) return hipSuccess;
  hipLaunchKernelGGL(bsr_product_kernel<KIND>, grid_for(16 * nb), dim3(kSolveThreads), 0, s, nb, bptr, bcol, bval, a);
  return hipGetLastError();
}
}  // namespace

hipError_t launch_product(const MatrixRef& A, const double* x, const double* b, double* y, hipStream_t s) {
  const ProductArgs a{x, b, nullptr, 0.0, 0.0, nullptr, y};
  if (A.adj) return b ? node_product<RESIDUAL>(A.nn, A.nnz, A.ptr, A.adj, A.vals, a, s)
                      : node_product<PRODUCT>(A.nn, A.nnz, A.ptr, A.adj, A.vals, a, s);
  return b ? bsr_product<RESIDUAL>(A.nn, A.ptr, A.bcol, A.vals, a, s)
           : bsr_product<PRODUCT>(A.nn, A.ptr, A.bcol, A.vals, a, s);
}

hipError_t launch_smooth(const MatrixRef& A, const double* binv, const double* b, const double* x, double c1,
                         double c2, double* d, double* y, hipStream_t s) {
  const ProductArgs a{x, b, binv, c1, c2, d, y};
  return A.adj ? node_product<SMOOTH>(A.nn, A.nnz, A.ptr, A.adj, A.vals, a, s)
               : bsr_product<SMOOTH>(A.nn, A.ptr, A.bcol, A.vals, a, s);
}

hipError_t launch_smooth_start(int64_t nn, const double* binv, const double* b, double c2, double* d, double* x,
                               hipStream_t s) {
  if (nn == 0) return hipSuccess;
  hipLaunchKernelGGL(smooth_start_kernel, grid_for(4 * nn), dim3(kSolveThreads), 0, s, nn, binv, b, c2, d, x);
  return hipGetLastError();
}

hipError_t launch_block_inverse(int64_t nn, const int64_t* rp, const int32_t* cols, const double* vals,
                                double* binv, int* status, hipStream_t s) {
  if (nn == 0) return hipSuccess;
  hipLaunchKernelGGL(block_inverse_kernel, grid_for(nn), dim3(kSolveThreads), 0, s, nn, rp, cols, vals, binv, status);
  return hipGetLastError();
}

hipError_t launch_bsr_block_inverse(int64_t nb, const int64_t* bptr, const int32_t* bcol, const double* bval,
                                    double* binv, int* status, hipStream_t s) {
  if (nb == 0) return hipSuccess;
  hipLaunchKernelGGL(bsr_block_inverse_kernel, grid_for(nb), dim3(kSolveThreads), 0, s, nb, bptr, bcol, bval, binv,
                     status);
  return hipGetLastError();
}

hipError_t launch_galerkin(int64_t ncb, const int64_t* gptr, const int64_t* gidx, const int32_t* brow,
                           const int64_t* rp, const double* fvals, double* cvals, hipStream_t s) {
  if (ncb == 0) return hipSuccess;
  hipLaunchKernelGGL(galerkin_kernel, grid_for(16 * ncb), dim3(kSolveThreads), 0, s, ncb, gptr, gidx, brow, rp, fvals,
                     cvals);
  return hipGetLastError();
}

hipError_t launch_restrict(int64_t nc, const int64_t* aptr, const int32_t* amem, const double* r, double* bc,
                           hipStream_t s) {
  if (nc == 0) return hipSuccess;
  hipLaunchKernelGGL(restrict_kernel, grid_for(16 * nc), dim3(kSolveThreads), 0, s, nc, aptr, amem, r, bc);
  return hipGetLastError();
}

hipError_t launch_prolong(int64_t nf, const int32_t* agg, const double* xc, double* x, hipStream_t s) {
  if (nf == 0) return hipSuccess;
  hipLaunchKernelGGL(prolong_kernel, grid_for(4 * nf), dim3(kSolveThreads), 0, s, nf, agg, xc, x);
  return hipGetLastError();
}

hipError_t launch_dense_matvec(int n, const double* M, const double* x, double* y, hipStream_t s) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(dense_matvec_kernel, grid_for(64 * (int64_t)n), dim3(kSolveThreads), 0, s, n, M, x, y);
  return hipGetLastError();
}

hipError_t launch_block_apply(int64_t nn, const double* binv, const double* x, double* y, hipStream_t s) {
  if (nn == 0) return hipSuccess;
  hipLaunchKernelGGL(block_apply_kernel, grid_for(nn), dim3(kSolveThreads), 0, s, nn, binv, x, y);
  return hipGetLastError();
}

hipError_t launch_multi_dot(int64_t n, int k, const double* V, int64_t ldv, const double* w, double* partial,
                            double* out, hipStream_t s, DgksTest test) {
  if (k == 0) return hipSuccess;
  const int nb = multi_dot_blocks(n);
  hipLaunchKernelGGL(multi_dot_partial_kernel, dim3(nb, (k + kDotGroup - 1) / kDotGroup), dim3(kSolveThreads), 0, s, n, k, V, ldv, w, partial, test);
  hipLaunchKernelGGL(multi_dot_final_kernel, dim3(k), dim3(kSolveThreads), 0, s, nb, partial, out, test);
  return hipGetLastError();
}

hipError_t launch_multi_axpy(int64_t n, int k, const double* V, int64_t ldv, const double* c, double sign, double* w,
                             hipStream_t s, DgksTest test) {
  if (n == 0 || k == 0) return hipSuccess;
  hipLaunchKernelGGL(multi_axpy_kernel, grid_for(n), dim3(kSolveThreads), 0, s, n, k, V, ldv, c, sign, w, test);
  return hipGetLastError();
}

hipError_t launch_arnoldi_end(int64_t n, double* w, const double* norms, const double* h1, int k1, const double* h2,
                              int k2, double* host, hipStream_t s) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(arnoldi_end_kernel, grid_for(n), dim3(kSolveThreads), 0, s, n, w, norms, h1, k1, h2, k2, host);
  return hipGetLastError();
}

hipError_t launch_arnoldi_start(int64_t n, double* q, hipStream_t s) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(arnoldi_start_kernel, grid_for(n), dim3(kSolveThreads), 0, s, n, q);
  return hipGetLastError();
}

hipError_t launch_scale(int64_t n, double a, const double* x, double* y, hipStream_t s) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(scale_kernel, grid_for(n), dim3(kSolveThreads), 0, s, n, a, x, y);
  return hipGetLastError();
}

}  // namespace goal
