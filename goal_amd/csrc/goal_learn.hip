// Learned element error indicator: per-element features of a primal state
// and a 12 -> 64 -> 64 -> 1 ReLU network (BF16 weights, FP32 biases and
// accumulation) with its forward pass, mean-squared-error gradient and Adam
// update.  The network predicts log10(eta_E / E) where eta_E is the nested-
// adjoint indicator of Nested::set_error (src/goal_nested.cpp:395-412); it
// has no counterpart in the reference.
//
// Every reduction runs in a fixed order (per-block partial sums, then one
// ordered pass), so a training run is bitwise reproducible.

#include "goal_kernels.hpp"

namespace goal {
namespace {

constexpr int kIn = kMlpIn, kHid = kMlpHidden;
constexpr int oW1 = kMlpOffW1, oB1 = kMlpOffB1, oW2 = kMlpOffW2, oB2 = kMlpOffB2, oW3 = kMlpOffW3,
              oB3 = kMlpOffB3, kP = kMlpParams;

// ------------------------------------------------------------- features

constexpr int kFeatThreads = 256;

__device__ inline double tet_volume(const double* X, const int32_t* v) {
  const double* a = X + 3 * v[0];
  const double* b = X + 3 * v[1];
  const double* c = X + 3 * v[2];
  const double* d = X + 3 * v[3];
  const double e1[3] = {b[0] - a[0], b[1] - a[1], b[2] - a[2]};
  const double e2[3] = {c[0] - a[0], c[1] - a[1], c[2] - a[2]};
  const double e3[3] = {d[0] - a[0], d[1] - a[1], d[2] - a[2]};
  return (e1[0] * (e2[1] * e3[2] - e2[2] * e3[1]) - e1[1] * (e2[0] * e3[2] - e2[2] * e3[0]) +
          e1[2] * (e2[0] * e3[1] - e2[1] * e3[0])) /
         6.0;
}

// Reference-configuration gradient of the vertex-interpolated displacement:
// H[i][j] = sum_k (U[k+1][i] - U[0][i]) Ji[j][k], Ji the inverse of the
// matrix whose rows are the edges 01, 02, 03.
__device__ inline void linear_grad(const double X[4][3], const double U[4][3], double H[9]) {
  double J[3][3];
  for (int r = 0; r < 3; ++r)
    for (int c = 0; c < 3; ++c) J[r][c] = X[r + 1][c] - X[0][c];
  const double det = J[0][0] * (J[1][1] * J[2][2] - J[1][2] * J[2][1]) -
                     J[0][1] * (J[1][0] * J[2][2] - J[1][2] * J[2][0]) +
                     J[0][2] * (J[1][0] * J[2][1] - J[1][1] * J[2][0]);
  double Ji[3][3];
  Ji[0][0] = (J[1][1] * J[2][2] - J[1][2] * J[2][1]) / det;
  Ji[0][1] = (J[0][2] * J[2][1] - J[0][1] * J[2][2]) / det;
  Ji[0][2] = (J[0][1] * J[1][2] - J[0][2] * J[1][1]) / det;
  Ji[1][0] = (J[1][2] * J[2][0] - J[1][0] * J[2][2]) / det;
  Ji[1][1] = (J[0][0] * J[2][2] - J[0][2] * J[2][0]) / det;
  Ji[1][2] = (J[0][2] * J[1][0] - J[0][0] * J[1][2]) / det;
  Ji[2][0] = (J[1][0] * J[2][1] - J[1][1] * J[2][0]) / det;
  Ji[2][1] = (J[0][1] * J[2][0] - J[0][0] * J[2][1]) / det;
  Ji[2][2] = (J[0][0] * J[1][1] - J[0][1] * J[1][0]) / det;
  for (int i = 0; i < 3; ++i)
    for (int j = 0; j < 3; ++j) {
      double s = 0.0;
      for (int k = 0; k < 3; ++k) s += (U[k + 1][i] - U[0][i]) * Ji[j][k];
      H[3 * i + j] = s;
    }
}

__device__ inline void load_vertices(const FeatureArgs& a, int64_t e, double X[4][3], double U[4][3]) {
  const int32_t* v = a.conn + e * a.npe;
  for (int i = 0; i < 4; ++i)
    for (int c = 0; c < 3; ++c) {
      X[i][c] = a.coords[3 * (int64_t)v[i] + c];
      U[i][c] = a.x[4 * (int64_t)v[i] + c];
    }
}

// Per element, into its row of elem_scratch: the von Mises integral, grad u and
// the volume, all that the recovery reads of it.  A wave's rows go out through
// LDS as one run: 53 us for 1.97 M tets, where each lane's own stores, 80 bytes
// apart, took 70.
constexpr int kRow = kFeatElem, kRowH = 1, kRowVol = 10;
static_assert(kRowVol < kRow && kRow <= 16 && kRow % 2 == 0, "one lane of sixteen per value, stored in pairs");
__global__ __launch_bounds__(kFeatThreads) void elem_geometry_kernel(FeatureArgs a) {
  __shared__ double stage[kFeatThreads / 64][64 * (kRow + 1)];
  const int64_t e = (int64_t)blockIdx.x * kFeatThreads + threadIdx.x;
  const int lane = threadIdx.x & 63;
  double* w = stage[threadIdx.x >> 6];
  if (e < a.num_elems) {
    double X[4][3], U[4][3], H[9];
    load_vertices(a, e, X, U);
    linear_grad(X, U, H);
    double* o = w + (kRow + 1) * lane;  // odd: the rows spread over the banks
    o[0] = a.elem_vm[e];
    for (int k = 0; k < 9; ++k) o[kRowH + k] = H[k];
    o[kRowVol] = tet_volume(a.coords, a.conn + e * a.npe);
    for (int k = kRowVol + 1; k < kRow; ++k) o[k] = 0.0;
  }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  const int64_t e0 = e - lane;
#pragma unroll
  for (int j = 0; j < kRow / 2; ++j) {
    const int i = (64 * j + lane) / (kRow / 2), k = 2 * ((64 * j + lane) % (kRow / 2));
    if (e0 + i < a.num_elems)
      reinterpret_cast<double2*>(a.elem_scratch + kRow * e0)[64 * j + lane] =
          double2{w[(kRow + 1) * i + k], w[(kRow + 1) * i + k + 1]};
  }
}

// Volume-weighted nodal means of the element von Mises stress and of grad u:
// node_scratch[n] = (sum int_e vm, sum |e| H_e) / sum |e| over the incident
// elements in ascending order.
// Sixteen lanes per node, one per value of an element's row, so a row comes as
// one run of one or two lines, and a node's elements four at a time; each sum
// keeps its order.  Bound by the lines the L2 delivers (about 36 a node).  1.97 M
// tets (343 K nodes): 106 us; with the von Mises integrals apart and 80-byte rows
// (2.6 lines an element) 184; with one thread per node 345.
__global__ __launch_bounds__(kFeatThreads) void recover_kernel(FeatureArgs a) {
  constexpr int kAhead = 4;
  const int c = threadIdx.x & 15;
  const int64_t n = (int64_t)blockIdx.x * (kFeatThreads / 16) + threadIdx.x / 16;
  if (n >= a.num_nodes) return;  // uniform per group of 16 lanes
  const int64_t k0 = a.inc_ptr[n], k1 = a.inc_ptr[n + 1];
  double s = 0.0;
  for (int64_t kb = k0; kb < k1; kb += 16) {  // sixteen incidences, one a lane
    const int32_t r = a.inc[kb + c < k1 ? kb + c : k0];
    const int32_t mine = a.npe == 4 ? r / 4 : r / 10;
    const int m = (int)(k1 - kb < 16 ? k1 - kb : 16);
    for (int j0 = 0; j0 < m; j0 += kAhead) {
      double x[kAhead];
#pragma unroll
      for (int j = 0; j < kAhead; ++j) {  // past the end: an element of this node again, not added
        const int64_t e = __shfl(mine, j0 + j, 16);  // by all sixteen: the source lane may be one without a value
        x[j] = c <= kRowVol ? a.elem_scratch[kRow * e + c] : 0.0;
      }
#pragma unroll
      for (int j = 0; j < kAhead; ++j) {
        const double vol = __shfl(x[j], kRowVol, 16);
        if (j0 + j < m) s += (c >= kRowH && c < kRowVol ? vol : 1.0) * x[j];
      }
    }
  }
  const double w = __shfl(s, kRowVol, 16);
  if (c < kRowVol) a.node_scratch[10 * n + c] = w > 0.0 ? s / w : 0.0;
}

__device__ inline float flog10(double v) { return (float)log10(v); }

// One element per thread.  Features (FP32):
//  0 log10 h (RMS edge length)        6 log10(vm / E + 1e-12)
//  1-3 centroid x, y, z               7 log10(|vm - vm*| / E + 1e-12)
//  4 log10(|x_c - qoi_x| + h)         8 log10(|grad u|_F + 1e-12)
//  5 1 if x_c < qoi_x else 0          9 log10(|grad u - (grad u)*|_F + 1e-12)
//                                     10 nu
//                                     11 log10(mean point eqps + 1e-9)
// vm is the element mean von Mises stress; a starred value is the mean over
// the element's four vertices of the recovered nodal value.  grad u uses the
// vertex displacements (linear interpolation).
__global__ __launch_bounds__(kFeatThreads) void features_kernel(FeatureArgs a) {
  const int64_t e = (int64_t)blockIdx.x * kFeatThreads + threadIdx.x;
  if (e >= a.num_elems) return;
  const int32_t* v = a.conn + e * a.npe;
  double X[4][3];
  for (int i = 0; i < 4; ++i)
    for (int c = 0; c < 3; ++c) X[i][c] = a.coords[3 * (int64_t)v[i] + c];
  const double* ge = a.elem_scratch + kRow * e;
  double star[10] = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
  for (int i = 0; i < 4; ++i) {
    const double* nv = a.node_scratch + 10 * (int64_t)v[i];
    for (int c = 0; c < 10; ++c) star[c] += 0.25 * nv[c];
  }
  double h2 = 0.0, d2 = 0.0;
  for (int k = 0; k < 9; ++k) {
    h2 += ge[kRowH + k] * ge[kRowH + k];
    d2 += (ge[kRowH + k] - star[1 + k]) * (ge[kRowH + k] - star[1 + k]);
  }
  double l2 = 0.0;
  for (int k = 0; k < 6; ++k) {
    const int p = k < 3 ? 0 : (k < 5 ? 1 : 2);
    const int q = k < 3 ? k + 1 : (k < 5 ? k - 1 : 3);
    for (int c = 0; c < 3; ++c) l2 += (X[p][c] - X[q][c]) * (X[p][c] - X[q][c]);
  }
  const double h = sqrt(l2 / 6.0);
  double xc[3];
  for (int c = 0; c < 3; ++c) xc[c] = 0.25 * (X[0][c] + X[1][c] + X[2][c] + X[3][c]);
  const MatParams m = a.mats[a.elem_set[e]];
  const double E = 9.0 * m.kappa * m.mu / (3.0 * m.kappa + m.mu);
  const double nu = (3.0 * m.kappa - 2.0 * m.mu) / (2.0 * (3.0 * m.kappa + m.mu));
  const double vm = ge[0] / ge[kRowVol];
  double eq = 0.0;
  if (a.eqps) {
    for (int q = 0; q < a.nq; ++q) eq += a.eqps[e * a.nq + q];
    eq /= a.nq;
  }
  float* f = a.feat + e * kIn;
  f[0] = flog10(h);
  f[1] = (float)xc[0];
  f[2] = (float)xc[1];
  f[3] = (float)xc[2];
  f[4] = flog10(fabs(xc[0] - a.qoi_x) + h);
  f[5] = xc[0] < a.qoi_x ? 1.0f : 0.0f;
  f[6] = flog10(fabs(vm) / E + 1e-12);
  f[7] = flog10(fabs(vm - star[0]) / E + 1e-12);
  f[8] = flog10(sqrt(h2) + 1e-12);
  f[9] = flog10(sqrt(d2) + 1e-12);
  f[10] = (float)nu;
  f[11] = flog10(eq + 1e-9);
}

// ---------------------------------------------------------------- network

__device__ inline float bf16_to_f32(uint16_t b) { return __uint_as_float((uint32_t)b << 16); }

// Round to nearest, ties to even (finite inputs).
__device__ inline uint16_t f32_to_bf16(float f) {
  uint32_t u = __float_as_uint(f);
  u += 0x7fffu + ((u >> 16) & 1u);
  return (uint16_t)(u >> 16);
}

__device__ inline float round_bf16(float f) { return bf16_to_f32(f32_to_bf16(f)); }

// ---------------------------------------------------------- forward (MFMA)
//
// Layers 1 and 2 run on the matrix cores as v_mfma_f32_16x16x16_bf16 with the
// samples as the N dimension.  For lane l, r = l % 16 and q = l / 16:
//   A operand  lane holds A[r][4q + i]      (weights: output row r of a block)
//   B operand  lane holds B[4q + i][r]      (inputs of sample r)
//   C/D        lane holds D[4q + i][r]      i = 0..3
// so the D of a layer-1 row block is, after bias, ReLU and rounding, exactly
// the B operand of layer 2 for the matching K block: the activations never
// leave the registers.  All weights sit in registers for the whole launch.
// The inputs of each product (normalized features, layer-1 activations) are
// rounded to BF16; accumulation is FP32.
typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kFwdThreads = 256;
constexpr int kFwdWaves = kFwdThreads / 64;
constexpr int kFwdUnroll = 4;

__device__ inline f32x4 mfma16(bf16x4 a, bf16x4 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, c, 0, 0, 0);
}

// y[i] = s_y * net(bf16((x[i] - mu) * is)) + mu_y + c * x[i][0].  Rows with a
// feature outside the training box [lo, hi] are counted in *ood.
__global__ __launch_bounds__(kFwdThreads) void mlp_forward_kernel(MlpArgs a, const float* x, int64_t n, float* y,
                                                                  int* ood) {
  const int lane = threadIdx.x & 63, r = lane & 15, q = lane >> 4;
  // the BF16 weights, staged through LDS with coalesced loads; each wave
  // then reads its operand fragments from there
  __shared__ uint16_t sw[kP + 1];
  for (int i = threadIdx.x; i < kP; i += kFwdThreads) sw[i] = a.wq[i];
  __syncthreads();
  bf16x4 A1[4], A2[4][4];
  float b1[4][4], b2[4][4], w3[4][4];
  for (int mb = 0; mb < 4; ++mb) {
    for (int i = 0; i < 4; ++i) {
      const int k = 4 * q + i;
      A1[mb][i] = k < kIn ? (short)sw[oW1 + (16 * mb + r) * kIn + k] : (short)0;
      const int row = 16 * mb + 4 * q + i;   // D row held by this lane
      b1[mb][i] = a.params[oB1 + row];
      b2[mb][i] = a.params[oB2 + row];
      w3[mb][i] = bf16_to_f32(sw[oW3 + row]);
    }
    for (int kb = 0; kb < 4; ++kb)
      for (int i = 0; i < 4; ++i) A2[mb][kb][i] = (short)sw[oW2 + (16 * mb + r) * kHid + 16 * kb + 4 * q + i];
  }
  float mu[4], is[4], lo[4], hi[4];
  for (int i = 0; i < 4; ++i) {
    const int k = 4 * q + i;
    mu[i] = k < kIn ? a.norms[k] : 0.0f;
    is[i] = k < kIn ? a.norms[kIn + k] : 0.0f;
    lo[i] = k < kIn ? a.norms[kMlpOffLo + k] : 0.0f;
    hi[i] = k < kIn ? a.norms[kMlpOffHi + k] : 0.0f;
  }
  const float b3 = a.params[oB3], mu_y = a.norms[2 * kIn], s_y = a.norms[2 * kIn + 1], cx = a.norms[kMlpOffC];
  const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
  const int64_t tiles = (n + 15) / 16;
  const int64_t wave = (int64_t)blockIdx.x * kFwdWaves + (threadIdx.x >> 6);
  const int64_t stride = (int64_t)gridDim.x * kFwdWaves;
  int outside = 0;  // rows of this lane outside the box (lanes q == 0 only)
  // kFwdUnroll consecutive tiles per iteration: their feature loads are all
  // issued before the first product, so each wave keeps several in flight.
  for (int64_t t0 = wave * kFwdUnroll; t0 < tiles; t0 += stride * kFwdUnroll) {   // uniform per wave
    float v[kFwdUnroll][4];
#pragma unroll
    for (int u = 0; u < kFwdUnroll; ++u) {
      const int64_t smp = (t0 + u) * 16 + r;
#pragma unroll
      for (int i = 0; i < 4; ++i) v[u][i] = (4 * q + i < kIn && smp < n) ? x[smp * kIn + 4 * q + i] : 0.0f;
    }
#pragma unroll
    for (int u = 0; u < kFwdUnroll; ++u) {
      const int64_t smp = (t0 + u) * 16 + r;
      const bool live = smp < n;
      bf16x4 B1;
      int out = 0;
      for (int i = 0; i < 4; ++i) {
        const int k = 4 * q + i;
        if (k < kIn && live) out |= !(v[u][i] >= lo[i] && v[u][i] <= hi[i]);
        B1[i] = (short)f32_to_bf16(k < kIn ? (v[u][i] - mu[i]) * is[i] : 0.0f);
      }
      bf16x4 B2[4];
      for (int mb = 0; mb < 4; ++mb) {
        const f32x4 z = mfma16(A1[mb], B1, zero);
        for (int i = 0; i < 4; ++i) B2[mb][i] = (short)f32_to_bf16(fmaxf(z[i] + b1[mb][i], 0.0f));
      }
      float o = 0.0f;
      for (int mb = 0; mb < 4; ++mb) {
        f32x4 z = zero;
        for (int kb = 0; kb < 4; ++kb) z = mfma16(A2[mb][kb], B2[kb], z);
        for (int i = 0; i < 4; ++i) o += w3[mb][i] * fmaxf(z[i] + b2[mb][i], 0.0f);
      }
      // sum the four row groups of sample r (lanes r, r+16, r+32, r+48)
      o += __shfl_xor(o, 16, 64);
      o += __shfl_xor(o, 32, 64);
      out |= __shfl_xor(out, 16, 64);
      out |= __shfl_xor(out, 32, 64);
      // feature 0 of sample r is v[u][0] of lane r (q == 0)
      if (q == 0 && live) {
        y[smp] = (o + b3) * s_y + mu_y + cx * v[u][0];
        outside += out ? 1 : 0;
      }
    }
  }
  // one atomic per wave: a row-by-row count on a single address serializes
  for (int off = 32; off > 0; off >>= 1) outside += __shfl_xor(outside, off, 64);
  if (lane == 0 && outside && ood) atomicAdd(ood, outside);
}

// Gradient of L = (1/B) sum_i (net(x_i) - t_i)^2, t_i = (y_i - mu_y - c x_i0)/s_y, over
// rows idx[0..B), on the matrix cores in FP32 (v_mfma_f32_16x16x4_f32) with the
// samples in tiles of 16.  For lane l, r = l % 16 and q = l / 16:
//   A operand  lane holds A[r][q],  B operand  B[q][r],
//   C/D        lane holds D[4q + i][r]      i = 0..3
// Wave w of four owns the 16 hidden units 16 w ..: its rows of both layers, of
// both deltas and of all parameter gradients, whose sums stay in its registers
// over the block's tiles.  Activations and deltas pass between the waves
// through LDS ([unit][sample], one word of padding).  Each block writes its
// sums to partial[block][kP] and its loss sum to partial_loss[block].
// Bound by the latency of its few products and barriers, not by their number:
// 16 samples per block instead of 64 put 256 blocks on the chip at a batch of
// 4096, and all four waves work instead of one (116 -> 11 us; with the
// reduction and Adam in one kernel a step takes 15 us instead of 140).
constexpr int kTile = 16, kGradThreads = 256, kPad = kTile + 1;

__device__ inline f32x4 mfma4(float a, float b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }

__global__ __launch_bounds__(kGradThreads) void mlp_grad_kernel(MlpArgs a, const float* x, const float* y,
                                                                const int32_t* idx, int64_t B, float* partial,
                                                                float* partial_loss) {
  __shared__ uint16_t sw[kP + 1];
  __shared__ float xs[kTile][kIn + 1], tgt[kTile], os[4][kTile];
  __shared__ float h1s[kHid][kPad], d2s[kHid][kPad], d1s[kHid][kPad];
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, r = lane & 15, q = lane >> 4;
  for (int i = tid; i < kP; i += kGradThreads) sw[i] = a.wq[i];
  __syncthreads();
  // operand fragments: W1 and W2 by rows of this wave's units, W2 by columns
  float A1[3], A2[16], A2t[16], b1[4], b2[4], w3[4];
  for (int k = 0; k < 3; ++k) A1[k] = bf16_to_f32(sw[oW1 + (16 * w + r) * kIn + 4 * k + q]);
  for (int k = 0; k < 16; ++k) {
    A2[k] = bf16_to_f32(sw[oW2 + (16 * w + r) * kHid + 4 * k + q]);
    A2t[k] = bf16_to_f32(sw[oW2 + (4 * k + q) * kHid + 16 * w + r]);
  }
  for (int i = 0; i < 4; ++i) {
    const int unit = 16 * w + 4 * q + i;
    b1[i] = a.params[oB1 + unit];
    b2[i] = a.params[oB2 + unit];
    w3[i] = bf16_to_f32(sw[oW3 + unit]);
  }
  const float b3 = a.params[oB3], mu_y = a.norms[2 * kIn], s_y = a.norms[2 * kIn + 1], cx = a.norms[kMlpOffC];
  const float invB = 1.0f / (float)B;
  const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
  f32x4 g2[4] = {zero, zero, zero, zero}, g1 = zero;
  float gw3[4] = {0, 0, 0, 0}, gb1[4] = {0, 0, 0, 0}, gb2[4] = {0, 0, 0, 0}, gb3 = 0.0f, loss = 0.0f;
  const int64_t tiles = (B + kTile - 1) / kTile;
  for (int64_t tile = blockIdx.x; tile < tiles; tile += gridDim.x) {
    if (tid < kTile * kIn) {
      const int s = tid / kIn, k = tid % kIn;
      const int64_t row = tile * kTile + s;
      float v = 0.0f;
      if (row < B) {
        const int64_t g = idx[row];
        const float raw = x[g * kIn + k];
        v = round_bf16((raw - a.norms[k]) * a.norms[kIn + k]);
        if (k == 0) tgt[s] = (y[g] - mu_y - cx * raw) / s_y;
      }
      xs[s][k] = v;
    }
    __syncthreads();
    // layer 1
    f32x4 z = zero;
    for (int k = 0; k < 3; ++k) z = mfma4(A1[k], xs[r][4 * k + q], z);
    float h1[4], h2[4];
    for (int i = 0; i < 4; ++i) {
      h1[i] = round_bf16(fmaxf(z[i] + b1[i], 0.0f));
      h1s[16 * w + 4 * q + i][r] = h1[i];
    }
    __syncthreads();
    // layer 2 and the output
    z = zero;
    for (int k = 0; k < 16; ++k) z = mfma4(A2[k], h1s[4 * k + q][r], z);
    float o = 0.0f;
    for (int i = 0; i < 4; ++i) {
      h2[i] = fmaxf(z[i] + b2[i], 0.0f);
      o += w3[i] * h2[i];
    }
    o += __shfl_xor(o, 16, 64);
    o += __shfl_xor(o, 32, 64);
    if (q == 0) os[w][r] = o;
    __syncthreads();
    const bool live = tile * kTile + r < B;
    const float res = live ? (os[0][r] + os[1][r]) + (os[2][r] + os[3][r]) + b3 - tgt[r] : 0.0f;
    const float d3 = 2.0f * res * invB;
    if (tid < kTile) {  // once per sample
      loss += res * res;
      gb3 += d3;
    }
    for (int i = 0; i < 4; ++i) {
      const float d2 = h2[i] > 0.0f ? d3 * w3[i] : 0.0f;
      d2s[16 * w + 4 * q + i][r] = d2;
      gb2[i] += d2;
      gw3[i] += d3 * h2[i];
    }
    __syncthreads();
    // d1 = W2^T d2 where the unit is active
    z = zero;
    for (int k = 0; k < 16; ++k) z = mfma4(A2t[k], d2s[4 * k + q][r], z);
    for (int i = 0; i < 4; ++i) {
      const float d1 = h1[i] > 0.0f ? z[i] : 0.0f;
      d1s[16 * w + 4 * q + i][r] = d1;
      gb1[i] += d1;
    }
    for (int k = 0; k < 4; ++k) {  // samples 4 k ..
      const float d = d2s[16 * w + r][4 * k + q];
      for (int b = 0; b < 4; ++b) g2[b] = mfma4(d, h1s[16 * b + r][4 * k + q], g2[b]);
    }
    __syncthreads();  // d1s is there
    for (int k = 0; k < 4; ++k) g1 = mfma4(d1s[16 * w + r][4 * k + q], r < kIn ? xs[4 * k + q][r] : 0.0f, g1);
    __syncthreads();  // the next tile overwrites xs, h1s and d2s
  }
  float* out = partial + (int64_t)blockIdx.x * kP;
  for (int i = 0; i < 4; ++i) {
    const int unit = 16 * w + 4 * q + i;
    for (int b = 0; b < 4; ++b) out[oW2 + unit * kHid + 16 * b + r] = g2[b][i];
    if (r < kIn) out[oW1 + unit * kIn + r] = g1[i];
    for (int off = 8; off > 0; off >>= 1) {  // over the samples
      gw3[i] += __shfl_xor(gw3[i], off, 64);
      gb1[i] += __shfl_xor(gb1[i], off, 64);
      gb2[i] += __shfl_xor(gb2[i], off, 64);
    }
    if (r == 0) {
      out[oW3 + unit] = gw3[i];
      out[oB1 + unit] = gb1[i];
      out[oB2 + unit] = gb2[i];
    }
  }
  if (w == 0) {
    for (int off = 8; off > 0; off >>= 1) {
      gb3 += __shfl_xor(gb3, off, 64);
      loss += __shfl_xor(loss, off, 64);
    }
    if (lane == 0) {
      out[oB3] = gb3;
      partial_loss[blockIdx.x] = loss;
    }
  }
}

struct AdamArgs {
  int step;  // 0: leave the parameters alone
  float lr, beta1, beta2, eps;
};

// grad[p] = sum_b partial[b][p]; loss = sum_b partial_loss[b] / B; and, for a
// training step, Adam (Kingma & Ba 2015, algorithm 1) on the FP32 master, the
// weight entries re-rounded into the BF16 copy.  A block takes 64 parameters,
// its 16 waves each every 16th row of partial: the rows' latencies overlap
// where one thread per parameter took them one after the other.
constexpr int kReduceSlices = 16;
__global__ __launch_bounds__(64 * kReduceSlices) void mlp_grad_reduce_kernel(MlpArgs a, const float* partial,
                                                                             const float* partial_loss, int nb,
                                                                             int64_t B, AdamArgs adam, float* grad,
                                                                             float* loss) {
  __shared__ float part[kReduceSlices][64];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, p = blockIdx.x * 64 + lane;
  float s = 0.0f;
  if (p < kP)
#pragma unroll 4
    for (int b = w; b < nb; b += kReduceSlices) s += partial[(int64_t)b * kP + p];
  part[w][lane] = s;
  __syncthreads();
  if (w == 0 && p < kP) {
    float g = 0.0f;
    for (int k = 0; k < kReduceSlices; ++k) g += part[k][lane];
    grad[p] = g;
    if (adam.step > 0) {
      const float m = adam.beta1 * a.adam_m[p] + (1.0f - adam.beta1) * g;
      const float v = adam.beta2 * a.adam_v[p] + (1.0f - adam.beta2) * g * g;
      a.adam_m[p] = m;
      a.adam_v[p] = v;
      const float mh = m / (1.0f - powf(adam.beta1, (float)adam.step));
      const float vh = v / (1.0f - powf(adam.beta2, (float)adam.step));
      const float q = a.params[p] - adam.lr * mh / (sqrtf(vh) + adam.eps);
      a.params[p] = q;
      a.wq[p] = f32_to_bf16(q);
    }
  }
  if (blockIdx.x == 0 && w == 1) {
    float t = 0.0f;
    for (int b = lane; b < nb; b += 64) t += partial_loss[b];
    for (int off = 32; off > 0; off >>= 1) t += __shfl_xor(t, off, 64);
    if (lane == 0) *loss = t / (float)B;
  }
}

__global__ void mlp_round_kernel(MlpArgs a) {
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p < kP) a.wq[p] = f32_to_bf16(a.params[p]);
}

}  // namespace

int mlp_grad_blocks(int64_t B) {
  const int64_t tiles = (B + kTile - 1) / kTile;
  return (int)std::min<int64_t>(std::max<int64_t>(tiles, 1), 256);
}

hipError_t launch_features(const FeatureArgs& a, hipStream_t s) {
  if (a.num_elems == 0) return hipSuccess;
  const unsigned ge = (unsigned)((a.num_elems + kFeatThreads - 1) / kFeatThreads);
  const unsigned gn = (unsigned)((a.num_nodes + kFeatThreads / 16 - 1) / (kFeatThreads / 16));
  hipLaunchKernelGGL(elem_geometry_kernel, dim3(ge), dim3(kFeatThreads), 0, s, a);
  hipLaunchKernelGGL(recover_kernel, dim3(gn), dim3(kFeatThreads), 0, s, a);
  hipLaunchKernelGGL(features_kernel, dim3(ge), dim3(kFeatThreads), 0, s, a);
  return hipGetLastError();
}

hipError_t launch_mlp_forward(const MlpArgs& a, const float* x, int64_t n, float* y, int* ood, hipStream_t s) {
  if (n == 0) return hipSuccess;
  // persistent: exactly the workgroups that are resident at once; each wave
  // loads the weights once, then walks groups of 16-row tiles
  static const int resident = [] {
    int occ = 0, dev = 0, cus = 256;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&occ, reinterpret_cast<const void*>(&mlp_forward_kernel),
                                                     kFwdThreads, 0) != hipSuccess ||
        occ < 1) {
      occ = 1;
      (void)hipGetLastError();
    }
    (void)hipGetDevice(&dev);
    (void)hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
    return occ * cus;
  }();
  const int64_t tiles = (n + 15) / 16;
  const int64_t groups = (tiles + kFwdUnroll - 1) / kFwdUnroll;
  const unsigned g = (unsigned)std::max<int64_t>(1, std::min<int64_t>((groups + kFwdWaves - 1) / kFwdWaves, resident));
  hipLaunchKernelGGL(mlp_forward_kernel, dim3(g), dim3(kFwdThreads), 0, s, a, x, n, y, ood);
  return hipGetLastError();
}

hipError_t launch_mlp_grad(const MlpArgs& a, const float* x, const float* y, const int32_t* idx, int64_t B,
                           float* partial, float* partial_loss, int step, float lr, float* grad, float* loss,
                           hipStream_t s) {
  if (B <= 0) return hipErrorInvalidValue;
  const int nb = mlp_grad_blocks(B);
  hipLaunchKernelGGL(mlp_grad_kernel, dim3(nb), dim3(kGradThreads), 0, s, a, x, y, idx, B, partial, partial_loss);
  hipLaunchKernelGGL(mlp_grad_reduce_kernel, dim3((kP + 63) / 64), dim3(64 * kReduceSlices), 0, s, a, partial,
                     partial_loss, nb, B, AdamArgs{step, lr, 0.9f, 0.999f, 1e-8f}, grad, loss);
  return hipGetLastError();
}

hipError_t launch_mlp_round(const MlpArgs& a, hipStream_t s) {
  hipLaunchKernelGGL(mlp_round_kernel, dim3((kP + 255) / 256), dim3(256), 0, s, a);
  return hipGetLastError();
}

}  // namespace goal
