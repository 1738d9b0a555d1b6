// Residual assembly without matrices: the residual of a step or line search
// (ASM_RESIDUAL), the error estimate's localization (ASM_LOCALIZE), and sums of
// per-element node values in general.
//
// residual_kernel takes one thread per quadrature point and keeps the whole
// evaluator chain (src/goal_assembly.cpp:65-88, src/goal_mechanics.cpp:97-146)
// in registers: gather, kinematics, model, weights.  An element's four points
// are the lanes of a quad; each ends with the coefficients alpha_i of N_a and
// beta_i of grad N_a in its residual rows, which are summed in barycentric
// form: with T_q[v] = beta . grad lambda_v and lambda_v(q) = B + (A - B) d_vq
//   vertex v:     (4 B - 1) sum T[v] + 4 (A - B) T_v[v]
//   edge (i, j):  4 B (sum T[i] + sum T[j]) + 4 (A - B) (T_i[j] + T_j[i])
// (alpha likewise), so lane q writes vertex q and edges (q, q + 1 mod 3) and
// (q, 3), q < 3, after exchanges inside the quad; no LDS, no barriers.
#include <algorithm>
#include <type_traits>

#include "goal_device.hpp"
#include "goal_kernels.hpp"

namespace goal {
namespace {

constexpr int kBlock = 256;
constexpr double kA = 0.5854101966249685, kB = 0.1381966011250105;  // lambda of the four points

template <int MODEL>
struct ModelOf;
template <>
struct ModelOf<MODEL_ELASTIC> {
  using type = dev::Elastic;
};
template <>
struct ModelOf<MODEL_NEOHOOKEAN> {
  using type = dev::NeoHookean;
};
template <>
struct ModelOf<MODEL_J2> {
  using type = dev::J2Model;
};

__device__ __forceinline__ double sel4(int i, double a, double b, double c, double d) {
  return i == 0 ? a : i == 1 ? b : i == 2 ? c : d;
}

// Lane permutations inside a quad; CTRL is a DPP quad_perm.
template <int CTRL>
__device__ __forceinline__ double quad(double v) {
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, 0xF, 0xF, true);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, 0xF, 0xF, true);
  return __hiloint2double(hi, lo);
}
constexpr int kXor1 = 0xB1, kXor2 = 0x4E, kNext = 0xC9, kFrom3 = 0xFF;  // kNext: 1, 2, 0, 3
__device__ __forceinline__ double quad_sum(double v) {
  v += quad<kXor1>(v);
  return v + quad<kXor2>(v);
}

__device__ __forceinline__ void put4(double* emr, int32_t rec, const double* r) {
  double2* o = reinterpret_cast<double2*>(emr + 4 * (int64_t)rec);
  o[0] = double2{r[0], r[1]};
  o[1] = double2{r[2], r[3]};
}

// Values of a nodal 4-vector field at a point: value and gradients along the
// barycentric coordinates 1..3 (differences against coordinate 0: a constant
// part drops out exactly).
template <int NN, int NQ>
struct Interp {
  double val[4], D[3][4];
  __device__ __forceinline__ void load(const double* x, const int32_t* ec, const double* lam) {
    double U[4][4];
#pragma unroll
    for (int i = 0; i < 4; ++i) val[i] = 0.0;
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const double* xn = x + 4 * (int64_t)ec[v];
      const double c = NN == 4 ? 1.0 : 4.0 * lam[v] - 1.0, N = NN == 4 ? lam[v] : lam[v] * (2.0 * lam[v] - 1.0);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        U[v][i] = c * xn[i];
        val[i] += N * xn[i];
      }
    }
    if constexpr (NN == 10) {
#pragma unroll
      for (int k = 0; k < 6; ++k) {
        const int i = k < 3 ? k : k - 3, j = k < 3 ? (k == 2 ? 0 : k + 1) : 3;
        const double* xn = x + 4 * (int64_t)ec[4 + k];
#pragma unroll
        for (int d = 0; d < 4; ++d) {
          U[i][d] += 4.0 * lam[j] * xn[d];
          U[j][d] += 4.0 * lam[i] * xn[d];
          val[d] += 4.0 * lam[i] * lam[j] * xn[d];
        }
      }
    }
#pragma unroll
    for (int v = 1; v < 4; ++v)
#pragma unroll
      for (int i = 0; i < 4; ++i) D[v - 1][i] = U[v][i] - U[0][i];
  }
  __device__ __forceinline__ double grad(const double gl[4][3], int i, int j) const {
    return D[0][i] * gl[1][j] + D[1][i] * gl[2][j] + D[2][i] * gl[3][j];
  }
};

template <int NN, int NQ, int MODEL, bool LOC>
__global__ __launch_bounds__(kBlock) void residual_kernel(AsmArgs a) {
  const int64_t t = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  const int64_t e = t / NQ;
  const int q = (int)(t % NQ);
  if (e >= a.num_elems) return;  // whole quads
  const int32_t* ec = a.conn + e * NN;
  double lam[4];
#pragma unroll
  for (int v = 0; v < 4; ++v) lam[v] = NQ == 1 ? 0.25 : (v == q ? kA : kB);
  const MatParams mp = a.mats[a.elem_set ? a.elem_set[e] : 0];
  Interp<NN, NQ> u;
  u.load(a.x, ec, lam);
  double gl[4][3], wdv, tau;
  {
    double X[4][3];
#pragma unroll
    for (int v = 0; v < 4; ++v)
#pragma unroll
      for (int c = 0; c < 3; ++c) X[v][c] = a.coords[3 * (int64_t)ec[v] + c];
    wdv = dev::tet_gradlambda(X, gl) * (NQ == 1 ? 1.0 / 6.0 : 1.0 / 24.0);
    tau = a.stabilization ? dev::stab_tau(X, mp) : 0.0;
  }
  double al[4], be[4][3];  // residual rows: al[i] N_a + be[i] . grad N_a
  {
    dev::QP qp;
#pragma unroll
    for (int j = 0; j < 3; ++j) {
#pragma unroll
      for (int i = 0; i < 3; ++i) qp.H[3 * i + j] = u.grad(gl, i, j);
      qp.g[j] = u.grad(gl, 3, j);
    }
#pragma unroll
    for (int k = 0; k < 9; ++k) qp.F[k] = qp.H[k] + ((k % 4 == 0) ? 1.0 : 0.0);
    qp.p = u.val[3];
    qp.J = dev::det3(qp.F);
    dev::inv3(qp.F, qp.J, qp.Fi);
    const int64_t n = a.num_elems * NQ;
    typename ModelOf<MODEL>::type m;
    if constexpr (MODEL == MODEL_J2) {
      double Fpo[9];
      for (int k = 0; k < 9; ++k) Fpo[k] = a.Fp_old[k * n + t];
      m.init(qp, mp, Fpo, a.eqps_old[t]);
      if (m.failed()) atomicOr(a.status, 1);
      if (!LOC && a.save_state) {
        a.eqps[t] = m.alpha;
        if (m.plastic) {
          double Fpn[9];
          m.new_Fp(Fpo, Fpn);
          for (int k = 0; k < 9; ++k) a.Fp[k * n + t] = Fpn[k];
        }
      }
    } else {
      m.init(qp, mp);
    }
    if (!LOC && a.save_state)
      for (int k = 0; k < 9; ++k) a.sigma[k * n + t] = m.sig[k];
    const double r1 = m.r1(qp);
    dev::Stab st;
    st.init(qp, tau);
    double s3[3];
    st.value(s3);
    if constexpr (!LOC) {
#pragma unroll
      for (int i = 0; i < 3; ++i) {
        al[i] = 0.0;
#pragma unroll
        for (int j = 0; j < 3; ++j) be[i][j] = m.P[3 * i + j] * wdv;
      }
      al[3] = r1 * wdv;
#pragma unroll
      for (int j = 0; j < 3; ++j) be[3][j] = s3[j] * wdv;
    } else {
      // DisplacementAdjoint / PressureAdjoint weights
      // (src/goal_displacement_adjoint.cpp:37-53, src/goal_pressure_adjoint.cpp:38-49)
      Interp<NN, NQ> z;
      z.load(a.z_diff, ec, lam);
#pragma unroll
      for (int i = 0; i < 3; ++i) {
        al[i] = 0.0;
#pragma unroll
        for (int j = 0; j < 3; ++j) {
          al[i] += m.P[3 * i + j] * wdv * z.grad(gl, i, j);
          be[i][j] = m.P[3 * i + j] * wdv * z.val[i];
        }
      }
      const double zp = z.val[3];
      z.load(a.z_coarse, ec, lam);
      al[3] = r1 * wdv * zp;
#pragma unroll
      for (int j = 0; j < 3; ++j) {
        al[3] += s3[j] * wdv * z.grad(gl, 3, j);
        be[3][j] = s3[j] * wdv * z.val[3];
      }
    }
  }
  double T[4][4];  // be[i] . grad lambda_v
#pragma unroll
  for (int i = 0; i < 4; ++i) {
#pragma unroll
    for (int v = 1; v < 4; ++v) T[v][i] = be[i][0] * gl[v][0] + be[i][1] * gl[v][1] + be[i][2] * gl[v][2];
    T[0][i] = -(T[1][i] + T[2][i] + T[3][i]);
  }
  const int32_t* rec = a.rec + e * NN;
  if constexpr (NQ == 1) {
    double r[4];
#pragma unroll
    for (int v = 0; v < 4; ++v) {
#pragma unroll
      // ten nodes: the vertex gradients vanish at the centroid; not left out, or a point whose stress is not
      // finite would not show in its vertices' rows
      for (int i = 0; i < 4; ++i) r[i] = NN == 4 ? 0.25 * al[i] + T[v][i] : -0.125 * al[i] + 0.0 * T[v][i];
      put4(a.emr, rec[v], r);
    }
    if constexpr (NN == 10) {
#pragma unroll
      for (int k = 0; k < 6; ++k) {
        const int vi = k < 3 ? k : k - 3, vj = k < 3 ? (k == 2 ? 0 : k + 1) : 3;
#pragma unroll
        for (int i = 0; i < 4; ++i) r[i] = 0.25 * al[i] + T[vi][i] + T[vj][i];
        put4(a.emr, rec[4 + k], r);
      }
    }
  } else {
    double rv[4], re[4], r3[4];  // vertex q, edges (q, q + 1 mod 3) and (q, 3)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const double S1 = quad_sum(T[1][i]), S2 = quad_sum(T[2][i]), S3 = quad_sum(T[3][i]), S0 = -(S1 + S2 + S3);
      const double Sa = quad_sum(al[i]);
      const double Sq = sel4(q, S0, S1, S2, S3);
      if constexpr (NN == 4) {
        rv[i] = Sq + kB * Sa + (kA - kB) * al[i];
      } else {
        constexpr double cB = 4.0 * kB - 1.0, cD = 4.0 * (kA - kB), eB = 4.0 * kB;
        constexpr double nB = kB * (2.0 * kB - 1.0), nD = kA * (2.0 * kA - 1.0) - nB, mB = 4.0 * kB * kB,
                         mD = 4.0 * kB * (kA - kB);
        rv[i] = cB * Sq + cD * sel4(q, T[0][i], T[1][i], T[2][i], T[3][i]) + nB * Sa + nD * al[i];
        // from lane q + 1 mod 3: its T[q]; it gives T[its own number - 1 mod 3]
        const double next_T = quad<kNext>(sel4(q, T[2][i], T[0][i], T[1][i], 0.0)), next_a = quad<kNext>(al[i]);
        const double Sn = sel4(q, S1, S2, S0, 0.0), Tn = sel4(q, T[1][i], T[2][i], T[0][i], 0.0);
        re[i] = eB * (Sq + Sn) + cD * (Tn + next_T) + mB * Sa + mD * (al[i] + next_a);
        const double t3 = sel4(q, quad<kFrom3>(T[0][i]), quad<kFrom3>(T[1][i]), quad<kFrom3>(T[2][i]), 0.0);
        r3[i] = eB * (Sq + S3) + cD * (T[3][i] + t3) + mB * Sa + mD * (al[i] + quad<kFrom3>(al[i]));
      }
    }
    put4(a.emr, rec[q], rv);
    if constexpr (NN == 10) {
      if (q < 3) {
        put4(a.emr, rec[4 + q], re);
        put4(a.emr, rec[7 + q], r3);
      }
    }
  }
}

// out[4 n + i] (+)= sum of emr[4 k + i] over node n's incidences k: 16 lanes a
// node, lane 4 j + i entry i of every fourth incidence, so that a node's
// records are read in whole 128-byte lines, four of them ahead of the sum.  Bound
// by the loads' latency where a node has many elements (320 tets around one node:
// 9.3 us for linear, 11 for quadratic ones; one load at a time 14 and 20, more than
// the node gather's 10.4), by HBM on large meshes (P2 64^3 190 us against 215; with
// two ahead 178 but 11 and 14 on the fans, with eight 216).
constexpr int kAhead = 4;
__global__ __launch_bounds__(kBlock) void node_sum_kernel(int64_t nn, const int64_t* inc_ptr, const double* emr,
                                                          int overwrite, double* out) {
  const int l = threadIdx.x & 15, i = l & 3;
  const int64_t n = (int64_t)blockIdx.x * (kBlock / 16) + threadIdx.x / 16;
  if (n >= nn) return;  // uniform per group of 16 lanes
  const int64_t k1 = inc_ptr[n + 1];
  double s = 0.0;
  for (int64_t k = inc_ptr[n] + (l >> 2); k < k1; k += 4 * kAhead) {
    double v[kAhead];
#pragma unroll
    for (int j = 0; j < kAhead; ++j) v[j] = emr[4 * (k + 4 * j < k1 ? k + 4 * j : k) + i];
#pragma unroll
    for (int j = 0; j < kAhead; ++j)
      if (k + 4 * j < k1) s += v[j];
  }
  s += __shfl_xor(s, 4, 64);
  s += __shfl_xor(s, 8, 64);
  if (l < 4) out[4 * n + i] = (overwrite ? 0.0 : out[4 * n + i]) + s;
}

template <int NN, int NQ, bool LOC>
hipError_t launch_model(const AsmArgs& a, hipStream_t s) {
  const dim3 grid((unsigned)((a.num_elems * NQ + kBlock - 1) / kBlock));
  switch (a.model) {
    case MODEL_ELASTIC: hipLaunchKernelGGL((residual_kernel<NN, NQ, MODEL_ELASTIC, LOC>), grid, dim3(kBlock), 0, s, a); break;
    case MODEL_NEOHOOKEAN: hipLaunchKernelGGL((residual_kernel<NN, NQ, MODEL_NEOHOOKEAN, LOC>), grid, dim3(kBlock), 0, s, a); break;
    case MODEL_J2: hipLaunchKernelGGL((residual_kernel<NN, NQ, MODEL_J2, LOC>), grid, dim3(kBlock), 0, s, a); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

template <bool LOC>
hipError_t launch_shape(int order, int quad_order, const AsmArgs& a, hipStream_t s) {
  if (order == 1) return quad_order == 1 ? launch_model<4, 1, LOC>(a, s) : launch_model<4, 4, LOC>(a, s);
  return quad_order == 1 ? launch_model<10, 1, LOC>(a, s) : launch_model<10, 4, LOC>(a, s);
}

}  // namespace

hipError_t launch_residual(int kind, int order, int quad_order, const AsmArgs& a, hipStream_t s) {
  if (a.num_elems == 0) return hipSuccess;
  if ((order != 1 && order != 2) || (quad_order != 1 && quad_order != 2)) return hipErrorInvalidValue;
  return kind == ASM_LOCALIZE ? launch_shape<true>(order, quad_order, a, s)
                              : launch_shape<false>(order, quad_order, a, s);
}

hipError_t launch_node_sum(int64_t nn, const int64_t* inc_ptr, const double* emr, int overwrite, double* out,
                           hipStream_t s) {
  if (nn == 0) return hipSuccess;
  hipLaunchKernelGGL(node_sum_kernel, dim3((unsigned)((nn + kBlock / 16 - 1) / (kBlock / 16))), dim3(kBlock), 0, s, nn,
                     inc_ptr, emr, overwrite, out);
  return hipGetLastError();
}

}  // namespace goal
