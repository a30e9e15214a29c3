// Crystal-plasticity kernels for gfx950 (FP64).
//
// Constitutive update per QP (the role of CP_PARAM::integration_algorithm,
// src/plasticity_model.cc:1148-1224, whose return map lives in the un-vendored GCM library):
//   unknowns x = (M, lambda, g), M = pF(n) pF(n+1)^-1
//   R_M      = M - I + dt sum_a gdot_a P_a - dt lambda pJ M^-T        (src/integration.cc:54-100)
//   R_lambda = pJ - 1,  pJ = det(pF(n)) / det(M)                      (:88-95)
//   R_g      = g (gs - g0 + dt h0 gdot) - (gs - g0) g_n - dt h0 gs gdot (:395-403)
//   gdot_a   = gdot0 (tau_a/g)|tau_a/g|^(1/m-1), tau_a = (C_e S):P_a,
//   C_e = eF^T eF, eF = F pF(n)^-1 M, and S either the cubic S = L : (C_e - I)/2
//   (src/TA_GA.cc:8-41) or the hyperelastic law of the material line (he_law below); the
//   kernels are instantiated per law
// Plain start: the reference's fully plastic predictor (initial_guess,
// src/initial_guess.cc:100-110: elastic part of step n kept, M_p = pF(n) F^-1 F(n) pF(n)^-1
// scaled to det 1) pulled back along M(a) = I + a (M_p - I) to max |tau_a|/g_n = 1 (8
// bisection steps, upper end kept; a = 0 below yield).  Newton on all eleven unknowns with
// backtracking on half the squared residual norm; converged when the full Newton step is
// below tol.  The 11x11 system is
// solved through the Schur complement of its (M, M) block: with the bordered structure
//   [A b c; d^T 0 0; e^T 0 f]
// one 9x9 elimination (in registers, unpivoted; the rare matrix that needs pivoting is solved
// again with it) serves the two right-hand sides of a Newton step, and a 6x6 one the
// nine columns of the tangent.  All of it runs in the crystal frame (see below).
//
// Kernels:
//   cp_kinematics  F(n+1) at every QP of a block (gather of the element nodes)
//   cp_start_kernel  the starting points (and the choice of a caller's start), one per lane
//   cp_newton      persistent: each wave works through a QP range, 64 QPs at a time
//   cp_tangent     at the converged state: tau, gdot, and per point the stress and the moduli that
//                  the element kernel contracts (qpbuf); for the three-field element Me, S, pJ
//                  and dMe/dF (Me = pF(n+1)^-1)
//   cp_tangent_pivot  the same for the points whose system needs pivoting
//   cp_elem        element rows: the reference contraction (compute_stiffness_matrix,
//                  src/constitutive_model.cc:1520-1616) is linear in the two gradients, so it is
//                  f_ab = sum_j T_bj dN_a,j, K_ab,wg = sum_jl dN_a,j A[b j][g l] dN_w,l with the
//                  first Piola-Kirchhoff stress T and its derivative A, formed per point
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <type_traits>

#include "pgf_device.h"
#include "pgf_math.h"

namespace pgf {
namespace {

using namespace dev;

typedef double dbl2 __attribute__((ext_vector_type(2)));

// Voigt helpers: index I -> (i,j) in xx,yy,zz,xy,yz,xz
__device__ __forceinline__ int vi(int I) { return I < 3 ? I : (I == 3 ? 0 : (I == 4 ? 1 : 0)); }
__device__ __forceinline__ int vj(int I) { return I < 3 ? I : (I == 3 ? 1 : 2); }

__device__ __forceinline__ void mm3(const double *A, const double *B, double *C) {
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int j = 0; j < 3; ++j) C[i * 3 + j] = A[i * 3] * B[j] + A[i * 3 + 1] * B[3 + j] + A[i * 3 + 2] * B[6 + j];
}
__device__ __forceinline__ void mtm3(const double *A, const double *B, double *C) {  // A^T B
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int j = 0; j < 3; ++j) C[i * 3 + j] = A[i] * B[j] + A[3 + i] * B[3 + j] + A[6 + i] * B[6 + j];
}
__device__ __forceinline__ void mmt3(const double *A, const double *B, double *C) {  // A B^T
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int j = 0; j < 3; ++j) C[i * 3 + j] = A[i * 3] * B[j * 3] + A[i * 3 + 1] * B[j * 3 + 1] + A[i * 3 + 2] * B[j * 3 + 2];
}
__device__ __forceinline__ double fma3(double a0, double b0, double a1, double b1, double a2, double b2) {
#pragma clang fp contract(off)
  return __builtin_fma(a0, b0, __builtin_fma(a1, b1, a2 * b2));
}
__device__ __forceinline__ void cubic_dot(const double *R, const double *cub, const double *X9, double *S6) {
#pragma clang fp contract(off)
  double E[9], T[9], Ep[9];
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int j = 0; j < 3; ++j) E[i * 3 + j] = 0.5 * (X9[i * 3 + j] + X9[j * 3 + i]);
#pragma unroll
  for (int i = 0; i < 3; ++i)  // T = E R
#pragma unroll
    for (int j = 0; j < 3; ++j) T[i * 3 + j] = fma3(E[i * 3 + 0], R[0 * 3 + j], E[i * 3 + 1], R[1 * 3 + j], E[i * 3 + 2], R[2 * 3 + j]);
#pragma unroll
  for (int i = 0; i < 3; ++i)  // E' = R^T T (symmetric: the upper triangle)
#pragma unroll
    for (int j = i; j < 3; ++j) Ep[i * 3 + j] = fma3(R[0 * 3 + i], T[0 * 3 + j], R[1 * 3 + i], T[1 * 3 + j], R[2 * 3 + i], T[2 * 3 + j]);
  const double tr = (Ep[0] + Ep[4]) + Ep[8];
  const double ct = cub[1] * tr;
  double Sp[9];
  Sp[0] = __builtin_fma(cub[0], Ep[0], ct);
  Sp[4] = __builtin_fma(cub[0], Ep[4], ct);
  Sp[8] = __builtin_fma(cub[0], Ep[8], ct);
  Sp[1] = Sp[3] = cub[2] * Ep[1];
  Sp[2] = Sp[6] = cub[2] * Ep[2];
  Sp[5] = Sp[7] = cub[2] * Ep[5];
#pragma unroll
  for (int i = 0; i < 3; ++i)  // T = S' R^T
#pragma unroll
    for (int j = 0; j < 3; ++j) T[i * 3 + j] = fma3(Sp[i * 3 + 0], R[j * 3 + 0], Sp[i * 3 + 1], R[j * 3 + 1], Sp[i * 3 + 2], R[j * 3 + 2]);
  double S[9];
#pragma unroll
  for (int i = 0; i < 3; ++i)  // S = R T (symmetric: the upper triangle)
#pragma unroll
    for (int j = i; j < 3; ++j) S[i * 3 + j] = fma3(R[i * 3 + 0], T[0 * 3 + j], R[i * 3 + 1], T[1 * 3 + j], R[i * 3 + 2], T[2 * 3 + j]);
  S6[0] = S[0];
  S6[1] = S[4];
  S6[2] = S[8];
  S6[3] = S[1];
  S6[4] = S[5];
  S6[5] = S[2];
}
__device__ __forceinline__ void v6_to_9(const double *s, double *S) {
  S[0] = s[0]; S[4] = s[1]; S[8] = s[2];
  S[1] = S[3] = s[3];
  S[5] = S[7] = s[4];
  S[2] = S[6] = s[5];
}

// Hyperelastic law of the intermediate configuration (law 1, as the CM model's elasticity on
// eF, src/constitutive_model.cc:998-1014): neo-Hookean deviatoric part (devStress_Mooney_Rivlin
// with m01 = 0, src/new_potentials.cc:329-358) and the volumetric potential of volPotFlag
// (:575-616), kappa = E / (3 (1 - 2 nu)):
//   S = 2 m10 d (I - tr(Ce)/3 Ci) + kappa J U'(J) Ci,   Ci = Ce^-1, d = det(Ce)^(-1/3), J = det eF
// Its tangent L = dS/dE (matStiff_Mooney_Rivlin, :376-432, with the volumetric terms) is used
// as a directional derivative on the symmetric part of X:
//   L : X = c1 (Ci:X) Ci + c2 ((Ci:X) I + tr(X) Ci) + c3 Ci X Ci
//   c1 = 4 m10 d tr(Ce)/9 + kappa (J U' + J^2 U''),  c2 = -4 m10 d / 3,  c3 = 4 m10 d tr(Ce)/3 - 2 kappa J U'
struct HeTan {
  double Ci[6], c1, c2, c3;
};

__device__ __forceinline__ void he_law(const CPMaterial &cm, const double *eF, const double *Ce, double *S6,
                                       HeTan &t) {
  const double J = det3(eF);
  double Ci9[9];
  inv3(Ce, Ci9);
  const double d = pow(det3(Ce), -1.0 / 3.0);
  const double trC = Ce[0] + Ce[4] + Ce[8];
  double dU, d2U;
  vol_pot(cm.vol_flag, J, dU, d2U);
  const double a = 2.0 * cm.m10 * d, pv = cm.kappa * J * dU;
  const double ci = pv - a * trC * (1.0 / 3.0);
#pragma unroll
  for (int I = 0; I < 6; ++I) {
    t.Ci[I] = Ci9[vi(I) * 3 + vj(I)];
    S6[I] = (I < 3 ? a : 0.0) + ci * t.Ci[I];
  }
  t.c1 = 2.0 * a * trC * (1.0 / 9.0) + cm.kappa * (J * dU + J * J * d2U);
  t.c2 = -2.0 * a * (1.0 / 3.0);
  t.c3 = 2.0 * a * trC * (1.0 / 3.0) - 2.0 * pv;
}

__device__ __forceinline__ void he_dot(const HeTan &t, const double *X9, double *out6) {
  const double x[6] = {X9[0], X9[4], X9[8], 0.5 * (X9[1] + X9[3]), 0.5 * (X9[5] + X9[7]), 0.5 * (X9[2] + X9[6])};
  const double *C = t.Ci;
  const double cx = C[0] * x[0] + C[1] * x[1] + C[2] * x[2] + 2.0 * (C[3] * x[3] + C[4] * x[4] + C[5] * x[5]);
  const double tx = x[0] + x[1] + x[2];
  double Ci9[9], X[9], T[9];
  v6_to_9(C, Ci9);
  v6_to_9(x, X);
  mm3(Ci9, X, T);
#pragma unroll
  for (int I = 0; I < 6; ++I) {
    const int i = vi(I), j = vj(I);
    const double r = T[i * 3] * Ci9[j] + T[i * 3 + 1] * Ci9[3 + j] + T[i * 3 + 2] * Ci9[6 + j];
    out6[I] = t.c1 * cx * C[I] + t.c2 * ((I < 3 ? cx : 0.0) + tx * C[I]) + t.c3 * r;
  }
}

// The stages of the local solve each fit the registers, their overlap does not.  pin makes a
// stage's results due at its end (in program order with the other asm), end_stage keeps the
// scheduler from mixing stages, and reload gives the lane's LDS slots under an index the
// compiler cannot see through, so that what is read after it is read from LDS, not kept.
__device__ __forceinline__ void end_stage() { __builtin_amdgcn_sched_barrier(0); }
template <int N>
__device__ __forceinline__ void pin(double (&x)[N]) {
#pragma unroll
  for (int i = 0; i < N; ++i) asm volatile("" : "+v"(x[i]));
}
__device__ __forceinline__ double *reload(double *slots, int lane) {
  asm volatile("" : "+v"(lane));
  return slots + lane;
}

// ------------------------------------------------------------------- the local solve
// The return map runs in the crystal frame: M, A = F pF(n)^-1 and the stress are rotated once per
// point (X' = R^T X R), and every quantity of the residual but the frame is rotation invariant.
// There the twelve Schmid tensors are P_a = kR6 s_a (x) n_k with entries of s and n in {0, +1, -1},
// so contractions with them are sums, and the cubic stiffness is three constants; nothing of the
// grain but R is read.  In the sample frame a system took about 260 operations of a Newton
// iteration's Jacobian, here about 60, and the slip directions, plane normals and the stiffness's
// frame were 72 doubles of the register file.
constexpr double kR6 = 0.40824829046386301637;  // 1 / sqrt(6)
// plane k's normal (1, 1, 1), with component k - 1 negative for k = 1, 2, 3
__device__ constexpr int n_sign(int k, int j) { return k == j + 1 ? -1 : 1; }
// slip direction of system a: the order of make_grain's table
__device__ constexpr int s_sign(int a, int i) {
  constexpr int t[12][3] = {{0, 1, -1}, {-1, 0, 1}, {1, -1, 0}, {0, 1, -1}, {1, 0, 1}, {1, 1, 0},
                            {0, 1, 1},  {1, 0, -1}, {1, 1, 0},  {0, 1, 1},  {1, 0, 1}, {1, -1, 0}};
  return t[a][i];
}
// +v, -v by a sign known at compile time (folds into the add that uses it)
__device__ __forceinline__ double pm(int s, double v) { return s > 0 ? v : -v; }
// s_a . x: the two components of system a's direction
__device__ __forceinline__ double s_dot(int a, const double *x) {
  return a % 3 == 0   ? x[1] + pm(s_sign(a, 2), x[2])
         : a % 3 == 1 ? pm(s_sign(a, 0), x[0]) + pm(s_sign(a, 2), x[2])
                      : x[0] + pm(s_sign(a, 1), x[1]);
}
__device__ __forceinline__ double n_dot(int k, double x0, double x1, double x2) {
  return (pm(n_sign(k, 0), x0) + pm(n_sign(k, 1), x1)) + pm(n_sign(k, 2), x2);
}
// y += s_a v (y of three, v known per system)
__device__ __forceinline__ void s_add(int a, double v, double *y) {
#pragma unroll
  for (int i = 0; i < 3; ++i)
    if (s_sign(a, i) != 0) y[i] += pm(s_sign(a, i), v);
}

// 3x3 products and inverse with explicit multiply-adds: what a residual pass and a fused pass
// both compute has the same bits in either kernel.
__device__ __forceinline__ void mul_ab(const double *A, const double *B, double *C) {
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int j = 0; j < 3; ++j) C[i * 3 + j] = fma3(A[i * 3], B[j], A[i * 3 + 1], B[3 + j], A[i * 3 + 2], B[6 + j]);
}
__device__ __forceinline__ void mul_atb(const double *A, const double *B, double *C) {
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int j = 0; j < 3; ++j) C[i * 3 + j] = fma3(A[i], B[j], A[3 + i], B[3 + j], A[6 + i], B[6 + j]);
}
__device__ __forceinline__ void mul_abt(const double *A, const double *B, double *C) {
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int j = 0; j < 3; ++j)
      C[i * 3 + j] = fma3(A[i * 3], B[j * 3], A[i * 3 + 1], B[j * 3 + 1], A[i * 3 + 2], B[j * 3 + 2]);
}
__device__ __forceinline__ double det2(double a, double b, double c, double d) {  // a b - c d
#pragma clang fp contract(off)
  return __builtin_fma(a, b, -(c * d));
}
// the inverse and determinant of m; false below the singularity threshold of inv3
__device__ __forceinline__ bool inv_det(const double *m, double *mi, double &det) {
#pragma clang fp contract(off)
  const double c0 = det2(m[4], m[8], m[5], m[7]), c1 = det2(m[5], m[6], m[3], m[8]), c2 = det2(m[3], m[7], m[4], m[6]);
  det = fma3(m[0], c0, m[1], c1, m[2], c2);
  const double r = 1.0 / det;
  mi[0] = r * c0;
  mi[3] = r * c1;
  mi[6] = r * c2;
  mi[1] = r * det2(m[2], m[7], m[1], m[8]);
  mi[4] = r * det2(m[0], m[8], m[2], m[6]);
  mi[7] = r * det2(m[1], m[6], m[0], m[7]);
  mi[2] = r * det2(m[1], m[5], m[2], m[4]);
  mi[5] = r * det2(m[2], m[3], m[0], m[5]);
  mi[8] = r * det2(m[0], m[4], m[1], m[3]);
  return fabs(det) >= 1.0e-15;
}
__device__ __forceinline__ void rot_in(const double *R, const double *X, double *Y) {  // R^T X R
  double T[9];
  mul_ab(X, R, T);
  mul_atb(R, T, Y);
}
__device__ __forceinline__ void rot_out(const double *R, const double *X, double *Y) {  // R X R^T
  double T[9];
  mul_ab(R, X, T);
  mul_abt(T, R, Y);
}
// The same of X = I + Y, as I + R^T Y R: the orthonormality error of R (1e-16) would otherwise come
// into the elastic strain, and times C / tau = 1e4 into the stress.
__device__ __forceinline__ void rot_in_1(const double *R, const double *X, double *Y) {
  const double D[9] = {X[0] - 1.0, X[1], X[2], X[3], X[4] - 1.0, X[5], X[6], X[7], X[8] - 1.0};
  rot_in(R, D, Y);
  Y[0] += 1.0;
  Y[4] += 1.0;
  Y[8] += 1.0;
}
__device__ __forceinline__ void rot_out_1(const double *R, const double *X, double *Y) {
  const double D[9] = {X[0] - 1.0, X[1], X[2], X[3], X[4] - 1.0, X[5], X[6], X[7], X[8] - 1.0};
  rot_out(R, D, Y);
  Y[0] += 1.0;
  Y[4] += 1.0;
  Y[8] += 1.0;
}

// What of the flow and hardening rule needs pow: 0 both, 1 the saturation stress (w != 0), 2 none.
// A kernel holds one form: twelve inlined pows are a quarter of the Newton kernel's code, which
// has to fit the instruction cache, and one pow's constants, kept across its loop, 40 registers.
enum : int { kFlowPow = 0, kFlowSat = 1, kFlowPlain = 2 };
// |r_a|^e of the power-law flow rule, e = 1/m - 1, for the twelve systems.  When e is a whole
// number (ie >= 0; the rate sensitivity m = 0.05 gives 19) it is formed by binary powering, a
// handful of multiplies where pow takes about 130 FP64 operations; the two agree to a few ulps.
template <int FLOW>
__device__ __forceinline__ void flow_pow(const double (&r)[12], double e, int ie, double (&w)[12]) {
  if constexpr (FLOW >= 1) {
    double b[12];
#pragma unroll
    for (int a = 0; a < 12; ++a) {
      b[a] = fabs(r[a]);
      w[a] = 1.0;
    }
    for (int k = ie; k; k >>= 1) {
      if (k & 1) {
#pragma unroll
        for (int a = 0; a < 12; ++a) w[a] *= b[a];
      }
#pragma unroll
      for (int a = 0; a < 12; ++a) b[a] *= b[a];
    }
  } else {
#pragma unroll
    for (int a = 0; a < 12; ++a) w[a] = pow(fabs(r[a]), e);
  }
}

// Elastic PK2 (Voigt) in the crystal frame from eF and Ce = eF^T eF: law 0 is the cubic
// S = L : (Ce - I)/2; law 1 is he_law, which also fills the tangent coefficients.  The
// multiply-adds are explicit, so that every kernel gives the same bits.
template <bool HE>
__device__ __forceinline__ void el_stress(const CPMaterial &cm, const double *eF, const double *Ce, double *S6,
                                          HeTan &t) {
  if constexpr (HE) {
    he_law(cm, eF, Ce, S6, t);
  } else {
#pragma clang fp contract(off)
    const double e0 = 0.5 * (Ce[0] - 1.0), e1 = 0.5 * (Ce[4] - 1.0), e2 = 0.5 * (Ce[8] - 1.0);
    const double ct = cm.c12 * ((e0 + e1) + e2), sh = 0.5 * cm.c44x2;
    S6[0] = __builtin_fma(cm.c11m12, e0, ct);
    S6[1] = __builtin_fma(cm.c11m12, e1, ct);
    S6[2] = __builtin_fma(cm.c11m12, e2, ct);
    S6[3] = sh * Ce[1];
    S6[4] = sh * Ce[5];
    S6[5] = sh * Ce[2];
  }
}

// eF = A M, C_e = eF^T eF, S and the twelve tau_a = (C_e S) : P_a
struct CPStress {
  double eF[9], Ce[9], S[6], tau[12];
  HeTan he;  // law 1: tangent coefficients at Ce
};
template <bool HE>
__device__ __forceinline__ void cp_stress(const CPMaterial &cm, const double *A, const double *M, CPStress &p) {
#pragma clang fp contract(off)
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int j = 0; j < 3; ++j) p.eF[i * 3 + j] = fma3(A[i * 3], M[j], A[i * 3 + 1], M[3 + j], A[i * 3 + 2], M[6 + j]);
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int j = i; j < 3; ++j)
      p.Ce[j * 3 + i] = p.Ce[i * 3 + j] = fma3(p.eF[i], p.eF[j], p.eF[3 + i], p.eF[3 + j], p.eF[6 + i], p.eF[6 + j]);
  el_stress<HE>(cm, p.eF, p.Ce, p.S, p.he);
  double S9[9], Sig[9];
  v6_to_9(p.S, S9);
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int j = 0; j < 3; ++j)
      Sig[i * 3 + j] = fma3(p.Ce[i * 3], S9[j], p.Ce[i * 3 + 1], S9[3 + j], p.Ce[i * 3 + 2], S9[6 + j]);
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    double u[3];
#pragma unroll
    for (int i = 0; i < 3; ++i) u[i] = n_dot(k, Sig[i * 3], Sig[i * 3 + 1], Sig[i * 3 + 2]);
#pragma unroll
    for (int a = 3 * k; a < 3 * k + 3; ++a) p.tau[a] = kR6 * s_dot(a, u);
  }
}

// Material-point evaluation at x = (M, lambda, g).  Returns false outside the domain, where p is
// of no use; every lane runs through it, since a branch around it would keep its registers
// live from one turn of the Newton loop to the next.
struct CPPoint : CPStress {
  double T[9];    // M^-T
  double N[9];    // dt sum_a gdot_a P_a
  double sd[12];  // dgdot_a / dtau_a with the sign of gdot_a
  double pJ, gsum, gs, dgs, R[11];
};

template <bool HE, int FLOW>
__device__ __forceinline__ bool cp_point(const CPMaterial &cm, const double *A, double det_pFn, double g_n, double dt,
                                         const double *x, CPPoint &p) {
  const double *M = x;
  const double lam = x[9], g = x[10];
  double Mi[9], dM;
  const bool valid = inv_det(M, Mi, dM) && dM > 0.0 && g > 0.0;
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int j = 0; j < 3; ++j) p.T[i * 3 + j] = Mi[j * 3 + i];
  p.pJ = det_pFn / dM;
  cp_stress<HE>(cm, A, M, p);
  // one reciprocal of g for the twelve systems (the divisions are software sequences)
  const double rg = 1.0 / g, cdg = cm.gd0_m * rg;
  double r[12], w[12], V[4][3] = {};  // V_k = sum over plane k of gdot_a s_a
#pragma unroll
  for (int a = 0; a < 12; ++a) r[a] = p.tau[a] * rg;
  flow_pow<FLOW>(r, cm.expo, cm.ipow, w);
  p.gsum = 0.0;
#pragma unroll
  for (int a = 0; a < 12; ++a) {
    const double gdot = cm.gd0 * r[a] * w[a];
    p.sd[a] = r[a] < 0.0 ? -(cdg * w[a]) : cdg * w[a];
    p.gsum += fabs(gdot);
    s_add(a, gdot, V[a / 3]);
  }
  p.gs = cm.gs0;
  p.dgs = 0.0;
  if (FLOW != kFlowPlain && cm.w != 0.0) {
    const bool flows = p.gsum / cm.gds > 1.0e-15;
    p.gs = flows ? cm.gs0 * pow(p.gsum / cm.gds, cm.w) : 0.0;
    p.dgs = flows ? cm.w * p.gs / p.gsum : 0.0;
  }
  const double dk = dt * kR6, dl = dt * lam * p.pJ;
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      double sl = 0.0;
#pragma unroll
      for (int k = 0; k < 4; ++k) sl += pm(n_sign(k, j), V[k][i]);
      p.N[i * 3 + j] = dk * sl;
      p.R[i * 3 + j] = M[i * 3 + j] - ((i == j) ? 1.0 : 0.0) + p.N[i * 3 + j] - dl * p.T[i * 3 + j];
    }
  p.R[9] = p.pJ - 1.0;
  p.R[10] = g * (p.gs - cm.g0 + dt * cm.h0 * p.gsum) - (p.gs - cm.g0) * g_n - dt * cm.h0 * p.gs * p.gsum;
  return valid;
}

// What one system's Q_a = sym(P_a S + 1/2 L:(C_e P_a)), d tau_a / d M = 2 A^T eF Q_a, shares
// with its plane: v = S n, and for law 1 Ci n.
struct CPPlane {
  double v[3], cn[3];
};
template <bool HE>
__device__ __forceinline__ void cp_plane(const CPStress &p, int k, CPPlane &q) {
  const double *S = p.S;
  q.v[0] = n_dot(k, S[0], S[3], S[5]);
  q.v[1] = n_dot(k, S[3], S[1], S[4]);
  q.v[2] = n_dot(k, S[5], S[4], S[2]);
  if constexpr (HE) {
    const double *C = p.he.Ci;
    q.cn[0] = n_dot(k, C[0], C[3], C[5]);
    q.cn[1] = n_dot(k, C[3], C[1], C[4]);
    q.cn[2] = n_dot(k, C[5], C[4], C[2]);
  }
}
// Q_a * 2 / kR6 in Voigt order.  P_a S = kR6 s (x) v, C_e P_a = kR6 w (x) n with w = C_e s.
// Law 0: L of w (x) n by its three constants.  Law 1: he_dot of sym(w (x) n), where Ci w = s and
// s . n = 0 leave c2 tr Ci + c3 sym(s (x) Ci n).
template <bool HE>
__device__ __forceinline__ void cp_q(const CPMaterial &cm, const CPStress &p, const CPPlane &pl, int a, double *q) {
  const int k = a / 3;
  double w[3];
#pragma unroll
  for (int i = 0; i < 3; ++i) w[i] = s_dot(a, p.Ce + 3 * i);  // C_e is symmetric
  const double tr = n_dot(k, w[0], w[1], w[2]);
#pragma unroll
  for (int I = 0; I < 6; ++I) {
    const int i = voigt_i(I), j = voigt_j(I);
    double x = 0.0;  // s_i v_j + s_j v_i
    if (s_sign(a, i) != 0) x += pm(s_sign(a, i), pl.v[j]);
    if (s_sign(a, j) != 0) x += pm(s_sign(a, j), pl.v[i]);
    if constexpr (HE) {
      double y = 0.0;  // s_i cn_j + s_j cn_i
      if (s_sign(a, i) != 0) y += pm(s_sign(a, i), pl.cn[j]);
      if (s_sign(a, j) != 0) y += pm(s_sign(a, j), pl.cn[i]);
      q[I] = x + p.he.c2 * tr * p.he.Ci[I] + 0.5 * p.he.c3 * y;
    } else if (I < 3) {
      q[I] = x + (cm.c11m12 * pm(n_sign(k, i), w[i]) + cm.c12 * tr);
    } else {
      q[I] = x + 0.5 * cm.c44x2 * (pm(n_sign(k, j), w[i]) + pm(n_sign(k, i), w[j]));
    }
  }
}

// The Jacobian of the local system at p is bordered,
//   [A b c; d^T 0 0; e^T 0 f],  d = -pJ M^-T, b = dt d,
// and A and e see dM only through the six numbers K dM = sym(A^T eF dM) (K_I: the diagonal
// entries of Y = AtE^T dM, then Y_ij + Y_ji), since dtau_a does:
//   e = es eq K,  A - c e^T / f = I + lp T (.)^T T + G K,  T = M^-T, lp = dt lambda pJ,
// less A's term lp T (x) T = (lambda / pJ) b d^T: where d . u = s is an equation of the system,
// that term only moves (lambda / pJ) s between A u and b y.
// G = sum_a dt dgdt_a / 6 (s_a n_k) (x) q_a - c (es eq) / f.  The power law gives the rest from
// what the point has: dgdot_a/dg = -gdot_a / (m g), so c = -N / (m g).
struct LocalLin {
  double G[9][6], eq[6], es, f;
};
// G and eq without the factors of cp_fold
template <bool HE>
__device__ __forceinline__ void cp_slip_sums(const CPMaterial &cm, const CPStress &p, const double *sd, LocalLin &L) {
#pragma unroll
  for (int I = 0; I < 6; ++I) L.eq[I] = 0.0;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    CPPlane pl;
    cp_plane<HE>(p, k, pl);
    double V[3][6] = {};
#pragma unroll
    for (int a = 3 * k; a < 3 * k + 3; ++a) {
      double q[6];
      cp_q<HE>(cm, p, pl, a, q);
#pragma unroll
      for (int I = 0; I < 6; ++I) {
        L.eq[I] += sd[a] * q[I];
        q[I] *= fabs(sd[a]);
#pragma unroll
        for (int i = 0; i < 3; ++i)
          if (s_sign(a, i) != 0) V[i][I] += pm(s_sign(a, i), q[I]);
      }
    }
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
      for (int j = 0; j < 3; ++j)
#pragma unroll
        for (int I = 0; I < 6; ++I)
          L.G[i * 3 + j][I] = k == 0 ? V[i][I] : L.G[i * 3 + j][I] + pm(n_sign(k, j), V[i][I]);
#pragma unroll
    for (int r = 0; r < 9; ++r) pin(L.G[r]);
    end_stage();
  }
}
__device__ __forceinline__ void cp_fold(const CPMaterial &cm, double dt, double g, double g_n, double gsum, double gs,
                                        double dgs, const double *c, LocalLin &L) {
  const double dRg = g * (dgs + dt * cm.h0) - dgs * g_n - dt * cm.h0 * (dgs * gsum + gs);
  L.f = (gs - cm.g0 + dt * cm.h0 * gsum) - dRg * gsum / (cm.m * g);
  L.es = dRg * kR6;
  const double as = dt * (kR6 * kR6), rf = L.es / L.f;
#pragma unroll
  for (int r = 0; r < 9; ++r) {
    const double cr = c[r] * rf;
#pragma unroll
    for (int I = 0; I < 6; ++I) L.G[r][I] = as * L.G[r][I] - cr * L.eq[I];
  }
}
// the matrix I + lp T (.)^T T + G K
__device__ __forceinline__ void cp_matrix(const LocalLin &L, const double *AtE, const double *T, double lp,
                                          double (&Ah)[81]) {
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      const int r = i * 3 + j;
      double G9[9];
      v6_to_9(L.G[r], G9);
      double lt[3];
#pragma unroll
      for (int l = 0; l < 3; ++l) lt[l] = lp * T[i * 3 + l];
#pragma unroll
      for (int k = 0; k < 3; ++k)
#pragma unroll
        for (int l = 0; l < 3; ++l)
          Ah[r * 9 + k * 3 + l] = ((i == k && j == l) ? 1.0 : 0.0) + AtE[k * 3] * G9[l] + AtE[k * 3 + 1] * G9[3 + l] +
                                  AtE[k * 3 + 2] * G9[6 + l] + lt[l] * T[k * 3 + j];
    }
}

// Gaussian elimination of A with NR right-hand sides, solutions in B, without pivoting; false
// where a multiplier exceeds max_mult or a pivot is no number, and the caller takes
// factor_pivot.  The local system is the identity plus the slip systems' positive part, so
// large multipliers are rare (above 1000 in 0.1% of the matrices of a plastic step), and partial
// pivoting by predicated swaps is more instructions than the elimination.  A Newton step only has
// to be a good direction: the residual, not the matrix, fixes the point that the iteration ends
// at, and at 1e6 its relative error stays near 1e-10.  A step that pivots is taken twice: with a bound
// of 1e3 a pass over 998,250 points takes 2333 us instead of 2277, and 3476 where every step pivots.
// The tangent is a result, and its bound lower; where every point's pivots, the pass takes 2564 us.
// (kMaxMultStep and kMaxMultTangent, unless the caller sets others.)
template <int N, int NR>
__device__ __forceinline__ bool eliminate(double (&A)[N * N], double (&B)[NR][N], double max_mult) {
  double lmax = 0.0, rd[N];
#pragma unroll
  for (int k = 0; k < N; ++k) {
    rd[k] = 1.0 / A[k * N + k];
#pragma unroll
    for (int i = k + 1; i < N; ++i) {
      const double l = A[i * N + k] * rd[k];
      lmax = fmax(lmax, fabs(l));
#pragma unroll
      for (int j = k + 1; j < N; ++j) A[i * N + j] -= l * A[k * N + j];
#pragma unroll
      for (int q = 0; q < NR; ++q) B[q][i] -= l * B[q][k];
    }
    asm volatile("" : "+v"(lmax));  // now, not from multipliers kept to the end
  }
#pragma unroll
  for (int i = N - 1; i >= 0; --i)
#pragma unroll
    for (int q = 0; q < NR; ++q) {
      double s = B[q][i];
#pragma unroll
      for (int j = i + 1; j < N; ++j) s -= A[i * N + j] * B[q][j];
      B[q][i] = s * rd[i];
    }
  return lmax <= max_mult && fabs(rd[N - 1]) < __builtin_huge_val();
}
// The same with partial pivoting, as factors and solutions: every lane that needs it takes part, its
// rows exchanged by selects, so that no index is known at run time only.  False for a singular matrix.
template <int N>
__device__ __forceinline__ bool factor_pivot(double (&A)[N * N], int (&piv)[N]) {
  bool ok = true;
#pragma unroll
  for (int k = 0; k < N; ++k) {
    int p = k;
    double amax = fabs(A[k * N + k]);
#pragma unroll
    for (int i = k + 1; i < N; ++i) {
      const double v = fabs(A[i * N + k]);
      p = v > amax ? i : p;
      amax = v > amax ? v : amax;
    }
    ok = ok && amax > 0.0;
    piv[k] = p;
#pragma unroll
    for (int i = k + 1; i < N; ++i)
#pragma unroll
      for (int j = 0; j < N; ++j) {
        const double x = A[k * N + j], y = A[i * N + j];
        A[k * N + j] = p == i ? y : x;
        A[i * N + j] = p == i ? x : y;
      }
    const double r = 1.0 / A[k * N + k];
    A[k * N + k] = r;
#pragma unroll
    for (int i = k + 1; i < N; ++i) {
      A[i * N + k] *= r;
#pragma unroll
      for (int j = k + 1; j < N; ++j) A[i * N + j] -= A[i * N + k] * A[k * N + j];
    }
  }
  return ok;
}
template <int N>
__device__ __forceinline__ void solve_pivot(const double (&A)[N * N], const int (&piv)[N], double (&b)[N]) {
#pragma unroll
  for (int k = 0; k < N; ++k)
#pragma unroll
    for (int i = k + 1; i < N; ++i) {
      const double x = b[k], y = b[i];
      b[k] = piv[k] == i ? y : x;
      b[i] = piv[k] == i ? x : y;
    }
#pragma unroll
  for (int k = 0; k < N; ++k)
#pragma unroll
    for (int i = k + 1; i < N; ++i) b[i] -= A[i * N + k] * b[k];
#pragma unroll
  for (int i = N - 1; i >= 0; --i) {
#pragma unroll
    for (int j = i + 1; j < N; ++j) b[i] -= A[i * N + j] * b[j];
    b[i] *= A[i * N + i];
  }
}

__device__ __forceinline__ double cp_merit(const CPPoint &p, double gscale) {
  double r = 0.0;
#pragma unroll
  for (int i = 0; i < 10; ++i) r += p.R[i] * p.R[i];
  const double rg = p.R[10] * gscale;
  return 0.5 * (r + rg * rg);
}

// max_a |tau_a| / g at M (elastic part eF = A M)
template <bool HE>
__device__ __forceinline__ double tau_ratio_max(const CPMaterial &cm, const double *A, const double *M, double rg) {
  CPStress p;
  cp_stress<HE>(cm, A, M, p);
  double mx = 0.0;
#pragma unroll
  for (int a = 0; a < 12; ++a) mx = fmax(mx, fabs(p.tau[a]));
  return mx * rg;
}

// Plain start x = (M, lambda_n, g_n) in the crystal frame: the fully plastic predictor
// Mp = pF(n) F^-1 F(n) pF(n)^-1 (not yet scaled to det 1), pulled back to yield.
template <bool HE>
__device__ __forceinline__ bool cp_start(const CPMaterial &cm, const double *A, double (&Mp)[9], double g_n,
                                         double lam_n, double *x) {
  const double dp = det3(Mp);
  if (!(dp > 0.0)) return false;
  const double c = 1.0 / cbrt(dp);
#pragma unroll
  for (int i = 0; i < 9; ++i) Mp[i] *= c;
  const double rg = 1.0 / g_n;
  const double I9[9] = {1, 0, 0, 0, 1, 0, 0, 0, 1};
  double al = 0.0;
  if (tau_ratio_max<HE>(cm, A, I9, rg) > 1.0) {
    al = 1.0;
    if (!(tau_ratio_max<HE>(cm, A, Mp, rg) > 1.0)) {
      double lo = 0.0, hi = 1.0;
      for (int k = 0; k < 8; ++k) {
        const double mid = 0.5 * (lo + hi);
        double Mm[9];
#pragma unroll
        for (int i = 0; i < 9; ++i) Mm[i] = I9[i] + mid * (Mp[i] - I9[i]);
        if (tau_ratio_max<HE>(cm, A, Mm, rg) > 1.0) lo = mid;
        else hi = mid;
      }
      al = hi;
    }
  }
#pragma unroll
  for (int i = 0; i < 9; ++i) x[i] = I9[i] + al * (Mp[i] - I9[i]);
  if (al > 0.0) {
    const double sc = 1.0 / cbrt(det3(x));
#pragma unroll
    for (int i = 0; i < 9; ++i) x[i] *= sc;
  }
  x[9] = lam_n;
  x[10] = g_n;
  return true;
}

// ------------------------------------------------------------------- kinematics kernel
template <int NNE>
__global__ __launch_bounds__(256) void cp_kinematics(CPArgs a) {
  constexpr int NQP = nqp_of(NNE);
  const int64_t tq = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (tq >= a.ne * NQP) return;
  const int64_t e = tq / NQP;
  const int ip = int(tq % NQP);
  double x[NNE * 3], u[NNE * 3];
#pragma unroll
  for (int n = 0; n < NNE; ++n) {
    const int32_t node = a.conn[e * NNE + n];
#pragma unroll
    for (int b = 0; b < 3; ++b) {
      x[n * 3 + b] = a.X[int64_t(node) * 3 + b];
      const int32_t d = a.dofid[int64_t(node) * 3 + b];
      double uu = 0.0;  // def_elem_total, src/utils.cc:1391-1412
      if (d > 0) uu = a.r[d - 1] + (a.d_r ? a.d_r[d - 1] : 0.0);
      else if (d < 0)  // the prescribed-load pass takes K at defl
        uu = (a.defl ? a.defl[-d - 1] : 0.0) + (a.defl_d && !(a.kin & kKinDefl) ? a.defl_d[-d - 1] : 0.0);
      u[n * 3 + b] = uu;
    }
  }
  double k, ee, z, wt;
  int_point(NNE, ip, k, ee, z, wt);
  double dN[NNE * 3];
  shape_dN<NNE>(k, ee, z, dN);
  double dX[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
  for (int n = 0; n < NNE; ++n)
#pragma unroll
    for (int ib = 0; ib < 3; ++ib)
#pragma unroll
      for (int ic = 0; ic < 3; ++ic) dX[ib * 3 + ic] += dN[n * 3 + ic] * x[n * 3 + ib];
  double Xi[9] = {};
  const double J0 = det3(dX);
  const bool ok = J0 > 0.0 && inv3(dX, Xi);
  double F[9] = {1, 0, 0, 0, 1, 0, 0, 0, 1};
#pragma unroll
  for (int n = 0; n < NNE; ++n) {
    double g[3];
#pragma unroll
    for (int ib = 0; ib < 3; ++ib)
      g[ib] = dN[n * 3 + 0] * Xi[0 * 3 + ib] + dN[n * 3 + 1] * Xi[1 * 3 + ib] + dN[n * 3 + 2] * Xi[2 * 3 + ib];
#pragma unroll
    for (int ib = 0; ib < 3; ++ib)
#pragma unroll
      for (int ic = 0; ic < 3; ++ic) F[ib * 3 + ic] += u[n * 3 + ib] * g[ic];
  }
  const int64_t q = a.qp_base + tq;
  if (a.kin & kKinRec) {
    double *rec = a.qpbuf + qrec(q);
#pragma unroll
    for (int i = 0; i < 9; ++i) rec[(kRecXi + i) * kRecStride] = Xi[i];
    rec[kRecW * kRecStride] = ok ? J0 * wt : 0.0;
    if (!ok) atomicAdd(a.err, 1);
    if (!(a.kin & kKinState)) {
#pragma unroll
      for (int i = 0; i < 9; ++i) rec[i * kRecStride] = F[i];
    }
  }
  if (!(a.kin & kKinState)) return;
  const double J = det3(F);
  bool okF = ok && J > 0.0;  // getJacobian, src/utils.cc:513-527
  if (a.tf_V) {
    // CM3F: the model integrates at (theta/J)^(1/3) F and keeps it as its F(n+1)
    // (run_integration_algorithm with tf_factor, src/constitutive_model.cc:810-818, :1109-1115)
    const double th = a.tf_V[e] + a.tf_dV[e];
    okF = okF && th > 0.0;
    const double fac = okF ? cbrt(th / J) : 1.0;
#pragma unroll
    for (int i = 0; i < 9; ++i) F[i] *= fac;
  }
#pragma unroll
  for (int i = 0; i < 9; ++i) a.F_np1[i * a.n_qp + q] = F[i];
  if (!okF) atomicAdd(a.err, 1);
}

// ------------------------------------------------------------------- start kernel
// The local Newton's starting points, one thread per QP, ahead of the Newton kernel: the plain
// start (the plastic predictor pulled back to yield, about ten stress evaluations) and, with a
// caller's start attached, which of the two has the lower residual merit.  In the Newton
// kernel a lane takes a new QP whenever its last one converges, so work done at a refill runs
// with the other lanes of the wave masked off; here it runs on every lane.  The QP's record in
// qpbuf holds the plain start x(0..10) and the choice kStartFlag (bit 0: the plain start
// failed, bit 1: take the caller's start) until the tangent kernel overwrites it.
constexpr int kStartFlag = 11;
template <bool HE, int FLOW>
__global__ __launch_bounds__(64) void cp_start_kernel(CPArgs a) {
  const int64_t q = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (q >= a.nq) return;
  const int64_t NQ = a.n_qp;
  const int64_t qg = a.qp_base + q;
  const CPMaterial cm = a.cpmats[0];
  const double *R = a.grains[a.qgrain[q]].R;
  double F[9], pFn[9], pFi[9], Fn[9], Fi[9], A[9] = {}, T[9], Mp[9], x[11], det_pFn = 1.0, det_F;
#pragma unroll
  for (int i = 0; i < 9; ++i) {
    F[i] = a.F_np1[i * NQ + qg];
    pFn[i] = a.pF_n[i * NQ + qg];
    Fn[i] = a.F_n[i * NQ + qg];
    x[i] = 0.0;
  }
  bool bad = !inv_det(pFn, pFi, det_pFn) || !inv_det(F, Fi, det_F);
  const double g_n = a.g_n[qg];
  x[9] = x[10] = 0.0;
  if (!bad) {
    mul_ab(F, pFi, T);
    rot_in_1(R, T, A);
    mul_ab(pFn, Fi, T);
    mul_ab(T, Fn, Mp);
    mul_ab(Mp, pFi, T);
    rot_in_1(R, T, Mp);
    bad = !cp_start<HE>(cm, A, Mp, g_n, a.lam_n[qg], x);
  }
  int flag = bad ? 1 : 0;
  if (a.warm) {
    // a caller's start is taken when its residual merit is below the plain start's
    const double gscale = 1.0 / (fabs(cm.gs0 - cm.g0) * g_n + 1e-300);
    double xw[11];
#pragma unroll
    for (int i = 0; i < 9; ++i) T[i] = a.warm[i * NQ + qg];
    rot_in_1(R, T, xw);
    xw[9] = a.warm[9 * NQ + qg];
    xw[10] = a.warm[10 * NQ + qg];
    CPPoint p;
    double mw = 0.0, mp = 0.0;
    const bool okw = cp_point<HE, FLOW>(cm, A, det_pFn, g_n, a.dt, xw, p);
    if (okw) mw = cp_merit(p, gscale);
    const bool okp = !bad && cp_point<HE, FLOW>(cm, A, det_pFn, g_n, a.dt, x, p);
    if (okp) mp = cp_merit(p, gscale);
    if (okw && (!okp || mw < mp)) flag |= 2;
  }
  double *row = a.qpbuf + qrec(qg);
#pragma unroll
  for (int i = 0; i < 11; ++i) row[i * kRecStride] = x[i];
  row[kStartFlag * kRecStride] = double(flag);
}

// ------------------------------------------------------------------- Newton kernel
// The lane's slots of the Newton kernel's LDS: A (9), x (11), dx (11), det pF(n), g(n), gscale.
constexpr int kA = 0, kX = 9, kDX = 20, kDet = 31, kGn = 32, kGs = 33;
// A step's system with pivoting, formed again from G and the residual's right-hand side (rec) and from
// A and x (pk): with a copy of the matrix in scratch memory a pass without pivoting took 125 us instead of
// 123 (10,368 points).
__device__ __forceinline__ bool step_pivot(const double *rec, const double *pk, double dt, double (&Ah)[81],
                                           double (&u)[2][9]) {
  LocalLin L;
  double M[9], Mi[9], A[9], eF[9], AtE[9], T[9], dM;
#pragma unroll
  for (int i = 0; i < 9; ++i) {
    M[i] = pk[(kX + i) * 64];
    A[i] = pk[(kA + i) * 64];
  }
  inv_det(M, Mi, dM);
  const double pJ = pk[kDet * 64] / dM;
  mm3(A, M, eF);
  mtm3(A, eF, AtE);
#pragma unroll
  for (int i = 0; i < 54; ++i) L.G[i / 6][i % 6] = rec[i * kRecStride];
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      const int r = i * 3 + j;
      T[r] = Mi[j * 3 + i];
      u[0][r] = rec[(54 + r) * kRecStride];
      u[1][r] = -pJ * T[r];
    }
  cp_matrix(L, AtE, T, dt * pk[(kX + 9) * 64] * pJ, Ah);
  int piv[9];
  const bool ok = factor_pivot<9>(Ah, piv);
  solve_pivot<9>(Ah, piv, u[0]);
  solve_pivot<9>(Ah, piv, u[1]);
  return ok;
}
// One wave per workgroup, one QP per lane: wave w works through QPs [w*chunk, (w+1)*chunk) of the
// block, or, with a.qnext set, draws them from one global queue.  Which lane takes a QP does not
// change its result.  A wave hands out new QPs when kRefill of its lanes are idle: at each idle lane it
// would wait for that QP's state too often (no gain over whole batches), and in whole batches it
// waits for the batch's last QP: with up to 25 iterations (178,752 QPs) the pass took 1000 us at 64,
// 900 at 48, 32 and 16; with a mean of 5 and at most 8 (998,250 QPs) all are within 2%.  The starting
// points come from cp_start_kernel (qpbuf).
//
// Bound by FP64 issue: a turn is about 3300 instructions for 64 QPs.  A turn has no divergent
// branch around its stages (values would be kept across it), and each stage is closed by pin, so
// the widest stretch, the 9 x 9 elimination, fits 300 registers with nothing spilled.  One wave
// per SIMD: at two, 256 registers spill and it takes 800 us instead of 740 (998,250 QPs; 2743 us
// in the sample frame, with the pivoting and the slip systems' tensors in registers).
template <bool HE, int FLOW>
__global__ __launch_bounds__(64) void cp_newton(CPArgs a, int64_t chunk) {
  const int lane = threadIdx.x;
  const int64_t NQ = a.n_qp;
  // The lane's QP data that lives across turns sits in LDS (lane-fastest; each lane touches
  // only its own slots), read where used, rather than in registers held through the material
  // point and the elimination: A (9), x (11), dx (11), det pF(n), g(n), gscale.  17 KB per wave.
  __shared__ double sPk[34 * 64];
  double *pk = sPk + lane;  // field i at pk[i * 64]
  constexpr int kRefill = 48;
  const double dt = a.dt;
  const CPMaterial cm = a.cpmats[0];  // one material for every CP point: wave-uniform, loaded once
  // the lane's phase: evaluate the start, a line-search trial x + alpha dx, the full step after 40
  // halvings without a decrease, or x once more, for a step with a pivoting elimination
  constexpr int kPhStart = 0, kPhTrial = 1, kPhFull = 2, kPhAgain = 3, kPhDone = 4;
  int64_t next = int64_t(blockIdx.x) * chunk;  // the range's first point that no lane has taken
  const int64_t q_hi = a.qnext ? a.nq : (next + chunk < a.nq ? next + chunk : a.nq);
  bool more = true;
  int64_t q = -1;  // the lane's point
  int kind = 0;    // its start: 0 plain, 1 the caller's (learned), 2 the caller's, then the plain fallback
  int phase = kPhDone, it = 0, it_att = 0, ls = 0;
  bool bad_start = false, failed = false;
  double f0 = 0.0, alpha = 1.0;
  for (;;) {
    const uint64_t idle = __ballot(phase == kPhDone);
    const int n_idle = __popcll(idle);
    if (n_idle == 64 || (more && n_idle >= kRefill)) {
      if (phase == kPhDone && q >= 0) {
        const int64_t qg = a.qp_base + q;
        a.iters[qg] = it | (kind << 24);  // iterations, and the start in the high byte
        if (failed) {
          atomicAdd(a.err, 1);
        } else {
          // pF(n+1) = M^-1 pF(n)
          double x[11], Mc[9], Mi[9] = {}, pFn[9], pF1[9], det;
#pragma unroll
          for (int i = 0; i < 11; ++i) x[i] = pk[(kX + i) * 64];
          rot_out_1(a.grains[a.qgrain[q]].R, x, Mc);
          inv_det(Mc, Mi, det);
#pragma unroll
          for (int i = 0; i < 9; ++i) pFn[i] = a.pF_n[i * NQ + qg];
          mul_ab(Mi, pFn, pF1);
#pragma unroll
          for (int i = 0; i < 9; ++i) a.pF_np1[i * NQ + qg] = pF1[i];
          a.Sc_np1[qg] = x[10];
          a.Sc_np1[NQ + qg] = x[9];
        }
      }
      if (phase == kPhDone) q = -1;
      if (more) {
        if (a.qnext) {
          unsigned long long base = 0;
          if (lane == 0) base = atomicAdd(a.qnext, (unsigned long long)n_idle);
          next = int64_t(__shfl((long long)base, 0));
        }
        const int64_t mine = next + __popcll(idle & ((1ull << lane) - 1));
        next += n_idle;
        more = next < q_hi;
        if (phase == kPhDone && mine < q_hi) {
          q = mine;
          const int64_t qg = a.qp_base + q;
          kind = it = it_att = ls = 0;
          failed = false;
          double F[9], pFn[9], pFi[9], T[9], A[9], det = 0.0;
#pragma unroll
          for (int i = 0; i < 9; ++i) {
            F[i] = a.F_np1[i * NQ + qg];
            pFn[i] = a.pF_n[i * NQ + qg];
            pFi[i] = 0.0;
          }
          const double *R = a.grains[a.qgrain[q]].R;
          inv_det(pFn, pFi, det);
          mul_ab(F, pFi, T);
          rot_in_1(R, T, A);
#pragma unroll
          for (int i = 0; i < 9; ++i) pk[(kA + i) * 64] = A[i];
          pk[kDet * 64] = det;
          const double g_n = a.g_n[qg];
          pk[kGn * 64] = g_n;
          pk[kGs * 64] = 1.0 / (fabs(cm.gs0 - cm.g0) * g_n + 1e-300);
          phase = kPhStart;
          // start: the caller's warm start where cp_start_kernel chose it, else the plain start
          const double *row = a.qpbuf + qrec(qg);
          const int flag = int(row[kStartFlag * kRecStride]);
          bad_start = (flag & 1) != 0;
          if (flag & 2) {
#pragma unroll
            for (int i = 0; i < 9; ++i) T[i] = a.warm[i * NQ + qg];
            rot_in_1(R, T, A);
#pragma unroll
            for (int i = 0; i < 9; ++i) pk[(kX + i) * 64] = A[i];
            pk[(kX + 9) * 64] = a.warm[9 * NQ + qg];
            pk[(kX + 10) * 64] = a.warm[10 * NQ + qg];
            kind = 1;
            bad_start = false;
          } else {
#pragma unroll
            for (int i = 0; i < 11; ++i) pk[(kX + i) * 64] = row[i * kRecStride];
          }
        }
      }
      if (!__any(phase != kPhDone)) break;
    }
    // One turn: every live lane evaluates the material point once, at its start or at its
    // line-search trial x + alpha dx; a lane whose start or accepted trial this is then takes a
    // Newton step from it.  A trial's evaluation is thus also the point of the next iteration.
    // A lane whose elimination asked for pivoting takes the same step once more in the next turn, beside
    // the wave's other lanes, with a copy of what its system is made of in the point's record.
    const bool again = phase == kPhAgain, turn = phase != kPhDone;
    const bool moved = phase == kPhTrial || phase == kPhFull;
    const double len = phase == kPhTrial ? alpha : (phase == kPhFull ? 1.0 : 0.0);
    double xc[11], A[9];
#pragma unroll
    for (int i = 0; i < 11; ++i) {
      const double x = pk[(kX + i) * 64], xm = x + len * pk[(kDX + i) * 64];
      xc[i] = moved ? xm : x;
    }
#pragma unroll
    for (int i = 0; i < 9; ++i) A[i] = pk[(kA + i) * 64];
    CPPoint p;
    bool valid = cp_point<HE, FLOW>(cm, A, pk[kDet * 64], pk[kGn * 64], dt, xc, p);
    valid = valid && !(phase == kPhStart && bad_start);
    const double merit = cp_merit(p, pk[kGs * 64]);
    const bool accept = turn && moved && valid && (phase == kPhFull || merit <= (1.0 - 1e-4 * alpha) * f0);
    bool fail = turn && !valid && phase != kPhTrial;
    if (turn && phase == kPhTrial && !accept) {
      alpha *= 0.5;
      if (++ls == 40) phase = kPhFull;  // no decrease found: the full step, if it is valid
    }
    if (accept) {
#pragma unroll
      for (int i = 0; i < 11; ++i) pk[(kX + i) * 64] = xc[i];
    }
    // the iteration that took this step may have been the last
    fail = fail || (accept && it_att >= cm.maxit);
    const bool step = turn && !fail && (accept || (!moved && valid));
    if (phase == kPhStart ? turn : (accept && step)) {
      ++it;
      ++it_att;
    }
    if (__builtin_amdgcn_readfirstlane(__any(step))) {
      // The point of this step (the start, or the accepted trial) is x in LDS.  The slip sums are
      // the widest stretch, so the residual waits in dx's slots and the frames are formed again
      // from A and x afterwards; e then takes those slots over the elimination.
      double Ah[81], u[2][9], f;
      const double lam = pk[(kX + 9) * 64], rhs_s = -p.R[9], rhs_t = -p.R[10];
      if (step) {
        f0 = merit;
#pragma unroll
        for (int i = 0; i < 9; ++i) pk[(kDX + i) * 64] = p.R[i];
      }
      pin(p.S);
      pin(p.sd);
      LocalLin L;
      end_stage();
      cp_slip_sums<HE>(cm, p, p.sd, L);
#pragma unroll
      for (int r = 0; r < 9; ++r) pin(L.G[r]);
      pin(L.eq);
      end_stage();
      pk = reload(sPk, lane);
      {
        double M[9], Mi[9], eF[9], AtE[9], T[9], E9[9], E9e[9], c[9], dM;
#pragma unroll
        for (int i = 0; i < 9; ++i) {
          M[i] = pk[(kX + i) * 64];
          A[i] = pk[(kA + i) * 64];
        }
        inv_det(M, Mi, dM);
        const double pJ = pk[kDet * 64] / dM, g = pk[(kX + 10) * 64], dl = dt * lam * pJ, mg = -1.0 / (cm.m * g);
        mm3(A, M, eF);
        mtm3(A, eF, AtE);
#pragma unroll
        for (int i = 0; i < 3; ++i)
#pragma unroll
          for (int j = 0; j < 3; ++j) {
            const int r = i * 3 + j;
            T[r] = Mi[j * 3 + i];
            u[0][r] = pk[(kDX + r) * 64];
            c[r] = mg * (u[0][r] - (M[r] - ((i == j) ? 1.0 : 0.0)) + dl * T[r]);  // N from the residual
          }
        cp_fold(cm, dt, g, pk[kGn * 64], p.gsum, p.gs, p.dgs, c, L);
        f = L.f;
        const double tf = rhs_t / f;
        v6_to_9(L.eq, E9);
        mm3(AtE, E9, E9e);
#pragma unroll
        for (int r = 0; r < 9; ++r) {
          u[0][r] = -u[0][r] - c[r] * tf;
          u[1][r] = -pJ * T[r];  // d
        }
        if (step) {
#pragma unroll
          for (int r = 0; r < 9; ++r) pk[(kDX + r) * 64] = L.es * E9e[r];
        }
        pin(u[0]);
        pin(u[1]);
#pragma unroll
        for (int r = 0; r < 9; ++r) pin(L.G[r]);
        if (again) {
          double *rec = a.qpbuf + qrec(a.qp_base + q) + kRecStep * kRecStride;
#pragma unroll
          for (int i = 0; i < 54; ++i) rec[i * kRecStride] = L.G[i / 6][i % 6];
#pragma unroll
          for (int i = 0; i < 9; ++i) rec[(54 + i) * kRecStride] = u[0][i];
        }
        end_stage();
        cp_matrix(L, AtE, T, dl, Ah);
      }
      pin(Ah);
      end_stage();
      pk = reload(sPk, lane);
      bool solved = eliminate<9, 2>(Ah, u, a.max_step);
      if (again) solved = step_pivot(a.qpbuf + qrec(a.qp_base + q) + kRecStep * kRecStride, pk, dt, Ah, u);
      double M[9], Mi[9], dM, du = 0.0, dv = 0.0, ex = 0.0, dx[11];
#pragma unroll
      for (int i = 0; i < 9; ++i) M[i] = pk[(kX + i) * 64];
      inv_det(M, Mi, dM);
      const double pJ = pk[kDet * 64] / dM;
#pragma unroll
      for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j) {
          const double d = -pJ * Mi[j * 3 + i];
          du += d * u[0][i * 3 + j];
          dv += d * u[1][i * 3 + j];
        }
      const double yd = (du - rhs_s) / dv;  // dt times the step's multiplier of b
#pragma unroll
      for (int i = 0; i < 9; ++i) {
        dx[i] = u[0][i] - yd * u[1][i];
        ex += pk[(kDX + i) * 64] * dx[i];
      }
      dx[9] = yd / dt - lam / pJ * rhs_s;
      dx[10] = (rhs_t - ex) / f;
      double size = 0.0;
#pragma unroll
      for (int i = 0; i < 9; ++i) size = fmax(size, fabs(dx[i]));
      size = fmax(size, fabs(dx[9]) * dt);
      size = fmax(size, fabs(dx[10]) / pk[kGn * 64]);
      if (step) {
        if (!solved) {
          fail = again;  // singular
          phase = kPhAgain;
        } else if (size < cm.tol) {
#pragma unroll
          for (int i = 0; i < 11; ++i) pk[(kX + i) * 64] = pk[(kX + i) * 64] + dx[i];
          phase = kPhDone;
        } else {  // backtracking on half the squared residual norm, from the full step
#pragma unroll
          for (int i = 0; i < 11; ++i) pk[(kDX + i) * 64] = dx[i];
          alpha = 1.0;
          ls = 0;
          phase = kPhTrial;
        }
      }
    }
    if (fail) {
      if (kind == 1) {
        // the warm start did not converge: fall back to the plain start with a fresh budget
        // (iterations keep counting)
        kind = 2;
        it_att = 0;
        const double *row = a.qpbuf + qrec(a.qp_base + q);
#pragma unroll
        for (int i = 0; i < 11; ++i) pk[(kX + i) * 64] = row[i * kRecStride];
        bad_start = (int(row[kStartFlag * kRecStride]) & 1) != 0;
        phase = kPhStart;
      } else {
        failed = true;
        phase = kPhDone;
      }
    }
  }
}

// ------------------------------------------------------------------- tangent kernel
// At the stored converged state (F, pF(n), pF(n+1), g, lambda): S, tau, gdot, Me, pJ and,
// with WITH_D, dMe/dF = pF(n)^-1 dM/dF from the implicit derivative of the local system.
//
// Column c = (i, j) of F moves the system like dM does, through six numbers: dtau_a/dF_c =
// kR6 q_a . kappa_c with kappa_c the symmetric part of u (x) w, u row i of R eF and w row j of
// R pF(n)^-1 M (products in the crystal frame, their outer index in the sample frame, where F
// is).  So with the hardening row eliminated its right-hand side is -G kappa_c, and
//   (B + G K) z_c = -G kappa_c,  B = I + lp T (.)^T T,
//   z_c = -H (I + K H)^-1 kappa_c,  H = B^-1 G:
// a 6 x 6 system serves the nine columns and the border's b, with no sum over slip systems and
// no 9 x 9 factor.  lp is of the order of the squared strain increment (1e-7 at 1e-3), so H
// comes by the series in lp, to the last bit.  A point where lp is not small, or where the
// 6 x 6 elimination meets a multiplier above kMaxMultTangent, is left to cp_tangent_pivot, which takes
// the 9 x 9 system with pivoting.  998,250 QPs in 575 us, of them 130 for the moduli, instead of the
// 1066 us of the sample-frame kernel with its pivoted 9 x 9 and without the moduli (25 instead of 61
// us for 10,368).
// Bound by FP64 issue and latency at one wave per SIMD: G, the columns and the frames are 512
// registers.  The columns run in a rolled loop with what is indexed by the column in LDS.
constexpr double kMaxLp = 0.01;

// X <- T X^T T scaled by c
__device__ __forceinline__ void lp_term(const double *T, double c, double *X) {
  double Y[9];
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int j = 0; j < 3; ++j)
      Y[i * 3 + j] = c * (T[i * 3] * X[j * 3] + T[i * 3 + 1] * X[j * 3 + 1] + T[i * 3 + 2] * X[j * 3 + 2]);
  mm3(Y, T, X);
}
// K X
__device__ __forceinline__ void k_of(const double *AtE, const double *X, double *k) {
  double Y[9];
  mtm3(AtE, X, Y);
#pragma unroll
  for (int I = 0; I < 3; ++I) k[I] = Y[I * 4];
  k[3] = Y[1] + Y[3];
  k[4] = Y[5] + Y[7];
  k[5] = Y[2] + Y[6];
}
__device__ __forceinline__ void kappa(const double *u, const double *w, double *k) {
#pragma unroll
  for (int I = 0; I < 3; ++I) k[I] = u[I] * w[I];
  k[3] = u[0] * w[1] + u[1] * w[0];
  k[4] = u[1] * w[2] + u[2] * w[1];
  k[5] = u[0] * w[2] + u[2] * w[0];
}

struct TangentPoint {
  double R[9], pFi[9], A[9], Me[9], x[11], pJ, g_n;
  CPPoint p;
};
template <bool HE, int FLOW>
__device__ __forceinline__ bool tangent_point(const CPArgs &a, const CPMaterial &cm, int64_t t, TangentPoint &q) {
  const int64_t NQ = a.n_qp, qg = a.qp_base + t;
  const double *R = a.grains[a.qgrain[t]].R;
  double F[9], pFn[9], pF1[9], T[9], det_pFn;
#pragma unroll
  for (int i = 0; i < 9; ++i) {
    q.R[i] = R[i];
    F[i] = a.F_np1[i * NQ + qg];
    pFn[i] = a.pF_n[i * NQ + qg];
    pF1[i] = a.pF_np1[i * NQ + qg];
  }
  q.g_n = a.g_n[qg];
  if (!inv_det(pFn, q.pFi, det_pFn) || !inv_det(pF1, q.Me, q.pJ)) return false;
  mul_ab(F, q.pFi, T);
  rot_in_1(q.R, T, q.A);
  mul_ab(pFn, q.Me, T);
  rot_in_1(q.R, T, q.x);  // M = pF(n) pF(n+1)^-1
  q.x[9] = a.Sc_np1[NQ + qg];
  q.x[10] = a.Sc_np1[qg];
  return cp_point<HE, FLOW>(cm, q.A, det_pFn, q.g_n, a.dt, q.x, q.p);
}
// U = R eF, W = R pF(n)^-1 M and R pF(n)^-1 (second indices in the crystal frame)
__device__ __forceinline__ void tangent_frames(const TangentPoint &q, double *U, double *W, double *RpFi) {
  mul_ab(q.R, q.p.eF, U);
  mul_ab(q.pFi, q.R, RpFi);
  mul_ab(RpFi, q.x, W);
}
// dMe/dF[:, c] = pF(n)^-1 dM/dF[:, c], from dM in the crystal frame
__device__ __forceinline__ void store_dMe(const TangentPoint &q, const double *RpFi, const double *dM, int c, double *out) {
  double H[9], D[9];
  mm3(RpFi, dM, H);
  mmt3(H, q.R, D);
#pragma unroll
  for (int r = 0; r < 9; ++r) out[(16 + c * 9 + r) * kRecStride] = D[r];
}

template <bool HE>
__device__ __forceinline__ void tangent_lin(const CPMaterial &cm, double dt, const TangentPoint &q, double *AtE,
                                            LocalLin &L) {
  double c[9];
  const double mg = -1.0 / (cm.m * q.x[10]);
#pragma unroll
  for (int r = 0; r < 9; ++r) c[r] = mg * q.p.N[r];
  cp_slip_sums<HE>(cm, q.p, q.p.sd, L);
  cp_fold(cm, dt, q.x[10], q.g_n, q.p.gsum, q.p.gs, q.p.dgs, c, L);
  mtm3(q.A, q.p.eF, AtE);
}

// What the element kernel needs of a point, at its deformation gradient Fr (the pass's; the state's
// own when the pass integrates): T = detJ w pJ Fr Sh, Sh = Me S Me^T, whose rows give the residual, and
// for a tangent the moduli A[b j][g l] = dT_bj / dF_gl.  With column (g, l)'s dM (crystal frame),
// U = Fr W and E = sym(U^T (e_g (x) w_l + V dM)) the strain's derivative, V = Fr R pF(n)^-1,
//   dSh = W (L:E) W^T + X + X^T, X = R pF(n)^-1 dM S W^T,
//   A[. j][g l] = detJ w pJ (Fr dSh + e_g (x) Sh_l)_.j
// (dM keeps det M, so -Sh tr(Me^-1 dMe) is zero).  On a lane per point this is 230 multiply-adds a
// column; in the element kernel, from dMe/dF, it ran on one lane of an element's sixteen and then
// on nine.
template <bool HE>
struct PointFrame {
  double Fr[9], U[9], W[9], RpFi[9], AtE[9], N[9], Sh[6], wq;
  HeTan t;
};
template <bool HE>
__device__ __forceinline__ void point_frame(const CPArgs &a, const CPMaterial &cm, int64_t t, const TangentPoint &q,
                                            bool moduli, PointFrame<HE> &f, double *T) {
  const int64_t qg = a.qp_base + t;
  const double *rec = a.qpbuf + qrec(qg);
  if (a.kin & kKinState) {
#pragma unroll
    for (int i = 0; i < 9; ++i) f.Fr[i] = a.F_np1[i * a.n_qp + qg];
  } else {
#pragma unroll
    for (int i = 0; i < 9; ++i) f.Fr[i] = rec[i * kRecStride];
  }
  f.wq = rec[kRecW * kRecStride] * q.pJ;
  double S9[9], V[9], Sh9[9];
  mul_ab(q.pFi, q.R, f.RpFi);
  mul_ab(f.RpFi, q.x, f.W);
  mul_ab(f.Fr, f.W, f.U);
  v6_to_9(q.p.S, S9);
  mul_abt(S9, f.W, f.N);
  mul_ab(f.W, f.N, Sh9);
#pragma unroll
  for (int I = 0; I < 6; ++I) f.Sh[I] = Sh9[vi(I) * 3 + vj(I)];
  v6_to_9(f.Sh, Sh9);
  mul_ab(f.Fr, Sh9, T);
#pragma unroll
  for (int i = 0; i < 9; ++i) T[i] *= f.wq;
  if (moduli) {
    mul_ab(f.Fr, f.RpFi, V);
    mul_atb(V, f.U, f.AtE);
    if constexpr (HE) {
      double Ce[9], Sx[6];
      mul_atb(f.U, f.U, Ce);
      he_law(cm, f.U, Ce, Sx, f.t);
    }
  }
}
// Column (g, l) of the moduli to the record, from its dM; u = row g of U, w = row l of W.
template <bool HE>
__device__ __forceinline__ void store_moduli(const CPMaterial &cm, const PointFrame<HE> &f, const double *u,
                                             const double *w, const double *dM, int g, int l, double *out) {
  double E[6], kd[6], dS[6];
  kappa(u, w, E);
  k_of(f.AtE, dM, kd);
#pragma unroll
  for (int I = 0; I < 6; ++I) E[I] += kd[I];
  if constexpr (HE) {
    const double E9[9] = {E[0], 0.5 * E[3], 0.5 * E[5], 0.5 * E[3], E[1], 0.5 * E[4], 0.5 * E[5], 0.5 * E[4], E[2]};
    he_dot(f.t, E9, dS);
  } else {
    const double tr = cm.c12 * (E[0] + E[1] + E[2]);
#pragma unroll
    for (int I = 0; I < 6; ++I) dS[I] = I < 3 ? cm.c11m12 * E[I] + tr : 0.5 * cm.c44x2 * E[I];
  }
  double dS9[9], X[9], Y[9], Z[9], H[9], Q[9], Sl[3];
  v6_to_9(dS, dS9);
  mul_ab(dM, f.N, Y);
  mul_ab(f.RpFi, Y, X);
  mul_ab(f.W, dS9, Z);
  mul_abt(Z, f.W, H);
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int j = i; j < 3; ++j) H[i * 3 + j] = H[j * 3 + i] = H[i * 3 + j] + X[i * 3 + j] + X[j * 3 + i];
  mul_ab(f.Fr, H, Q);
  Sl[0] = l == 0 ? f.Sh[0] : (l == 1 ? f.Sh[3] : f.Sh[5]);
  Sl[1] = l == 0 ? f.Sh[3] : (l == 1 ? f.Sh[1] : f.Sh[4]);
  Sl[2] = l == 0 ? f.Sh[5] : (l == 1 ? f.Sh[4] : f.Sh[2]);
  double *o = out + (kRecA + (g * 3 + l) * 9) * kRecStride;
#pragma unroll
  for (int b = 0; b < 3; ++b)
#pragma unroll
    for (int j = 0; j < 3; ++j) o[(b * 3 + j) * kRecStride] = f.wq * (Q[b * 3 + j] + (b == g ? Sl[j] : 0.0));
}

// What the tangent kernel leaves in a point's record: T; T and the moduli; or, for the
// three-field element, Me, S, pJ and dMe/dF.
enum : int { kOutPoint = 0, kOutModuli = 1, kOutMe = 2 };

// The record of a point without a tangent: nothing of an earlier pass reaches the element.
template <int OUT>
__device__ __forceinline__ void zero_record(double *out) {
  if constexpr (OUT == kOutMe) {
#pragma unroll
    for (int i = 0; i < 97; ++i) out[i * kRecStride] = 0.0;
  } else {
#pragma unroll
    for (int i = 0; i < 9; ++i) out[i * kRecStride] = 0.0;
    if constexpr (OUT == kOutModuli) {
#pragma unroll
      for (int i = 0; i < 81; ++i) out[(kRecA + i) * kRecStride] = 0.0;
    }
  }
}

// The lanes' LDS of the tangent kernel, field i of a lane at [i * 64]: the columns' kappa -- then their
// solutions -- and the U, W of the moduli, by a run-time column.  36 KB per wave.
constexpr int kColY = 0, kColU = 54, kColW = 63;
template <bool HE, int FLOW, int OUT>
__device__ __forceinline__ double *tangent_slots() {
  __shared__ double sCol[(OUT == kOutPoint ? 1 : 72) * 64];
  return sCol + threadIdx.x;
}
// Column c of the tangent from its dM, in a rolled loop over the columns: U and W in the lane's LDS.
template <bool HE, int OUT>
__device__ __forceinline__ void store_column(const CPMaterial &cm, const TangentPoint &q, const PointFrame<HE> &f,
                                             const double *RpFi, const double *col, const double *dM, int c,
                                             double *out) {
  if constexpr (OUT == kOutModuli) {
    const int g = c / 3, l = c - 3 * g;
    double u[3], w[3];
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      u[i] = col[(kColU + g * 3 + i) * 64];
      w[i] = col[(kColW + l * 3 + i) * 64];
    }
    store_moduli<HE>(cm, f, u, w, dM, g, l, out);
  } else {
    store_dMe(q, RpFi, dM, c, out);
  }
}
// What store_column needs: the point's T to the record and its frame, with U and W to the lane's LDS, or
// R pF(n)^-1.
template <bool HE, int OUT>
__device__ __forceinline__ void open_columns(const CPArgs &a, const CPMaterial &cm, int64_t t, const TangentPoint &q,
                                             PointFrame<HE> &f, double *RpFi, double *col, double *out) {
  if constexpr (OUT == kOutModuli) {
    double T[9];
    point_frame<HE>(a, cm, t, q, true, f, T);
#pragma unroll
    for (int i = 0; i < 9; ++i) out[i * kRecStride] = T[i];  // where Fr was
#pragma unroll
    for (int i = 0; i < 9; ++i) {
      col[(kColU + i) * 64] = f.U[i];
      col[(kColW + i) * 64] = f.W[i];
    }
  } else {
    mul_ab(q.pFi, q.R, RpFi);
  }
}

template <bool HE, int FLOW, int OUT>
__global__ __launch_bounds__(64) void cp_tangent(CPArgs a, int64_t nqb) {
  const int64_t t = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (t >= nqb) return;
  const int64_t NQ = a.n_qp;
  const int64_t qg = a.qp_base + t;
  const CPMaterial cm = a.cpmats[0];
  double *out = a.qpbuf + qrec(qg);  // field i at out[i * kRecStride]
  TangentPoint q;
  if (!tangent_point<HE, FLOW>(a, cm, t, q)) {
    atomicAdd(a.err, 1);
    zero_record<OUT>(out);
    return;
  }
  const CPPoint &p = q.p;
  {
    const double rg = 1.0 / q.x[10];
#pragma unroll
    for (int al = 0; al < 12; ++al) {
      a.tau[al * NQ + qg] = p.tau[al];
      a.gdot[al * NQ + qg] = (fabs(p.sd[al]) * cm.m * q.x[10]) * (p.tau[al] * rg);
    }
    if constexpr (OUT == kOutMe) {
      double S9[9], S[9];
      v6_to_9(p.S, S9);
      rot_out(q.R, S9, S);
#pragma unroll
      for (int i = 0; i < 9; ++i) out[i * kRecStride] = q.Me[i];
#pragma unroll
      for (int I = 0; I < 6; ++I) out[(9 + I) * kRecStride] = S[voigt_i(I) * 3 + voigt_j(I)];
      out[15 * kRecStride] = q.pJ;
    }
  }
  if constexpr (OUT == kOutPoint) {
    PointFrame<HE> f;
    double T[9];
    point_frame<HE>(a, cm, t, q, false, f, T);
#pragma unroll
    for (int i = 0; i < 9; ++i) out[i * kRecStride] = T[i];
  } else {
    LocalLin L;
    double AtE[9];
    tangent_lin<HE>(cm, a.dt, q, AtE, L);
    const double lp = a.dt * q.x[9] * p.pJ;
    double v[9];  // B^-1 T, T the border's b and d up to factors
#pragma unroll
    for (int r = 0; r < 9; ++r) v[r] = p.T[r];
    bool ok = fabs(lp) <= kMaxLp;
    {  // H = B^-1 G and v by the series sum (-lp)^k (T (.)^T T)^k
      double tv[9], size = fabs(lp);
#pragma unroll
      for (int r = 0; r < 9; ++r) tv[r] = v[r];
      for (double sz = size; ok && sz > 1e-17; sz *= 2.0 * size) {
        lp_term(p.T, -lp, tv);
#pragma unroll
        for (int r = 0; r < 9; ++r) v[r] += tv[r];
      }
#pragma unroll
      for (int I = 0; I < 6; ++I) {
        double h[9], th[9];
#pragma unroll
        for (int r = 0; r < 9; ++r) h[r] = th[r] = L.G[r][I];
        for (double sz = size; ok && sz > 1e-17; sz *= 2.0 * size) {
          lp_term(p.T, -lp, th);
#pragma unroll
          for (int r = 0; r < 9; ++r) h[r] += th[r];
        }
#pragma unroll
        for (int r = 0; r < 9; ++r) L.G[r][I] = h[r];
      }
    }
    double *col = tangent_slots<HE, FLOW, OUT>();
    {
      double U[9], W[9], RpFi[9], S6[36], Y[10][6];
      tangent_frames(q, U, W, RpFi);
#pragma unroll
      for (int I = 0; I < 6; ++I) {
        double h[9], k6[6];
#pragma unroll
        for (int r = 0; r < 9; ++r) h[r] = L.G[r][I];
        k_of(AtE, h, k6);
#pragma unroll
        for (int J = 0; J < 6; ++J) S6[J * 6 + I] = k6[J] + (I == J ? 1.0 : 0.0);
      }
#pragma unroll
      for (int c = 0; c < 9; ++c) kappa(U + (c / 3) * 3, W + (c % 3) * 3, Y[c]);
      k_of(AtE, v, Y[9]);
      ok = eliminate<6, 10>(S6, Y, a.max_tangent) && ok;
#pragma unroll
      for (int c = 0; c < 9; ++c)
#pragma unroll
        for (int I = 0; I < 6; ++I) col[(kColY + c * 6 + I) * 64] = Y[c][I];
#pragma unroll
      for (int r = 0; r < 9; ++r)
#pragma unroll
        for (int I = 0; I < 6; ++I) v[r] -= L.G[r][I] * Y[9][I];
    }
    if (!ok) {
      const uint64_t m = __ballot(1);
      if (int(threadIdx.x) == __builtin_ctzll(m)) a.pivots[blockIdx.x] = m;
      return;
    }
    double dv = 0.0;
#pragma unroll
    for (int r = 0; r < 9; ++r) dv += p.T[r] * v[r];
    const double rdv = 1.0 / dv;
    PointFrame<HE> f;
    double RpFi[9];
    open_columns<HE, OUT>(a, cm, t, q, f, RpFi, col, out);
#pragma unroll 1
    for (int c = 0; c < 9; ++c) {
      double dM[9], du = 0.0, y[6];
#pragma unroll
      for (int I = 0; I < 6; ++I) y[I] = col[(kColY + c * 6 + I) * 64];
#pragma unroll
      for (int r = 0; r < 9; ++r) {
        double z = 0.0;
#pragma unroll
        for (int I = 0; I < 6; ++I) z -= L.G[r][I] * y[I];
        dM[r] = z;
        du += p.T[r] * z;
      }
      du *= rdv;
#pragma unroll
      for (int r = 0; r < 9; ++r) dM[r] -= du * v[r];
      store_column<HE, OUT>(cm, q, f, RpFi, col, dM, c, out);
    }
  }
}

// The points that cp_tangent has left to the 9 x 9 system with pivoting, by the masks of its waves: a
// wave looks through `waves` of them, takes a mask's points together and clears it.  A launch of its
// own: beside the common path, in one kernel, it costs that path registers (cp_tangent 705 us instead of
// 575 on 998,250 points), and as a function called there the compiler lost the other lanes' values.
// A tangent pass over 82,944 points that all come here takes 214 us, beside 151 where none does (with
// the points one after another, each lane's system in LDS, 8.2 ms; in the sample frame, where every point
// pivoted, 337).  With nothing to do it takes 5 us, as long as any short launch.
template <bool HE, int FLOW, int OUT>
__device__ __forceinline__ void tangent_pivot(const CPArgs &a, const CPMaterial &cm, int64_t t) {
  double *out = a.qpbuf + qrec(a.qp_base + t), *col = tangent_slots<HE, FLOW, OUT>();
  TangentPoint q;
  if (!tangent_point<HE, FLOW>(a, cm, t, q)) return;  // counted by cp_tangent
  LocalLin L;
  double Ah[81], v[9];
  int piv[9];
  {
    double U[9], W[9], RpFi[9], AtE[9];
    tangent_frames(q, U, W, RpFi);
#pragma unroll
    for (int c = 0; c < 9; ++c) {
      double kp[6];
      kappa(U + (c / 3) * 3, W + (c % 3) * 3, kp);
#pragma unroll
      for (int I = 0; I < 6; ++I) col[(kColY + c * 6 + I) * 64] = kp[I];
    }
    tangent_lin<HE>(cm, a.dt, q, AtE, L);
    cp_matrix(L, AtE, q.p.T, a.dt * q.x[9] * q.p.pJ, Ah);
  }
  if (!factor_pivot<9>(Ah, piv)) {
    atomicAdd(a.err, 1);
    zero_record<OUT>(out);
    return;
  }
#pragma unroll
  for (int r = 0; r < 9; ++r) v[r] = q.p.T[r];
  solve_pivot<9>(Ah, piv, v);
  double dv = 0.0;
#pragma unroll
  for (int r = 0; r < 9; ++r) dv += q.p.T[r] * v[r];
  const double rdv = 1.0 / dv;
  PointFrame<HE> f;
  double RpFi[9];
  open_columns<HE, OUT>(a, cm, t, q, f, RpFi, col, out);
#pragma unroll 1
  for (int c = 0; c < 9; ++c) {
    double dM[9], du = 0.0, y[6];
#pragma unroll
    for (int I = 0; I < 6; ++I) y[I] = col[(kColY + c * 6 + I) * 64];
#pragma unroll
    for (int r = 0; r < 9; ++r) {
      dM[r] = 0.0;
#pragma unroll
      for (int I = 0; I < 6; ++I) dM[r] -= L.G[r][I] * y[I];
    }
    solve_pivot<9>(Ah, piv, dM);
#pragma unroll
    for (int r = 0; r < 9; ++r) du += q.p.T[r] * dM[r];
    du *= rdv;
#pragma unroll
    for (int r = 0; r < 9; ++r) dM[r] -= du * v[r];
    store_column<HE, OUT>(cm, q, f, RpFi, col, dM, c, out);
  }
}
template <bool HE, int FLOW, int OUT>
__global__ __launch_bounds__(64) void cp_tangent_pivot(CPArgs a, int64_t n_waves, int waves) {
  const CPMaterial cm = a.cpmats[0];
  const int64_t w0 = int64_t(blockIdx.x) * waves, w1 = w0 + waves < n_waves ? w0 + waves : n_waves;
#pragma unroll 1
  for (int64_t w = w0; w < w1; ++w) {
    const uint64_t m = a.pivots[w];
    if (!m) continue;
    if ((m >> threadIdx.x) & 1) tangent_pivot<HE, FLOW, OUT>(a, cm, w * 64 + threadIdx.x);
    if (threadIdx.x == 0) a.pivots[w] = 0;
  }
}

// ------------------------------------------------------------------- element kernel
// Rows of the displacement element from the points' records: with T and the moduli A of
// store_moduli, f_ab = sum_j T_bj dN_a,j and K_ab,wg = sum_l (sum_j dN_a,j A[b j][g l]) dN_w,l.
// One lane per row, the points one after another.  Bound by memory: 490 us for 998,250 tet4, 2.3 GB
// moved at 4.8 TB/s, the rate of a copy.  (1417 us with the point's tensors formed here; 716 with the
// rows stored by their lanes, 8 bytes every 104, instead of through LDS; 538 with each store's
// staging offset loaded just before it.)
template <int NNE, int MODE, bool STG>
__global__ __launch_bounds__(256) void cp_elem(CPElemArgs a, int64_t e_begin, int64_t e_end) {
  constexpr int NQP = nqp_of(NNE);
  constexpr int NDE = NNE * 3;
  constexpr int TPE = (NNE == 4) ? 16 : 32;
  constexpr int EPB = 256 / TPE;
  constexpr int QPB = EPB * NQP;  // points per workgroup: a power of two
  constexpr bool RES = (MODE & MODE_RESIDUAL) != 0;
  constexpr bool TAN = (MODE & MODE_TANGENT) != 0;
  constexpr bool DFL = (MODE & MODE_DEFL_LOAD) != 0;  // K times the prescribed increments
  static_assert(!DFL || (TAN && !RES), "MODE_DEFL_LOAD goes with MODE_TANGENT alone");
  static_assert(256 % QPB == 0, "a thread's point is its index modulo QPB");
  constexpr bool WK = TAN && !DFL;  // K rows are written
  constexpr bool WR = RES || DFL;   // the residual entry is written
  __shared__ double s_dl[EPB][DFL ? NDE : 1];
  __shared__ int32_t s_dof[EPB][NDE], s_node[EPB][NNE];
  __shared__ double s_dN[EPB][NQP][NDE];
  __shared__ double s_T[EPB][NQP][RES ? 9 : 1];
  // staging offsets: loaded with the nodes, so that the stores at the end wait for no load
  __shared__ int64_t s_so[EPB][WK && STG ? NNE : 1];
  constexpr int LD = NDE + 1;
  constexpr int EPW = 64 / TPE;
  constexpr int kD = EPB * NQP * (TAN ? 81 : 1);
  constexpr int RE = stage_round(EPW, NDE, kD);
  constexpr int kS = WK && STG ? 4 * RE * NDE * LD : 0;
  __shared__ double s_work[kD > kS ? kD : kS];  // A[b j][g l], row-major, then the staged rows
  auto s_D = reinterpret_cast<double (*)[NQP][TAN ? 81 : 1]>(s_work);

  const int slot = threadIdx.x / TPE, lane = threadIdx.x % TPE;
  const int64_t ie = e_begin + int64_t(blockIdx.x) * EPB + slot;
  const bool active = ie < e_end;
  const int64_t e = (a.elist && active) ? int64_t(a.elist[ie]) : ie;
  if (active && lane < NNE) {
    const int32_t node = a.conn[e * NNE + lane];
    s_node[slot][lane] = node;
    if constexpr (WK && STG) s_so[slot][lane] = a.soff[e * NNE + lane];
#pragma unroll
    for (int b = 0; b < 3; ++b) {
      const int32_t d = a.dofid[int64_t(node) * 3 + b];
      s_dof[slot][lane * 3 + b] = d;
      if constexpr (DFL) s_dl[slot][lane * 3 + b] = (d < 0 && a.defl_d) ? a.defl_d[-d - 1] : 0.0;
    }
  }
  {
    // A thread reads fields of one point, 256 / QPB apart, so that eight consecutive threads read
    // the eight consecutive doubles a field has in a group of records.
    const int qi = threadIdx.x % QPB, sl = qi / NQP, ip = qi % NQP;
    const int64_t iq = e_begin + int64_t(blockIdx.x) * EPB + sl;
    if (iq < e_end) {
      const int64_t eq = a.elist ? int64_t(a.elist[iq]) : iq;
      const double *qb = a.qpbuf + qrec(a.qp_base + eq * NQP + ip);
      if constexpr (TAN) {
        for (int f = threadIdx.x / QPB; f < 81; f += 256 / QPB)
          s_D[sl][ip][(f % 9) * 9 + f / 9] = qb[(kRecA + f) * kRecStride];
      }
      if constexpr (RES) {
        for (int f = threadIdx.x / QPB; f < 9; f += 256 / QPB) s_T[sl][ip][f] = qb[f * kRecStride];
      }
      if (threadIdx.x < QPB) {
        double k, ee, z, wt, Xi[9];
        int_point(NNE, ip, k, ee, z, wt);
        double dN[NDE];
        shape_dN<NNE>(k, ee, z, dN);
#pragma unroll
        for (int i = 0; i < 9; ++i) Xi[i] = qb[(kRecXi + i) * kRecStride];
#pragma unroll
        for (int n = 0; n < NNE; ++n)
#pragma unroll
          for (int ib = 0; ib < 3; ++ib)
            s_dN[sl][ip][n * 3 + ib] =
                dN[n * 3 + 0] * Xi[0 * 3 + ib] + dN[n * 3 + 1] * Xi[1 * 3 + ib] + dN[n * 3 + 2] * Xi[2 * 3 + ib];
      }
    }
  }
  __syncthreads();
  const bool rowlane = active && lane < NDE;
  const int ra = lane / 3, rb = lane % 3;
  double K[TAN ? NDE : 1];
  if constexpr (TAN) {
#pragma unroll
    for (int i = 0; i < NDE; ++i) K[i] = 0.0;
  }
  double fe = 0.0;
  if (rowlane) {
#pragma unroll 1
  for (int ip = 0; ip < NQP; ++ip) {
    const double *dN = s_dN[slot][ip];
    const double ga[3] = {dN[ra * 3], dN[ra * 3 + 1], dN[ra * 3 + 2]};
    if constexpr (RES) {
      const double *T = &s_T[slot][ip][rb * 3];
      fe += T[0] * ga[0] + T[1] * ga[1] + T[2] * ga[2];
    }
    if constexpr (TAN) {
      const double *A = &s_D[slot][ip][rb * 27];
      double zz[9];
#pragma unroll
      for (int c = 0; c < 9; ++c) zz[c] = ga[0] * A[c] + ga[1] * A[9 + c] + ga[2] * A[18 + c];
#pragma unroll
      for (int w = 0; w < NNE; ++w) {
        const double h0 = dN[w * 3], h1 = dN[w * 3 + 1], h2 = dN[w * 3 + 2];
#pragma unroll
        for (int g = 0; g < 3; ++g) K[w * 3 + g] += zz[g * 3] * h0 + zz[g * 3 + 1] * h1 + zz[g * 3 + 2] * h2;
      }
    }
  }
  if constexpr (TAN) {
    double diag = 0.0;
#pragma unroll
    for (int i = 0; i < NDE; ++i) diag = (i == lane) ? K[i] : diag;
    if (!isnormal(diag)) atomicAdd(a.err, 1);
  }
  if constexpr (DFL) {  // f_defl row: K row . prescribed increments (src/load.cc:190-215)
    double s = 0.0;
#pragma unroll
    for (int i = 0; i < NDE; ++i) s += K[i] * s_dl[slot][i];
    fe = s;
  }
  }  // rowlane
  if constexpr (WK && STG) {
    // Gather mode: each wave lays RE of its elements' rows out in LDS as the staging blocks
    // ([node a][row b][K row, residual]) and copies each node block (3 (NDE+1) doubles,
    // zero-padded to whole lines) to its staging offset, consecutive lanes on consecutive doubles.
    // Rows of prescribed DOFs are copied too (nothing reads them; it keeps every line whole);
    // nodes without free DOFs have no block.  No wave waits for another's rows.
    constexpr int PB = stage_block(NNE);
    constexpr int PB2 = PB / 2;  // two doubles per lane (blocks are whole 128-byte lines)
    lds_barrier();  // every lane is done with the moduli
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), wl = threadIdx.x % 64;
    double *st = s_work + wave * (RE * NDE * LD);
#pragma unroll 1
    for (int r0 = wave * EPW; r0 < (wave + 1) * EPW; r0 += RE) {
      if (rowlane && slot >= r0 && slot < r0 + RE) {
        double *row = st + ((slot - r0) * NDE + lane) * LD;
#pragma unroll
        for (int i = 0; i < NDE; ++i) row[i] = K[i];
        row[NDE] = fe;
      }
      __builtin_amdgcn_wave_barrier();
      for (int idx = wl; idx < RE * NNE * PB2; idx += 64) {
        const int el = idx / (NNE * PB2), o = idx - el * (NNE * PB2);
        const int na = o / PB2, ob = 2 * (o - na * PB2);
        if (e_begin + int64_t(blockIdx.x) * EPB + r0 + el >= e_end) continue;
        const int64_t so = s_so[r0 + el][na];
        if (so < 0) continue;
        const double *src = st + (el * NDE + na * 3) * LD + ob;
        dbl2 v;
        v.x = (ob < 3 * LD) ? src[0] : 0.0;
        v.y = (ob + 1 < 3 * LD) ? src[1] : 0.0;
        // streamed past L2: the gather reads it in a later launch
        __builtin_nontemporal_store(v, reinterpret_cast<dbl2 *>(a.stage + so + ob));
      }
      __builtin_amdgcn_wave_barrier();
    }
    return;
  }
  if (!rowlane) return;
  const int32_t dof = s_dof[slot][lane];
  if (dof <= 0) return;
  if constexpr (STG) {  // gather mode, no K rows: the entry alone
    a.stage[int64_t(a.rslot[e * NNE + ra]) * 3 + rb] = fe;
    return;
  }
  const int16_t *off = a.off + (e * NNE + ra) * NNE;
  if constexpr (WR) {
    if (off[ra] <= -2) a.f[dof - 1] = fe;
    else a.f[dof - 1] += fe;
  }
  if constexpr (WK) {
    const int32_t node = s_node[slot][ra];
    int bp = 0;
#pragma unroll
    for (int j = 0; j < 3; ++j) bp += (j < rb && s_dof[slot][ra * 3 + j] > 0) ? 1 : 0;
    double *row = a.vals + (int64_t(a.row_start[node]) + int64_t(bp) * a.rowlen[node]);
    constexpr int H1 = (NNE + 1) / 2;
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      const int w0 = half ? H1 : 0, w1 = half ? NNE : H1;
      int pos[3 * H1];
      double old[3 * H1];
#pragma unroll
      for (int w = w0; w < w1; ++w) {
        const int o = off[w];
        const bool first = o <= -2;
        const int base = first ? (-o - 2) : o;
        int gp = 0;
#pragma unroll
        for (int gg = 0; gg < 3; ++gg) {
          const bool fr = (o != -1) && s_dof[slot][w * 3 + gg] > 0;
          pos[(w - w0) * 3 + gg] = fr ? base + gp : -1;
          gp += fr ? 1 : 0;
          old[(w - w0) * 3 + gg] = (fr && !first) ? row[base + gp - 1] : 0.0;
        }
      }
#pragma unroll
      for (int w = w0; w < w1; ++w)
#pragma unroll
        for (int gg = 0; gg < 3; ++gg) {
          const int pp = pos[(w - w0) * 3 + gg];
          if (pp >= 0) row[pp] = old[(w - w0) * 3 + gg] + K[w * 3 + gg];
        }
    }
  }
}

// ------------------------------------------------------------------- CM3F element kernel
// The three-field (CM3F) element of crystal plasticity with the hyperelastic law, condensed to
// the displacement DOFs (ConstitutiveModelIntregrate::integrate_ss, src/constitutive_model.cc
// :720-880, total Lagrangian, one theta and one P per element; the blocks of CM_ThreeField,
// src/constitutive_model_3f.cc:189-470; condense_K_3F_to_1F / condense_F_3F_to_1F,
// src/condense.cc:304-385).  Per QP, from the tangent pass's qpbuf: M = pF(n+1)^-1, pJ and
// dM/dFb (Fb = (theta/J)^(1/3) F, the model's F); eF = F M with the unscaled F, Sd and Ld the
// deviatoric PK2 and tangent of the neo-Hookean law at eF, dU, ddU = kappa U', kappa U'' at
// theta_e = theta det M.  For a DOF k (node a, component b) with G_k = e_b (x) dN_a:
//   Phi_k = sym(G_k^T F), Psi_k = M^T Phi_k M, tr_k = tr(G_k F^-1),
//   dM_k = dM/dFb : dFb/du_k, dFb/du_k = f (G_k - tr_k/3 F), Lambda_k = tr(M^-1 dM_k),
//   X_k = Psi_k + sym(M^T F^T F dM_k) (the change of the elastic strain),
// and with cw = detJ w pJ (1/Jn), r_k = Psi_k : Sd + P J tr_k:
//   Ru_k  += cw r_k,                       Kup_k += cw J tr_k,
//   Kuu_kl += cw (Psi_k : Ld : X_l + P J (tr_k tr_l - tr(G_k F^-1 G_l F^-1))
//                 + sym(G_k^T G_l) : M Sd M^T + 2 (Phi_k M Sd) : dM_l - Lambda_l r_k),
//   Kut_k += cw (2 sym(M^T Phi_k dM_t) : Sd + Psi_k : Ld : X_t - Lambda_t r_k),
//   Ktu_k += cw (JM (ddU theta JM + dU) - (dU JM - P)) Lambda_k,
//   Rp += cw (J - theta), Rt += cw (dU JM - P), Ktt += cw (JM dU Lambda_t + JM^2 ddU
//   - Lambda_t (dU JM - P)), Ktp -= cw, with the theta direction dM_t = dM/dFb : Fb/(3 theta).
// The element's rows: one lane per DOF row, the QPs one at a time through LDS (the QP's
// tensors, then every column's LX = Ld : X, dM, tr, Lambda, then the row sums).
template <int NNE, int MODE, bool STG>
__global__ __launch_bounds__(256) void cp_tf_elem(CPElemArgs a, int64_t e_begin, int64_t e_end) {
  constexpr int NQP = nqp_of(NNE);
  constexpr int NDE = NNE * 3;
  constexpr int TPE = (NNE == 4) ? 16 : 32;
  constexpr int EPB = 256 / TPE;
  constexpr bool RES = (MODE & MODE_RESIDUAL) != 0;
  constexpr bool TAN = (MODE & MODE_TANGENT) != 0;
  constexpr bool DFL = (MODE & MODE_DEFL_LOAD) != 0;
  static_assert(!DFL || (TAN && !RES), "MODE_DEFL_LOAD goes with MODE_TANGENT alone");
  constexpr bool WK = TAN && !DFL;
  constexpr bool WR = RES || DFL;
  // per QP tensors in s_q: Fr 0, M 9, M^-1 18, M^T Cr 27, Sd 36, M Sd M^T 45, Ci (Voigt) 54,
  // c1 c2 c3 60, dM/dFb : Fr 63, dM_t 72, Ld : X_t (Voigt) 81, cw 87, J 88, JM 89, dU 90,
  // ddU 91, f 92, Lambda_t 93, dU JM - P 94, M Sd 95, M Sd dM_t^T 104, Fr^-1 113
  constexpr int QD = 122;
  constexpr int CD = 17;  // per DOF column: LX (Voigt) 0, dM 6, tr 15, Lambda 16
  __shared__ double s_x[EPB][NDE], s_u[EPB][NDE];
  __shared__ double s_dl[EPB][DFL ? NDE : 1];
  __shared__ int32_t s_dof[EPB][NDE], s_node[EPB][NNE];
  __shared__ double s_dN[EPB][NQP][NDE], s_w[EPB][NQP];
  __shared__ double s_q[EPB][QD], s_D[EPB][81], s_col[EPB][NDE][CD], s_gn[EPB][NDE];
  __shared__ double s_vec[EPB][2][NDE];

  const int slot = threadIdx.x / TPE, lane = threadIdx.x % TPE;
  const int64_t ie = e_begin + int64_t(blockIdx.x) * EPB + slot;
  const bool active = ie < e_end;
  const int64_t e = (a.elist && active) ? int64_t(a.elist[ie]) : ie;
  if (active && lane < NNE) {
    const int32_t node = a.conn[e * NNE + lane];
    s_node[slot][lane] = node;
#pragma unroll
    for (int b = 0; b < 3; ++b) {
      s_x[slot][lane * 3 + b] = a.X[int64_t(node) * 3 + b];
      const int32_t d = a.dofid[int64_t(node) * 3 + b];
      s_dof[slot][lane * 3 + b] = d;
      double u = 0.0, dl = 0.0;
      if (d > 0) {
        u = a.r[d - 1] + (a.d_r ? a.d_r[d - 1] : 0.0);
      } else if (d < 0) {
        dl = a.defl_d ? a.defl_d[-d - 1] : 0.0;
        u = (a.defl ? a.defl[-d - 1] : 0.0) + (DFL ? 0.0 : dl);
      }
      s_u[slot][lane * 3 + b] = u;
      if constexpr (DFL) s_dl[slot][lane * 3 + b] = dl;
    }
  }
  __syncthreads();
  if (active && lane < NQP) {  // physical shape-function gradients and detJ w of every QP
    const int ip = lane;
    double k, ee, z, wt;
    int_point(NNE, ip, k, ee, z, wt);
    double dN[NDE];
    shape_dN<NNE>(k, ee, z, dN);
    double dX[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
    for (int n = 0; n < NNE; ++n)
#pragma unroll
      for (int ib = 0; ib < 3; ++ib)
#pragma unroll
        for (int ic = 0; ic < 3; ++ic) dX[ib * 3 + ic] += dN[n * 3 + ic] * s_x[slot][n * 3 + ib];
    const double J0 = det3(dX);
    double Xi[9];
    const bool ok = J0 > 0.0 && inv3(dX, Xi);
    if (!ok) atomicAdd(a.err, 1);
#pragma unroll
    for (int n = 0; n < NNE; ++n)
#pragma unroll
      for (int ib = 0; ib < 3; ++ib)
        s_dN[slot][ip][n * 3 + ib] =
            dN[n * 3 + 0] * Xi[0 * 3 + ib] + dN[n * 3 + 1] * Xi[1 * 3 + ib] + dN[n * 3 + 2] * Xi[2 * 3 + ib];
    s_w[slot][ip] = ok ? J0 * wt : 0.0;
  }
  const double theta = active ? a.tf_V[e] + a.tf_dV[e] : 1.0;
  const double Pp = active ? a.tf_P[e] + a.tf_dP[e] : 0.0;
  const CPMaterial cm = a.cpmats[0];
  const bool rowlane = active && lane < NDE;
  const int ra = lane / 3, rb = lane % 3;
  double K[NDE];
#pragma unroll
  for (int i = 0; i < NDE; ++i) K[i] = 0.0;
  double Ru = 0.0, Kup = 0.0, Kut = 0.0, Ktu = 0.0, Rp = 0.0, Rt = 0.0, Ktt = 0.0, Ktp = 0.0;
  __syncthreads();
#pragma unroll 1
  for (int ip = 0; ip < NQP; ++ip) {
    if (active) {
      const double *qb = a.qpbuf + qrec(a.qp_base + e * NQP + ip);
      for (int f = lane; f < 81; f += TPE) s_D[slot][(f % 9) * 9 + f / 9] = qb[(16 + f) * kRecStride];
    }
    lds_barrier();
    // the QP's tensors in three rounds, lanes of an element working side by side
    double *q = s_q[slot];
    if (active && lane == 0) {  // Fr, M, M^-1, Fr^-1, J, det M
      const double *dN = s_dN[slot][ip];
      double Fr[9] = {1, 0, 0, 0, 1, 0, 0, 0, 1};
#pragma unroll
      for (int n = 0; n < NNE; ++n)
#pragma unroll
        for (int ib = 0; ib < 3; ++ib)
#pragma unroll
          for (int ic = 0; ic < 3; ++ic) Fr[ib * 3 + ic] += s_u[slot][n * 3 + ib] * dN[n * 3 + ic];
      const double *qb = a.qpbuf + qrec(a.qp_base + e * NQP + ip);
      double Me[9], Mi[9], Fi[9];
#pragma unroll
      for (int i = 0; i < 9; ++i) Me[i] = qb[i * kRecStride];
      const double J = det3(Fr);
      const bool okq = J > 0.0 && theta > 0.0 && inv3(Fr, Fi) && inv3(Me, Mi);
      if (!okq) atomicAdd(a.err, 1);
#pragma unroll
      for (int i = 0; i < 9; ++i) {
        q[i] = Fr[i];
        q[9 + i] = Me[i];
        q[18 + i] = Mi[i];
        q[113 + i] = Fi[i];
      }
      q[87] = okq ? s_w[slot][ip] * qb[15 * kRecStride] : 0.0;  // detJ w / Jn, 1/Jn = pJ
      q[88] = J;
      q[89] = det3(Me);
      q[92] = okq ? cbrt(theta / J) : 1.0;
    }
    lds_barrier();
    if (active && lane == 0) {  // M^T Cr
      double Cr[9], MtC[9];
      mtm3(q, q, Cr);
      mtm3(q + 9, Cr, MtC);
#pragma unroll
      for (int i = 0; i < 9; ++i) q[27 + i] = MtC[i];
    } else if (active && lane == 1) {
      // neo-Hookean deviatoric PK2 and tangent coefficients at Ce = (F M)^T F M (he_law
      // without kappa), and the volumetric derivatives at theta_e = theta det M
      double eF[9], Ce[9], Ci9[9];
      mm3(q, q + 9, eF);
      mtm3(eF, eF, Ce);
      inv3(Ce, Ci9);
      const double d = pow(det3(Ce), -1.0 / 3.0);
      const double trC = Ce[0] + Ce[4] + Ce[8];
      const double aa = 2.0 * cm.m10 * d;
#pragma unroll
      for (int i = 0; i < 9; ++i) q[36 + i] = aa * ((i % 4 == 0) ? 1.0 : 0.0) - aa * trC * (1.0 / 3.0) * Ci9[i];
#pragma unroll
      for (int I = 0; I < 6; ++I) q[54 + I] = Ci9[vi(I) * 3 + vj(I)];
      q[60] = 2.0 * aa * trC * (1.0 / 9.0);
      q[61] = -2.0 * aa * (1.0 / 3.0);
      q[62] = 2.0 * aa * trC * (1.0 / 3.0);
      const double JM = q[89];
      double dU, ddU;
      vol_pot(cm.vol_flag, theta * JM, dU, ddU);
      q[90] = dU * cm.kappa;
      q[91] = ddU * cm.kappa;
      q[94] = dU * cm.kappa * JM - Pp;
    } else if (active && lane >= 2 && lane < 11) {  // row r of dM/dFb : Fr and of dM_t
      const int r = lane - 2;
      double sd = 0.0;
#pragma unroll
      for (int c = 0; c < 9; ++c) sd += s_D[slot][r * 9 + c] * q[c];
      q[63 + r] = sd;
      q[72 + r] = q[92] / (3.0 * theta) * sd;  // dM_t = f / (3 theta) dM/dFb : Fr
    }
    lds_barrier();
    if (active && lane == 0) {  // tr(M^-1 dM_t) and Ld : sym(M^T Cr dM_t)
      double Lt = 0.0;
#pragma unroll
      for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j) Lt += q[18 + i * 3 + j] * q[72 + j * 3 + i];
      q[93] = Lt;
      double T[9], Xt[9], LXt[6];
      mm3(q + 27, q + 72, T);
#pragma unroll
      for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j) Xt[i * 3 + j] = 0.5 * (T[i * 3 + j] + T[j * 3 + i]);
      HeTan td;
#pragma unroll
      for (int I = 0; I < 6; ++I) td.Ci[I] = q[54 + I];
      td.c1 = q[60];
      td.c2 = q[61];
      td.c3 = q[62];
      he_dot(td, Xt, LXt);
#pragma unroll
      for (int I = 0; I < 6; ++I) q[81 + I] = LXt[I];
    } else if (active && lane == 1) {  // M Sd, M Sd M^T, M Sd dM_t^T
      double MeSd[9];
      mm3(q + 9, q + 36, MeSd);
#pragma unroll
      for (int i = 0; i < 9; ++i) q[95 + i] = MeSd[i];
#pragma unroll
      for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j) {
          q[45 + i * 3 + j] = MeSd[i * 3 + 0] * q[9 + j * 3 + 0] + MeSd[i * 3 + 1] * q[9 + j * 3 + 1] +
                              MeSd[i * 3 + 2] * q[9 + j * 3 + 2];
          q[104 + i * 3 + j] = MeSd[i * 3 + 0] * q[72 + j * 3 + 0] + MeSd[i * 3 + 1] * q[72 + j * 3 + 1] +
                               MeSd[i * 3 + 2] * q[72 + j * 3 + 2];
        }
    }
    lds_barrier();
    const double *dN = s_dN[slot][ip];
    double Psi[9], Phi[9];
    if (rowlane) {  // the DOF's column data, and the row's own Psi
      const double *Fr = q, *Me = q + 9, *Fi = q + 113;
      const double ga[3] = {dN[ra * 3], dN[ra * 3 + 1], dN[ra * 3 + 2]};
#pragma unroll
      for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j) Phi[i * 3 + j] = 0.5 * (ga[i] * Fr[rb * 3 + j] + ga[j] * Fr[rb * 3 + i]);
      double T[9];
      mm3(Phi, Me, T);
      mtm3(Me, T, Psi);
      // g_a = F^-T dN_a: tr_k = g_a,b
      double g[3];
#pragma unroll
      for (int i = 0; i < 3; ++i) g[i] = ga[0] * Fi[0 * 3 + i] + ga[1] * Fi[1 * 3 + i] + ga[2] * Fi[2 * 3 + i];
      s_gn[slot][lane] = g[rb];
      const double trk = g[rb], fac = q[92];
      double dM[9];
#pragma unroll
      for (int r = 0; r < 9; ++r) {
        const double *Dr = s_D[slot] + r * 9 + rb * 3;
        dM[r] = fac * (Dr[0] * ga[0] + Dr[1] * ga[1] + Dr[2] * ga[2] - trk * (1.0 / 3.0) * q[63 + r]);
      }
      double Lk = 0.0;
#pragma unroll
      for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j) Lk += q[18 + i * 3 + j] * dM[j * 3 + i];
      double X[9], V[9];
      mm3(q + 27, dM, V);
#pragma unroll
      for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j) X[i * 3 + j] = Psi[i * 3 + j] + 0.5 * (V[i * 3 + j] + V[j * 3 + i]);
      HeTan td;
#pragma unroll
      for (int I = 0; I < 6; ++I) td.Ci[I] = q[54 + I];
      td.c1 = q[60];
      td.c2 = q[61];
      td.c3 = q[62];
      double LX[6];
      he_dot(td, X, LX);
      double *col = s_col[slot][lane];
#pragma unroll
      for (int I = 0; I < 6; ++I) col[I] = LX[I];
#pragma unroll
      for (int r = 0; r < 9; ++r) col[6 + r] = dM[r];
      col[15] = trk;
      col[16] = Lk;
    }
    lds_barrier();
    if (active) {
      const double cw = q[87], J = q[88], JM = q[89], dU = q[90], ddU = q[91], Lt = q[93], vt = q[94];
      Rp += cw * (J - theta);  // compute_Rp
      Rt += cw * vt;           // compute_Rt
      Ktt += cw * (JM * dU * Lt + JM * JM * ddU - Lt * vt);  // compute_Ktt
      Ktp -= cw;               // compute_Ktp
    }
    if (rowlane) {
      const double cw = q[87], J = q[88], JM = q[89], dU = q[90], ddU = q[91], Lt = q[93], vt = q[94];
      const double *Sd = q + 36;
      double PsiS = 0.0;
#pragma unroll
      for (int i = 0; i < 9; ++i) PsiS += Psi[i] * Sd[i];
      const double trk = s_col[slot][lane][15], Lk = s_col[slot][lane][16];
      const double rk = PsiS + Pp * J * trk;
      // Psi : Ld : X_t and 2 sym(M^T Phi dM_t) : Sd = 2 Phi : (M Sd dM_t^T)
      const double *LXt = q + 81, *W = q + 104;
      const double PLt = Psi[0] * LXt[0] + Psi[4] * LXt[1] + Psi[8] * LXt[2] +
                         2.0 * (Psi[1] * LXt[3] + Psi[5] * LXt[4] + Psi[2] * LXt[5]);
      double DtS = 0.0;
#pragma unroll
      for (int i = 0; i < 9; ++i) DtS += 2.0 * Phi[i] * W[i];
      Ru += cw * rk;                                                // compute_Ru
      Kup += cw * J * trk;                                          // compute_Kup
      Kut += cw * (DtS + PLt - Lt * rk);                            // compute_Kut
      Ktu += cw * (JM * (ddU * theta * JM + dU) * Lk - Lk * vt);    // compute_Ktu
      if constexpr (TAN) {
        // Z = 2 Phi_k M Sd, t = M Sd M^T dN_a
        double Z[9];
        mm3(Phi, q + 95, Z);
        const double *Sh = q + 45;
        const double ga[3] = {dN[ra * 3], dN[ra * 3 + 1], dN[ra * 3 + 2]};
        double ta[3];
#pragma unroll
        for (int i = 0; i < 3; ++i) ta[i] = Sh[i * 3] * ga[0] + Sh[i * 3 + 1] * ga[1] + Sh[i * 3 + 2] * ga[2];
        double gk[3];  // g_a (F^-T dN_a), all three components
#pragma unroll
        for (int i = 0; i < 3; ++i) gk[i] = s_gn[slot][ra * 3 + i];
        // not unrolled: the column data are read from LDS one column at a time (unrolled, the
        // compiler hoists all of them and spills)
#pragma unroll 1
        for (int l = 0; l < NDE; ++l) {
          const int w = l / 3, bp = l % 3;
          const double *col = s_col[slot][l];
          const double PLX = Psi[0] * col[0] + Psi[4] * col[1] + Psi[8] * col[2] +
                             2.0 * (Psi[1] * col[3] + Psi[5] * col[4] + Psi[2] * col[5]);
          double dMS = 0.0;
#pragma unroll
          for (int i = 0; i < 9; ++i) dMS += 2.0 * Z[i] * col[6 + i];
          const double GGS = (bp == rb) ? ta[0] * dN[w * 3] + ta[1] * dN[w * 3 + 1] + ta[2] * dN[w * 3 + 2] : 0.0;
          const double tr2 = gk[bp] * s_gn[slot][w * 3 + rb];
          K[l] += cw * (PLX + Pp * J * (trk * col[15] - tr2) + GGS + dMS - col[16] * rk);  // compute_Kuu
        }
      }
    }
    lds_barrier();  // the next QP overwrites s_q, s_D, s_col, s_gn
  }
  // condensation: K = Kuu - Kup Ktu / Ktp + Kup Ktt Kpu / (Ktp Kpt) - Kut Kpu / Kpt, with
  // Kpu = Kup^T, Kpt = Ktp (IntegrateThreeFieldStiffness::out_loop, constitutive_model.cc:531-555)
  if (rowlane) {
    s_vec[slot][0][lane] = Kup;
    s_vec[slot][1][lane] = Ktu;
  }
  lds_barrier();
  double fe = 0.0;
  if (rowlane) {
    const double Kpt = Ktp;
    if constexpr (TAN) {
#pragma unroll
      for (int l = 0; l < NDE; ++l)
        K[l] = K[l] - Kup / Ktp * s_vec[slot][1][l] + Kup / Ktp * Ktt / Kpt * s_vec[slot][0][l] -
               Kut / Kpt * s_vec[slot][0][l];
      double diag = 0.0;
#pragma unroll
      for (int i = 0; i < NDE; ++i) diag = (i == lane) ? K[i] : diag;
      if (!isnormal(diag)) atomicAdd(a.err, 1);
    }
    if constexpr (RES) fe = Ru + Kup / Ktp * Ktt / Kpt * Rp - Kup / Ktp * Rt - Kut / Kpt * Rp;
    if constexpr (DFL) {
      double s = 0.0;
#pragma unroll
      for (int i = 0; i < NDE; ++i) s += K[i] * s_dl[slot][i];
      fe = s;
    }
    if constexpr (RES) {  // the element update's data (compute_d_theta_dP)
      double *tb = a.tf_buf + e * kTfBuf;
      tb[lane] = Kup;
      tb[kTfKtu + lane] = Ktu;
      if (lane == 0) {
        tb[NDE] = Rp;
        tb[NDE + 1] = Rt;
        tb[NDE + 2] = Ktt;
        tb[NDE + 3] = -Ktp;
      }
    }
  }
  if (!rowlane) return;
  const int32_t dof = s_dof[slot][lane];
  if (dof <= 0) return;
  constexpr int LD = NDE + 1;
  if constexpr (STG) {  // gather mode: the row straight into its staging block, or the entry alone
    if constexpr (WK) {
      double *srow = a.stage + a.soff[e * NNE + ra] + rb * LD;
#pragma unroll
      for (int i = 0; i < NDE; ++i) srow[i] = K[i];
      if constexpr (WR) srow[NDE] = fe;
    } else {
      a.stage[int64_t(a.rslot[e * NNE + ra]) * 3 + rb] = fe;
    }
    return;
  }
  const int16_t *off = a.off + (e * NNE + ra) * NNE;
  if constexpr (WR) {
    if (off[ra] <= -2) a.f[dof - 1] = fe;
    else a.f[dof - 1] += fe;
  }
  if constexpr (WK) {
    const int32_t node = s_node[slot][ra];
    int bp = 0;
#pragma unroll
    for (int j = 0; j < 3; ++j) bp += (j < rb && s_dof[slot][ra * 3 + j] > 0) ? 1 : 0;
    double *row = a.vals + (int64_t(a.row_start[node]) + int64_t(bp) * a.rowlen[node]);
#pragma unroll
    for (int w = 0; w < NNE; ++w) {
      const int o = off[w];
      if (o == -1) continue;
      const bool first = o <= -2;
      const int base = first ? (-o - 2) : o;
      int gp = 0;
#pragma unroll
      for (int gg = 0; gg < 3; ++gg) {
        if (s_dof[slot][w * 3 + gg] <= 0) continue;
        double *p = row + base + gp;
        *p = first ? K[w * 3 + gg] : *p + K[w * 3 + gg];
        ++gp;
      }
    }
  }
}

template <int NNE, int MODE>
void launch_tfe(const CPElemArgs &a, int64_t e0, int64_t e1, hipStream_t s) {
  constexpr int TPE = (NNE == 4) ? 16 : 32;
  constexpr int EPB = 256 / TPE;
  const int64_t n = e1 - e0;
  if (n <= 0) return;
  const unsigned grid = unsigned((n + EPB - 1) / EPB);
  if (a.stage) cp_tf_elem<NNE, MODE, true><<<grid, 256, 0, s>>>(a, e0, e1);
  else cp_tf_elem<NNE, MODE, false><<<grid, 256, 0, s>>>(a, e0, e1);
}

template <int NNE>
void launch_tfe_mode(int mode, const CPElemArgs &a, int64_t e0, int64_t e1, hipStream_t s) {
  switch (mode & (MODE_RESIDUAL | MODE_TANGENT | MODE_DEFL_LOAD)) {
    case MODE_RESIDUAL: launch_tfe<NNE, MODE_RESIDUAL>(a, e0, e1, s); break;
    case MODE_TANGENT: launch_tfe<NNE, MODE_TANGENT>(a, e0, e1, s); break;
    case MODE_RESIDUAL | MODE_TANGENT: launch_tfe<NNE, MODE_RESIDUAL | MODE_TANGENT>(a, e0, e1, s); break;
    case MODE_TANGENT | MODE_DEFL_LOAD: launch_tfe<NNE, MODE_TANGENT | MODE_DEFL_LOAD>(a, e0, e1, s); break;
    default: break;
  }
}

template <int NNE>
void launch_kin(const CPArgs &a, hipStream_t s) {
  const int64_t n = a.ne * nqp_of(NNE);
  if (n <= 0) return;
  cp_kinematics<NNE><<<unsigned((n + 255) / 256), 256, 0, s>>>(a);
}

template <int NNE, int MODE>
void launch_ce(const CPElemArgs &a, int64_t e0, int64_t e1, hipStream_t s) {
  constexpr int TPE = (NNE == 4) ? 16 : 32;
  constexpr int EPB = 256 / TPE;
  const int64_t n = e1 - e0;
  if (n <= 0) return;
  const unsigned grid = unsigned((n + EPB - 1) / EPB);
  if (a.stage) cp_elem<NNE, MODE, true><<<grid, 256, 0, s>>>(a, e0, e1);
  else cp_elem<NNE, MODE, false><<<grid, 256, 0, s>>>(a, e0, e1);
}

template <int NNE>
void launch_ce_mode(int mode, const CPElemArgs &a, int64_t e0, int64_t e1, hipStream_t s) {
  switch (mode & (MODE_RESIDUAL | MODE_TANGENT | MODE_DEFL_LOAD)) {
    case MODE_RESIDUAL: launch_ce<NNE, MODE_RESIDUAL>(a, e0, e1, s); break;
    case MODE_TANGENT: launch_ce<NNE, MODE_TANGENT>(a, e0, e1, s); break;
    case MODE_RESIDUAL | MODE_TANGENT: launch_ce<NNE, MODE_RESIDUAL | MODE_TANGENT>(a, e0, e1, s); break;
    case MODE_TANGENT | MODE_DEFL_LOAD: launch_ce<NNE, MODE_TANGENT | MODE_DEFL_LOAD>(a, e0, e1, s); break;
    default: break;
  }
}

// ------------------------------------------------------------------- output variables
// One thread per element of a block: the stress from the stored state at the level, as
// constitutive_model_update_output_variables forms it (src/constitutive_model.cc:1738-1875):
// eF = F pF^-1 (J2 and the hyperelastic model: the elastic left stretch from Cp^-1), the elastic
// stress of the model on eF, sigma = eF eS eF^T / theta_e, S = theta F^-1 sigma F^-T,
// E = (F^T F - I)/2 per QP; sigma and e = (I - (F F^T)^-1)/2 (compute_Eulerian_Almansi_strain,
// src/utils.cc:46-56) averaged over the element with detJ w, shear strains doubled.
template <int NNE>
__global__ __launch_bounds__(256) void output_kernel(OutArgs o) {
  constexpr int NQP = nqp_of(NNE);
  const int64_t e = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (e >= o.ne) return;
  double x[NNE * 3];
#pragma unroll
  for (int n = 0; n < NNE; ++n) {
    const int32_t node = o.conn[e * NNE + n];
#pragma unroll
    for (int b = 0; b < 3; ++b) x[n * 3 + b] = o.X[int64_t(node) * 3 + b];
  }
  // the reference's output order XX, YY, ZZ, YZ, XZ, XY as (i, j)
  const int oi[6] = {0, 1, 2, 1, 0, 0}, oj[6] = {0, 1, 2, 2, 2, 1};
  double vol = 0.0, sa[6] = {0, 0, 0, 0, 0, 0}, ea[6] = {0, 0, 0, 0, 0, 0};
  const DevMaterial m = o.mats[o.mat ? o.mat[e] : 0];
  for (int ip = 0; ip < NQP; ++ip) {
    double k, ee, z, wt;
    int_point(NNE, ip, k, ee, z, wt);
    double dN[NNE * 3];
    shape_dN<NNE>(k, ee, z, dN);
    double dX[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
    for (int n = 0; n < NNE; ++n)
#pragma unroll
      for (int ib = 0; ib < 3; ++ib)
#pragma unroll
        for (int ic = 0; ic < 3; ++ic) dX[ib * 3 + ic] += dN[n * 3 + ic] * x[n * 3 + ib];
    const double w = det3(dX) * wt;
    const int64_t q = o.qp_base + e * NQP + ip;
    const int64_t NQ = o.n_qp;
    double F[9], Fi[9];
#pragma unroll
    for (int i = 0; i < 9; ++i) F[i] = o.F[i * NQ + q];
    const double J = det3(F);
    inv3(F, Fi);
    double sig[9];  // Cauchy
    if (o.model == PGF_MODEL_CRYSTAL_PLASTICITY) {
      const CPMaterial cm = o.cpmats[0];
      double pF[9], pFi[9], eF[9], Ce[9], S6[6], S9[9], T[9];
#pragma unroll
      for (int i = 0; i < 9; ++i) pF[i] = o.P[i * NQ + q];
      inv3(pF, pFi);
      mm3(F, pFi, eF);
      mtm3(eF, eF, Ce);
      if (cm.law == 1) {
        HeTan t;
        he_law(cm, eF, Ce, S6, t);
      } else {
        double E[9];
#pragma unroll
        for (int i = 0; i < 9; ++i) E[i] = 0.5 * (Ce[i] - ((i % 4 == 0) ? 1.0 : 0.0));
        const double cub[3] = {cm.c11m12, cm.c12, cm.c44x2};
        cubic_dot(o.grains[o.qgrain[q - o.qp_base]].R, cub, E, S6);
      }
      v6_to_9(S6, S9);
      const double rte = 1.0 / det3(eF);
      mm3(eF, S9, T);
#pragma unroll
      for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j)
          sig[i * 3 + j] = rte * (T[i * 3] * eF[j * 3] + T[i * 3 + 1] * eF[j * 3 + 1] + T[i * 3 + 2] * eF[j * 3 + 2]);
    } else {
      // bbar_e = J^-2/3 F Cp^-1 F^T (Cp^-1 = I for the hyperelastic model); tau = G dev bbar_e +
      // kappa J U'(J) 1, scaled by (1 - w) with J2 damage; sigma = tau / J
      double Cn[9] = {1, 0, 0, 0, 1, 0, 0, 0, 1};
      if (o.model == PGF_MODEL_J2_PLASTICITY) {
        const double c6[6] = {o.P[0 * NQ + q], o.P[1 * NQ + q], o.P[2 * NQ + q],
                              o.P[3 * NQ + q], o.P[4 * NQ + q], o.P[5 * NQ + q]};
        Cn[0] = c6[0]; Cn[4] = c6[1]; Cn[8] = c6[2];
        Cn[1] = Cn[3] = c6[3];
        Cn[5] = Cn[7] = c6[4];
        Cn[2] = Cn[6] = c6[5];
      }
      double T[9], b[9];
      mm3(F, Cn, T);
#pragma unroll
      for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j)
          b[i * 3 + j] = T[i * 3] * F[j * 3] + T[i * 3 + 1] * F[j * 3 + 1] + T[i * 3 + 2] * F[j * 3 + 2];
      const double cj = cbrt(J);
      const double Jm23 = 1.0 / (cj * cj);
      const double tr3 = (b[0] + b[4] + b[8]) * (1.0 / 3.0);
      double dU, d2U;
      vol_pot(m.volPotFlag, J, dU, d2U);
      const double om = (o.model == PGF_MODEL_J2_PLASTICITY && m.mu > 0.0) ? 1.0 - o.Sc[2 * NQ + q] : 1.0;
      const double rJ = 1.0 / J;
      if (o.model == PGF_MODEL_HYPER_ELASTICITY && m.devPotFlag == 2) {
        // the linear law in C: tau = G (b b - b) + kappa J U'(J) 1
        double bb[9];
        mm3(b, b, bb);
#pragma unroll
        for (int i = 0; i < 9; ++i) sig[i] = rJ * (m.G * (bb[i] - b[i]) + ((i % 4 == 0) ? m.kappa * J * dU : 0.0));
      } else {
#pragma unroll
        for (int i = 0; i < 9; ++i)
          sig[i] = om * rJ * (m.G * Jm23 * (b[i] - ((i % 4 == 0) ? tr3 : 0.0)) + ((i % 4 == 0) ? m.kappa * J * dU : 0.0));
      }
    }
    // S = J F^-1 sigma F^-T, E = (F^T F - I)/2, e = (I - (F F^T)^-1)/2 = (I - Fi^T Fi)/2
    double T[9], S9[9], C[9], bi[9];
    mm3(Fi, sig, T);
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
      for (int j = 0; j < 3; ++j)
        S9[i * 3 + j] = J * (T[i * 3] * Fi[j * 3] + T[i * 3 + 1] * Fi[j * 3 + 1] + T[i * 3 + 2] * Fi[j * 3 + 2]);
    mtm3(F, F, C);
    mtm3(Fi, Fi, bi);
#pragma unroll
    for (int I = 0; I < 6; ++I) {
      const int ij = oi[I] * 3 + oj[I];
      o.S[I * NQ + q] = S9[ij];
      o.E[I * NQ + q] = 0.5 * (C[ij] - (I < 3 ? 1.0 : 0.0));
      sa[I] += w * sig[ij];
      ea[I] += w * (I < 3 ? 1.0 : 2.0) * 0.5 * ((I < 3 ? 1.0 : 0.0) - bi[ij]);
    }
    vol += w;
  }
  const double rv = 1.0 / vol;
#pragma unroll
  for (int I = 0; I < 6; ++I) {
    o.sig[I * o.ne + e] = sa[I] * rv;
    o.eps[I * o.ne + e] = ea[I] * rv;
  }
}

// ------------------------------------------------------------------- learned warm start
// Features of one QP (device QP order rows of 34): F(n) pF(n)^-1, F(n+1) - F(n), tau_a(n)/g(n),
// grain quaternion; with shift/scale the row is normalised as (x - shift) * scale.
__global__ void cp_features(CPArgs a, const float *gquat, const float *shift, const float *scale, float *X) {
  const int64_t t = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (t >= a.nq) return;
  const int64_t NQ = a.n_qp, qg = a.qp_base + t;
  double Fn[9], pFn[9], pFi[9], Fe[9];
#pragma unroll
  for (int i = 0; i < 9; ++i) {
    Fn[i] = a.F_n[i * NQ + qg];
    pFn[i] = a.pF_n[i * NQ + qg];
  }
  if (!inv3(pFn, pFi)) {
#pragma unroll
    for (int i = 0; i < 9; ++i) pFi[i] = (i % 4 == 0) ? 1.0 : 0.0;
  }
  mm3(Fn, pFi, Fe);
  float f[34];
#pragma unroll
  for (int i = 0; i < 9; ++i) {
    f[i] = float(Fe[i]);
    f[9 + i] = float(a.F_np1[i * NQ + qg] - Fn[i]);
  }
  // the resolved shear stresses at n over the slip resistance at n (the flow rule's ratio)
  const double rg = 1.0 / a.g_n[qg];
#pragma unroll
  for (int i = 0; i < 12; ++i) f[18 + i] = float(a.tau_n[i * NQ + qg] * rg);
  const int gid = a.qgrain[t];
#pragma unroll
  for (int i = 0; i < 4; ++i) f[30 + i] = gquat[gid * 4 + i];
  float *row = X + qg * 34;
#pragma unroll
  for (int i = 0; i < 34; ++i) row[i] = shift ? (f[i] - shift[i]) * scale[i] : f[i];
}

// Targets: dt * gamma_dot(n+1), rows of 12.
__global__ void cp_targets(CPArgs a, float *T) {
  const int64_t t = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (t >= a.nq) return;
  const int64_t NQ = a.n_qp, qg = a.qp_base + t;
#pragma unroll
  for (int i = 0; i < 12; ++i) T[qg * 12 + i] = float(a.dt * a.gdot[i * NQ + qg]);
}

// Warm start from predicted slip increments (block-local rows of Y, ldy apart):
// M = I - sum_a dgamma_a P_a (first order in the increments), lambda = lambda(n) and g from
// the closed-form hardening update at the predicted total slip rate.
__global__ void cp_warm_from_slip(CPArgs a, const float *Y, int ldy, const float *out_scale, double *warm) {
  const int64_t t = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (t >= a.nq) return;
  const int64_t NQ = a.n_qp, qg = a.qp_base + t;
  const DevGrain &gr = a.grains[a.qgrain[t]];
  const CPMaterial cm = a.cpmats[0];
  double dg[12], gsum = 0.0;
#pragma unroll
  for (int i = 0; i < 12; ++i) {
    dg[i] = double(Y[t * ldy + i]) / double(out_scale[i]);
    gsum += fabs(dg[i]);
  }
  gsum /= a.dt;
#pragma unroll
  for (int i = 0; i < 9; ++i) {
    double s = 0.0;
#pragma unroll
    for (int al = 0; al < 12; ++al) s += dg[al] * gr.P[al][i];
    warm[i * NQ + qg] = ((i % 4 == 0) ? 1.0 : 0.0) - s;
  }
  double gs = cm.gs0;
  if (cm.w != 0.0) gs = (gsum / cm.gds > 1.0e-15) ? cm.gs0 * pow(gsum / cm.gds, cm.w) : 0.0;
  const double g_n = a.g_n[qg];
  const double num = (gs - cm.g0) * g_n + a.dt * cm.h0 * gs * gsum;
  const double den = gs - cm.g0 + a.dt * cm.h0 * gsum;
  warm[9 * NQ + qg] = a.lam_n[qg];
  warm[10 * NQ + qg] = (den != 0.0 && num / den > 0.0) ? num / den : g_n;
}

}  // namespace

void launch_cp_features(const CPArgs &a, const float *gquat, const float *shift, const float *scale, float *X,
                        hipStream_t s) {
  if (a.nq > 0) cp_features<<<unsigned((a.nq + 255) / 256), 256, 0, s>>>(a, gquat, shift, scale, X);
}
void launch_cp_targets(const CPArgs &a, float *T, hipStream_t s) {
  if (a.nq > 0) cp_targets<<<unsigned((a.nq + 255) / 256), 256, 0, s>>>(a, T);
}
void launch_cp_warm_from_slip(const CPArgs &a, const float *Y, int ldy, const float *out_scale, double *warm,
                              hipStream_t s) {
  if (a.nq > 0) cp_warm_from_slip<<<unsigned((a.nq + 255) / 256), 256, 0, s>>>(a, Y, ldy, out_scale, warm);
}

void launch_output(int nne, const OutArgs &o, hipStream_t s) {
  if (o.ne <= 0) return;
  const unsigned grid = unsigned((o.ne + 255) / 256);
  if (nne == 4) output_kernel<4><<<grid, 256, 0, s>>>(o);
  else if (nne == 10) output_kernel<10><<<grid, 256, 0, s>>>(o);
  else if (nne == 8) output_kernel<8><<<grid, 256, 0, s>>>(o);
}

void launch_cp_kinematics(int nne, const CPArgs &a, hipStream_t s) {
  if (nne == 4) launch_kin<4>(a, s);
  else if (nne == 10) launch_kin<10>(a, s);
  else if (nne == 8) launch_kin<8>(a, s);
}

__global__ void cp_queue_reset(unsigned long long *q) { *q = 0; }
// resident waves of the persistent Newton kernel on an MI355X: 256 CUs x 4 SIMDs, one wave each
constexpr int64_t kQueueWaves = 1024;

// run(HE, FLOW) for the material's elastic law and flow rule
template <class F>
void by_law(const CPArgs &a, F run) {
  const auto flow = [&](auto he) {
    if (a.flow == kFlowPlain) run(he, std::integral_constant<int, kFlowPlain>{});
    else if (a.flow == kFlowSat) run(he, std::integral_constant<int, kFlowSat>{});
    else run(he, std::integral_constant<int, kFlowPow>{});
  };
  if (a.law == 1) flow(std::true_type{});
  else flow(std::false_type{});
}

void launch_cp_newton(const CPArgs &a, int64_t chunk, hipStream_t s) {
  const int64_t nq = a.nq;
  if (nq <= 0) return;
  CPArgs b = a;
  // Up to two batches per wave the queue has nothing to balance (380 us against 373 for a pass over
  // 100,736 QPs); above, it keeps the waves filled (178,752 QPs, up to 25 iterations: 1000 -> 900).
  if (nq <= 2 * 64 * kQueueWaves) b.qnext = nullptr;
  if (b.qnext) {
    // one persistent wave per SIMD of the chip (the kernel takes more than 256 registers of a lane),
    // draining the global queue; the counter is reset by a kernel, so a captured pass replays it
    cp_queue_reset<<<1, 1, 0, s>>>(b.qnext);
    chunk = 64;
  } else if (chunk < 64) {
    chunk = 64;
  }
  const unsigned grid = b.qnext ? unsigned(std::min<int64_t>((nq + 63) / 64, kQueueWaves))
                                : unsigned((nq + chunk - 1) / chunk);
  const unsigned sgrid = unsigned((nq + 63) / 64);
  const auto run = [&](auto he, auto fl) {
    constexpr bool HE = decltype(he)::value;
    constexpr int FLOW = decltype(fl)::value;
    cp_start_kernel<HE, FLOW><<<sgrid, 64, 0, s>>>(a);
    cp_newton<HE, FLOW><<<grid, 64, 0, s>>>(b, chunk);
  };
  by_law(a, run);
}

void launch_cp_tangent(const CPArgs &a, bool with_D, hipStream_t s) {
  const int64_t nq = a.nq;
  if (nq <= 0) return;
  const unsigned grid = unsigned((nq + 63) / 64);
  // masks per wave of cp_tangent_pivot: one until the chip's 1024 waves are busy twice over, few
  // enough waves beyond that a launch that finds nothing stays short
  const unsigned waves = (grid + 2 * kQueueWaves - 1) / (2 * kQueueWaves);
  by_law(a, [&](auto he, auto fl) {
    constexpr bool HE = decltype(he)::value;
    constexpr int FLOW = decltype(fl)::value;
    const auto columns = [&](auto out) {
      constexpr int OUT = decltype(out)::value;
      cp_tangent<HE, FLOW, OUT><<<grid, 64, 0, s>>>(a, nq);
      cp_tangent_pivot<HE, FLOW, OUT><<<(grid + waves - 1) / waves, 64, 0, s>>>(a, grid, int(waves));
    };
    if (a.tf) columns(std::integral_constant<int, kOutMe>{});
    else if (with_D) columns(std::integral_constant<int, kOutModuli>{});
    else cp_tangent<HE, FLOW, kOutPoint><<<grid, 64, 0, s>>>(a, nq);
  });
}

void launch_cp_elem(int nne, int mode, const CPElemArgs &a, int64_t e0, int64_t e1, hipStream_t s) {
  if (nne == 4) launch_ce_mode<4>(mode, a, e0, e1, s);
  else if (nne == 10) launch_ce_mode<10>(mode, a, e0, e1, s);
  else if (nne == 8) launch_ce_mode<8>(mode, a, e0, e1, s);
}
void launch_cp_tf_elem(int nne, int mode, const CPElemArgs &a, int64_t e0, int64_t e1, hipStream_t s) {
  if (nne == 4) launch_tfe_mode<4>(mode, a, e0, e1, s);
  else if (nne == 10) launch_tfe_mode<10>(mode, a, e0, e1, s);
  else if (nne == 8) launch_tfe_mode<8>(mode, a, e0, e1, s);
}

}  // namespace pgf
