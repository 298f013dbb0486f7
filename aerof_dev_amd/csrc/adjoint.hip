// adjoint.hip -- transposed residual derivatives on gfx950:
//   dRdU^T lambda and dRdX^T lambda for the second-order residual
//   R_i = (1/V_i) (sum_edges +-F(V_ij, V_ji, n_ij) + sum_faces F_b(V_i, n_f/3))
// (SpaceOperator::computeTransposeDerivativeOfResidual, SpaceOperator.C:1235-1304,
//  and the sensitivity operators of EdgeSet, Edge.C:1452-1728, on the same
//  residual; the reference builds per-edge sparse operator blocks, here each
//  edge contracts its local derivatives with the adjoint weights at once).
//
// The MUSCL gradients are recomputed by a forward residual pass at the start
// of each call; nothing from an earlier forward evaluation is kept.
//
// Stages (all deterministic: per-edge, per-tet and per-face results go to
// their own slots and each node sums its slots in a fixed order):
//   1. forward residual: V, LSQ gradients g, R (scaled); mu = lambda/V
//   2. k_adj_edges  one lane per edge: w = mu_i - mu_j; w^T dF/d(V_ij, V_ji, n)
//      by the reverse mode of the Roe flux, then reverse through the Van Albada
//      reconstruction by hand -> per edge: Vbar_i, c_i, Vbar_j, c_j, dxbar,
//      nbar; its first blocks: the same per boundary-face slot
//   3. k_adj_nodes  one lane per node: sums its slots -> Vbar, Gbar, the dx
//      part of Xbar; then the reverse of the LSQ gradients' own node.  With
//      M g = sum_j dx_ij (V_j - V_i), M = sum_j dx_ij dx_ij^T and H = M^-1 Gbar,
//        d(Gbar . g) = sum_j d[dx_ij . H (V_j - V_i)] - H . (dM g),
//      so H and the symmetric S = -(H g^T + g H^T) are all that is passed on
//   4. k_adj_lsq    one lane per node, with K = H_i + H_j:
//      Vbar_i -= K dx_ij, Xbar_i -= K (V_j - V_i) + (S_i + S_j) dx_ij, then
//      Ubar = (dV/dU)^T Vbar
//   5. k_adj_tets / k_adj_faces: control-volume, dual-normal and face-normal
//      geometry, reverse over each element's coordinates
//   6. k_adj_xgather: Xbar_i plus its tet and face slots
#include <hip/hip_runtime.h>

#include <type_traits>

#include "context.h"
#include "device_dual.h"
#include "device_sens.h"
#include "host_internal.h"

namespace aerofx {

struct Adjoint {
  double *EVi = nullptr;  // il<10> (first order il<5>) over edge positions: Vbar_i, c_i (Gbar_i[d*5+k] = c_i[k] dx[d])
  double *EVj = nullptr;  // the same of the upper end
  double *EXd = nullptr;  // il<3> over edge positions: dxbar
  double *EXn = nullptr;  // il<3> over edge positions: nbar
  double *FV = nullptr;   // [3F][5] Vbar of each node face slot
  double *FN = nullptr;   // [3F][3] its share of the face normal's, at 3 f + local vertex
  double *mu = nullptr;   // il<5>: lambda / V
  double *cvb = nullptr;  // [N] -mu . R
  double *Vb = nullptr;   // il<5>
  double *H = nullptr;    // il<15>
  double *S = nullptr;    // il<6>
  double *Xb = nullptr;   // il<3>
  double *R = nullptr;    // [N][5] forward residual (scaled)
  double *TX = nullptr;   // [T][12]
  double *FX = nullptr;   // [F][9]
  double *Jf = nullptr;   // [F] per-face objective values, then the sum at [F]
  double *h_J = nullptr;  // pinned
  int *tets = nullptr;    // [T][4]
  int *tpos = nullptr;    // [T][6] edge positions
  int *faces = nullptr;   // [F][3]
  int *ntrow = nullptr;   // [N+1]
  int *ntslot = nullptr;  // [4T] 4*t + local vertex
  int *nfslot = nullptr;  // [3F] 3*f + local vertex, in the order of tab.fidx
};

namespace {

constexpr int kAdjBlock = 256;
// ElemTet edge -> (end, end) table (ElemTetCore.C:19-21)
constexpr int kEnd[6][2] = {{0, 1}, {0, 2}, {0, 3}, {1, 2}, {1, 3}, {2, 3}};

__device__ __forceinline__ double seed(int dir, int k) { return dir == k ? 1.0 : 0.0; }

// Reverse mode of roeflux7 (device_physics.h) with evitno = 0, the edge
// call: given the weights g on the five flux components, returns
// bL = g^T dphi/dUg, bR = g^T dphi/dUd and be = g^T dphi/den.  The forward
// statements are repeated in their order (the same upwind branch), then each is
// reversed in the opposite order: one forward and one reverse sweep, with each
// reciprocal and root formed once.
__device__ __forceinline__ void roeflux7_vjp(const Gas &gs, const double e[3], const double L[5], const double R[5],
                                             const double g[5], double bL[5], double bR[5], double be[3]) {
#pragma clang fp contract(on)
  const double gam = gs.gam, gam1 = gs.gam1, invgam1 = gs.invgam1, ps = gs.pstiff;
  // ---- forward
  const double rn2 = e[0] * e[0] + e[1] * e[1] + e[2] * e[2];
  const double invnorm = frsq(rn2);
  const double rnorm = sqrt_from_rsq(rn2, invnorm);
  const double n0 = e[0] * invnorm, n1 = e[1] * invnorm, n2 = e[2] * invnorm;
  const double vitg2 = L[1] * L[1] + L[2] * L[2] + L[3] * L[3];
  const double vitd2 = R[1] * R[1] + R[2] * R[2] + R[3] * R[3];
  const double is1 = frsq(L[0]), is2 = frsq(R[0]);
  const double s1 = sqrt_from_rsq(L[0], is1), s2 = sqrt_from_rsq(R[0], is2);
  const double ener1 = (L[4] + gam * ps) * invgam1 + 0.5 * L[0] * vitg2;
  const double ener2 = (R[4] + gam * ps) * invgam1 + 0.5 * R[0] * vitd2;
  const double usro = frcp(s1 + s2);
  const double m2 = s1 * L[1] + s2 * R[1], m3 = s1 * L[2] + s2 * R[2], m4n = s1 * L[3] + s2 * R[3];
  const double u2 = m2 * usro, u3 = m3 * usro, u4 = m4n * usro;
  const double A1 = (ener1 + L[4]) * is1, A2 = (ener2 + R[4]) * is2;
  const double u5 = (A1 + A2) * usro;
  const double VdotNt = n0 * u2 + n1 * u3 + n2 * u4;
  const bool left = VdotNt > 0.0;
  const double *S = left ? L : R;
  const double vit2 = left ? vitg2 : vitd2;
  const double VdotN = S[1] * n0 + S[2] * n1 + S[3] * n2;
  const double H0 = gam * (S[4] + ps) + 0.5 * gam1 * S[0] * vit2;
  const double iS0 = left ? is1 * is1 : is2 * is2;
  const double H = H0 * invgam1 * iS0;
  const double p0 = S[0] * VdotN;
  const double p1 = p0 * S[1] + S[4] * n0, p2 = p0 * S[2] + S[4] * n1, p3 = p0 * S[3] + S[4] * n2;
  const double p4 = p0 * H;
  const double qir = 0.5 * (u2 * u2 + u3 * u3 + u4 * u4);
  const double cr2 = gam1 * (u5 - qir);
  const double icr = frsq(cr2);
  const double cr = sqrt_from_rsq(cr2, icr);
  const double icr2 = icr * icr;
  const double vp4 = VdotNt + cr, vp5 = VdotNt - cr;
  const double r = cr, sm = -cr, cb = -cr, itb = -icr;
  const double d1 = -L[0] + R[0];
  const double d2 = -L[0] * L[1] + R[0] * R[1];
  const double d3 = -L[0] * L[2] + R[0] * R[2];
  const double d4 = -L[0] * L[3] + R[0] * R[3];
  const double a1 = VdotNt * d1 - n0 * d2 - n1 * d3 - n2 * d4;
  const double a2 = qir * d1 - u2 * d2 - u3 * d3 - u4 * d4 + (ener2 - ener1);
  double flur4 = 0.0, flur5 = 0.0, mm = 0.0, tt = 0.0;
  if (!left) {
    mm = vp4 > 0.0 ? vp4 : 0.0;
    tt = cb * a1 + gam1 * sm * itb * a2;
    flur4 = mm * tt;
  } else {
    mm = vp5 < 0.0 ? vp5 : 0.0;
    tt = -cb * a1 + (-gam1 * r * itb * a2);
    flur5 = -mm * tt;
  }
  const double fs = flur4 + flur5;
  const double rs = r * flur4 + sm * flur5;
  const double X0 = fs, X1 = n0 * rs + u2 * fs, X2 = n1 * rs + u3 * fs, X3 = n2 * rs + u4 * fs,
               X4 = VdotNt * rs + u5 * fs;
  const double q0 = p0 - 0.5 * X0 * icr2, q1 = p1 - X1 * 0.5 * icr2, q2 = p2 - X2 * 0.5 * icr2,
               q3 = p3 - X3 * 0.5 * icr2, q4 = p4 - X4 * 0.5 * icr2;
  // ---- reverse
  double bLl[5] = {0.0, 0.0, 0.0, 0.0, 0.0}, bRr[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
  // phi_k = q_k rnorm
  double b_rnorm = g[0] * q0 + g[1] * q1 + g[2] * q2 + g[3] * q3 + g[4] * q4;
  const double bq0 = g[0] * rnorm, bq1 = g[1] * rnorm, bq2 = g[2] * rnorm, bq3 = g[3] * rnorm, bq4 = g[4] * rnorm;
  // q_k = p_k - X_k icr2 / 2
  const double c = 0.5 * icr2;
  const double b_icr2 = -0.5 * (bq0 * X0 + bq1 * X1 + bq2 * X2 + bq3 * X3 + bq4 * X4);
  const double bX0 = -c * bq0, bX1 = -c * bq1, bX2 = -c * bq2, bX3 = -c * bq3, bX4 = -c * bq4;
  double b_p0 = bq0;
  const double b_p1 = bq1, b_p2 = bq2, b_p3 = bq3, b_p4 = bq4;
  // X_k
  double b_fs = bX0 + u2 * bX1 + u3 * bX2 + u4 * bX3 + u5 * bX4;
  const double b_rs = n0 * bX1 + n1 * bX2 + n2 * bX3 + VdotNt * bX4;
  double b_n0 = rs * bX1, b_n1 = rs * bX2, b_n2 = rs * bX3;
  double b_u2 = fs * bX1, b_u3 = fs * bX2, b_u4 = fs * bX3, b_u5 = fs * bX4;
  double b_VdotNt = rs * bX4;
  // rs = r flur4 + sm flur5, fs = flur4 + flur5
  const double b_flur4 = b_fs + r * b_rs, b_flur5 = b_fs + sm * b_rs;
  double b_r = flur4 * b_rs, b_sm = flur5 * b_rs, b_cb = 0.0, b_itb = 0.0, b_a1 = 0.0, b_a2 = 0.0;
  double b_vp4 = 0.0, b_vp5 = 0.0;
  if (!left) {
    // flur4 = mm tt, tt = cb a1 + ((gam1 sm) itb) a2
    const double b_mm = tt * b_flur4, b_tt = mm * b_flur4;
    b_vp4 = vp4 > 0.0 ? b_mm : 0.0;
    b_cb += a1 * b_tt;
    b_a1 += cb * b_tt;
    const double k = gam1 * sm * itb;
    b_a2 += k * b_tt;
    const double b_k = a2 * b_tt;
    b_sm += gam1 * itb * b_k;
    b_itb += gam1 * sm * b_k;
  } else {
    // flur5 = -mm tt, tt = -cb a1 + (((-gam1) r) itb) a2
    const double b_mm = -tt * b_flur5, b_tt = -mm * b_flur5;
    b_vp5 = vp5 < 0.0 ? b_mm : 0.0;
    b_cb += -a1 * b_tt;
    b_a1 += -cb * b_tt;
    const double k = -gam1 * r * itb;
    b_a2 += k * b_tt;
    const double b_k = a2 * b_tt;
    b_r += -gam1 * itb * b_k;
    b_itb += -gam1 * r * b_k;
  }
  // a2 = qir d1 - u2 d2 - u3 d3 - u4 d4 + (ener2 - ener1)
  double b_qir = d1 * b_a2;
  double b_d1 = qir * b_a2, b_d2 = -u2 * b_a2, b_d3 = -u3 * b_a2, b_d4 = -u4 * b_a2;
  b_u2 += -d2 * b_a2;
  b_u3 += -d3 * b_a2;
  b_u4 += -d4 * b_a2;
  double b_ener1 = -b_a2, b_ener2 = b_a2;
  // a1 = VdotNt d1 - n0 d2 - n1 d3 - n2 d4
  b_VdotNt += d1 * b_a1;
  b_d1 += VdotNt * b_a1;
  b_n0 += -d2 * b_a1;
  b_n1 += -d3 * b_a1;
  b_n2 += -d4 * b_a1;
  b_d2 += -n0 * b_a1;
  b_d3 += -n1 * b_a1;
  b_d4 += -n2 * b_a1;
  // d1..d4
  bLl[0] += -b_d1 - L[1] * b_d2 - L[2] * b_d3 - L[3] * b_d4;
  bRr[0] += b_d1 + R[1] * b_d2 + R[2] * b_d3 + R[3] * b_d4;
  bLl[1] += -L[0] * b_d2;
  bLl[2] += -L[0] * b_d3;
  bLl[3] += -L[0] * b_d4;
  bRr[1] += R[0] * b_d2;
  bRr[2] += R[0] * b_d3;
  bRr[3] += R[0] * b_d4;
  // r = cr, sm = -cr, cb = -cr, itb = -1/cr; vp4 = VdotNt + cr, vp5 = VdotNt - cr
  double b_cr = b_r - b_sm - b_cb + b_itb * icr2 + b_vp4 - b_vp5;
  b_VdotNt += b_vp4 + b_vp5;
  // icr2 = 1/cr2, cr = sqrt(cr2), cr2 = gam1 (u5 - qir)
  const double b_cr2 = -icr2 * icr2 * b_icr2 + 0.5 * b_cr * icr;
  b_u5 += gam1 * b_cr2;
  b_qir += -gam1 * b_cr2;
  // qir = (u2^2 + u3^2 + u4^2) / 2
  b_u2 += u2 * b_qir;
  b_u3 += u3 * b_qir;
  b_u4 += u4 * b_qir;
  // p1..p4 = p0 S_k + S4 n_k, p0 H
  b_p0 += S[1] * b_p1 + S[2] * b_p2 + S[3] * b_p3 + H * b_p4;
  double bS[5];
  bS[1] = p0 * b_p1;
  bS[2] = p0 * b_p2;
  bS[3] = p0 * b_p3;
  bS[4] = n0 * b_p1 + n1 * b_p2 + n2 * b_p3;
  b_n0 += S[4] * b_p1;
  b_n1 += S[4] * b_p2;
  b_n2 += S[4] * b_p3;
  const double b_H = p0 * b_p4;
  // p0 = S0 VdotN
  bS[0] = VdotN * b_p0;
  const double b_VdotN = S[0] * b_p0;
  // H = H0 / (gam1 S0), H0 = gam (S4 + ps) + gam1 S0 vit2 / 2
  const double b_H0 = b_H * invgam1 * iS0;
  bS[0] += -H * b_H * iS0 + 0.5 * gam1 * vit2 * b_H0;
  bS[4] += gam * b_H0;
  const double b_vit2 = 0.5 * gam1 * S[0] * b_H0;
  // VdotN = S1 n0 + S2 n1 + S3 n2
  bS[1] += n0 * b_VdotN;
  bS[2] += n1 * b_VdotN;
  bS[3] += n2 * b_VdotN;
  b_n0 += S[1] * b_VdotN;
  b_n1 += S[2] * b_VdotN;
  b_n2 += S[3] * b_VdotN;
  double b_vitg2 = 0.0, b_vitd2 = 0.0;
  if (left) {
#pragma unroll
    for (int k = 0; k < 5; ++k) bLl[k] += bS[k];
    b_vitg2 += b_vit2;
  } else {
#pragma unroll
    for (int k = 0; k < 5; ++k) bRr[k] += bS[k];
    b_vitd2 += b_vit2;
  }
  // VdotNt = n0 u2 + n1 u3 + n2 u4
  b_n0 += u2 * b_VdotNt;
  b_n1 += u3 * b_VdotNt;
  b_n2 += u4 * b_VdotNt;
  b_u2 += n0 * b_VdotNt;
  b_u3 += n1 * b_VdotNt;
  b_u4 += n2 * b_VdotNt;
  // u5 = (A1 + A2) usro, A1 = (ener1 + L4) / s1, A2 = (ener2 + R4) / s2
  double b_usro = (A1 + A2) * b_u5;
  const double b_A1 = usro * b_u5, b_A2 = usro * b_u5;
  b_ener1 += b_A1 * is1;
  bLl[4] += b_A1 * is1;
  double b_s1 = -A1 * is1 * b_A1;
  b_ener2 += b_A2 * is2;
  bRr[4] += b_A2 * is2;
  double b_s2 = -A2 * is2 * b_A2;
  // u_c = m_c usro, m_c = s1 L_c + s2 R_c
  b_usro += m2 * b_u2 + m3 * b_u3 + m4n * b_u4;
  const double b_m2 = usro * b_u2, b_m3 = usro * b_u3, b_m4 = usro * b_u4;
  b_s1 += L[1] * b_m2 + L[2] * b_m3 + L[3] * b_m4;
  b_s2 += R[1] * b_m2 + R[2] * b_m3 + R[3] * b_m4;
  bLl[1] += s1 * b_m2;
  bLl[2] += s1 * b_m3;
  bLl[3] += s1 * b_m4;
  bRr[1] += s2 * b_m2;
  bRr[2] += s2 * b_m3;
  bRr[3] += s2 * b_m4;
  // usro = 1 / (s1 + s2)
  b_s1 += -usro * usro * b_usro;
  b_s2 += -usro * usro * b_usro;
  // ener = (p + gam ps) / gam1 + rho vit / 2
  bLl[4] += invgam1 * b_ener1;
  bLl[0] += 0.5 * vitg2 * b_ener1;
  b_vitg2 += 0.5 * L[0] * b_ener1;
  bRr[4] += invgam1 * b_ener2;
  bRr[0] += 0.5 * vitd2 * b_ener2;
  b_vitd2 += 0.5 * R[0] * b_ener2;
  // s = sqrt(rho)
  bLl[0] += 0.5 * b_s1 * is1;
  bRr[0] += 0.5 * b_s2 * is2;
  // vit2 = |u|^2
#pragma unroll
  for (int k = 1; k < 4; ++k) {
    bLl[k] += 2.0 * L[k] * b_vitg2;
    bRr[k] += 2.0 * R[k] * b_vitd2;
  }
  // n = e invnorm, invnorm = 1/rnorm, rnorm = sqrt(rn2)
  const double b_invnorm = e[0] * b_n0 + e[1] * b_n1 + e[2] * b_n2;
  b_rnorm += -invnorm * invnorm * b_invnorm;
  const double b_rn2 = 0.5 * b_rnorm * invnorm;
  be[0] = invnorm * b_n0 + 2.0 * e[0] * b_rn2;
  be[1] = invnorm * b_n1 + 2.0 * e[1] * b_rn2;
  be[2] = invnorm * b_n2 + 2.0 * e[2] * b_rn2;
#pragma unroll
  for (int k = 0; k < 5; ++k) {
    bL[k] = bLl[k];
    bR[k] = bRr[k];
  }
}

// d VA(a, b) / da and / db of the Van Albada function q = num / den (RecFcn.h:269-281)
__device__ __forceinline__ void va_partials(double a, double b, double &da, double &db) {
#pragma clang fp contract(on)
  const double eps = 1.e-16;
  const double a2 = a * a, b2 = b * b, ab = a * b;
  const double id = frcp(a2 + b2 + 2.0 * eps);
  const bool pos = ab > 0.0, zero = ab == 0.0;
  const double num = pos ? ab * (a + b) + eps * (a + b) : (zero ? 0.5 * eps * (a + b) : 0.0);
  const double q2 = 2.0 * (num * id);
  const double na = pos ? 2.0 * ab + (b2 + eps) : (zero ? 0.5 * eps : 0.0);
  const double nb = pos ? 2.0 * ab + (a2 + eps) : (zero ? 0.5 * eps : 0.0);
  da = (na - q2 * a) * id;
  db = (nb - q2 * b) * id;
}

}  // namespace

// mu = lambda / V, and what each control volume's derivative weighs:
// R_i = F_i / V_i, so d/dV_i (lambda_i . R_i) = -mu_i . R_i
__global__ __launch_bounds__(kAdjBlock) void k_adj_mu(DevTables t, const double *__restrict__ lam,
                                                      const double *__restrict__ R, double *__restrict__ mu,
                                                      double *__restrict__ cvb) {
  const int n = blockIdx.x * kAdjBlock + threadIdx.x;
  if (n >= t.N) return;
  const double ic = t.invcv[n];
  double m[5], s = 0.0;
#pragma unroll
  for (int k = 0; k < 5; ++k) {
    m[k] = lam[5 * (size_t)n + k] * ic;
    s += m[k] * R[5 * (size_t)n + k];
  }
  store_il<5>(t.sh, mu, n, m);
  cvb[n] = -s;
}

// ---------------------------------------------------------------------------
// 2. per edge
// ---------------------------------------------------------------------------
// A boundary-face slot: mu^T d(face flux) / d(V, face normal / 3).
template <bool WANTX, int SH>
__device__ __forceinline__ void adj_face_slot(const DevTables &t, const double *__restrict__ V,
                                              const double *__restrict__ mu, const FluxConsts &fc,
                                              const int *__restrict__ nfslot, int q, double *__restrict__ FV,
                                              double *__restrict__ FN) {
  const int n = t.fnode[q], face = t.fidx[q];
  const int code = t.fcode[face];
  double Vn[5], m[5], nf[3];
  load_il<5>(Lay<SH>(), V, n, Vn);
  load_il<5>(Lay<SH>(), mu, n, m);
#pragma unroll
  for (int a = 0; a < 3; ++a) nf[a] = t.fnorm3[3 * (size_t)face + a];
#pragma unroll 1
  for (int dir = 0; dir < (WANTX ? 8 : 5); ++dir) {
    Dual nv[3], vv[5], fl[5];
#pragma unroll
    for (int a = 0; a < 3; ++a) nv[a] = Dual(nf[a], seed(dir, 5 + a));
#pragma unroll
    for (int k = 0; k < 5; ++k) vv[k] = Dual(Vn[k], seed(dir, k));
    face_flux(fc, code, nv, vv, fl);
    double s = 0.0;
#pragma unroll
    for (int k = 0; k < 5; ++k) s += m[k] * fl[k].d;
    if (dir < 5)
      FV[5 * (size_t)q + dir] = s;
    else
      FN[3 * (size_t)nfslot[q] + dir - 5] = s;
  }
}

// One edge (i, j) at position pos: e[0..5) = Vbar and e[5..10) = c of each end
// (Gbar[5a+k] = c_k dx[a]: the sums form the products), dxbar, and nbar to its
// place.
template <bool SECOND, bool WANTX, bool NT, int SH>
__device__ __forceinline__ void adj_edge(const DevTables &t, const double *__restrict__ V,
                                         const double *__restrict__ grad, const double *__restrict__ mu,
                                         const FluxConsts &fc, int i, int j, int pos, double *__restrict__ EXn,
                                         double ei[10], double ej[10], double dxb[3]) {
  double VL[5], VR[5], dV[5], g[5], di[5], dj[5];
  {
    double mj[5];
    load_il<5>(Lay<SH>(), mu, i, g);
    load_il<5>(Lay<SH>(), mu, j, mj);
#pragma unroll
    for (int k = 0; k < 5; ++k) g[k] -= mj[k];
  }
  load_il<5>(Lay<SH>(), V, i, VL);
  load_il<5>(Lay<SH>(), V, j, VR);
  if (SECOND) {
    double xi[3], dx[3], gi[15], gj[15];
    load_il<3>(Lay<SH>(), t.X3, i, xi);
    load_il<3>(Lay<SH>(), t.X3, j, dx);
#pragma unroll
    for (int a = 0; a < 3; ++a) dx[a] -= xi[a];
    load_il<15>(Lay<SH>(), grad, i, gi);
    load_il<15>(Lay<SH>(), grad, j, gj);
#pragma unroll
    for (int k = 0; k < 5; ++k) {
      di[k] = dx[0] * gi[k] + dx[1] * gi[5 + k] + dx[2] * gi[10 + k];
      dj[k] = dx[0] * gj[k] + dx[1] * gj[5 + k] + dx[2] * gj[10 + k];
      const double a = VL[k], b = VR[k];
      dV[k] = b - a;
      reconstruct(fc.beta, a, di[k], b, dj[k], VL[k], VR[k]);
    }
  }
  double nv[3], fb[13];
  stream_load<3, NT>(Lay<SH>(), t.pnormal, pos, nv);
#pragma unroll
  for (int d = 0; d < 13; ++d) fb[d] = 0.0;
  if (!(nv[0] * nv[0] + nv[1] * nv[1] + nv[2] * nv[2] < 1e-36))
    roeflux7_vjp(fc.gas, nv, VL, VR, g, fb, fb + 5, fb + 10);
  if (WANTX) stream_store<3, NT>(Lay<SH>(), EXn, pos, fb + 10);
  if (!SECOND) {
#pragma unroll
    for (int k = 0; k < 5; ++k) {
      ei[k] = fb[k];
      ej[k] = fb[5 + k];
    }
    return;
  }
  const double beta = fc.beta, beta2 = 1.0 - 2.0 * beta;
#pragma unroll
  for (int k = 0; k < 5; ++k) {
    const double d = beta2 * dV[k];
    double da_i, db_i, da_j, db_j;
    va_partials(d + 2.0 * beta * di[k], dV[k], da_i, db_i);
    va_partials(d + 2.0 * beta * dj[k], dV[k], da_j, db_j);
    const double Lb = fb[k], Rb = fb[5 + k];
    const double A = 0.5 * Lb * da_i, B = 0.5 * Lb * db_i;
    const double A2 = -0.5 * Rb * da_j, B2 = -0.5 * Rb * db_j;
    const double dVb = B + B2 + beta2 * (A + A2);
    ei[k] = Lb - dVb;
    ej[k] = Rb + dVb;
    ei[5 + k] = 2.0 * beta * A;
    ej[5 + k] = 2.0 * beta * A2;
  }
  if (WANTX) {
    const double *g2 = grad;
    asm volatile("" : "+s"(g2));
    double h[15];
#pragma unroll
    for (int a = 0; a < 3; ++a) dxb[a] = 0.0;
    load_il<15>(Lay<SH>(), g2, i, h);
#pragma unroll
    for (int a = 0; a < 3; ++a)
#pragma unroll
      for (int k = 0; k < 5; ++k) dxb[a] += ei[5 + k] * h[5 * a + k];
    load_il<15>(Lay<SH>(), g2, j, h);
#pragma unroll
    for (int a = 0; a < 3; ++a)
#pragma unroll
      for (int k = 0; k < 5; ++k) dxb[a] += ej[5 + k] * h[5 * a + k];
  }
}

// A boundary-face slot in the first nfb blocks, then ROWS: a wave per 64 nodes,
// lane r takes the upper edges of its node in turn and sums the node's own side
// in LDS (23 values a lane; registers are short: two waves per SIMD need all
// 256, and what the sums need of an edge is read again), so half of the records
// are neither written nor read again; otherwise a wave per (64 nodes, k-th upper
// edge).  Everything is read and written by
// position, so what is not gathered is contiguous.  The gradients are read again
// after the flux for dxbar rather than held across it.  ROWS 2: streams past the
// caches, which keep the gathered node data (815k nodes, 5.6M edges: 1013 -> 530
// us, 619 by entries, 568 by rows; the node pass 342 -> 241; 5 TB/s counted).
template <bool SECOND, bool WANTX, int ROWS, int SH>
__global__ __launch_bounds__(kAdjBlock) __attribute__((amdgpu_waves_per_eu(2, 2))) void k_adj_edges(
    DevTables t, int nfb, const double *__restrict__ V, const double *__restrict__ grad,
    const double *__restrict__ mu, FluxConsts fc, const int *__restrict__ nfslot, double *__restrict__ EVi,
    double *__restrict__ EVj, double *__restrict__ EXd, double *__restrict__ EXn, double *__restrict__ FV,
    double *__restrict__ FN, double *__restrict__ Vb, double *__restrict__ Gb, double *__restrict__ Xb) {
  constexpr int W = SECOND ? 10 : 5;
  if ((int)blockIdx.x < nfb) {
    const int q = blockIdx.x * kAdjBlock + threadIdx.x;
    if (q < 3 * t.F) adj_face_slot<WANTX, SH>(t, V, mu, fc, nfslot, q, FV, FN);
    return;
  }
  const int nw = ROWS ? t.ns : t.nup;
  const int nb = (nw + kAdjBlock / kWave - 1) / (kAdjBlock / kWave);
  const int w = xcd_chunk(blockIdx.x - nfb, nb) * (kAdjBlock / kWave) + (int)(threadIdx.x / kWave);
  if (w >= nw) return;
  double ei[10], ej[10], dxb[3];
  if (!ROWS) {
    const UpperEntry u = upper_entry<SH>(t, w);
    if (!u.act) return;
    adj_edge<SECOND, WANTX, false, SH>(t, V, grad, mu, fc, u.i, t.up.idx[u.pos], u.pos, EXn, ei, ej, dxb);
    store_il<W>(Lay<SH>(), EVi, u.pos, ei);
    store_il<W>(Lay<SH>(), EVj, u.pos, ej);
    if (SECOND && WANTX) store_il<3>(Lay<SH>(), EXd, u.pos, dxb);
    return;
  }
  const int sl = w, kb = t.up.kptr[sl], i = sl * kWave + lane_id();
  const int deg = i < t.N ? t.eup[i + 1] - t.eup[i] : 0;
  __shared__ double sums[kAdjBlock / kWave][23][kWave];
  double(*sum)[kWave] = sums[threadIdx.x / kWave];
  const int lane = lane_id(), ke = t.up.kptr[sl + 1];
#pragma unroll
  for (int q = 0; q < 23; ++q) sum[q][lane] = 0.0;
  for (int k = kb; k < ke; ++k) {
    const bool act = k - kb < deg;
    const int pos = t.up.koff[k] + lanes_below(act);
    if (!act) continue;
    int own = i;
    asm volatile("" : "+v"(own));  // the own side is read anew for each edge
    const int j = t.up.idx[pos];
    adj_edge<SECOND, WANTX, ROWS == 2, SH>(t, V, grad, mu, fc, own, j, pos, EXn, ei, ej, dxb);
    stream_store<W, ROWS == 2>(Lay<SH>(), EVj, pos, ej);
#pragma unroll
    for (int q = 0; q < 5; ++q) sum[q][lane] += ei[q];
    const double *X = t.X3;
    asm volatile("" : "+s"(X));
    double x[3], dx[3];
    load_il<3>(Lay<SH>(), X, own, x);
    load_il<3>(Lay<SH>(), X, j, dx);
#pragma unroll
    for (int a = 0; a < 3; ++a) dx[a] -= x[a];
#pragma unroll
    for (int a = 0; a < 3; ++a)
#pragma unroll
      for (int q = 0; q < 5; ++q) sum[5 + 5 * a + q][lane] += ei[5 + q] * dx[a];
    if (WANTX) {
      stream_store<3, ROWS == 2>(Lay<SH>(), EXd, pos, dxb);
#pragma unroll
      for (int a = 0; a < 3; ++a) sum[20 + a][lane] -= dxb[a];
    }
  }
  if (i >= t.N) return;
  double o[15];
#pragma unroll
  for (int q = 0; q < 5; ++q) o[q] = sum[q][lane];
  store_il<5>(Lay<SH>(), Vb, i, o);
#pragma unroll
  for (int q = 0; q < 15; ++q) o[q] = sum[5 + q][lane];
  store_il<15>(Lay<SH>(), Gb, i, o);
  if (WANTX) {
#pragma unroll
    for (int a = 0; a < 3; ++a) o[a] = sum[20 + a][lane];
    store_il<3>(Lay<SH>(), Xb, i, o);
  }
}

// ---------------------------------------------------------------------------
// 3. per node: edge slots in edge order, then faces
// ---------------------------------------------------------------------------
// one edge slot: Vbar, and Gbar += c dx^T with dx = X_j - X_i of the edge (i, j)
template <bool SECOND>
__device__ __forceinline__ void add_slot(const double *ev, const double dx[3], double vb[5], double gb[15]) {
#pragma unroll
  for (int k = 0; k < 5; ++k) vb[k] += ev[k];
  if (SECOND) {
#pragma unroll
    for (int a = 0; a < 3; ++a)
#pragma unroll
      for (int k = 0; k < 5; ++k) gb[5 * a + k] += ev[5 + k] * dx[a];
  }
}

// A wave per 64 nodes: the slots of the upper edges are contiguous (ROWS: the
// edge pass left their sums in Vb, H and Xb), those of the lower ones are
// gathered, and both ends' coordinates follow from the adjacency
// rows, whose first entries are the lower neighbours.  Bound by the slots' bytes
// (624 -> 241 us at 815k nodes, 342 with both ends' slots).
template <bool SECOND, bool WANTX, bool ROWS, int SH>
__global__ __launch_bounds__(kAdjBlock) void k_adj_nodes(DevTables t, const double *__restrict__ grad,
                                                         const double *__restrict__ EVi,
                                                         const double *__restrict__ EVj,
                                                         const double *__restrict__ EXd,
                                                         const double *__restrict__ FV, double *__restrict__ Vb,
                                                         double *__restrict__ H, double *__restrict__ S,
                                                         double *__restrict__ Xb) {
  constexpr int W = SECOND ? 10 : 5;
  const int sl = wave_slice(t);
  if (sl >= t.ns) return;
  const int n = sl * kWave + lane_id();
  const bool live = n < t.N;
  double vb[5] = {0.0, 0.0, 0.0, 0.0, 0.0}, gb[15], xb[3] = {0.0, 0.0, 0.0}, xn[3] = {0.0, 0.0, 0.0};
#pragma unroll
  for (int q = 0; q < 15; ++q) gb[q] = 0.0;
  if (SECOND) load_il<3>(Lay<SH>(), t.X3, min(n, t.N - 1), xn);
  if (ROWS && live) {
    load_il<5>(Lay<SH>(), Vb, n, vb);
    load_il<15>(Lay<SH>(), H, n, gb);
    if (WANTX) load_il<3>(Lay<SH>(), Xb, n, xb);
  }
  // edges (m, n), m < n: the j-side slots
  {
    const int deg = live ? t.lrow[n + 1] - t.lrow[n] : 0, all = live ? t.rowptr[n + 1] - t.rowptr[n] : 0;
    const int kb = t.lo.kptr[sl], ke = t.lo.kptr[sl + 1], ab = t.nb.kptr[sl];
    for (int k = 0; k < ke - kb; ++k) {
      const bool act = k < deg;
      const int q = t.lo.koff[kb + k] + lanes_below(act), e = t.nb.koff[ab + k] + lanes_below(k < all);
      if (!act) continue;
      const int pos = t.lo.idx[q];
      double ev[W], dx[3] = {0.0, 0.0, 0.0}, d[3];
      load_il<W>(Lay<SH>(), EVj, pos, ev);
      if (SECOND) {
        load_il<3>(Lay<SH>(), t.X3, t.nb.idx[e], dx);
#pragma unroll
        for (int a = 0; a < 3; ++a) dx[a] = xn[a] - dx[a];
      }
      if (SECOND && WANTX) {
        load_il<3>(Lay<SH>(), EXd, pos, d);
#pragma unroll
        for (int a = 0; a < 3; ++a) xb[a] += d[a];
      }
      add_slot<SECOND>(ev, dx, vb, gb);
    }
  }
  // edges (n, m), n < m: the i-side slots
  if (!ROWS) {
    const int deg = live ? t.eup[n + 1] - t.eup[n] : 0;
    const int kb = t.up.kptr[sl], ke = t.up.kptr[sl + 1];
    for (int k = 0; k < ke - kb; ++k) {
      const bool act = k < deg;
      const int pos = t.up.koff[kb + k] + lanes_below(act);
      if (!act) continue;
      double ev[W], dx[3] = {0.0, 0.0, 0.0}, d[3];
      load_il<W>(Lay<SH>(), EVi, pos, ev);
      if (SECOND) {
        load_il<3>(Lay<SH>(), t.X3, t.up.idx[pos], dx);
#pragma unroll
        for (int a = 0; a < 3; ++a) dx[a] -= xn[a];
      }
      if (SECOND && WANTX) {
        load_il<3>(Lay<SH>(), EXd, pos, d);
#pragma unroll
        for (int a = 0; a < 3; ++a) xb[a] -= d[a];
      }
      add_slot<SECOND>(ev, dx, vb, gb);
    }
  }
  if (!live) return;
  for (int q = t.frow[n]; q < t.frow[n + 1]; ++q)
#pragma unroll
    for (int k = 0; k < 5; ++k) vb[k] += FV[5 * (size_t)q + k];
  store_il<5>(Lay<SH>(), Vb, n, vb);
  if (WANTX) store_il<3>(Lay<SH>(), Xb, n, xb);
  if (!SECOND) return;
  double L[6];
#pragma unroll
  for (int q = 0; q < 6; ++q) L[q] = t.lsq6[6 * (size_t)n + q];
#pragma unroll
  for (int k = 0; k < 5; ++k) {
    double w[3];
    lsq_weights(L, gb[k], gb[5 + k], gb[10 + k], w);
#pragma unroll
    for (int a = 0; a < 3; ++a) gb[5 * a + k] = w[a];
  }
  store_il<15>(Lay<SH>(), H, n, gb);
  if (WANTX) {
    double gn[15], s[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
    load_il<15>(Lay<SH>(), grad, n, gn);
    int e = 0;
#pragma unroll
    for (int a = 0; a < 3; ++a)
#pragma unroll
      for (int b = a; b < 3; ++b, ++e)
#pragma unroll
        for (int k = 0; k < 5; ++k) s[e] -= gb[5 * a + k] * gn[5 * b + k] + gb[5 * b + k] * gn[5 * a + k];
    store_il<6>(Lay<SH>(), S, n, s);
  }
}

// ---------------------------------------------------------------------------
// 4. per node: reverse of the LSQ gradients, then U
// ---------------------------------------------------------------------------
// Bound by the gathers of H, S, V and X (29 values an entry, where the weights of
// both ends were formed per entry from their factors; 376 -> 229 us at 815k nodes).
template <bool SECOND, bool WANTX, int SH>
__global__ __launch_bounds__(kAdjBlock) void k_adj_lsq(DevTables t, const double *__restrict__ V,
                                                       const double *__restrict__ U, Gas gas,
                                                       const double *__restrict__ Vb, const double *__restrict__ H,
                                                       const double *__restrict__ S, double *__restrict__ Ub,
                                                       double *__restrict__ Xb) {
  const int sl = wave_slice(t);
  if (sl >= t.ns) return;
  const int n = sl * kWave + lane_id();
  const bool live = n < t.N;
  const int nn = min(n, t.N - 1);
  double vb[5], Vn[5], xb[3] = {0.0, 0.0, 0.0};
  load_il<5>(Lay<SH>(), Vb, nn, vb);
  load_il<5>(Lay<SH>(), V, nn, Vn);
  if (SECOND) {
    // sum over j of dx and of V_j - V_i: what the node's own H and S multiply
    double xn[3], sx[3] = {0.0, 0.0, 0.0}, sv[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
    load_il<3>(Lay<SH>(), t.X3, nn, xn);
    const int deg = live ? t.rowptr[n + 1] - t.rowptr[n] : 0;
    const int kb = t.nb.kptr[sl], ke = t.nb.kptr[sl + 1];
    auto add = [&](const double h[15], const double s[6], const double dx[3], const double dV[5]) {
#pragma unroll
      for (int k = 0; k < 5; ++k) vb[k] -= h[k] * dx[0] + h[5 + k] * dx[1] + h[10 + k] * dx[2];
      if (WANTX) {
#pragma unroll
        for (int a = 0; a < 3; ++a)
#pragma unroll
          for (int k = 0; k < 5; ++k) xb[a] -= h[5 * a + k] * dV[k];
        xb[0] -= s[0] * dx[0] + s[1] * dx[1] + s[2] * dx[2];
        xb[1] -= s[1] * dx[0] + s[3] * dx[1] + s[4] * dx[2];
        xb[2] -= s[2] * dx[0] + s[4] * dx[1] + s[5] * dx[2];
      }
    };
    for (int k = 0; k < ke - kb; ++k) {
      const bool act = k < deg;
      const int pos = t.nb.koff[kb + k] + lanes_below(act);
      if (!act) continue;
      const int m = t.nb.idx[pos];
      double h[15], s[6], dx[3], dV[5];
      load_il<3>(Lay<SH>(), t.X3, m, dx);
      load_il<15>(Lay<SH>(), H, m, h);
      if (WANTX) {
        load_il<5>(Lay<SH>(), V, m, dV);
        load_il<6>(Lay<SH>(), S, m, s);
#pragma unroll
        for (int q = 0; q < 5; ++q) {
          dV[q] -= Vn[q];
          sv[q] += dV[q];
        }
      }
#pragma unroll
      for (int a = 0; a < 3; ++a) {
        dx[a] -= xn[a];
        sx[a] += dx[a];
      }
      add(h, s, dx, dV);
    }
    double h[15], s[6];
    load_il<15>(Lay<SH>(), H, nn, h);
    if (WANTX) load_il<6>(Lay<SH>(), S, nn, s);
    add(h, s, sx, sv);
  }
  if (!live) return;
  if (WANTX) {
    double x[3];
    load_il<3>(Lay<SH>(), Xb, n, x);
#pragma unroll
    for (int a = 0; a < 3; ++a) x[a] += xb[a];
    store_il<3>(Lay<SH>(), Xb, n, x);
  }
  if (Ub) {
    // V = (rho, u / rho, (gam - 1) (E - rho |u|^2 / 2) - gam pstiff)
    const double ir = 1.0 / U[5 * (size_t)n], gp = gas.gam1 * vb[4];
    double q = 0.0, r = 0.0, ub[5];
#pragma unroll
    for (int k = 1; k < 4; ++k) {
      ub[k] = vb[k] * ir - gp * Vn[k];
      q += Vn[k] * Vn[k];
      r += Vn[k] * vb[k];
    }
    ub[0] = vb[0] - r * ir + 0.5 * gp * q;
    ub[4] = gp;
#pragma unroll
    for (int k = 0; k < 5; ++k) Ub[5 * (size_t)n + k] = ub[k];
  }
}

// ---------------------------------------------------------------------------
// 5. geometry: per tet (control volumes, dual normals), per boundary face
// ---------------------------------------------------------------------------
__device__ __forceinline__ void load_x4(const double *__restrict__ X4, int n, double x[3]) {
  const double4 p = *reinterpret_cast<const double4 *>(X4 + 4 * (size_t)n);
  x[0] = p.x;
  x[1] = p.y;
  x[2] = p.z;
}
// z += s (x x y)
__device__ __forceinline__ void add_cross(double s, const double x[3], const double y[3], double z[3]) {
  z[0] += s * (x[1] * y[2] - x[2] * y[1]);
  z[1] += s * (x[2] * y[0] - x[0] * y[2]);
  z[2] += s * (x[0] * y[1] - x[1] * y[0]);
}

// The tet's share of each quantity is a product of coordinate differences, so
// its reverse is a few cross products: with p = c - d, r = (a - c) + (b - d) and
// w the weight of an edge, d(w . p x r) = dp . r x w + dr . w x p.  Bound by the
// gathers of six nbar (659 -> 215 us for 4.7M tets; 12 passes in dual numbers
// before, and 282 us with each lane storing its own 96 bytes: the vector cache
// takes a store of 64 scattered pieces one piece at a time, so they go out
// through LDS as whole lines).
template <int SH>
__global__ __launch_bounds__(kAdjBlock) void k_adj_tets(int T, const int4 *__restrict__ tets,
                                                        const int *__restrict__ tpos,
                                                        const double *__restrict__ X4,
                                                        const double *__restrict__ cvb,
                                                        const double *__restrict__ EXn, double *__restrict__ TX) {
#pragma clang fp contract(on)
  const int nblk = (T + kAdjBlock - 1) / kAdjBlock;
  __shared__ double2 out[6 * kAdjBlock];
  const int t0 = xcd_chunk(blockIdx.x, nblk) * kAdjBlock, t1 = t0 + (int)threadIdx.x;
  const int t = min(t1, T - 1);  // the lanes past the last tet repeat it and store nothing
  const int4 d4 = tets[t];
  const int nd[4] = {d4.x, d4.y, d4.z, d4.w};
  int ps[6];
#pragma unroll
  for (int e = 0; e < 6; e += 2) {
    const int2 q = *reinterpret_cast<const int2 *>(tpos + 6 * (size_t)t + e);
    ps[e] = q.x;
    ps[e + 1] = q.y;
  }
  double x[4][3], z[4][3], cv = 0.0;
#pragma unroll
  for (int v = 0; v < 4; ++v) {
    load_x4(X4, nd[v], x[v]);
    cv += cvb[nd[v]];
#pragma unroll
    for (int a = 0; a < 3; ++a) z[v][a] = 0.0;
  }
  // ElemTet::computeVolume (ElemTetCore.C:31-44): v3 . (v1 x v2) / 6, a quarter
  // of it to each vertex
  {
    double e[3][3];
#pragma unroll
    for (int v = 0; v < 3; ++v)
#pragma unroll
      for (int a = 0; a < 3; ++a) e[v][a] = x[v + 1][a] - x[0][a];
    const double s = cv * (1.0 / 24.0);
    add_cross(s, e[1], e[2], z[1]);
    add_cross(s, e[2], e[0], z[2]);
    add_cross(s, e[0], e[1], z[3]);
#pragma unroll
    for (int a = 0; a < 3; ++a) z[0][a] -= z[1][a] + z[2][a] + z[3][a];
  }
  // dual-face normals (ElemTetCore.C:281-330)
#pragma unroll
  for (int e = 0; e < 6; ++e) {
    const int a = kEnd[e][0], b = kEnd[e][1], c = kOpp[e][0], d = kOpp[e][1];
    double w[3], p[3], r[3], gp[3] = {0.0, 0.0, 0.0}, gr[3] = {0.0, 0.0, 0.0};
    load_il<3>(Lay<SH>(), EXn, ps[e], w);
    const double s = nd[a] < nd[b] ? 1.0 / 24.0 : -1.0 / 24.0;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      p[k] = x[c][k] - x[d][k];
      r[k] = (x[a][k] - x[c][k]) + (x[b][k] - x[d][k]);
    }
    add_cross(s, r, w, gp);
    add_cross(s, w, p, gr);
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      z[a][k] += gr[k];
      z[b][k] += gr[k];
      z[c][k] += gp[k] - gr[k];
      z[d][k] -= gp[k] + gr[k];
    }
  }
  double2 *o = out + 6 * threadIdx.x;
#pragma unroll
  for (int v = 0; v < 4; v += 2) {
    o[3 * v / 2] = make_double2(z[v][0], z[v][1]);
    o[3 * v / 2 + 1] = make_double2(z[v][2], z[v + 1][0]);
    o[3 * v / 2 + 2] = make_double2(z[v + 1][1], z[v + 1][2]);
  }
  __syncthreads();
  double2 *g = reinterpret_cast<double2 *>(TX) + 6 * (size_t)t0;
  const int n = 6 * min(kAdjBlock, T - t0);
#pragma unroll
  for (int r = 0; r < 6; ++r) {
    const int q = (int)threadIdx.x + r * kAdjBlock;
    if (q < n) g[q] = out[q];
  }
}

__global__ __launch_bounds__(kAdjBlock) void k_adj_faces(int F, const int *__restrict__ faces,
                                                         const double *__restrict__ X4,
                                                         const double *__restrict__ FN, double *__restrict__ FX) {
  const int f = blockIdx.x * kAdjBlock + threadIdx.x;
  if (f >= F) return;
  double x[3][3], nb[3] = {0.0, 0.0, 0.0};
#pragma unroll
  for (int v = 0; v < 3; ++v) {
    load_x4(X4, faces[3 * (size_t)f + v], x[v]);
#pragma unroll
    for (int a = 0; a < 3; ++a) nb[a] += FN[9 * (size_t)f + 3 * v + a];
  }
  // a third of FaceTria::computeNormal (FaceTriaCore.C:31-37, 288-292):
  // (x2 - x0) x (x1 - x0) / 6
  double p[3], q[3], gp[3] = {0.0, 0.0, 0.0}, gq[3] = {0.0, 0.0, 0.0};
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    p[a] = x[2][a] - x[0][a];
    q[a] = x[1][a] - x[0][a];
  }
  add_cross(1.0 / 6.0, q, nb, gp);
  add_cross(1.0 / 6.0, nb, p, gq);
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    FX[9 * (size_t)f + a] = -(gp[a] + gq[a]);
    FX[9 * (size_t)f + 3 + a] = gq[a];
    FX[9 * (size_t)f + 6 + a] = gp[a];
  }
}

// ---------------------------------------------------------------------------
// 6. per node: Xbar
// ---------------------------------------------------------------------------
// Four lanes per node, each every fourth slot: the slot lists are read in whole
// lines and four gathers per node are in flight (688 -> 215 us at 815k nodes, with
// the neighbours' S moved to the pass that reads them anyway).
__global__ __launch_bounds__(kAdjBlock) void k_adj_xgather(DevTables t, const double *__restrict__ Xb,
                                                           const int *__restrict__ ntrow,
                                                           const int *__restrict__ ntslot,
                                                           const double *__restrict__ TX,
                                                           const int *__restrict__ nfslot,
                                                           const double *__restrict__ FX,
                                                           double *__restrict__ out) {
  const int nb = (t.N + kAdjBlock / 4 - 1) / (kAdjBlock / 4);
  const int n = xcd_chunk(blockIdx.x, nb) * (kAdjBlock / 4) + (int)(threadIdx.x >> 2), r = threadIdx.x & 3;
  double xb[3] = {0.0, 0.0, 0.0};
  if (n < t.N) {
    const int q1 = ntrow[n + 1];
#pragma unroll 4
    for (int q = ntrow[n] + r; q < q1; q += 4) {
      const double *s = TX + 3 * (size_t)ntslot[q];  // 4 t + v
      const double2u p = *reinterpret_cast<const double2u *>(s);
      xb[0] += p.x;
      xb[1] += p.y;
      xb[2] += s[2];
    }
    for (int q = t.frow[n] + r; q < t.frow[n + 1]; q += 4) {
      const double *s = FX + 3 * (size_t)nfslot[q];  // 3 f + v
#pragma unroll
      for (int a = 0; a < 3; ++a) xb[a] += s[a];
    }
  }
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    xb[a] += __shfl_xor(xb[a], 1);
    xb[a] += __shfl_xor(xb[a], 2);
  }
  if (n < t.N && r < 3) out[3 * (size_t)n + r] = Xb[il<3>(t.sh, n, r)] + (r == 0 ? xb[0] : (r == 1 ? xb[1] : xb[2]));
}

// edge id -> position, and the tets' edge ids to positions
__global__ __launch_bounds__(kAdjBlock) void k_adj_epos(int E, const int *__restrict__ pedge, int *__restrict__ epos) {
  const int p = blockIdx.x * kAdjBlock + threadIdx.x;
  if (p < E) epos[pedge[p]] = p;
}
__global__ __launch_bounds__(kAdjBlock) void k_adj_tpos(long long n, const int *__restrict__ epos,
                                                        int *__restrict__ tpos) {
  const long long k = (long long)blockIdx.x * kAdjBlock + threadIdx.x;
  if (k < n) tpos[k] = epos[tpos[k]];
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
void free_adjoint(aerofx_ctx *c) {
  if (c->adj && c->adj->h_J) (void)hipHostFree(c->adj->h_J);
  delete c->adj;  // device memory is owned by the context allocation list
  c->adj = nullptr;
}

namespace {

inline dim3 grid_for(long long n) { return dim3((unsigned)((n + kAdjBlock - 1) / kAdjBlock)); }

template <class T>
int alloc_n(aerofx_ctx *c, size_t n, T **out) {
  void *p = nullptr;
  int rc = ctx_alloc(c, n * sizeof(T), &p);
  *out = static_cast<T *>(p);
  return rc;
}

template <class T>
int upload_vec(aerofx_ctx *c, const std::vector<T> &v, T **out) {
  int rc = alloc_n(c, v.size() ? v.size() : 1, out);
  if (rc) return rc;
  if (v.empty()) return 0;
  hipError_t e = hipMemcpy(*out, v.data(), v.size() * sizeof(T), hipMemcpyHostToDevice);
  return e == hipSuccess ? 0 : set_hip_error(e, "adjoint table upload");
}

int ensure_adjoint(aerofx_ctx *c) {
  if (c->adj) return 0;
  const int N = c->N, E = c->E, T = c->T, F = c->F;
  int rc = ensure_elem_tables(c);
  if (rc) return rc;
  Adjoint *a = new Adjoint();
  const ElemTables &el = *c->elem;
  a->tets = el.tets;
  a->faces = el.faces;
  a->ntrow = el.ntrow;
  a->ntslot = el.ntslot;
  a->nfslot = el.nfslot;
  const size_t F1 = std::max(F, 1);
  if ((rc = alloc_n(c, il_count<10>(c->tab.sh, E), &a->EVi)) || (rc = alloc_n(c, il_count<10>(c->tab.sh, E), &a->EVj)) ||
      (rc = alloc_n(c, il_count<3>(c->tab.sh, E), &a->EXd)) || (rc = alloc_n(c, il_count<3>(c->tab.sh, E), &a->EXn)) ||
      (rc = alloc_n(c, 15 * F1, &a->FV)) || (rc = alloc_n(c, 9 * F1, &a->FN)) ||
      (rc = alloc_n(c, il_count<5>(c->tab.sh, N), &a->mu)) || (rc = alloc_n(c, (size_t)N, &a->cvb)) ||
      (rc = alloc_n(c, il_count<5>(c->tab.sh, N), &a->Vb)) || (rc = alloc_n(c, il_count<15>(c->tab.sh, N), &a->H)) ||
      (rc = alloc_n(c, il_count<3>(c->tab.sh, N), &a->Xb)) || (rc = alloc_n(c, il_count<6>(c->tab.sh, N), &a->S)) ||
      (rc = alloc_n(c, 5 * (size_t)N, &a->R)) || (rc = alloc_n(c, 12 * (size_t)std::max(T, 1), &a->TX)) ||
      (rc = alloc_n(c, 9 * F1, &a->FX)) || (rc = alloc_n(c, (size_t)F + 1, &a->Jf)) ||
      (rc = upload_vec(c, c->tet_edges, &a->tpos))) {
    delete a;
    return rc;
  }
  if (T > 0) {
    // the positions of the tets' edges (dxbar's buffer holds the map meanwhile)
    int *epos = reinterpret_cast<int *>(a->EXd);
    hipLaunchKernelGGL(k_adj_epos, grid_for(E), dim3(kAdjBlock), 0, c->stream, E, c->tab.pedge, epos);
    hipLaunchKernelGGL(k_adj_tpos, grid_for(6LL * T), dim3(kAdjBlock), 0, c->stream, 6LL * T, epos, a->tpos);
  }
  hipError_t e = hipHostMalloc((void **)&a->h_J, sizeof(double), hipHostMallocDefault);
  if (e != hipSuccess) {
    delete a;
    return set_hip_error(e, "adjoint set-up");
  }
  c->adj = a;
  return 0;
}

}  // namespace

int ensure_elem_tables(aerofx_ctx *c) {
  if (c->elem) return 0;
  const int N = c->N, E = c->E, T = c->T, F = c->F;
  if ((int)c->tets.size() != 4 * T || (int)c->tet_edges.size() != 6 * T || (int)c->faces.size() != 3 * F)
    return set_error(AEROFX_ERR_STATE, "element tables missing from the context");
  // node -> (tet, vertex) slots in tet order; node -> (face, vertex) in the
  // order of tab.fidx; edge -> (tet, local edge) slots in tet order
  std::vector<int> ntrow(N + 1, 0), ntslot(4 * (size_t)T), nfslot(3 * (size_t)F);
  std::vector<int> etrow(E + 1, 0), etslot(6 * (size_t)T);
  for (size_t k = 0; k < 4 * (size_t)T; ++k) ntrow[c->tets[k] + 1]++;
  for (int n = 0; n < N; ++n) ntrow[n + 1] += ntrow[n];
  {
    std::vector<int> fill(ntrow.begin(), ntrow.end() - 1);
    for (size_t k = 0; k < 4 * (size_t)T; ++k) ntslot[fill[c->tets[k]]++] = (int)k;
  }
  {
    std::vector<int> frow(N + 1, 0);
    for (size_t k = 0; k < 3 * (size_t)F; ++k) frow[c->faces[k] + 1]++;
    for (int n = 0; n < N; ++n) frow[n + 1] += frow[n];
    std::vector<int> fill(frow.begin(), frow.end() - 1);
    for (size_t k = 0; k < 3 * (size_t)F; ++k) nfslot[fill[c->faces[k]]++] = (int)k;
  }
  for (size_t k = 0; k < 6 * (size_t)T; ++k) etrow[c->tet_edges[k] + 1]++;
  for (int l = 0; l < E; ++l) etrow[l + 1] += etrow[l];
  {
    std::vector<int> fill(etrow.begin(), etrow.end() - 1);
    for (size_t k = 0; k < 6 * (size_t)T; ++k) etslot[fill[c->tet_edges[k]]++] = (int)k;
  }
  ElemTables *el = new ElemTables();
  int rc;
  if ((rc = upload_vec(c, c->tets, &el->tets)) || (rc = upload_vec(c, c->faces, &el->faces)) || (rc = upload_vec(c, ntrow, &el->ntrow)) ||
      (rc = upload_vec(c, ntslot, &el->ntslot)) || (rc = upload_vec(c, nfslot, &el->nfslot)) ||
      (rc = upload_vec(c, etrow, &el->etrow)) || (rc = upload_vec(c, etslot, &el->etslot))) {
    delete el;
    return rc;
  }
  c->elem = el;
  return 0;
}

// From this many 64-node slices the edge pass takes whole rows, and from the
// second its streams bypass the caches.  (dR/dU)^T / both products in us, by
// entries, by rows, by rows past the caches: at 562 slices 122 / 157, 121 / 169,
// -; 1839: 213 / 364, 194 / 348, 210 / 348; 4292: 502 / 867, 465 / 814, 452 / 791;
// 14261: 1494 / 2683, 1340 / 2510, 1304 / 2426.  Below, there are too few waves
// for the 1024 SIMDs, and then the edge data still fit the caches.
constexpr int kAdjRowSlices = 1536, kAdjStreamSlices = 3072;

template <bool SECOND, bool WANTX, int ROWS, int SH>
static int adjoint_stages(aerofx_ctx *c, const double *U, const double *lam, double *Ub, double *Xout) {
  Adjoint *a = c->adj;
  const DevTables &t = c->tab;
  const dim3 b(kAdjBlock);
  // 1.
  hipLaunchKernelGGL(k_adj_mu, grid_for(t.N), b, 0, c->stream, t, lam, a->R, a->mu, a->cvb);
  // 2.
  const int nfb = (3 * t.F + kAdjBlock - 1) / kAdjBlock;
  const int nb = ((ROWS ? t.ns : t.nup) + kAdjBlock / kWave - 1) / (kAdjBlock / kWave);
  if (nfb + nb)
    hipLaunchKernelGGL((k_adj_edges<SECOND, WANTX, ROWS, SH>), dim3((unsigned)(nfb + nb)), b, 0, c->stream, t, nfb, c->d_V,
                       c->d_grad, a->mu, c->fc, a->nfslot, a->EVi, a->EVj, a->EXd, a->EXn, a->FV, a->FN,
                       a->Vb, a->H, a->Xb);
  // 3.
  hipLaunchKernelGGL((k_adj_nodes<SECOND, WANTX, ROWS != 0, SH>), slice_grid(t.ns), b, 0, c->stream, t, c->d_grad, a->EVi, a->EVj,
                     a->EXd, a->FV, a->Vb, a->H, a->S, a->Xb);
  // 4.
  hipLaunchKernelGGL((k_adj_lsq<SECOND, WANTX, SH>), slice_grid(t.ns), b, 0, c->stream, t, c->d_V, U, c->gas, a->Vb, a->H,
                     a->S, Ub, a->Xb);
  int rc;
  // the Navier-Stokes Galerkin term (its element derivative, transposed)
  if (c->viscous && Ub && (rc = launch_visc_adjoint(c, lam, Ub))) return rc;
  if (WANTX) {
    // 5.
    if (c->T > 0)
      hipLaunchKernelGGL(k_adj_tets<SH>, grid_for(c->T), b, 0, c->stream, c->T, (const int4 *)a->tets, a->tpos, t.X4,
                         a->cvb, a->EXn, a->TX);
    // the Navier-Stokes Galerkin term's coordinate derivative, per element
    if (c->T > 0 && (rc = launch_visc_adjoint_x(c, lam, a->TX))) return rc;
    if (c->F > 0)
      hipLaunchKernelGGL(k_adj_faces, grid_for(c->F), b, 0, c->stream, c->F, a->faces, t.X4, a->FN, a->FX);
    // 6.
    hipLaunchKernelGGL(k_adj_xgather, grid_for(4LL * t.N), b, 0, c->stream, t, a->Xb, a->ntrow, a->ntslot, a->TX,
                       a->nfslot, a->FX, Xout);
  }
  hipError_t e = hipGetLastError();
  return e == hipSuccess ? 0 : set_hip_error(e, "adjoint launch");
}

int launch_adjoint(aerofx_ctx *c, const double *U, const double *lam, double *Ub, double *Xout) {
  int rc = ensure_adjoint(c);
  // forward pass: V, gradients (recomputed), R
  if (rc || (rc = launch_residual(c, U, c->adj->R, true))) return rc;
  const DevTables &t = c->tab;
  const bool second = c->p.second_order != 0, rows = second && t.sh && row_waves(t.ns, kAdjRowSlices, c->max_degree);
  auto stages = [&](auto wantx) {
    constexpr bool X = decltype(wantx)::value;
    const auto f = rows && t.ns >= kAdjStreamSlices ? adjoint_stages<true, X, 2, kGroupShift>
                   : rows                           ? adjoint_stages<true, X, 1, kGroupShift>
                   : second && t.sh                 ? adjoint_stages<true, X, 0, kGroupShift>
                   : second                         ? adjoint_stages<true, X, 0, 0>
                   : t.sh                           ? adjoint_stages<false, X, 0, kGroupShift>
                                                    : adjoint_stages<false, X, 0, 0>;
    return f(c, U, lam, Ub, Xout);
  };
  return Xout ? stages(std::true_type()) : stages(std::false_type());
}

// ---------------------------------------------------------------------------
// force objective on slip-wall faces: J = sum_f sum_{v in f} p_v (n_f / 3) . d
// (the wall flux carries p n, FluxFcnDescSG.C:779-789, so this is the
// pressure force on the wall projected on d)
// ---------------------------------------------------------------------------
// per face: J_f, and the coordinate derivative of J_f (9 slots)
__global__ __launch_bounds__(kAdjBlock) void k_lift_faces(int F, int sh, const int *__restrict__ faces,
                                                          const int *__restrict__ fcode,
                                                          const double *__restrict__ fnorm3,
                                                          const double *__restrict__ X4,
                                                          const double *__restrict__ V, double d0, double d1,
                                                          double d2, double *__restrict__ Jf,
                                                          double *__restrict__ FX) {
  const int f = blockIdx.x * kAdjBlock + threadIdx.x;
  if (f >= F) return;
  const int code = fcode[f];
  const bool wall = is_wall_code(code);
  int nd[3];
  double psum = 0.0;
#pragma unroll
  for (int v = 0; v < 3; ++v) {
    nd[v] = faces[3 * (size_t)f + v];
    psum += V[il<5>(sh, nd[v], 4)];
  }
  if (!wall) psum = 0.0;
  const double *nv = fnorm3 + 3 * (size_t)f;
  Jf[f] = psum * (nv[0] * d0 + nv[1] * d1 + nv[2] * d2);
  if (!FX) return;
  // d J_f / d x: J_f = psum (1/3) (0.5 (x2 - x0) x (x1 - x0)) . d
  double x[3][3];
#pragma unroll
  for (int v = 0; v < 3; ++v) {
    const double4 xv = *reinterpret_cast<const double4 *>(X4 + 4 * (size_t)nd[v]);
    x[v][0] = xv.x;
    x[v][1] = xv.y;
    x[v][2] = xv.z;
  }
  const double third = 1.0 / 3.0;
#pragma unroll 1
  for (int dir = 0; dir < 9; ++dir) {
    Dual p[3], q[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      p[a] = Dual(x[2][a], seed(dir, 6 + a)) - Dual(x[0][a], seed(dir, a));
      q[a] = Dual(x[1][a], seed(dir, 3 + a)) - Dual(x[0][a], seed(dir, a));
    }
    Dual c0 = p[1] * q[2] - p[2] * q[1];
    Dual c1 = p[2] * q[0] - p[0] * q[2];
    Dual c2 = p[0] * q[1] - p[1] * q[0];
    FX[9 * (size_t)f + dir] = psum * third * 0.5 * (c0.d * d0 + c1.d * d1 + c2.d * d2);
  }
}

// per node: dJ/dU (through p(U)) and dJ/dX (face slots)
__global__ __launch_bounds__(kAdjBlock) void k_lift_nodes(DevTables t, const double *__restrict__ U, Gas gas,
                                                          const int *__restrict__ nfslot,
                                                          const double *__restrict__ FX, double d0, double d1,
                                                          double d2, double *__restrict__ dJdU,
                                                          double *__restrict__ dJdX) {
  const int n = blockIdx.x * kAdjBlock + threadIdx.x;
  if (n >= t.N) return;
  double w = 0.0, xb[3] = {0.0, 0.0, 0.0};
  for (int q = t.frow[n]; q < t.frow[n + 1]; ++q) {
    const int f = t.fidx[q];
    const int code = t.fcode[f];
    if (!is_wall_code(code)) continue;
    const double *nv = t.fnorm3 + 3 * (size_t)f;
    w += nv[0] * d0 + nv[1] * d1 + nv[2] * d2;
    if (dJdX) {
      const size_t sl = nfslot[q];
      const size_t ff = sl / 3, v = sl - 3 * ff;
#pragma unroll
      for (int a = 0; a < 3; ++a) xb[a] += FX[9 * ff + 3 * v + a];
    }
  }
  if (dJdU) {
    double u[5];
#pragma unroll
    for (int k = 0; k < 5; ++k) u[k] = U[5 * (size_t)n + k];
#pragma unroll 1
    for (int dir = 0; dir < 5; ++dir) {
      Dual ud[5], vd[5];
#pragma unroll
      for (int k = 0; k < 5; ++k) ud[k] = Dual(u[k], seed(dir, k));
      prim_from_cons(ud, gas, vd);
      dJdU[5 * (size_t)n + dir] = w * vd[4].d;
    }
  }
  if (dJdX)
#pragma unroll
    for (int a = 0; a < 3; ++a) dJdX[3 * (size_t)n + a] = xb[a];
}

// J = sum of the per-face values in face order (one block)
__global__ void k_sum_ordered(int F, const double *__restrict__ Jf, double *__restrict__ out) {
  __shared__ double sh[256];
  const int per = (F + 255) / 256;
  const int b0 = threadIdx.x * per, b1 = min(F, b0 + per);
  double s = 0.0;
  for (int f = b0; f < b1; ++f) s += Jf[f];
  sh[threadIdx.x] = s;
  __syncthreads();
  if (threadIdx.x == 0) {
    double tot = 0.0;
    for (int k = 0; k < 256; ++k) tot += sh[k];
    *out = tot;
  }
}

}  // namespace aerofx

using namespace aerofx;

extern "C" int aerofx_adjoint_residual(aerofx_ctx *ctx, const double *U, const double *lambda,
                                       double *dRdU_T_lambda, double *dRdX_T_lambda) {
  if (!ctx || !U || !lambda) return set_error(AEROFX_ERR_ARG, "adjoint_residual: null argument");
  if (ctx->fc.low_mach)
    return set_error(AEROFX_ERR_STATE, "adjoint_residual: not available with low-Mach preconditioning");
  if (int rf = refuse_failsafe_nodes(ctx, "adjoint_residual")) return rf;
  if (!dRdU_T_lambda && !dRdX_T_lambda) return AEROFX_OK;
  int rc = launch_adjoint(ctx, U, lambda, dRdU_T_lambda, dRdX_T_lambda);
  if (rc) return rc;
  hipError_t e = hipStreamSynchronize(ctx->stream);
  return e == hipSuccess ? AEROFX_OK : set_hip_error(e, "adjoint_residual");
}

extern "C" int aerofx_wall_force(aerofx_ctx *ctx, const double *U, const double dir[3], double *J,
                                 double *dJdU, double *dJdX) {
  if (!ctx || !U || !dir || !J) return set_error(AEROFX_ERR_ARG, "wall_force: null argument");
  int rc = ensure_adjoint(ctx);
  if (rc) return rc;
  Adjoint *a = ctx->adj;
  const DevTables &t = ctx->tab;
  if ((rc = launch_primitive_il(ctx, U))) return rc;
  if (ctx->F > 0) {
    hipLaunchKernelGGL(k_lift_faces, grid_for(ctx->F), dim3(kAdjBlock), 0, ctx->stream, ctx->F, t.sh, a->faces, t.fcode,
                       t.fnorm3, t.X4, ctx->d_V, dir[0], dir[1], dir[2], a->Jf, dJdX ? a->FX : nullptr);
    // the viscous stress on the wall faces (PostFcnNS::computeForce)
    if ((rc = launch_visc_force(ctx, dir, a->Jf, dJdU || dJdX))) return rc;
    hipLaunchKernelGGL(k_sum_ordered, dim3(1), dim3(256), 0, ctx->stream, ctx->F, a->Jf, a->Jf + ctx->F);
  } else {
    hipLaunchKernelGGL(k_sum_ordered, dim3(1), dim3(256), 0, ctx->stream, 0, a->Jf, a->Jf);  // no faces: J = 0
  }
  if (dJdU || dJdX)
    hipLaunchKernelGGL(k_lift_nodes, grid_for(t.N), dim3(kAdjBlock), 0, ctx->stream, t, U, ctx->gas, a->nfslot,
                       a->FX, dir[0], dir[1], dir[2], dJdU, dJdX);
  if ((dJdU || dJdX) && (rc = launch_visc_force_gather(ctx, dJdU, dJdX))) return rc;
  hipError_t e = hipGetLastError();
  if (e == hipSuccess) e = hipMemcpyAsync(a->h_J, a->Jf + ctx->F, sizeof(double), hipMemcpyDeviceToHost, ctx->stream);
  if (e == hipSuccess) e = hipStreamSynchronize(ctx->stream);
  if (e != hipSuccess) return set_hip_error(e, "wall_force");
  *J = *a->h_J;
  return AEROFX_OK;
}
