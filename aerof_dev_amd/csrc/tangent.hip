// tangent.hip -- forward-mode derivative of the residual on gfx950:
//   dR = (dR/dU) dU + (dR/dX) dX
// for the second-order residual R_i = (1/V_i)(sum_edges +-F(V_ij, V_ji, n_ij)
// + sum_faces F_b(V_i, n_f/3)).  This is the directional derivative
// SpaceOperator::computeDerivativeOfResidual (SpaceOperator.C:917-1070) and
// EdgeSet::computeDerivativeOfFiniteVolumeTerm (Edge.C:1494-1573) form for a
// shape perturbation dX (with dU the state perturbation: the exact product of
// the second-order Jacobian that MatVecProdH2 applies, MatVecProd.C:1293+).
// Every quantity the residual computes from X is differentiated: dual-face
// normals and control volumes (per tet, ElemTetCore.C:31-44, 281-330), face
// normals (FaceTriaCore.C:31-37), LSQ moments, Cholesky factors and weights,
// the gradients, the reconstruction distances and the fluxes.
//
// The numbers are Dual (value, derivative along the one seeded direction)
// pushed through the same templated routines the residual uses.  Stages:
//   1. forward residual: V, LSQ gradients, raw flux sums S (the MUSCL
//      gradients are recomputed, nothing from an earlier call is kept)
//   2. geometry, when the mesh moves: dn per edge (its tets in tet order), a
//      quarter of each tet's volume derivative, dn_f per boundary face
//   3. per node: dV(U) and the gradients' derivative
//   4. per edge and boundary face: reconstruction and flux in Dual
//   5. per node: dS = sum over upper edges of dF - sum over lower edges of dF
//      + faces; dR = dS / V - S dV / V^2
// Sums are in fixed orders: deterministic from run to run.
#include <hip/hip_runtime.h>

#include "context.h"
#include "device_dual.h"
#include "device_sens.h"
#include "host_internal.h"

namespace aerofx {

struct Tangent {
  double *S = nullptr;    // [N][5] raw flux sums of the forward pass
  double *dV = nullptr;   // il<5>
  double *dG = nullptr;   // il<15>
  double *dn = nullptr;   // il<3> over edge positions
  double *dvol = nullptr; // [T] a quarter of each tet's volume derivative
  double *dfn = nullptr;  // [F][3] full face normal
  double *dF = nullptr;   // il<5> over edge positions
  double *dFf = nullptr;  // [3F][5] boundary-face fluxes' derivatives, per node face slot
  // the state part of the exact product operator (MatVecProdH2), kept from
  // its selection: primitive state and LSQ gradients, laid out as d_V and
  // d_grad
  double *V0 = nullptr, *G0 = nullptr;
};

void free_tangent(aerofx_ctx *c) {
  delete c->tan;  // device memory is owned by the context allocation list
  c->tan = nullptr;
}

namespace {

constexpr int kTanBlock = 256;

__device__ __forceinline__ Dual coord(const double *__restrict__ X4, const double *__restrict__ dX, int n, int a) {
  return Dual(X4[4 * (size_t)n + a], dX ? dX[3 * (size_t)n + a] : 0.0);
}
__device__ __forceinline__ void load_xdx(const double *__restrict__ X4, const double *__restrict__ dX, int n,
                                         double x[3], double dx[3]) {
  const double4 p = *reinterpret_cast<const double4 *>(X4 + 4 * (size_t)n);
  x[0] = p.x;
  x[1] = p.y;
  x[2] = p.z;
#pragma unroll
  for (int a = 0; a < 3; ++a) dx[a] = dX[3 * (size_t)n + a];
}
__device__ __forceinline__ int pick_id(const int4 &d, int k) { return k == 0 ? d.x : (k == 1 ? d.y : (k == 2 ? d.z : d.w)); }

// ---------------------------------------------------------------------------
// 2. geometry
// ---------------------------------------------------------------------------
// dn of the edge at position pos: over the tets around it in tet order.  The
// median dual face of edge (a, b) in a tet with opposite vertices c, d
// (ElemTet::computeEdgeNormalsGCL1 with Xn == Xnp1, ElemTetCore.C:281-330, 1.5 p x r
// of the face centroids p, r from the centroid) is (c - d) x (a + b - c - d) / 24,
// so a tet adds two cross products and only its two other vertices are loaded
// (162 -> 29 us at 52k nodes; all four vertices, the centroids and their
// products in dual numbers before).  The differences of near vertices also
// round at the edge's scale: against extended precision the error of a tet's
// term is 1e-16 (3e-14 with centroids of vertices far from the origin).
__global__ __launch_bounds__(kTanBlock) void k_tan_edge_normals(DevTables t, const int *__restrict__ etrow,
                                                                const int *__restrict__ etslot,
                                                                const int4 *__restrict__ tets,
                                                                const double *__restrict__ dX,
                                                                double *__restrict__ dn) {
#pragma clang fp contract(on)
  const int pos = xcd_chunk(blockIdx.x, (t.E + kTanBlock - 1) / kTanBlock) * kTanBlock + (int)threadIdx.x;
  if (pos >= t.E) return;
  const int l = t.pedge[pos];
  const int2 ij = t.eij[l];
  double xi[3], xj[3], di[3], dj[3];
  load_xdx(t.X4, dX, ij.x, xi, di);
  load_xdx(t.X4, dX, ij.y, xj, dj);
  double acc[3] = {0.0, 0.0, 0.0};
  // four tets at a time, so that their index chains overlap; the places past the
  // last tet repeat it with weight zero
  const int q1 = etrow[l + 1];
  for (int q0 = etrow[l]; q0 < q1; q0 += 4) {
    int s[4], nc[4], nd[4];
    double sg[4];
#pragma unroll
    for (int b = 0; b < 4; ++b) s[b] = etslot[min(q0 + b, q1 - 1)];
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      const int tt = s[b] / 6, e = s[b] - 6 * tt;
      const int4 d4 = tets[tt];
      int oc = 0, od = 0;
#pragma unroll
      for (int k = 0; k < 6; ++k)
        if (k == e) {
          oc = kOpp[k][0];
          od = kOpp[k][1];
        }
      nc[b] = pick_id(d4, oc);
      nd[b] = pick_id(d4, od);
      // oriented from the lower to the higher node id
      sg[b] = q0 + b >= q1 ? 0.0 : (pick_id(d4, e < 3 ? 0 : (e < 5 ? 1 : 2)) == ij.x ? 1.0 : -1.0);
    }
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      double xc[3], xd[3], dc[3], dd[3], p[3], dp[3], r[3], dr[3];
      load_xdx(t.X4, dX, nc[b], xc, dc);
      load_xdx(t.X4, dX, nd[b], xd, dd);
#pragma unroll
      for (int a = 0; a < 3; ++a) {
        p[a] = sg[b] * (xc[a] - xd[a]);
        dp[a] = sg[b] * (dc[a] - dd[a]);
        r[a] = (xi[a] - xc[a]) + (xj[a] - xd[a]);
        dr[a] = (di[a] - dc[a]) + (dj[a] - dd[a]);
      }
      acc[0] += (dp[1] * r[2] - dp[2] * r[1]) + (p[1] * dr[2] - p[2] * dr[1]);
      acc[1] += (dp[2] * r[0] - dp[0] * r[2]) + (p[2] * dr[0] - p[0] * dr[2]);
      acc[2] += (dp[0] * r[1] - dp[1] * r[0]) + (p[0] * dr[1] - p[1] * dr[0]);
    }
  }
#pragma unroll
  for (int a = 0; a < 3; ++a) acc[a] *= 1.0 / 24.0;
  store_il<3>(t.sh, dn, pos, acc);
}

// a quarter of each tet's volume derivative (ElemTet::computeVolume,
// ElemTetCore.C:31-44); the node pass sums them in tet order
__global__ __launch_bounds__(kTanBlock) void k_tan_vol(int T, const int4 *__restrict__ tets,
                                                       const double *__restrict__ X4, const double *__restrict__ dX,
                                                       double *__restrict__ dvol) {
#pragma clang fp contract(on)
  const int t = blockIdx.x * kTanBlock + threadIdx.x;
  if (t >= T) return;
  const int4 d4 = tets[t];
  const int id[4] = {d4.x, d4.y, d4.z, d4.w};
  double x[4][3], dx[4][3];
#pragma unroll
  for (int k = 0; k < 4; ++k) load_xdx(X4, dX, id[k], x[k], dx[k]);
  double e[3][3], de[3][3];
#pragma unroll
  for (int k = 0; k < 3; ++k)
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      e[k][a] = x[k + 1][a] - x[0][a];
      de[k][a] = dx[k + 1][a] - dx[0][a];
    }
  double s = 0.0;
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    const double *a = e[(k + 1) % 3], *b = e[(k + 2) % 3], *d = de[k];
    s += d[0] * (a[1] * b[2] - a[2] * b[1]) + d[1] * (a[2] * b[0] - a[0] * b[2]) + d[2] * (a[0] * b[1] - a[1] * b[0]);
  }
  dvol[t] = 0.25 * (1.0 / 6.0) * s;
}

// dn_f = d(0.5 (x2 - x0) x (x1 - x0)) (FaceTria::computeNormal, FaceTriaCore.C:31-37)
__global__ __launch_bounds__(kTanBlock) void k_tan_faces(int F, const int *__restrict__ faces,
                                                         const double *__restrict__ X4,
                                                         const double *__restrict__ dX, double *__restrict__ dfn) {
  const int f = blockIdx.x * kTanBlock + threadIdx.x;
  if (f >= F) return;
  Dual x[3][3];
#pragma unroll
  for (int v = 0; v < 3; ++v) {
    const int nd = faces[3 * (size_t)f + v];
#pragma unroll
    for (int a = 0; a < 3; ++a) x[v][a] = coord(X4, dX, nd, a);
  }
  Dual p[3], q[3];
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    p[a] = x[2][a] - x[0][a];
    q[a] = x[1][a] - x[0][a];
  }
  dfn[3 * (size_t)f] = (0.5 * (p[1] * q[2] - p[2] * q[1])).d;
  dfn[3 * (size_t)f + 1] = (0.5 * (p[2] * q[0] - p[0] * q[2])).d;
  dfn[3 * (size_t)f + 2] = (0.5 * (p[0] * q[1] - p[1] * q[0])).d;
}

// ---------------------------------------------------------------------------
// 3. per node: dV and, at second order, the derivative of the gradients
// ---------------------------------------------------------------------------
__device__ __forceinline__ void load_v(const double *__restrict__ U, const double *__restrict__ dU, int n,
                                       const Gas &gas, Dual v[5]) {
  Dual u[5];
#pragma unroll
  for (int k = 0; k < 5; ++k) u[k] = Dual(U[5 * (size_t)n + k], dU ? dU[5 * (size_t)n + k] : 0.0);
  prim_from_cons(u, gas, v);
}

// dV alone; with the mesh fixed the gradients are linear in V, so theirs are
// the gradients of dV (launch_gradients_il)
__global__ __launch_bounds__(kTanBlock) void k_tan_dv(int N, int sh, const double *__restrict__ U,
                                                      const double *__restrict__ dU, Gas gas,
                                                      double *__restrict__ dV, const int *__restrict__ done) {
  if (done && *done) return;
  const int n = blockIdx.x * kTanBlock + threadIdx.x;
  if (n >= N) return;
  Dual v[5];
  load_v(U, dU, n, gas, v);
  const double d[5] = {v[0].d, v[1].d, v[2].d, v[3].d, v[4].d};
  store_il<5>(sh, dV, n, d);
}

// the derivative of the gradients with the mesh moving: g solves M g = b with the
// moments M = sum dx dx^T and b = sum dx dV, so
//   dg = M^-1 (db - dM g) = M^-1 sum ddx (dV - dx . g) + dx (ddV - ddx . g):
// one sweep over the neighbours, and the weights of the gradient pass (linear in
// dx) apply M^-1.
template <int SH>
__global__ __launch_bounds__(kTanBlock) void k_tan_grad(DevTables t, const double *__restrict__ V,
                                                        const double *__restrict__ grad,
                                                        const double *__restrict__ dV,
                                                        const double *__restrict__ dX, double *__restrict__ dG) {
  const int sl = wave_slice(t);
  if (sl >= t.ns) return;
  const int n = sl * kWave + lane_id(), nn = min(n, t.N - 1);
  const int deg = n < t.N ? t.rowptr[n + 1] - t.rowptr[n] : 0;
  double vn[5], wn[5], gn[15], xn[3], yn[3], acc[15];
  load_il<5>(Lay<SH>(), V, nn, vn);
  load_il<5>(Lay<SH>(), dV, nn, wn);
  load_il<15>(Lay<SH>(), grad, nn, gn);
  load_il<3>(Lay<SH>(), t.X3, nn, xn);
#pragma unroll
  for (int a = 0; a < 3; ++a) yn[a] = dX[3 * (size_t)nn + a];
#pragma unroll
  for (int q = 0; q < 15; ++q) acc[q] = 0.0;
  const int kb = t.nb.kptr[sl], ke = t.nb.kptr[sl + 1];
  for (int w = kb; w < ke; ++w) {
    const bool act = w - kb < deg;
    const int pos = t.nb.koff[w] + lanes_below(act);
    if (!act) continue;
    const int m = t.nb.idx[pos];
    double vm[5], wm[5], dx[3], dy[3];
    load_il<5>(Lay<SH>(), V, m, vm);
    load_il<5>(Lay<SH>(), dV, m, wm);
    load_il<3>(Lay<SH>(), t.X3, m, dx);
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      dy[a] = dX[3 * (size_t)m + a] - yn[a];
      dx[a] -= xn[a];
    }
#pragma unroll
    for (int q = 0; q < 5; ++q) {
      const double e = (vm[q] - vn[q]) - (dx[0] * gn[q] + dx[1] * gn[5 + q] + dx[2] * gn[10 + q]);
      const double f = (wm[q] - wn[q]) - (dy[0] * gn[q] + dy[1] * gn[5 + q] + dy[2] * gn[10 + q]);
#pragma unroll
      for (int a = 0; a < 3; ++a) acc[5 * a + q] += dy[a] * e + dx[a] * f;
    }
  }
  if (n >= t.N) return;
  double L[6];
#pragma unroll
  for (int q = 0; q < 6; ++q) L[q] = t.lsq6[6 * (size_t)n + q];
#pragma unroll
  for (int q = 0; q < 5; ++q) {
    double w[3];
    lsq_weights(L, acc[q], acc[5 + q], acc[10 + q], w);
#pragma unroll
    for (int a = 0; a < 3; ++a) acc[5 * a + q] = w[a];
  }
  store_il<15>(Lay<SH>(), dG, n, acc);
}

// ---------------------------------------------------------------------------
// 4. per edge: reconstruction and Roe flux in Dual; boundary-face fluxes
// ---------------------------------------------------------------------------
// A wave per (64 nodes, k-th upper edge), as the residual's flux pass on small
// meshes; the first nfb blocks take the boundary-face slots.  MOVE: the mesh
// moves (dX, dn, dfn), otherwise their derivatives are zero and not read.
// Bound by the gathers of both ends' 46 values (44 us at 104k nodes; selection,
// time step and two products there 512 -> 296 us, with the flux's derivative by
// position and summed as the residual's).
template <bool SECOND, bool MOVE, int SH>
__global__ __launch_bounds__(kTanBlock) void k_tan_flux(DevTables t, int nfb, const double *__restrict__ V,
                                                        const double *__restrict__ grad,
                                                        const double *__restrict__ dV,
                                                        const double *__restrict__ dG,
                                                        const double *__restrict__ dX,
                                                        const double *__restrict__ dn,
                                                        const double *__restrict__ dfn, FluxConsts fc,
                                                        double *__restrict__ dF, double *__restrict__ dFf,
                                                        const int *__restrict__ done) {
  if (done && *done) return;
  if ((int)blockIdx.x < nfb) {
    const int q = blockIdx.x * kTanBlock + threadIdx.x;
    if (q >= 3 * t.F) return;
    const int n = t.fnode[q], face = t.fidx[q];
    double v[5], dv[5];
    load_il<5>(Lay<SH>(), V, n, v);
    load_il<5>(Lay<SH>(), dV, n, dv);
    Dual Vn[5], nv[3], fl[5];
#pragma unroll
    for (int k = 0; k < 5; ++k) Vn[k] = Dual(v[k], dv[k]);
    const double third = 1.0 / 3.0;
#pragma unroll
    for (int a = 0; a < 3; ++a)
      nv[a] = Dual(t.fnorm3[3 * (size_t)face + a], MOVE ? third * dfn[3 * (size_t)face + a] : 0.0);
    face_flux(fc, t.fcode[face], nv, Vn, fl);
#pragma unroll
    for (int k = 0; k < 5; ++k) dFf[5 * (size_t)q + k] = fl[k].d;
    return;
  }
  const int nb = (t.nup + kTanBlock / kWave - 1) / (kTanBlock / kWave);
  const int w = xcd_chunk(blockIdx.x - nfb, nb) * (kTanBlock / kWave) + (int)(threadIdx.x / kWave);
  if (w >= t.nup) return;
  const UpperEntry u = upper_entry<SH>(t, w);
  if (!u.act) return;
  const int i = u.i, pos = u.pos;
  const int j = t.up.idx[pos];
  Dual Vi[5], Vj[5], Vij[5], Vji[5];
  {
    double a[5], b[5];
    load_il<5>(Lay<SH>(), V, i, a);
    load_il<5>(Lay<SH>(), dV, i, b);
#pragma unroll
    for (int k = 0; k < 5; ++k) Vi[k] = Dual(a[k], b[k]);
    load_il<5>(Lay<SH>(), V, j, a);
    load_il<5>(Lay<SH>(), dV, j, b);
#pragma unroll
    for (int k = 0; k < 5; ++k) Vj[k] = Dual(a[k], b[k]);
  }
  if (SECOND) {
    double xi[3], xj[3], gi[15], gj[15], hi[15], hj[15];
    load_il<3>(Lay<SH>(), t.X3, i, xi);
    load_il<3>(Lay<SH>(), t.X3, j, xj);
    Dual dx[3];
#pragma unroll
    for (int a = 0; a < 3; ++a)
      dx[a] = Dual(xj[a] - xi[a], MOVE ? dX[3 * (size_t)j + a] - dX[3 * (size_t)i + a] : 0.0);
    load_il<15>(Lay<SH>(), grad, i, gi);
    load_il<15>(Lay<SH>(), dG, i, hi);
    load_il<15>(Lay<SH>(), grad, j, gj);
    load_il<15>(Lay<SH>(), dG, j, hj);
#pragma unroll
    for (int k = 0; k < 5; ++k) {
      const Dual ddVij = dx[0] * Dual(gi[k], hi[k]) + dx[1] * Dual(gi[5 + k], hi[5 + k]) +
                         dx[2] * Dual(gi[10 + k], hi[10 + k]);
      const Dual ddVji = dx[0] * Dual(gj[k], hj[k]) + dx[1] * Dual(gj[5 + k], hj[5 + k]) +
                         dx[2] * Dual(gj[10 + k], hj[10 + k]);
      reconstruct(fc.beta, Vi[k], ddVij, Vj[k], ddVji, Vij[k], Vji[k]);
    }
  } else {
#pragma unroll
    for (int k = 0; k < 5; ++k) {
      Vij[k] = Vi[k];
      Vji[k] = Vj[k];
    }
  }
  double n0[3], n1[3] = {0.0, 0.0, 0.0};
  load_il<3>(Lay<SH>(), t.pnormal, pos, n0);
  if (MOVE) load_il<3>(Lay<SH>(), dn, pos, n1);
  const Dual nv[3] = {Dual(n0[0], n1[0]), Dual(n0[1], n1[1]), Dual(n0[2], n1[2])};
  Dual f[5];
  if (n0[0] * n0[0] + n0[1] * n0[1] + n0[2] * n0[2] >= 1e-36) roe_flux(fc.gas, nv, Vij, Vji, f);
  const double d[5] = {f[0].d, f[1].d, f[2].d, f[3].d, f[4].d};
  store_il<5>(Lay<SH>(), dF, pos, d);
}

// ---------------------------------------------------------------------------
// 5. per node: dS and dR (+ p / dt, the backward-Euler time term of the exact
//    product, when dt is given)
// ---------------------------------------------------------------------------
template <bool MOVE, int SH>
__global__ __launch_bounds__(kTanBlock) void k_tan_nodes(DevTables t, const double *__restrict__ S,
                                                         const int *__restrict__ ntrow,
                                                         const int *__restrict__ ntslot,
                                                         const double *__restrict__ dvol,
                                                         const double *__restrict__ dF,
                                                         const double *__restrict__ dFf,
                                                         const double *__restrict__ p, const double *__restrict__ dt,
                                                         double *__restrict__ dR, const int *__restrict__ done) {
  if (done && *done) return;
  const int sl = wave_slice(t);
  if (sl >= t.ns) return;
  const int n = sl * kWave + lane_id();
  const bool live = n < t.N;
  double s[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
  add_slots<false>(Lay<SH>(), t.up, sl, live ? t.eup[n + 1] - t.eup[n] : 0, dF, s);
  add_slots<true>(Lay<SH>(), t.lo, sl, live ? t.lrow[n + 1] - t.lrow[n] : 0, dF, s);
  if (!live) return;
  for (int q = t.frow[n]; q < t.frow[n + 1]; ++q)
#pragma unroll
    for (int k = 0; k < 5; ++k) s[k] += dFf[5 * (size_t)q + k];
  // R = S * (1/V): dR = dS / V + S d(1/V) = dS / V - S dV / V^2
  const double ic = t.invcv[n];
  if (MOVE) {
    double dcv = 0.0;
#pragma unroll 8
    for (int q = ntrow[n]; q < ntrow[n + 1]; ++q) dcv += dvol[ntslot[q] >> 2];
    const double dic = -dcv * ic * ic;
#pragma unroll
    for (int k = 0; k < 5; ++k) dR[5 * (size_t)n + k] = s[k] * ic + S[5 * (size_t)n + k] * dic;
  } else {
    const double it = dt ? 1.0 / dt[n] : 0.0;
#pragma unroll
    for (int k = 0; k < 5; ++k) {
      const double r = s[k] * ic;
      dR[5 * (size_t)n + k] = dt ? r + p[5 * (size_t)n + k] * it : r;
    }
  }
}

template <class T>
int alloc_n(aerofx_ctx *c, size_t n, T **out) {
  void *p = nullptr;
  int rc = ctx_alloc(c, n * sizeof(T), &p);
  *out = static_cast<T *>(p);
  return rc;
}

int ensure_tangent(aerofx_ctx *c) {
  if (c->tan) return 0;
  int rc = ensure_elem_tables(c);
  if (rc) return rc;
  Tangent *g = new Tangent();
  const size_t N = c->N, E = c->E, F = std::max(c->F, 1);
  if ((rc = alloc_n(c, 5 * N, &g->S)) || (rc = alloc_n(c, il_count<5>(c->tab.sh, N), &g->dV)) ||
      (rc = alloc_n(c, il_count<15>(c->tab.sh, N), &g->dG)) || (rc = alloc_n(c, il_count<3>(c->tab.sh, E), &g->dn)) ||
      (rc = alloc_n(c, (size_t)c->T, &g->dvol)) || (rc = alloc_n(c, 3 * F, &g->dfn)) ||
      (rc = alloc_n(c, il_count<5>(c->tab.sh, E), &g->dF)) || (rc = alloc_n(c, 15 * F, &g->dFf))) {
    delete g;
    return rc;
  }
  c->tan = g;
  return 0;
}

inline dim3 grid_for(long long n) { return dim3((unsigned)((n + kTanBlock - 1) / kTanBlock)); }

template <bool SECOND, bool MOVE>
void launch_flux(aerofx_ctx *c, const double *V, const double *G, const double *dX, const int *done) {
  const Tangent *g = c->tan;
  const DevTables &t = c->tab;
  const int nfb = (3 * t.F + kTanBlock - 1) / kTanBlock;
  const unsigned nb = (unsigned)((t.nup + kTanBlock / kWave - 1) / (kTanBlock / kWave));
  const auto k = t.sh ? k_tan_flux<SECOND, MOVE, kGroupShift> : k_tan_flux<SECOND, MOVE, 0>;
  if (nfb + nb)
    hipLaunchKernelGGL(k, dim3(nfb + nb), dim3(kTanBlock), 0, c->stream, t, nfb, V, G, g->dV, g->dG, dX, g->dn, g->dfn,
                       c->fc, g->dF, g->dFf, done);
}

// stages 3 to 5 about the state U with its V and gradients G
int launch_stages(aerofx_ctx *c, const double *U, const double *V, const double *G, const double *dU,
                  const double *dX, const double *dt, double *dR, const int *done) {
  Tangent *g = c->tan;
  const ElemTables &el = *c->elem;
  const DevTables &t = c->tab;
  const bool second = c->p.second_order != 0;
  hipLaunchKernelGGL(k_tan_dv, grid_for(t.N), dim3(kTanBlock), 0, c->stream, t.N, t.sh, U, dU, c->gas, g->dV, done);
  if (second && dX) {
    hipLaunchKernelGGL(t.sh ? k_tan_grad<kGroupShift> : k_tan_grad<0>, slice_grid(t.ns), dim3(kTanBlock), 0,
                       c->stream, t, V, G, g->dV, dX, g->dG);
  } else if (second) {
    if (int rc = launch_gradients_il(c, g->dV, g->dG, done)) return rc;
  }
  if (second && dX)
    launch_flux<true, true>(c, V, G, dX, done);
  else if (second)
    launch_flux<true, false>(c, V, G, nullptr, done);
  else if (dX)
    launch_flux<false, true>(c, V, G, dX, done);
  else
    launch_flux<false, false>(c, V, G, nullptr, done);
  if (dX) {
    const auto k = t.sh ? k_tan_nodes<true, kGroupShift> : k_tan_nodes<true, 0>;
    hipLaunchKernelGGL(k, slice_grid(t.ns), dim3(kTanBlock), 0, c->stream, t, g->S, el.ntrow, el.ntslot, g->dvol, g->dF,
                       g->dFf, nullptr, nullptr, dR, done);
  } else {
    const auto k = t.sh ? k_tan_nodes<false, kGroupShift> : k_tan_nodes<false, 0>;
    hipLaunchKernelGGL(k, slice_grid(t.ns), dim3(kTanBlock), 0, c->stream, t, g->S, nullptr, nullptr, nullptr, g->dF,
                       g->dFf, dU, dt, dR, done);
  }
  // the Navier-Stokes Galerkin term
  return launch_visc_tangent(c, V, dU, dX, dR, done);
}

}  // namespace

int launch_tangent(aerofx_ctx *c, const double *U, const double *dU, const double *dX, double *dR) {
  int rc = ensure_tangent(c);
  if (rc) return rc;
  Tangent *g = c->tan;
  const ElemTables &el = *c->elem;
  const DevTables &t = c->tab;
  // 1. forward pass: V, gradients, raw flux sums
  if ((rc = launch_residual(c, U, g->S, false))) return rc;
  // 2. geometry
  if (dX) {
    if (t.E > 0)
      hipLaunchKernelGGL(k_tan_edge_normals, grid_for(t.E), dim3(kTanBlock), 0, c->stream, t, el.etrow, el.etslot,
                         (const int4 *)el.tets, dX, g->dn);
    if (c->T > 0)
      hipLaunchKernelGGL(k_tan_vol, grid_for(c->T), dim3(kTanBlock), 0, c->stream, c->T, (const int4 *)el.tets, t.X4, dX,
                         g->dvol);
    if (t.F > 0)
      hipLaunchKernelGGL(k_tan_faces, grid_for(t.F), dim3(kTanBlock), 0, c->stream, t.F, el.faces, t.X4, dX, g->dfn);
  }
  // 3.-5.
  if ((rc = launch_stages(c, U, c->d_V, c->d_grad, dU, dX, nullptr, dR, nullptr))) return rc;
  hipError_t e = hipGetLastError();
  return e == hipSuccess ? 0 : set_hip_error(e, "tangent launch");
}

// MatVecProdH2::evaluate (MatVecProd.C:1560-1609) as a matrix-free exact
// product: the forward pass at Q leaves its primitive state and LSQ gradients
// in the tangent workspace (the mesh does not move: no geometry terms).
int launch_h2_select(aerofx_ctx *c, const double *Q) {
  int rc = ensure_tangent(c);
  if (rc) return rc;
  Tangent *g = c->tan;
  const DevTables &t = c->tab;
  if (!g->V0) {  // both or neither
    double *V0 = nullptr, *G0 = nullptr;
    if ((rc = alloc_n(c, il_count<5>(c->tab.sh, t.N), &V0))) return rc;
    if ((rc = alloc_n(c, il_count<15>(c->tab.sh, t.N), &G0))) {
      ctx_release(c, V0);
      return rc;
    }
    g->V0 = V0;
    g->G0 = G0;
  }
  const ResidualBufs b{g->V0, g->G0, c->d_Fm, c->d_P};
  return launch_residual_with(c, b, Q, g->S, false);
}

// MatVecProdH2::apply (MatVecProd.C:1647-1670): y = (dR/dU) p + p / dt at the
// selected Q (dt NULL: no time term); every kernel returns at once when
// *done != 0 (device-resident Krylov loops).
int launch_h2_apply(aerofx_ctx *c, const double *Q, const double *p, const double *dt, double *y,
                    const int *done) {
  Tangent *g = c->tan;
  if (!g || !g->V0) return set_error(AEROFX_ERR_STATE, "h2 apply: operator not selected");
  int rc;
  if ((rc = launch_stages(c, Q, g->V0, g->G0, p, nullptr, dt, y, done))) return rc;
  // the wall rows of the Navier-Stokes conditions (after the time term)
  if ((rc = launch_bcs_product(c, Q, p, y, done))) return rc;
  hipError_t e = hipGetLastError();
  return e == hipSuccess ? 0 : set_hip_error(e, "h2 apply launch");
}

}  // namespace aerofx

using namespace aerofx;

extern "C" int aerofx_residual_derivative(aerofx_ctx *c, const double *U, const double *dU, const double *dX,
                                          double *dR) {
  if (!c || !U || !dR) return set_error(AEROFX_ERR_ARG, "residual_derivative: null argument");
  if (c->fc.low_mach)
    return set_error(AEROFX_ERR_STATE, "residual_derivative: not available with low-Mach preconditioning");
  if (int rf = refuse_failsafe_nodes(c, "residual_derivative")) return rf;
  int rc = launch_tangent(c, U, dU, dX, dR);
  if (rc) return rc;
  hipError_t e = hipMemcpyAsync(c->h_err, c->d_err, sizeof(int), hipMemcpyDeviceToHost, c->stream);
  if (e == hipSuccess) e = hipStreamSynchronize(c->stream);
  if (e != hipSuccess) return set_hip_error(e, "residual_derivative sync");
  return c->h_err[0];
}
