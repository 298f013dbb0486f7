// residual.hip -- the FP64 edge residual on gfx950.
//
// SpaceOperator<5>::computeResidual (SpaceOperator.C:524-634), all
// deterministic (no atomics on floating-point data):
//
//  1. k_gradients_halo (k_gradients for meshes whose neighbourhoods do not fit
//     it)  one lane per node n walks its neighbours m in ascending
//     order (= ascending edge id) accumulating W(R_n, X_m - X_n) (V_m - V_n):
//     the reference's LSQ edge loop (SubDomain.C:137-159, 297-374) with the
//     same per-node addition order.  The pass also writes V = V(U), which
//     later passes gather, interleaved.
//  2. k_flux_edges each edge flux once (MUSCL + Van Albada + Roe's flux,
//     Edge.C:372-439), a wave per 64 lower nodes i: lane r takes the edges of
//     node i in turn, so its state, coordinates and gradients stay in
//     registers and the +f contributions P_i are summed in edge order (large
//     meshes), or a wave per (64 nodes, k-th upper edge) (small ones).
//     Boundary-face fluxes (Face.C:356-389) per face slot by further blocks.
//  3. k_flux_nodes node-parallel: R_n = (sum over lower edges (m, n), m
//     ascending, of -f, gathered from Fm) + P_n + boundary-face fluxes in face
//     order, times 1/V_n (SpaceOperator.C:599-624).
//
// Layouts: il and RowSlices (context.h).  blockIdx is remapped so that each XCD
// sweeps one contiguous node range, keeping the RCM neighbour window in its
// L2.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "context.h"
#include "host_internal.h"

namespace aerofx {

// neighbours per load batch of the per-entry gradient pass (measured at 128^3
// with record gathers: 2 -> 0.317 ms, 4 -> 0.310, 6 -> 0.307, 8 -> 0.301; from
// 10 on the batch no longer stays in registers)
constexpr int kGradChunk = 8;

// ---------------------------------------------------------------------------
// 1. gradients: one lane per node, neighbours in ascending order (= the
//    reference's edge order), so every node's sums are formed exactly as in
//    the reference's sequential edge loop.
// ---------------------------------------------------------------------------
// where a state comes from: U or V as [N][5], or the interleaved V
enum { kFromU = 0, kFromV = 1, kFromVil = 2 };
template <int FROM, class L>
__device__ __forceinline__ void load_state(L lay, const double *__restrict__ W, int n, double w[5]) {
  if (FROM == kFromVil) {
    load_il<5>(lay, W, n, w);
  } else {
#pragma unroll
    for (int k = 0; k < 5; ++k) w[k] = W[5 * (size_t)n + k];
  }
}
template <int FROM>
__device__ __forceinline__ void to_prim(const double w[5], const Gas &gas, double v[5]) {
  if (FROM == kFromU) {
    prim_from_cons(w, gas, v);
  } else {
#pragma unroll
    for (int k = 0; k < 5; ++k) v[k] = w[k];
  }
}
template <class L>
__device__ __forceinline__ void load_x(L lay, const DevTables &t, int n, double x[3]) {
  load_il<3>(lay, t.X3, n, x);
}

// ... from the records
__device__ __forceinline__ void load_x4(const DevTables &t, int n, double x[3]) {
  const double4 p = *reinterpret_cast<const double4 *>(t.X4 + 4 * (size_t)n);
  x[0] = p.x;
  x[1] = p.y;
  x[2] = p.z;
}

__device__ __forceinline__ void load_lsq(const DevTables &t, int n, double L[6]) {
#pragma unroll
  for (int q = 0; q < 6; ++q) L[q] = t.lsq6[6 * (size_t)n + q];
}

// acc += W(L, X_m - X_n) (V_m - V_n) (SubDomain.C:137-159, 297-374),
// variables V0 <= q < V1
template <int V0 = 0, int V1 = 5>
__device__ __forceinline__ void lsq_add(const double L[6], const double xm[3], const double xn[3],
                                        const double Vm[5], const double Vn[5], double acc[15]) {
  const double or11 = L[0], or22 = L[1], or33 = L[2], r12or11 = L[3], r23or22 = L[4], psi = L[5];
  const double dx0 = xm[0] - xn[0], dx1 = xm[1] - xn[1], dx2 = xm[2] - xn[2];
  const double alpha1 = dx0 * or11 * or11;
  const double alpha2 = (dx1 - r12or11 * dx0) * or22 * or22;
  const double alpha3 = (dx2 - r23or22 * dx1 + psi * dx0) * or33 * or33;
  const double w0 = alpha1 - r12or11 * alpha2 + psi * alpha3;
  const double w1 = alpha2 - r23or22 * alpha3;
  const double w2 = alpha3;
#pragma unroll
  for (int q = V0; q < V1; ++q) {
    const double d = Vm[q] - Vn[q];
    acc[q] += w0 * d;
    acc[5 + q] += w1 * d;
    acc[10 + q] += w2 * d;
  }
}

// kFromU also writes V (Vout); OUT3: gradients to ddx, ddy, ddz [N][5].
// Each lane walks its own row: of records (U or V [N][5], X4) a gather is one or
// two lines, and row order and slice order cost the same to index (by slices and
// with interleaved coordinates the pass took 176 us at 439k nodes, 112 so).
template <int FROM, bool OUT3>
__global__ __launch_bounds__(kBlock) void k_gradients(DevTables t, const double *__restrict__ W, Gas gas,
                                                      double *__restrict__ Vout, double *__restrict__ grad,
                                                      double *__restrict__ ddx, double *__restrict__ ddy,
                                                      double *__restrict__ ddz, int *__restrict__ err,
                                                      const int *__restrict__ done) {
  if (done && *done) return;
  if (err && blockIdx.x == 0 && threadIdx.x == 0) *err = 0;  // the flux pass follows in stream order
  const int sl = wave_slice(t);
  const int n = sl * kWave + lane_id();
  if (n >= t.N) return;
  double Vn[5], xn[3];
  {
    double w[5];
    load_state<FROM>(t.sh, W, n, w);
    to_prim<FROM>(w, gas, Vn);
  }
  if (Vout) store_il<5>(t.sh, Vout, n, Vn);
  load_x4(t, n, xn);
  double L[6], acc[15];
  load_lsq(t, n, L);
#pragma unroll
  for (int q = 0; q < 15; ++q) acc[q] = 0.0;
  // Neighbours in chunks of kGradChunk: the chunk's states and coordinates
  // are requested together and the next chunk's indices are prefetched, so a
  // row costs about one memory latency per chunk.  The sums are still formed
  // one neighbour at a time in ascending order.
  const int e0 = t.rowptr[n], e1 = t.rowptr[n + 1];
  int mi[kGradChunk];
#pragma unroll
  for (int k = 0; k < kGradChunk; ++k) mi[k] = e0 + k < e1 ? t.adj[e0 + k] : n;
  for (int e = e0; e < e1; e += kGradChunk) {
    double Wm[kGradChunk][5], xm[kGradChunk][3];
#pragma unroll
    for (int k = 0; k < kGradChunk; ++k) {
      load_state<FROM>(t.sh, W, mi[k], Wm[k]);
      load_x4(t, mi[k], xm[k]);
    }
#pragma unroll
    for (int k = 0; k < kGradChunk; ++k) mi[k] = e + kGradChunk + k < e1 ? t.adj[e + kGradChunk + k] : n;
#pragma unroll
    for (int k = 0; k < kGradChunk; ++k) {
      if (e + k >= e1) break;
      double Vm[5];
      to_prim<FROM>(Wm[k], gas, Vm);
      lsq_add(L, xm[k], xn, Vm, Vn, acc);
    }
  }
  if (!OUT3 && t.fs_mask && t.fs_mask[n]) {
    // DistNodalGrad::limit with failsafe tags (DistNodalGrad.C:1083-1104)
#pragma unroll
    for (int q = 0; q < 15; ++q) acc[q] = 0.0;
  }
  if (!OUT3) {
    store_il<15>(t.sh, grad, n, acc);
  } else {
#pragma unroll
    for (int k = 0; k < 5; ++k) {
      ddx[5 * (size_t)n + k] = acc[k];
      ddy[5 * (size_t)n + k] = acc[5 + k];
      ddz[5 * (size_t)n + k] = acc[10 + k];
    }
  }
}

// The same through LDS, a slice at a time per workgroup: the slice's
// neighbours overlap (about 14 * 64 adjacency entries are 480 different nodes
// in RCM or row order, runs of consecutive ids).  Each node of the halo is
// loaded once, by consecutive lanes, and the entries read LDS: 16-B pairs,
// consecutive lanes on consecutive nodes.  The pass is bound by the loads in
// flight: four workgroups per CU (by LDS, 64 B a halo node, five): two
// waves share the halo and split the variables, the workgroups stay for
// several slices and request the next one's data before they compute, and the
// tables are padded to one length per slice, so those requests depend on one
// earlier load only.  The sums are k_gradients', term for term.  At 2.1M nodes
// 266 us (kernel trace), at 275k 37, with U -> V in the same pass; k_gradients
// takes 252 and 34 from plain records of V, and a conversion of U before it 28
// at 2.1M.  Without the overlap 266 + 28, with one wave per slice 366 + 28.
constexpr int kHaloWaves = 2;
constexpr int kHaloThreads = kWave * kHaloWaves;
constexpr int kHaloBatch = 4;   // halo nodes a lane has in flight
constexpr int kHaloPairs = 8;   // place pairs (two entries) requested together

template <int FROM>
struct HaloLoad {
  double w[kHaloBatch][5], x[kHaloBatch][3];
  __device__ __forceinline__ void request(const DevTables &t, const double *__restrict__ U,
                                          const int m[kHaloBatch]) {
#pragma unroll
    for (int r = 0; r < kHaloBatch; ++r) {
      load_state<FROM>(Lay<kGroupShift>(), U, m[r], w[r]);
      load_x(Lay<kGroupShift>(), t, m[r], x[r]);
    }
  }
  // pair q of halo node h to sp[q * cap + h]: (V0, V1) (V2, V3) (V4, X0) (X1, X2)
  __device__ __forceinline__ void put(const Gas &gas, double2 *sp, int cap, int r0) {
#pragma unroll
    for (int r = 0; r < kHaloBatch; ++r) {
      const int h = r0 + r * kHaloThreads + (int)threadIdx.x;
      if (h >= cap) break;
      double v[5];
      to_prim<FROM>(w[r], gas, v);
      sp[h] = make_double2(v[0], v[1]);
      sp[cap + h] = make_double2(v[2], v[3]);
      sp[2 * cap + h] = make_double2(v[4], x[r][0]);
      sp[3 * cap + h] = make_double2(x[r][1], x[r][2]);
    }
  }
};

__device__ __forceinline__ void halo_ids(const DevTables &t, int sl, int r0, int m[kHaloBatch]) {
  const int *halo = t.halo + (size_t)sl * t.halo_cap;
#pragma unroll
  for (int r = 0; r < kHaloBatch; ++r) m[r] = halo[min(r0 + r * kHaloThreads + (int)threadIdx.x, t.halo_cap - 1)];
}

// this lane's node: state, coordinates, factors, degree and the places of its
// first entries
struct HaloRow {
  double w[5], xn[3], L[6];
  int deg;
  uint32_t loc[kHaloPairs];
  template <int FROM>
  __device__ __forceinline__ void request(const DevTables &t, const double *__restrict__ U, int sl) {
    const int nn = min(sl * kWave + lane_id(), t.N - 1);
    load_state<FROM>(Lay<kGroupShift>(), U, nn, w);
    load_x(Lay<kGroupShift>(), t, nn, xn);
    load_lsq(t, nn, L);
    deg = t.rowptr[nn + 1] - t.rowptr[nn];
    places(t, sl, 0);
  }
  __device__ __forceinline__ void places(const DevTables &t, int sl, int p0) {
    const uint32_t *q = t.hloc + (size_t)sl * t.halo_pairs * kWave + lane_id();
#pragma unroll
    for (int p = 0; p < kHaloPairs; ++p) loc[p] = p0 + p < t.halo_pairs ? q[(p0 + p) * kWave] : 0;
  }
};

// variables V0 <= q < V1 of this lane's gradients
template <int V0, int V1>
__device__ __forceinline__ void halo_sums(const DevTables &t, const double2 *sp, HaloRow &row, const double Vn[5],
                                          int sl, int n, double *__restrict__ grad) {
  const int cap = t.halo_cap;
  double acc[15];
#pragma unroll
  for (int q = 0; q < 15; ++q) acc[q] = 0.0;
  for (int p0 = 0; p0 < t.halo_pairs; p0 += kHaloPairs) {
    if (p0) row.places(t, sl, p0);
#pragma unroll
    for (int k = 0; k < 2 * kHaloPairs; ++k) {
      if (2 * p0 + k >= 2 * t.halo_pairs) break;
      const int hm = k & 1 ? row.loc[k >> 1] >> 16 : row.loc[k >> 1] & 0xffffu;
      const double2 b = sp[cap + hm], c = sp[2 * cap + hm], d = sp[3 * cap + hm];
      const double2 a = V0 < 2 ? sp[hm] : make_double2(0.0, 0.0);
      const double Vm[5] = {a.x, a.y, b.x, b.y, c.x}, xm[3] = {c.y, d.x, d.y};
      if (2 * p0 + k < row.deg) lsq_add<V0, V1>(row.L, xm, row.xn, Vm, Vn, acc);
    }
  }
  if (t.fs_mask && t.fs_mask[n]) {
    // DistNodalGrad::limit with failsafe tags (DistNodalGrad.C:1083-1104)
#pragma unroll
    for (int q = 0; q < 15; ++q) acc[q] = 0.0;
  }
#pragma unroll
  for (int d = 0; d < 3; ++d)
#pragma unroll
    for (int q = V0; q < V1; ++q) grad[il<15>(kGroupShift, n, 5 * d + q)] = acc[5 * d + q];
}

// The workgroups b, b + 8, ... take turns over the b % 8-th part of the slices
// (the XCD they run on).
template <int FROM>
__global__ __launch_bounds__(kHaloThreads) void k_gradients_halo(DevTables t, const double *__restrict__ U, Gas gas,
                                                                 double *__restrict__ Vout,
                                                                 double *__restrict__ grad, int *__restrict__ err,
                                                                 const int *__restrict__ done) {
  if (done && *done) return;
  extern __shared__ double2 sp[];
  const int cap = t.halo_cap;
  if (err && blockIdx.x == 0 && threadIdx.x == 0) *err = 0;  // the flux pass follows in stream order
  const int xcd = blockIdx.x % kNumXcd, turn = blockIdx.x / kNumXcd;
  const int step = ((int)gridDim.x - xcd + kNumXcd - 1) / kNumXcd;  // workgroups of this part
  const int s0 = (int)((long long)t.ns * xcd / kNumXcd), s1 = (int)((long long)t.ns * (xcd + 1) / kNumXcd);
  int sl = s0 + turn;
  if (sl >= s1) return;
  HaloLoad<FROM> load;
  HaloRow row;
  int m[kHaloBatch];
  halo_ids(t, sl, 0, m);
  row.request<FROM>(t, U, sl);
  load.request(t, U, m);
  int next = sl + step;
  if (next < s1) halo_ids(t, next, 0, m);
  while (true) {
    load.put(gas, sp, cap, 0);
    for (int r0 = kHaloBatch * kHaloThreads; r0 < cap; r0 += kHaloBatch * kHaloThreads) {
      // a halo beyond one batch: its remainder without the overlap
      int mr[kHaloBatch];
      halo_ids(t, sl, r0, mr);
      load.request(t, U, mr);
      load.put(gas, sp, cap, r0);
    }
    HaloRow cur = row;
    double Vn[5];
    to_prim<FROM>(cur.w, gas, Vn);
    __syncthreads();
    const bool more = next < s1;
    if (more) {
      load.request(t, U, m);
      row.request<FROM>(t, U, next);
    }
    const int n = sl * kWave + lane_id();
    if (n < t.N) {
      if ((int)threadIdx.x < kWave) {
        if (Vout) store_il<5>(Lay<kGroupShift>(), Vout, n, Vn);
        halo_sums<0, 3>(t, sp, cur, Vn, sl, n, grad);
      } else {
        halo_sums<3, 5>(t, sp, cur, Vn, sl, n, grad);
      }
    }
    if (!more) return;
    sl = next;
    next += step;
    if (next < s1) halo_ids(t, next, 0, m);
    __syncthreads();
  }
}

// ---------------------------------------------------------------------------
// 2. edge fluxes, computed once per edge
// ---------------------------------------------------------------------------
// One edge: reconstruction, check and flux.  LM: the spatial low-Mach flux
// (ROEFLUX5) with the edge length |X_j - X_i| in Turkel's beta.  bi, bj: the
// sides whose reconstruction is non-physical (checkReconstructedValues,
// EdgeCore.C:137-166, VarFcnSGEuler.h:90-110).
template <bool SECOND, bool LM>
__device__ __forceinline__ void edge_flux(const FluxConsts &fc, const double Vi[5], const double xi[3],
                                          const double *gi, const double Vj[5], const double xj[3],
                                          const double *gj, const double nv[3], double f[5], bool &bi, bool &bj) {
  const Gas &g = fc.gas;
  double Vij[5], Vji[5];
  double length = 1.0, dx0 = 0.0, dx1 = 0.0, dx2 = 0.0;
  if (SECOND || LM) {
    dx0 = xj[0] - xi[0];
    dx1 = xj[1] - xi[1];
    dx2 = xj[2] - xi[2];
  }
  if (LM) length = sqrt(dx0 * dx0 + dx1 * dx1 + dx2 * dx2);
  if (SECOND) {
#pragma unroll
    for (int k = 0; k < 5; ++k) {
      const double ddVij = dx0 * gi[k] + dx1 * gi[5 + k] + dx2 * gi[10 + k];
      const double ddVji = dx0 * gj[k] + dx1 * gj[5 + k] + dx2 * gj[10 + k];
      reconstruct(fc.beta, Vi[k], ddVij, Vj[k], ddVji, Vij[k], Vji[k]);
    }
  } else {
#pragma unroll
    for (int k = 0; k < 5; ++k) {
      Vij[k] = Vi[k];
      Vji[k] = Vj[k];
    }
  }
  bi = Vij[0] <= 0.0 || Vij[4] + g.pstiff <= 0.0;
  bj = Vji[0] <= 0.0 || Vji[4] + g.pstiff <= 0.0;
  if (nv[0] * nv[0] + nv[1] * nv[1] + nv[2] * nv[2] < 1e-36) {
#pragma unroll
    for (int k = 0; k < 5; ++k) f[k] = 0.0;
  } else if (LM) {
    roe_turkel_flux(g, fc.lm, true, nv, length, Vij, Vji, f);
  } else {
    roe_flux(g, nv, Vij, Vji, f);
  }
}

// flux of boundary-face slot q (a face of node fnode[q]) into Ff[q]
template <int SH>
__device__ __forceinline__ void face_slot_flux(const DevTables &t, const double *__restrict__ V, const FluxConsts &fc,
                                               int q, double *__restrict__ Ff) {
  const int n = t.fnode[q], face = t.fidx[q];
  const int code = t.fcode[face];
  const double nv[3] = {t.fnorm3[3 * (size_t)face], t.fnorm3[3 * (size_t)face + 1], t.fnorm3[3 * (size_t)face + 2]};
  double Vn[5], fl[5];
  load_state<kFromVil>(Lay<SH>(), V, n, Vn);
  if (is_wall_code(code)) {
    wallflux(nv, 0.0, Vn, fl);
  } else {
    const double *ub = (code == AEROFX_BC_INLET || code == -AEROFX_BC_INLET) ? fc.ub_in : fc.ub_out;
    boundflux5(fc.gas, nv, 0.0, Vn, ub, fl);
  }
#pragma unroll
  for (int k = 0; k < 5; ++k) Ff[5 * (size_t)q + k] = fl[k];
}

// ALL: a wave per slice, lane r takes the upper edges of its node in turn
// (node data in registers, P summed here); otherwise a wave per (slice, k)
// pair.  The first nfb blocks take the boundary-face slots.
template <bool SECOND, bool LM, bool ALL, int SH>
__global__ __launch_bounds__(kBlock) void k_flux_edges(DevTables t, int nfb, const double *__restrict__ V,
                                                       const double *__restrict__ grad, FluxConsts fc,
                                                       double *__restrict__ Fm, double *__restrict__ P,
                                                       double *__restrict__ Ff, int *__restrict__ err,
                                                       int *__restrict__ tag0, const int *__restrict__ done) {
  if (done && *done) return;
  if ((int)blockIdx.x < nfb) {
    const int q = blockIdx.x * kBlock + (int)threadIdx.x;
    if (q < 3 * t.F) face_slot_flux<SH>(t, V, fc, q, Ff);
    return;
  }
  const int nw = ALL ? t.ns : t.nup;
  const int nb = (nw + kBlock / kWave - 1) / (kBlock / kWave);
  const int w = xcd_chunk(blockIdx.x - nfb, nb) * (kBlock / kWave) + (int)(threadIdx.x / kWave);
  if (w >= nw) return;
  const int lane = lane_id();
  // (upper_entry's edge, with the own state requested before its place is known)
  constexpr bool places = !ALL && SH == 0;
  const int at = w * kWave + lane, sl = ALL ? w : (places ? 0 : t.upslice[w]);
  const int kb = places ? 0 : t.up.kptr[sl], ke = ALL ? t.up.kptr[sl + 1] : 0;
  const int i = places ? t.uprow[min(at, t.E - 1)] : sl * kWave + lane;
  const bool live = places ? at < t.E : i < t.N;
  const int ii = places || live ? i : t.N - 1;
  const int deg = !places && live ? t.eup[i + 1] - t.eup[i] : 0;
  double Vi[5], xi[3] = {0.0, 0.0, 0.0}, gi[15];
  load_state<kFromVil>(Lay<SH>(), V, ii, Vi);
  if (SECOND || LM) load_x(Lay<SH>(), t, ii, xi);
  if (SECOND) load_il<15>(Lay<SH>(), grad, ii, gi);
  double p[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
  for (int kk = ALL ? kb : w; kk < (ALL ? ke : w + 1); ++kk) {
    const bool act = places ? live : kk - kb < deg;
    const int pos = places ? at : t.up.koff[kk] + lanes_below(act);
    if (!act) continue;
    const int j = t.up.idx[pos];
    double Vj[5], xj[3] = {0.0, 0.0, 0.0}, gj[15];
    load_state<kFromVil>(Lay<SH>(), V, j, Vj);
    if (SECOND || LM) load_x(Lay<SH>(), t, j, xj);
    if (SECOND) load_il<15>(Lay<SH>(), grad, j, gj);
    double nv[3];
    stream_load<3, ALL>(Lay<SH>(), t.pnormal, pos, nv);
    double f[5];
    bool bi, bj;
    edge_flux<SECOND, LM>(fc, Vi, xi, gi, Vj, xj, gj, nv, f, bi, bj);
    if (bi || bj) {
      atomicAdd(err, (int)bi + (int)bj);
      if (tag0) {  // with the failsafe the failing sides are tagged
        if (bi) tag0[i] = 1;
        if (bj) tag0[j] = 1;
      }
    }
    stream_store<5, ALL>(Lay<SH>(), Fm, pos, f);
#pragma unroll
    for (int k = 0; k < 5; ++k) p[k] += f[k];
  }
  if (ALL && live) store_il<5>(Lay<SH>(), P, i, p);
}

__global__ __launch_bounds__(kBlock) void k_face_flux(DevTables t, const double *__restrict__ V, FluxConsts fc,
                                                      double *__restrict__ Ff, const int *__restrict__ done) {
  if (done && *done) return;
  const int q = blockIdx.x * kBlock + (int)threadIdx.x;
  if (q < 3 * t.F) {
    if (t.sh) face_slot_flux<kGroupShift>(t, V, fc, q, Ff);
    else face_slot_flux<0>(t, V, fc, q, Ff);
  }
}

// ---------------------------------------------------------------------------
// 1'. gradients with the strip's node data staged in LDS.  A block covers a
//     strip of consecutive nodes [n0, n1) (one lane each); every node the
//     strip touches (the strip and all neighbours, ascending ids) is loaded
//     once: consecutive lanes take consecutive staged nodes, so the loads
//     coalesce, and U -> V is converted once per staged node instead of once
//     per adjacency entry.  The sums are the per-lane kernel's, term for term.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(kGradStrip) void k_gradients_staged(DevTables t, const double *__restrict__ U, Gas gas,
                                                                 double *__restrict__ Vout,
                                                                 double *__restrict__ grad, int *__restrict__ err,
                                                                 const int *__restrict__ done) {
  if (done && *done) return;
  __shared__ double sv[8 * kGradHalo];  // field f of staged node h at sv[f * kGradHalo + h]: V (5), X (3)
  const int b = xcd_chunk(blockIdx.x, t.ngb);
  const int4 s = t.gb4[b];
  const int tid = threadIdx.x;
  if (err && blockIdx.x == 0 && tid == 0) *err = 0;  // the flux pass follows in stream order
  const int H = s.w - s.z;
  // every staged node's loads are issued before any is used: one memory
  // latency per block instead of one per staged node
  constexpr int PER = (kGradHalo + kGradStrip - 1) / kGradStrip;
  double u[PER][5];
  double4 x[PER];
#pragma unroll
  for (int r = 0; r < PER; ++r) {
    const int h = tid + r * kGradStrip;
    const int g = h < H ? t.ghalo[s.z + h] : t.ghalo[s.z];
#pragma unroll
    for (int k = 0; k < 5; ++k) u[r][k] = U[5 * (size_t)g + k];
    x[r] = *reinterpret_cast<const double4 *>(t.X4 + 4 * (size_t)g);
  }
#pragma unroll
  for (int r = 0; r < PER; ++r) {
    const int h = tid + r * kGradStrip;
    if (h < H) {
      double v[5];
      prim_from_cons(u[r], gas, v);
#pragma unroll
      for (int k = 0; k < 5; ++k) sv[k * kGradHalo + h] = v[k];
      sv[5 * kGradHalo + h] = x[r].x;
      sv[6 * kGradHalo + h] = x[r].y;
      sv[7 * kGradHalo + h] = x[r].z;
    }
  }
  __syncthreads();
  const int n = s.x + tid;
  if (n >= s.y) return;
  const int hn = t.gown[b] + tid;
  double Vn[5];
#pragma unroll
  for (int k = 0; k < 5; ++k) {
    Vn[k] = sv[k * kGradHalo + hn];
    Vout[il<5>(t.sh, n, k)] = Vn[k];
  }
  const double xn[3] = {sv[5 * kGradHalo + hn], sv[6 * kGradHalo + hn], sv[7 * kGradHalo + hn]};
  double L[6], acc[15];
  load_lsq(t, n, L);
#pragma unroll
  for (int q = 0; q < 15; ++q) acc[q] = 0.0;
  const int e0 = t.rowptr[n], e1 = t.rowptr[n + 1];
  for (int e = e0; e < e1; ++e) {
    const int hm = t.gloc[e];
    const double xm[3] = {sv[5 * kGradHalo + hm], sv[6 * kGradHalo + hm], sv[7 * kGradHalo + hm]};
    double Vm[5];
#pragma unroll
    for (int q = 0; q < 5; ++q) Vm[q] = sv[q * kGradHalo + hm];
    lsq_add(L, xm, xn, Vm, Vn, acc);
  }
  store_il<15>(t.sh, grad, n, acc);
}

// ---------------------------------------------------------------------------
// 2'. edge fluxes with the strip's node data staged in LDS.  A block covers
//     the edges of consecutive rows (lower nodes) [r0, r1); the rows and the
//     upper ends of their edges (ascending ids) are loaded once, consecutive
//     lanes taking consecutive fields of a node.  With plain records those
//     are consecutive doubles; in the interleaved layout a field's pair lies
//     in a plane of its own, so a load touches a line per two fields and the
//     lines are shared by the lanes of neighbouring nodes.  Lane k computes
//     edge l0 + k from LDS exactly as the per-lane kernel does; the fluxes go
//     through the same LDS for the per-row sums P.  Boundary faces take a
//     launch of their own (k_face_flux).  An option, not the default: it
//     measures 158 us a second-order residual at 275k nodes and 1155 at 2.1M,
//     against 131 and 923 of the passes above (on plain records 182 and 1236).
// ---------------------------------------------------------------------------
template <bool SECOND>
__global__ __launch_bounds__(kFluxStrip) void k_flux_staged(DevTables t, const double *__restrict__ V,
                                                            const double *__restrict__ grad, FluxConsts fc,
                                                            double *__restrict__ Fm, double *__restrict__ P,
                                                            int *__restrict__ err, const int *__restrict__ done) {
  if (done && *done) return;
  // staged node h: record sh[h * NF ...] = V (5), X (3), gradients (15); the
  // odd record length spreads the lanes' reads of random records over the
  // LDS banks, and consecutive lanes staging one record write consecutive
  // addresses
  constexpr int NF = SECOND ? 23 : 5;
  constexpr int HS = kFluxHalo;
  constexpr int FS = kFluxStrip + 1;
  // the flux staging [5][FS] reuses the node staging [HS][NF]
  __shared__ double sh[NF * HS > 5 * FS ? NF * HS : 5 * FS];
  __shared__ int sidx[HS];
  const int b = xcd_chunk(blockIdx.x, t.nfb);
  const int4 ch = t.fb4[b];
  const int2 hr = t.fbh[b];
  const int r0 = ch.x, r1 = ch.y, l0 = ch.z, l1 = ch.w;
  const int H = hr.y - hr.x;
  const int tid = threadIdx.x;
  for (int h = tid; h < H; h += kFluxStrip) sidx[h] = t.fhalo[hr.x + h];
  __syncthreads();
  // all of a lane's staging loads are in flight together (consecutive lanes on
  // consecutive fields: V 5, X 3 of 4, gradients 15 of 16), so a block waits
  // one memory latency
  constexpr int PV = (5 * HS + kFluxStrip - 1) / kFluxStrip;
  constexpr int PX = (4 * HS + kFluxStrip - 1) / kFluxStrip;
  constexpr int PG = (16 * HS + kFluxStrip - 1) / kFluxStrip;
  double rv[PV], rx[SECOND ? PX : 1], rg[SECOND ? PG : 1];
#pragma unroll
  for (int r = 0; r < PV; ++r) {
    const int q = tid + r * kFluxStrip;
    const int h = q / 5, f = q - 5 * h;
    rv[r] = q < 5 * H ? V[il<5>(t.sh, sidx[min(h, H - 1)], f)] : 0.0;
  }
  if (SECOND) {
#pragma unroll
    for (int r = 0; r < PX; ++r) {
      const int q = tid + r * kFluxStrip;
      rx[r] = q < 4 * H ? t.X4[4 * (size_t)sidx[min(q >> 2, H - 1)] + (q & 3)] : 0.0;
    }
#pragma unroll
    for (int r = 0; r < PG; ++r) {
      const int q = tid + r * kFluxStrip;
      rg[r] = q < 16 * H && (q & 15) < 15 ? grad[il<15>(t.sh, sidx[min(q >> 4, H - 1)], q & 15)] : 0.0;
    }
  }
#pragma unroll
  for (int r = 0; r < PV; ++r) {
    const int q = tid + r * kFluxStrip;
    const int h = q / 5, f = q - 5 * h;
    if (q < 5 * H) sh[h * NF + f] = rv[r];
  }
  if (SECOND) {
#pragma unroll
    for (int r = 0; r < PX; ++r) {
      const int q = tid + r * kFluxStrip;
      if (q < 4 * H && (q & 3) < 3) sh[(q >> 2) * NF + 5 + (q & 3)] = rx[r];
    }
#pragma unroll
    for (int r = 0; r < PG; ++r) {
      const int q = tid + r * kFluxStrip;
      if (q < 16 * H && (q & 15) < 15) sh[(q >> 4) * NF + 8 + (q & 15)] = rg[r];
    }
  }
  __syncthreads();
  const int ne = l1 - l0;
  double f[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
  if (tid < ne) {
    const int l = l0 + tid;
    const uint32_t loc = t.floc[l];
    const double *si = sh + (int)(loc & 0xffffu) * NF, *sj = sh + (int)(loc >> 16) * NF;
    double Vi[5], Vj[5];
#pragma unroll
    for (int k = 0; k < 5; ++k) {
      Vi[k] = si[k];
      Vj[k] = sj[k];
    }
    double nv[3];
    load_il<3>(t.sh, t.pnormal, t.epos[l], nv);
    bool bi, bj;
    edge_flux<SECOND, false>(fc, Vi, si + 5, si + 8, Vj, sj + 5, sj + 8, nv, f, bi, bj);
    if (bi || bj) atomicAdd(err, (int)bi + (int)bj);
  }
  __syncthreads();  // the node staging is dead: reuse it for the fluxes
  double *sf = sh;
#pragma unroll
  for (int k = 0; k < 5; ++k) sf[k * FS + tid] = f[k];
  __syncthreads();
  if (tid < ne) store_il<5>(t.sh, Fm, t.epos[l0 + tid], f);
  const int nr = r1 - r0;
  for (int idx = tid; idx < nr * 5; idx += kFluxStrip) {
    const int rr = idx / 5, q = idx - 5 * rr;
    const int r = r0 + rr;
    const int eb = t.eup[r] - l0, eend = t.eup[r + 1] - l0;
    double s = 0.0;
    for (int e = eb; e < eend; ++e) s += sf[q * FS + e];
    P[il<5>(t.sh, r, q)] = s;
  }
}

// ---------------------------------------------------------------------------
// 3. node assembly: lower edges, upper-edge sum, faces, 1/V
// ---------------------------------------------------------------------------
// P null: the upper-edge sum is formed here from the edge fluxes, in edge
// order.  vg (or null): the node sums of the Navier-Stokes Galerkin
// contributions (momentum and energy), added before the 1/V scaling.
// host_err (or null): pinned copy of the error count of the finished flux
// pass, so a synchronous caller needs no copy of its own.
template <int SH>
__global__ __launch_bounds__(kBlock) void k_flux_nodes(DevTables t, const double *__restrict__ Fm,
                                                       const double *__restrict__ P, const double *__restrict__ Ff,
                                                       int scale, const double *__restrict__ vg,
                                                       const int *__restrict__ err, int *__restrict__ host_err,
                                                       double *__restrict__ R, const int *__restrict__ done) {
  if (done && *done) return;
  if (host_err && blockIdx.x == 0 && threadIdx.x == 0)
    __hip_atomic_store(host_err, *err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  const int sl = wave_slice(t);
  if (sl >= t.ns) return;
  const int lane = lane_id();
  const int n = sl * kWave + lane;
  const bool live = n < t.N;
  double s[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
  add_slots<true>(Lay<SH>(), t.lo, sl, live ? t.lrow[n + 1] - t.lrow[n] : 0, Fm, s);
  if (P) {
    if (live) {
      double p[5];
      load_il<5>(Lay<SH>(), P, n, p);
#pragma unroll
      for (int k = 0; k < 5; ++k) s[k] += p[k];
    }
  } else {
    double p[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
    add_slots<false>(Lay<SH>(), t.up, sl, live ? t.eup[n + 1] - t.eup[n] : 0, Fm, p);
#pragma unroll
    for (int k = 0; k < 5; ++k) s[k] += p[k];
  }
  if (!live) return;
  for (int q = t.frow[n]; q < t.frow[n + 1]; ++q)
#pragma unroll
    for (int k = 0; k < 5; ++k) s[k] += Ff[5 * (size_t)q + k];
  if (vg) {
    double g[4];
    load_il<4>(Lay<SH>(), vg, n, g);
#pragma unroll
    for (int k = 0; k < 4; ++k) s[1 + k] += g[k];
  }
  const double ic = t.invcv[n];
#pragma unroll
  for (int k = 0; k < 5; ++k) R[5 * (size_t)n + k] = scale ? s[k] * ic : s[k];
}

// V = V(U), as [N][5] (IL false) or interleaved; clears *err (or null)
template <bool IL>
__global__ __launch_bounds__(kBlock) void k_primitive(int N, int sh, const double *__restrict__ U, Gas g,
                                                      double *__restrict__ V, int *__restrict__ err,
                                                      const int *__restrict__ done) {
  if (done && *done) return;
  const int n = blockIdx.x * kBlock + threadIdx.x;
  if (err && n == 0) *err = 0;
  if (n >= N) return;
  double u[5], v[5];
#pragma unroll
  for (int k = 0; k < 5; ++k) u[k] = U[5 * (size_t)n + k];
  prim_from_cons(u, g, v);
#pragma unroll
  for (int k = 0; k < 5; ++k) V[IL ? il<5>(sh, n, k) : 5 * (size_t)n + k] = v[k];
}

__global__ void k_zero_int(int *p, int n, const int *done) {
  if (done && *done) return;
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0;
}

// ---------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------
// Slices from which a wave takes whole rows of edges and the streamed data
// bypass the caches; below, one edge per lane keeps more waves busy and the
// fluxes (40 B an edge) are still cached when the node pass reads them.  Flux
// and node pass, rows against edges: 106 / 104 us at 275k nodes (4291
// slices), 192 / 202 at 531k (8304), 672 / 757 at 2.1M.
constexpr int kRowWaveSlices = 6144;

static size_t halo_lds(const DevTables &t) { return 4 * sizeof(double2) * (size_t)t.halo_cap; }
// as many workgroups as fit all CUs (by LDS, and four by the registers)
static dim3 halo_grid(const DevTables &t) {
  const int fit = (int)std::max<size_t>(1, std::min<size_t>(4, kLdsPerCu / halo_lds(t)));
  return dim3((unsigned)std::min((t.ns + kNumXcd - 1) / kNumXcd * kNumXcd, kNumCu * fit));
}

template <bool SECOND, bool LM>
static void launch_flux_edges(aerofx_ctx *c, const ResidualBufs &b, bool all, const int *done) {
  const DevTables &t = c->tab;
  const int nfb = (3 * t.F + kBlock - 1) / kBlock;
  const dim3 grid(nfb + slice_grid(all ? t.ns : t.nup).x);
  if (grid.x == 0) return;
  const auto k = all    ? k_flux_edges<SECOND, LM, true, kGroupShift>
                 : t.sh ? k_flux_edges<SECOND, LM, false, kGroupShift>
                        : k_flux_edges<SECOND, LM, false, 0>;
  hipLaunchKernelGGL(k, grid, dim3(kBlock), 0, c->stream, t, nfb, b.V, b.grad, c->fc, b.Fm, b.P, c->d_Ff, c->d_err,
                     b.tag0, done);
}

int launch_residual_with(aerofx_ctx *c, const ResidualBufs &b, const double *U, double *R, bool scale,
                         const int *done, int *host_err) {
  const DevTables &t = c->tab;
  // the staged kernels evaluate Roe's flux only, without the failsafe
  const bool staged = t.ngb > 0 && c->residual_kernels == AEROFX_RESIDUAL_STAGED && !c->fc.low_mach && !c->failsafe;
  const bool rows = t.sh && row_waves(t.ns, kRowWaveSlices, c->max_degree);
  const bool all = staged || rows;  // P formed by the flux pass
  const dim3 ngrid((t.N + kBlock - 1) / kBlock), blk(kBlock);
  if (c->p.second_order) {
    ProfScope ps(c, AEROFX_TIMER_NODAL_GRAD);
    if (staged) {
      hipLaunchKernelGGL(k_gradients_staged, dim3(t.ngb), dim3(kGradStrip), 0, c->stream, t, U, c->gas, b.V,
                         b.grad, c->d_err, done);
    } else if (t.halo_cap) {
      hipLaunchKernelGGL(k_gradients_halo<kFromU>, halo_grid(t), dim3(kHaloThreads), halo_lds(t), c->stream, t, U, c->gas,
                         b.V, b.grad, c->d_err, done);
    } else {
      hipLaunchKernelGGL((k_gradients<kFromU, false>), slice_grid(t.ns), blk, 0, c->stream, t, U, c->gas, b.V,
                         b.grad, nullptr, nullptr, nullptr, c->d_err, done);
    }
  } else {
    hipLaunchKernelGGL(k_primitive<true>, ngrid, blk, 0, c->stream, t.N, t.sh, U, c->gas, b.V, c->d_err, done);
  }
  {
    ProfScope ps(c, AEROFX_TIMER_FV_TERM);
    if (staged) {
      if (t.F > 0)
        hipLaunchKernelGGL(k_face_flux, dim3((3 * t.F + kBlock - 1) / kBlock), blk, 0, c->stream, t, b.V, c->fc,
                           c->d_Ff, done);
      if (c->p.second_order)
        hipLaunchKernelGGL(k_flux_staged<true>, dim3(t.nfb), dim3(kFluxStrip), 0, c->stream, t, b.V, b.grad,
                           c->fc, b.Fm, b.P, c->d_err, done);
      else
        hipLaunchKernelGGL(k_flux_staged<false>, dim3(t.nfb), dim3(kFluxStrip), 0, c->stream, t, b.V, b.grad,
                           c->fc, b.Fm, b.P, c->d_err, done);
    } else if (c->p.second_order && c->fc.low_mach) {
      launch_flux_edges<true, true>(c, b, rows, done);
    } else if (c->p.second_order) {
      launch_flux_edges<true, false>(c, b, rows, done);
    } else if (c->fc.low_mach) {
      launch_flux_edges<false, true>(c, b, rows, done);
    } else {
      launch_flux_edges<false, false>(c, b, rows, done);
    }
  }
  // the Navier-Stokes Galerkin term (SpaceOperator.C:570-573): its element
  // pass and node sums, added by the node pass (or, without the contribution
  // buffer, the per-node kernel after it)
  const bool fold = c->viscous && c->d_visc_c;
  if (fold) {
    int rc = launch_visc_elements(c, b.V, done);
    if (rc || (rc = launch_visc_sum(c, done))) return rc;
  }
  {
    ProfScope ps(c, AEROFX_TIMER_FV_NODES);
    hipLaunchKernelGGL(t.sh ? k_flux_nodes<kGroupShift> : k_flux_nodes<0>, slice_grid(t.ns), blk, 0, c->stream, t,
                       b.Fm, all ? b.P : nullptr, c->d_Ff, scale ? 1 : 0, fold ? c->d_visc_g : nullptr, c->d_err,
                       host_err, R, done);
  }
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return set_hip_error(e, "residual launch");
  return fold ? 0 : launch_visc_residual(c, b.V, R, scale, done);
}

int launch_residual(aerofx_ctx *c, const double *U, double *R, bool scale, const int *done) {
  const ResidualBufs b{c->d_V, c->d_grad, c->d_Fm, c->d_P};
  return launch_residual_with(c, b, U, R, scale, done);
}

// SubDomain::finalizeTags (SubDomainCore.C:5177-5188) in its edge order: for
// each edge (i, j) tag1[i] = tag1[j] = tag0[i] + tag0[j], so a node keeps the
// value of its last edge (the last entry of its adjacency row, which is in
// edge order); then DistNodalGrad::fix (DistNodalGrad.C:1265-1284): the node
// is first order from now on if tag1 is set.
__global__ void k_fs_finalize(DevTables t, const int *__restrict__ tag0, int *__restrict__ tag1,
                              int *__restrict__ mask) {
  const int n = blockIdx.x * kBlock + threadIdx.x;
  if (n >= t.N) return;
  const int e0 = t.rowptr[n], e1 = t.rowptr[n + 1];
  if (e1 > e0) tag1[n] = tag0[n] + tag0[t.adj[e1 - 1]];
  if (tag1[n]) mask[n] = 1;
}

// the count that the residual's node pass left in h_err[0]
static int read_error_count(aerofx_ctx *c, int *count) {
  hipError_t e = hipStreamSynchronize(c->stream);
  if (e != hipSuccess) return set_hip_error(e, "residual error count");
  *count = c->h_err[0];
  return 0;
}

int residual_failsafe(aerofx_ctx *c, const ResidualBufs &b, const double *U, double *R, bool scale, int *count) {
  const bool fs = c->failsafe && c->p.second_order;
  ResidualBufs b1 = b;
  const int N = c->N;
  b1.tag0 = fs ? c->d_fs : nullptr;
  int rc = launch_residual_with(c, b1, U, R, scale, nullptr, c->h_err);
  if (rc || (rc = read_error_count(c, count))) return rc;
  if (!fs || *count == 0) return 0;
  // Domain::computeFiniteVolumeTerm with failsafe (Domain.C:884-917)
  hipLaunchKernelGGL(k_fs_finalize, dim3((N + kBlock - 1) / kBlock), dim3(kBlock), 0, c->stream, c->tab, c->d_fs,
                     c->d_fs + N, c->d_fs + 2 * (size_t)N);
  c->fs_any = true;
  if ((rc = launch_residual_with(c, b, U, R, scale, nullptr, c->h_err)) || (rc = read_error_count(c, count))) return rc;
  // FailSafe = On clears the tags after the fix; AlwaysOn keeps them
  if (c->failsafe == 1) hipLaunchKernelGGL(k_zero_int, dim3((2 * N + 63) / 64), dim3(64), 0, c->stream, c->d_fs,
                                           2 * N, nullptr);
  hipError_t e = hipGetLastError();
  return e == hipSuccess ? 0 : set_hip_error(e, "failsafe launch");
}

int refuse_failsafe_nodes(aerofx_ctx *c, const char *who) {
  if (!c->fs_any) return 0;
  return set_error(AEROFX_ERR_STATE, std::string(who) +
                                         ": failsafe first-order nodes are set (aerofx_ctx_reset_failsafe clears them)");
}

int launch_gradients_il(aerofx_ctx *c, const double *W, double *grad, const int *done) {
  const DevTables &t = c->tab;
  if (t.halo_cap)
    hipLaunchKernelGGL(k_gradients_halo<kFromVil>, halo_grid(t), dim3(kHaloThreads), halo_lds(t), c->stream, t, W,
                       c->gas, nullptr, grad, nullptr, done);
  else
    hipLaunchKernelGGL((k_gradients<kFromVil, false>), slice_grid(t.ns), dim3(kBlock), 0, c->stream, t, W, c->gas,
                       nullptr, grad, nullptr, nullptr, nullptr, nullptr, done);
  hipError_t e = hipGetLastError();
  return e == hipSuccess ? 0 : set_hip_error(e, "gradients launch");
}

int launch_gradients_v(aerofx_ctx *c, const double *V, double *ddx, double *ddy, double *ddz) {
  hipLaunchKernelGGL((k_gradients<kFromV, true>), slice_grid(c->tab.ns), dim3(kBlock), 0, c->stream, c->tab, V,
                     c->gas, nullptr, nullptr, ddx, ddy, ddz, nullptr, nullptr);
  hipError_t e = hipGetLastError();
  return e == hipSuccess ? 0 : set_hip_error(e, "gradients launch");
}

int launch_primitive(aerofx_ctx *c, const double *U, double *V) {
  hipLaunchKernelGGL(k_primitive<false>, dim3((c->N + kBlock - 1) / kBlock), dim3(kBlock), 0, c->stream, c->N, c->tab.sh,
                     U, c->gas, V, nullptr, nullptr);
  hipError_t e = hipGetLastError();
  return e == hipSuccess ? 0 : set_hip_error(e, "primitive launch");
}

int launch_primitive_il(aerofx_ctx *c, const double *U) {
  hipLaunchKernelGGL(k_primitive<true>, dim3((c->N + kBlock - 1) / kBlock), dim3(kBlock), 0, c->stream, c->N, c->tab.sh,
                     U, c->gas, c->d_V, nullptr, nullptr);
  hipError_t e = hipGetLastError();
  return e == hipSuccess ? 0 : set_hip_error(e, "primitive launch");
}

}  // namespace aerofx
