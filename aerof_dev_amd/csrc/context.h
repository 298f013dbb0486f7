// context.h -- the per-mesh context behind the C ABI (internal).
#pragma once
#include <hip/hip_runtime.h>

#include <functional>
#include <string>
#include <vector>

#include "aerofx.h"
#include "device_physics.h"
#include "device_viscous.h"

namespace aerofx {

constexpr int kBlock = 256;       // threads per block of the edge/entry kernels
constexpr int kMaxRows = 64;      // node rows per block (LDS staging bound)
constexpr int kNumXcd = 8;        // MI355X: 8 XCDs, blocks dealt round-robin
constexpr int kNumCu = 256;
constexpr size_t kLdsPerCu = 160 * 1024;
constexpr int kPad = kBlock + 1;  // LDS row stride (odd: conflict-free)
// LDS-staged residual passes: strips of consecutive nodes (gradients) or
// rows (fluxes) whose touched nodes are loaded into LDS once per block.
//   gradient strip: <= kGradStrip nodes (one lane each), <= kGradHalo staged
//                   nodes of 8 doubles (V, X): 61,440 B of LDS
//   flux strip:     <= kFluxStrip edges (one lane each), <= kFluxHalo staged
//                   nodes of 23 doubles (V, X, gradients): 35,328 B of LDS
constexpr int kGradStrip = 128;
constexpr int kGradHalo = 960;
constexpr int kFluxStrip = 256;
constexpr int kFluxHalo = 192;

// Faces of every wall code take the wall flux (FluxFcn.h:270-276): slip,
// adiabatic and isothermal walls, fixed or moving.
__host__ __device__ inline bool is_wall_code(int code) {
  const int a = code < 0 ? -code : code;
  return a == AEROFX_BC_SLIP_WALL || a == AEROFX_BC_ADIABATIC_WALL || a == AEROFX_BC_ISOTHERMAL_WALL;
}

// Block b of a launch runs on XCD b % 8; remap so that each XCD sweeps one
// contiguous range of chunks (its L2 then holds that range's neighbours).
__device__ __forceinline__ int xcd_chunk(int b, int nchunks) {
  const int q = nchunks / kNumXcd, r = nchunks % kNumXcd;
  const int x = b % kNumXcd, k = b / kNumXcd;
  return x * q + min(x, r) + k;
}

// 5x5 block storage interleaved in groups of 64 blocks: element q of block e
// at (e / 64) * 1600 + q * 64 + e % 64, so that 64 lanes reading element q of
// 64 consecutive blocks touch one contiguous 512 B (FP64) segment.
__host__ __device__ inline size_t blk64_base(size_t e) { return (e >> 6) * (64 * 25) + (e & 63); }
constexpr int kBlkStride = 64;
inline size_t blk64_count(size_t nblocks) { return (nblocks + 63) / 64 * 64 * 25; }

// Node and edge data of W doubles per item that the passes gather (primitive
// state, gradients, coordinates, fluxes): groups of 64 items, the fields of a
// group in planes of two (the last of an odd W alone), so a lane loads 16 B
// and 64 lanes reading neighbouring items touch a contiguous piece of each
// plane.  The vector cache takes one access per clock, each up to 64 B of four
// consecutive lanes: with records of 40 to 128 B a gather costs 43 to 64
// accesses per load and wave, which took 85 % of the flux pass's clocks; from
// the planes it takes about 28 over the neighbours of 64 consecutive nodes in
// RCM order (flux and node pass at 2.1M nodes 864 -> 727 us).
// The groups have 1 << sh items: 64 (sh = kGroupShift), or one (sh = 0), plain
// records, 15 and 3 fields padded to whole lines, where the numbering scatters
// a node's neighbours: the planes of an item that no lane beside reads cost a
// line each (DevTables::sh).  The passes that gather most are instantiated for
// either, the others read the shift.
constexpr int kGroupShift = 6;
// One layout fixed at compile time (kGroupShift or 0), for the passes that are
// instantiated for each; where a layout is read from the tables it is the int.
template <int SH>
struct Lay {};
typedef double double2u __attribute__((ext_vector_type(2), aligned(8)));  // 16-byte access at 8-byte alignment
template <int W>
constexpr int record_size() {
  return W == 15 ? 16 : (W == 3 ? 4 : W);
}
template <int W>
__host__ __device__ __forceinline__ size_t il_group(int sh, size_t n) {
  return (n >> sh) * (sh ? 64 * W : record_size<W>());
}
template <int W>
__host__ __device__ __forceinline__ size_t il(int sh, size_t n, int k) {
  const size_t g = il_group<W>(sh, n), l = n & ((1u << sh) - 1);
  return k < (W & ~1) ? g + ((size_t)(k >> 1) << (sh + 1)) + 2 * l + (k & 1) : g + ((size_t)(W - 1) << sh) + l;
}
template <int W>
inline size_t il_count(int sh, size_t n) {
  return sh ? (n + 63) / 64 * 64 * W : n * record_size<W>();
}
template <int W>
__device__ __forceinline__ void load_il(int sh, const double *__restrict__ p, int n, double v[W]) {
  const double *q = p + il_group<W>(sh, n);
  const int l = n & ((1 << sh) - 1);
#pragma unroll
  for (int k = 0; k < W / 2; ++k) {
    const double2u a = *reinterpret_cast<const double2u *>(q + (k << (sh + 1)) + 2 * l);
    v[2 * k] = a.x;
    v[2 * k + 1] = a.y;
  }
  if (W & 1) v[W - 1] = q[((W - 1) << sh) + l];
}
template <int W>
__device__ __forceinline__ void store_il(int sh, double *__restrict__ p, int n, const double v[W]) {
  double *q = p + il_group<W>(sh, n);
  const int l = n & ((1 << sh) - 1);
#pragma unroll
  for (int k = 0; k < W / 2; ++k) {
    const double2u a = {v[2 * k], v[2 * k + 1]};
    *reinterpret_cast<double2u *>(q + (k << (sh + 1)) + 2 * l) = a;
  }
  if (W & 1) q[((W - 1) << sh) + l] = v[W - 1];
}

template <int W, int SH>
__device__ __forceinline__ void load_il(Lay<SH>, const double *__restrict__ p, int n, double v[W]) {
  if constexpr (SH == 0) return load_il<W>(0, p, n, v);
  const double *q = p + ((size_t)n >> 6) * (64 * W);
  const int l = n & 63;
#pragma unroll
  for (int k = 0; k < W / 2; ++k) {
    const double2 a = *reinterpret_cast<const double2 *>(q + k * 128 + 2 * l);
    v[2 * k] = a.x;
    v[2 * k + 1] = a.y;
  }
  if (W & 1) v[W - 1] = q[(W - 1) * 64 + l];
}
template <int W, int SH>
__device__ __forceinline__ void store_il(Lay<SH>, double *__restrict__ p, int n, const double v[W]) {
  if constexpr (SH == 0) return store_il<W>(0, p, n, v);
  double *q = p + ((size_t)n >> 6) * (64 * W);
  const int l = n & 63;
#pragma unroll
  for (int k = 0; k < W / 2; ++k) *reinterpret_cast<double2 *>(q + k * 128 + 2 * l) = make_double2(v[2 * k], v[2 * k + 1]);
  if (W & 1) q[(W - 1) * 64 + l] = v[W - 1];
}

// Rows of a CSR table regrouped for one wave per 64 consecutive rows (a
// slice): entry k of all rows of slice s that have one, consecutively from
// koff[kptr[s] + k], in row order.  Lane r finds its entry by counting the
// lanes below it that have one, so nothing is padded whatever the degrees.
struct RowSlices {
  const int *kptr;  // [slices + 1] first (slice, k) pair of each slice
  const int *koff;  // per (slice, k): its first entry
  const int *idx;   // the entries
};

__device__ __forceinline__ int lanes_below(bool active) {
  const unsigned long long b = __ballot(active);
  return __builtin_amdgcn_mbcnt_hi((unsigned)(b >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)b, 0u));
}

// 64 B of LDS per halo node: 512 nodes (about a slice's in RCM or row order)
// leave room for five workgroups per CU, of which registers let four run
constexpr int kHaloCap = 1024;
constexpr int kHaloRow = 64;  // bounds the padding of the places

// Device-resident mesh tables.  All arrays are laid out for the kernel that
// streams them: contiguous per node row or per edge.
struct DevTables {
  int N, E, F;
  int ns;                // 64-node slices
  int sh;                // group size of the interleaved arrays, 1 << sh items
  const double *X4;      // [N][4] coordinates padded to 32 B
  const double *X3;      // il<3>: coordinates
  const int *fs_mask;    // [N] failsafe first-order nodes (gradients zeroed), or null
  const double *lsq6;    // [N][6] (1/r11, 1/r22, 1/r33, r12/r11, r23/r22, psi)
  const double *invcv;   // [N] 1/ctrlVol
  const double *cv;      // [N] ctrlVol
  // gradient pass: node adjacency, rows sorted ascending (= edge-id order)
  int ngchunks;
  const int *gchunk;     // [ngchunks+1] row starts; a row of more than kBlock entries is a chunk alone
  int nglong;
  const int *glong;      // [nglong] the rows of more than kBlock entries
  const int *rowptr;     // [N+1]
  const int *adj;        // [2E]
  const int *eidx;       // [2E] edge id of each adjacency entry
  const int *mirror;     // [2E] entry (m, n) of the entry (n, m)
  // residual passes: all neighbours, upper neighbours (the edge storage order
  // of the flux pass: an edge's position is its place in up.idx) and, per
  // lower neighbour, the position of that edge
  RowSlices nb, up, lo;
  // gradient pass through LDS: the different neighbours of each slice
  // (halo_cap per slice, in the order its entries first name them, the last
  // repeated), and the places among them of the entries 2 p (low half) and
  // 2 p + 1 of row r of a slice at [(slice * halo_pairs + p) * 64 + r];
  // halo_cap = 0: a slice has more than kHaloCap or a row more than kHaloRow,
  // the pass gathers per entry
  int halo_cap, halo_pairs;
  const int *halo;
  const uint32_t *hloc;
  int nup;               // waves of the passes by entries: (slice, k) pairs of up, or with records 64 edges each
  const int *upslice;    // [nup] the pairs' slices (with records null)
  const int *uprow;      // [E] row of each position (with records, else null)
  const int *pedge;      // [E] edge id at each position
  const double *pnormal; // il<3> over positions: dual-face area vectors
  const int *eup;        // [N+1] first edge whose lower node is i
  const int2 *eij;       // [E] edge endpoints (i, j), i < j

  const double *normal;  // [E][3] dual-face area vector oriented i -> j
  // flux pass B: per node, lower-edge slots and boundary faces
  const int *lrow;       // [N+1] lower-list pointers
  const int *ledge;      // [E] edges (m, n), m < n, of node n, ascending m
  const int *frow;       // [N+1] face-list pointers
  const int *fidx;       // [3F] faces touching each node, ascending
  const int *fnode;      // [3F] node of each face slot
  const int *fcode;      // [F] boundary code
  const double *fnorm3;  // [F][3] (1/3) face normal
  const double *fnorm;   // [F][3] face normal
  // LDS-staged passes (ngb == 0: the mesh does not fit, per-lane kernels run)
  int ngb;               // gradient strips
  const int4 *gb4;       // [ngb] (first node, end node, first halo entry, end halo entry)
  const int *gown;       // [ngb] halo position of the strip's first node
  const int *ghalo;      // staged node ids, ascending within each strip
  const uint16_t *gloc;  // [2E] halo position of each adjacency entry's neighbour
  int nfb;               // flux strips
  const int4 *fb4;       // [nfb] (first row, end row, first edge, end edge)
  const int2 *fbh;       // [nfb] (first halo entry, end halo entry)
  const int *fhalo;      // staged node ids, ascending within each strip
  const uint32_t *floc;  // [E] halo position of i | halo position of j << 16
  const int *epos;       // [E] position of each edge in the flux storage
};

constexpr int kWave = 64;
__device__ __forceinline__ int lane_id() { return (int)threadIdx.x & (kWave - 1); }
// slice of this wave: blocks of four slices, one contiguous range per XCD
__device__ __forceinline__ int wave_slice(const DevTables &t) {
  const int nb = (t.ns + kBlock / kWave - 1) / (kBlock / kWave);
  return xcd_chunk(blockIdx.x, nb) * (kBlock / kWave) + (int)(threadIdx.x / kWave);
}
// Whole rows of edges per wave (flux and adjoint edge passes): from `from`
// slices on, unless a node has so many neighbours that the pass waits for the
// lane that takes its row.  An edge there costs some 1.5 us (flux), 3 us
// (adjoint).  By rows and by entries, one node of 31 / 47 / 60 neighbours beside
// 456k nodes: flux and node pass with the gradients 246 / 276 / 311 and 238 / 249
// / 263 us, (dR/dU)^T 793 / 882 / 960 and 820 / 842 / 868; 47 / 100 / 127 / 200
// beside 2.1M nodes: 957 / 1014 / 1067 / 1210 and 999 / 989 / 1010 / 1059, 2938 /
// 3192 / 3382 / 3837 and 3293 / 3337 / 3383 / 3531.
inline bool row_waves(int ns, int from, int max_degree) {
  return ns >= from && max_degree <= (ns / 384 > 32 ? ns / 384 : 32);
}
// The edge of this lane in wave w of a pass by entries (t.nup waves): row, place
// in the edge storage and whether there is one.  A wave takes the k-th upper edges
// of a slice; with records (SH = 0) 64 consecutive places, since a scattered
// numbering leaves half of a slice's k-th places empty (its nodes have from 0 to
// all neighbours above them).
struct UpperEntry {
  int i = 0, pos = 0;
  bool act = false;
};
template <int SH>
__device__ __forceinline__ UpperEntry upper_entry(const DevTables &t, int w) {
  UpperEntry u;
  if (SH == 0) {
    const int at = w * kWave + lane_id();
    u.act = at < t.E;
    u.pos = u.act ? at : t.E - 1;
    u.i = t.uprow[u.pos];
  } else {
    const int sl = t.upslice[w];
    u.i = sl * kWave + lane_id();
    u.act = u.i < t.N && w - t.up.kptr[sl] < t.eup[min(u.i, t.N - 1) + 1] - t.eup[min(u.i, t.N - 1)];
    u.pos = t.up.koff[w] + lanes_below(u.act);
  }
  return u;
}
inline dim3 slice_grid(int ns) { return dim3((unsigned)((ns + kBlock / kWave - 1) / (kBlock / kWave))); }

// the passes' streamed data of large meshes: past the caches, which then keep
// the gathered node data (flux pass at 2.1M nodes 492 -> 468 us, the node pass
// after it 212 -> 205; at 275k nodes the fluxes would miss the cache instead:
// 106 -> 109 us)
typedef double nt_double2 __attribute__((ext_vector_type(2)));
template <int W, bool NT, int SH>
__device__ __forceinline__ void stream_load(Lay<SH> lay, const double *__restrict__ p, int n, double v[W]) {
  static_assert(!NT || SH == kGroupShift, "records share lines between stores");
  if (!NT) return load_il<W>(lay, p, n, v);
  const double *q = p + ((size_t)n >> 6) * (64 * W);
  const int l = n & 63;
#pragma unroll
  for (int k = 0; k < W / 2; ++k) {
    const nt_double2 a = __builtin_nontemporal_load(reinterpret_cast<const nt_double2 *>(q + k * 128 + 2 * l));
    v[2 * k] = a.x;
    v[2 * k + 1] = a.y;
  }
  if (W & 1) v[W - 1] = __builtin_nontemporal_load(q + (W - 1) * 64 + l);
}
template <int W, bool NT, int SH>
__device__ __forceinline__ void stream_store(Lay<SH> lay, double *__restrict__ p, int n, const double v[W]) {
  static_assert(!NT || SH == kGroupShift, "records share lines between stores");
  if (!NT) return store_il<W>(lay, p, n, v);
  double *q = p + ((size_t)n >> 6) * (64 * W);
  const int l = n & 63;
#pragma unroll
  for (int k = 0; k < W / 2; ++k) {
    const nt_double2 a = {v[2 * k], v[2 * k + 1]};
    __builtin_nontemporal_store(a, reinterpret_cast<nt_double2 *>(q + k * 128 + 2 * l));
  }
  if (W & 1) __builtin_nontemporal_store(v[W - 1], q + (W - 1) * 64 + l);
}

// s -= (LOWER: edge positions in rows.idx) or += (upper edges: the entries'
// own places) the fluxes of this lane's row, in row order; four entries'
// loads in flight together.
template <bool LOWER, int SH>
__device__ __forceinline__ void add_slots(Lay<SH> lay, const RowSlices &rows, int sl, int deg, const double *__restrict__ Fm,
                                          double s[5]) {
  constexpr int B = 4;
  const int kb = rows.kptr[sl], kn = rows.kptr[sl + 1] - kb;
  for (int k0 = 0; k0 < kn; k0 += B) {
    int pos[B];
#pragma unroll
    for (int u = 0; u < B; ++u) {
      const int off = k0 + u < kn ? rows.koff[kb + k0 + u] : 0;
      const bool act = k0 + u < deg;
      const int e = off + lanes_below(act);
      pos[u] = act ? (LOWER ? rows.idx[e] : e) : 0;
    }
    double v[B][5];
#pragma unroll
    for (int u = 0; u < B; ++u) load_il<5>(lay, Fm, pos[u], v[u]);
#pragma unroll
    for (int u = 0; u < B; ++u)
      if (k0 + u < deg) {
#pragma unroll
        for (int k = 0; k < 5; ++k) s[k] = LOWER ? s[k] - v[u][k] : s[k] + v[u][k];
      }
  }
}

struct FluxConsts {
  Gas gas;
  double beta;
  double ub_in[5], ub_out[5];
  int low_mach;  // 1: spatial low-Mach preconditioning (ROEFLUX5 and its ROEJAC6)
  LowMach lm;
};

int set_hip_error(hipError_t e, const char *what);
struct Krylov;
struct Adjoint;
struct BlockSolver;
struct Tangent;
struct Ilu;
struct FgWork;

// Element tables of the geometry derivatives (device copies, built on first
// use): the adjoint and the tangent passes sum per-element contributions per
// node or per edge in element order.
struct ElemTables {
  int *tets = nullptr;    // [T][4]
  int *faces = nullptr;   // [F][3]
  int *ntrow = nullptr;   // [N+1]
  int *ntslot = nullptr;  // [4T] 4 t + local vertex, ascending t per node
  int *nfslot = nullptr;  // [3F] 3 f + local vertex, in the order of DevTables::fidx
  int *etrow = nullptr;   // [E+1]
  int *etslot = nullptr;  // [6T] 6 t + local edge, ascending t per edge
};

}  // namespace aerofx

struct aerofx_ctx {
  int N = 0, T = 0, F = 0, E = 0;
  aerofx_params p{};
  aerofx::Gas gas{};
  aerofx::FluxConsts fc{};
  hipStream_t own_stream = nullptr, stream = nullptr;
  // host copies of the set-up tables
  std::vector<int> ptr;
  std::vector<double> cv, normals, fnorm, lsq;
  std::vector<int> tets, faces, tet_edges;  // element tables for the adjoint geometry terms
  std::vector<int> fcodes;                  // face codes
  // device
  aerofx::DevTables tab{};
  std::vector<void *> allocs;
  double *d_V = nullptr;     // il<5>: primitive state of the last residual
  double *d_grad = nullptr;  // il<15>: LSQ gradients, field d*5+k
  double *d_Fm = nullptr;    // il<5> over positions: edge fluxes
  double *d_P = nullptr;     // il<5>: per-node sums over upper edges
  double *d_Ff = nullptr;    // [3F][5] boundary-face fluxes, per node face slot
  int *d_err = nullptr;      // [0] reconstruction errors, [1] singular blocks, [2] bad states
  bool staged_tried = false;  // the staged family's tables were built, or do not fit
  int residual_kernels = AEROFX_RESIDUAL_PER_LANE;  // AEROFX_RESIDUAL_PER_LANE or _STAGED
  // Newton.FailSafe: 0 off, 1 on, 2 always on; d_fs [3N] = tag0, tag1, mask
  // (DistSVec<int,2> tag of Domain and the node tags of DistNodalGrad)
  int failsafe = 0;
  int *d_fs = nullptr;
  bool fs_any = false;  // some node is first order by the failsafe
  int check_final_res = 0;  // KspData checkFinalRes: GMRES reports -999 above its target
  int max_degree = 0;        // most neighbours of a node
  // laminar Navier-Stokes terms (viscous.hip): constants, node types, the
  // wall nodes (node, type) and the viscous time-step scratch
  int viscous = 0;
  aerofx::NsConsts ns{};
  std::vector<int> node_type;
  int nwall = 0, wall_cap = 0;
  int2 *d_wall = nullptr;
  double *d_idtv = nullptr;
  double *d_visc_c = nullptr;  // [4T][5] element contributions of the Galerkin term, in node-slot order
                               // (the residual's, whose density row is zero: [4T][4])
  double *d_visc_g = nullptr;  // il<4>: their node sums
  int *d_visc_chunk = nullptr; // row chunks of the Galerkin Jacobian pass; visc_chunks of them (0: a row is too long)
  int visc_chunks = 0;
  double *d_adj_tmp = nullptr;  // [N][5] the adjoint with the wall rows masked
  // viscous wall force: element of each face, per node the wall-face element
  // slots (4 f + k), per slot the derivatives [4F][5] / [4F][3]
  int *d_face_elem = nullptr, *d_nfe_row = nullptr, *d_nfe_slot = nullptr;
  double *d_force_u = nullptr, *d_force_x = nullptr;
  // the elements by their lowest node: vertices, and node-slot positions of the vertices
  int4 *d_visc_tets = nullptr, *d_visc_pos = nullptr;
  // device address of this GPU's static scratch array of
  // aerofx_residual_noalloc (looked up at ctx_create; null if that failed,
  // with the reason in noalloc_err)
  char *noalloc_scratch = nullptr;
  std::string noalloc_err;
  int *h_err = nullptr;
  // implicit operators (jacobian.hip) and Krylov workspace (krylov.hip)
  int jac_precision = -1;    // 0: FP64 blocks, 1: FP32 blocks
  void *d_jacD = nullptr, *d_jacB = nullptr, *d_jacDi = nullptr;  // current precision's
  void *jac_store[2][3] = {{nullptr, nullptr, nullptr}, {nullptr, nullptr, nullptr}};  // [precision][D, B, Di]
  long long jac_version = 0;  // bumped at every assembly
  // off-diagonal blocks in mirror order (slot e holds the block of the
  // mirror entry), so the transposed apply reads them as the forward one
  // does; rebuilt before transposed use when the assembly is newer
  void *jac_mirror[2] = {nullptr, nullptr};
  long long mirror_version = -1;
  int mirror_precision = -1;
  double *d_fjac = nullptr;    // [3F][25] boundary-face Jacobians, per node face slot
  // MatVecProd of aerofx_gmres and the Newton driver (AEROFX_MVP_*) and the
  // scratch of the finite-difference products, allocated on first use:
  // Q, Fa, Fb, F0 [5N] each, reduction partials [kDotBlocks], scalars [16]
  int mvp_type = AEROFX_MVP_H1, mvp_order = 1;
  const double *mvp_Q = nullptr, *mvp_F0 = nullptr, *mvp_dt = nullptr;
  double *d_fd = nullptr;
  double *d_dt = nullptr;
  aerofx::Krylov *ksp = nullptr;
  aerofx::Adjoint *adj = nullptr;
  aerofx::ElemTables *elem = nullptr;
  aerofx::Tangent *tan = nullptr;
  // preconditioner of the Krylov solves (AEROFX_PREC_*), taking effect at the
  // next Jacobian assembly; the RAS / ILU(0) subdomain size in nodes
  int prec_type = AEROFX_PREC_JACOBI;
  int prec_subdomain = 256;
  aerofx::Ilu *ilu = nullptr;
  aerofx::FgWork *fgm = nullptr;  // flexible GMRES workspace (fgmres.hip)
  aerofx::BlockSolver *blk = nullptr;
  int blk_tune = 0;  // autotuned waves per workgroup of the block update, 0: not yet
  // per-kernel timers (the reference's Timer buckets, Timer.h:12-15)
  bool prof = false;
  struct Pending {
    int bucket;
    hipEvent_t a, b;
  };
  std::vector<Pending> pending;
  std::vector<hipEvent_t> pool;
  double timer_ms[AEROFX_NUM_TIMERS] = {0};
  long long timer_n[AEROFX_NUM_TIMERS] = {0};
};

namespace aerofx {

// Brackets one kernel launch with events on the context stream when
// profiling is on.
struct ProfScope {
  aerofx_ctx *c;
  int bucket;
  hipEvent_t a = nullptr;
  ProfScope(aerofx_ctx *ctx, int b);
  ~ProfScope();
};

// device allocation owned by the context, and its early release
int ctx_alloc(aerofx_ctx *c, size_t bytes, void **out);
void ctx_release(aerofx_ctx *c, void *p);

__global__ void k_zero_int(int *p, int n, const int *done);

// laminar Navier-Stokes terms (viscous.hip), no-ops with the terms off:
// R += Galerkin term (/ V if scale); H1 += its blocks, then the wall
// conditions (U: the state, for isothermal walls); F's wall rows; the
// viscous time-step term (idtv = NULL when not used)
int launch_visc_residual(aerofx_ctx *c, const double *V, double *R, bool scale, const int *done);
// the element pass alone into the contribution buffer (the node pass of the
// residual sums it)
int launch_visc_elements(aerofx_ctx *c, const double *V, const int *done);
// their node sums into d_visc_g
int launch_visc_sum(aerofx_ctx *c, const int *done);
int launch_visc_jacobian(aerofx_ctx *c, const double *U, int precision);
int launch_bcs_residual(aerofx_ctx *c, const double *U, double *F, const int *done);
int launch_visc_idtv(aerofx_ctx *c, double **idtv);
// dR += (d Galerkin / dU) dU / V at the primitive state V; the wall rows of
// a product y = A p
int launch_visc_tangent(aerofx_ctx *c, const double *V, const double *dU, const double *dX, double *dR,
                        const int *done);
// the viscous wall force: Jf[f] += -(tau n_f) . dir on the wall faces (and
// the slot derivatives when derivs), then dJdU / dJdX += their node sums
int launch_visc_force(aerofx_ctx *c, const double dir[3], double *Jf, bool derivs);
int launch_visc_force_gather(aerofx_ctx *c, double *dJdU, double *dJdX);
// TX[t][12] += the Galerkin part of the element's coordinate adjoint
int launch_visc_adjoint_x(aerofx_ctx *c, const double *lam, double *TX);
int launch_bcs_product(aerofx_ctx *c, const double *U, const double *p, double *y, const int *done);
// Ub += (d Galerkin / dU)^T lam (the residual's 1/V included), at c->d_V
int launch_visc_adjoint(aerofx_ctx *c, const double *lam, double *Ub);
// the wall rows of the transposed Jacobian A^T psi = (dR/dU)^T P psi + B^T psi:
// pre: Ppsi = P psi; post: y += B^T psi
int launch_bcs_adjoint(aerofx_ctx *c, const double *U, const double *psi, double *Ppsi, double *y, bool pre);
// AEROFX_ERR_STATE when the Navier-Stokes terms are on
int refuse_viscous(aerofx_ctx *c, const char *who);

// residual passes (residual.hip); all enqueue on c->stream; every kernel
// returns at once when done != nullptr and *done != 0 (device-resident
// Krylov loops with a matrix-free operator)
int launch_residual(aerofx_ctx *c, const double *U, double *R, bool scale, const int *done = nullptr);
// the same passes with their scratch (primitive state V, gradients, edge
// fluxes Fm and upper-edge sums P, laid out as d_V, d_grad, d_Fm and d_P of
// the context) given explicitly; the error count still goes to c->d_err[0],
// and to host_err (pinned) when that is given
struct ResidualBufs {
  double *V, *grad, *Fm, *P;
  int *tag0 = nullptr;  // failsafe: sides of non-physical reconstructions are tagged here
};
// The residual with Newton.FailSafe (Domain.C:864-917): with the failsafe on
// and a non-physical reconstruction in the pass, the nodes are tagged
// (finalizeTags), their gradients zeroed from then on (DistNodalGrad::fix and
// limit) and the pass re-run.  Synchronises; *count = the non-physical
// reconstructions of the pass that stands.
int residual_failsafe(aerofx_ctx *c, const ResidualBufs &b, const double *U, double *R, bool scale, int *count);
// AEROFX_ERR_STATE while failsafe first-order nodes are set (the derivative
// passes differentiate the full second-order residual)
int refuse_failsafe_nodes(aerofx_ctx *c, const char *who);
int launch_residual_with(aerofx_ctx *c, const ResidualBufs &b, const double *U, double *R, bool scale,
                         const int *done = nullptr, int *host_err = nullptr);
// tables of the LDS-staged family, built when it is first selected
int ensure_staged(aerofx_ctx *c);
// LSQ gradients (il<15>) of a field laid out as d_V
int launch_gradients_il(aerofx_ctx *c, const double *W, double *grad, const int *done);
int launch_gradients_v(aerofx_ctx *c, const double *V, double *ddx, double *ddy, double *ddz);
int launch_primitive(aerofx_ctx *c, const double *U, double *V);  // V [N][5]
int launch_primitive_il(aerofx_ctx *c, const double *U);          // c->d_V

// implicit operators (jacobian.hip)
int launch_timestep(aerofx_ctx *c, double cfl, double *dt);
// U: the state of the wall conditions (needed with the Navier-Stokes terms)
int launch_jacobian(aerofx_ctx *c, const double *dt, int precision, const double *U = nullptr);
// trans: apply the transposed operator (adjoint solves)
int launch_h1_apply(aerofx_ctx *c, const double *p, double *y, bool trans = false);
// builds the mirrored off-diagonal blocks of the current assembly if they are
// older than it (enqueued on c->stream; call outside graph capture)
int ensure_mirror(aerofx_ctx *c);
int launch_prec_apply(aerofx_ctx *c, const double *y, double *x, bool trans = false);
// variants that return at once when *done != 0 (device-resident Krylov loops)
int launch_h1_apply_flag(aerofx_ctx *c, const double *p, double *y, const int *done, bool trans = false);
int launch_prec_apply_flag(aerofx_ctx *c, const double *y, double *x, const int *done, bool trans = false);
// V = (src - sum_{k < nsub} h_k Vb_k) * (*scale) then x = P V (the Arnoldi step's
// last Gram-Schmidt update and normalisation fused with the preconditioner)
int launch_prec_norm_flag(aerofx_ctx *c, const double *src, const double *scale, const double *Vb, size_t ldv,
                          int nsub, const double *h, double *V, double *x, const int *done, bool trans = false);
// Gram-Schmidt update pass of Arnoldi step j fused with the preconditioner
// (delayed reorthogonalisation; coefficients in coef, layout in krylov.hip)
constexpr int kMaxBasisCoef = 32;
int launch_dcgs_update(aerofx_ctx *c, double *V, size_t ldv, int j, const double *w, const double *coef,
                       const int *done, const int *jlast, double *x, bool trans);
void free_krylov(aerofx_ctx *c);
void free_adjoint(aerofx_ctx *c);
void free_tangent(aerofx_ctx *c);
// RAS / ILU(0) (ilu.hip): tables for subdomains of B nodes, numericILU of the
// current H1 (zero pivots counted in d_err[1]), and the solve x = M^-1 y
// (returning at once when done != nullptr and *done != 0)
void free_ilu(aerofx_ctx *c);
// flexible GMRES over nrhs right-hand sides rhs, x [nrhs][5N] (fgmres.hip):
// apply(x, y, nq): y_q = A x_q for q < nq; prec(v, z, nq, &inner): z_q ~
// M^-1 v_q (any, possibly varying, approximate inverse), adding its inner
// iterations.  Stops when every ||rhs_q - A x_q|| <= eps ||rhs_q|| or after
// max_outer steps; outer restart mo (<= 31).
struct FgOps {
  std::function<int(const double *, double *, int)> apply;
  std::function<int(const double *, double *, int, int *)> prec;
};
struct FgResult {
  int converged = 0, outer_its = 0, inner_its = 0;
  double res0 = 0.0, res = 0.0;  // the worst right-hand side: ||rhs||, ||rhs - A x||
};
int fgmres_solve(aerofx_ctx *c, int nrhs, const double *rhs, double *x, int mo, double eps, int max_outer,
                 const FgOps &ops, FgResult *res);
void free_fgmres(aerofx_ctx *c);
int ensure_ilu(aerofx_ctx *c, int B);
int launch_ilu_factor(aerofx_ctx *c);
int launch_ilu_solve(aerofx_ctx *c, const double *y, double *x, const int *done);
// c->elem (adjoint.hip)
int ensure_elem_tables(aerofx_ctx *c);
// dR = (dR/dU) dU + (dR/dX) dX at U (tangent.hip; dU, dX may be NULL),
// enqueued on c->stream; the forward residual it runs leaves R (raw flux
// sums) in the tangent workspace
int launch_tangent(aerofx_ctx *c, const double *U, const double *dU, const double *dX, double *dR);
// the exact product operator (tangent.hip): select keeps the forward pass at
// Q; apply gives y = (dR/dU) p + p / dt (dt may be NULL), every kernel
// returning at once when done != nullptr and *done != 0
int launch_h2_select(aerofx_ctx *c, const double *Q);
int launch_h2_apply(aerofx_ctx *c, const double *Q, const double *p, const double *dt, double *y,
                    const int *done);
// (dR/dU)^T lam -> Ub and/or (dR/dX)^T lam -> Xout (adjoint.hip), enqueued on c->stream
int launch_adjoint(aerofx_ctx *c, const double *U, const double *lam, double *Ub, double *Xout);
void free_block(aerofx_ctx *c);
// LINPACK inverse of FP32 5x5 blocks on a given stream (zero-pivot count in
// d_err[1], cleared first)
int launch_invert_f32(aerofx_ctx *c, hipStream_t stream, const float *D, float *Di);

}  // namespace aerofx
