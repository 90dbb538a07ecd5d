// Residual and Jacobian of the MPFA-O Richards path (subsystems (b), (c)).
//
//  k_cell_state   per cell: van Genuchten / Mualem / EOS state, rho, Kr/mu and their
//                 pressure derivatives, and the accumulation term (TS or SNES form)
//                 (TDyUpdateState_Richards_MPFAO, src/fv/mpfao/tdympfao.c:2527-2594;
//                  tdympfao_ts.c:191-212; tdympfao_snes.c:19-30, 112-123);
//                 per boundary face: P_bnd and Kr/mu on the boundary
//                 (tdympfao_utils.c:24-99, 690-759)
//  k_rows         per flux row (face*4 + subface): T.P from the vertex's columns,
//                 upwinded rho^2 kr/mu flux (TDyMPFAOIFunction_Vertices, tdympfao_ts.c:12-150);
//                 k_rows_general where a vertex has any number of columns
//  k_cell_gather  per cell: R = sum over its 6 faces x 4 subfaces (+/- by orientation)
//                 + accumulation
//  k_cell_jac     per cell, one pass: the Jacobian row from its 24 flux rows'
//                 derivatives (TDyMPFAOIJacobian_Vertices, 235-456) + the
//                 accumulation diagonal, optionally the residual as well
//
// Flux rows are stored face-major (row = face*4 + subface), the reference's
// Trans_mat row numbering; T is an 8-wide ELL block stored by pairs of columns
// (trans_index) so that consecutive lanes read consecutive 16-byte pairs.
#include "tdyhip_internal.h"
#include "tdyhip_math.h"

namespace tdyhip {

// Launch-time inputs that a replayed hipGraph must not freeze: when `dyn` is
// set, dtime = dyn[0] and shift = dyn[1] are read from device memory (the
// solver updates them between replays); when `stop` is set and nonzero the
// launch returns at once (the Newton solver's device-side gating).
struct StateParams {
  double vg_m, vg_alpha, x0, x1, dx, pref, dtime, shift;
  double c0, c1, c2, c3;
  int density_type, form;  // form: 0 TS, 1 SNES
  const double *dyn;
  const int *stop;
};

struct CellStateArgs {
  int nc;
  StateParams sp;
  const double *U, *Udot, *phi, *Sr, *vol, *accum_prev;
  FlowState *st;
  double *dM, *d2M, *acc;
};

__device__ inline void cell_state(const CellStateArgs &a, int c) {
  const StateParams &sp = a.sp;
  const double p = a.U[c];
  const double sr = a.Sr[c];
  double S, dS, d2S;
  vg_saturation(sp.vg_m, sp.vg_alpha, sr, sp.pref - p, S, dS, d2S);
  const double Se = (S - sr) / (1.0 - sr);
  double Kr, dKr;
  const double cc[4] = {sp.c0, sp.c1, sp.c2, sp.c3};
  mualem_kr(sp.vg_m, sp.x0, sp.x1, sp.dx, cc, Se, Kr, dKr);
  dKr *= 1.0 / (1.0 - sr);
  double rho, drho, d2rho;
  water_density(sp.density_type, p, rho, drho, d2rho);
  const double vis = kViscosity, dvis = 0.0;
  a.st[c] = FlowState{rho, Kr / vis, drho, dKr * dS / vis - Kr / (vis * vis) * dvis};
  const double ph = a.phi[c];
  const double dM = drho * ph * S + rho * ph * dS;
  const double d2M = 2.0 * dS * drho * ph + S * d2rho * ph + d2S * rho * ph;
  a.dM[c] = dM;
  a.d2M[c] = d2M;
  if (sp.form == 0) {
    a.acc[c] = dM * a.Udot[c] * a.vol[c];
  } else {
    a.acc[c] = rho * ph * S * a.vol[c] / (sp.dyn ? sp.dyn[0] : sp.dtime) - a.accum_prev[c];
  }
}

// rho phi S V / dt at Uprev (TDyMPFAOSNESPreSolve, tdympfao_snes.c:32-64)
// Diagnostics of TDyUpdateDiagnostics_MPFAO (src/fv/mpfao/tdympfao.c:2759-2786):
// liquid saturation and the reference's "liquid mass" rho*V per cell, plus the
// water mass rho*phi*S*V that a mass balance needs.
__global__ void k_diagnostics(int nc, StateParams sp, const double *__restrict__ U, const double *__restrict__ phi,
                              const double *__restrict__ Sr, const double *__restrict__ vol, double *__restrict__ S_o,
                              double *__restrict__ mass_o, double *__restrict__ water_o) {
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= nc) return;
  const double p = U[c];
  double S, dS, d2S;
  vg_saturation(sp.vg_m, sp.vg_alpha, Sr[c], sp.pref - p, S, dS, d2S);
  double rho, drho, d2rho;
  water_density(sp.density_type, p, rho, drho, d2rho);
  if (S_o) S_o[c] = S;
  if (mass_o) mass_o[c] = rho * vol[c];
  if (water_o) water_o[c] = rho * phi[c] * S * vol[c];
}

__global__ void k_snes_presolve(int nc, StateParams sp, const double *__restrict__ U,
                                const double *__restrict__ phi, const double *__restrict__ Sr,
                                const double *__restrict__ vol, double *__restrict__ accum_prev) {
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= nc) return;
  double S, dS, d2S, rho, drho, d2rho;
  vg_saturation(sp.vg_m, sp.vg_alpha, Sr[c], sp.pref - U[c], S, dS, d2S);
  water_density(sp.density_type, U[c], rho, drho, d2rho);
  accum_prev[c] = rho * phi[c] * S * vol[c] / sp.dtime;
}

struct BndStateArgs {
  int nbnd;
  StateParams sp;
  const double *U;
  const int32_t *bnd_cell;
  const double *Sr, *pbnd_fn;
  double *Pbnd;
  FlowState *st;  // boundary entries; rho and the zero derivatives are written at setup
};

__device__ inline void bnd_state(const BndStateArgs &a, int b) {
  const StateParams &sp = a.sp;
  const int c = a.bnd_cell[b];
  const double P = a.pbnd_fn ? a.pbnd_fn[b] : a.U[c];
  a.Pbnd[b] = P;
  const double sr = a.Sr[c];
  double S, dS, d2S;
  vg_saturation(sp.vg_m, sp.vg_alpha, sr, sp.pref - P, S, dS, d2S);
  const double Se = (S - sr) / (1.0 - sr);
  double Kr, dKr;
  const double cc[4] = {sp.c0, sp.c1, sp.c2, sp.c3};
  mualem_kr(sp.vg_m, sp.x0, sp.x1, sp.dx, cc, Se, Kr, dKr);
  a.st[b].ukvr = Kr / kViscosity;
}

// State of cell i < nc, or of boundary face i - nc (which depends on U alone,
// so both share a launch).
__device__ inline void state_entry(const CellStateArgs &a, const BndStateArgs &b, int i) {
  if (i < a.nc) cell_state(a, i);
  else if (i - a.nc < b.nbnd) bnd_state(b, i - a.nc);
}
__global__ void k_cell_state(CellStateArgs a, BndStateArgs b) {
  if (a.sp.stop && *a.sp.stop) return;
  state_entry(a, b, blockIdx.x * blockDim.x + threadIdx.x);
}

// boundary rho frozen at (Pref, Tref) (tdympfao.c:297-336)
__global__ void k_bnd_init(int nbnd, FlowState *__restrict__ st, double rho) {
  const int b = blockIdx.x * blockDim.x + threadIdx.x;
  if (b < nbnd) st[b] = FlowState{rho, 0.0, 0.0, 0.0};
}

struct RowArgs {
  int nc;
  int64_t nrows;
  double pref;
  const int32_t *face_cells;
  const int32_t *face_verts;
  const uint8_t *face_flags;
  const int32_t *vcols;
  const double *T;
  const double *G;
  const double *U;
  const double *Pbnd;
  const FlowState *st;
  double *flux;
  const int *stop;
};

constexpr int kRowBlock = 256;  // k_rows workgroup size

// The arithmetic of one flux row (TDyMPFAOIFunction_Vertices,
// tdympfao_ts.c:12-150; TDyMPFAOIJacobian_Vertices, 235-456), shared by the
// residual's row kernel and the Jacobian's cell kernel so that both take the
// same T.P and the same upwind side.  Inputs: the row's 8 transmissibilities
// T and the vertex's columns ck with their pressures P, rho at the two sides,
// the gravity term G.
__device__ inline double row_tp(const double (&T)[kMaxCols], const int (&ck)[kMaxCols],
                                const double (&P)[kMaxCols]) {
  double TP = 0.0;
#pragma unroll
  for (int k = 0; k < kMaxCols; k++) TP = ck[k] >= 0 ? fma(T[k], P[k], TP) : TP;
  return TP;
}
__device__ inline double row_den(double rho_up, double rho_dn) {
  double den = 0.0;
  den += rho_up;
  den += rho_dn;
  return den * 0.5;
}
__device__ inline bool row_upwind_up(double TP, double den, double G) { return fma(den, G, TP) < 0.0; }
__device__ inline double row_flux(double TP, double den, double G, double ukvr, bool zero) {
  double fluxm = den * ukvr * (-TP);
  fluxm += -(den * den) * ukvr * G;
  return zero ? 0.0 : fluxm;
}
// what d(flux) adds in the column of one side of the row beyond rho_bar
// lambda T: the derivatives dden of rho_bar and dl of kr/mu by that side's
// pressure (0 for a boundary side), negated like the flux
__device__ inline double side_extra(double TP, double den, double G, double ukvr, double dden, double dl) {
  return (dden * ukvr + den * dl) * TP + (2.0 * dden * ukvr + den * dl) * (den * G);
}

// the columns of vertex v and their pressures (padding reads U[0], unused)
__device__ inline void vertex_columns(const RowArgs &a, int v, int (&ck)[kMaxCols], double (&P)[kMaxCols]) {
  const int4 c0 = *reinterpret_cast<const int4 *>(a.vcols + (int64_t)v * kMaxCols);
  const int4 c1 = *reinterpret_cast<const int4 *>(a.vcols + (int64_t)v * kMaxCols + 4);
  ck[0] = c0.x; ck[1] = c0.y; ck[2] = c0.z; ck[3] = c0.w;
  ck[4] = c1.x; ck[5] = c1.y; ck[6] = c1.z; ck[7] = c1.w;
#pragma unroll
  for (int k = 0; k < kMaxCols; k++) {
    const int col = ck[k];
    P[k] = *(col < a.nc ? a.U + (col < 0 ? 0 : col) : a.Pbnd + (col - a.nc));
  }
}

// the row's transmissibilities, four 16-byte loads
__device__ inline void row_trans(const double *__restrict__ T, int64_t nrows, int64_t r, double (&t)[kMaxCols]) {
  const double2 *p = reinterpret_cast<const double2 *>(T) + r;
#pragma unroll
  for (int k = 0; k < kMaxCols / 2; k++) {
    const double2 q = p[k * nrows];
    t[2 * k] = q.x;
    t[2 * k + 1] = q.y;
  }
}
// rho and kr / mu of a face side
__device__ inline double2 side_state(const FlowState *st, int i) {
  return *reinterpret_cast<const double2 *>(&st[i].rho);
}
__device__ inline double2 side_derivs(const FlowState *st, int i) {
  return *reinterpret_cast<const double2 *>(&st[i].drho);
}

// Thread per flux row: the residual's flux rows (the Jacobian is assembled by
// k_cell_jac, one pass per cell).
__device__ inline void flux_row(const RowArgs &a, int64_t r) {
  const int f = (int)(r >> 2);
  const uint8_t fl = a.face_flags[f];
  double flux = 0.0;
  if (!(fl & kFaceNoFlow)) {
    const int2 ud = *reinterpret_cast<const int2 *>(a.face_cells + 2 * f);
    const int up = ud.x, dn = ud.y;
    int ck[kMaxCols];
    double P[kMaxCols], T[kMaxCols];
    vertex_columns(a, a.face_verts[r], ck, P);
    row_trans(a.T, a.nrows, r, T);
    const double2 su = side_state(a.st, flow_index(a.nc, up)), sd = side_state(a.st, flow_index(a.nc, dn));
    const double G = a.G[r];
    const double den = row_den(su.x, sd.x);
    const double TP = row_tp(T, ck, P);
    const bool upwind_up = row_upwind_up(TP, den, G);
    const int uw = upwind_up ? up : dn;
    const double ukvr = upwind_up ? su.y : sd.y;
    // a seepage face's boundary side carries no flux while its pressure is at
    // or below the reference pressure
    const bool zero = uw < 0 && (fl & kFaceSeepage) && a.Pbnd[-uw - 1] <= a.pref;
    flux = row_flux(TP, den, G, ukvr, zero);
  }
  a.flux[r] = flux;
}

__global__ void __launch_bounds__(kRowBlock) k_rows(RowArgs a) {
  if (a.stop && *a.stop) return;  // uniform over the workgroup
  const int64_t r = (int64_t)blockIdx.x * kRowBlock + threadIdx.x;
  if (r < a.nrows) flux_row(a, r);
}

// ---------------------------------------------------------------- general (prism) meshes
// Flux rows whose vertex has any number of columns: the row's T entries sit in
// its vertex's block (row-major, columns = the region's cells, then its
// Dirichlet faces).  The physics is k_rows' (tdympfao_ts.c:12-150, 235-456).
//
// A workgroup per run of consecutive vertices (at most kGrpRows rows, kGrpT
// entries, kGrpCols columns): their T blocks, one contiguous run, and their
// columns' pressures go to LDS first, all loads coalesced or gathered once per
// vertex, then a thread per row sums its own.  Bound by reading T.  The
// Jacobian needs three numbers of a row beside T itself: rho_bar lambda (0 for
// a row that carries no flux) and what each side adds in its own column
// (side_extra); k_gather_general_J forms the derivatives from T again.
// 200k prisms, residual rows 106 -> 66 us, the Jacobian's 202 -> 84 us against a
// wavefront per vertex, whose rows strode over T and gathered every pressure
// themselves (18 of 64 lanes busy), and which wrote every entry's derivative.
// Rows without a block (a triangle's fourth sub-face, no-flow faces) keep the
// zeros written at setup.
// (a single vertex may hold up to 80 x 64 entries: 48 cells, 16 Dirichlet faces)
constexpr int kGrpRows = 256, kGrpT = 4096, kGrpTMax = 5120, kGrpCols = 512;
struct GenGroup {       // a run of vertices
  int32_t row, nrow;    // block rows
  int32_t t, nt;        // T entries
  int32_t cell, ncell;  // columns: cells (ccell), then Dirichlet faces (vdcol)
  int32_t dir, ndir;
};
struct GenRow {           // a block row, relative to its group
  uint16_t t, cell, dir;  // first T entry, first cell, first Dirichlet column
  uint8_t ncell, ndir;
};
struct GenRowArgs {
  int nc;
  double pref;
  const GenGroup *grp;
  const GenRow *brd;
  const int32_t *brow;  // flux row of each block row, blocks in vertex order
  const int32_t *face_cells;
  const uint8_t *face_flags;
  const int32_t *ccell, *vdcol;
  const double *T, *G, *U, *Pbnd;
  const FlowState *st;
  double *flux, *lam;
  double2 *side;
  const int *stop;
};

template <bool WITH_R, bool WITH_J>
__global__ void __launch_bounds__(kGrpRows) k_rows_general(GenRowArgs a) {
  extern __shared__ double gen_lds[];  // the columns' pressures, then the run's T entries
  double *Ps = gen_lds, *Ts = gen_lds + kGrpCols;
  if (a.stop && *a.stop) return;
  const GenGroup g = a.grp[blockIdx.x];
  const int t = threadIdx.x;
  // the row's own data beside the staging
  const bool live = t < g.nrow;
  const int r = live ? a.brow[g.row + t] : 0, f = r >> 2;
  const GenRow d = live ? a.brd[g.row + t] : GenRow{};
  {
    double v[kGrpT / kGrpRows];
    int col[kGrpCols / kGrpRows];
#pragma unroll
    for (int i = 0; i < kGrpCols / kGrpRows; i++) {
      const int e = t + i * kGrpRows;
      col[i] = e < g.ncell ? a.ccell[g.cell + e] : e < g.ncell + g.ndir ? a.vdcol[g.dir + e - g.ncell] : 0;
    }
#pragma unroll
    for (int i = 0; i < kGrpT / kGrpRows; i++) {
      const int e = t + i * kGrpRows;
      v[i] = e < g.nt ? a.T[(int64_t)g.t + e] : 0.0;
    }
#pragma unroll
    for (int i = 0; i < kGrpCols / kGrpRows; i++) {
      const int e = t + i * kGrpRows;
      if (e < g.ncell + g.ndir) Ps[e] = e < g.ncell ? a.U[col[i]] : a.Pbnd[col[i]];
    }
#pragma unroll
    for (int i = 0; i < kGrpT / kGrpRows; i++) {
      const int e = t + i * kGrpRows;
      if (e < g.nt) Ts[e] = v[i];
    }
    for (int e = t + kGrpT; e < g.nt; e += kGrpRows) Ts[e] = a.T[(int64_t)g.t + e];
  }
  const int2 ud = *reinterpret_cast<const int2 *>(a.face_cells + 2 * f);
  const uint8_t fl = a.face_flags[f];
  const double G = a.G[r];
  const int up = ud.x, dn = ud.y;
  const FlowState su = a.st[flow_index(a.nc, up)], sd = a.st[flow_index(a.nc, dn)];
  __syncthreads();
  if (!live) return;
  double TP = 0.0;
#pragma unroll 4
  for (int j = 0; j < d.ncell; j++) TP += Ts[d.t + j] * Ps[d.cell + j];
  for (int j = 0; j < d.ndir; j++) TP += Ts[d.t + d.ncell + j] * Ps[g.ncell + d.dir + j];
  const double den = row_den(su.rho, sd.rho);
  const bool upwind_up = (TP + den * G < 0.0);
  const int uw = upwind_up ? up : dn;
  const double ukvr = upwind_up ? su.ukvr : sd.ukvr;
  const bool zero = uw < 0 && (fl & kFaceSeepage) && a.Pbnd[-uw - 1] <= a.pref;
  if (WITH_R) a.flux[r] = row_flux(TP, den, G, ukvr, zero);
  if (WITH_J) {
    a.lam[r] = zero ? 0.0 : den * ukvr;
    a.side[r] = zero ? double2{0.0, 0.0}
                     : double2{side_extra(TP, den, G, ukvr, 0.5 * su.drho, upwind_up ? su.dukvr : 0.0),
                               side_extra(TP, den, G, ukvr, 0.5 * sd.drho, upwind_up ? 0.0 : sd.dukvr)};
  }
}

// Jacobian row of each cell (CSR in the vertex-adjacency pattern, or the
// solver's ELL): its faces' flux rows in a fixed (face, sub-face) order, then
// the sides' terms and the accumulation diagonal.  kGenJLanes lanes own one
// row, summed in LDS (up to kGenJSlots entries), every slot written once.
// Lanes l and l + 16 of the 24 rows first read the rows' metadata and factors
// (face lf = i/4, sub-face i%4); then a lane per column loads T and its slot
// eight rows at a time and adds factor * T row by row with LDS adds, which
// need no answer (200k prisms 218 -> 171 us against read, add and write back,
// 32 lanes per cell): a wavefront's LDS operations run in program order and a
// flux row reaches each slot at most once (its columns are distinct cells),
// so every slot is summed in row order.  The rows' terms in the cell's own
// column and, per face, in the other cell's are reduced over the lanes first.
constexpr int kGenJBlock = 256;
constexpr int kGenJLanes = 16;  // lanes per cell: columns of a flux row (a row of more loops)
constexpr int kGenJSlots = 64;
struct GenGatherArgs {
  int nc, form, ell_w;
  int jbs;               // ELL: block size of the block-contiguous layout (see jac_row_addr)
  const int32_t *perm;   // ELL: position of row c (nullptr: CSR at jrp[c])
  double shift, dtime;
  const int32_t *cell_faces, *face_cells, *rtoff, *rinfo, *jrp, *jdiag;
  const uint8_t *face_flags, *gslot, *nslot;
  const double *T, *lam, *dM, *d2M, *Udot, *vol;
  const double2 *side;
  double *J;
  const double *dyn;  // device dtime / shift (see StateParams), or nullptr
  const int *stop;
};

// Slot of each face's other cell in the cell's Jacobian row (0xff for a
// boundary or absent face), built once at setup: one thread per cell and face.
__global__ void __launch_bounds__(256) k_gen_neighbour_slots(int nc, const int32_t *__restrict__ cell_faces,
                                                             const int32_t *__restrict__ face_cells,
                                                             const int32_t *__restrict__ jrp,
                                                             const int32_t *__restrict__ jcols,
                                                             uint8_t *__restrict__ nslot) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= (int64_t)nc * 6) return;
  const int c = (int)(i / 6), f = cell_faces[i];
  uint8_t s = 0xff;
  if (f >= 0) {
    const int o = face_cells[2 * f] == c ? face_cells[2 * f + 1] : face_cells[2 * f];
    if (o >= 0) {
      const int r0 = jrp[c];
      int lo = r0, hi = jrp[c + 1] - 1;
      while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if (jcols[mid] < o) lo = mid + 1; else hi = mid;
      }
      s = (uint8_t)(lo - r0);
    }
  }
  nslot[i] = s;
}

// Slot table of the general Jacobian gather, built once at setup: entry
// to + j of flux row r (its cell column j) has the column's slot in the up
// cell's Jacobian row at gslot[2*(to+j)] and in the down cell's at
// gslot[2*(to+j)+1] (0xff for a boundary side or a no-flow face).  One
// thread per flux row; the slot is found by binary search in the sorted row.
__global__ void __launch_bounds__(256) k_gen_slot_table(int64_t nrows, const int32_t *__restrict__ face_cells,
                                                        const uint8_t *__restrict__ face_flags,
                                                        const int32_t *__restrict__ rtoff,
                                                        const int32_t *__restrict__ rinfo,
                                                        const int32_t *__restrict__ roc,
                                                        const int32_t *__restrict__ ccell,
                                                        const int32_t *__restrict__ jrp,
                                                        const int32_t *__restrict__ jcols,
                                                        uint8_t *__restrict__ gslot) {
  const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= nrows) return;
  const int to = rtoff[r];
  if (to < 0) return;
  const int f = (int)(r >> 2);
  const int ncell = rinfo[r] & 0xff;
  const int32_t *cols = ccell + roc[r];
  const bool noflow = (face_flags[f] & kFaceNoFlow) != 0;
  for (int side = 0; side < 2; side++) {
    const int c = face_cells[2 * f + side];
    for (int j = 0; j < ncell; j++) {
      uint8_t s = 0xff;
      if (c >= 0 && !noflow) {
        const int r0 = jrp[c];
        int lo = r0, hi = jrp[c + 1] - 1;
        while (lo < hi) {
          const int mid = (lo + hi) >> 1;
          if (jcols[mid] < cols[j]) lo = mid + 1; else hi = mid;
        }
        s = (uint8_t)(lo - r0);
      }
      gslot[2 * ((int64_t)to + j) + side] = s;
    }
  }
}

__global__ void __launch_bounds__(kGenJBlock) k_gather_general_J(GenGatherArgs a) {
  constexpr int CPB = kGenJBlock / kGenJLanes;  // cells per workgroup
  constexpr int NR = 24;                        // flux rows of a cell: 6 faces x 4 sub-faces
  constexpr int RB = 8;                         // rows whose loads are in flight together
  static_assert(2 * kGenJLanes >= NR && 64 % kGenJLanes == 0, "a cell's lanes hold its rows and share a wavefront");
  __shared__ double acc[CPB][kGenJSlots + 1];
  if (a.stop && *a.stop) return;
  const int g = threadIdx.x / kGenJLanes, l = threadIdx.x % kGenJLanes;
  const int base = (threadIdx.x & 63) - l;  // the cell's first lane within the wavefront
  const int c = blockIdx.x * CPB + g;
  if (c >= a.nc) return;  // uniform over the cell's lanes (the wavefront's other cells are independent)
  const int r0 = a.jrp[c], len = a.jrp[c + 1] - r0;
  for (int k = l; k < len; k += kGenJLanes) acc[g][k] = 0.0;
  wave_lds_fence();
  // rows l and l + 16: T at T[to ..], the columns' slots, the signed factor,
  // and the sums of the sides' terms (this cell's, the other cell's)
  int to[2], ns[2];  // ns: columns | side << 8
  double fac[2], self = 0.0, other[2];
#pragma unroll
  for (int h = 0; h < 2; h++) {
    const int i = l + h * kGenJLanes;
    to[h] = -1; ns[h] = 0; fac[h] = 0.0; other[h] = 0.0;
    const int f = i < NR ? a.cell_faces[c * 6 + (i >> 2)] : -1;
    if (f >= 0 && !(a.face_flags[f] & kFaceNoFlow)) {
      const int64_t r = (int64_t)f * 4 + (i & 3);
      to[h] = a.rtoff[r];
      if (to[h] >= 0) {
        const bool up = a.face_cells[2 * f] == c;
        const double s = up ? -1.0 : 1.0;
        const double2 x = a.side[r];
        ns[h] = (a.rinfo[r] & 0xff) | (up ? 0 : 0x100);
        fac[h] = s * a.lam[r];
        self += s * (up ? x.x : x.y);
        other[h] = s * (up ? x.y : x.x);
      }
    }
  }
#pragma unroll
  for (int off = 1; off < kGenJLanes; off <<= 1) self += __shfl_xor(self, off, 64);
#pragma unroll
  for (int h = 0; h < 2; h++) {
    other[h] += __shfl_xor(other[h], 1, 64);
    other[h] += __shfl_xor(other[h], 2, 64);
  }
#pragma unroll
  for (int i0 = 0; i0 < NR; i0 += RB) {
    double tv[RB], fv[RB];
    int sv[RB];
#pragma unroll
    for (int k = 0; k < RB; k++) {
      const int h = (i0 + k) / kGenJLanes, src = base + (i0 + k) % kGenJLanes;
      const int ti = __shfl(to[h], src, 64), ni = __shfl(ns[h], src, 64);
      fv[k] = __shfl(fac[h], src, 64);
      const bool on = ti >= 0 && l < (ni & 0xff);
      tv[k] = on ? a.T[ti + l] : 0.0;
      sv[k] = on ? a.gslot[2 * ((int64_t)ti + l) + (ni >> 8)] : -1;
    }
#pragma unroll
    for (int k = 0; k < RB; k++) {
      if (sv[k] >= 0) atomicAdd(&acc[g][sv[k]], fv[k] * tv[k]);
      // columns past the lanes (regions of more than kGenJLanes cells): the rest of the same row
      const int h = (i0 + k) / kGenJLanes, src = base + (i0 + k) % kGenJLanes;
      const int ti = __shfl(to[h], src, 64), ni = __shfl(ns[h], src, 64);
      for (int j = l + kGenJLanes; ti >= 0 && j < (ni & 0xff); j += kGenJLanes)
        atomicAdd(&acc[g][a.gslot[2 * ((int64_t)ti + j) + (ni >> 8)]], fv[k] * a.T[ti + j]);
    }
  }
#pragma unroll
  for (int h = 0; h < 2; h++) {
    const int lf = (l + h * kGenJLanes) >> 2;
    if ((l & 3) == 0 && lf < 6) {  // a face each: its other cell's slot is its own
      const int s = a.nslot[(int64_t)c * 6 + lf];
      if (s != 0xff) atomicAdd(&acc[g][s], other[h]);
    }
  }
  if (l == 0) {
    const double shift = a.dyn ? a.dyn[1] : a.shift, dtime = a.dyn ? a.dyn[0] : a.dtime;
    const double dvc = (a.form == 0) ? (shift * a.dM[c] + a.d2M[c] * a.Udot[c]) * a.vol[c]
                                     : a.dM[c] * a.vol[c] * (1.0 / dtime);
    atomicAdd(&acc[g][a.jdiag[c]], self + dvc);
  }
  wave_lds_fence();
  int64_t st = 1;
  double *row = a.J + r0;
  if (a.perm) {
    const int64_t p = a.perm[c], bs = a.jbs;
    row = a.J + (p / bs * a.ell_w) * bs + p % bs;
    st = bs;
  }
  const int nslot = a.perm ? a.ell_w : len;  // ELL rows are padded to ell_w slots with zeros
  for (int k = l; k < nslot; k += kGenJLanes) row[k * st] = k < len ? acc[g][k] : 0.0;
}

struct GatherArgs {
  int nc;
  int64_t nrows;
  int form;  // 0 TS, 1 SNES
  double shift, dtime;
  const int32_t *cell_faces, *face_cells;
  const uint8_t *face_flags, *jdslot;
  const double *flux, *acc, *dM, *d2M, *Udot, *vol;
  const double *src;   // source_sink per cell, or nullptr (TS form: scaled by the volume)
  const int32_t *jrp;  // CSR row starts, or nullptr for the slot-major ELL layout
  const int32_t *perm; // ELL: position of row c (nullptr: c)
  int jbs;             // ELL: block size bs of the block-contiguous layout (slot k of position p at
                       // (p/bs*ell_w + k)*bs + p%bs)
  int ell_w;           // ELL width (slots written per row in the ELL layout)
  double *R, *J;
  const double *dyn;   // device dtime / shift (see StateParams), or nullptr
  const int *stop;
};

constexpr int kGatherBlock = 128;
constexpr int kJacSlots = 27;  // vertex-adjacency row length of a hexahedral mesh

// Where cell c's Jacobian row starts and the distance between its slots: CSR
// values at jrp[c] (stride 1), or the solver's block-contiguous ELL.
__device__ inline void jac_row_addr(const GatherArgs &a, int c, int64_t &base, int64_t &stride) {
  if (a.jrp) { base = a.jrp[c]; stride = 1; return; }
  const int64_t p = a.perm ? a.perm[c] : c, bs = a.jbs;
  base = (p / bs * a.ell_w) * bs + p % bs;
  stride = bs;
}

// R[c] from the flux rows: the cell's faces' four rows summed in sub-face
// order, +/- by orientation, then the accumulation and the source
// (tdympfao_ts.c:191-212, tdympfao_snes.c:112-123).
__device__ inline double cell_residual(const GatherArgs &a, int c, double s) {
  double r = s + a.acc[c];
  if (a.src) r -= (a.form == 0) ? a.src[c] * a.vol[c] : a.src[c];
  return r;
}

// Per-cell residual gather (thread per cell): every cell owns its entry, so
// the result does not depend on scheduling.
__device__ inline void cell_gather(const GatherArgs &a, int c) {
  double s = 0.0;
#pragma unroll
  for (int lf = 0; lf < 6; lf++) {
    const int f = a.cell_faces[c * 6 + lf];
    if (f < 0) continue;  // a prism has 5 faces (a triangle's fourth flux row is zero)
    const double4 q = *reinterpret_cast<const double4 *>(a.flux + (int64_t)f * 4);
    const double fs = ((q.x + q.y) + q.z) + q.w;
    s += (a.face_cells[2 * f] == c) ? fs : -fs;
  }
  a.R[c] = cell_residual(a, c, s);
}

__global__ void __launch_bounds__(kGatherBlock) k_cell_gather(GatherArgs a) {
  if (a.stop && *a.stop) return;
  const int c = blockIdx.x * kGatherBlock + threadIdx.x;
  if (c < a.nc) cell_gather(a, c);
}

// Single-pass Jacobian (and, WITH_R, residual) of a hexahedral mesh
// (TDyMPFAOIJacobian_Vertices, tdympfao_ts.c:235-456, evaluated from the
// cell's side): eight lanes per cell, one per corner.  The three faces of the
// cell that meet at a corner have one flux row each at that corner's vertex;
// the three rows share the vertex's 8 columns and pressures (gathered once)
// and the 8 slots of the cell's Jacobian row those columns occupy, so the lane
// sums the rows' derivatives in registers (face order) and stages the 8 sums
// and their slots in LDS.  Then the eight lanes add the eight corners into the
// row in corner order, a lane per column (a fixed summation order, so the
// result does not depend on scheduling; one lane per cell adding all 64
// values left the wavefront's other lanes idle: CSR at 1M cells 651 -> 611 us,
// block layout 617 -> 551 us, 95k cells 51 -> 44 us), the accumulation diagonal
// follows, and the lanes write the row.  Each flux row is evaluated by both cells of its face;
// the second read of T hits the cache when the two cells run close together,
// which `order` (position -> cell: the block-Jacobi layout's row list, -1
// padding) and the XCD-grouped workgroup numbering arrange.
//   crow[c*8 + j]: the corner's three rows as 5-bit (face slot * 4 + sub-face)
//                  codes in face order (bits 0-4, 5-9, 10-14), the cell's index
//                  in the region of the corner's vertex (bits 15-17),
//                  whether the cell is each row's up cell (bits 18, 19, 20),
//                  and the index of each row's other cell there (bits 21-29)
//   cell_verts[c*8 + j]: the corner's vertex
//   jslot[v*64 + li*8 + k]: slot of column k of vertex v's region in the row
//                  of the region's cell li (255: not a cell column)
// A no-flow face's row is evaluated like the others, at the cell itself on
// both sides (every read in range), and dropped.
struct CellJacArgs {
  const int32_t *order;  // position -> cell, or nullptr (position i is cell i)
  int64_t npos;
  int xcd_groups;        // 0: workgroups in launch order; else the launch is 8 * xcd_groups workgroups
  const uint32_t *crow;
  const int32_t *cell_verts;
  const uint8_t *jslot;
};

constexpr int kCellJacBlock = 256;                // lanes per workgroup
constexpr int kCellJacCells = kCellJacBlock / 8;  // cells per workgroup

// block blk of the cells (in `order`): kCellJacCells cells, 8 lanes each
template <bool WITH_R>
__device__ inline void cell_jac_block(const RowArgs &ra, const GatherArgs &a, const CellJacArgs &cj, int64_t blk) {
  __shared__ double sd[kMaxCols][kCellJacBlock];     // corner sums: column k of lane t at sd[k][t]
  __shared__ uint64_t sw[kCellJacBlock];             // their slots (one byte per column)
  __shared__ double sf[WITH_R ? 24 : 1][kCellJacCells];  // flux of row lf*4+q of cell cl
  __shared__ double acc[kJacSlots + 1][kCellJacCells];   // the row (slot kJacSlots: non-cell columns)
  const int t = threadIdx.x, cl = t >> 3, corner = t & 7;
  const int64_t i = blk * kCellJacCells + cl;
  const int c = i < cj.npos ? (cj.order ? cj.order[i] : (int)i) : -1;  // -1: no cell
  double dv = 0.0;  // the accumulation's diagonal entry
  int dslot = 0;
  if (c >= 0) {
    for (int sl = corner; sl < kJacSlots; sl += 8) acc[sl][cl] = 0.0;
    {
      const double shift = a.dyn ? a.dyn[1] : a.shift, dtime = a.dyn ? a.dyn[0] : a.dtime;
      dv = (a.form == 0) ? (shift * a.dM[c] + a.d2M[c] * a.Udot[c]) * a.vol[c] : a.dM[c] * a.vol[c] * (1.0 / dtime);
      dslot = a.jdslot[c];
    }
    const unsigned code = cj.crow[(int64_t)c * 8 + corner];
    const int v = cj.cell_verts[(int64_t)c * 8 + corner];
    // the cell's faces beside the code that picks three of them: one trip to
    // memory less before T
    const int2 *cf = reinterpret_cast<const int2 *>(a.cell_faces + (int64_t)c * 6);
    const int2 f01 = cf[0], f23 = cf[1], f45 = cf[2];
    const int li = (code >> 15) & 7;
    int fr[3], lfq[3];
#pragma unroll
    for (int m = 0; m < 3; m++) {
      lfq[m] = (code >> (5 * m)) & 31;
      const int lf = lfq[m] >> 2;
      const int2 pr = lf < 2 ? f01 : lf < 4 ? f23 : f45;
      fr[m] = (lf & 1) ? pr.y : pr.x;
    }
    int ck[kMaxCols];
    double P[kMaxCols];
    vertex_columns(ra, v, ck, P);
    const uint64_t w = *reinterpret_cast<const uint64_t *>(cj.jslot + (int64_t)v * 64 + li * 8);
    // the three rows' loads together, both sides' states (a no-flow face's row
    // runs at the cell on both sides, every read in range, and is dropped)
    int up[3], dn[3];
    bool noflow[3], seep[3];
    double T[3][kMaxCols], G[3];
    double2 su[3], sd2[3], du2[3], dd2[3];  // rho and kr / mu, and their derivatives, of the two sides
#pragma unroll
    for (int m = 0; m < 3; m++) {
      const int f = fr[m];
      const int64_t r = (int64_t)f * 4 + (lfq[m] & 3);
      const uint8_t fl = a.face_flags[f];
      const int2 ud = *reinterpret_cast<const int2 *>(a.face_cells + 2 * f);
      noflow[m] = (fl & kFaceNoFlow) != 0;
      seep[m] = (fl & kFaceSeepage) != 0;
      up[m] = noflow[m] ? c : ud.x;
      dn[m] = noflow[m] ? c : ud.y;
      row_trans(ra.T, ra.nrows, r, T[m]);
      G[m] = ra.G[r];
      const int iu = flow_index(ra.nc, up[m]), id = flow_index(ra.nc, dn[m]);
      su[m] = side_state(ra.st, iu);
      sd2[m] = side_state(ra.st, id);
      du2[m] = side_derivs(ra.st, iu);
      dd2[m] = side_derivs(ra.st, id);
    }
    double TP[3], den[3], ukvr[3], du[3], pb[3];
    bool upw[3];
    int uw[3];
#pragma unroll
    for (int m = 0; m < 3; m++) {
      TP[m] = row_tp(T[m], ck, P);
      den[m] = row_den(su[m].x, sd2[m].x);
      upw[m] = row_upwind_up(TP[m], den[m], G[m]);
      uw[m] = upw[m] ? up[m] : dn[m];
    }
#pragma unroll
    for (int m = 0; m < 3; m++) {
      ukvr[m] = upw[m] ? su[m].y : sd2[m].y;
      du[m] = upw[m] ? du2[m].y : dd2[m].y;
      pb[m] = ra.Pbnd[uw[m] < 0 ? -uw[m] - 1 : 0];  // Pbnd always holds at least one entry
    }
    // Row m adds s (rho_bar lambda) T to the corner's columns, s the sign of
    // its flux in this cell's residual (0 for a row that carries none); the
    // derivatives of rho_bar and kr/mu go to the columns of its two sides, this
    // cell's own (column li) and the other cell's (tdympfao_ts.c:439-444).
    // Boundary-pressure and padding columns gather values nobody reads.
    double sum[kMaxCols], self = 0.0, other[3];
#pragma unroll
    for (int k = 0; k < kMaxCols; k++) sum[k] = 0.0;
#pragma unroll
    for (int m = 0; m < 3; m++) {
      const bool zero = noflow[m] | ((uw[m] < 0) & seep[m] & (pb[m] <= ra.pref));
      const bool is_up = (code >> (18 + m)) & 1;
      const double s = zero ? 0.0 : is_up ? -1.0 : 1.0;
      const double sl = s * (den[m] * ukvr[m]);
#pragma unroll
      for (int k = 0; k < kMaxCols; k++) sum[k] = fma(sl, T[m][k], sum[k]);
      const double xu = side_extra(TP[m], den[m], G[m], ukvr[m], 0.5 * du2[m].x, upw[m] ? du2[m].y : 0.0);
      const double xd = side_extra(TP[m], den[m], G[m], ukvr[m], 0.5 * dd2[m].x, upw[m] ? 0.0 : dd2[m].y);
      self += s * (is_up ? xu : xd);
      other[m] = s * (is_up ? xd : xu);
      if (WITH_R) sf[lfq[m]][cl] = noflow[m] ? 0.0 : row_flux(TP[m], den[m], G[m], ukvr[m], zero);
    }
#pragma unroll
    for (int k = 0; k < kMaxCols; k++) sd[k][t] = sum[k];
    // (each lane adds to its own entries: plain LDS adds, in order)
    atomicAdd(&sd[li][t], self);
#pragma unroll
    for (int m = 0; m < 3; m++)
      if (((code >> (18 + m)) & 1 ? dn[m] : up[m]) >= 0) atomicAdd(&sd[(code >> (21 + 3 * m)) & 7][t], other[m]);
    sw[t] = w;
  }
  // a cell's eight lanes share a wavefront: no barrier from here on
  wave_lds_fence();
  if (c < 0) return;
  // corner by corner, lane k adds column k's sum into its slot: a region's
  // cells are distinct, so a corner's 8 slots are (apart from kJacSlots,
  // which is never read), and every slot is summed in corner order
  const int base8 = t - corner;
  unsigned sl[8];
  double v[8];
#pragma unroll
  for (int j = 0; j < 8; j++) {
    const unsigned b = (unsigned)(sw[base8 + j] >> (8 * corner)) & 0xffu;
    sl[j] = b == 0xffu ? kJacSlots : b;
    v[j] = sd[corner][base8 + j];
  }
#pragma unroll
  for (int j = 0; j < 8; j++) {
    acc[sl[j]][cl] += v[j];
    wave_lds_fence();
  }
  if (corner == 0) acc[dslot][cl] += dv;
  if (WITH_R) {
    // fluxes by face in face order, then accumulation, then the source
    // (tdympfao_ts.c:191-212, tdympfao_snes.c:112-123)
    double fs = 0.0;
    if (corner < 6) {
      const int f = a.cell_faces[c * 6 + corner];
      fs = ((sf[corner * 4][cl] + sf[corner * 4 + 1][cl]) + sf[corner * 4 + 2][cl]) + sf[corner * 4 + 3][cl];
      if (a.face_cells[2 * f] != c) fs = -fs;
    }
    double s = 0.0;
#pragma unroll
    for (int lf = 0; lf < 6; lf++) s += __shfl(fs, (base8 & 63) + lf, 64);
    if (corner == 0) a.R[c] = cell_residual(a, c, s);
  }
  wave_lds_fence();
  int64_t base = c, stride = 1;
  jac_row_addr(a, c, base, stride);
  const int len = a.jrp ? a.jrp[c + 1] - a.jrp[c] : a.ell_w;
  for (int sl = corner; sl < len; sl += 8) a.J[base + (int64_t)sl * stride] = acc[sl][cl];
}

template <bool WITH_R>
__global__ void __launch_bounds__(kCellJacBlock) k_cell_jac(RowArgs ra, GatherArgs a, CellJacArgs cj) {
  if (a.stop && *a.stop) return;  // uniform over the workgroup
  // with xcd_groups, hardware round-robin places workgroup w on XCD w % 8:
  // give XCD x the contiguous run of blocks [x * xcd_groups, (x + 1) * xcd_groups)
  const int64_t blk = cj.xcd_groups ? (int64_t)(blockIdx.x % 8) * cj.xcd_groups + blockIdx.x / 8 : blockIdx.x;
  cell_jac_block<WITH_R>(ra, a, cj, blk);
}

// ---------------------------------------------------------------- fused multi-request launches
// One launch runs the same evaluation for several independent problems (the
// requests of a serving batch), each a segment of the grid: a workgroup
// belongs to the segment whose block range holds it and computes exactly
// what the single-problem kernel computes for its local block, so each
// request's result is the same bit for bit whatever else shares the launch.
// A segment whose stop flag is set does nothing.
constexpr int kMaxSeg = 32;
struct SegBlocks {
  int nseg;
  int64_t start[kMaxSeg + 1];  // first global block of each segment; start[nseg] = the grid
};
__device__ inline int seg_find(const SegBlocks &sb, int64_t b) {
  int s = 0;
  while (s + 1 < sb.nseg && b >= sb.start[s + 1]) s++;
  return s;
}
struct SegProblem {  // one request's arguments of every fused launch
  CellStateArgs cs;
  BndStateArgs bs;
  RowArgs ra;
  GatherArgs ga;
  CellJacArgs cj;
  const int *stop;
};

__global__ void __launch_bounds__(256) k_seg_state(const SegProblem *__restrict__ P, SegBlocks sb) {
  const int s = seg_find(sb, blockIdx.x);
  if (P[s].stop && *P[s].stop) return;
  state_entry(P[s].cs, P[s].bs, (int)((blockIdx.x - sb.start[s]) * 256 + threadIdx.x));
}
__global__ void __launch_bounds__(kRowBlock) k_seg_rows(const SegProblem *__restrict__ P, SegBlocks sb) {
  const int s = seg_find(sb, blockIdx.x);
  if (P[s].stop && *P[s].stop) return;
  const int64_t r = (blockIdx.x - sb.start[s]) * kRowBlock + threadIdx.x;
  if (r < P[s].ra.nrows) flux_row(P[s].ra, r);
}
__global__ void __launch_bounds__(kGatherBlock) k_seg_cell_gather(const SegProblem *__restrict__ P, SegBlocks sb) {
  const int s = seg_find(sb, blockIdx.x);
  if (P[s].stop && *P[s].stop) return;
  const int c = (int)((blockIdx.x - sb.start[s]) * kGatherBlock + threadIdx.x);
  if (c < P[s].ga.nc) cell_gather(P[s].ga, c);
}
__global__ void __launch_bounds__(kCellJacBlock) k_seg_cell_jac(const SegProblem *__restrict__ P, SegBlocks sb) {
  // the segment is uniform over the workgroup: its arguments are copied out
  // once (scalar loads) rather than read through the table at every use
  const int s = __builtin_amdgcn_readfirstlane(seg_find(sb, blockIdx.x));
  if (P[s].stop && *P[s].stop) return;
  const RowArgs ra = P[s].ra;
  const GatherArgs ga = P[s].ga;
  const CellJacArgs cj = P[s].cj;
  cell_jac_block<false>(ra, ga, cj, blockIdx.x - sb.start[s]);
}

__global__ void k_fill(int64_t n, double *__restrict__ x, double val) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) x[i] = val;
}

// Velocity recovery (TDyMPFAORecoverVelocity, tdympfao_utils.c:103-217, 219-532):
// the potential of each cell is Phi = p + rho(p) |g| z_c, and every flux row
// q of face f adds -(T_row . Phi) / A_f to vel[f].  A boundary column takes
// the boundary-pressure function value (no gravity term) when one is set,
// else Phi of the face's cell (tdympfao_utils.c:314-324).
//
// One lane per flux row (T is read coalesced, as by k_rows); a face's four
// lanes add their rows in sub-face order, so the result is deterministic.
// Bound by reading T and by the potentials, evaluated per column: no scratch,
// so calls on several streams do not meet.  (One thread per face, its rows'
// columns strided over the wavefront: 325 -> 153 us at 442,368 cells.)
struct VelArgs {
  int nc, nf, general, has_fn, density_type;
  int64_t nrows;
  double gabs;  // |g|
  const uint8_t *face_flags;
  const int32_t *face_verts, *vcols;                          // hexahedra: rows by vertex columns
  const double *T;                                            // hexahedra: pairs of columns over rows (trans_index)
  const int32_t *rtoff, *rinfo, *roc, *rdc, *ccell, *vdcol;   // general meshes: per-row blocks
  const double *Tgen;
  const int32_t *bnd_cell;
  const double *U, *cell_z, *pbnd_fn, *face_area;
  double *vel;
  int32_t *count;
};

__device__ inline double vel_phi_cell(const VelArgs &a, int c) {
  double rho, drho, d2rho;
  water_density(a.density_type, a.U[c], rho, drho, d2rho);
  return a.U[c] + rho * a.gabs * a.cell_z[c];
}

__device__ inline double vel_phi_bnd(const VelArgs &a, int b) {
  return a.has_fn ? a.pbnd_fn[b] : vel_phi_cell(a, a.bnd_cell[b]);
}

__global__ void __launch_bounds__(256) k_velocity(VelArgs a) {
  const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int q = (int)(r & 3);
  const bool in = r < a.nrows;
  const int f = in ? (int)(r >> 2) : 0;
  double v = 0.0;
  int n = 0;
  if (in && !(a.face_flags[f] & kFaceNoFlow)) {
    double tp = 0.0;
    bool row = true;
    if (a.general) {
      const int to = a.rtoff[r];
      row = to >= 0;  // not the fourth row of a triangle
      if (row) {
        const int ncell = a.rinfo[r] & 0xff, ndir = (a.rinfo[r] >> 8) & 0xff;
        const int32_t *cols = a.ccell + a.roc[r];
        const int32_t *dcols = a.vdcol + a.rdc[r];
        const double *Tr = a.Tgen + to;
#pragma unroll 4
        for (int j = 0; j < ncell; j++) tp += Tr[j] * vel_phi_cell(a, cols[j]);
        for (int j = 0; j < ndir; j++) tp += Tr[ncell + j] * vel_phi_bnd(a, dcols[j]);
      }
    } else {
      const int4 *vc = reinterpret_cast<const int4 *>(a.vcols + (int64_t)a.face_verts[r] * kMaxCols);
      const int4 c0 = vc[0], c1 = vc[1];
      const int ck[kMaxCols] = {c0.x, c0.y, c0.z, c0.w, c1.x, c1.y, c1.z, c1.w};
      double T[kMaxCols], P[kMaxCols], z[kMaxCols];
      row_trans(a.T, a.nrows, r, T);
#pragma unroll
      for (int k = 0; k < kMaxCols; k++) {
        const int c = ck[k] < 0 || ck[k] >= a.nc ? 0 : ck[k];
        P[k] = a.U[c];
        z[k] = a.cell_z[c];
      }
#pragma unroll
      for (int k = 0; k < kMaxCols; k++) {
        double rho, drho, d2rho;
        water_density(a.density_type, P[k], rho, drho, d2rho);
        const double phi = ck[k] < a.nc ? P[k] + rho * a.gabs * z[k] : vel_phi_bnd(a, ck[k] - a.nc);
        if (ck[k] >= 0) tp += T[k] * phi;
      }
    }
    if (row) {
      v = -tp / a.face_area[f];
      n = 1;
    }
  }
  // the face's rows in sub-face order, in its first lane
  const int l0 = (threadIdx.x & 63) - q;
  double s = __shfl(v, l0, 64);
  int m = __shfl(n, l0, 64);
#pragma unroll
  for (int k = 1; k < 4; k++) {
    s += __shfl(v, l0 + k, 64);
    m += __shfl(n, l0 + k, 64);
  }
  if (in && q == 0) {
    a.vel[f] = s;
    if (a.count) a.count[f] = m;
  }
}

}  // namespace tdyhip

