// Newton's inner linear solve on the device (subsystem (d)): ELL SpMV,
// block-Jacobi ILU(0) and the BLAS-1 pieces of GMRES(m), templated on the
// Krylov precision.
//
// The reference leaves this to PETSc (KSPGMRES, restart 30, left
// preconditioning, classical Gram-Schmidt; PCILU(0) serial / PCBJACOBI+ILU(0)
// parallel; driven from src/tdyti.c:135,188).
//
// Block-Jacobi ILU(0): cells are partitioned (host) into compact blocks of at
// most BS cells (BS = 64: one wavefront per block; BS = 256 or 512: one 4- or
// 8-wave workgroup per block; at 512 the FP64 factor holds 125 KB of LDS).  Inside a block rows keep their global order;
// entries coupling different blocks are dropped.  The factorization (IKJ)
// and the two triangular solves advance level by level (levels of the
// in-block dependency DAG, computed on the host) with the block's rows in
// LDS, so no grid-wide synchronisation is ever needed.  The Jacobian is held
// block by block (slot s of row t of block b at (b*W + s)*BS + t) so every sweep
// is coalesced.
#include "tdyhip_internal.h"

namespace tdyhip {

constexpr int kBlkMax = 512;  // max rows per block
constexpr int kW = 27;        // max in-block entries per row (hexahedral vertex adjacency)
constexpr int kLU = 13;       // max strictly lower (upper) entries per row
// Factored block layout per row (slot-major, stride BS): slots 0..12 L
// multipliers (the nearest column first), 13..25 U entries (the nearest column
// first), 26 the inverse diagonal; padded L/U slots hold 0 and point at the zero
// entry x[BS] of the apply kernel's LDS vector.
//
// Chains: runs of consecutive rows (at most kChainMax, within 16 lanes) whose
// only coupling inside the run is to the row before, as the lines of a brick.
// The triangular sweeps solve a chain at once, so their levels are those of
// the chains (14 for an 8x8x4 brick, against 34 of its rows).
constexpr int kChainMax = 8;
constexpr uint16_t kChainLink = 0x8000;  // row t couples to row t-1 (forward) or t+1 (backward) of its chain

// Per-block arrays are strided by the block width BS (64, 256 or 512).
struct BJLayout {
  int nblocks = 0;
  int bs = 0;                  // stride / launch width (64, 256 or 512)
  int32_t *d_row = nullptr;    // nblocks*bs global row (-1 pad)
  int32_t *d_jpos = nullptr;   // nblocks*kW*bs position in the ELL Jacobian less the block's first entry (-1 pad)
  int ell_w = 0;               // ELL width W: block b's entries start at b*W*bs
  uint8_t *d_diag = nullptr;   // nblocks*bs slot of the diagonal
  uint8_t *d_nslot = nullptr;  // nblocks*bs number of slots
  uint16_t *d_swL = nullptr;   // nblocks*bs: level of each row's chain in the forward sweep, | kChainLink
  uint16_t *d_swU = nullptr;   // nblocks*bs: the same for the backward sweep
  int32_t *d_nsw = nullptr;    // nblocks*2 (forward, backward level counts)
  int32_t *d_nlu = nullptr;    // nblocks: L/U slots in use (the factor writes and the sweeps read only
                               // these); nullptr when every block uses all kLU
  int32_t *d_bw = nullptr;     // nblocks: ELL slots in use (the block's longest row; the SpMV reads only
                               // these); nullptr when every block reads all W
  uint16_t *d_cL = nullptr;    // nblocks*kLU*bs local column of L slot (bs = zero entry)
  uint16_t *d_cU = nullptr;    // nblocks*kLU*bs local column of U slot
  // Factorization: rows by level (lrow, levels starting at lptr[0..nlev]) and,
  // per row, 16 bytes for each of 32 lanes, lane d standing for slot d: bytes
  // 0..12 the slot of row k_p (k_p the column of lower slot p) that holds slot
  // d's column (kNoSlot: none, or d <= p), then slot d's column (16 bits) and the row's
  // diagonal slot.
  uint16_t *d_lrow = nullptr;  // nblocks*bs
  uint16_t *d_lptr = nullptr;  // nblocks*(bs+1)
  int32_t *d_nlev = nullptr;   // nblocks: levels
  uint4 *d_ftab = nullptr;     // nblocks*bs*kFacLanes
  // Shared index patterns: every index table above except d_row (and the
  // solver's int16 column offsets) holds one entry per pattern, block b using
  // pattern d_pat[b]; nullptr: every block has its own.
  int32_t *d_pat = nullptr;    // nblocks
  int npat = 0;
};

constexpr int kFacLanes = 32;   // lanes per row of the factorization
constexpr uint8_t kNoSlot = kW; // a row's slot past its entries: holds 0 in the factorization's LDS

// ---------------------------------------------------------------- device-resident GMRES cycle
// State shared by the kernels of one restart cycle; `done` makes every later
// kernel of the cycle return at once, so the host launches a whole cycle and
// synchronises once.
struct GmresDev {
  double tol;      // stopping tolerance on the preconditioned residual
  double inv_h;    // 1/h(j+1,j) or 1/beta for the next basis vector
  double resid;    // current residual estimate |g(j+1)|
  int done;        // cycle finished (converged, breakdown, or iteration cap)
  int converged;
  int its;         // total Arnoldi steps
  int jcur;        // basis vectors completed in this cycle
  int maxit;
  int finished;    // the solve is over: converged, iteration cap, or a non-finite residual
  int diverged;    // a non-finite residual estimate (KSP_DIVERGED_NANORINF)
  int jlast;       // columns of the last cycle that ended (its Hessenberg solve)
};

// ---------------------------------------------------------------- ILU(0) factor
// IKJ elimination level by level, half a wavefront per row, lane d holding the
// row's slot d in a register.  The rows k_p a row eliminates with are finished,
// so everything read of them (their entry in slot d's column, one LDS read per
// lower slot, and the reciprocal pivot of the lane's own column) is in flight
// before the first multiplier; what remains per lower slot is a product, a
// broadcast through scalar registers and a multiply-add.  The next level's table
// entries are fetched a level ahead.
//
// Bound by that chain: 34 levels of an 8x8x4 brick.  (Values updated in LDS by
// lists of pairs, four lanes per row, waited for about eight LDS round trips
// and a division per lower slot: 8x8x4 bricks, 1M cells 1825 -> 472 us, FP32 at
// 442,368 cells 657 -> 150, 63k 215 -> 74; 4x4x4 bricks, 4k cells 85 -> 31.)
constexpr int kFacPitch = kW + 2;  // a row's LDS pitch: its slots, the zero kNoSlot points at, odd
template <int BS>
struct FactorLanes {
  static constexpr int NT = BS == 64 ? 256 : 512;
  static constexpr int ROWS = NT / kFacLanes;  // rows at once
};

template <class TV>
__device__ inline TV lane_bcast(TV v, int lane);  // lane uniform
template <>
__device__ inline float lane_bcast<float>(float v, int lane) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}
template <>
__device__ inline double lane_bcast<double>(double v, int lane) {
  const uint64_t u = __double_as_longlong(v);
  const uint32_t lo = __builtin_amdgcn_readlane((int)u, lane), hi = __builtin_amdgcn_readlane((int)(u >> 32), lane);
  return __longlong_as_double((long long)((uint64_t)hi << 32 | lo));
}

template <class TV, int BS>
__global__ void __launch_bounds__(FactorLanes<BS>::NT)
k_bj_factor(BJLayout L, const double *__restrict__ J, TV *__restrict__ fac, int *__restrict__ status) {
  constexpr int NT = FactorLanes<BS>::NT, ROWS = FactorLanes<BS>::ROWS;
  __shared__ TV a[BS * kFacPitch];
  __shared__ TV piv[BS];  // reciprocal pivots of the finished rows
  __shared__ uint16_t lrow[BS], lptr[BS + 1];
  const int b = blockIdx.x, tid = threadIdx.x;
  // index tables of the block's pattern (shared by identical blocks); values per block
  const int pb = L.d_pat ? L.d_pat[b] : b;
  const int64_t base = (int64_t)pb * BS;
  const int64_t ibase = (int64_t)pb * kW * BS;
  const int64_t sbase = (int64_t)b * kW * BS;
  const int nlev = L.d_nlev[pb];
  {
    // the block's value loads, a batch in flight together
    constexpr int NB = 14;
    const double *Jb = J + (int64_t)b * L.ell_w * BS;
    for (int e0 = tid; e0 < kW * BS; e0 += NB * NT) {
      int32_t pos[NB];
      TV v[NB];
#pragma unroll
      for (int i = 0; i < NB; i++) pos[i] = e0 + i * NT < kW * BS ? L.d_jpos[ibase + e0 + i * NT] : -1;
#pragma unroll
      for (int i = 0; i < NB; i++) v[i] = pos[i] >= 0 ? (TV)Jb[pos[i]] : (TV)0;  // relative to the block's first position
#pragma unroll
      for (int i = 0; i < NB; i++) {
        const int e = e0 + i * NT;
        if (e < kW * BS) a[(e % BS) * kFacPitch + e / BS] = v[i];
      }
    }
  }
  for (int r = tid; r < BS; r += NT) {
    a[r * kFacPitch + kNoSlot] = (TV)0;
    piv[r] = (TV)0;
    lrow[r] = L.d_lrow[base + r];
  }
  for (int r = tid; r <= nlev; r += NT) lptr[r] = L.d_lptr[(int64_t)pb * (BS + 1) + r];
  __syncthreads();
  const int d = tid % kFacLanes, hw = tid / kFacLanes;
  const bool hi = (tid & 32) != 0;
  const uint4 *tab = L.d_ftab + (int64_t)pb * BS * kFacLanes + d;
  auto fetch = [&](int j, int end) {  // the table entry of the level's row j (a row past the end re-reads row 0's)
    return tab[(int64_t)(j < end ? lrow[j] : 0) * kFacLanes];
  };
  uint4 nt = fetch(lptr[0] + hw, lptr[1]);
  for (int l = 0; l < nlev; l++) {
    const int j0 = lptr[l], j1 = lptr[l + 1], j2 = l + 1 < nlev ? lptr[l + 2] : j1;
    for (int jb = j0; jb < j1; jb += ROWS) {  // uniform over the workgroup
      const int j = jb + hw;
      const bool live = j < j1;
      const uint4 tb = nt;
      nt = jb + ROWS < j1 ? fetch(jb + ROWS + hw, j1) : fetch(j1 + hw, j2);
      const int r = live ? lrow[j] : 0;
      const int c = (tb.w >> 8) & 0xffff, di = live ? (int)(tb.w >> 24) : 0;
      TV v = d < kW ? a[r * kFacPitch + d] : (TV)0;
      const TV ip = d < di ? piv[c] : (TV)0;
      const int pmax = max(__builtin_amdgcn_readlane(di, 0), __builtin_amdgcn_readlane(di, 32));
      const uint32_t tw[4] = {tb.x, tb.y, tb.z, tb.w};
      TV src[kLU];
#pragma unroll
      for (int p = 0; p < kLU; p++)
        if (p < pmax) {
          const int k0 = __builtin_amdgcn_readlane(c, p), k1 = __builtin_amdgcn_readlane(c, 32 + p);
          src[p] = a[(hi ? k1 : k0) * kFacPitch + ((tw[p / 4] >> (8 * (p % 4))) & 0xff)];
        }
#pragma unroll
      for (int p = 0; p < kLU; p++)
        if (p < pmax) {
          const TV m = v * ip;
          const TV m0 = lane_bcast(m, p), m1 = lane_bcast(m, 32 + p);
          v -= (hi ? m1 : m0) * src[p];
        }
      if (live && d < kW) {
        a[r * kFacPitch + d] = d < di ? v * ip : v;
        if (d == di) {
          piv[r] = (TV)1 / v;
          if (v == (TV)0) atomicOr(status, 1);
        }
      }
    }
    __syncthreads();
  }
  // split layout: L multipliers and U entries by distance from the diagonal, reciprocal pivot
  const int nlu = L.d_nlu ? L.d_nlu[pb] : kLU;
  for (int e = tid; e < nlu * BS; e += NT) {
    const int p = e / BS, t = e % BS;
    const int di = L.d_diag[base + t], ns = L.d_nslot[base + t];
    fac[sbase + (int64_t)p * BS + t] = (p < di) ? a[t * kFacPitch + di - 1 - p] : (TV)0;
    const int q = di + 1 + p;
    fac[sbase + (int64_t)(kLU + p) * BS + t] = (q < ns) ? a[t * kFacPitch + q] : (TV)0;
  }
  for (int t = tid; t < BS; t += NT) fac[sbase + (int64_t)(2 * kLU) * BS + t] = piv[t];
}

// This thread's share of p[0..n) in a workgroup of NT threads: the sum of
// p[c] over c = t, t + NT, ... in increasing c, its loads issued eight at a
// time (a rolled loop would wait for each load before the next).
template <int NT, class TV>
__device__ inline TV strided_sum(const TV *__restrict__ p, int n) {
  TV s = 0;
  int c = threadIdx.x;
  for (; c + 7 * NT < n; c += 8 * NT) {
    TV v[8];
#pragma unroll
    for (int i = 0; i < 8; i++) v[i] = p[c + i * NT];
#pragma unroll
    for (int i = 0; i < 8; i++) s += v[i];
  }
  for (; c < n; c += NT) s += p[c];
  return s;
}

// Sum over an NT-thread workgroup; every thread gets the result.
template <int NT, class TV>
__device__ inline TV block_sum_n(TV v, TV *sh) {
  const int t = threadIdx.x;
  for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
  if ((t & 63) == 0) sh[t >> 6] = v;
  __syncthreads();
  TV s = 0;
#pragma unroll
  for (int w = 0; w < NT / 64; w++) s += sh[w];
  __syncthreads();
  return s;
}

// ---------------------------------------------------------------- coarse right-hand side
// The coarse correction acts on what the block-Jacobi sweeps leave:
//   w = w_bj + P z,  z = Ac^-1 R (r - A w_bj)   (w_bj = BJ^-1 r)
// with R the block sums and P the blocks' constant prolongation (coarse.hip).
// R A w_bj needs no second matvec: row j of block b meets R A only in the
// few blocks its column of A reaches, C[q][j] = sum of A_ij over the rows i of
// neighbour block q, so the workgroup that has just swept block b sums its
// contributions C[q][.] w_bj to every neighbour q and stores each in a slot of
// the receiving block that nobody else writes (no atomics, a fixed order).
// A block's own column sums (q = itself, all its rows) are one coalesced value
// per row; the others are listed by neighbour, each neighbour's list padded to
// teams of 8 lanes (kCoarsePad).
constexpr int kCQ = 32;  // neighbour blocks of a block (itself included)
constexpr uint16_t kCoarsePad = 0xffff;
// Teams a block's lists may hold: rows of 27 entries in 27 lists, each list's
// last team short.  (Rows of up to 32 entries, scattered over a block's 32
// neighbours, could need more: the set-up counts them, build_coarse.)
constexpr int coarse_teams(int bs) { return bs * 27 / 8 + kCQ; }
struct CoarseRestrict {
  const double *cown = nullptr;    // nblocks*bs: the own block's column sums
  const int32_t *eptr = nullptr;   // nblocks+1: first list entry of each block (multiples of 8)
  const uint16_t *cent = nullptr;  // list entries: row of the block | neighbour << 9
  const double *cval = nullptr;    // their column sums
  const uint16_t *tq = nullptr;    // nblocks*(kCQ+1): first 8-entry team of each neighbour
  const uint8_t *ownq = nullptr;   // nblocks: the own block's place among the neighbours
  const int32_t *wdst = nullptr;   // nblocks*kCQ: where the contribution to neighbour q goes in rcs (-1 none)
  const uint8_t *gsl = nullptr;    // nblocks*kCQ: which of the groups the block reaches neighbour q is in (255 none)
  const int32_t *w2dst = nullptr;  // nblocks*kCQ: where the sum over its s-th group goes in r2c (-1 none)
  double *rcs = nullptr;           // nblocks*kCQ: received contributions; nullptr: no coarse correction
  double *r2c = nullptr;           // received contributions by group
};

// Per-neighbour sums of a block: thread q < kCQ returns the sum of neighbour q
// (the own block's: of `own` over the workgroup; another's: of value(e) over
// its list of ne entries, teams i0 .. i1-1).  Every thread calls it; one
// barrier inside.
template <int BS, class F>
__device__ inline double coarse_block_sums(int ne, int i0, int i1, bool ownq, int t, double own, F &&value) {
  __shared__ double tm[coarse_teams(BS)];
  __shared__ double ow[BS / 64];
  for (int off = 32; off > 0; off >>= 1) own += __shfl_down(own, off, 64);
  if ((t & 63) == 0) ow[t >> 6] = own;
  for (int e = t; e < ne; e += BS) {  // ne is a multiple of 8: a team's lanes stay together
    double v = value(e);
    v += __shfl_xor(v, 1, 64);
    v += __shfl_xor(v, 2, 64);
    v += __shfl_xor(v, 4, 64);
    if ((t & 7) == 0) tm[e >> 3] = v;
  }
  __syncthreads();
  double s = 0.0;
  if (t < kCQ) {
    for (int i = i0; i < i1; i++) s += tm[i];
    if (ownq) {
#pragma unroll
      for (int w = 0; w < BS / 64; w++) s += ow[w];
    }
  }
  return s;
}

// What a thread of block b reads for its part of the coarse right-hand side:
// its row's own column sum, its first list entries, and (thread q < kCQ)
// neighbour q's teams and destinations.
template <int BS>
struct CoarseRegs {
  static constexpr int PRE = BS == 64 ? 4 : 2;  // list entries held (a whole brick's has up to 5 or 2 per thread)
  int e0, ne;
  double own, val[PRE];
  unsigned ent[PRE];
  int i0 = 0, i1 = 0, dst = -1, dst2 = -1, grp = 255;
  bool ownq = false;
};
template <int BS>
__device__ inline void coarse_load(const CoarseRestrict &R, int b, int t, CoarseRegs<BS> &c) {
  c.e0 = R.eptr[b];
  c.ne = R.eptr[b + 1] - c.e0;
  c.own = R.cown[(int64_t)b * BS + t];
#pragma unroll
  for (int k = 0; k < CoarseRegs<BS>::PRE; k++) {
    const bool in = t + k * BS < c.ne;
    c.val[k] = in ? R.cval[c.e0 + t + k * BS] : 0.0;
    c.ent[k] = in ? R.cent[c.e0 + t + k * BS] : kCoarsePad;
  }
  if (t < kCQ) {
    c.i0 = R.tq[b * (kCQ + 1) + t];
    c.i1 = R.tq[b * (kCQ + 1) + t + 1];
    c.ownq = t == R.ownq[b];
    c.dst = R.wdst[b * kCQ + t];
    c.dst2 = R.w2dst[b * kCQ + t];
    c.grp = R.gsl[b * kCQ + t];
  }
}

// After the sweeps (x: w_bj of the block, rr: the block sum of its right-hand
// side): the block's contributions to R (r - A w_bj), per neighbour block and
// summed per neighbour group.  Every thread calls it.
template <class TV, int BS>
__device__ inline void coarse_scatter(const CoarseRestrict &R, const CoarseRegs<BS> &c, const TV *x, const double &rr,
                                      int b, int t) {
  __shared__ double qv[kCQ];
  __shared__ uint8_t qg[kCQ];
  constexpr int PRE = CoarseRegs<BS>::PRE;
  const double s = coarse_block_sums<BS>(c.ne, c.i0, c.i1, c.ownq, t, c.own * (double)x[t], [&](int e) {
    double v = 0.0;
    unsigned w = kCoarsePad;
    bool held = false;
#pragma unroll
    for (int k = 0; k < PRE; k++)
      if (e == t + k * BS) { v = c.val[k]; w = c.ent[k]; held = true; }
    if (!held) { v = R.cval[c.e0 + e]; w = R.cent[c.e0 + e]; }
    return v * (double)x[w == kCoarsePad ? BS : w & 511];  // x[BS] is 0
  });
  if (t < kCQ) {
    const double v = (c.ownq ? rr : 0.0) - s;
    if (c.dst >= 0) R.rcs[c.dst] = v;
    qv[t] = v;
    qg[t] = (uint8_t)c.grp;
    wave_lds_fence();  // one wavefront
    if (c.dst2 >= 0) {
      double g = 0.0;
#pragma unroll
      for (int q = 0; q < kCQ; q++) g += qg[q] == t ? qv[q] : 0.0;
      R.r2c[c.dst2] = g;
    }
  }
}

// Block sum of the right-hand side x, left in LDS (rr) by thread 0; the
// sweeps' barriers come before its use.
template <class TV, int BS>
__device__ inline void restrict_block(const TV *x, double &rr, int t) {
  __shared__ TV sh[BS / 64];
  const TV s = block_sum_n<BS>(x[t], sh);
  if (t == 0) rr = (double)s;
}

// The same, and in the same pass the block sum of v (this thread's entry of
// the basis vector) into rv[b].
template <class TV, int BS>
__device__ inline void restrict_block2(const TV *x, double &rr, TV v, double *rv, int b, int t) {
  __shared__ TV sh[2][BS / 64];
  TV a = x[t];
  for (int off = 32; off > 0; off >>= 1) {
    a += __shfl_down(a, off, 64);
    v += __shfl_down(v, off, 64);
  }
  if ((t & 63) == 0) {
    sh[0][t >> 6] = a;
    sh[1][t >> 6] = v;
  }
  __syncthreads();
  if (t == 0) {
    TV s = 0, q = 0;
#pragma unroll
    for (int w = 0; w < BS / 64; w++) {
      s += sh[0][w];
      q += sh[1][w];
    }
    rr = (double)s;
    rv[b] = (double)q;
  }
  __syncthreads();
}

// ---------------------------------------------------------------- ILU(0) apply: y = (LU)^-1 r
// Forward and backward sweeps over the block's levels with x (BS+1 entries,
// x[BS] == 0 the target of padded slots) in LDS.  Every thread of the block
// must call this; x[t] holds the right-hand side on entry and the solution on
// return.
//
// A chain's rows are one level: each forms its right-hand side less the other
// chains' products, and the recurrence along the chain, s_t += a_t s_(t-1), is
// three register-shift steps with the products of consecutive a_t (a_t = 0 at
// a chain's first row), formed once beside the loads.
//
// Between two barriers of a level stand LDS reads, the row's products and one
// LDS write: on grids too small to hide it, that chain is the kernel's time,
// so the products go into four sums (levels of thirteen dependent
// multiply-adds: 1M cells 106.7 -> 101.4 us; by chains of rows instead of rows
// 101.4 -> 89.4, FP32 at 442,368 rows 31.6 -> 22.9, 46k rows 19.0 -> 15.5; means
// over a solve's launches, those that return at once past its end among them.
// The launches that work take 110 us at 1M rows, 4.5 TB/s).
template <class TV>
struct SweepRegs {  // a thread's row: factor entries and their local columns
  TV vl[kLU], vu[kLU], dinv;
  TV al[3], au[3];  // products of 1, 2, 4 consecutive chain couplings
  uint16_t cl[kLU], cu[kLU];
  int levL, levU, nL, nU;
};
// v of the lane N before (row_shr) or after (row_shl) within 16 lanes, else 0
template <int CTRL>
__device__ inline float lane_shift(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, true));
}
template <int CTRL>
__device__ inline double lane_shift(double v) {
  const uint64_t u = __double_as_longlong(v);
  const uint32_t lo = __builtin_amdgcn_update_dpp(0, (int)u, CTRL, 0xf, 0xf, true);
  const uint32_t hi = __builtin_amdgcn_update_dpp(0, (int)(u >> 32), CTRL, 0xf, 0xf, true);
  return __longlong_as_double((long long)((uint64_t)hi << 32 | lo));
}
constexpr int kShr = 0x110, kShl = 0x100;  // + lanes
template <int DIR, class TV>
__device__ inline TV chain_solve(TV s, const TV (&a)[3]) {
  s += a[0] * lane_shift<DIR + 1>(s);
  s += a[1] * lane_shift<DIR + 2>(s);
  s += a[2] * lane_shift<DIR + 4>(s);
  return s;
}
template <class TV, int BS>
__device__ inline void bj_sweeps_load(const BJLayout &L, const TV *__restrict__ fac, int b, int t, SweepRegs<TV> &r) {
  const int pb = L.d_pat ? L.d_pat[b] : b;  // index tables of the block's pattern
  const int64_t base = (int64_t)pb * BS;
  const int64_t sbase = (int64_t)b * kW * BS;
  const int64_t cbase = (int64_t)pb * kLU * BS;
  const int nlu = L.d_nlu ? L.d_nlu[pb] : kLU;  // slots past it hold 0 against the zero entry x[BS]
#pragma unroll
  for (int p = 0; p < kLU; p++) {
    const bool in = p < nlu;
    r.vl[p] = in ? fac[sbase + (int64_t)p * BS + t] : (TV)0;
    r.vu[p] = in ? fac[sbase + (int64_t)(kLU + p) * BS + t] : (TV)0;
    r.cl[p] = in ? L.d_cL[cbase + (int64_t)p * BS + t] : (uint16_t)BS;
    r.cu[p] = in ? L.d_cU[cbase + (int64_t)p * BS + t] : (uint16_t)BS;
  }
  r.dinv = fac[sbase + (int64_t)(2 * kLU) * BS + t];
  const int wl = L.d_swL[base + t], wu = L.d_swU[base + t];
  r.nL = L.d_nsw[2 * pb];
  r.nU = L.d_nsw[2 * pb + 1];
  r.levL = wl & ~kChainLink;
  r.levU = wu & ~kChainLink;
  // the chain's couplings leave the products: slot 0 is the nearest column
  const bool ll = wl & kChainLink, lu = wu & kChainLink;
  r.al[0] = ll ? -r.vl[0] : (TV)0;
  r.au[0] = lu ? -r.vu[0] * r.dinv : (TV)0;
  r.vl[0] = ll ? (TV)0 : r.vl[0];
  r.vu[0] = lu ? (TV)0 : r.vu[0];
  r.cl[0] = ll ? (uint16_t)BS : r.cl[0];
  r.cu[0] = lu ? (uint16_t)BS : r.cu[0];
  r.al[1] = r.al[0] * lane_shift<kShr + 1>(r.al[0]);
  r.al[2] = r.al[1] * lane_shift<kShr + 2>(r.al[1]);
  r.au[1] = r.au[0] * lane_shift<kShl + 1>(r.au[0]);
  r.au[2] = r.au[1] * lane_shift<kShl + 2>(r.au[1]);
}
// x - sum v[p] x[c[p]], the products in four sums
template <class TV>
__device__ inline TV sweep_row(const TV *x, TV s, const TV (&v)[kLU], const uint16_t (&c)[kLU]) {
  TV xv[kLU];
#pragma unroll
  for (int p = 0; p < kLU; p++) xv[p] = x[c[p]];
  TV q[4] = {s, (TV)0, (TV)0, (TV)0};
#pragma unroll
  for (int p = 0; p < kLU; p++) q[p & 3] -= v[p] * xv[p];
  return (q[0] + q[1]) + (q[2] + q[3]);
}
template <class TV, int BS>
__device__ inline void bj_sweeps_run(const SweepRegs<TV> &r, TV *x, int t) {
  __syncthreads();
  // forward: branch-free inner loop, all LDS reads of a level in flight together
  for (int l = 0; l < r.nL; l++) {
    if (r.levL == l) x[t] = chain_solve<kShr>(sweep_row(x, x[t], r.vl, r.cl), r.al);
    __syncthreads();
  }
  for (int l = 0; l < r.nU; l++) {
    if (r.levU == l) x[t] = chain_solve<kShl>(sweep_row(x, x[t], r.vu, r.cu) * r.dinv, r.au);
    __syncthreads();
  }
}
template <class TV, int BS>
__device__ inline void bj_sweeps(const BJLayout &L, const TV *__restrict__ fac, TV *x, int b, int t) {
  SweepRegs<TV> r;
  bj_sweeps_load<TV, BS>(L, fac, b, t, r);
  bj_sweeps_run<TV, BS>(r, x, t);
}

template <class TV, int BS>
__global__ void __launch_bounds__(BS) k_bj_apply(BJLayout L, const TV *__restrict__ fac, const TV *__restrict__ r,
                                                 TV *__restrict__ y, const int *__restrict__ stop = nullptr,
                                                 CoarseRestrict cr = CoarseRestrict{}) {
  __shared__ TV x[BS + 1];
  __shared__ double rr;
  if (stop && *stop) return;  // uniform over the workgroup
  const int b = blockIdx.x, t = threadIdx.x;
  const int row = L.d_row[(int64_t)b * BS + t];
  x[t] = row >= 0 ? r[row] : (TV)0;
  if (t == 0) x[BS] = (TV)0;
  if (cr.rcs) restrict_block<TV, BS>(x, rr, t);  // cr is uniform
  bj_sweeps<TV, BS>(L, fac, x, b, t);
  if (row >= 0) y[row] = x[t];
  if (cr.rcs) {
    CoarseRegs<BS> cg;
    coarse_load<BS>(cr, b, t, cg);
    coarse_scatter<TV, BS>(cr, cg, x, rr, b, t);
  }
}

// ---------------------------------------------------------------- block-ordered SpMV
// The solver's Jacobian is stored block-contiguous over the block layout:
// slot k of position p = b*bs + t at a[(b*W + k)*bs + t], its global column at
// the same place of ecol (or of the block pattern's table, see ecol_addr);
// the global row of p is L.d_row[p] (-1 for padding positions).

// Column of slot k at block position p: an int32 global column, or an int16
// offset from the row (used when every offset of the mesh fits, which halves
// the index bytes of every SpMV).
template <class TI>
__device__ inline int blk_col(const TI *__restrict__ ecol, int64_t q, int row) {
  if (sizeof(TI) == 2) return row + (int)ecol[q];
  return (int)ecol[q];
}

// UNROLL: issue a hexahedral row's 27 loads at once (more registers, more
// memory-level parallelism); worth it where occupancy is set by other phases.
// Slot k's column index sits at ecol[eb + k*es]: eb = p, es = NB in the
// slot-major layout; eb = (pattern*W)*bs + t, es = bs with shared patterns.
template <class TV, class TI, bool UNROLL = (sizeof(TV) == 4)>
__device__ inline TV blk_row(int64_t ab, int64_t as, int W, int row, const TI *__restrict__ ecol, int64_t eb,
                             int64_t es, const TV *__restrict__ a, const TV *__restrict__ x) {
  TV s = 0;
  if (UNROLL && W == kW) {
    int c[kW];
    TV v[kW];
#pragma unroll
    for (int k = 0; k < kW; k++) {
      c[k] = blk_col(ecol, eb + k * es, row);
      v[k] = a[ab + k * as];
    }
#pragma unroll
    for (int k = 0; k < kW; k++) s += v[k] * x[c[k]];
  } else {
    for (int k = 0; k < W; k++) s += a[ab + k * as] * x[blk_col(ecol, eb + k * es, row)];
  }
  return s;
}

// The solver's ELL arrays (Jacobian values, column indices, coarse slot
// map) are block-contiguous: slot k of position p = b*bs + t (block b, row t
// of the block) at (b*W + k)*bs + t, so a block's W slots are one contiguous
// run of W*bs entries (one DRAM stream per workgroup instead of W streams
// NB apart).  Index tables shared by the blocks of one pattern sit at
// (pattern*W + k)*bs + t.
__device__ inline int64_t ell_base(int64_t p, int bs, int W) {
  const int64_t b = p / bs;
  return (b * W) * bs + (p - b * bs);
}

// Base and stride of block position p's column indices (see blk_row).
__device__ inline void ecol_addr(const int32_t *__restrict__ pat, int bs, int W, int64_t p, int64_t &eb, int64_t &es) {
  if (pat) {
    const int64_t b = p / bs;
    eb = ((int64_t)pat[b] * W) * bs + (p - b * bs);
  } else {
    eb = ell_base(p, bs, W);
  }
  es = bs;
}

// y[row(p)] = (A x)[row(p)]
template <class TV, class TI>
__global__ void __launch_bounds__(256) k_spmv_blk(int64_t NB, int W, const int32_t *__restrict__ rowof,
                                                  const TI *__restrict__ ecol, const int32_t *__restrict__ pat,
                                                  int bs, const int32_t *__restrict__ bw, const TV *__restrict__ a,
                                                  const TV *__restrict__ x, TV *__restrict__ y,
                                                  const int *__restrict__ stop = nullptr) {
  if (stop && *stop) return;
  const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= NB) return;
  const int row = rowof[p];
  if (row < 0) return;
  int64_t eb, es;
  ecol_addr(pat, bs, W, p, eb, es);
  y[row] = blk_row<TV, TI, true>(ell_base(p, bs, W), bs, bw ? bw[p / bs] : W, row, ecol, eb, es, a, x);
}

// Arnoldi column j: Hessenberg entries from h[0..j] (dots) and hj1 = h[j+1]
// (||w||^2), previous Givens rotations, the new rotation, residual estimate
// and stop test.  Rotation i turns (entry i, entry i+1) into (final entry i,
// the entry i+1 that rotation i+1 reads), so the running entry stays in a
// register and nothing written is read back from memory.
// hr, csr, snr: where h[0..j], cs[0..j-1] and sn[0..j-1] are read (the
// arrays themselves, or copies in LDS); cs[j] and sn[j] are written to cs, sn.
__device__ inline void arnoldi_update(GmresDev *gd, int j, int m, const double *hr, double hj1,
                                      double *__restrict__ H, double *__restrict__ cs, double *__restrict__ sn,
                                      double *__restrict__ g, const double *csr, const double *snr) {
  const int ld = m + 1;
  const double hn = sqrt(hj1);
  double a = hr[0];
  for (int i = 0; i < j; i++) {
    const double c = hr[i + 1], ci = csr[i], si = snr[i];
    H[i + j * ld] = ci * a + si * c;
    a = -si * a + ci * c;
  }
  const double c = hn;
  const double d = sqrt(a * a + c * c);
  const double csj = d > 0 ? a / d : 1.0, snj = d > 0 ? c / d : 0.0;
  cs[j] = csj;
  sn[j] = snj;
  H[j + j * ld] = d;
  H[j + 1 + j * ld] = 0.0;
  const double gj = g[j], gj1 = -snj * gj;
  g[j + 1] = gj1;
  g[j] = csj * gj;
  const int its = gd->its + 1;
  gd->its = its;
  gd->jcur = j + 1;
  const double resid = fabs(gj1);
  gd->resid = resid;
  gd->inv_h = hn > 0.0 ? 1.0 / hn : 0.0;
  const bool bad = !isfinite(resid) || !isfinite(hn);
  const int conv = !bad && (resid <= gd->tol || hn == 0.0);
  gd->converged = conv;
  if (bad) gd->diverged = 1;
  const bool fin = conv || bad || its >= gd->maxit;  // finished is 0 on entry (the step runs only while not done)
  if (fin) gd->finished = 1;
  if (fin || j + 1 == m) gd->done = 1;
}

// ---------------------------------------------------------------- fused Arnoldi matvec
// The previous Arnoldi column, finished inside the next matvec (NORM mode):
// ||u||^2 is the sum of the nchunk norm partials, reduced by every workgroup
// in the same fixed order; workgroup 0 also stores it and runs the Givens
// update of column j.
struct NormArgs {
  const void *part = nullptr;
  int nchunk = 0, j = 0, m = 0;
  double *h = nullptr, *H = nullptr, *cs = nullptr, *sn = nullptr, *g = nullptr;
};

// One GMRES step's  V_j = s u  and  out = M^-1 A V_j = s M^-1 A u  (s = 1/||u||
// read on the device, or with NORM formed here from the norm partials of the
// previous step): the block's rows of A u go straight into LDS and the
// triangular sweeps follow, so neither A u nor a separate scaling pass
// touches HBM; while some workgroups sweep their levels, others stream their
// rows of A.  u and out must be different vectors.
//
// EARLY (grids of at most two waves per SIMD, kEarlyWaves): the factor, the
// schedule and the coarse lists are loaded before the product instead of
// after it, in registers a larger grid needs for its occupancy: 46k rows 20.0 ->
// 19.0 us, 63k 20.9 -> 19.7, 4k in 64-row blocks 10.3 -> 9.5 (with the four sums).
constexpr int kEarlyWaves = 2048;
template <class TV, int BS, class TI, bool NORM, bool EARLY>
__global__ void __launch_bounds__(BS) __attribute__((amdgpu_waves_per_eu(EARLY ? 2 : 4))) k_bj_spmv_apply(BJLayout L, int64_t NB, int W, const TI *__restrict__ ecol,
                                                      const TV *__restrict__ a, const TV *__restrict__ u,
                                                      GmresDev *__restrict__ gd, TV *__restrict__ vj,
                                                      const TV *__restrict__ fac, TV *__restrict__ out,
                                                      const int *__restrict__ stop, CoarseRestrict cr,
                                                      NormArgs na, double *__restrict__ rv) {
  __shared__ TV x[BS + 1];
  __shared__ double rr;
  __shared__ TV shn[BS / 64];
  __shared__ int stop_s;
  const int b = blockIdx.x, t = threadIdx.x;
  SweepRegs<TV> sr;
  if (EARLY) bj_sweeps_load<TV, BS>(L, fac, b, t, sr);
  TV sc;
  if (NORM) {
    // workgroup 0 of this same launch may set the stop flag: read it once
    if (t == 0) stop_s = stop ? *stop : 0;
    __syncthreads();
    if (stop_s) return;  // uniform over the workgroup
    const TV *part = static_cast<const TV *>(na.part);
    TV s = 0;
    s = strided_sum<BS>(part, na.nchunk);
    s = block_sum_n<BS>(s, shn);
    const double hn = sqrt((double)s);
    sc = (TV)(hn > 0.0 ? 1.0 / hn : 0.0);
    if (b == 0 && t == 0) {
      na.h[na.j + 1] = (double)s;
      arnoldi_update(gd, na.j, na.m, na.h, (double)s, na.H, na.cs, na.sn, na.g, na.cs, na.sn);
    }
  } else {
    if (stop && *stop) return;  // uniform over the workgroup
    sc = (TV)gd->inv_h;
  }
  const int64_t p = (int64_t)b * BS + t;
  const int row = L.d_row[p];
  // the sweeps below hold ~100 registers anyway: the unrolled row costs no occupancy here
  int64_t eb, es;
  ecol_addr(L.d_pat, BS, W, p, eb, es);
  const int wb = L.d_bw ? L.d_bw[b] : W;  // slots past the block's longest row are padding
  x[t] = row >= 0 ? sc * blk_row<TV, TI, true>(((int64_t)b * W) * BS + t, BS, wb, row, ecol, eb, es, a, u) : (TV)0;
  const TV vv = row >= 0 ? sc * u[row] : (TV)0;
  if (row >= 0) vj[row] = vv;
  if (t == 0) x[BS] = (TV)0;
  // cr is uniform; rv: the block sums of V_j, for the coarse terms of the multi-dot
  if (cr.rcs) restrict_block2<TV, BS>(x, rr, vv, rv, b, t);
  if (!EARLY) bj_sweeps_load<TV, BS>(L, fac, b, t, sr);
  CoarseRegs<BS> cg;
  if (EARLY && cr.rcs) coarse_load<BS>(cr, b, t, cg);
  bj_sweeps_run<TV, BS>(sr, x, t);
  if (row >= 0) out[row] = x[t];
  if (!EARLY && cr.rcs) coarse_load<BS>(cr, b, t, cg);
  if (cr.rcs) coarse_scatter<TV, BS>(cr, cg, x, rr, b, t);
}

// A restart's preconditioned residual out = M_BJ^-1 (b - J y) in one pass:
// the block's rows of b - J y (FP64, the difference taken in FP64 and then
// rounded to TV, as a separate product and difference would give) go into
// LDS, the sweeps follow, and the block's part of the coarse right-hand side
// when the coarse correction is on.
template <class TV, int BS, class TI>
__global__ void __launch_bounds__(BS) __attribute__((amdgpu_waves_per_eu(4))) k_bj_resid_apply(BJLayout L, int W, const TI *__restrict__ ecol,
                                                       const double *__restrict__ J, const double *__restrict__ y,
                                                       const double *__restrict__ bvec, const TV *__restrict__ fac,
                                                       TV *__restrict__ out, const int *__restrict__ stop,
                                                       CoarseRestrict cr) {
  __shared__ TV x[BS + 1];
  __shared__ double rr;
  if (stop && *stop) return;  // uniform over the workgroup
  const int b = blockIdx.x, t = threadIdx.x;
  const int64_t p = (int64_t)b * BS + t;
  const int row = L.d_row[p];
  int64_t eb, es;
  ecol_addr(L.d_pat, BS, W, p, eb, es);
  const int wb = L.d_bw ? L.d_bw[b] : W;
  x[t] = row >= 0 ? (TV)(bvec[row] - blk_row<double, TI, true>(((int64_t)b * W) * BS + t, BS, wb, row, ecol, eb, es, J, y))
                  : (TV)0;
  if (t == 0) x[BS] = (TV)0;
  if (cr.rcs) restrict_block<TV, BS>(x, rr, t);  // cr is uniform
  bj_sweeps<TV, BS>(L, fac, x, b, t);
  if (row >= 0) out[row] = x[t];
  if (cr.rcs) {
    CoarseRegs<BS> cg;
    coarse_load<BS>(cr, b, t, cg);
    coarse_scatter<TV, BS>(cr, cg, x, rr, b, t);
  }
}

// ---------------------------------------------------------------- BLAS-1 with deterministic reductions
constexpr int kRedBlock = 256;
constexpr int kRedPerThread = 2;
constexpr int kChunk = kRedBlock * kRedPerThread;
// Rows per thread of the multi-vector kernels.  (Four FP32 rows per thread,
// to match FP64's bytes in flight, halves the workgroups and measured slower:
// multi-dot 27 -> 30 us, update 14.5 -> 21 us at 1M rows.)
template <class TV>
struct Red {
  static constexpr int E = kRedPerThread;
  static constexpr int chunk = kRedBlock * E;
};

template <class TV>
__device__ inline TV block_sum(TV v, TV *sh) {
  const int t = threadIdx.x;
  for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
  if ((t & 63) == 0) sh[t >> 6] = v;
  __syncthreads();
  TV s = 0;
  if (t == 0)
    for (int w = 0; w < kRedBlock / 64; w++) s += sh[w];
  __syncthreads();
  return s;
}

// Sum of 32 per-lane values over a wavefront by recursive halving: at each
// step a lane keeps one half of its values, adds the partner's copy of that
// half and hands over the other half (16 + 8 + 4 + 2 + 1 exchanges), then one
// more exchange completes the pair.  Afterwards lanes 2j and 2j+1 both hold
// the wavefront sum of value j.
template <int HALF, class TV>
__device__ inline void halve_step(TV (&v)[32], int lane) {
  const bool upper = (lane & (2 * HALF)) != 0;
#pragma unroll
  for (int k = 0; k < HALF; k++) {
    const TV send = upper ? v[k] : v[HALF + k];
    const TV keep = upper ? v[HALF + k] : v[k];
    v[k] = keep + __shfl_xor(send, 2 * HALF, 64);
  }
}

// NS (8, 16 or 32) values: the halving steps use lane bits log2(NS)..1, so
// value j ends in lanes with (lane >> 1) % NS == j; the lane bits left over
// (bit 0, and bits 5 / 4 for fewer values) are summed by plain exchanges.
template <int NS, class TV>
__device__ inline TV wave_reduce_scatter(TV (&v)[32]) {
  const int lane = threadIdx.x & 63;
  if (NS >= 32) halve_step<16>(v, lane);
  if (NS >= 16) halve_step<8>(v, lane);
  halve_step<4>(v, lane);
  halve_step<2>(v, lane);
  halve_step<1>(v, lane);
  TV r = v[0] + __shfl_xor(v[0], 1, 64);
  if (NS <= 16) r += __shfl_xor(r, 32, 64);
  if (NS <= 8) r += __shfl_xor(r, 16, 64);
  return r;
}

// The coarse solve run by the first `parts` workgroups of a multi-dot launch
// (0: none), with their terms of the dots.
struct CoarseDot {
  int parts = 0;                                // parts of the groups, in group order
  int ng = 0, gsz = 0, g2max = 0;               // groups, blocks of a group, entries of r2c of a group (at most)
  int nov = 0;                                  // columns of G1 (0: level 2 alone)
  const int32_t *gmem = nullptr;                // ng*gsz blocks of each group (-1 pad)
  const int32_t *gov = nullptr;                 // ng*nov blocks of each group with its overlap (-1 pad)
  const double *G1 = nullptr, *M = nullptr;     // group and level-2 parts of the coarse inverse (coarse.hip)
  const double *rcs = nullptr, *r2c = nullptr;  // contributions to the restricted residual, by block and by group
  const int32_t *g2ptr = nullptr;               // ng+1: each group's entries of r2c
  const double *RV = nullptr;                   // block sums of the basis vectors, rv_ld per vector
  int64_t rv_ld = 0;
  double *z1 = nullptr;                         // coarse correction per block (out)
};
template <class TV>
__device__ void coarse_level1_dots(const CoarseDot &cd, int part, int nv, TV *partial, int pstride);

// Coarse prolongation applied on the fly: w[i] += z1[pos[i] >> bs_log2]
// (pos = block-layout position of row i).  z1 == nullptr: none.
struct Prolong {
  const double *z1 = nullptr;
  const int32_t *pos = nullptr;
  int bs_log2 = 0;
};

// Two adjacent rows per lane, read as one 16-byte (FP64) or 8-byte (FP32)
// access when the rows' addresses allow it (ldv and the row even); the last
// odd row of a vector is read alone.
template <class TV> struct Pair2;
template <> struct Pair2<double> { using T = double2; };
template <> struct Pair2<float> { using T = float2; };
template <class TV>
__device__ inline void load2(const TV *__restrict__ p, int64_t r, int64_t n, bool vec, TV &a, TV &b) {
  if (vec && r + 1 < n) {
    const typename Pair2<TV>::T q = *reinterpret_cast<const typename Pair2<TV>::T *>(p + r);
    a = q.x;
    b = q.y;
  } else {
    a = r < n ? p[r] : (TV)0;
    b = r + 1 < n ? p[r + 1] : (TV)0;
  }
}

// The row pairs (r, r + 1) of vectors V_j0 .. V_j0+cnt-1 (cnt <= NS, the
// same for the whole workgroup) passed to f(j, a, b) in order.  The loads
// carry only workgroup-uniform guards, so all of them are issued before the
// first product instead of one at a time.  The chunk must hold both rows and
// the pair be aligned (ldv and r even).
template <class TV, int NS, class F>
__device__ inline void load_pairs(const TV *__restrict__ V, int64_t ldv, int64_t r, int j0, int cnt, F &&f) {
  using P = typename Pair2<TV>::T;
  const TV *p = V + (int64_t)j0 * ldv + r;
  P q[NS];
#pragma unroll
  for (int j = 0; j < NS; j++)
    if (j < cnt) q[j] = *reinterpret_cast<const P *>(p + (int64_t)j * ldv);
#pragma unroll
  for (int j = 0; j < NS; j++)
    if (j < cnt) f(j, q[j].x, q[j].y);
}

// The rows r and r + 1 of vectors V_j0 .. V_j0+cnt-1 (cnt <= NS, the same for
// the whole workgroup): `load` issues every load before the first one is
// waited for, which a loop over vectors of runtime count, or one whose loads
// sit behind per-lane bounds checks, does not.  Rows past the end read the last
// rows instead; the caller drops what becomes of them.
template <class TV, int NS>
struct VecRows {
  using P = typename Pair2<TV>::T;
  P q[NS];
  __device__ inline void load(const TV *__restrict__ V, int64_t ldv, int64_t n, int64_t r, int j0, int cnt) {
    const TV *p = V + (int64_t)j0 * ldv;
    if (((ldv | n) & 1) == 0) {  // pairs aligned: one access each
      p += min(r, n - 2);
#pragma unroll
      for (int j = 0; j < NS; j++)
        if (j < cnt) q[j] = *reinterpret_cast<const P *>(p + (int64_t)j * ldv);
    } else {
      const int64_t ra = min(r, n - 1), rb = min(r + 1, n - 1);
#pragma unroll
      for (int j = 0; j < NS; j++)
        if (j < cnt) {
          q[j].x = p[(int64_t)j * ldv + ra];
          q[j].y = p[(int64_t)j * ldv + rb];
        }
    }
  }
};

// partial[j*nchunk + chunk] = <w, V_j> over the chunk, j = 0..nv-1.  Each
// thread holds two adjacent rows and accumulates up to NS dots in registers;
// one reduce-scatter per wavefront and one barrier per group of NS vectors
// finish the chunk.
//
// BATCH (FP64 on small grids, kBatchGrid): the NS vectors' loads in flight
// together, in registers that cost a large grid its occupancy.
//
// COARSE: the launch's first cd.parts workgroups run the coarse solve; its
// registers would set the occupancy of the row chunks at NS <= 16 (74), so
// the budget is held to 7 waves per SIMD there, except on small grids.
template <class TV, int NS, bool COARSE, bool BATCH>
__global__ void __launch_bounds__(kRedBlock) __attribute__((amdgpu_waves_per_eu(COARSE && NS <= 16 && !BATCH ? 7 : 1))) k_mdot(int64_t n, int nv, const TV *__restrict__ V, int64_t ldv,
                                                    const TV *__restrict__ w, TV *__restrict__ partial, int nchunk,
                                                    const int *__restrict__ stop, CoarseDot cd) {
  static_assert(Red<TV>::E == 2, "two rows per thread");
  __shared__ TV red[kRedBlock / 64][NS];
  if (stop && *stop) return;
  // partial[j*nchunk + c]: c < cd.parts the coarse workgroups' terms, then one per row chunk
  if (COARSE && (int)blockIdx.x < cd.parts) {
    coarse_level1_dots<TV>(cd, blockIdx.x, nv, partial, nchunk);
    return;
  }
  const int chunk = blockIdx.x - cd.parts;
  const int t = threadIdx.x, lane = t & 63, wv_id = t >> 6;
  const int64_t r0 = (int64_t)chunk * Red<TV>::chunk + 2 * t;
  const bool vec = (ldv & 1) == 0;
  TV w0, w1;
  load2(w, r0, n, true, w0, w1);  // 0 past the end
  // FP32: every chunk but a ragged last one issues its NS loads together
  // (8-byte accesses: 22.4 -> 19.4 us at 1M rows).  A large FP64 grid keeps one
  // load at a time, which measured faster there (30.8 against 32.7 us): its
  // 16-byte loads already keep enough bytes in flight at the higher occupancy.
  const bool full = sizeof(TV) == 4 && vec && (int64_t)(chunk + 1) * Red<TV>::chunk <= n;
  for (int j0 = 0; j0 < nv; j0 += NS) {
    TV acc[32];
#pragma unroll
    for (int j = 0; j < 32; j++) acc[j] = 0;
    if (BATCH) {
      const int cnt = min(NS, nv - j0);
      VecRows<TV, NS> v;
      v.load(V, ldv, n, r0, j0, cnt);
#pragma unroll
      for (int j = 0; j < NS; j++)
        if (j < cnt) {
          acc[j] += w0 * v.q[j].x;
          acc[j] += w1 * v.q[j].y;
        }
    } else if (full) {
      load_pairs<TV, NS>(V, ldv, r0, j0, min(NS, nv - j0), [&](int j, TV v0, TV v1) {
        acc[j] += w0 * v0;
        acc[j] += w1 * v1;
      });
    } else {
#pragma unroll
      for (int j = 0; j < NS; j++) {
        if (j0 + j < nv) {
          TV v0, v1;
          load2(V + (int64_t)(j0 + j) * ldv, r0, n, vec, v0, v1);
          acc[j] += w0 * v0;
          acc[j] += w1 * v1;
        }
      }
    }
    const TV r = wave_reduce_scatter<NS>(acc);
    if ((lane & 1) == 0 && (lane >> 1) < NS) red[wv_id][lane >> 1] = r;
    __syncthreads();
    if (t < NS && j0 + t < nv) {
      TV s = 0;
#pragma unroll
      for (int q = 0; q < kRedBlock / 64; q++) s += red[q][t];
      partial[(int64_t)(j0 + t) * nchunk + cd.parts + chunk] = s;
    }
    __syncthreads();
  }
}

// out[j] = sum_c partial[j*nchunk + c] (fixed order)
template <class TV>
__global__ void k_reduce_partials(int nv, int nchunk, const TV *__restrict__ partial, double *__restrict__ out,
                                  const int *__restrict__ stop = nullptr) {
  __shared__ TV sh[kRedBlock / 64];
  if (stop && *stop) return;
  const int j = blockIdx.x;
  TV s = 0;
  s = strided_sum<kRedBlock>(partial + (int64_t)j * nchunk, nchunk);
  s = block_sum(s, sh);
  if (threadIdx.x == 0) out[j] = (double)s;
}

// w -= sum_j h[j] V_j ; partial[chunk] = ||w||^2 over the chunk (two
// adjacent rows per thread, as k_mdot).  DOTS: h itself is still the
// multi-dot's npart partials per vector; every workgroup sums them, eight
// lanes a vector in a fixed order, and workgroup 0 stores them for the
// Arnoldi update, so no launch of its own stands between the two kernels;
// the vectors' rows are on their way while it does.
constexpr int kMaxpyVecs = 200;  // basis vectors at most (the restart length)
template <class TV, bool DOTS>
__global__ void __launch_bounds__(kRedBlock) k_maxpy_norm(int64_t n, int nv, const TV *__restrict__ V, int64_t ldv,
                                                          double *__restrict__ h, TV *__restrict__ w,
                                                          TV *__restrict__ partial,
                                                          const int *__restrict__ stop = nullptr,
                                                          Prolong pro = Prolong{}, const TV *__restrict__ dots = nullptr,
                                                          int npart = 0) {
  __shared__ TV sh[kRedBlock / 64];
  __shared__ double hs[DOTS ? kMaxpyVecs : 1];
  if (stop && *stop) return;
  const int64_t r0 = (int64_t)blockIdx.x * Red<TV>::chunk + 2 * threadIdx.x;
  TV x0, x1;
  load2(w, r0, n, true, x0, x1);
  constexpr int NB = 32;
  VecRows<TV, DOTS ? NB : 1> q;
  if (DOTS) q.load(V, ldv, n, r0, 0, min(NB, nv));
  if (pro.z1) {  // the coarse prolongation
    if (r0 < n) x0 += (TV)pro.z1[pro.pos[r0] >> pro.bs_log2];
    if (r0 + 1 < n) x1 += (TV)pro.z1[pro.pos[r0 + 1] >> pro.bs_log2];
  }
  if (DOTS) {
    const int l = threadIdx.x % 8;
    for (int v = threadIdx.x / 8; v < nv; v += kRedBlock / 8) {
      const TV *p = dots + (int64_t)v * npart;
      TV s = 0;
      for (int c = l; c < npart; c += 64) {
        TV d[8];
#pragma unroll
        for (int u = 0; u < 8; u++) d[u] = c + 8 * u < npart ? p[c + 8 * u] : (TV)0;
#pragma unroll
        for (int u = 0; u < 8; u++) s += d[u];
      }
      s += __shfl_xor(s, 1, 64);
      s += __shfl_xor(s, 2, 64);
      s += __shfl_xor(s, 4, 64);
      if (l == 0) {
        hs[v] = (double)s;
        if (blockIdx.x == 0) h[v] = (double)s;
      }
    }
    __syncthreads();
  }
  if constexpr (DOTS) {
    for (int j0 = 0; j0 < nv; j0 += NB) {
      const int cnt = min(NB, nv - j0);
      if (j0 > 0) q.load(V, ldv, n, r0, j0, cnt);
#pragma unroll
      for (int j = 0; j < NB; j++)
        if (j < cnt) {
          const TV hj = (TV)hs[j0 + j];
          x0 -= hj * q.q[j].x;
          x1 -= hj * q.q[j].y;
        }
    }
  } else {
    const bool vec = (ldv & 1) == 0;
    for (int j = 0; j < nv; j++) {
      TV v0, v1;
      load2(V + (int64_t)j * ldv, r0, n, vec, v0, v1);
      const TV hj = (TV)h[j];
      x0 -= hj * v0;
      x1 -= hj * v1;
    }
  }
  TV s = 0;
  if (r0 + 1 < n) {
    *reinterpret_cast<typename Pair2<TV>::T *>(w + r0) = typename Pair2<TV>::T{x0, x1};
    s += x0 * x0;
    s += x1 * x1;
  } else if (r0 < n) {
    w[r0] = x0;
    s += x0 * x0;
  }
  s = block_sum(s, sh);
  if (threadIdx.x == 0) partial[blockIdx.x] = s;
}

// partial[chunk] = <x, y>
template <class TX, class TY>
__global__ void __launch_bounds__(kRedBlock) k_dot(int64_t n, const TX *__restrict__ x, const TY *__restrict__ y,
                                                   double *__restrict__ partial, const int *__restrict__ stop = nullptr) {
  __shared__ double sh[kRedBlock / 64];
  if (stop && *stop) return;
  const int64_t i0 = (int64_t)blockIdx.x * kChunk + threadIdx.x;
  double s = 0;
#pragma unroll
  for (int e = 0; e < kRedPerThread; e++) {
    const int64_t i = i0 + (int64_t)e * kRedBlock;
    if (i < n) s += (double)x[i] * (double)y[i];
  }
  s = block_sum(s, sh);
  if (threadIdx.x == 0) partial[blockIdx.x] = s;
}

template <class TV>
__global__ void k_scale_copy(int64_t n, TV a, const TV *__restrict__ x, TV *__restrict__ y) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) y[i] = a * x[i];
}

template <class TA, class TB>
__global__ void k_convert(int64_t n, const TA *__restrict__ a, TB *__restrict__ b) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) b[i] = (TB)a[i];
}

// dyn: the solver's device-resident parameters (SolverWS::dyn); cap: iterations
// this attempt gets at most.
__global__ void k_gmres_init(GmresDev *gd, int *status, const double *__restrict__ dyn, int cap) {
  gd->its = 0;
  gd->done = 0;
  gd->converged = 0;
  gd->finished = 0;
  gd->diverged = 0;
  gd->jcur = 0;
  gd->maxit = min((int)dyn[4], cap);
  *status = 0;
}

// Start of a cycle: beta = sqrt(h[0]) from a norm reduction; sets tol on the first cycle.
// After the solve has finished, a later cycle is empty: no columns, stop flag set.
__global__ void k_cycle_start(GmresDev *gd, const double *__restrict__ h, double *__restrict__ g, int m,
                              const double *__restrict__ dyn, int first) {
  if (!first && gd->finished) {
    gd->jcur = 0;
    gd->done = 1;
    return;
  }
  const double beta = sqrt(h[0]);
  if (first) gd->tol = fmax(dyn[2] * beta, dyn[3]);
  for (int i = 0; i <= m; i++) g[i] = 0.0;
  g[0] = beta;
  gd->resid = beta;
  gd->jcur = 0;
  gd->inv_h = beta > 0.0 ? 1.0 / beta : 0.0;
  const bool bad = !isfinite(beta);
  const int conv = !bad && !(beta > gd->tol);
  gd->converged = conv;
  if (bad) gd->diverged = 1;
  gd->finished = conv || bad || gd->its >= gd->maxit;
  gd->done = gd->finished;
}

// h[j+1] = sum of the nchunk norm partials (fixed order, as k_reduce_partials)
// and the Arnoldi/Givens update of column j, in one workgroup.
template <class TV>
__global__ void __launch_bounds__(kRedBlock) k_norm_arnoldi(int nchunk, const TV *__restrict__ partial, GmresDev *gd,
                                                            int j, int m, double *__restrict__ h,
                                                            double *__restrict__ H, double *__restrict__ cs,
                                                            double *__restrict__ sn, double *__restrict__ g) {
  __shared__ TV sh[kRedBlock / 64];
  __shared__ double hs[kRedBlock], css[kRedBlock], sns[kRedBlock];  // h, cs, sn read by the update
  if (gd->done) return;
  const int t = threadIdx.x;
  const bool staged = j < kRedBlock;  // the columns fit: the update reads them from LDS
  if (staged) {
    if (t <= j) hs[t] = h[t];
    if (t < j) { css[t] = cs[t]; sns[t] = sn[t]; }
  }
  TV s = 0;
  s = strided_sum<kRedBlock>(partial, nchunk);
  s = block_sum(s, sh);  // its barriers also order the LDS copies above
  if (t == 0) {
    h[j + 1] = (double)s;
    if (staged) arnoldi_update(gd, j, m, hs, (double)s, H, cs, sn, g, css, sns);
    else arnoldi_update(gd, j, m, h, (double)s, H, cs, sn, g, cs, sn);
  }
}

// y = H(1:j,1:j)^-1 g(1:j) for the j = jcur columns of the cycle
__global__ void k_hess_solve(GmresDev *gd, int m, const double *__restrict__ H, const double *__restrict__ g,
                             double *__restrict__ y) {
  const int ld = m + 1, j = gd->jcur;
  gd->jlast = j;
  for (int i = j - 1; i >= 0; i--) {
    double s = g[i];
    for (int k = i + 1; k < j; k++) s -= H[i + k * ld] * y[k];
    y[i] = s / H[i + i * ld];
  }
}

// The same with the cycle's Hessenberg columns staged in LDS by the
// workgroup and y formed in LDS, so the one thread's back substitution waits
// on no global load or store (same operations, same order).  Dynamic LDS:
// ((m + 1) * m + m) doubles.
constexpr int kHessLdsMaxM = 64;
__global__ void __launch_bounds__(256) k_hess_solve_lds(GmresDev *gd, int m, const double *__restrict__ H,
                                                        const double *__restrict__ g, double *__restrict__ y) {
  extern __shared__ double hs[];
  const int ld = m + 1, j = gd->jcur;
  for (int e = threadIdx.x; e < ld * j; e += blockDim.x) hs[e] = H[e];
  __syncthreads();
  if (threadIdx.x != 0) return;
  gd->jlast = j;
  double *ys = hs + (size_t)ld * m;
  for (int i = j - 1; i >= 0; i--) {
    double s = g[i];
    for (int k = i + 1; k < j; k++) s -= hs[i + k * ld] * ys[k];
    ys[i] = s / hs[i + i * ld];
  }
  for (int i = 0; i < j; i++) y[i] = ys[i];
}

// x += sum_{k<jcur} y[k] V_k
template <class TV, class TX>
__global__ void k_gemv_update_dev(int64_t n, int mmax, const TV *__restrict__ V, int64_t ldv,
                                  const double *__restrict__ c, const GmresDev *__restrict__ gd, TX *__restrict__ x) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int nv = gd->jcur < mmax ? gd->jcur : mmax;
  TV s = 0;
  for (int j = 0; j < nv; j++) s += (TV)c[j] * V[j * ldv + i];
  x[i] += (TX)s;
}

// w = x - lambda*y
__global__ void k_waxpy(int64_t n, double lambda, const double *__restrict__ x, const double *__restrict__ y,
                        double *__restrict__ w, const int *__restrict__ stop = nullptr) {
  if (stop && *stop) return;
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) w[i] = x[i] - lambda * y[i];
}

}  // namespace tdyhip
