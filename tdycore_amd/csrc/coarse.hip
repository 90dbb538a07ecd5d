// Coarse correction for the block-Jacobi ILU(0) preconditioner (optional;
// PETSc's default that the reference runs with is one-level block Jacobi).
//
//   w = BJ^-1 r,   M^-1 r = w + P z,   z = Z P^T (r - A w)
//
// One coarse unknown per ILU block (P: constant on a block's rows), with the
// Galerkin operator A1 = P^T A P; the coarse solve Z ~ A1^-1 acts on what the
// sweeps leave of r (the residual after block Jacobi, formed by the sweep
// kernels themselves: CoarseRestrict in krylov.hip).  The blocks are
// aggregated into at most kNG (small meshes kNG / 2) groups of at most kGMax;
// P2 is constant on a group's blocks, A2 = P2^T A1 P2 is inverted exactly as a
// dense matrix, and
//
//   Z r = P2 y + S (r - A1 P2 y),   y = A2^-1 P2^T r,
//
// with S the restricted Schwarz sum over the groups: a group's blocks with a
// layer of neighbour blocks (at most kOV in all) are solved exactly and the
// group's own blocks keep the result.  Everything of Z that depends on the
// matrix alone is formed once per Newton step, per group: G1 (the own rows of
// the overlapped inverse) and M = (P2 - G1 A1 P2) A2^-1, so an application is
// z = [G1 M] [r of the overlap; P2^T r], one small dense product per group.
// With a block per group (up to kNG / 2 blocks) the level-2 solve is A1^-1 itself
// and G1 is left out.
//
// Against the additive form BJ^-1 r + P (G1 + P2 A2^-1 P2^T) P^T r without
// overlap (GMRES(30) iterations to rtol 1e-5, first Newton systems): layered
// 96x96x48 box 89 -> 44 (A1 solved exactly: 42), 64x64x32 67 -> 38, rotated
// tensors 56x40x28 49 -> 23, 16^3 in 64-row blocks 30 -> 17.
//
// Everything is linear and fixed for one Newton step, so GMRES sees a
// constant preconditioner.  All reductions run in a fixed order, so the
// correction is deterministic.
#include "tdyhip_internal.h"

namespace tdyhip {

constexpr int kGMax = 64;   // blocks per group
constexpr int kOV = 128;    // blocks of a group with its overlap
constexpr int kNG = 128;    // level-2 unknowns

struct CoarseLayout {
  int nb = 0, ng = 0, gsz = 0;    // blocks, groups, max blocks per group
  int nov = 0;                    // blocks of a group with overlap, at most (0: a block per group)
  int g2max = 0;                  // entries of r2c of a group, at most
  uint8_t *cq = nullptr;          // W*NB, block-contiguous as the ELL: place of slot k's column block among the neighbours of p's block (255 none)
  uint8_t *tslot = nullptr;       // W*NB: slot of row i's mirror entry A_ci in the row c of its slot k (255 none)
  int32_t *gmem = nullptr;        // ng*gsz: blocks of each group (-1 pad)
  int32_t *gov = nullptr;         // ng*nov: blocks of each group, then its overlap (-1 pad)
  uint8_t *gpos = nullptr;        // ng*nov*kCQ: place in gov of each member's neighbour q (255 none)
  uint16_t *gent = nullptr;       // per group max(nov, gsz)*kCQ: entries member*kCQ + q of its members' A1 rows by group
  uint16_t *gep = nullptr;        // ng*(ng+1): each group's first entry in gent
  int32_t *g2ptr = nullptr;       // ng+1: each group's entries of r2c
  double *cown = nullptr, *cval = nullptr;  // column sums (CoarseRestrict)
  double *A1 = nullptr;           // nb*kCQ: Galerkin rows (column = neighbour position)
  double *G1 = nullptr;           // ng*nov*gsz: own rows of each overlapped inverse (column-major per group)
  double *A2 = nullptr;           // ng*ng: level-2 operator, inverted in place
  double *M = nullptr;            // ng*ng*gsz: level-2 part of the coarse inverse (column-major per group)
  double *z1 = nullptr;           // nb: coarse correction per block
  CoarseRestrict R;               // the sweep kernels' part
  int *status = nullptr;          // nonzero: singular coarse block
};

// Slot of row i in the row c of its slot k's column (the pattern is
// symmetric), found once per workspace by binary search: one thread per
// position and slot.
__global__ void __launch_bounds__(256) k_coarse_tslot(int64_t NB, int W, int bs, const int32_t *__restrict__ rowof,
                                                      const int32_t *__restrict__ jrp,
                                                      const int32_t *__restrict__ jcols, uint8_t *__restrict__ tslot) {
  const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= NB * W) return;
  const int64_t b = e / ((int64_t)W * bs);
  const int k = (int)((e / bs) % W);
  const int i = rowof[b * bs + e % bs];
  uint8_t s = 255;
  if (i >= 0 && k < jrp[i + 1] - jrp[i]) {
    const int c = jcols[jrp[i] + k], r0 = jrp[c];
    int lo = r0, hi = jrp[c + 1] - 1;
    while (lo < hi) {
      const int mid = (lo + hi) >> 1;
      if (jcols[mid] < i) lo = mid + 1; else hi = mid;
    }
    if (jcols[lo] == i) s = (uint8_t)(lo - r0);
  }
  tslot[e] = s;
}

// Column sums C of each block's rows by neighbour block (see CoarseRestrict)
// and from them A1: one workgroup per block, one thread per row j.  A_ij sits
// in row i of slot k's column, at the mirror slot; a thread's sums by
// neighbour go to its own LDS column, then the lists read them.  A1's entry
// of (neighbour, this block) is the sum of one list.
template <int BS, class TI>
__global__ void __launch_bounds__(BS) k_coarse_cols(CoarseLayout C, int W, int bs_log2, const int32_t *__restrict__ rowof,
                                                    const int32_t *__restrict__ perm, const TI *__restrict__ ecol,
                                                    const int32_t *__restrict__ pat, const double *__restrict__ J) {
  __shared__ double acc[kCQ][BS];
  const int b = blockIdx.x, t = threadIdx.x;
  const int row = rowof[(int64_t)b * BS + t];
  const int64_t e0 = ((int64_t)b * W) * BS + t;  // block-contiguous ELL: slot k at e0 + k*BS
  int64_t eb, es;
  ecol_addr(pat, BS, W, (int64_t)b * BS + t, eb, es);
#pragma unroll
  for (int q = 0; q < kCQ; q++) acc[q][t] = 0.0;
  constexpr int kBatch = 8;  // slots whose loads are in flight together
  for (int k0 = 0; k0 < W; k0 += kBatch) {
    uint8_t q[kBatch], ts[kBatch];
    int32_t p[kBatch];
    double v[kBatch];
#pragma unroll
    for (int u = 0; u < kBatch; u++) {
      const int k = k0 + u;
      const bool in = row >= 0 && k < W;
      q[u] = in ? C.cq[e0 + (int64_t)k * BS] : (uint8_t)255;
      ts[u] = in ? C.tslot[e0 + (int64_t)k * BS] : (uint8_t)255;
      p[u] = in ? blk_col(ecol, eb + k * es, row) : 0;
    }
#pragma unroll
    for (int u = 0; u < kBatch; u++) p[u] = perm[p[u]];
#pragma unroll
    for (int u = 0; u < kBatch; u++)
      v[u] = q[u] != 255 && ts[u] != 255 ? J[((((int64_t)(p[u] >> bs_log2) * W + ts[u]) << bs_log2)) + (p[u] & (BS - 1))] : 0.0;
#pragma unroll
    for (int u = 0; u < kBatch; u++)
      if (q[u] != 255) acc[q[u]][t] += v[u];
  }
  const double own = acc[C.R.ownq[b]][t];
  C.cown[(int64_t)b * BS + t] = own;
  __syncthreads();
  const int l0 = C.R.eptr[b], q = t < kCQ ? t : 0;
  const double s = coarse_block_sums<BS>(C.R.eptr[b + 1] - l0, C.R.tq[b * (kCQ + 1) + q], C.R.tq[b * (kCQ + 1) + q + 1],
                                         t == C.R.ownq[b], t, own, [&](int e) {
    const unsigned w = C.R.cent[l0 + e];
    const double v = w == kCoarsePad ? 0.0 : acc[w >> 9][w & 511];
    C.cval[l0 + e] = v;
    return v;
  });
  if (t < kCQ) {
    const int d = C.R.wdst[b * kCQ + t];
    if (d >= 0) C.A1[d] = s;
  }
}

// Max over a wavefront's 64 lanes, the same in every lane: register
// exchanges within each row of 16 lanes (lane ^ 1, lane ^ 2, the mirrors
// within 8 and 16 lanes), then the four rows' values.
template <int CTRL>
__device__ inline double dpp_max(double v) {
  const uint64_t u = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_update_dpp(0, (int)u, CTRL, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(u >> 32), CTRL, 0xf, 0xf, true);
  return fmax(v, __longlong_as_double((long long)((uint64_t)(uint32_t)hi << 32 | (uint32_t)lo)));
}
__device__ inline double lane_value(double v, int lane) {  // lane uniform
  const uint64_t u = __double_as_longlong(v);
  const uint32_t lo = __builtin_amdgcn_readlane((int)u, lane), hi = __builtin_amdgcn_readlane((int)(u >> 32), lane);
  return __longlong_as_double((long long)((uint64_t)hi << 32 | lo));
}
__device__ inline double wave_max(double v) {
  v = dpp_max<0xB1>(v);   // quad_perm [1,0,3,2]
  v = dpp_max<0x4E>(v);   // quad_perm [2,3,0,1]
  v = dpp_max<0x141>(v);  // row_half_mirror
  v = dpp_max<0x140>(v);  // row_mirror
  return fmax(fmax(lane_value(v, 0), lane_value(v, 16)), fmax(lane_value(v, 32), lane_value(v, 48)));
}

// Gauss-Jordan inverse with row pivoting of an n x n matrix (n <= N) in the
// registers of a 256-thread workgroup: lane l of wavefront w holds columns
// w*CW .. w*CW + CW-1 of rows l and (N = 128) l + 64; zero outside n x n.
// The pivot of column k is the row of largest |M[i][k]| not yet taken (the
// first such row); rows are not moved:
//   row p = row p / M[p][k], 1 / M[p][k] at column k;
//   row i = row i - (M[i][k] / M[p][k]) row p, -M[i][k] / M[p][k] at column k.
// On true, the entry of row i at register j is entry (s.rdst[i], s.cdst[c]) of
// the inverse, c = s.col(n, w, j).  false (for every thread): a zero or NaN
// pivot.
//
// Bound by the latency of the n dependent steps.  The wavefront that holds
// column k finds the pivot with register exchanges (each lane divides by its
// own candidate meanwhile) and publishes it with the column through LDS, one
// barrier a step (the column is double-buffered); the pivot row reaches the
// other lanes through scalar registers.  The column's wavefront rotates its
// registers by one column a step, so the current column is always register 0
// and the loop stays rolled: a small body, as its first pass through the
// instruction cache costs more than a step.  128 x 128 alone 318 -> 170 us,
// 64 x 64 164 -> 51 us against 4x4 tiles per thread with the pivot search, both
// rows and the column published in turn (four barriers a step).  (At 128 x 128 a
// lane's 64 values and the pivot row's 32 take 248 + 32 registers and 140 bytes of
// scratch.)
template <int N>
struct TiledGJ {
  static constexpr int NT = 256, RL = N / 64, CW = N / 4;
  double colk[2][N];
  double inv[2];
  int pk[2], flag[2];
  int rdst[N], cdst[N];
  static __device__ inline int col(int n, int w, int j) {
    return w * CW + (w == n / CW ? (j + n % CW) % CW : j);
  }
};

template <int N>
__device__ inline bool gj_invert_tiles(double (&m)[TiledGJ<N>::RL][TiledGJ<N>::CW], int n, TiledGJ<N> &s) {
  constexpr int RL = TiledGJ<N>::RL, CW = TiledGJ<N>::CW;
  const int t = threadIdx.x, lane = t & 63, w = __builtin_amdgcn_readfirstlane(t >> 6);
  bool open[RL];  // rows not yet taken
#pragma unroll
  for (int a = 0; a < RL; a++) open[a] = lane + 64 * a < n;
  for (int k = 0; k < n; k++) {
    const int f = k & 1;
    const bool mine = w == k / CW;
    if (mine) {
      double mx = -1.0, val = 0.0;
      bool nan = false;
#pragma unroll
      for (int a = 0; a < RL; a++) {
        const double v = open[a] ? fabs(m[a][0]) : -1.0;
        nan |= v != v;
        if (v > mx) { mx = v; val = m[a][0]; }
      }
      const double vinv = 1.0 / val;
      const double wm = wave_max(mx);
      // the first row that holds the maximum: rows l before rows l + 64
      int p = -1;
#pragma unroll
      for (int a = RL - 1; a >= 0; a--) {
        const uint64_t hit = __ballot(open[a] && fabs(m[a][0]) == wm);
        if (hit) p = __builtin_ctzll(hit) + 64 * a;
      }
      const bool bad = !(wm > 0.0) || __ballot(nan) != 0;
      // (a lane whose two rows both hold the maximum took, and divided by, the first)
      const double inv = lane_value(vinv, p < 0 ? 0 : p & 63);
      if (lane == 0) {
        s.pk[f] = p;
        s.inv[f] = inv;
        s.flag[f] = bad;
        s.cdst[k] = p;
      }
#pragma unroll
      for (int a = 0; a < RL; a++) s.colk[f][lane + 64 * a] = m[a][0];
    }
    __syncthreads();
    if (s.flag[f]) return false;  // uniform over the workgroup
    const int p = __builtin_amdgcn_readfirstlane(s.pk[f]), pl = p & 63;
    const double inv = s.inv[f];
    if (t == 0) s.rdst[p] = k;
    if (w * CW >= n) continue;  // no columns here
    double l[RL];
    bool piv[RL];
#pragma unroll
    for (int a = 0; a < RL; a++) {
      piv[a] = lane + 64 * a == p;
      open[a] = open[a] && !piv[a];
      l[a] = s.colk[f][lane + 64 * a] * inv;
    }
    double rp[CW];  // row p of these columns
    if (RL == 1 || p < 64) {
#pragma unroll
      for (int j = 0; j < CW; j++) rp[j] = lane_value(m[0][j], pl);
    } else {
#pragma unroll
      for (int j = 0; j < CW; j++) rp[j] = lane_value(m[RL - 1][j], pl);
    }
#pragma unroll
    for (int a = 0; a < RL; a++) {
#pragma unroll
      for (int j = 0; j < CW; j++) m[a][j] -= l[a] * rp[j];
      if (piv[a]) {
#pragma unroll
        for (int j = 0; j < CW; j++) m[a][j] = rp[j] * inv;
      }
    }
    if (mine) {
#pragma unroll
      for (int a = 0; a < RL; a++) {
#pragma unroll
        for (int j = 0; j + 1 < CW; j++) m[a][j] = m[a][j + 1];
        m[a][CW - 1] = piv[a] ? inv : -l[a];
      }
    }
  }
  __syncthreads();
  return true;
}

// One workgroup per group (N >= nov): the group's row of
// A2, G1 = the own rows of the inverse of A1 on the group's blocks with their
// overlap, and H = P2 - G1 A1 P2 over the own blocks (left in M for
// k_coarse_fold).  The members' A1 rows are staged in LDS, all their loads in
// flight together; each thread picks its tile of the matrix from them by
// the places gpos, and the matrix is inverted in registers.  Sums over the
// groups' neighbours follow the static lists gent (entries member * kCQ + q
// by the neighbour's group), so no thread looks at an entry it does not need.
template <int N>
__global__ void __launch_bounds__(TiledGJ<N>::NT) k_coarse_groups(CoarseLayout C) {
  constexpr int NT = TiledGJ<N>::NT, RL = TiledGJ<N>::RL, CW = TiledGJ<N>::CW;
  __shared__ TiledGJ<N> gs;
  __shared__ double aq[N * kCQ];   // A1 row of each member
  __shared__ uint8_t ps[N * kCQ];  // place of each neighbour in the group with overlap
  __shared__ uint16_t ge[N * kCQ], gp[kNG + 1];
  __shared__ int mem[N];
  const int g = blockIdx.x, t = threadIdx.x, G = C.gsz, nov = C.nov, ng = C.ng;
  const int nm = nov ? nov : G;  // members listed
  const int mt = t < nm ? (nov ? C.gov[g * nov + t] : C.gmem[g * G + t]) : -1;
  const int ot = t < G ? C.gmem[g * G + t] : -1;
  if (t < N) mem[t] = mt;
  // members with overlap (own members first), own members
  const int nt = __syncthreads_count(mt >= 0), n = __syncthreads_count(ot >= 0);
  for (int e = t; e < nm * kCQ; e += NT) ge[e] = C.gent[(int64_t)g * nm * kCQ + e];
  for (int h = t; h <= ng; h += NT) gp[h] = C.gep[(int64_t)g * (ng + 1) + h];
  for (int e = t; e < N * kCQ; e += NT) {
    const int i = e / kCQ, q = e % kCQ;
    aq[e] = i < nt ? C.A1[(int64_t)mem[i] * kCQ + q] : 0.0;
    ps[e] = i < nt && nov ? C.gpos[((int64_t)g * nov + i) * kCQ + q] : (uint8_t)255;
  }
  __syncthreads();
  // A2[g][h]: the own members' entries of group h, in the order of the list
  for (int h = t; h < ng; h += NT) {
    double sum = 0.0;
    for (int e = gp[h]; e < gp[h + 1]; e++) sum += ge[e] < n * kCQ ? aq[ge[e]] : 0.0;
    C.A2[(int64_t)g * ng + h] = sum;
  }
  double *g1 = C.G1 + (int64_t)g * nov * G;
  if (nov) {
    const int lane = t & 63, w = t >> 6;
    double m[RL][CW];
#pragma unroll
    for (int a = 0; a < RL; a++) {
#pragma unroll
      for (int j = 0; j < CW; j++) m[a][j] = 0.0;
#pragma unroll 2
      for (int q = 0; q < kCQ; q++) {
        const int p = (int)ps[(lane + 64 * a) * kCQ + q] - w * CW;
        const double v = aq[(lane + 64 * a) * kCQ + q];
#pragma unroll
        for (int j = 0; j < CW; j++) m[a][j] = p == j ? v : m[a][j];
      }
    }
    if (!gj_invert_tiles<N>(m, nt, gs)) {
      if (t == 0) atomicOr(C.status, 1);
      return;
    }
    // G1 column-major (entry (i, j) at j*G + i, zero past the members): the
    // coarse solve reads it coalesced
    for (int e = t; e < nov * G; e += NT)
      if (e / G >= nt || e % G >= n) g1[e] = 0.0;
#pragma unroll
    for (int a = 0; a < RL; a++) {
      const int i = lane + 64 * a < nt ? gs.rdst[lane + 64 * a] : n;
#pragma unroll
      for (int j = 0; j < CW; j++) {
        const int c = gs.col(nt, w, j);
        if (i < n && c < nt) g1[(int64_t)gs.cdst[c] * G + i] = m[a][j];
      }
    }
    __syncthreads();
  }
  // H: each thread a row and every nch-th group
  const int rp = G <= 8 ? 8 : G <= 32 ? 32 : 64;
  const int i = t % rp, nch = NT / rp;
  if (i < G)
    for (int h = t / rp; h < ng; h += nch) {
      double s = h == g && i < n ? 1.0 : 0.0;
      if (nov) {
#pragma unroll 4
        for (int e = gp[h]; e < gp[h + 1]; e++) s -= g1[(ge[e] / kCQ) * G + i] * aq[ge[e]];
      }
      C.M[((int64_t)g * ng + h) * G + i] = s;
    }
}

// M = H A2^-1 of group g (one workgroup of 256 threads per group, groups of
// at most 2*RB blocks; H in M on entry): each thread a column and half of the
// rows, A2^-1 read by rows, H through LDS K groups at a time.  Small in LDS
// so that it fits beside the factor's workgroups.  (It does not look at the
// status: the factor beside it may set it while a workgroup's threads read, and
// they would part at the barriers.  After a singular block M is not used.)
constexpr int kFoldThreads = 2 * kNG;
template <int RB, int K>
__global__ void __launch_bounds__(kFoldThreads) k_coarse_fold(CoarseLayout C) {
  __shared__ double hs[K][2 * RB];
  const int g = blockIdx.x, t = threadIdx.x, G = C.gsz, ng = C.ng;
  const int col = t % kNG, r0 = (t / kNG) * RB;
  double *M = C.M + (int64_t)g * ng * G;
  double s[RB];
#pragma unroll
  for (int r = 0; r < RB; r++) s[r] = 0.0;
  for (int h0 = 0; h0 < ng; h0 += K) {
    for (int e = t; e < K * 2 * RB; e += kFoldThreads) {
      const int h = h0 + e / (2 * RB), i = e % (2 * RB);
      hs[e / (2 * RB)][i] = h < ng && i < G ? M[(int64_t)h * G + i] : 0.0;
    }
    double a[K];
#pragma unroll
    for (int u = 0; u < K; u++) a[u] = h0 + u < ng && col < ng ? C.A2[(int64_t)(h0 + u) * ng + col] : 0.0;
    __syncthreads();
    if (r0 < G) {
#pragma unroll
      for (int u = 0; u < K; u++)
#pragma unroll
        for (int r = 0; r < RB; r++) s[r] += hs[u][r0 + r] * a[u];
    }
    __syncthreads();
  }
#pragma unroll
  for (int r = 0; r < RB; r++)
    if (col < ng && r0 + r < G) M[(int64_t)col * G + r0 + r] = s[r];
}

// Single workgroup: A <- A^-1 (n <= N, row-major), the matrix in registers;
// the level-2 inverse A2 <- A2^-1.
template <int N>
__device__ inline void dense_invert(double *A, int n, int *status) {
  constexpr int RL = TiledGJ<N>::RL, CW = TiledGJ<N>::CW;
  __shared__ TiledGJ<N> gs;
  const int t = threadIdx.x, lane = t & 63, w = t >> 6;
  double m[RL][CW];
#pragma unroll
  for (int a = 0; a < RL; a++)
#pragma unroll
    for (int j = 0; j < CW; j++)
      m[a][j] = (lane + 64 * a < n && w * CW + j < n) ? A[(int64_t)(lane + 64 * a) * n + w * CW + j] : 0.0;
  if (!gj_invert_tiles<N>(m, n, gs)) {
    if (t == 0) atomicOr(status, 1);
    return;
  }
#pragma unroll
  for (int a = 0; a < RL; a++) {
    if (lane + 64 * a >= n) continue;
    const int i = gs.rdst[lane + 64 * a];
#pragma unroll
    for (int j = 0; j < CW; j++) {
      const int c = gs.col(n, w, j);
      if (c < n) A[(int64_t)i * n + gs.cdst[c]] = m[a][j];
    }
  }
}

template <int N>
__global__ void __launch_bounds__(TiledGJ<N>::NT) k_coarse_invert(CoarseLayout C) { dense_invert<N>(C.A2, C.ng, C.status); }

// Test kernel: A <- A^-1 for one dense n x n row-major matrix (n <= N) by
// gj_invert_tiles<N> in one workgroup; N = 64 and 128 are the widths the
// coarse set-up uses.  *status set on a zero pivot.
template <int N>
__global__ void __launch_bounds__(TiledGJ<N>::NT) k_test_dense_invert(double *A, int n, int *status) {
  dense_invert<N>(A, n, status);
}

// An application of Z for one part of a group (one workgroup of kL1Threads
// per part of kL1Rows of the group's blocks):
//   z1 = G1 r + M r2,
// r the restricted residual of the group's blocks with their overlap (each
// block's received contributions summed) and r2 that of every group.  Every
// workgroup sums what it needs itself, so one launch finishes the coarse
// solve.  Bound by latency: with 16 rows a thread holds 8 columns of G1 and of
// M, all loaded before the one barrier, and the groups' lists are summed with
// 16 loads in flight.  (Whole groups of 33 blocks per workgroup, their
// columns in batches of four, held the multi-dot to 27 us at 1M rows.)  z1
// of the part's blocks is left in zs (LDS, zero past the members) and written
// to cd.z1; the members in ms.  Every thread calls it.
constexpr int kL1Threads = 256, kL1Rows = 16;
static_assert(kL1Threads == 2 * kOV, "two threads per block of the overlap");
__host__ __device__ inline int coarse_parts(int gsz) { return (gsz + kL1Rows - 1) / kL1Rows; }
__device__ inline void coarse_z1(const CoarseDot &cd, int part, double *zs, int *ms) {
  constexpr int NP = kNG * 8 / kL1Threads;     // passes of 8-lane teams over the groups
  constexpr int NCH = kL1Threads / kL1Rows;    // column chunks: chunk ch has columns ch, ch + NCH, ...
  constexpr int NCOL = kNG / NCH;
  static_assert(kOV == kNG, "as many columns of G1 as of M");
  __shared__ double rs[kOV], r2s[kNG], zc[kL1Threads / 64][kL1Rows];
  const int t = threadIdx.x, G = cd.gsz, ng = cd.ng, nov = cd.nov;
  const int np = coarse_parts(G), g = part / np, i0 = (part % np) * kL1Rows;
  const int i = i0 + t % kL1Rows, ch = t / kL1Rows;
  const bool row = i < G;
  // r2[h]: eight lanes per group
  {
    int e[NP], e1[NP];
    double s[NP];
#pragma unroll
    for (int p = 0; p < NP; p++) {
      const int h = p * (kL1Threads / 8) + t / 8;
      e[p] = h < ng ? cd.g2ptr[h] + t % 8 : 0;
      e1[p] = h < ng ? cd.g2ptr[h + 1] : 0;
      s[p] = 0.0;
    }
    for (int k = 0; k < cd.g2max; k += 32) {
      double v[NP][4];
#pragma unroll
      for (int p = 0; p < NP; p++)
#pragma unroll
        for (int u = 0; u < 4; u++) v[p][u] = e[p] + k + 8 * u < e1[p] ? cd.r2c[e[p] + k + 8 * u] : 0.0;
#pragma unroll
      for (int p = 0; p < NP; p++)
#pragma unroll
        for (int u = 0; u < 4; u++) s[p] += v[p][u];
    }
#pragma unroll
    for (int p = 0; p < NP; p++) {
      double q = s[p];
      q += __shfl_xor(q, 1, 64);
      q += __shfl_xor(q, 2, 64);
      q += __shfl_xor(q, 4, 64);
      const int h = p * (kL1Threads / 8) + t / 8;
      if (t % 8 == 0) r2s[h] = h < ng ? q : 0.0;
    }
  }
  const int bt = t < kL1Rows && i0 + t < G ? cd.gmem[g * G + i0 + t] : -1;
  const int bo = t / 2 < nov ? cd.gov[g * nov + t / 2] : -1;
  const double *g1 = cd.G1 + (int64_t)g * nov * G + i, *mm = cd.M + (int64_t)g * ng * G + i;
  double gv[NCOL], mv[NCOL];
#pragma unroll
  for (int u = 0; u < NCOL; u++) {
    const int c = ch + NCH * u;
    gv[u] = row && c < nov ? g1[(int64_t)c * G] : 0.0;
    mv[u] = row && c < ng ? mm[(int64_t)c * G] : 0.0;
  }
  // r of the overlap's blocks: two threads per block, half of its contributions each
  {
    double s = 0.0;
    if (bo >= 0) {
      const double2 *rc = reinterpret_cast<const double2 *>(cd.rcs + (int64_t)bo * kCQ + (t % 2) * (kCQ / 2));
#pragma unroll
      for (int u = 0; u < kCQ / 4; u++) {
        const double2 q = rc[u];
        s += q.x;
        s += q.y;
      }
    }
    s += __shfl_xor(s, 1, 64);
    if (t % 2 == 0) rs[t / 2] = s;
  }
  if (t < kL1Rows) ms[t] = bt;
  __syncthreads();
  double z = 0.0;
#pragma unroll
  for (int u = 0; u < NCOL; u++) {
    z += gv[u] * rs[ch + NCH * u];
    z += mv[u] * r2s[ch + NCH * u];
  }
  // the chunks: four per wavefront by exchanges, then the wavefronts in order
  z += __shfl_xor(z, 16, 64);
  z += __shfl_xor(z, 32, 64);
  if ((t & 63) < kL1Rows) zc[t >> 6][t % kL1Rows] = z;
  __syncthreads();
  if (t < kL1Rows) {
    double zz = 0.0;
    if (bt >= 0) {
#pragma unroll
      for (int w = 0; w < kL1Threads / 64; w++) zz += zc[w][t];
      cd.z1[bt] = zz;
    }
    zs[t] = zz;
  }
  __syncthreads();
}

__global__ void __launch_bounds__(kL1Threads) k_coarse_level1(CoarseDot cd, const int *__restrict__ stop) {
  __shared__ double zs[kL1Rows];
  __shared__ int ms[kL1Rows];
  if (stop && *stop) return;
  coarse_z1(cd, blockIdx.x, zs, ms);
}

// In a multi-dot launch: z1 of a group's part as above, then the part's
// terms of the dots with the nv basis vectors.  V_v . (w_bj + P z1) splits
// into V_v . w_bj (the row-chunk workgroups) and RV_v . z1 with RV_v the
// block sums of V_v; this part adds sum over its blocks of RV_v[b] z1[b], two
// members per thread and the eight pairs in order, to partial[v * pstride +
// part].
template <class TV>
__device__ void coarse_level1_dots(const CoarseDot &cd, int part, int nv, TV *partial, int pstride) {
  static_assert(kL1Threads == kRedBlock, "the multi-dot's workgroup size");
  __shared__ double zs[kL1Rows];
  __shared__ int ms[kL1Rows];
  __shared__ double cps[kL1Rows / 2][32];
  coarse_z1(cd, part, zs, ms);
  const int t = threadIdx.x, v = t % 32, c = t / 32;  // vector, pair of members
  const int b0 = ms[2 * c], b1 = ms[2 * c + 1];
  for (int v0 = 0; v0 < nv; v0 += 32) {
    double q = 0.0;
    if (v0 + v < nv) {
      const double *rv = cd.RV + (int64_t)(v0 + v) * cd.rv_ld;
      const double x0 = b0 >= 0 ? rv[b0] : 0.0, x1 = b1 >= 0 ? rv[b1] : 0.0;
      q += x0 * zs[2 * c];
      q += x1 * zs[2 * c + 1];
    }
    cps[c][v] = q;
    __syncthreads();
    if (t < 32 && v0 + t < nv) {
      double p = cps[0][t];
#pragma unroll
      for (int k = 1; k < kL1Rows / 2; k++) p += cps[k][t];
      partial[(int64_t)(v0 + t) * pstride + part] = (TV)p;
    }
    __syncthreads();
  }
}

// Prolongation: out[row] += z1[b] for the rows of block b.
template <class TV, int BS>
__global__ void __launch_bounds__(BS) k_coarse_prolong(CoarseLayout C, const int32_t *__restrict__ rowof,
                                                       TV *__restrict__ out, const int *__restrict__ stop) {
  if (stop && *stop) return;
  const int b = blockIdx.x, t = threadIdx.x;
  const int row = rowof[(int64_t)b * BS + t];
  if (row >= 0) out[row] += (TV)C.z1[b];
}

}  // namespace tdyhip
