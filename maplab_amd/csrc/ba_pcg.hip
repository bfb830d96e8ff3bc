// ba_pcg.hip -- deflated, block-Jacobi preconditioned conjugate gradients on
// the reduced camera system S y = b (FP64).
//
// Block-Jacobi (inverse 6x6 diagonal blocks of S, Ceres' SCHUR_JACOBI) leaves
// a handful of very small eigenvalues on long trajectories: smooth, global
// modes of the vertex chain. They are removed by deflation (Saad, Yeung,
// Erhel, Guyomarc'h, "A deflated version of the conjugate gradient
// algorithm", SIAM J. Sci. Comput. 21, 2000) with a coarse space
// W = [H | R]: H the piecewise-linear "hat" functions over the vertex order
// (K nodes, 6 K columns), R up to 16 dense columns recycled from earlier
// solves (Ritz vectors of the preconditioned operator for its smallest
// eigenvalues, from each solve's Lanczos coefficients; see the ritz kernels
// below). x0 = W E^-1 W'b, E = W'SW, and every search direction is made
// S-orthogonal to W with mu = E^-1 (SW)'z. The iteration converges to the
// same solution as plain PCG (the tolerance is on the true residual
// recursion): the hat space cuts iterations 3-4x on long random-walk maps,
// the recycled vectors another 2-3x on the solves that follow a rejected
// LM step (same linearization, new damping).
//
// Rows of S are handled in groups of 42 vertices (252 entries); SW is stored
// per group, column-major over the group's window of coarse columns (the hat
// columns its rows couple to, then the dense ones), so that (SW)'z of a group
// is a set of coalesced column dot products.
//
// Per LM step: k_defl_sr (SW), k_defl_e and k_defl_dense (E, R'b),
// k_defl_prep (state, E^-1 by the sweep operator, y = E^-1 W'b). With
// block-Jacobi k_pcg_start and one launch per iteration, k_pcg_step, follow where
// that pays (step_pays); otherwise k_defl_init (x0, r0, z0 and the first per-group partials)
// and two launches per iteration: k_pcg_spmv (sums the previous
// per-group partials; p = z - W mu + beta p_prev and
// q = S z + beta S p_prev - (SW) mu) and k_pcg_update (x, r, z and the
// per-group partials r'z, r'r, E^-1 (SW)'z). Every sum of partials runs in
// the same fixed order, so the set-up and the iteration are deterministic.
// With more groups than one LDS chunk of k_pcg_spmv holds, the work-group of
// k_pcg_update (or k_defl_init) that finishes last sums the groups' partials
// once, into part1, and k_pcg_spmv reads that one vector; the only atomic is
// the integer arrival counter that picks this work-group.
//
// The deflation holds for any SPD preconditioner: with the learned one
// (z = L^-T (I - K)' (I - K) L^-1 r, K strictly block-lower-triangular),
// k_defl_init and k_pcg_update stop at t = L^-1 r, and k_pcg_lower,
// k_pcg_upper (the two row sweeps) and k_defl_partials (the same group
// partials) follow; the hat space is kept, the recycled columns are not
// (their Rayleigh-Ritz step is taken with respect to block-Jacobi's M).
#include "ba_pcg.h"

#include <algorithm>

#include "ba_device.h"
#include "ba_reduce.h"

namespace mlba {

constexpr int kMaxHatNodes = 15;
constexpr int kMaxRitz = kPcgMaxRitz;
constexpr int kMaxCoarse = 6 * kMaxHatNodes + kMaxRitz;  // 106 columns
constexpr int kRowsPerGroup = 42;
constexpr int kGroupThreads = 6 * kRowsPerGroup;  // 252 entries (row, component) per group
constexpr int kGroupBlock = 1024;                 // threads of the per-group kernels
constexpr int kPartChunk = 2048;                  // doubles of partials summed per LDS pass

struct PcgState {
  double rz[2];     // r'z of iteration k in rz[k & 1] (written by k_pcg_spmv)
  double bb;        // |b|^2
  double tol_rel2;  // tol^2
  double tol2;      // (tol |b|)^2
  int32_t iters;
  int32_t done;
  int32_t max_iters;
  int32_t defl_ok;  // E was positive definite: the deflation is applied
  uint32_t arrive;  // work-groups that wrote their partials in the current launch
  int32_t pad;
};

struct PcgArgs {
  int32_t Pvar, ne;            // ne = neh + nr coarse columns (0: no deflation)
  int32_t neh, nr;             // hat (6 K) and dense columns
  int32_t K, groups;
  int32_t gwh, n6;             // hat columns of a group window; 6 Pvar
  int32_t zcap, pad3;
  const int32_t* row_ptr;
  const int32_t* col_var;
  const double* S;
  const double* Minv;
  const double* b;
  const int32_t* hat_node;     // Pvar: first hat node of the vertex (0 without deflation)
  const double* hat_w;         // 2 Pvar: weights of hat_node and hat_node + 1 (0 without deflation)
  const int32_t* node_range;   // 2 K: first and last vertex of each hat's support
  const int32_t* grp_lo;       // groups: first hat node of the group's window of SW columns
  int32_t gw, pad2;            // window width in columns (gwh hat + nr dense)
  const double* R;             // nr x 6 Pvar dense columns
  const int32_t* blk_hat;      // per block of S: hat node of its column vertex
  const double* blk_w;         // per block of S: the two hat weights of its column vertex
  const int32_t* blk_rng;      // Pvar x K x 2: blocks of row i in the support of hat k
  double* SR;                  // groups x gw x 252: SW entry (group row t, window column lc)
  double* E;                   // ne x ne
  double* Einv;                // ne x ne
  double* EinvW;               // groups x gw x ne: the rows of E^-1 of each group's window columns
  double* x;
  double* r;
  double* z;
  double* p0;
  double* p1;
  double* q;
  double* part;                // Pvar: p'q of each row
  double* part2;               // groups x (3 + ne): r'z, r'r, b'b and E^-1 (SW)'z of the group's rows
  double* part1;               // 3 + ne: part2 summed over the groups (with reduce1)
  int32_t reduce1, pad4;       // the groups' partials exceed one LDS chunk of k_pcg_spmv
  double* y;                   // ne: E^-1 W'b
  double* cden;                // nr: R'b
  double* Zh;                  // zcap x 6 Pvar: deflated preconditioned residuals
  double* coef;                // 2 zcap: r'z and alpha per iteration
  PcgState* st;
  // k_pcg_step: what other rows read is kept twice, iteration k reads copy
  // k & 1 and writes the other.
  int32_t wgs, step_G;         // work-groups of k_pcg_step, rows of each
  double* zvp;                 // 2 x Pvar x 18: z, v = M S p and p of each row
  double* cvec;                // 2 x kMaxCoarse: (SW)'z
  double* spart;               // 2 x wgs x (kStepScalars + ne) partials
  double* zpart;               // wgs x ne: the work-groups' (SW)'z
  const double* linv;          // learned preconditioner (with kmat): L_i^-1, 36 Pvar
  const float* kmat;           // K_ij, 36 nnzb
  const int32_t* diag_pos;
  const int32_t* tpos;
  double* t;                   // L^-1 r
  double* u;                   // (I - K) L^-1 r
};

__device__ inline double hat_weight(const PcgArgs& a, int i, int k) {
  const int n0 = a.hat_node[i];
  return n0 == k ? a.hat_w[2 * i] : (n0 + 1 == k ? a.hat_w[2 * i + 1] : 0.0);
}

__device__ inline double* sr_col(const PcgArgs& a, int g, int lc) {
  return a.SR + ((size_t)g * a.gw + lc) * kGroupThreads;
}

// Coarse column of window column lc of a group whose hat window starts at
// column c0 (6 x its first node); -1 past the last hat column.
__device__ inline int win_col(const PcgArgs& a, int c0, int lc) {
  if (lc >= a.gwh) return a.neh + (lc - a.gwh);
  return c0 + lc < a.neh ? c0 + lc : -1;
}

// Block sums of three values (blockDim.x = 64 x waves, at most 16 waves), in
// every thread.
__device__ inline void block_sum3(double& v0, double& v1, double& v2, double* lds) {
  const int nw = blockDim.x >> 6, w = threadIdx.x >> 6;
  v0 = wave_sum(v0);
  v1 = wave_sum(v1);
  v2 = wave_sum(v2);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) {
    lds[w] = v0;
    lds[16 + w] = v1;
    lds[32 + w] = v2;
  }
  __syncthreads();
  double s0 = 0.0, s1 = 0.0, s2 = 0.0;
  for (int k = 0; k < nw; ++k) {
    s0 += lds[k];
    s1 += lds[16 + k];
    s2 += lds[32 + k];
  }
  v0 = s0;
  v1 = s1;
  v2 = s2;
}

// SW for the hat columns, one block row of S per work-group:
// (SH)_i = sum_j S_ij H_j over the group window's hat columns, written into
// the group window. Thread o owns entry (component o % 6, window column
// o / 6) of hat node k and sums, in order, the row's blocks whose vertex lies
// in the hat's support: a contiguous range of the row (blk_rng), each with
// weight w0 or w1 of its vertex (its first hat node is k or k - 1).
__global__ __launch_bounds__(256) void k_defl_sr(PcgArgs a) {
  const int i = blockIdx.x, g = i / kRowsPerGroup, t0 = 6 * (i - g * kRowsPerGroup);
  const int c0 = 6 * a.grp_lo[g];
  for (int o = threadIdx.x; o < 6 * a.gwh; o += blockDim.x) {
    const int comp = o % 6, lc = o / 6, col = win_col(a, c0, lc);
    double acc = 0.0;
    if (col >= 0) {
      const int k = col / 6, cc = col % 6;
      const int lo = a.blk_rng[2 * (i * a.K + k)], hi = a.blk_rng[2 * (i * a.K + k) + 1];
#pragma unroll 4
      for (int kb = lo; kb < hi; ++kb) {
        const int n0 = a.blk_hat[kb];
        const double w0 = a.blk_w[2 * kb], w1 = a.blk_w[2 * kb + 1];
        acc += (n0 == k ? w0 : w1) * a.S[(size_t)36 * kb + 6 * comp + cc];
      }
    }
    sr_col(a, g, lc)[t0 + comp] = acc;
  }
}

// SW for the dense columns (or S Rn for the recycling), one block row per
// work-group of six waves: wave w takes the dense columns 3 w .. 3 w + 2 for
// all six components (so R_j is read once per block, not once per
// component), lane l sums over the row's blocks l, l + 64, ... the products
// S_ij[comp][:] . R_c[6 j ..], then a fixed-order wave sum per (component,
// column). Writes the group window (dense part) or a plain column-major
// buffer.
constexpr int kDenseThreads = 384;
constexpr int kDenseColsPerWave = (kMaxRitz + kDenseThreads / 64 - 1) / (kDenseThreads / 64);  // 3
template <bool kWindow>
__global__ __launch_bounds__(kDenseThreads) void k_row_dense(PcgArgs a, const int32_t* __restrict__ row_ptr,
                                                             const int32_t* __restrict__ col_var,
                                                             const double* __restrict__ S,
                                                             const double* __restrict__ R, int32_t nr, int32_t n6,
                                                             double* __restrict__ out) {
  const int i = blockIdx.x, wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int c0 = wave * kDenseColsPerWave;
  if (c0 >= nr) return;  // the whole wave: no barrier in this kernel
  const int rb = row_ptr[i], re = row_ptr[i + 1];
  double acc[6][kDenseColsPerWave];
#pragma unroll
  for (int comp = 0; comp < 6; ++comp)
#pragma unroll
    for (int m = 0; m < kDenseColsPerWave; ++m) acc[comp][m] = 0.0;
  for (int kb = rb + lane; kb < re; kb += 64) {
    const double* sb = S + (size_t)36 * kb;
    double sv[36];
#pragma unroll
    for (int e = 0; e < 36; ++e) sv[e] = sb[e];
    const double* rj = R + 6 * col_var[kb];
#pragma unroll
    for (int m = 0; m < kDenseColsPerWave; ++m) {
      if (c0 + m < nr) {
        const double* r = rj + (size_t)(c0 + m) * n6;
        const double r0 = r[0], r1 = r[1], r2 = r[2], r3 = r[3], r4 = r[4], r5 = r[5];
#pragma unroll
        for (int comp = 0; comp < 6; ++comp) {
          const double* s6 = sv + 6 * comp;
          acc[comp][m] += ((s6[0] * r0 + s6[1] * r1) + (s6[2] * r2 + s6[3] * r3)) + (s6[4] * r4 + s6[5] * r5);
        }
      }
    }
  }
#pragma unroll
  for (int m = 0; m < kDenseColsPerWave; ++m) {
    const int c = c0 + m;
    if (c >= nr) break;
#pragma unroll
    for (int comp = 0; comp < 6; ++comp) {
      const double v = wave_sum(acc[comp][m]);
      if (lane == 0) {
        if (kWindow) {
          const int g = i / kRowsPerGroup;
          sr_col(a, g, a.gwh + c)[6 * (i - g * kRowsPerGroup) + comp] = v;
        } else {
          out[(size_t)c * n6 + 6 * i + comp] = v;
        }
      }
    }
  }
}

// Entry (e, col) of SW from the group windows.
__device__ inline double sw_entry(const PcgArgs& a, int e, int col) {
  const int g = e / kGroupThreads;
  const int lc = col >= a.neh ? a.gwh + (col - a.neh) : col - 6 * a.grp_lo[g];
  return (lc >= 0 && lc < a.gw) ? sr_col(a, g, lc)[e - g * kGroupThreads] : 0.0;
}

// E = W'(SW) for the hat rows: one wave per (hat node k, column oc) sums the
// six rows (k, comp) over the hat's support (lanes take every 64th support
// row, then a fixed-order wave sum). A dense column's entries are also the
// transposed (dense, hat) entries. The dense-dense block is k_defl_dense's.
__global__ __launch_bounds__(64) void k_defl_e(PcgArgs a) {
  const int k = blockIdx.x, oc = blockIdx.y, lane = threadIdx.x;
  double s[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
  for (int i = a.node_range[2 * k] + lane; i <= a.node_range[2 * k + 1]; i += 64) {
    const double w = hat_weight(a, i, k);
#pragma unroll
    for (int comp = 0; comp < 6; ++comp) s[comp] += w * sw_entry(a, 6 * i + comp, oc);
  }
#pragma unroll
  for (int comp = 0; comp < 6; ++comp) {
    const double v = wave_sum(s[comp]);
    if (lane == 0) {
      a.E[(size_t)(6 * k + comp) * a.ne + oc] = v;
      if (oc >= a.neh) a.E[(size_t)oc * a.ne + 6 * k + comp] = v;
    }
  }
}

// Dense block of E and R'b, one work-group per entry: (a, b < nr) is
// R_a'(SR)_b over all rows, (a, nr) is R_a'b.
__global__ __launch_bounds__(256) void k_defl_dense(PcgArgs a) {
  __shared__ double lds[4];
  const int ra = blockIdx.x, cb = blockIdx.y;
  const double* Ra = a.R + (size_t)ra * a.n6;
  double s = 0.0;
  for (int e = threadIdx.x; e < a.n6; e += blockDim.x)
    s += Ra[e] * (cb < a.nr ? sw_entry(a, e, a.neh + cb) : a.b[e]);
  s = block_sum256(s, lds);
  if (threadIdx.x == 0) {
    if (cb < a.nr)
      a.E[(size_t)(a.neh + ra) * a.ne + a.neh + cb] = s;
    else
      a.cden[ra] = s;
  }
}

constexpr int kPrepThreads = 1024;
constexpr int kInvTile = 16;
constexpr int kInvTiles = (kMaxCoarse + kInvTile - 1) / kInvTile;  // 7
constexpr int kInvPad = kInvTile + 1;                              // LDS pitch of a 16-wide panel
constexpr int kInvWaves = kPrepThreads / 64;
constexpr int kInvPerWave = (kInvTiles * (kInvTiles + 1) / 2 + kInvWaves - 1) / kInvWaves;  // lower tiles of a wave

typedef double double4v __attribute__((ext_vector_type(4)));  // v_mfma_f64_16x16x4's accumulator

__device__ inline double readlane_f64(double v, int lane) {
  const int2 u = __builtin_bit_cast(int2, v);
  return __builtin_bit_cast(double, make_int2(__builtin_amdgcn_readlane(u.x, lane), __builtin_amdgcn_readlane(u.y, lane)));
}
// Lane kLane of every 16 lanes.
template <int kLane>
__device__ inline double row_lane_f64(double v) {
  const int2 u = __builtin_bit_cast(int2, v);
  constexpr int kCtrl = 0x150 + kLane;  // row_newbcast
  return __builtin_bit_cast(double, make_int2(__builtin_amdgcn_update_dpp(0, u.x, kCtrl, 0xf, 0xf, true),
                                              __builtin_amdgcn_update_dpp(0, u.y, kCtrl, 0xf, 0xf, true)));
}

// Sweeps pivots kP .. 15 of a symmetric 16 x 16 tile (lane l, value i: row
// 4 i + l / 16, column l % 16). False if a pivot is not positive.
template <int kP>
__device__ inline bool sweep_tile(double4v& t, int lane) {
  if constexpr (kP == kInvTile) {
    return true;
  } else {
    constexpr int kI = kP / 4, kG = kP % 4;
    const double p = readlane_f64(t[kI], 16 * kG + kP), ip = 1.0 / p;
    const double rowp = __shfl(t[kI], 16 * kG + (lane & 15));  // (p, own column)
    const double w = rowp * ip;
    const bool own_col = (lane & 15) == kP;
    double4v n;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const double colp = row_lane_f64<kP>(t[i]);  // (own row, p)
      n[i] = own_col ? colp * ip : fma(-colp, w, t[i]);
    }
    if ((lane >> 4) == kG) n[kI] = own_col ? -ip : w;
    t = n;
    return sweep_tile<kP + 1>(t, lane) && p > 0.0;
  }
}

// Solve set-up (one work-group): the PCG state, c = W'b, E^-1 by the sweep
// operator on the lower triangle (Goodnight, "A tutorial on the SWEEP
// operator", Amer. Statistician 33, 1979: sweeping pivot k of a symmetric A
// maps a_kk -> -1/a_kk, a_ik -> a_ik / a_kk, a_ij -> a_ij - a_ik a_kj / a_kk,
// keeps A symmetric, and sweeping every pivot gives -A^-1; E is SPD, so the
// pivots are the positive Cholesky pivots and no pivoting is needed). Then
// y = E^-1 c. A non-positive pivot disables deflation for this solve (E^-1 = 0,
// y = 0, defl_ok = 0).
//
// Sixteen pivots are swept at once: with the 16 x 16 tile A_kk swept (-P) by
// its wave, in registers, L_i = A_ik P for the other tile rows i, the panel
// becomes L and A_ij -= L_i A_jk'. The lower tiles stay in registers, two a
// wave, as the matrix instruction's accumulators; the panel and L go through
// LDS. One pivot at a time, every entry a register of one of 1024 threads, is
// a barrier, a divide and a column through LDS per pivot: 106 columns took
// about 100 us that way and take 35 so, 34 columns 13. Columns past ne are those
// of the identity.
__global__ __launch_bounds__(kPrepThreads) void k_defl_prep(PcgArgs a, double tol, int32_t max_iters) {
  __shared__ union {
    struct {
      double panel[2][kInvTiles * kInvTile][kInvPad];  // A_ik by row, of step k in panel[k & 1]
      double l[kInvTiles * kInvTile][kInvPad];
      double pinv[2][kInvTile][kInvPad];
    } s;
    double inv[kMaxCoarse * kMaxCoarse];
  } sh;
  __shared__ double cpart[kPrepThreads];
  __shared__ double cvec[kMaxCoarse];
  __shared__ int bad;
  const int ne = a.ne, tid = threadIdx.x;
  if (tid == 0) {
    PcgState* st = a.st;
    st->rz[0] = st->rz[1] = 0.0;
    st->bb = 0.0;
    st->tol_rel2 = tol * tol;
    st->tol2 = 0.0;
    st->iters = 0;
    st->done = 0;
    st->max_iters = max_iters;
    st->defl_ok = 0;
    st->arrive = 0;
    bad = 0;
  }
  if (ne == 0) return;
  // The wave's lower tiles (ti, tj), ti >= tj, row by row; ti = -1: none.
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), nt = (ne + kInvTile - 1) / kInvTile;
  const int lr = lane >> 4, lc = lane & 15;
  double4v v[kInvPerWave];
  int ti[kInvPerWave], tj[kInvPerWave];
#pragma unroll
  for (int m = 0; m < kInvPerWave; ++m) {
    int e = wave + m * kInvWaves, r = 0;
    while (e > r) e -= ++r;
    ti[m] = r < nt ? r : -1;
    tj[m] = e;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int row = kInvTile * r + 4 * i + lr, col = kInvTile * e + lc;
      v[m][i] = ti[m] < 0 ? 0.0 : (max(row, col) < ne ? a.E[(size_t)max(row, col) * ne + min(row, col)] : (row == col ? 1.0 : 0.0));
    }
  }
  // c = W'b: thread (column, g) sums the support rows lo + g, lo + g + G, ...
  // of a hat column; dense columns come from k_defl_dense.
  {
    const int G = kPrepThreads / ne, col = tid % ne, g = tid / ne, k = col / 6, comp = col % 6;
    double acc = 0.0;
    if (g < G) {
      if (col < a.neh) {
        for (int i = a.node_range[2 * k] + g; i <= a.node_range[2 * k + 1]; i += G)
          acc += hat_weight(a, i, k) * a.b[6 * i + comp];
      } else if (g == 0) {
        acc = a.cden[col - a.neh];
      }
    }
    cpart[tid] = acc;
    __syncthreads();
    if (tid < ne) {
      double c = 0.0;
      for (int gg = 0; gg < G; ++gg) c += cpart[gg * ne + tid];
      cvec[tid] = c;
    }
  }
  for (int k = 0; k < nt; ++k) {
    double(*panel)[kInvPad] = sh.s.panel[k & 1];
    double(*pinv)[kInvPad] = sh.s.pinv[k & 1];
    // The panel (the previous step's readers use the other buffer), and the
    // swept tile by the wave that holds it.
#pragma unroll
    for (int m = 0; m < kInvPerWave; ++m) {
      if (ti[m] > k && tj[m] == k)
#pragma unroll
        for (int i = 0; i < 4; ++i) panel[kInvTile * ti[m] + 4 * i + lr][lc] = v[m][i];
      if (ti[m] == k && tj[m] < k)
#pragma unroll
        for (int i = 0; i < 4; ++i) panel[kInvTile * tj[m] + lc][4 * i + lr] = v[m][i];
    }
#pragma unroll
    for (int m = 0; m < kInvPerWave; ++m)
      if (ti[m] == k && tj[m] == k) {
        const bool ok = sweep_tile<0>(v[m], lane);
        if (!ok && lane == 0) bad = 1;
#pragma unroll
        for (int i = 0; i < 4; ++i) pinv[4 * i + lr][lc] = -v[m][i];
      }
    __syncthreads();
    if (wave < nt && wave != k) {  // L_i = A_ik P
      double4v acc = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
      for (int q = 0; q < 4; ++q)
        acc = __builtin_amdgcn_mfma_f64_16x16x4f64(panel[kInvTile * wave + lc][4 * q + lr], pinv[4 * q + lr][lc], acc,
                                                   0, 0, 0);
#pragma unroll
      for (int i = 0; i < 4; ++i) sh.s.l[kInvTile * wave + 4 * i + lr][lc] = acc[i];
    }
    __syncthreads();
#pragma unroll
    for (int m = 0; m < kInvPerWave; ++m) {
      if (ti[m] < 0 || (ti[m] == k && tj[m] == k)) continue;
      if (tj[m] == k) {
#pragma unroll
        for (int i = 0; i < 4; ++i) v[m][i] = sh.s.l[kInvTile * ti[m] + 4 * i + lr][lc];
      } else if (ti[m] == k) {
#pragma unroll
        for (int i = 0; i < 4; ++i) v[m][i] = sh.s.l[kInvTile * tj[m] + lc][4 * i + lr];
      } else {
#pragma unroll
        for (int q = 0; q < 4; ++q)
          v[m] = __builtin_amdgcn_mfma_f64_16x16x4f64(-sh.s.l[kInvTile * ti[m] + lc][4 * q + lr],
                                                      panel[kInvTile * tj[m] + lc][4 * q + lr], v[m], 0, 0, 0);
      }
    }
  }
  __syncthreads();
  const bool ok = bad == 0;
  // E^-1 = -(swept matrix), both triangles (a diagonal tile is symmetric up to
  // rounding: its lower triangle counts).
#pragma unroll
  for (int m = 0; m < kInvPerWave; ++m) {
    if (ti[m] < 0) continue;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int row = kInvTile * ti[m] + 4 * i + lr, col = kInvTile * tj[m] + lc;
      if (row < ne && col <= row) {
        const double x = ok ? -v[m][i] : 0.0;
        sh.inv[row * ne + col] = x;
        sh.inv[col * ne + row] = x;
      }
    }
  }
  __syncthreads();
  const int n2 = ne * ne;
  for (int e = tid; e < n2; e += kPrepThreads) a.Einv[e] = sh.inv[e];
  if (tid == 0) a.st->defl_ok = ok ? 1 : 0;
  // y = E^-1 c: thread (row, part) sums a contiguous part of the columns.
  const int nparts = kPrepThreads / ne, row = tid % ne, part = tid / ne, len = (ne + nparts - 1) / nparts;
  double yv = 0.0;
  if (part < nparts)
    for (int c = part * len; c < min(ne, (part + 1) * len); ++c) yv += sh.inv[row * ne + c] * cvec[c];
  cpart[tid] = yv;
  __syncthreads();
  if (tid < ne) {
    double y = 0.0;
    for (int pp = 0; pp < nparts; ++pp) y += cpart[pp * ne + tid];
    a.y[tid] = y;
  }
}

// Operands of a group's partials that do not change during the solve, loaded
// into registers at the start of the per-group kernels (kGroupBlock threads)
// so that their latency overlaps the kernel's reductions: wave w holds the
// SW window columns w + 16 m, its lanes the group entries lane + 64 j; thread
// (row, part) of E^-1 holds the entries of its part of the window columns.
constexpr int kGroupWaves = kGroupBlock / 64;
constexpr int kSrCols = (kMaxCoarse + kGroupWaves - 1) / kGroupWaves;
constexpr int kSrRows = (kGroupThreads + 63) / 64;
constexpr int einv_per_thread() {
  int m = 0;
  for (int ne = 1; ne <= kMaxCoarse; ++ne) {
    const int parts = kGroupBlock / ne, len = (ne + parts - 1) / parts;
    m = len > m ? len : m;
  }
  return m;
}
constexpr int kEinvPer = einv_per_thread();

struct GroupLoads {
  double sr[kSrCols][kSrRows];
  double einv[kEinvPer];
};

// The E^-1 entries come from the per-group copy EinvW (addresses that do not
// depend on a prior load) or, with kFromEinv, from E^-1 itself.
template <bool kFromEinv>
__device__ inline void load_group(const PcgArgs& a, int g, GroupLoads& L) {
  const int ne = a.ne, tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
#pragma unroll
  for (int m = 0; m < kSrCols; ++m) {
    const int lc = wave + kGroupWaves * m;
#pragma unroll
    for (int j = 0; j < kSrRows; ++j) {
      const int t = lane + 64 * j;
      L.sr[m][j] = (ne && lc < a.gw && t < kGroupThreads) ? sr_col(a, g, lc)[t] : 0.0;
    }
  }
#pragma unroll
  for (int m = 0; m < kEinvPer; ++m) L.einv[m] = 0.0;
  if (ne == 0) return;
  const int nparts = kGroupBlock / ne, rrow = tid % ne, part = tid / ne, gw = a.gw;
  const int len = (gw + nparts - 1) / nparts;
  const int c0 = kFromEinv ? 6 * a.grp_lo[g] : 0;
  if (part < nparts) {
#pragma unroll
    for (int m = 0; m < kEinvPer; ++m) {
      const int lc = part * len + m;
      if (m < len && lc < gw) {
        if (kFromEinv) {
          const int gc = win_col(a, c0, lc);
          L.einv[m] = gc >= 0 ? a.Einv[(size_t)gc * ne + rrow] : 0.0;  // E^-1 is symmetric
        } else {
          L.einv[m] = a.EinvW[((size_t)g * gw + lc) * ne + rrow];
        }
      }
    }
  }
}

// Per-group partials of group g: out = {rz, rr, bb, E^-1 (SW)'z}; zloc holds
// the group's z (0 past the last row). (SW)'z is non-zero only on the group's
// window of columns, so E^-1 (SW)'z needs only those columns of E^-1 (window
// columns past the last coarse column have zero SW and E^-1 entries).
__device__ inline void group_partials(const PcgArgs& a, int g, const GroupLoads& L, const double* zloc, double rz,
                                      double rr, double bb, double* cs, double* mpart, double* out) {
  const int ne = a.ne, tid = threadIdx.x;
  if (tid == 0) {
    out[0] = rz;
    out[1] = rr;
    out[2] = bb;
  }
  if (ne == 0) return;
  const int wave = tid >> 6, lane = tid & 63, w = a.gw;
#pragma unroll
  for (int m = 0; m < kSrCols; ++m) {
    const int lc = wave + kGroupWaves * m;
    if (lc < w) {
      double s = 0.0;
#pragma unroll
      for (int j = 0; j < kSrRows; ++j) {
        const int t = lane + 64 * j;
        if (t < kGroupThreads) s += L.sr[m][j] * zloc[t];
      }
      s = wave_sum(s);
      if (lane == 0) cs[lc] = s;
    }
  }
  __syncthreads();
  const int nparts = kGroupBlock / ne, part = tid / ne, len = (w + nparts - 1) / nparts;
  double m = 0.0;
  if (part < nparts) {
#pragma unroll
    for (int j = 0; j < kEinvPer; ++j) {
      const int lc = part * len + j;
      if (j < len && lc < w) m += L.einv[j] * cs[lc];
    }
  }
  mpart[tid] = m;
  __syncthreads();
  if (tid < ne) {
    double mu = 0.0;
    for (int pp = 0; pp < nparts; ++pp) mu += mpart[pp * ne + tid];
    out[3 + tid] = mu;
  }
}

// With a.reduce1: the work-group that writes the last group's partials sums
// every group's, in group order (the order k_pcg_spmv sums them in without
// reduce1), into part1 and re-arms the counter. Which work-group arrives last
// does not change the sum.
// The partials are written by the first two waves (thread 0 and threads
// below ne <= 106); only they release their stores at device scope (an L2
// write-back, since each XCD has its own L2), and only the last work-group
// acquires (an L2 invalidate): a full fence in every wave of every
// work-group would invalidate the L2 under the other work-groups' loads.
// The summing work-group stages whole groups' partials through LDS (red,
// kRedChunk doubles), every load of a pass in flight at once.
static_assert(3 + kMaxCoarse <= 128, "the group partials are written by the first two waves");
constexpr int kRedChunk = 4096;
constexpr int kRedPer = kRedChunk / kGroupBlock;

__device__ inline void sum_partials_if_last(const PcgArgs& a, bool* last, double* red) {
  const int tid = threadIdx.x, stride = 3 + a.ne;
  if (tid < 128) __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
  __syncthreads();
  if (tid == 0) *last = atomicAdd(&a.st->arrive, 1u) == (uint32_t)a.groups - 1u;
  __syncthreads();
  if (!*last) return;
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");  // every group's partials are visible here
  const int per = kRedChunk / stride;
  double acc = 0.0;
  for (int g0 = 0; g0 < a.groups; g0 += per) {
    const int ng = min(per, a.groups - g0), n = ng * stride;
    const double* src = a.part2 + (size_t)g0 * stride;
    double v[kRedPer];
#pragma unroll
    for (int m = 0; m < kRedPer; ++m) {
      const int q = tid + kGroupBlock * m;
      v[m] = q < n ? src[q] : 0.0;
    }
    __syncthreads();  // the previous pass is summed
#pragma unroll
    for (int m = 0; m < kRedPer; ++m) red[tid + kGroupBlock * m] = v[m];
    __syncthreads();
    if (tid < stride) {
#pragma unroll 8
      for (int gg = 0; gg < ng; ++gg) acc += red[gg * stride + tid];
    }
  }
  if (tid < stride) a.part1[tid] = acc;
  if (tid == 0) a.st->arrive = 0u;
}

// t_e = (L_i^-1 r_i)_comp for entry e = 6 i + comp; rloc holds the group's r.
__device__ inline double lower_solve_entry(const PcgArgs& a, int row, int comp, const double* rloc, int base) {
  const double* Li = a.linv + (size_t)36 * row + 6 * comp;
  double s = 0.0;
  for (int m = 0; m <= comp; ++m) s += Li[m] * rloc[base + m];
  return s;
}

// x0 = W y, r0 = b - (SW) y, p = 0 on one group of rows per work-group; with
// block-Jacobi z0 = M^-1 r0 and the group's partials, with the learned
// preconditioner t0 = L^-1 r0 (k_pcg_lower, k_pcg_upper and
// k_defl_partials follow).
template <bool kLearned>
__global__ __launch_bounds__(kGroupBlock) void k_defl_init(PcgArgs a) {
  __shared__ double rloc[kGroupThreads];
  __shared__ double zloc[kGroupThreads];
  __shared__ double lds[48];
  __shared__ double cs[kMaxCoarse];
  __shared__ double mpart[kGroupBlock];
  __shared__ double ys[kMaxCoarse];
  const int ne = a.ne, tid = threadIdx.x, P = a.Pvar, g = blockIdx.x;
  GroupLoads L;
  if (!kLearned) load_group<true>(a, g, L);
  for (int c = tid; c < ne; c += blockDim.x) ys[c] = a.y[c];
  if (ne) {
    // The group's window rows of E^-1 for k_pcg_update.
    const int c0 = 6 * a.grp_lo[g];
    for (int e = tid; e < a.gw * ne; e += blockDim.x) {
      const int lc = e / ne, col = e - lc * ne, gc = win_col(a, c0, lc);
      a.EinvW[(size_t)g * a.gw * ne + e] = gc >= 0 ? a.Einv[(size_t)gc * ne + col] : 0.0;
    }
  }
  __syncthreads();
  const int row = g * kRowsPerGroup + tid / 6, comp = tid % 6;
  const bool active = tid < kGroupThreads && row < P;
  double rv = 0.0, bv = 0.0;
  if (active) {
    const int e = 6 * row + comp;
    bv = a.b[e];
    double sy = 0.0, xv = 0.0;
    if (ne) {
      const int c0 = 6 * a.grp_lo[g];
      for (int lc = 0; lc < a.gw; ++lc) {
        const int gc = win_col(a, c0, lc);
        if (gc >= 0) sy += sr_col(a, g, lc)[tid] * ys[gc];
      }
      const int n0 = a.hat_node[row];
      const double w0 = a.hat_w[2 * row], w1 = a.hat_w[2 * row + 1];
      xv = w0 * ys[6 * n0 + comp] + (w1 != 0.0 ? w1 * ys[6 * (n0 + 1) + comp] : 0.0);
      for (int c = 0; c < a.nr; ++c) xv += a.R[(size_t)c * a.n6 + e] * ys[a.neh + c];
    }
    rv = bv - sy;
    a.x[e] = xv;
    a.r[e] = rv;
    a.p0[e] = 0.0;
  }
  if (tid < kGroupThreads) rloc[tid] = rv;
  __syncthreads();
  if (kLearned) {
    if (active) a.t[6 * row + comp] = lower_solve_entry(a, row, comp, rloc, tid - comp);
    return;
  }
  double zv = 0.0;
  if (active) {
    const double* M = a.Minv + (size_t)36 * row + 6 * comp;
    const int base = tid - comp;
    for (int c = 0; c < 6; ++c) zv += M[c] * rloc[base + c];
    a.z[6 * row + comp] = zv;
  }
  if (tid < kGroupThreads) zloc[tid] = zv;
  double rz = rv * zv, rr = rv * rv, bb = bv * bv;
  block_sum3(rz, rr, bb, lds);
  group_partials(a, g, L, zloc, rz, rr, bb, cs, mpart, a.part2 + (size_t)g * (3 + ne));
  __shared__ bool last;
  __shared__ double red[kRedChunk];
  if (a.reduce1) sum_partials_if_last(a, &last, red);
}

// Iteration k: stops when |r|^2 <= tol2 or k = max_iters, else
// q = S p_k with p_k = z - W mu + beta p_{k-1}, evaluated as
// S z + beta S p_{k-1} - (SW) mu so that the row's block products (the bulk
// of the loads) do not wait for the sums of the previous update's per-group
// partials (r'z, r'r and mu); the own row's p_k is stored and
// part[i] = p_k,i . q_i. Thread t < 252 handles component t % 6 of every 42nd
// block of the row and window columns t / 6 + 42 m of (SW)_i. kReduced reads
// the summed partials (part1) instead of summing every group's.
template <bool kReduced>
__global__ __launch_bounds__(256) void k_pcg_spmv(PcgArgs a, int32_t k, const double* __restrict__ p_prev,
                                                  double* __restrict__ p_cur) {
  __shared__ double chunk[kReduced ? 1 : kPartChunk];
  __shared__ double sums[3 + kMaxCoarse];
  __shared__ double ysz[kGroupThreads], ysp[kGroupThreads], ysw[kGroupThreads];
  PcgState* st = a.st;
  const int32_t done = st->done, max_iters = st->max_iters;
  const double rz_prev = st->rz[(k + 1) & 1], tol2_prev = st->tol2, tol_rel2 = st->tol_rel2;
  const int ne = a.ne, tid = threadIdx.x, stride = 3 + ne;
  const int i = blockIdx.x, comp = tid % 6, g = tid / 6;
  // Every read of the work-group is issued before its first wait (each
  // dependent round of global loads costs microseconds): the state, the first
  // chunk of group partials, the row's own z, p_{k-1} and hat weights, (SW)_i
  // and the block products.
  constexpr int kChunkPer = kReduced ? 1 : kPartChunk / 256;
  const int per_chunk = kPartChunk / stride, ng0 = min(per_chunk, a.groups);
  double pre[kChunkPer];
  if (kReduced) {
    pre[0] = tid < stride ? a.part1[tid] : 0.0;
  } else {
#pragma unroll
    for (int m = 0; m < kChunkPer; ++m) {
      const int q = tid + 256 * m;
      pre[m] = q < ng0 * stride ? a.part2[q] : 0.0;
    }
  }
  double z_own = 0.0, p_own = 0.0, hw0 = 0.0, hw1 = 0.0, r_own[kMaxRitz];
  int hn0 = 0;
#pragma unroll
  for (int c = 0; c < kMaxRitz; ++c) r_own[c] = 0.0;
  if (tid < 6) {
    z_own = a.z[6 * i + tid];
    p_own = p_prev[6 * i + tid];
    if (ne) {
      hn0 = a.hat_node[i];
      hw0 = a.hat_w[2 * i];
      hw1 = a.hat_w[2 * i + 1];
#pragma unroll
      for (int c = 0; c < kMaxRitz; ++c)
        if (c < a.nr) r_own[c] = a.R[(size_t)c * a.n6 + 6 * i + tid];
    }
  }
  constexpr int kSwCols = (kMaxCoarse + kRowsPerGroup - 1) / kRowsPerGroup;
  double sz = 0.0, sp = 0.0, sw[kSwCols] = {};
  const int gi = i / kRowsPerGroup, c0 = 6 * (ne ? a.grp_lo[gi] : 0);
  if (tid < kGroupThreads) {
    const int rb = a.row_ptr[i], re = a.row_ptr[i + 1];
#pragma unroll 4
    for (int kb = rb + g; kb < re; kb += kRowsPerGroup) {
      const int j = a.col_var[kb];
      const double* srow = a.S + (size_t)36 * kb + 6 * comp;
#pragma unroll
      for (int c = 0; c < 6; ++c) {
        sz += srow[c] * a.z[6 * j + c];
        sp += srow[c] * p_prev[6 * j + c];
      }
    }
    if (ne) {
      const int t = 6 * (i - gi * kRowsPerGroup) + comp;
#pragma unroll
      for (int m = 0; m < kSwCols; ++m) {
        const int lc = g + m * kRowsPerGroup;
        if (lc < a.gw) sw[m] = sr_col(a, gi, lc)[t];
      }
    }
  }
  if (done) return;  // the same value in every thread of the work-group
  if (kReduced) {
    if (tid < stride) sums[tid] = pre[0];
  } else {
    // Fixed-order sum of the group partials, a chunk of whole groups per pass.
#pragma unroll
    for (int m = 0; m < kChunkPer; ++m) chunk[tid + 256 * m] = pre[m];
    __syncthreads();
    double acc = 0.0;
    if (tid < stride) {
#pragma unroll 8
      for (int gg = 0; gg < ng0; ++gg) acc += chunk[gg * stride + tid];
    }
    for (int g0 = ng0; g0 < a.groups; g0 += per_chunk) {
      const int ng = min(per_chunk, a.groups - g0);
      __syncthreads();
      for (int q = tid; q < ng * stride; q += blockDim.x) chunk[q] = a.part2[(size_t)g0 * stride + q];
      __syncthreads();
      if (tid < stride) {
#pragma unroll 8
        for (int gg = 0; gg < ng; ++gg) acc += chunk[gg * stride + tid];
      }
    }
    if (tid < stride) sums[tid] = acc;
  }
  __syncthreads();
  const double* mu_s = sums + 3;
  const double rz = sums[0], rr = sums[1];
  double tol2;
  bool stop;
  if (k == 0) {
    const double bb = sums[2];
    tol2 = tol_rel2 * bb;
    stop = bb <= 0.0 || max_iters <= 0 || rr <= tol2;
    if (blockIdx.x == 0 && tid == 0) {
      st->bb = bb;
      st->tol2 = tol2;
    }
  } else {
    tol2 = tol2_prev;
    stop = rr <= tol2 || k >= max_iters;
  }
  if (stop) {
    if (blockIdx.x == 0 && tid == 0) {
      st->iters = k;
      st->done = 1;
    }
    return;
  }
  const double beta = k > 0 ? rz / rz_prev : 0.0;
  if (blockIdx.x == 0 && tid == 0) {
    st->rz[k & 1] = rz;
    st->iters = k;
    if (k < a.zcap) a.coef[2 * k] = rz;
  }
  if (tid < kGroupThreads) {
    double w = 0.0;
    if (ne) {
#pragma unroll
      for (int m = 0; m < kSwCols; ++m) {
        const int lc = g + m * kRowsPerGroup, gc = lc < a.gw ? win_col(a, c0, lc) : -1;
        if (gc >= 0) w += sw[m] * mu_s[gc];
      }
    }
    ysz[tid] = sz;
    ysp[tid] = sp;
    ysw[tid] = w;
  }
  __syncthreads();
  if (tid < 6) {
    double qz = 0.0, qp = 0.0, qw = 0.0;
#pragma unroll 6
    for (int gg = 0; gg < kRowsPerGroup; ++gg) {
      qz += ysz[6 * gg + tid];
      qp += ysp[6 * gg + tid];
      qw += ysw[6 * gg + tid];
    }
    const double qa = qz + beta * qp - qw;
    double zh = z_own;  // deflated preconditioned residual z - W mu
    if (ne) {
      double wm = hw0 * mu_s[6 * hn0 + tid] + (hw1 != 0.0 ? hw1 * mu_s[6 * (hn0 + 1) + tid] : 0.0);
#pragma unroll
      for (int c = 0; c < kMaxRitz; ++c)
        if (c < a.nr) wm += r_own[c] * mu_s[a.neh + c];
      zh -= wm;
    }
    const double pa = zh + beta * p_own;
    a.q[6 * i + tid] = qa;
    p_cur[6 * i + tid] = pa;
    if (k < a.zcap) a.Zh[(size_t)k * a.n6 + 6 * i + tid] = zh;
    ysz[tid] = pa * qa;
  }
  __syncthreads();
  if (tid == 0) a.part[i] = ((ysz[0] + ysz[1]) + (ysz[2] + ysz[3])) + (ysz[4] + ysz[5]);
}

// alpha = r'z / p'q; x += alpha p; r -= alpha q on one group of rows per
// work-group; with block-Jacobi z = M^-1 r and the group's partials r'z, r'r,
// E^-1 (SW)'z, with the learned preconditioner t = L^-1 r (k_pcg_lower,
// k_pcg_upper and k_defl_partials follow).
template <bool kLearned>
__global__ __launch_bounds__(kGroupBlock) void k_pcg_update(PcgArgs a, int32_t k, const double* __restrict__ p_cur) {
  __shared__ double rloc[kGroupThreads];
  __shared__ double zloc[kGroupThreads];
  __shared__ double lds[48];
  __shared__ double cs[kMaxCoarse];
  __shared__ double mpart[kGroupBlock];
  const PcgState* st = a.st;
  const int32_t done = st->done;
  const double rz = st->rz[k & 1];
  const int ne = a.ne, tid = threadIdx.x, P = a.Pvar, g = blockIdx.x;
  const int row = g * kRowsPerGroup + tid / 6, comp = tid % 6;
  const bool active = tid < kGroupThreads && row < P;
  GroupLoads L;
  if (!kLearned) load_group<false>(a, g, L);
  // The group's vectors and preconditioner rows (M^-1 or L^-1), loaded
  // before the reduction.
  double xv = 0.0, pv = 0.0, rv = 0.0, qv = 0.0, M[6] = {};
  if (active) {
    const int e = 6 * row + comp;
    xv = a.x[e];
    pv = p_cur[e];
    rv = a.r[e];
    qv = a.q[e];
    const double* Mr = (kLearned ? a.linv : a.Minv) + (size_t)36 * row + 6 * comp;
#pragma unroll
    for (int c = 0; c < 6; ++c) M[c] = (!kLearned || c <= comp) ? Mr[c] : 0.0;
  }
  // p'q, summed by every group in the same order.
  double pq = 0.0, unused0 = 0.0, unused1 = 0.0;
  for (int r = tid; r < P; r += blockDim.x) pq += a.part[r];
  if (done) return;  // the same value in every thread
  block_sum3(pq, unused0, unused1, lds);
  const double alpha = rz / pq;
  if (g == 0 && tid == 0 && k < a.zcap) a.coef[2 * k + 1] = alpha;
  if (active) {
    const int e = 6 * row + comp;
    a.x[e] = xv + alpha * pv;
    rv -= alpha * qv;
    a.r[e] = rv;
  }
  if (tid < kGroupThreads) rloc[tid] = rv;
  __syncthreads();
  double zv = 0.0;
  if (active) {
    const int base = tid - comp;
#pragma unroll
    for (int c = 0; c < 6; ++c) zv += M[c] * rloc[base + c];
    (kLearned ? a.t : a.z)[6 * row + comp] = zv;
  }
  if (kLearned) return;
  if (tid < kGroupThreads) zloc[tid] = zv;
  double rzg = rv * zv, rr = rv * rv, zero = 0.0;
  block_sum3(rzg, rr, zero, lds);
  group_partials(a, g, L, zloc, rzg, rr, 0.0, cs, mpart, a.part2 + (size_t)g * (3 + ne));
  __shared__ bool last;
  __shared__ double red[kRedChunk];
  if (a.reduce1) sum_partials_if_last(a, &last, red);
}

// Learned preconditioner, after t = L^-1 r: u_i = t_i - sum_{j < i} K_ij t_j,
// one wave per row (lanes take every 64th lower block, then a fixed-order
// wave sum).
__global__ __launch_bounds__(64) void k_pcg_lower(PcgArgs a) {
  if (a.st->done) return;
  const int i = blockIdx.x, lane = threadIdx.x;
  double acc[6] = {0, 0, 0, 0, 0, 0};
  for (int pos = a.row_ptr[i] + lane; pos < a.diag_pos[i]; pos += 64) {
    const int j = a.col_var[pos];
    const float* K = a.kmat + (size_t)36 * pos;
    const double* tj = a.t + 6 * (size_t)j;
#pragma unroll
    for (int r = 0; r < 6; ++r) {
      double s = 0.0;
#pragma unroll
      for (int c = 0; c < 6; ++c) s += (double)K[6 * r + c] * tj[c];
      acc[r] += s;
    }
  }
#pragma unroll
  for (int r = 0; r < 6; ++r) acc[r] = wave_sum(acc[r]);
  if (lane < 6) {
    double v = acc[0];
#pragma unroll
    for (int r = 1; r < 6; ++r)
      if (lane == r) v = acc[r];
    a.u[6 * i + lane] = a.t[6 * i + lane] - v;
  }
}

// w_j = u_j - sum_{i > j} K_ij' u_i, z_j = L_j^-T w_j; one wave per row (K_ij
// is stored in row i, at the transposed position of block (j, i)).
__global__ __launch_bounds__(64) void k_pcg_upper(PcgArgs a) {
  __shared__ double w[6];
  if (a.st->done) return;
  const int j = blockIdx.x, lane = threadIdx.x;
  double acc[6] = {0, 0, 0, 0, 0, 0};
  for (int pos = a.diag_pos[j] + 1 + lane; pos < a.row_ptr[j + 1]; pos += 64) {
    const int i = a.col_var[pos];
    const float* K = a.kmat + (size_t)36 * a.tpos[pos];
    const double* ui = a.u + 6 * (size_t)i;
#pragma unroll
    for (int c = 0; c < 6; ++c) {
      double s = 0.0;
#pragma unroll
      for (int r = 0; r < 6; ++r) s += (double)K[6 * r + c] * ui[r];
      acc[c] += s;
    }
  }
#pragma unroll
  for (int c = 0; c < 6; ++c) acc[c] = wave_sum(acc[c]);
  if (lane < 6) {
    double v = acc[0];
#pragma unroll
    for (int c = 1; c < 6; ++c)
      if (lane == c) v = acc[c];
    w[lane] = a.u[6 * j + lane] - v;
  }
  __syncthreads();
  if (lane < 6) {
    const double* Lj = a.linv + (size_t)36 * j;
    double s = 0.0;
    for (int m = lane; m < 6; ++m) s += Lj[6 * m + lane] * w[m];
    a.z[6 * j + lane] = s;
  }
}

// Learned preconditioner: the group's partials r'z, r'r (b'b with
// `with_b`) and E^-1 (SW)'z from r and z, one group of rows per work-group,
// as k_pcg_update and k_defl_init form them with block-Jacobi.
__global__ __launch_bounds__(kGroupBlock) void k_defl_partials(PcgArgs a, int32_t with_b) {
  __shared__ double zloc[kGroupThreads];
  __shared__ double lds[48];
  __shared__ double cs[kMaxCoarse];
  __shared__ double mpart[kGroupBlock];
  const int32_t done = a.st->done;
  const int ne = a.ne, tid = threadIdx.x, P = a.Pvar, g = blockIdx.x;
  const int row = g * kRowsPerGroup + tid / 6, comp = tid % 6;
  const bool active = tid < kGroupThreads && row < P;
  GroupLoads L;
  load_group<false>(a, g, L);
  double rv = 0.0, zv = 0.0, bv = 0.0;
  if (active) {
    const int e = 6 * row + comp;
    rv = a.r[e];
    zv = a.z[e];
    if (with_b) bv = a.b[e];
  }
  if (done) return;  // the same value in every thread
  if (tid < kGroupThreads) zloc[tid] = zv;
  double rz = rv * zv, rr = rv * rv, bb = bv * bv;
  block_sum3(rz, rr, bb, lds);
  group_partials(a, g, L, zloc, rz, rr, bb, cs, mpart, a.part2 + (size_t)g * (3 + ne));
  __shared__ bool last;
  __shared__ double red[kRedChunk];
  if (a.reduce1) sum_partials_if_last(a, &last, red);
}

// Plain block-Jacobi PCG of a small system in one work-group, for systems
// without a coarse space (the automatic space starts at 32 vertices). A
// system of 10 keyframes needs about 40 iterations, and as two launches each
// they cost 10.5 us an iteration on MI355X (launch and two dependent rounds
// of global loads, not the 54 x 54 product): 450 us a solve, 3.6 ms of the
// 6.3 ms that 10 LM iterations took (2.7 ms with this). Here an iteration is
// 2.0 us (37 of them 75 us, set-up included). S stays in
// registers, dense: wave w holds columns 12 w .. 12 w + 11 of rows lane,
// lane + 64 and lane + 128 (36 doubles a thread, which is what 1024 threads
// leave room for and why 31 vertices are the limit); the waves' sums of a row
// meet in LDS, and wave 0 keeps the vectors, so an iteration is two barriers.
// Sums run in a fixed order.
constexpr int kSmallVertices = 31;
// A launch that cannot stop early (a residual that is not a number, a tolerance
// below what 64 bits reach) runs all its iterations: at 2 us each at most 33 ms go
// into one launch; a larger cap is iterated by launches that the host polls.
constexpr int kSmallIterations = 16384;
constexpr int kSmallRows = 192;
constexpr int kSmallWaves = 16;
constexpr int kSmallCols = kSmallRows / kSmallWaves;  // two blocks of columns a wave
constexpr int kSmallRowsPerLane = kSmallRows / 64;

__global__ __launch_bounds__(64 * kSmallWaves) void k_pcg_small(PcgArgs a, double tol, int32_t max_iters,
                                                                double* __restrict__ iters_out) {
  __shared__ double red[kSmallWaves][kSmallRows];
  __shared__ double ps[kSmallRows], rs[kSmallRows], xs[kSmallRows], Ms[6][kSmallRows];
  __shared__ int16_t pos[32][32];
  __shared__ int stop;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, n = a.n6, P = a.Pvar;
  const int bi = tid >> 5;  // block row
  pos[bi][tid & 31] = -1;
  __syncthreads();
  if (bi < P)
    for (int kb = a.row_ptr[bi] + (tid & 31); kb < a.row_ptr[bi + 1]; kb += 32) pos[bi][a.col_var[kb]] = (int16_t)kb;
  __syncthreads();
  double s[kSmallRowsPerLane][kSmallCols];
#pragma unroll
  for (int j = 0; j < kSmallRowsPerLane; ++j) {
    const int row = lane + 64 * j;
#pragma unroll
    for (int h = 0; h < kSmallCols / 6; ++h) {
      const int kb = row < n ? pos[row / 6][kSmallCols / 6 * wave + h] : -1;
      const double* sb = a.S + (size_t)36 * max(kb, 0) + 6 * (row % 6);
#pragma unroll
      for (int c = 0; c < 6; ++c) s[j][6 * h + c] = kb >= 0 ? sb[c] : 0.0;
    }
  }
  // Wave 0's vectors (rows lane + 64 j) live in LDS, the registers are S's;
  // z takes red[0], which holds wave 0's own sums only between the barriers.
  double rz = 0.0, rr = 0.0, tol2 = 0.0;
  auto apply_minv = [&]() {
    // rs is written and read by wave 0 alone.
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    double t0 = 0.0, t1 = 0.0;
#pragma unroll
    for (int j = 0; j < kSmallRowsPerLane; ++j) {
      const int row = lane + 64 * j, base = row - row % 6;
      double v = 0.0;
#pragma unroll
      for (int c = 0; c < 6; ++c) v += Ms[c][row] * rs[base + c];
      red[0][row] = v;
      const double rv = rs[row];
      t0 += rv * v;
      t1 += rv * rv;
    }
    rz = wave_sum(t0);
    rr = wave_sum(t1);
  };
  if (wave == 0) {
    for (int row = lane; row < kSmallRows; row += 64) {
      xs[row] = ps[row] = 0.0;
      rs[row] = row < n ? a.b[row] : 0.0;
      for (int c = 0; c < 6; ++c) Ms[c][row] = row < n ? a.Minv[(size_t)6 * row + c] : 0.0;
    }
    apply_minv();
    tol2 = tol * tol * rr;
  }
  double rz_prev = 0.0;
  int k = 0;
  while (true) {
    if (wave == 0) {
      const bool end = k == 0 ? (rr <= 0.0 || max_iters <= 0 || rr <= tol2) : (rr <= tol2 || k >= max_iters);
      const double beta = k > 0 ? rz / rz_prev : 0.0;
      rz_prev = rz;
#pragma unroll
      for (int j = 0; j < kSmallRowsPerLane; ++j) ps[lane + 64 * j] = red[0][lane + 64 * j] + beta * ps[lane + 64 * j];
      if (lane == 0) stop = end;
    }
    __syncthreads();
    if (stop) break;  // the same value in every thread
    double acc[kSmallRowsPerLane] = {};
#pragma unroll
    for (int c = 0; c < kSmallCols; ++c) {
      const double pc = ps[kSmallCols * wave + c];
#pragma unroll
      for (int j = 0; j < kSmallRowsPerLane; ++j) acc[j] += s[j][c] * pc;
    }
#pragma unroll
    for (int j = 0; j < kSmallRowsPerLane; ++j) red[wave][lane + 64 * j] = acc[j];
    __syncthreads();
    if (wave == 0) {
      double q[kSmallRowsPerLane], t = 0.0;
#pragma unroll
      for (int j = 0; j < kSmallRowsPerLane; ++j) {
        q[j] = 0.0;
#pragma unroll 4
        for (int w = 0; w < kSmallWaves; ++w) q[j] += red[w][lane + 64 * j];
        t += ps[lane + 64 * j] * q[j];
      }
      const double alpha = rz / wave_sum(t);
#pragma unroll
      for (int j = 0; j < kSmallRowsPerLane; ++j) {
        const int row = lane + 64 * j;
        xs[row] += alpha * ps[row];
        rs[row] -= alpha * q[j];
      }
      apply_minv();
    }
    ++k;
  }
  if (wave == 0) {
    for (int row = lane; row < n; row += 64) a.x[row] = xs[row];
    if (lane == 0) *iters_out = (double)k;
  }
}

// ------------------------------------------------------------ block-Jacobi step

// One PCG iteration in one launch. A launch that reads what the one before it
// wrote costs several us here whatever it computes (launch, then dependent
// rounds of global loads), and an iteration as a product and an update was
// two of them. CG needs a global sum for alpha = r'z / p's (s = S p) and a
// second one after it, r'z and the deflation's c = (SW)'z - W'r of the new z and
// r. The second follows from the first by linearity: with v = M s formed at the
// end of an iteration,
//   r+ = r - alpha s, z+ = z - alpha v,
//   r+'z+ = r'z - 2 alpha s'z + alpha^2 s'v,   r+'r+ alike,
//   c+ = c - alpha ((SW)'v - W's),
// so one launch sums all of these and the next one starts from them: each row
// takes r+, its own z+ = M r+ (formed anew, so that the recurrences for the
// scalars run over one iteration only), mu = E^-1 c+ of its window, and the
// product of its row with z+ = z - alpha v and p as three sums that do not
// wait for alpha. c is carried over at most kStepRefresh iterations and then
// summed anew from z and r: carried through the whole solve, its rounding error
// stays at 1e-16 of the first c while r falls, and the residual stagnates at
// 1e-11. W'r is zero but for the errors of the c before it, which reach r through
// W mu; the direction z - W E^-1 c takes them out again (the A-DEF2 operator of
// Tang, Nabben, Vuik and Erlangga, J. Sci. Comput. 39, 2009). With c = (SW)'z
// they stay: a 1500-keyframe ring took 57 iterations for 49, its recycled columns
// came to depend on the hat functions, and the next solve did not converge. The
// term costs 0.3 us an iteration.
//
// A work-group of 1024 threads takes G rows, so that at most 256 work-groups
// (one a CU) publish the partials that every work-group sums. Component t % 6
// of every kBlocks-th block of a row is thread t's; with one row a work-group
// three quarters of the waves have no product and sum the partials meanwhile.
// A work-group reads about 0.4 MB (its rows of S, E^-1 and 256 x 113 partials),
// and the kernel is bound by that behind four dependent rounds of loads: more
// rows with fewer work-groups (500 keyframes: 125 work-groups 18.8 us, 250
// 15.5 us) and the partials summed once by the work-group that ends last
// (24 us) are slower. Sums run in a fixed order.
//
// Where it pays (step_pays; MI355X, whole solves with the 15-node space, two
// launches -> one, us an iteration). A work-group has G rows of B blocks and
// takes them side by side, so its product lasts as long as G B blocks, where the
// two launches give every row a work-group and grow with the vertices:
//   up to 512 vertices (G <= 2) always: walks 60 vertices 18 -> 12, 500 33.5 ->
//     27.6; rings that every keyframe sees whole, B = vertices: 120 20.8 -> 15.7,
//     256 24.3 -> 20.8, 512 34.1 -> 30.3;
//   up to 1024 (G = 4) from 5 B vertices on: 1000 vertices (B 155) 27.6 -> 24.3,
//     800 (152) 23.2 -> 23.2, 1000 (201) 31.8 -> 31.6, 600 (150) 22.5 -> 23.6, 800
//     (211) 28.4 -> 31.0, rings 600 40 -> 45, 1000 79 -> 82;
//   up to 2048 (G = 8) from 12 B vertices on: 2000 (149) 37.7 -> 32.6, 2040 (186)
//     46.9 -> 46.3, 1400 (156) 34.2 -> 33.2, 1050 (155) 27.4 -> 31.3, 1600 (172)
//     38.8 -> 41.2, 1200 (206) 33.2 -> 46.0, rings 1100 136 -> 197, 2000 287 -> 311;
//   above 2048, 256 work-groups of 8 rows, a compute unit runs two of them one
//     after the other: 2300 39.7 -> 60.1, 4000 57.2 -> 68.6, 5000 64.5 -> 102.
constexpr int kStepScalars = 7;  // p's, r'z, s'z, s'v, r'r, r's, s's (k_pcg_start: r'z, r'r, b'b in 1, 4, 5)
constexpr int kStepStride = kStepScalars + kMaxCoarse;
constexpr int kStepThreads = 1024;
constexpr int kStepFlight = 16;  // a thread's partials in flight
constexpr int kStepVertices = 2048;
constexpr int kStepRefresh = 8;  // every launch k with k % 8 = 0 sums (SW)'z as well
constexpr double kStepCancel = 1e-12;  // r'r by recurrence holds to about 1e-15 of the last one: 3 digits here
static_assert(kStepStride <= 128, "128 threads hold the partials of one work-group");

int32_t step_rows(int32_t Pvar) {
  return Pvar <= 256 ? 1 : (Pvar <= 512 ? 2 : (Pvar <= 1024 ? 4 : 8));
}
int32_t step_wgs(int32_t Pvar) { return (Pvar + step_rows(Pvar) - 1) / step_rows(Pvar); }

template <int G>
struct StepShape {
  static constexpr int kProduct = G == 1 ? 256 : kStepThreads;  // threads of the products
  static constexpr int kT = kProduct / G;                       // threads of a row
  static constexpr int kBlocks = (kT < 256 ? kT : 256) / 6;     // blocks of a row at once
  static constexpr int kFirst = kProduct < kStepThreads ? kProduct : 0;  // first thread of the sums
  static constexpr int kSlices = (kStepThreads - kFirst) / 128;
  static constexpr int kCols = (kMaxCoarse + kBlocks - 1) / kBlocks;
  static constexpr int kRitz = (kMaxRitz + kBlocks - 1) / kBlocks;
};

// Slice sl (the same in a wave) of entry t of the sum of wgs work-groups' partials.
template <int kSlices>
__device__ inline double step_slice(const double* part, int wgs, int stride, int t, int sl) {
  double acc = 0.0;
  if (t >= stride) return acc;
  // The loads of a pass differ by a uniform number of bytes.
  const uint32_t own = 8u * (uint32_t)t;
  for (int w0 = sl; w0 < wgs; w0 += kStepFlight * kSlices) {
    double v[kStepFlight];
#pragma unroll
    for (int m = 0; m < kStepFlight; ++m) {
      const int w = w0 + m * kSlices;
      const char* row = reinterpret_cast<const char*>(part + (size_t)min(w, wgs - 1) * stride);
      v[m] = *reinterpret_cast<const double*>(row + own);
      if (w >= wgs) v[m] = 0.0;
    }
#pragma unroll
    for (int m = 0; m < kStepFlight; ++m) acc += v[m];
  }
  return acc;
}

// A row's hat part of W: its nodes n, n + 1 and their weights.
struct StepHat {
  int32_t n;
  double w0, w1;
};

// Entry of W in a row's component comp and hat column gc.
__device__ inline double hat_entry(const StepHat& h, int gc, int comp) {
  const int node = gc / 6;
  if (gc - 6 * node != comp) return 0.0;
  return node == h.n ? h.w0 : (node == h.n + 1 ? h.w1 : 0.0);
}

// Coarse column e of the sum over a work-group's rows of the window products
// tmp[row][window column][component] and, to be subtracted, the dense columns'
// den[row][column][component].
template <int G>
__device__ inline double step_column(const PcgArgs& a, int i0, int e, const double (*tmp)[kMaxCoarse][6],
                                     const double (*den)[kMaxRitz][6]) {
  double s = 0.0;
#pragma unroll
  for (int g = 0; g < G; ++g) {
    if (i0 + g < a.Pvar) {
      const int lc = e >= a.neh ? a.gwh + (e - a.neh) : e - 6 * a.grp_lo[(i0 + g) / kRowsPerGroup];
      if (lc >= 0 && lc < a.gw && (e >= a.neh || lc < a.gwh)) {
        const double* t = tmp[g][lc];
        s += ((t[0] + t[1]) + (t[2] + t[3])) + (t[4] + t[5]);
        if (e >= a.neh) {
          const double* d = den[g][e - a.neh];
          s -= ((d[0] + d[1]) + (d[2] + d[3])) + (d[4] + d[5]);
        }
      }
    }
  }
  return s;
}

// Publishes a work-group's partials: the scalars over its rows' entries
// (sc[e]) and the coarse columns of tmp.
template <int G>
__device__ inline void step_publish(const PcgArgs& a, int i0, const double (*sc)[kStepScalars],
                                    const double (*tmp)[kMaxCoarse][6], const double (*den)[kMaxRitz][6],
                                    double* part) {
  const int tid = threadIdx.x, stride = kStepScalars + a.ne;
  double* out = part + (size_t)blockIdx.x * stride;
  if (tid < kStepScalars) {
    double s = 0.0;
#pragma unroll
    for (int e = 0; e < 6 * G; ++e) s += sc[e][tid];
    out[tid] = s;
  } else if (tid < stride) {
    out[tid] = step_column<G>(a, i0, tid - kStepScalars, tmp, den);
  }
}

// x0 = W y, r0 = b - (SW) y, z0 = M r0, p = v = s = 0 and the first partials.
template <int G>
__global__ __launch_bounds__(kStepThreads) void k_pcg_start(PcgArgs a) {
  using Sh = StepShape<G>;
  __shared__ double sc[6 * G][kStepScalars];
  __shared__ double tmp[G][kMaxCoarse][6];
  __shared__ double ys[kMaxCoarse], rows[G][6], rowr[G][6], den[G][kMaxRitz][6], red[G][Sh::kBlocks][6];
  __shared__ StepHat hat[G];
  const int tid = threadIdx.x, i0 = blockIdx.x * G, ne = a.ne;
  const int g = min(tid / Sh::kT, G - 1), t = tid - g * Sh::kT, comp = t % 6, bs = t / 6, i = i0 + g;
  const bool row_ok = i < a.Pvar, lane_in = t < 6 * Sh::kBlocks, lane_ok = row_ok && lane_in;
  const int gi = row_ok ? i / kRowsPerGroup : 0, c0 = ne ? 6 * a.grp_lo[gi] : 0;
  for (int c = tid; c < ne; c += kStepThreads) ys[c] = a.y[c];
  double sw[Sh::kCols] = {};
  if (ne && lane_ok) {
#pragma unroll
    for (int m = 0; m < Sh::kCols; ++m) {
      const int lc = bs + Sh::kBlocks * m;
      if (lc < a.gw) sw[m] = sr_col(a, gi, lc)[6 * (i - gi * kRowsPerGroup) + comp];
    }
  }
  __syncthreads();
  if (lane_in) {
    double sy = 0.0;
    if (ne) {
#pragma unroll
      for (int m = 0; m < Sh::kCols; ++m) {
        const int lc = bs + Sh::kBlocks * m, gc = lc < a.gw ? win_col(a, c0, lc) : -1;
        if (gc >= 0) sy += sw[m] * ys[gc];
      }
    }
    red[g][bs][comp] = sy;
  }
  __syncthreads();
  if (t < 6) {
    double rv = 0.0, bv = 0.0, zv = 0.0, M[6];
    const int e = 6 * i + comp;
    if (row_ok) {
      double xv = 0.0, s = 0.0;
      bv = a.b[e];
      for (int k = 0; k < Sh::kBlocks; ++k) s += red[g][k][comp];
      if (ne) {
        const int n0 = a.hat_node[i];
        const double w0 = a.hat_w[2 * i], w1 = a.hat_w[2 * i + 1];
        if (comp == 0) hat[g] = StepHat{n0, w0, w1};
        xv = w0 * ys[6 * n0 + comp] + (w1 != 0.0 ? w1 * ys[6 * (n0 + 1) + comp] : 0.0);
        for (int c = 0; c < a.nr; ++c) xv += a.R[(size_t)c * a.n6 + e] * ys[a.neh + c];
      }
      rv = bv - s;
      a.x[e] = xv;
      a.r[e] = rv;
      a.q[e] = 0.0;
    }
#pragma unroll
    for (int c = 0; c < 6; ++c) M[c] = row_ok ? a.Minv[(size_t)36 * i + 6 * comp + c] : 0.0;
#pragma unroll
    for (int c = 0; c < 6; ++c) zv += M[c] * __shfl(rv, (tid & 63) - comp + c);
    if (row_ok) {
      double* o = a.zvp + (size_t)18 * i + comp;
      o[0] = zv;
      o[6] = 0.0;
      o[12] = 0.0;
    }
    rows[g][comp] = zv;
    rowr[g][comp] = rv;
    double* o = sc[6 * g + comp];
    o[0] = o[2] = o[3] = o[6] = 0.0;
    o[1] = rv * zv;
    o[4] = rv * rv;
    o[5] = bv * bv;
  }
  __syncthreads();
  if (ne && lane_in) {
    const double z = rows[g][comp], r = rowr[g][comp];
#pragma unroll
    for (int m = 0; m < Sh::kCols; ++m) {
      const int lc = bs + Sh::kBlocks * m;
      if (lc < kMaxCoarse) tmp[g][lc][comp] = sw[m] * z - (row_ok && lc < a.gwh ? hat_entry(hat[g], c0 + lc, comp) * r : 0.0);
    }
#pragma unroll
    for (int m = 0; m < Sh::kRitz; ++m) {
      const int c = bs + Sh::kBlocks * m;
      if (c < kMaxRitz) den[g][c][comp] = row_ok && c < a.nr ? a.R[(size_t)c * a.n6 + 6 * i + comp] * r : 0.0;
    }
  }
  __syncthreads();
  step_publish<G>(a, i0, sc, tmp, den, a.spart);
}

// Iteration k: takes step k - 1 (x, r), then stops when |r|^2 <= tol2 or
// k = max_iters, else forms direction k and its product. Where |r|^2 was too
// small a difference to stop on, launch k + 1 finds it summed and stops without
// a step, after k iterations.
template <int G>
__global__ __launch_bounds__(kStepThreads) void k_pcg_step(PcgArgs a, int32_t k) {
  using Sh = StepShape<G>;
  __shared__ double sc[6 * G][kStepScalars];
  __shared__ double tmp[G][kMaxCoarse][6];
  __shared__ double lds[Sh::kSlices][128], ldz[Sh::kSlices][128];
  __shared__ double sums[128], cs[kMaxCoarse], mus[kMaxCoarse], rows[G][6], rowz[G][6], rowq[G][6], rowr[G][6];
  __shared__ double red[G][Sh::kBlocks][6], wred[G][kMaxRitz][6];
  __shared__ StepHat hat[G];
  PcgState* st = a.st;
  const int odd = k & 1, ne = a.ne, stride = kStepScalars + ne;
  const double* __restrict__ in = a.zvp + (odd ? (size_t)18 * a.Pvar : 0);
  double* __restrict__ out = a.zvp + (odd ? 0 : (size_t)18 * a.Pvar);
  const double* __restrict__ c_in = a.cvec + (odd ? kMaxCoarse : 0);
  double* __restrict__ c_out = a.cvec + (odd ? 0 : kMaxCoarse);
  const int tid = threadIdx.x, i0 = blockIdx.x * G;
  const int g = min(tid / Sh::kT, G - 1), t = tid - g * Sh::kT, comp = t % 6, bs = t / 6, i = i0 + g;
  const bool row_ok = i < a.Pvar, lane_in = t < 6 * Sh::kBlocks, lane_ok = row_ok && lane_in;
  const bool fresh = k > 0 && (k - 1) % kStepRefresh == 0;  // (SW)'z of the last launch was summed anew
  // done is 1 + the launch that stopped: a work-group of that launch which
  // starts late still takes the last step.
  const int32_t done = st->done, max_iters = st->max_iters;
  const double tol2_prev = st->tol2, tol_rel2 = st->tol_rel2;
  // Coarse columns of the work-group's windows: hat columns ulo .. ulo + nh, then the dense ones.
  const int gi = row_ok ? i / kRowsPerGroup : 0;
  const int c0 = ne ? 6 * a.grp_lo[gi] : 0;
  int ulo = 0, nh = 0;
  if (ne) {
    const int la = 6 * a.grp_lo[i0 / kRowsPerGroup], lb = 6 * a.grp_lo[(min(i0 + G, a.Pvar) - 1) / kRowsPerGroup];
    ulo = min(la, lb);
    nh = min(max(la, lb) + a.gwh, a.neh) - ulo;
  }
  // Slice of the sums, the same in a wave.
  const int tc = (tid - Sh::kFirst) & 127;
  const int sl = __builtin_amdgcn_readfirstlane(tid >= Sh::kFirst ? (tid - Sh::kFirst) >> 7 : kStepThreads);
  const int nu = nh + a.nr, uc = tc < nh ? ulo + tc : a.neh + (tc - nh);
  constexpr int kEinvCols = (kMaxCoarse + Sh::kSlices - 1) / Sh::kSlices;
  double sw[Sh::kCols] = {}, rc[Sh::kRitz] = {}, ei[kEinvCols] = {};
  double az = 0.0, av = 0.0, ap = 0.0;
  double xv = 0.0, rv = 0.0, sv = 0.0, pv = 0.0, hw0 = 0.0, hw1 = 0.0, M[6] = {};
  int hn0 = 0;
  if (lane_ok) {
    const int re = a.row_ptr[i + 1];
#pragma unroll 2
    for (int kb = a.row_ptr[i] + bs; kb < re; kb += Sh::kBlocks) {
      const double2* x2 = reinterpret_cast<const double2*>(in + (size_t)18 * a.col_var[kb]);
      const double2* s2 = reinterpret_cast<const double2*>(a.S + (size_t)36 * kb + 6 * comp);
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        const double2 sb = s2[c], zz = x2[c], vv = x2[3 + c], pp = x2[6 + c];
        az += sb.x * zz.x;
        az += sb.y * zz.y;
        av += sb.x * vv.x;
        av += sb.y * vv.y;
        ap += sb.x * pp.x;
        ap += sb.y * pp.y;
      }
    }
    if (ne) {
#pragma unroll
      for (int m = 0; m < Sh::kCols; ++m) {
        const int lc = bs + Sh::kBlocks * m;
        if (lc < a.gw) sw[m] = sr_col(a, gi, lc)[6 * (i - gi * kRowsPerGroup) + comp];
      }
#pragma unroll
      for (int m = 0; m < Sh::kRitz; ++m) {
        const int c = bs + Sh::kBlocks * m;
        if (c < a.nr) rc[m] = a.R[(size_t)c * a.n6 + 6 * i + comp];
      }
    }
    if (t < 6) {
      const int e = 6 * i + comp;
      xv = a.x[e];
      rv = a.r[e];
      sv = a.q[e];
      pv = in[(size_t)18 * i + 12 + comp];
#pragma unroll
      for (int c = 0; c < 6; ++c) M[c] = a.Minv[(size_t)36 * i + 6 * comp + c];
      if (ne) {
        hn0 = a.hat_node[i];
        hw0 = a.hat_w[2 * i];
        hw1 = a.hat_w[2 * i + 1];
      }
    }
  }
  __builtin_amdgcn_sched_barrier(0);
  if (sl < Sh::kSlices) {
#pragma unroll
    for (int m = 0; m < kEinvCols; ++m) {
      const int c = sl + Sh::kSlices * m;
      ei[m] = tc < nu && c < ne ? a.Einv[(size_t)c * ne + uc] : 0.0;
    }
    if (fresh)
      ldz[sl][tc] = step_slice<Sh::kSlices>(a.zpart, a.wgs, ne, tc, sl);
    else if (sl == 0 && tc < ne)
      cs[tc] = k > 0 ? c_in[tc] : 0.0;
    lds[sl][tc] = step_slice<Sh::kSlices>(a.spart + (odd ? (size_t)a.wgs * stride : 0), a.wgs, stride, tc, sl);
  }
  if (done && done != k + 1) return;  // the same value in every thread
  __syncthreads();
  if (tid < stride) {
    double s = 0.0;
#pragma unroll
    for (int q = 0; q < Sh::kSlices; ++q) s += lds[q][tid];
    sums[tid] = s;
  }
  if (fresh && tid < ne) {
    double s = 0.0;
#pragma unroll
    for (int q = 0; q < Sh::kSlices; ++q) s += ldz[q][tid];
    cs[tid] = s;
  }
  __syncthreads();
  const double rz_old = sums[1];
  double rz = rz_old, rr = sums[4], alpha = 0.0, beta = 0.0, tol2 = tol2_prev;
  bool stop, take = k > 0;  // take: step k - 1 is taken
  if (k == 0) {
    const double bb = sums[5];
    tol2 = tol_rel2 * bb;
    stop = bb <= 0.0 || max_iters <= 0 || rr <= tol2;
  } else if (rr <= tol2) {
    // The last launch's r'r, summed from r itself, was small enough.
    stop = true;
    take = false;
  } else {
    alpha = rz_old / sums[0];
    // r'r and r'z of the new r are differences of numbers as large as the old
    // ones. A result below kStepCancel of r'r has few or no digits left and may
    // come out negative: it stops nothing, this launch sums r'r anew.
    rz += alpha * (alpha * sums[3] - 2.0 * sums[2]);
    rr += alpha * (alpha * sums[6] - 2.0 * sums[5]);
    beta = rz < 0.0 ? 0.0 : rz / rz_old;
    stop = (rr <= tol2 && rr > kStepCancel * sums[4]) || k >= max_iters;
  }
  if (t < 6 && lane_ok && take) {
    const int e = 6 * i + comp;
    rv -= alpha * sv;
    a.x[e] = xv + alpha * pv;
    a.r[e] = rv;
  }
  if (blockIdx.x == 0 && tid == 0) {
    if (k == 0) {
      st->bb = sums[5];
      st->tol2 = tol2;
    } else if (take && k - 1 < a.zcap) {
      a.coef[2 * (k - 1) + 1] = alpha;
    }
    if (!stop && k < a.zcap) a.coef[2 * k] = rz;
    st->iters = k > 0 && !take ? k - 1 : k;
    if (stop) st->done = k + 1;
  }
  if (stop) return;  // the same value in every thread
  // c, and mu = E^-1 c on the work-group's windows.
  const double ca = k > 0 ? -alpha : 1.0;  // cs is zero at k = 0
  if (blockIdx.x == 0 && tid < ne) c_out[tid] = cs[tid] + ca * sums[kStepScalars + tid];
  if (sl < Sh::kSlices) {
    double mp = 0.0;
#pragma unroll
    for (int m = 0; m < kEinvCols; ++m) {
      const int c = sl + Sh::kSlices * m;
      if (c < ne) mp += ei[m] * (cs[c] + ca * sums[kStepScalars + c]);
    }
    lds[sl][tc] = mp;
  }
  __syncthreads();
  if (tid >= Sh::kFirst && tid - Sh::kFirst < nu) {
    double m = 0.0;
#pragma unroll
    for (int q = 0; q < Sh::kSlices; ++q) m += lds[q][tc];
    mus[uc] = m;
  }
  __syncthreads();
  if (lane_in) {
    double y = az - alpha * av + beta * ap;
    if (ne) {
#pragma unroll
      for (int m = 0; m < Sh::kCols; ++m) {
        const int lc = bs + Sh::kBlocks * m, gc = lc < a.gw ? win_col(a, c0, lc) : -1;
        if (gc >= 0) y -= sw[m] * mus[gc];
      }
#pragma unroll
      for (int m = 0; m < Sh::kRitz; ++m) {
        const int c = bs + Sh::kBlocks * m;
        if (c < kMaxRitz) wred[g][c][comp] = c < a.nr ? rc[m] * mus[a.neh + c] : 0.0;
      }
    }
    red[g][bs][comp] = y;
  }
  __syncthreads();
  if (t < 6) {
    double q = 0.0, zv = 0.0, vv = 0.0;
#pragma unroll
    for (int b = 0; b < Sh::kBlocks; ++b) q += red[g][b][comp];
#pragma unroll
    for (int c = 0; c < 6; ++c) {
      const int l = (tid & 63) - comp + c;
      zv += M[c] * __shfl(rv, l);
      vv += M[c] * __shfl(q, l);
    }
    double zh = zv;  // deflated preconditioned residual z - W mu
    if (ne) {
      double wm = hw0 != 0.0 ? hw0 * mus[6 * hn0 + comp] : 0.0;
      if (hw1 != 0.0) wm += hw1 * mus[6 * (hn0 + 1) + comp];
#pragma unroll
      for (int c = 0; c < kMaxRitz; ++c) wm += wred[g][c][comp];
      zh -= wm;
    }
    const double pn = zh + beta * pv;
    if (row_ok) {
      double* o = out + (size_t)18 * i + comp;
      o[0] = zv;
      o[6] = vv;
      o[12] = pn;
      a.q[6 * i + comp] = q;
      if (k < a.zcap) a.Zh[(size_t)k * a.n6 + 6 * i + comp] = zh;
    }
    rows[g][comp] = row_ok ? vv : 0.0;
    rowz[g][comp] = row_ok ? zv : 0.0;
    rowq[g][comp] = row_ok ? q : 0.0;
    rowr[g][comp] = row_ok ? rv : 0.0;
    if (comp == 0) hat[g] = StepHat{hn0, hw0, hw1};
    double* o = sc[6 * g + comp];
    o[0] = row_ok ? pn * q : 0.0;
    o[1] = row_ok ? rv * zv : 0.0;
    o[2] = row_ok ? q * zv : 0.0;
    o[3] = row_ok ? q * vv : 0.0;
    o[4] = row_ok ? rv * rv : 0.0;
    o[5] = row_ok ? rv * q : 0.0;
    o[6] = row_ok ? q * q : 0.0;
  }
  __syncthreads();
  if (ne && lane_in) {
    const double v = rows[g][comp], q = rowq[g][comp];
    const StepHat h = hat[g];
#pragma unroll
    for (int m = 0; m < Sh::kCols; ++m) {
      const int lc = bs + Sh::kBlocks * m;
      if (lc < kMaxCoarse) tmp[g][lc][comp] = sw[m] * v - (lc < a.gwh ? hat_entry(h, c0 + lc, comp) * q : 0.0);
    }
#pragma unroll
    for (int m = 0; m < Sh::kRitz; ++m) {
      const int c = bs + Sh::kBlocks * m;
      if (c < kMaxRitz) wred[g][c][comp] = rc[m] * q;
    }
  }
  __syncthreads();
  step_publish<G>(a, i0, sc, tmp, wred, a.spart + (odd ? 0 : (size_t)a.wgs * stride));
  if (k % kStepRefresh != 0 || ne == 0) return;
  __syncthreads();
  if (lane_in) {
    const double z = rowz[g][comp], r = rowr[g][comp];
    const StepHat h = hat[g];
#pragma unroll
    for (int m = 0; m < Sh::kCols; ++m) {
      const int lc = bs + Sh::kBlocks * m;
      if (lc < kMaxCoarse) tmp[g][lc][comp] = sw[m] * z - (lc < a.gwh ? hat_entry(h, c0 + lc, comp) * r : 0.0);
    }
#pragma unroll
    for (int m = 0; m < Sh::kRitz; ++m) {
      const int c = bs + Sh::kBlocks * m;
      if (c < kMaxRitz) wred[g][c][comp] = rc[m] * r;
    }
  }
  __syncthreads();
  if (tid < ne) a.zpart[(size_t)blockIdx.x * ne + tid] = step_column<G>(a, i0, tid, tmp, wred);
}

// Clears the convergence flag and lifts the iteration limit so that one more
// iteration runs (kernel timing only).
__global__ void k_pcg_reopen(PcgState* st) {
  st->done = 0;
  st->max_iters = st->iters + 2;
  st->tol2 = -1.0;
}

// ------------------------------------------------------------ recycling
// After a solve, Ritz vectors of its Lanczos process (Saad, Yeung, Erhel,
// Guyomarc'h 2000, sec. 4; Stathopoulos & Orginos, "Computing and deflating
// eigenvalues while solving multiple right-hand side linear systems", SIAM
// J. Sci. Comput. 32, 2010): the stored deflated preconditioned residuals
// z_k - W mu_k, scaled by 1 / sqrt(r_k'z_k), are the Lanczos vectors of the
// deflated preconditioned operator, and the CG coefficients give its
// tridiagonal matrix. The host takes the eigenvectors of that tridiagonal
// for its smallest eigenvalues (Y), k_ritz_form forms Rn = Zh' Y, and a
// Rayleigh-Ritz step on span[R, Rn] with respect to (S, M) (k_row_dense for S Rn,
// k_ritz_gram, a small generalized eigenproblem on the host, k_ritz_merge)
// keeps the best r vectors for the next solve.

constexpr int kRitzFormThreads = 256;
constexpr int kMaxLanczos = 64;

// Rn[c] = sum_j Zh[j] Y[j][c], one thread per (entry, column).
__global__ __launch_bounds__(kRitzFormThreads) void k_ritz_form(int32_t n6, int32_t m, int32_t r,
                                                                const double* __restrict__ Zh,
                                                                const double* __restrict__ Y, double* __restrict__ Rn) {
  __shared__ double Ys[kMaxLanczos];
  const int c = blockIdx.y;
  for (int t = threadIdx.x; t < m; t += blockDim.x) Ys[t] = Y[t * r + c];
  __syncthreads();
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= n6) return;
  double acc = 0.0;
#pragma unroll 8
  for (int j = 0; j < m; ++j) acc += Zh[(size_t)j * n6 + e] * Ys[j];
  Rn[(size_t)c * n6 + e] = acc;
}

// Gram matrices of Y = [R | Rn], one work-group per entry (a, b):
// A_ab = Y_a'(S Y_b) (S R from the group windows of this solve's SW),
// B_ab = Y_a'(M Y_b) with M the 6x6 diagonal blocks of S.
__global__ __launch_bounds__(256) void k_ritz_gram(PcgArgs a, int32_t r, const double* __restrict__ Rn,
                                                   const double* __restrict__ SRn, const int32_t* __restrict__ diag_pos,
                                                   double* __restrict__ AB) {
  __shared__ double lds[4];
  const int ia = blockIdx.x, ib = blockIdx.y, nb = a.nr + r;
  const double* Ya = ia < a.nr ? a.R + (size_t)ia * a.n6 : Rn + (size_t)(ia - a.nr) * a.n6;
  const double* Yb = ib < a.nr ? a.R + (size_t)ib * a.n6 : Rn + (size_t)(ib - a.nr) * a.n6;
  double sa = 0.0, sb = 0.0;
  for (int e = threadIdx.x; e < a.n6; e += blockDim.x) {
    const double sy = ib < a.nr ? sw_entry(a, e, a.neh + ib) : SRn[(size_t)(ib - a.nr) * a.n6 + e];
    const int i = e / 6, comp = e % 6;
    const double* Mi = a.S + (size_t)36 * diag_pos[i] + 6 * comp;
    const double* yb = Yb + 6 * i;
    const double my = ((Mi[0] * yb[0] + Mi[1] * yb[1]) + (Mi[2] * yb[2] + Mi[3] * yb[3])) + (Mi[4] * yb[4] + Mi[5] * yb[5]);
    sa += Ya[e] * sy;
    sb += Ya[e] * my;
  }
  sa = block_sum256(sa, lds);
  __syncthreads();
  sb = block_sum256(sb, lds);
  if (threadIdx.x == 0) {
    AB[(size_t)ia * nb + ib] = sa;
    AB[(size_t)nb * nb + (size_t)ia * nb + ib] = sb;
  }
}

// Rnext[c] = sum_a R[a] Cm[a][c] + sum_a Rn[a] Cm[nr_old + a][c], one
// thread per (entry, column).
__global__ __launch_bounds__(256) void k_ritz_merge(int32_t n6, const double* __restrict__ R, int32_t nr_old,
                                                    const double* __restrict__ Rn, int32_t r,
                                                    const double* __restrict__ Cm, int32_t r_next,
                                                    double* __restrict__ Rnext) {
  __shared__ double Cs[2 * kMaxRitz];
  const int nb = nr_old + r, c = blockIdx.y;
  for (int t = threadIdx.x; t < nb; t += blockDim.x) Cs[t] = Cm[t * r_next + c];
  __syncthreads();
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= n6) return;
  double acc = 0.0;
  for (int ia = 0; ia < nb; ++ia)
    acc += (ia < nr_old ? R[(size_t)ia * n6 + e] : Rn[(size_t)(ia - nr_old) * n6 + e]) * Cs[ia];
  Rnext[(size_t)c * n6 + e] = acc;
}

// ------------------------------------------------------------ launchers

size_t pcg_state_bytes() { return sizeof(PcgState); }
int32_t pcg_max_hat_nodes() { return kMaxHatNodes; }
int32_t pcg_max_ritz() { return kMaxRitz; }
int32_t pcg_max_lanczos() { return kMaxLanczos; }
int32_t pcg_group_rows() { return kRowsPerGroup; }
int32_t pcg_update_groups(int32_t Pvar) { return (Pvar + kRowsPerGroup - 1) / kRowsPerGroup; }
bool pcg_deflation_applied(const void* state_host) {
  return static_cast<const PcgState*>(state_host)->defl_ok != 0;
}

static PcgArgs make_args(const PcgBuffers& B) {
  PcgArgs a;
  a.Pvar = B.Pvar;
  a.K = B.K;
  a.neh = 6 * B.K;
  a.nr = B.K > 0 ? B.nr : 0;
  a.ne = a.neh + a.nr;
  a.groups = pcg_update_groups(B.Pvar);
  a.gwh = B.gwh;
  a.gw = B.gwh + a.nr;
  a.n6 = 6 * B.Pvar;
  a.zcap = std::min(B.zcap, kMaxLanczos);
  a.pad2 = a.pad3 = 0;
  a.row_ptr = B.row_ptr; a.col_var = B.col_var; a.S = B.S; a.Minv = B.Minv; a.b = B.b;
  a.hat_node = B.hat_node; a.hat_w = B.hat_w; a.node_range = B.node_range; a.grp_lo = B.grp_lo; a.R = B.R;
  a.blk_hat = B.blk_hat; a.blk_w = B.blk_w; a.blk_rng = B.blk_rng;
  a.SR = B.SR; a.E = B.E; a.Einv = B.Einv; a.EinvW = B.Einv + (size_t)a.ne * a.ne;
  a.x = B.x; a.r = B.r; a.z = B.z; a.p0 = B.p0; a.p1 = B.p1; a.q = B.q;
  a.part = B.part; a.part2 = B.part2; a.y = B.y; a.cden = B.cden; a.Zh = B.Zh; a.coef = B.coef;
  // part2 holds groups + 1 rows of partials; the last one is part1.
  a.part1 = B.part2 + (size_t)a.groups * (3 + a.ne);
  a.reduce1 = B.partials == 0 ? (a.groups > kPartChunk / (3 + a.ne) ? 1 : 0) : (B.partials == 2 ? 1 : 0);
  a.pad4 = 0;
  a.step_G = step_rows(a.Pvar);
  a.wgs = step_wgs(a.Pvar);
  a.zvp = B.step;
  a.cvec = a.zvp + 36 * (size_t)a.Pvar;
  a.spart = a.cvec + 2 * kMaxCoarse;
  a.zpart = a.spart + 2 * (size_t)a.wgs * kStepStride;
  a.st = static_cast<PcgState*>(B.state_dev);
  a.linv = B.linv; a.kmat = B.kmat; a.diag_pos = B.diag_pos; a.tpos = B.tpos; a.t = B.t; a.u = B.u;
  return a;
}

// With the learned preconditioner: z = L^-T (I - K)' (I - K) t after t = L^-1 r,
// then the group partials.
static void launch_learned_z(hipStream_t s, const PcgArgs& a, int32_t with_b) {
  k_pcg_lower<<<a.Pvar, 64, 0, s>>>(a);
  k_pcg_upper<<<a.Pvar, 64, 0, s>>>(a);
  k_defl_partials<<<a.groups, kGroupBlock, 0, s>>>(a, with_b);
}

static void launch_update(hipStream_t s, const PcgArgs& a, int32_t k, const double* p_cur) {
  if (a.kmat) {
    k_pcg_update<true><<<a.groups, kGroupBlock, 0, s>>>(a, k, p_cur);
    launch_learned_z(s, a, 0);
  } else {
    k_pcg_update<false><<<a.groups, kGroupBlock, 0, s>>>(a, k, p_cur);
  }
}

static void launch_spmv(hipStream_t s, const PcgArgs& a, int32_t k, const double* p_prev, double* p_cur) {
  if (a.reduce1)
    k_pcg_spmv<true><<<a.Pvar, 256, 0, s>>>(a, k, p_prev, p_cur);
  else
    k_pcg_spmv<false><<<a.Pvar, 256, 0, s>>>(a, k, p_prev, p_cur);
}

static void launch_step_start(hipStream_t s, const PcgArgs& a) {
  switch (a.step_G) {
    case 1: k_pcg_start<1><<<a.wgs, kStepThreads, 0, s>>>(a); break;
    case 2: k_pcg_start<2><<<a.wgs, kStepThreads, 0, s>>>(a); break;
    case 4: k_pcg_start<4><<<a.wgs, kStepThreads, 0, s>>>(a); break;
    default: k_pcg_start<8><<<a.wgs, kStepThreads, 0, s>>>(a);
  }
}

static void launch_step(hipStream_t s, const PcgArgs& a, int32_t k) {
  switch (a.step_G) {
    case 1: k_pcg_step<1><<<a.wgs, kStepThreads, 0, s>>>(a, k); break;
    case 2: k_pcg_step<2><<<a.wgs, kStepThreads, 0, s>>>(a, k); break;
    case 4: k_pcg_step<4><<<a.wgs, kStepThreads, 0, s>>>(a, k); break;
    default: k_pcg_step<8><<<a.wgs, kStepThreads, 0, s>>>(a, k);
  }
}

// Whether an iteration in one launch is the faster form (k_pcg_step): S has at
// most a fifth, with eight rows a work-group a twelfth, of its blocks.
static bool step_pays(int32_t Pvar, int64_t nnzb) {
  if (Pvar <= 0 || Pvar > kStepVertices) return false;
  const int32_t G = step_rows(Pvar);
  const int64_t sparse = G <= 2 ? 0 : (G == 4 ? 5 : 12);
  return (int64_t)Pvar * Pvar >= sparse * nnzb;
}

bool pcg_step_applies(const PcgBuffers& B) { return B.kmat == nullptr && step_pays(B.Pvar, B.nnzb); }

size_t pcg_step_doubles(int32_t Pvar, int64_t nnzb) {
  if (!step_pays(Pvar, nnzb)) return 0;
  return 36 * (size_t)Pvar + 2 * kMaxCoarse + (size_t)step_wgs(Pvar) * (2 * kStepStride + kMaxCoarse);
}

bool pcg_small_applies(const PcgBuffers& B, int32_t max_iters) {
  return B.K == 0 && B.kmat == nullptr && B.Pvar > 0 && B.Pvar <= kSmallVertices && max_iters <= kSmallIterations;
}

bool launch_pcg_small(hipStream_t s, const PcgBuffers& B, double tol, int32_t max_iters, double* iters_out) {
  if (!pcg_small_applies(B, max_iters)) return false;
  k_pcg_small<<<1, 64 * kSmallWaves, 0, s>>>(make_args(B), tol, max_iters, iters_out);
  return hipGetLastError() == hipSuccess;
}

// Deflated PCG solve of S y = b. The host polls the state after `first`
// iterations, then every `poll` iterations. With `probe` (three events), the
// kernels of one more iteration (k_pcg_step, or k_pcg_spmv and then
// k_pcg_update) are each launched `probe_reps` times back to back after the
// solve and timed as two batches, the second empty with k_pcg_step (x, r and
// z then hold extra steps). Returns the iteration count or -1 on a launch
// error.
int launch_pcg_deflated(hipStream_t s, const PcgBuffers& B, double tol, int32_t max_iters, int32_t first,
                        int32_t poll, const hipEvent_t* probe, int32_t probe_reps) {
  const int32_t Pvar = B.Pvar;
  if (Pvar <= 0) return 0;
  if (B.K > kMaxHatNodes || B.nr > kMaxRitz || B.nr < 0) return -1;
  const bool learned = B.kmat != nullptr, step = pcg_step_applies(B);
  if (learned && (B.nr > 0 || B.zcap > 0 || probe || !B.linv || !B.diag_pos || !B.tpos || !B.t || !B.u)) return -1;
  const PcgArgs a = make_args(B);
  double* p0 = B.p0;
  double* p1 = B.p1;
  const int groups = a.groups;
  if (a.ne > 0) {
    k_defl_sr<<<Pvar, 256, 0, s>>>(a);
    if (a.nr > 0)
      k_row_dense<true><<<Pvar, kDenseThreads, 0, s>>>(a, a.row_ptr, a.col_var, a.S, a.R, a.nr, a.n6, nullptr);
    k_defl_e<<<dim3(a.K, a.ne), 64, 0, s>>>(a);
    if (a.nr > 0) k_defl_dense<<<dim3(a.nr, a.nr + 1), 256, 0, s>>>(a);
  }
  k_defl_prep<<<1, kPrepThreads, 0, s>>>(a, tol, max_iters);
  if (learned) {
    k_defl_init<true><<<groups, kGroupBlock, 0, s>>>(a);
    launch_learned_z(s, a, 1);
  } else if (step) {
    launch_step_start(s, a);
  } else {
    k_defl_init<false><<<groups, kGroupBlock, 0, s>>>(a);
  }
  PcgState* hs = static_cast<PcgState*>(B.state_host);
  int k = 0;
  while (true) {
    const int n = std::min(k == 0 ? std::max(first, 1) : poll, max_iters - k);
    for (int j = 0; j < n; ++j, ++k) {
      if (step) {
        launch_step(s, a, k);
      } else {
        launch_spmv(s, a, k, (k & 1) ? p1 : p0, (k & 1) ? p0 : p1);
        launch_update(s, a, k, (k & 1) ? p0 : p1);
      }
    }
    // At k = max_iters this launch only records the final state (k_pcg_step
    // also takes the last step).
    if (k >= max_iters) {
      if (step) launch_step(s, a, k);
      else launch_spmv(s, a, k, p0, p1);
    }
    if (hipMemcpyAsync(hs, a.st, sizeof(PcgState), hipMemcpyDeviceToHost, s) != hipSuccess) return -1;
    if (hipStreamSynchronize(s) != hipSuccess) return -1;
    if (hs->done || k >= max_iters) break;
  }
  if (hipGetLastError() != hipSuccess) return -1;
  const int iters = hs->iters;
  if (probe && iters > 0) {
    // Re-open the state for one timed iteration k = iters.
    k_pcg_reopen<<<1, 1, 0, s>>>(a.st);
    const int kk = iters;
    if (hipEventRecord(probe[0], s) != hipSuccess) return -1;
    for (int j = 0; j < probe_reps; ++j) {
      if (step) launch_step(s, a, kk);
      else launch_spmv(s, a, kk, (kk & 1) ? p1 : p0, (kk & 1) ? p0 : p1);
    }
    if (hipEventRecord(probe[1], s) != hipSuccess) return -1;
    for (int j = 0; j < probe_reps && !step; ++j) k_pcg_update<false><<<groups, kGroupBlock, 0, s>>>(a, kk, (kk & 1) ? p0 : p1);
    if (hipEventRecord(probe[2], s) != hipSuccess) return -1;
    if (hipGetLastError() != hipSuccess) return -1;
  }
  return iters;
}

void launch_ritz_form(hipStream_t s, int32_t Pvar, int32_t m, int32_t r, const double* Zh, const double* Y,
                      double* Rn) {
  const int n6 = 6 * Pvar;
  if (n6 <= 0 || m <= 0 || m > kMaxLanczos || r <= 0 || r > kMaxRitz) return;
  k_ritz_form<<<dim3((n6 + kRitzFormThreads - 1) / kRitzFormThreads, r), kRitzFormThreads, 0, s>>>(n6, m, r, Zh, Y,
                                                                                                 Rn);
}

void launch_ritz_spmv(hipStream_t s, int32_t Pvar, int32_t r, const int32_t* row_ptr, const int32_t* col_var,
                      const double* S, const double* Rn, double* SRn) {
  if (Pvar <= 0 || r <= 0 || r > kMaxRitz) return;
  k_row_dense<false><<<Pvar, kDenseThreads, 0, s>>>(PcgArgs{}, row_ptr, col_var, S, Rn, r, 6 * Pvar, SRn);
}

void launch_ritz_gram(hipStream_t s, const PcgBuffers& B, int32_t r, const double* Rn, const double* SRn,
                      const int32_t* diag_pos, double* AB) {
  const PcgArgs a = make_args(B);
  const int nb = a.nr + r;
  if (B.Pvar <= 0 || r <= 0 || r > kMaxRitz || a.K <= 0) return;
  k_ritz_gram<<<dim3(nb, nb), 256, 0, s>>>(a, r, Rn, SRn, diag_pos, AB);
}

void launch_ritz_merge(hipStream_t s, int32_t Pvar, const double* R, int32_t nr_old, const double* Rn, int32_t r,
                       const double* Cm, int32_t r_next, double* Rnext) {
  const int n6 = 6 * Pvar;
  if (n6 <= 0 || r_next <= 0 || r_next > kMaxRitz || nr_old + r > 2 * kMaxRitz) return;
  k_ritz_merge<<<dim3((n6 + 255) / 256, r_next), 256, 0, s>>>(n6, R, nr_old, Rn, r, Cm, r_next, Rnext);
}

}  // namespace mlba
