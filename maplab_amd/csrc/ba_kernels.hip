// ba_kernels.hip -- gfx950 kernels of the visual bundle-adjustment path.
//
// One LM iteration on the device (names match the launchers at the bottom):
//   k_vertex_prep     R_I_M and |q|^2 of every vertex (state or candidate)
//   k_linearize<1>    per observation: residual, its Jacobian by the landmark
//                     in the IMU frame, robust correction
//                     (VisualReprojectionError::Evaluate + ceres Corrector);
//                     per landmark: V, g reductions in LDS
//   k_linearize<0>    the same chain, cost only (candidate evaluation)
//   k_pose_rows       per variable vertex: unscaled gradient, diag(F'F) and
//                     the direct observation block sum Jo^T Jo
//   k_schur_factors   per factor block, per linearization: P, p and k
//   k_landmark_prep   per landmark: T of Z = C (C V C + D^2)^-1 C = T'T, T g and
//                     the anchor's factor and self product
//   k_schur_tiles     partial sums of the upper blocks of the reduced camera
//                     system S over segments of 16 x 16-block tiles
//   k_schur_finalize  S blocks and rhs from the partials, both triangles
//   k_block_inverse   block-Jacobi preconditioner (6x6 inverses of diag(S))
//   (ba_pcg.hip)      deflated block-Jacobi PCG on S
//   k_back_substitute landmark step and the LM model cost change
//   k_step_vertices   vertex step and x (+) step (JPL Plus)
//   k_candidate_landmarks
//   k_gradient_norm   max |x - Plus(x, -g)|
//   k_evaluate_full   every reference Jacobian block (Evaluate parity API)
// All reductions are fixed-order (per-tile partials summed by one block,
// S blocks by one wave each, the tile sums of a landmark split over several
// linearization tiles added in tile order), so results repeat bit for bit
// run to run.
#include <hip/hip_ext.h>

#include "ba_device.h"
#include "ba_math.h"
#include "ba_reduce.h"
#include "ba_tiles.h"

namespace mlba {

// ------------------------------------------------------------ utilities

// L^-1 (rows i00; i10 i11; i20 i21 i22) of the Cholesky factor L of a symmetric
// positive definite 3x3 matrix given as (xx xy xz yy yz zz); returns false
// when not positive definite.
__device__ inline bool spd3_inverse_factor(const double* a, double* out) {
  const double l00 = sqrt(a[0]);
  if (!(l00 > 0.0)) return false;
  const double l10 = a[1] / l00, l20 = a[2] / l00;
  const double d11 = a[3] - l10 * l10;
  if (!(d11 > 0.0)) return false;
  const double l11 = sqrt(d11);
  const double l21 = (a[4] - l20 * l10) / l11;
  const double d22 = a[5] - l20 * l20 - l21 * l21;
  if (!(d22 > 0.0)) return false;
  const double l22 = sqrt(d22);
  const double i00 = 1.0 / l00, i11 = 1.0 / l11, i22 = 1.0 / l22;
  const double i10 = -l10 * i00 * i11;
  const double i21 = -l21 * i11 * i22;
  out[0] = i00;
  out[1] = i10;
  out[2] = i11;
  out[3] = -(l20 * i00 + l21 * i10) * i22;
  out[4] = i21;
  out[5] = i22;
  return true;
}

// T x and T'x of a lower-triangular 3x3 T (rows t0; t1 t2; t3 t4 t5).
__device__ inline void tri_vec(const double* t, const double* x, double* out) {
  out[0] = t[0] * x[0];
  out[1] = t[1] * x[0] + t[2] * x[1];
  out[2] = t[3] * x[0] + t[4] * x[1] + t[5] * x[2];
}
__device__ inline void trit_vec(const double* t, const double* x, double* out) {
  out[0] = t[0] * x[0] + t[1] * x[1] + t[3] * x[2];
  out[1] = t[2] * x[1] + t[4] * x[2];
  out[2] = t[5] * x[2];
}

__device__ inline void sym3_full(const double* s, double* m) {
  m[0] = s[0]; m[1] = s[1]; m[2] = s[2];
  m[3] = s[1]; m[4] = s[3]; m[5] = s[4];
  m[6] = s[2]; m[7] = s[4]; m[8] = s[5];
}

// Anchor map M = [-|q_a|^2 [p_B]x , R_B_LM] (3x6): the anchor-vertex
// tangent Jacobian of an observation is J_landmark * M
// (visual-error-term-inl.h:199-224 with the JPL lift).
__device__ inline void anchor_map(const double* pB, const double* Ra, double n2, double* M) {
  // -n2 [p]x = -n2 [[0,-z,y],[z,0,-x],[-y,x,0]]
  M[0] = 0.0;         M[1] = n2 * pB[2];  M[2] = -n2 * pB[1];
  M[6] = -n2 * pB[2]; M[7] = 0.0;         M[8] = n2 * pB[0];
  M[12] = n2 * pB[1]; M[13] = -n2 * pB[0]; M[14] = 0.0;
  for (int r = 0; r < 3; ++r)
    for (int c = 0; c < 3; ++c) M[r * 6 + 3 + c] = Ra[r * 3 + c];
}

// ------------------------------------------------------------ vertices

// The 12-double rotation record of a vertex: R_I_M (JPL, 9), |q|^2, 0, 0.
__device__ inline void vertex_rotation(const double* q, double* __restrict__ out) {
  double R[9];
  rot_jpl(q, R);
  for (int i = 0; i < 9; ++i) out[i] = R[i];
  out[9] = q[0] * q[0] + q[1] * q[1] + q[2] * q[2] + q[3] * q[3];
  out[10] = 0.0;
  out[11] = 0.0;
}

__global__ void k_vertex_prep(int32_t P, const double* __restrict__ vert, double* __restrict__ vR) {
  const int v = blockIdx.x * blockDim.x + threadIdx.x;
  if (v >= P) return;
  vertex_rotation(vert + 7 * v, vR + 12 * v);
}

// ------------------------------------------------------------ linearization

struct ObsEval {
  double r[2];
  double K[6];   // d r / d p_I, row-major 2x3
  double G[9];   // d p_I / d p_B
  double pI[3];  // the landmark in the observer's IMU frame
  bool failed;
};

// G = d p_I / d p_B of a pose-coupled observation by vertex v of a landmark
// anchored in vertex a: R_I_M R_M_B, over the mission frames for kGlobal.
__device__ inline void landmark_to_imu(const DevTopology& t, int32_t type, int32_t a, int32_t v, const double* Ra,
                                       const double* Rv, double* G) {
  double H[9];  // d p_M / d p_B
  for (int i = 0; i < 3; ++i)
    for (int j = 0; j < 3; ++j) H[i * 3 + j] = Ra[j * 3 + i];
  if (type == kTypeGlobal) {
    const double* TL = t.mission_T + 12 * t.vertex_mission[a];
    const double* TM = t.mission_T + 12 * t.vertex_mission[v];
    double T1[9];
    mat3_mul(TL, H, T1);  // R_G_LM R_LM_B
    for (int i = 0; i < 3; ++i)
      for (int j = 0; j < 3; ++j) H[i * 3 + j] = TM[i] * T1[j] + TM[3 + i] * T1[3 + j] + TM[6 + i] * T1[6 + j];
  }
  mat3_mul(Rv, H, G);
}

// Residual of one observation, of landmark l (anchored in vertex a) by vertex
// v, and the factors of its Jacobians (visual-error-term-inl.h:13-379).
template <bool kJac>
__device__ inline void eval_observation(const DevTopology& t, int o, int32_t meta, int32_t l, int32_t v, int32_t a,
                                        const double* __restrict__ vert, const double* __restrict__ vR,
                                        const double* __restrict__ lm, ObsEval& e) {
  const int32_t type = obs_type(meta);
  const DevCamera& cam = t.cams[obs_camera(meta)];
  const double* pB = lm + 3 * l;
  double* pI = e.pI;
  if (type == kTypeKeyframe) {
    pI[0] = pB[0]; pI[1] = pB[1]; pI[2] = pB[2];
    if (kJac)
      for (int i = 0; i < 9; ++i) e.G[i] = (i % 4 == 0) ? 1.0 : 0.0;
  } else {
    const double* Rv = vR + 12 * v;
    const double* Ra = vR + 12 * a;        // R_B_LM
    const double* pa = vert + 7 * a + 4;   // p_LM_B
    double pM[3];
    mat3t_vec(Ra, pB, pM);
    pM[0] += pa[0]; pM[1] += pa[1]; pM[2] += pa[2];
    if (type == kTypeGlobal) {
      const double* TL = t.mission_T + 12 * t.vertex_mission[a];
      const double* TM = t.mission_T + 12 * t.vertex_mission[v];
      double pG[3], d[3];
      mat3_vec(TL, pM, pG);
      for (int i = 0; i < 3; ++i) d[i] = pG[i] + TL[9 + i] - TM[9 + i];
      mat3t_vec(TM, d, pM);
    }
    const double* pv = vert + 7 * v + 4;
    const double dm[3] = {pM[0] - pv[0], pM[1] - pv[1], pM[2] - pv[2]};
    mat3_vec(Rv, dm, pI);
    if (kJac) landmark_to_imu(t, type, a, v, Ra, Rv, e.G);
  }
  double pC[3];
  mat3_vec(cam.R_C_I, pI, pC);
  pC[0] += cam.p_C_I[0]; pC[1] += cam.p_C_I[1]; pC[2] += cam.p_C_I[2];
  double kp[2], jp[6];
  const int32_t status = project_camera(cam.model, cam.xi, cam.dist_type, cam.intr, cam.dist, cam.width, cam.height, pC, kp, jp);
  e.failed = projection_failed(status, pC, kp);
  const double sinv = t.obs_sinv[o];
  const double* meas = t.obs_kp + 2 * o;
  if (e.failed) {
    e.r[0] = e.r[1] = 0.0;
  } else {
    e.r[0] = (kp[0] - meas[0]) * sinv;
    e.r[1] = (kp[1] - meas[1]) * sinv;
  }
  if (!kJac) return;
  if (e.failed) {
    for (int i = 0; i < 6; ++i) e.K[i] = 0.0;
    for (int i = 0; i < 3; ++i) pI[i] = 0.0;
    return;
  }
  // K = (d kp / d p_C) * sigma^-1 * R_C_I.
  for (int r = 0; r < 2; ++r)
    for (int c = 0; c < 3; ++c)
      e.K[r * 3 + c] = sinv * (jp[r * 3] * cam.R_C_I[c] + jp[r * 3 + 1] * cam.R_C_I[3 + c] +
                               jp[r * 3 + 2] * cam.R_C_I[6 + c]);
}

// The observer's tangent Jacobian (2x6, [rot 3 | pos 3]) from an observation
// record: rotation |q|^2 (K_r x p_I), position -K_r R_I_M. Rv is the vertex's
// 12-double rotation record.
template <class Rec>
__device__ inline void observer_jacobian(const Rec& rec, const double* Rv, double* Jo) {
  const double n2 = Rv[9];
  for (int r = 0; r < 2; ++r) {
    const double k0 = rec.K(3 * r), k1 = rec.K(3 * r + 1), k2 = rec.K(3 * r + 2);
    Jo[r * 6 + 0] = n2 * (k1 * rec.p(2) - k2 * rec.p(1));
    Jo[r * 6 + 1] = n2 * (k2 * rec.p(0) - k0 * rec.p(2));
    Jo[r * 6 + 2] = n2 * (k0 * rec.p(1) - k1 * rec.p(0));
    for (int c = 0; c < 3; ++c) Jo[r * 6 + 3 + c] = -(k0 * Rv[c] + k1 * Rv[3 + c] + k2 * Rv[6 + c]);
  }
}

// Loss scale of one observation: HuberLoss(delta * sigma) with delta 3 / 10
// (optimization-terms-addition.cc:189-198), Cauchy(scale_px / sigma).
__device__ inline double loss_scale(const DevLoss& loss, int32_t type, double sinv) {
  if (loss.type == 0) return (type == kTypeGlobal ? 10.0 : 3.0) / sinv;
  if (loss.type == 1) return loss.scale_px * sinv;
  return 1.0;
}

// Per observation: robust-corrected residual and Jacobian K into obs_rec;
// per landmark: sum Jl'Jl over the store vertex's own observations (V_own) and
// over the pose-coupled ones (V_mission), g = sum Jl'r, g_mission; per tile: cost and fixed cost.
//
// With kF32 K is rounded (Rec32) right after the correction and every later
// product (V, g here; J'J, W, the model cost in the readers) uses the rounded
// values, so S stays the Schur complement of J'J of one Jacobian; records are
// Rec32 (residual and p_I in FP64).
//
// Records leave through LDS, so that consecutive lanes write consecutive 16
// bytes: written by its own thread, a record is six stores of which each touches
// 64 rows of 96 bytes: 188 -> 164 us for 2.9M observations of 500 keyframes, 358
// -> 311 for 5.1M of 1000 (and k_schur_factors, which writes so too, 185 -> 134,
// 327 -> 229).
//
// The landmark sums meet in LDS: nine values per observation (V and g), value-
// major; thread (run, value) adds its landmark's run of observations in order,
// the pose-coupled ones and the store vertex's own separately, so all 256
// threads share the sums (a run's first thread alone adding 18 values left
// nine tenths of the tile idle).
constexpr int kLinVals = 9;  // V (6), g (3)

template <bool kJac, bool kF32 = false>
__global__ __launch_bounds__(kObsTile) void k_linearize(DevTopology t, const double* __restrict__ vert,
                                                         const double* __restrict__ vR,
                                                         const double* __restrict__ lm, DevLoss loss,
                                                         const int32_t* __restrict__ tile_begin,
                                                         void* __restrict__ obs_rec,
                                                         double* __restrict__ lm_acc,
                                                         double* __restrict__ split_part,
                                                         double* __restrict__ tile_cost) {
  constexpr int kRecWords = (kF32 ? (int)sizeof(Rec32) : kObsRecord * 8) / 16;  // 16-byte words of a record
  __shared__ union {
    double red[kJac ? kLinVals : 1][kJac ? kObsTile + 1 : 1];
    double2 rec[kJac ? kObsTile * kRecWords : 1];
  } sh;
  __shared__ int32_t seg[kJac ? kObsTile : 1];    // landmark of each observation
  __shared__ uint8_t own[kJac ? kObsTile : 1];    // made by the store vertex (not pose-coupled)
  __shared__ int16_t head[kJac ? kObsTile + 1 : 1];  // first observation of each run
  __shared__ int32_t wave_runs[4];
  __shared__ double lds4[4];
  const int tid = threadIdx.x;
  const int b = tile_begin[blockIdx.x], e = tile_begin[blockIdx.x + 1];
  const int o = b + tid;
  double acc[kLinVals];
  for (int i = 0; i < kLinVals; ++i) acc[i] = 0.0;
  double cost = 0.0, fixed = 0.0;
  int32_t l = -1;
  bool pose_coupled = true;
  if (o < e) {
    l = t.obs_landmark[o];
    // What the evaluation's loads start from comes with the flags, so that an
    // active landmark's evaluation waits one round for them and an inactive
    // one's is skipped. 500 keyframes, all active / 60 % inactive / three
    // quarters of the tiles inactive: 138 / 125 / 65 us, cost only 46 / 38 / 18;
    // evaluated whatever the flags say 138 / 138 / 131 and 47 / 46 / 45; loaded
    // after the flags 143 / 125 / 67 and 46 / 38 / 19.
    const int32_t meta = t.obs_meta[o], v = t.obs_vertex[o];
    const uint32_t flags = t.lm_flags[l];
    const int32_t a = t.lm_anchor[l];
    double rec[kObsRecord] = {};
    if (flags & kLmActive) {
      ObsEval ev;
      eval_observation<kJac>(t, o, meta, l, v, a, vert, vR, lm, ev);
      const int32_t type = obs_type(meta);
      const double s = ev.r[0] * ev.r[0] + ev.r[1] * ev.r[1];
      double rho[3];
      robust_loss(loss.type, loss_scale(loss, type, t.obs_sinv[o]), s, rho);
      pose_coupled = type != kTypeKeyframe;
      const bool has_var = !(flags & kLmConstant) ||
                           (pose_coupled && (obs_observer_var(meta) || t.vertex_var[a] >= 0));
      if (has_var) cost = 0.5 * rho[0]; else fixed = 0.5 * rho[0];
      if (kJac) {
        // ceres Corrector: J~ = sqrt(rho') (I - alpha r r'/|r|^2) J, r~ = rs r.
        const double sq1 = sqrt(rho[1]);
        double rs = sq1, asq = 0.0;
        if (s > 0.0 && rho[2] > 0.0) {
          const double alpha = 1.0 - sqrt(1.0 + 2.0 * s * rho[2] / rho[1]);
          rs = sq1 / (1.0 - alpha);
          asq = alpha / s;
        }
        rec[0] = ev.r[0] * rs;
        rec[1] = ev.r[1] * rs;
        for (int c = 0; c < 3; ++c) {
          const double rtj = ev.K[c] * ev.r[0] + ev.K[3 + c] * ev.r[1];
          rec[2 + c] = sq1 * (ev.K[c] - asq * ev.r[0] * rtj);
          rec[5 + c] = sq1 * (ev.K[3 + c] - asq * ev.r[1] * rtj);
        }
        if (kF32)
          for (int i = 0; i < 6; ++i) {
            const float hi = (float)rec[2 + i];
            rec[2 + i] = (double)hi + (double)bf16_value(bf16_round((float)(rec[2 + i] - (double)hi)));
          }
        for (int i = 0; i < 3; ++i) rec[8 + i] = ev.pI[i];
        double J[6];
        for (int r = 0; r < 2; ++r)
          for (int c = 0; c < 3; ++c)
            J[r * 3 + c] = rec[2 + 3 * r] * ev.G[c] + rec[3 + 3 * r] * ev.G[3 + c] + rec[4 + 3 * r] * ev.G[6 + c];
        acc[0] = J[0] * J[0] + J[3] * J[3];
        acc[1] = J[0] * J[1] + J[3] * J[4];
        acc[2] = J[0] * J[2] + J[3] * J[5];
        acc[3] = J[1] * J[1] + J[4] * J[4];
        acc[4] = J[1] * J[2] + J[4] * J[5];
        acc[5] = J[2] * J[2] + J[5] * J[5];
        for (int c = 0; c < 3; ++c) acc[6 + c] = J[c] * rec[0] + J[3 + c] * rec[1];
      }
    }
    if (kJac) {
      if (kF32) {
        Rec32* out = reinterpret_cast<Rec32*>(sh.rec) + tid;
        for (int i = 0; i < 2; ++i) out->r[i] = rec[i];
        for (int i = 0; i < 3; ++i) out->p[i] = rec[8 + i];
        out->unused = 0;
        for (int i = 0; i < 6; ++i) {
          const float hi = (float)rec[2 + i];  // the sum rounds back to its parts
          out->K[i] = hi;
          out->lo[i] = bf16_round((float)(rec[2 + i] - (double)hi));
        }
      } else {
        for (int i = 0; i < kRecWords; ++i) sh.rec[kRecWords * tid + i] = make_double2(rec[2 * i], rec[2 * i + 1]);
      }
    }
  }
  if (kJac) {
    // Records are 96 or 80 bytes and the array is 256-byte aligned.
    __syncthreads();
    double2* out = static_cast<double2*>(obs_rec) + (size_t)kRecWords * b;
    for (int i = tid; i < kRecWords * (e - b); i += kObsTile) out[i] = sh.rec[i];
    __syncthreads();
  }
  if (kJac) {
    for (int i = 0; i < kLinVals; ++i) sh.red[i][tid] = acc[i];
    seg[tid] = l;
    own[tid] = pose_coupled ? 0 : 1;
    __syncthreads();
    // Runs of one landmark, in order: first observations into head.
    const bool first = o < e && (tid == 0 || seg[tid - 1] != l);
    const uint64_t mask = __ballot(first);
    const int lane = tid & 63, wave = tid >> 6;
    if (lane == 0) wave_runs[wave] = __popcll(mask);
    __syncthreads();
    int before = __popcll(mask & ((1ull << lane) - 1ull)), runs = 0;
    for (int w = 0; w < 4; ++w) {
      if (w < wave) before += wave_runs[w];
      runs += wave_runs[w];
    }
    if (first) head[before] = (int16_t)tid;
    if (tid == 0) head[runs] = (int16_t)(e - b);
    __syncthreads();
    for (int it = tid; it < runs * kLinVals; it += kObsTile) {
      const int run = it / kLinVals, c = it - run * kLinVals;
      const int k0 = head[run], k1 = head[run + 1];
      double sum = 0.0, sum_own = 0.0;
      for (int k = k0; k < k1; ++k) {
        const double v = sh.red[c][k];
        if (own[k]) sum_own += v; else sum += v;
      }
      const int32_t lr = seg[k0];
      // A split landmark owns its tiles whole: the tile's sum goes to the
      // tile's slot, and k_split_sum adds the slots in tile order.
      double* dst = (t.lm_flags[lr] & kLmSplit) ? split_part + (size_t)kLmAcc * blockIdx.x
                                                : lm_acc + (size_t)kLmAcc * lr;
      // V_own, V_mission (6 each), then g, g_mission (3 each).
      const int at = c < 6 ? c : 6 + c, step = c < 6 ? 6 : 3;
      dst[at] = c < 6 ? sum_own : sum + sum_own;
      dst[at + step] = sum;
    }
  }
  const double c_sum = block_sum256(cost, lds4);
  const double f_sum = block_sum256(fixed, lds4);
  if (tid == 0) {
    tile_cost[2 * blockIdx.x] = c_sum;
    tile_cost[2 * blockIdx.x + 1] = f_sum;
  }
}

// Accumulators of the landmarks split over several tiles: the tile sums of
// each, added in tile order. split_tiles[2k], [2k+1] = first tile, tile count.
__global__ void k_split_sum(int32_t n, const int32_t* __restrict__ ids, const int32_t* __restrict__ split_tiles,
                            const double* __restrict__ split_part, double* __restrict__ lm_acc) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n * kLmAcc) return;
  const int k = i / kLmAcc, c = i % kLmAcc;
  const int t0 = split_tiles[2 * k], nt = split_tiles[2 * k + 1];
  double s = 0.0;
  for (int j = 0; j < nt; ++j) s += split_part[(size_t)kLmAcc * (t0 + j) + c];
  lm_acc[(size_t)kLmAcc * ids[k] + c] = s;
}

// ------------------------------------------------------------ vertex rows

// Per variable vertex: unscaled gradient g = J'r and diag(J'J) of its six
// tangent columns, over its incidences (observations it makes and the
// landmarks anchored in it).
template <bool kF32>
__global__ __launch_bounds__(kRowThreads) void k_pose_rows(DevTopology t, const double* __restrict__ vert,
                                                            const double* __restrict__ vR,
                                                            const double* __restrict__ lm,
                                                            const void* __restrict__ obs_rec,
                                                            const double* __restrict__ lm_acc,
                                                            double* __restrict__ pose_grad,
                                                            double* __restrict__ pose_diag,
                                                            double* __restrict__ pose_jtj) {
  constexpr int kVals = 12 + 21;  // gradient, diagonal, upper triangle of sum Jo^T Jo
  __shared__ double red[kRowThreads / 64][kVals];
  const int i = blockIdx.x;
  const int ib = t.inc_ptr[i], ie = t.inc_ptr[i + 1];
  double g[6] = {0, 0, 0, 0, 0, 0}, d[6] = {0, 0, 0, 0, 0, 0}, jj[21];
  for (int k = 0; k < 21; ++k) jj[k] = 0.0;
  const double* Rv = vR + 12 * t.var_vertex[i];
  for (int k = ib + threadIdx.x; k < ie; k += kRowThreads) {
    const int32_t x = t.inc[k];
    if (x >= 0) {
      const RecView<kF32> rec(obs_rec, x);
      double Jo[12];
      observer_jacobian(rec, Rv, Jo);
      for (int c = 0; c < 6; ++c) {
        g[c] += Jo[c] * rec.r(0) + Jo[6 + c] * rec.r(1);
        d[c] += Jo[c] * Jo[c] + Jo[6 + c] * Jo[6 + c];
      }
      int u = 0;
      for (int r = 0; r < 6; ++r)
        for (int c = r; c < 6; ++c, ++u) jj[u] += Jo[r] * Jo[c] + Jo[6 + r] * Jo[6 + c];
    } else {
      const int32_t l = -1 - x;
      const int32_t a = t.lm_anchor[l];
      double M[18], VLM[9];
      anchor_map(lm + 3 * l, vR + 12 * a, vR[12 * a + 9], M);
      const double* acc = lm_acc + (size_t)kLmAcc * l;
      sym3_full(acc + 6, VLM);
      const double* gLM = acc + 15;
      for (int c = 0; c < 6; ++c) {
        const double m0 = M[c], m1 = M[6 + c], m2 = M[12 + c];
        g[c] += m0 * gLM[0] + m1 * gLM[1] + m2 * gLM[2];
        d[c] += m0 * (VLM[0] * m0 + VLM[1] * m1 + VLM[2] * m2) + m1 * (VLM[3] * m0 + VLM[4] * m1 + VLM[5] * m2) +
                m2 * (VLM[6] * m0 + VLM[7] * m1 + VLM[8] * m2);
      }
    }
  }
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  for (int c = 0; c < 6; ++c) {
    g[c] = wave_sum(g[c]);
    d[c] = wave_sum(d[c]);
  }
  for (int k = 0; k < 21; ++k) jj[k] = wave_sum(jj[k]);
  if (lane == 0) {
    for (int c = 0; c < 6; ++c) { red[wave][c] = g[c]; red[wave][6 + c] = d[c]; }
    for (int k = 0; k < 21; ++k) red[wave][12 + k] = jj[k];
  }
  __syncthreads();
  if (threadIdx.x < 12) {
    double s = 0.0;
    for (int w = 0; w < kRowThreads / 64; ++w) s += red[w][threadIdx.x];
    if (threadIdx.x < 6) pose_grad[6 * i + threadIdx.x] = s;
    else pose_diag[6 * i + threadIdx.x - 6] = s;
  } else if (threadIdx.x >= 64 && threadIdx.x < 100) {
    const int e = threadIdx.x - 64, r = min(e / 6, e % 6), c = max(e / 6, e % 6);
    const int u = r * 6 - r * (r - 1) / 2 + (c - r);  // index of (r, c), r <= c, in the upper triangle
    double s = 0.0;
    for (int w = 0; w < kRowThreads / 64; ++w) s += red[w][12 + u];
    pose_jtj[36 * i + e] = s;
  }
}

// ceres Jacobi scaling: c = 1 / (1 + sqrt(diag(J'J))) of every tangent column.
__global__ void k_jacobi_scaling(int32_t Pvar, int32_t L, int32_t use, const double* __restrict__ pose_diag,
                                 const double* __restrict__ lm_acc, double* __restrict__ pose_scale,
                                 double* __restrict__ lm_scale) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < 6 * Pvar) pose_scale[i] = use ? 1.0 / (1.0 + sqrt(pose_diag[i])) : 1.0;
  if (i < 3 * L) {
    const int l = i / 3, c = i % 3;
    const int di = c == 0 ? 0 : (c == 1 ? 3 : 5);
    const double* V = lm_acc + (size_t)kLmAcc * l;
    lm_scale[i] = use ? 1.0 / (1.0 + sqrt(V[di] + V[6 + di])) : 1.0;
  }
}

// ------------------------------------------------------------ landmark pivot

// T_l with Z_l = T'T = C (C V C + D^2)^-1 C, D^2 = clamp(diag(C V C)) / mu
// (ceres LevenbergMarquardtStrategy diagonal), and T_l g_l, so that the Schur
// factors read both from one record of their (scattered) landmark. Zero for
// inactive and constant landmarks.
//
// For a landmark whose anchor vertex is variable also the anchor's factor
// (see the Schur complement below): U_a = T R with R = Z^-1 - V_mission =
// V_own + D^2 / C^2 (formed so, not as a difference), the negated self product
// -V_mission Z R and the rhs part -(g_mission - V_mission Z g). A constant
// landmark has Z = 0, but its observations couple its anchor all the same:
// T = e I with U_a = I / e gives those products exactly, and e = 1e-20 makes
// the observations' own products vanish.
__global__ void k_landmark_prep(DevTopology t, const double* __restrict__ lm_acc,
                                const double* __restrict__ lm_scale, double inv_mu, double min_diag,
                                double max_diag, double* __restrict__ lm_z, double* __restrict__ lm_anc,
                                int32_t* __restrict__ fail) {
  const int l = blockIdx.x * blockDim.x + threadIdx.x;
  if (l >= t.L) return;
  double* z = lm_z + (size_t)kLmZ * l;
  double* an = lm_anc + (size_t)kLmAnchor * l;
  const uint32_t flags = t.lm_flags[l];
  const double* acc = lm_acc + (size_t)kLmAcc * l;
  const bool anchored = (flags & kLmAnchorVar) != 0;
  double T[6] = {0, 0, 0, 0, 0, 0}, damp[3] = {0, 0, 0};
  bool zero = !(flags & kLmActive);
  if (!zero && !(flags & kLmConstant)) {
    const double* c = lm_scale + 3 * l;
    double A[6];
    for (int i = 0; i < 6; ++i) A[i] = acc[i] + acc[6 + i];
    A[0] *= c[0] * c[0]; A[1] *= c[0] * c[1]; A[2] *= c[0] * c[2];
    A[3] *= c[1] * c[1]; A[4] *= c[1] * c[2]; A[5] *= c[2] * c[2];
    const double d[3] = {fmin(fmax(A[0], min_diag), max_diag) * inv_mu, fmin(fmax(A[3], min_diag), max_diag) * inv_mu,
                         fmin(fmax(A[5], min_diag), max_diag) * inv_mu};
    A[0] += d[0];
    A[3] += d[1];
    A[5] += d[2];
    if (spd3_inverse_factor(A, T)) {
      T[0] *= c[0]; T[1] *= c[0]; T[2] *= c[1];
      T[3] *= c[0]; T[4] *= c[1]; T[5] *= c[2];
      for (int k = 0; k < 3; ++k) damp[k] = d[k] / (c[k] * c[k]);
    } else {
      atomicAdd(fail, 1);
      for (int k = 0; k < 6; ++k) T[k] = 0.0;
      zero = true;
    }
  }
  const double* g = acc + 12;
  double y[3] = {0, 0, 0};
  if (!zero) tri_vec(T, g, y);
  const bool pinned = !zero && (flags & kLmConstant) && anchored;
  constexpr double kPin = 1e-20;
  if (pinned) T[0] = T[2] = T[5] = kPin;
  for (int i = 0; i < 6; ++i) z[i] = T[i];
  for (int i = 0; i < 3; ++i) z[6 + i] = y[i];
  if (!anchored) return;
  double U[9] = {}, X[6] = {}, h[3] = {};
  if (!zero) {
    const double* V = acc + 6;
    const double* gm = acc + 15;
    if (pinned) {
      U[0] = U[4] = U[8] = 1.0 / kPin;
      for (int i = 0; i < 6; ++i) X[i] = -V[i];
      for (int i = 0; i < 3; ++i) h[i] = -gm[i];
    } else {
      double R[9], VM[9], B[9];
      sym3_full(acc, R);
      for (int k = 0; k < 3; ++k) R[4 * k] += damp[k];
      sym3_full(V, VM);
      for (int c = 0; c < 3; ++c) {  // U = T R, B = T V_mission, column by column
        const double r[3] = {R[c], R[3 + c], R[6 + c]}, m[3] = {VM[c], VM[3 + c], VM[6 + c]};
        double o[3];
        tri_vec(T, r, o);
        for (int k = 0; k < 3; ++k) U[3 * k + c] = o[k];
        tri_vec(T, m, o);
        for (int k = 0; k < 3; ++k) B[3 * k + c] = o[k];
      }
      double W[9];  // V_mission Z R = B'U
      for (int r = 0; r < 3; ++r)
        for (int c = 0; c < 3; ++c) W[3 * r + c] = B[r] * U[c] + B[3 + r] * U[3 + c] + B[6 + r] * U[6 + c];
      X[0] = -W[0];
      X[1] = -0.5 * (W[1] + W[3]);
      X[2] = -0.5 * (W[2] + W[6]);
      X[3] = -W[4];
      X[4] = -0.5 * (W[5] + W[7]);
      X[5] = -W[8];
      for (int c = 0; c < 3; ++c) h[c] = B[c] * y[0] + B[3 + c] * y[1] + B[6 + c] * y[2] - gm[c];
    }
  }
  for (int i = 0; i < 9; ++i) an[i] = U[i];
  for (int i = 0; i < 6; ++i) an[9 + i] = X[i];
  for (int i = 0; i < 3; ++i) an[15 + i] = h[i];
}

// ------------------------------------------------------------ Schur complement

// The reduced camera system
//   S = F'F + D^2 - sum_l W_l' Z_l W_l,  rhs = F'r - sum_l W_l' Z_l g_l
// (ceres' Schur eliminator, schur_eliminator_impl.h, restated on the
// anchor-lifted blocks) from factors of the landmark-pose blocks. With
// E(p) = [[p]x | -I] (3x6) and the row transform D_i = diag(|q_i|^2 I, R_i) C_i
// of the vertex of row i (R_I_M, column scaling C_i), the Jacobians factor as
//   J_observer C = K E(p_I) D_i                 (p_I: landmark in the IMU frame)
//   J_anchor C   = -J_landmark E(p_B) D_a       (J_landmark times the anchor map)
// and with P = J_landmark' K, summed over the observations of landmark l by
// the vertex (they share p_I), and k = K'r, l's products with Z = T'T are
//   S_ij -= D_i' E_i' (U_i' U_j) E_j D_j,       U = T P      (3x3)
//   rhs_i += D_i' E_i' (k - U_i' T g)
// The anchor a of l joins them with U_a = T R, R = Z^-1 - V_mission: an
// observation x with the anchor gives W_x'(Z V_mission - I) A = -W_x' Z R A,
// and the anchor with itself V_mission - V_mission Z V_mission =
// V_mission Z R, which k_landmark_prep forms (as its rhs part). So a staged
// factor is U and p (12 doubles) for both sides of every product, where the
// plain blocks W and W'Z are 36, and a product is 27 + 72 multiply-adds with
// 24 doubles read from LDS instead of 108 with 36. The row transforms are
// applied once per block of S, by k_schur_finalize.
// Factor blocks (P, p) and k are stored landmark-major (rows ascending), per
// linearization. An anchor's block keeps p_B.
template <bool kF32>
__global__ __launch_bounds__(256) void k_schur_factors(
    DevTopology t, int32_t n_g, const int32_t* __restrict__ g_row, const int32_t* __restrict__ g_inc_ptr,
    const int32_t* __restrict__ g_inc, const double* __restrict__ vR, const double* __restrict__ lm,
    const void* __restrict__ obs_rec, double* __restrict__ gf, double* __restrict__ gk) {
  // Blocks leave through LDS, as k_linearize's records do.
  __shared__ double2 sf[256 * kFactor / 2];
  __shared__ double sk[256 * 3];
  const int tid = threadIdx.x, g0 = blockIdx.x * 256, n = min(256, n_g - g0);
  const int g = min(g0 + tid, n_g - 1);  // the last work-group's spare threads repeat the last block
  const int m0 = g_inc_ptr[g], m1 = g_inc_ptr[g + 1];
  double f[kFactor] = {}, k[3] = {0, 0, 0};
  const int32_t x0 = g_inc[m0];
  if (x0 < 0) {
    const int32_t l = -1 - x0;
    if (t.lm_flags[l] & kLmActive)
      for (int c = 0; c < 3; ++c) f[9 + c] = lm[3 * l + c];
  } else {
    const int v = t.var_vertex[g_row[g]], la = t.lm_anchor[t.obs_landmark[x0]];
    double G[9];
    landmark_to_imu(t, obs_type(t.obs_meta[x0]), la, v, vR + 12 * la, vR + 12 * v, G);
    for (int m = m0; m < m1; ++m) {
      const RecView<kF32> rec(obs_rec, g_inc[m]);
      for (int r = 0; r < 2; ++r) {
        const double k0 = rec.K(3 * r), k1 = rec.K(3 * r + 1), k2 = rec.K(3 * r + 2), rr = rec.r(r);
        for (int a = 0; a < 3; ++a) {
          const double jl = k0 * G[a] + k1 * G[3 + a] + k2 * G[6 + a];
          f[3 * a] += jl * k0;
          f[3 * a + 1] += jl * k1;
          f[3 * a + 2] += jl * k2;
        }
        k[0] += k0 * rr;
        k[1] += k1 * rr;
        k[2] += k2 * rr;
      }
      // A failed projection's record is zero, p_I included.
      if (rec.p(0) != 0.0 || rec.p(1) != 0.0 || rec.p(2) != 0.0)
        for (int c = 0; c < 3; ++c) f[9 + c] = rec.p(c);
    }
  }
  for (int c = 0; c < kFactor / 2; ++c) sf[kFactor / 2 * tid + c] = make_double2(f[2 * c], f[2 * c + 1]);
  for (int c = 0; c < 3; ++c) sk[3 * tid + c] = k[c];
  __syncthreads();
  double2* out = reinterpret_cast<double2*>(gf + (size_t)kFactor * g0);
  for (int i = tid; i < kFactor / 2 * n; i += 256) out[i] = sf[i];
  for (int i = tid; i < 3 * n; i += 256) gk[(size_t)3 * g0 + i] = sk[i];
}

// LDS of one round of a tile: the staged factors of one or two batches (U and
// p), on diagonal tiles their rhs vectors and the anchors' self products, the
// batches' pair lists and the segment's batch words. Entries are slot-minor,
// the factor's in pairs of 16 bytes (row r of U and p_r are [2 r][s] and
// [2 r + 1][s]), so that the staging writes of consecutive threads hit
// consecutive banks and a product's 24 doubles are 12 reads.
struct TileLds {
  union {
    double2 f[kFactor / 2][2 * kBatchSlots];
    struct {
      double2 f[kFactor / 2][kBatchSlots];
      double h[3][kBatchSlots];
      double x[6][kBatchSlots];
      uint8_t anchor[kBatchSlots];
    } diag;
  };
  uint32_t pairs[2][kBatchPairs / 2];
  int4 bt[kSegmentBatches];
};

struct TileArgs {
  const int4* batches;
  const int2* slots;
  const uint16_t* batch_off;
  const uint32_t* pairs;  // the pair list as 32-bit words (batches start on a word)
  const double* gf;
  const double* gk;
  const double* lm_z;
  const double* lm_anc;
};

// A thread's part of a segment.
struct TilePart {
  int32_t tid, np, blk, part;
};

// A thread's index loads of one batch (two rounds ahead): its slot's word and
// its part's pair range.
struct TileIdx {
  int2 slot;
  int32_t pb, pe;
};

// A thread's data loads of one batch (one round ahead): its slot's factor (P,
// or U for an anchor, and p), its landmark's T, its share of the pair list; on
// diagonal tiles T g, k (or the anchor's rhs) and the anchor's self product.
template <bool kDiag>
struct TileStage {
  double f[kFactor], z[kDiag ? 9 : 6], h[kDiag ? 3 : 1], x[kDiag ? 6 : 1];
  uint32_t pw[kPairWords];
  TileIdx q;
};

__device__ inline void tile_idx(TileIdx& q, const TileArgs& ta, const int4& bt, int b, const TilePart& me) {
  q.slot = make_int2(-1, 0);
  if (me.tid < bt.y) q.slot = ta.slots[bt.x + me.tid];
  q.pb = q.pe = 0;
  if (me.np) {
    const uint16_t* off = ta.batch_off + (size_t)b * (kTileBlocks + 1);
    q.pb = off[me.blk] + me.part;
    q.pe = off[me.blk + 1];
  }
}

template <bool kDiag>
__device__ inline void tile_data(TileStage<kDiag>& st, const TileIdx& q, const TileArgs& ta, const int4& bt, int tid) {
  st.q = q;
  const int nw = (bt.w + 1) >> 1;
  const uint32_t* pw = ta.pairs + (bt.z >> 1);
#pragma unroll
  for (int k = 0; k < kPairWords; ++k) {
    const int j = tid + k * kTileBlocks;
    st.pw[k] = j < nw ? pw[j] : 0u;
  }
  if (q.slot.x < 0) return;
  const uint32_t lw = (uint32_t)q.slot.y;
  const size_t l = lw & ~kSlotAnchor;
  const bool anc = (lw & kSlotAnchor) != 0;
  const double* fp = ta.gf + (size_t)kFactor * q.slot.x;
  const double* an = ta.lm_anc + kLmAnchor * l;
  const double* up = anc ? an : fp;
#pragma unroll
  for (int e = 0; e < 9; ++e) st.f[e] = up[e];
#pragma unroll
  for (int e = 9; e < kFactor; ++e) st.f[e] = fp[e];
  const double* zp = ta.lm_z + kLmZ * l;
#pragma unroll
  for (int e = 0; e < (kDiag ? 9 : 6); ++e) st.z[e] = zp[e];
  if (kDiag) {
    const double* hp = anc ? an + 15 : ta.gk + (size_t)3 * q.slot.x;
#pragma unroll
    for (int e = 0; e < 3; ++e) st.h[e] = hp[e];
    if (anc)
#pragma unroll
      for (int e = 0; e < 6; ++e) st.x[e] = an[9 + e];
  }
}

// A batch's staged data into LDS: U = T P (an anchor's is ready), p, and on
// diagonal tiles h = k - U'T g.
template <bool kDiag>
__device__ inline void tile_stage(TileLds& sh, const TileStage<kDiag>& st, int tid, int half) {
#pragma unroll
  for (int j = 0; j < kPairWords; ++j) sh.pairs[half][tid + j * kTileBlocks] = st.pw[j];
  if (st.q.slot.x < 0) return;
  const double* z = st.z;
  const bool anc = ((uint32_t)st.q.slot.y & kSlotAnchor) != 0;
  double u[9];
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    const double p0 = st.f[c], p1 = st.f[3 + c], p2 = st.f[6 + c];
    u[c] = anc ? p0 : z[0] * p0;
    u[3 + c] = anc ? p1 : z[1] * p0 + z[2] * p1;
    u[6 + c] = anc ? p2 : z[3] * p0 + z[4] * p1 + z[5] * p2;
  }
#pragma unroll
  for (int r = 0; r < 3; ++r) {
    const double2 lo = make_double2(u[3 * r], u[3 * r + 1]), hi = make_double2(u[3 * r + 2], st.f[9 + r]);
    if (kDiag) {
      sh.diag.f[2 * r][tid] = lo;
      sh.diag.f[2 * r + 1][tid] = hi;
    } else {
      sh.f[2 * r][half * kBatchSlots + tid] = lo;
      sh.f[2 * r + 1][half * kBatchSlots + tid] = hi;
    }
  }
  if (kDiag) {
#pragma unroll
    for (int c = 0; c < 3; ++c)
      sh.diag.h[c][tid] = anc ? st.h[c] : st.h[c] - (u[c] * z[6] + u[3 + c] * z[7] + u[6 + c] * z[8]);
#pragma unroll
    for (int c = 0; c < 6; ++c) sh.diag.x[c][tid] = st.x[c];
    sh.diag.anchor[tid] = anc ? 1 : 0;
  }
}

// One segment of a tile. Per round (one batch on a diagonal tile, two on the
// others): every thread stages its slot's factor of each batch in LDS and its
// share of the pair lists, then each thread adds the products of its part of
// its block's pairs in list order, one batch's after the other's in one loop: a
// wave's loop lasts as long as its busiest part, and over two batches the
// parts' shares are more even (a part has 1.9 pairs a batch, the busiest 6.6).
// A part of a diagonal block of a diagonal tile also adds the rhs of its
// pairs' factors. Loads are software-pipelined: while a round's products run,
// the next round's data loads and the index loads of the one after that are in
// flight. Each part's sums go to its own slot of the segment's partial.
template <bool kDiag>
__device__ inline void tile_segment(TileLds& sh, const TileArgs& ta, const int4& sg, uint32_t tw,
                                    double* __restrict__ out_base) {
  constexpr int kHalves = kDiag ? 1 : 2;
  constexpr int kSlots = kHalves * kBatchSlots;
  TilePart me;
  me.tid = threadIdx.x;
  me.np = seg_thread_parts(tw);
  me.blk = seg_thread_block(tw);
  me.part = seg_thread_part(tw);
  const int tid = me.tid, np = me.np, nb = sg.y - sg.x;
  const bool rhs_part = kDiag && np && me.blk / kTileBand == me.blk % kTileBand;
  const double2(*fl)[kSlots] =
      kDiag ? reinterpret_cast<const double2(*)[kSlots]>(sh.diag.f) : reinterpret_cast<const double2(*)[kSlots]>(sh.f);
  // Sums of [p_i]x X [p_j]x, [p_i]x X, X [p_j]x and X over the pairs, X =
  // U_i' U_j; of p_i x h and h.
  double rr[9], rp[9], pr[9], pp[9], racc[kDiag ? 6 : 1];
#pragma unroll
  for (int e = 0; e < 9; ++e) rr[e] = rp[e] = pr[e] = pp[e] = 0.0;
#pragma unroll
  for (int c = 0; c < (kDiag ? 6 : 1); ++c) racc[c] = 0.0;
  TileIdx q[kHalves];
  TileStage<kDiag> st[kHalves];
#pragma unroll
  for (int h = 0; h < kHalves; ++h) {
    if (h < nb) {
      tile_idx(q[h], ta, sh.bt[h], sg.x + h, me);
      tile_data(st[h], q[h], ta, sh.bt[h], tid);
    } else {
      q[h].slot = make_int2(-1, 0);
      q[h].pb = q[h].pe = 0;
      st[h].q = q[h];
    }
    if (kHalves + h < nb) tile_idx(q[h], ta, sh.bt[kHalves + h], sg.x + kHalves + h, me);
  }
  for (int k = 0; k < nb; k += kHalves) {
    __syncthreads();
    int n0 = 0, total = 0, b0 = 0, b1 = 0;
#pragma unroll
    for (int h = 0; h < kHalves; ++h) {
      if (k + h < nb) {
        tile_stage(sh, st[h], tid, h);
        const int n = np && st[h].q.pe > st[h].q.pb ? (st[h].q.pe - st[h].q.pb + np - 1) / np : 0;
        if (h == 0) {
          n0 = n;
          b0 = st[h].q.pb;
        } else {
          b1 = st[h].q.pb;
        }
        total += n;
      }
    }
    __syncthreads();
#pragma unroll
    for (int h = 0; h < kHalves; ++h) {
      const int kn = k + kHalves + h, kq = kn + kHalves;
      if (kn < nb) tile_data(st[h], q[h], ta, sh.bt[kn], tid);
      if (kq < nb) tile_idx(q[h], ta, sh.bt[kq], sg.x + kq, me);
    }
    for (int it = 0; it < total; ++it) {
      const bool second = kHalves == 2 && it >= n0;
      const int p = second ? b1 + (it - n0) * np : b0 + it * np;
      const uint32_t w = reinterpret_cast<const uint16_t*>(sh.pairs[second ? 1 : 0])[p];
      const int base = second ? kBatchSlots : 0;
      const int x = base + (int)(w & 255u), y = base + (int)(w >> 8);
      const double2 a0 = fl[0][x], a1 = fl[1][x], b0v = fl[0][y], b1v = fl[1][y];
      const double2 a2 = fl[2][x], a3 = fl[3][x], b2v = fl[2][y], b3v = fl[3][y];
      const double2 a4 = fl[4][x], a5 = fl[5][x], b4v = fl[4][y], b5v = fl[5][y];
      double X[9];
      X[0] = a0.x * b0v.x + a2.x * b2v.x + a4.x * b4v.x;
      X[1] = a0.x * b0v.y + a2.x * b2v.y + a4.x * b4v.y;
      X[2] = a0.x * b1v.x + a2.x * b3v.x + a4.x * b5v.x;
      X[3] = a0.y * b0v.x + a2.y * b2v.x + a4.y * b4v.x;
      X[4] = a0.y * b0v.y + a2.y * b2v.y + a4.y * b4v.y;
      X[5] = a0.y * b1v.x + a2.y * b3v.x + a4.y * b5v.x;
      X[6] = a1.x * b0v.x + a3.x * b2v.x + a5.x * b4v.x;
      X[7] = a1.x * b0v.y + a3.x * b2v.y + a5.x * b4v.y;
      X[8] = a1.x * b1v.x + a3.x * b3v.x + a5.x * b5v.x;
      if (kDiag && x == y && sh.diag.anchor[x]) {
        X[0] = sh.diag.x[0][x]; X[4] = sh.diag.x[3][x]; X[8] = sh.diag.x[5][x];
        X[1] = X[3] = sh.diag.x[1][x];
        X[2] = X[6] = sh.diag.x[2][x];
        X[5] = X[7] = sh.diag.x[4][x];
      }
      const double px = a1.y, py = a3.y, pz = a5.y;
      const double qx = b1v.y, qy = b3v.y, qz = b5v.y;
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        pp[c] += X[c];
        pp[3 + c] += X[3 + c];
        pp[6 + c] += X[6 + c];
        rp[c] += py * X[6 + c] - pz * X[3 + c];
        rp[3 + c] += pz * X[c] - px * X[6 + c];
        rp[6 + c] += px * X[3 + c] - py * X[c];
      }
      double Y[9];
#pragma unroll
      for (int r = 0; r < 3; ++r) {
        Y[3 * r] = X[3 * r + 1] * qz - X[3 * r + 2] * qy;
        Y[3 * r + 1] = X[3 * r + 2] * qx - X[3 * r] * qz;
        Y[3 * r + 2] = X[3 * r] * qy - X[3 * r + 1] * qx;
      }
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        pr[c] += Y[c];
        pr[3 + c] += Y[3 + c];
        pr[6 + c] += Y[6 + c];
        rr[c] += py * Y[6 + c] - pz * Y[3 + c];
        rr[3 + c] += pz * Y[c] - px * Y[6 + c];
        rr[6 + c] += px * Y[3 + c] - py * Y[c];
      }
      if (kDiag && rhs_part) {
        const double h0 = sh.diag.h[0][x], h1 = sh.diag.h[1][x], h2 = sh.diag.h[2][x];
        racc[0] += py * h2 - pz * h1;
        racc[1 % (kDiag ? 6 : 1)] += pz * h0 - px * h2;
        racc[2 % (kDiag ? 6 : 1)] += px * h1 - py * h0;
        racc[3 % (kDiag ? 6 : 1)] += h0;
        racc[4 % (kDiag ? 6 : 1)] += h1;
        racc[5 % (kDiag ? 6 : 1)] += h2;
      }
    }
  }
  if (np) {
    // -E_i' X E_j and E_i' h, E' = [-[p]x; -I].
    double* out = out_base + (size_t)tid * kPartEntries;
#pragma unroll
    for (int r = 0; r < 3; ++r)
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        out[6 * r + c] = rr[3 * r + c];
        out[6 * r + 3 + c] = -rp[3 * r + c];
        out[6 * (3 + r) + c] = pr[3 * r + c];
        out[6 * (3 + r) + 3 + c] = -pp[3 * r + c];
      }
    if (kDiag)
#pragma unroll
      for (int c = 0; c < 6; ++c) out[36 + c] = -racc[c % (kDiag ? 6 : 1)];
  }
}

// One work item = one segment of a tile (I, J). Work-groups take items_per_wg
// consecutive items of the dispatch order; with xcd_map each XCD walks a
// contiguous range of work-groups (work-group b runs on XCD b mod 8). Neither
// changes a partial.
__global__ __launch_bounds__(kTileBlocks) __attribute__((amdgpu_waves_per_eu(2))) void k_schur_tiles(
    int32_t n_segs, int32_t items_per_wg, int32_t xcd_map, const int32_t* __restrict__ seg_order,
    const int4* __restrict__ segs, const uint32_t* __restrict__ seg_thread, TileArgs ta,
    double* __restrict__ partial) {
  __shared__ TileLds sh;
  const int wgs = (n_segs + items_per_wg - 1) / items_per_wg;
  const int per_xcd = gridDim.x / 8;
  const int wg = xcd_map ? (int)(blockIdx.x % 8) * per_xcd + (int)(blockIdx.x / 8) : (int)blockIdx.x;
  if (wg >= wgs) return;
  const int tid = threadIdx.x;
  for (int it = 0; it < items_per_wg; ++it) {
    const int si = wg * items_per_wg + it;
    if (si >= n_segs) break;
    const int sid = seg_order[si];
    const int4 sg = segs[sid];
    const uint32_t tw = seg_thread[(size_t)sid * kTileBlocks + tid];
    __syncthreads();
    if (tid < sg.y - sg.x) sh.bt[tid] = ta.batches[sg.x + tid];
    __syncthreads();
    double* out = partial + (size_t)sid * kTilePartial;
    if (sg.z == sg.w)
      tile_segment<true>(sh, ta, sg, tw, out);
    else
      tile_segment<false>(sh, ta, sg, tw, out);
  }
}

// S_ij = D_i' (sum of the block's part slots) D_j (segments in segment order,
// parts in part order, listed per upper block; D the row transforms), plus on
// S_ii the direct observation term C_i (sum Jo^T Jo) C_i and the LM diagonal
// D^2 / radius; written to S_ij and S_ji = S_ij^T. One thread per entry; the
// first six threads of a diagonal block also sum the rhs of its row. A
// work-group of seven 36-thread groups takes seven blocks, or with kWide one
// block whose slots k, k + 7, ... group k sums, the seven sums then added in
// group order: a small system has few blocks of many slots each.
constexpr int kFinalizeGroups = 7;

template <bool kWide>
__global__ __launch_bounds__(252) void k_schur_finalize(DevTopology t, int32_t nub, const int4* __restrict__ ublk,
                                                        const int32_t* __restrict__ uslot_ptr,
                                                        const int32_t* __restrict__ uslot,
                                                        const double* __restrict__ partial,
                                                        const double* __restrict__ vR,
                                                        const double* __restrict__ pose_scale,
                                                        const double* __restrict__ pose_diag,
                                                        const double* __restrict__ pose_jtj, double inv_mu,
                                                        double min_diag, double max_diag, double* __restrict__ S,
                                                        double* __restrict__ rhs) {
  __shared__ double red[kFinalizeGroups][kPartEntries];
  __shared__ double mid[kFinalizeGroups][36];
  const int grp = threadIdx.x / 36, e = threadIdx.x % 36, r = e / 6, c = e % 6;
  const int u = kWide ? (int)blockIdx.x : (int)blockIdx.x * kFinalizeGroups + grp;
  const bool valid = u < nub;
  constexpr int st = kWide ? kFinalizeGroups : 1;
  const int4 ub = valid ? ublk[u] : make_int4(0, 0, 0, 1);
  const bool diag = ub.z == ub.w, rhs_entry = diag && e < 6;
  double v = 0.0, g = 0.0;
  if (valid) {
    const int ke = uslot_ptr[u + 1];
    int k = uslot_ptr[u] + (kWide ? grp : 0);
    // Four slots' loads in flight at a time; the sums keep slot order.
    for (; k + 3 * st < ke; k += 4 * st) {
      const double* p0 = partial + (size_t)uslot[k] * kPartEntries;
      const double* p1 = partial + (size_t)uslot[k + st] * kPartEntries;
      const double* p2 = partial + (size_t)uslot[k + 2 * st] * kPartEntries;
      const double* p3 = partial + (size_t)uslot[k + 3 * st] * kPartEntries;
      const double a0 = p0[e], a1 = p1[e], a2 = p2[e], a3 = p3[e];
      v += a0;
      v += a1;
      v += a2;
      v += a3;
      if (rhs_entry) {
        const double b0 = p0[36 + e], b1 = p1[36 + e], b2 = p2[36 + e], b3 = p3[36 + e];
        g += b0;
        g += b1;
        g += b2;
        g += b3;
      }
    }
    for (; k < ke; k += st) {
      const double* p = partial + (size_t)uslot[k] * kPartEntries;
      v += p[e];
      if (rhs_entry) g += p[36 + e];
    }
  }
  red[grp][e] = v;
  if (rhs_entry) red[grp][36 + e] = g;
  __syncthreads();
  if (kWide) {
    double a = red[0][e], b = rhs_entry ? red[0][36 + e] : 0.0;
    for (int q = 1; q < kFinalizeGroups; ++q) {
      a += red[q][e];
      if (rhs_entry) b += red[q][36 + e];
    }
    __syncthreads();
    red[grp][e] = a;
    if (rhs_entry) red[grp][36 + e] = b;
    __syncthreads();
  }
  // Sums times D_j from the right, then D_i' from the left.
  const double* raw = red[grp];
  const double* Ri = vR + 12 * t.var_vertex[ub.z];
  const double* Rj = vR + 12 * (diag || !valid ? t.var_vertex[ub.z] : t.var_vertex[ub.w]);
  double x;
  if (c < 3) x = raw[e] * Rj[9];
  else x = raw[6 * r + 3] * Rj[c - 3] + raw[6 * r + 4] * Rj[c] + raw[6 * r + 5] * Rj[3 + c];
  mid[grp][e] = x;
  __syncthreads();
  if (!valid || (kWide && grp > 0)) return;
  const double* m = mid[grp];
  if (r < 3) v = m[e] * Ri[9];
  else v = m[18 + c] * Ri[r - 3] + m[24 + c] * Ri[r] + m[30 + c] * Ri[3 + r];
  const int i = ub.z, j = ub.w;
  v *= pose_scale[6 * i + r] * pose_scale[6 * j + c];
  if (diag) {
    v += pose_scale[6 * i + r] * pose_scale[6 * i + c] * pose_jtj[36 * i + e];
    if (r == c) {
      const double sc = pose_scale[6 * i + c];
      v += fmin(fmax(sc * sc * pose_diag[6 * i + c], min_diag), max_diag) * inv_mu;
    }
    if (rhs_entry) {
      const double* h = raw + 36;
      const double y = e < 3 ? h[e] * Ri[9] : h[3] * Ri[e - 3] + h[4] * Ri[e] + h[5] * Ri[3 + e];
      rhs[6 * i + e] = y * pose_scale[6 * i + e];
    }
  }
  S[(size_t)36 * ub.x + e] = v;
  if (ub.y != ub.x) S[(size_t)36 * ub.y + c * 6 + r] = v;
}

// ------------------------------------------------------------ landmark admission

struct QualityArgs {
  int32_t min_observers, pad;
  double min_angle_deg;  // smallest accepted max disparity angle of the incidence rays
  double max_dist, min_dist;
  double max_reproj2;    // squared; <= 0: check off
};

// Camera centre and landmark of observation o: ray = c_G - p_G (unit, with
// its length) and the landmark's depth in the camera. The frame chain is
// T_G_C = T_G_M T_M_I T_C_I^-1 and p_C = T_C_I T_M_I^-1 T_G_M^-1 p_G
// (landmark-quality-metrics.cc:118-127).
__device__ inline void quality_ray(const DevTopology& t, const double* __restrict__ vert,
                                   const double* __restrict__ vR, int o, const double* pG, double* ray,
                                   double* dist, double* pC) {
  const int v = t.obs_vertex[o];
  const DevCamera& cam = t.cams[obs_camera(t.obs_meta[o])];
  const double* Rv = vR + 12 * v;           // R_I_M
  const double* pv = vert + 7 * v + 4;      // p_M_I
  const double* TM = t.mission_T + 12 * t.vertex_mission[v];
  double cI[3], cM[3], cG[3];
  mat3t_vec(cam.R_C_I, cam.p_C_I, cI);
  for (int a = 0; a < 3; ++a) cI[a] = -cI[a];
  mat3t_vec(Rv, cI, cM);
  for (int a = 0; a < 3; ++a) cM[a] += pv[a];
  mat3_vec(TM, cM, cG);
  for (int a = 0; a < 3; ++a) cG[a] += TM[9 + a];
  double d[3], pM[3], pI[3];
  for (int a = 0; a < 3; ++a) d[a] = pG[a] - TM[9 + a];
  mat3t_vec(TM, d, pM);
  for (int a = 0; a < 3; ++a) pM[a] -= pv[a];
  mat3_vec(Rv, pM, pI);
  mat3_vec(cam.R_C_I, pI, pC);
  for (int a = 0; a < 3; ++a) pC[a] += cam.p_C_I[a];
  for (int a = 0; a < 3; ++a) ray[a] = cG[a] - pG[a];
  *dist = sqrt(ray[0] * ray[0] + ray[1] * ray[1] + ray[2] * ray[2]);
}

// Observation o of a landmark at pG: its signed distance enters smin, a pixel
// error above the threshold sets bad, and the unit ray goes to ray; returns
// whether the ray is valid.
template <bool kReproj>
__device__ inline bool quality_observation(const DevTopology& t, const double* __restrict__ vert,
                                           const double* __restrict__ vR, const QualityArgs& q, int o,
                                           const double* pG, double& smin, int& bad, double* ray) {
  double dist, pC[3];
  quality_ray(t, vert, vR, o, pG, ray, &dist, pC);
  smin = fmin(smin, pC[2] < 0.0 ? -dist : dist);
  if (kReproj) {
    const DevCamera& cam = t.cams[obs_camera(t.obs_meta[o])];
    double kp[2], jp[6];
    const int st = project_camera(cam.model, cam.xi, cam.dist_type, cam.intr, cam.dist, cam.width, cam.height, pC, kp, jp);
    double e2 = 1.7976931348623157e308;
    if (st == kVisible || st == kOutsideImage) {
      const double du = kp[0] - t.obs_kp[2 * o], dv = kp[1] - t.obs_kp[2 * o + 1];
      e2 = du * du + dv * dv;
    }
    if (e2 > q.max_reproj2) bad = 1;
  }
  const double inv = dist > 0.0 ? 1.0 / dist : 0.0;
  for (int k = 0; k < 3; ++k) ray[k] *= inv;
  return dist > 0.0;
}

// Landmark l in G from its store vertex and mission.
__device__ inline void landmark_in_G(const DevTopology& t, const double* __restrict__ vert,
                                     const double* __restrict__ vR, const double* __restrict__ lm, int l, double* pG) {
  const int a = t.lm_anchor[l];
  const double* TA = t.mission_T + 12 * t.vertex_mission[a];
  double pM[3];
  mat3t_vec(vR + 12 * a, lm + 3 * l, pM);
  for (int k = 0; k < 3; ++k) pM[k] += vert[7 * a + 4 + k];
  mat3_vec(TA, pM, pG);
  for (int k = 0; k < 3; ++k) pG[k] += TA[9 + k];
}

// The verdict; fewer than two valid rays give angle 0 (mincos 1).
__device__ inline uint8_t quality_verdict(const QualityArgs& q, double smin, int bad, double mincos) {
  if (bad || smin > q.max_dist || smin < q.min_dist) return 0;
  const double angle_deg = acos(fmin(mincos, 1.0)) * (180.0 / 3.14159265358979323846);
  return angle_deg < q.min_angle_deg ? 0 : 1;
}

// isVisualLandmarkWellConstrained of every landmark: signed distance to the
// closest observer, optional reprojection check, smallest |cos| over the
// pairs of unit rays. A landmark has about ten observers, so a wave takes
// four landmarks at once, one for each row of 16 lanes (at most
// kQualityRowRays rays each in LDS); lane i of a row pairs its ray with rays
// i + 1, i + 2, ... i + n / 2 (cyclically), which meets every pair. A landmark
// with more observers is then taken by the whole wave, its first kQualityRays
// rays in the same LDS and the rest recomputed. Minima do not depend on the
// order, so neither does the result. 120000 landmarks of 300 keyframes, whole
// call: 335 us with one landmark a wave (10 of its 64 lanes at work), 95 us.
constexpr int kQualityRowRays = 64;
constexpr int kQualityRays = 4 * kQualityRowRays;
constexpr int kQualityWaves = 2;  // waves a work-group (14 KB of LDS)

template <bool kReproj>
__global__ __launch_bounds__(64 * kQualityWaves) void k_landmark_quality(
    DevTopology t, const double* __restrict__ vert, const double* __restrict__ vR, const double* __restrict__ lm,
    QualityArgs q, uint8_t* __restrict__ good) {
  __shared__ double ray_lds[kQualityWaves][kQualityRays][3];
  __shared__ uint8_t valid_lds[kQualityWaves][kQualityRays];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, row = lane >> 4, rl = lane & 15;
  const int l0 = 4 * (blockIdx.x * kQualityWaves + wave);
  double(*rays)[3] = ray_lds[wave];
  uint8_t* valid = valid_lds[wave];
  // LDS is written and read by one wave alone: no barrier, only the order.
  auto lds_order = [] {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  };
  const double kMax = 1.7976931348623157e308;  // DBL_MAX
  {
    const int l = l0 + row, base = row * kQualityRowRays;
    const int ob = l < t.L ? t.lm_begin[l] : 0, n_all = l < t.L ? t.lm_begin[l + 1] - ob : 0;
    const bool mine = l < t.L && n_all >= q.min_observers && n_all <= kQualityRowRays;
    const int n = mine ? n_all : 0;
    double smin = kMax;
    int bad = 0;
    if (n > 0) {
      double pG[3];
      landmark_in_G(t, vert, vR, lm, l, pG);
      for (int oi = rl; oi < n; oi += 16)
        valid[base + oi] = quality_observation<kReproj>(t, vert, vR, q, ob + oi, pG, smin, bad, rays[base + oi]);
    }
    smin = row_min(smin);
    bad = ((__ballot(bad) >> (16 * row)) & 0xFFFFu) != 0;
    lds_order();
    double mincos = 1.0;
    for (int i = rl; i < n; i += 16) {
      if (!valid[base + i]) continue;
      const double r0 = rays[base + i][0], r1 = rays[base + i][1], r2 = rays[base + i][2];
      for (int d = 1; d <= n / 2; ++d) {
        const int k = i + d, j = base + (k < n ? k : k - n);
        if (valid[j]) mincos = fmin(mincos, fabs(r0 * rays[j][0] + r1 * rays[j][1] + r2 * rays[j][2]));
      }
    }
    mincos = row_min(mincos);
    if (l < t.L && n_all <= kQualityRowRays && rl == 0)
      good[l] = n_all >= q.min_observers ? quality_verdict(q, smin, bad, mincos) : 0;
    lds_order();
  }
  for (int s = 0; s < 4 && l0 + s < t.L; ++s) {
    const int l = l0 + s, ob = t.lm_begin[l], n = t.lm_begin[l + 1] - ob;
    if (n <= kQualityRowRays) continue;
    if (n < q.min_observers) {
      if (lane == 0) good[l] = 0;
      continue;
    }
    double pG[3];
    landmark_in_G(t, vert, vR, lm, l, pG);
    double smin = kMax;
    int bad = 0;
    for (int oi = lane; oi < n; oi += 64) {
      double ray[3];
      const bool ok = quality_observation<kReproj>(t, vert, vR, q, ob + oi, pG, smin, bad, ray);
      if (oi < kQualityRays) {
        for (int k = 0; k < 3; ++k) rays[oi][k] = ray[k];
        valid[oi] = ok;
      }
    }
    smin = wave_min(smin);
    bad = __any(bad);
    lds_order();
    double mincos = 1.0;
    if (!bad && !(smin > q.max_dist || smin < q.min_dist)) {
      auto ray_of = [&](int i, double* r) -> bool {
        if (i < kQualityRays) {
          for (int k = 0; k < 3; ++k) r[k] = rays[i][k];
          return valid[i];
        }
        double unused = kMax;
        int none = 0;
        return quality_observation<false>(t, vert, vR, q, ob + i, pG, unused, none, r);
      };
      for (int i = 0; i + 1 < n; ++i) {
        double ri[3];
        if (!ray_of(i, ri)) continue;
        for (int j = i + 1 + lane; j < n; j += 64) {
          double rj[3];
          if (ray_of(j, rj)) mincos = fmin(mincos, fabs(ri[0] * rj[0] + ri[1] * rj[1] + ri[2] * rj[2]));
        }
      }
    }
    mincos = wave_min(mincos);
    if (lane == 0) good[l] = quality_verdict(q, smin, bad, mincos);
    lds_order();
  }
}

// ------------------------------------------------------------ PCG

// 6x6 SPD inverse of every diagonal block of S (block-Jacobi preconditioner).
__global__ void k_block_inverse(int32_t Pvar, const int32_t* __restrict__ diag_pos, const double* __restrict__ S,
                                double* __restrict__ Minv, int32_t* __restrict__ fail) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= Pvar) return;
  const double* A = S + (size_t)36 * diag_pos[i];
  double L[36];
  for (int k = 0; k < 36; ++k) L[k] = 0.0;
  bool ok = true;
  for (int j = 0; j < 6; ++j) {
    double s = A[j * 6 + j];
    for (int k = 0; k < j; ++k) s -= L[j * 6 + k] * L[j * 6 + k];
    if (!(s > 0.0)) { ok = false; s = 1.0; }
    const double ljj = sqrt(s);
    L[j * 6 + j] = ljj;
    for (int r = j + 1; r < 6; ++r) {
      double v = A[r * 6 + j];
      for (int k = 0; k < j; ++k) v -= L[r * 6 + k] * L[j * 6 + k];
      L[r * 6 + j] = v / ljj;
    }
  }
  if (!ok) atomicAdd(fail, 1);
  // Columns of A^-1 by forward / backward substitution.
  double* out = Minv + (size_t)36 * i;
  for (int c = 0; c < 6; ++c) {
    double y[6];
    for (int r = 0; r < 6; ++r) {
      double s = (r == c) ? 1.0 : 0.0;
      for (int k = 0; k < r; ++k) s -= L[r * 6 + k] * y[k];
      y[r] = s / L[r * 6 + r];
    }
    for (int r = 5; r >= 0; --r) {
      double s = y[r];
      for (int k = r + 1; k < 6; ++k) s -= L[k * 6 + r] * y[k];
      y[r] = s / L[r * 6 + r];
    }
    for (int r = 0; r < 6; ++r) out[r * 6 + c] = y[r];
  }
}

// ------------------------------------------------------------ step

// Landmark step and model cost change. With y the solution of the scaled
// system, w = C_p y_p (per vertex) and u = C_l y_l = Z_l (g_l - sum W' y_p):
// J y = Jl u + Jo w_o + Jl M w_a per observation and
// model_cost_change = sum (J y)'r - |J y|^2 / 2 (ceres ComputeTrustRegionStep).
// From the records, J y = K (s + G (u + M w_a)), s = |q|^2 p_I x w_rot -
// R_I_M w_pos, G = R_I_M R_M_B, so the landmark side is taken in the landmark's
// mission frame: the sums of R_M_I K'K s per landmark, then R_M_B' u once.
// One work-group per linearization tile of whole landmarks: each observation
// record is read once; the landmark sums are taken by the segment heads in a
// fixed order. Tiles of landmarks split over several tiles are left to
// k_back_substitute_split (their part entries are zero here). u of inactive
// or observation-less landmarks is not written (kept zero).
__device__ inline void landmark_step(const DevTopology& t, int l, const double* __restrict__ vR,
                                     const double* __restrict__ lm, const double* __restrict__ lm_acc,
                                     const double* __restrict__ lm_z, const double* __restrict__ w,
                                     double* tv, double* u, double* Mwa) {
  const uint32_t flags = t.lm_flags[l];
  const double* acc = lm_acc + (size_t)kLmAcc * l;
  Mwa[0] = Mwa[1] = Mwa[2] = 0.0;
  if (flags & kLmAnchorVar) {
    const int a = t.lm_anchor[l];
    double M[18];
    anchor_map(lm + 3 * l, vR + 12 * a, vR[12 * a + 9], M);
    const double* wa = w + 6 * t.vertex_var[a];
    for (int r = 0; r < 3; ++r) {
      double s = 0.0;
      for (int c = 0; c < 6; ++c) s += M[r * 6 + c] * wa[c];
      Mwa[r] = s;
    }
  }
  u[0] = u[1] = u[2] = 0.0;
  if (!(flags & kLmConstant)) {
    if (flags & kLmAnchorVar) {
      double VLM[9];
      sym3_full(acc + 6, VLM);
      for (int a = 0; a < 3; ++a) tv[a] -= VLM[a * 3] * Mwa[0] + VLM[a * 3 + 1] * Mwa[1] + VLM[a * 3 + 2] * Mwa[2];
    }
    double y[3];
    tri_vec(lm_z + (size_t)kLmZ * l, tv, y);
    trit_vec(lm_z + (size_t)kLmZ * l, y, u);
  }
}

// Vector x between the landmark's mission frame and the observer's IMU frame
// of a pose-coupled observation by vertex v: to_imu R_I_M (R_M_LM) x, else the
// transpose.
__device__ inline void rotate_observer(const DevTopology& t, int32_t type, int l, int v, const double* Rv, bool to_imu,
                                       const double* x, double* out) {
  double m[3];
  if (type != kTypeGlobal) {
    if (to_imu) mat3_vec(Rv, x, out);
    else mat3t_vec(Rv, x, out);
    return;
  }
  const double* TL = t.mission_T + 12 * t.vertex_mission[t.lm_anchor[l]];
  const double* TM = t.mission_T + 12 * t.vertex_mission[v];
  double g[3];
  if (to_imu) {
    mat3_vec(TL, x, g);
    mat3t_vec(TM, g, m);
    mat3_vec(Rv, m, out);
  } else {
    mat3t_vec(Rv, x, m);
    mat3_vec(TM, m, g);
    mat3t_vec(TL, g, out);
  }
}

// s of an observation: |q|^2 p_I x w_rot - R_I_M w_pos (J_observer w = K s).
template <class Rec>
__device__ inline void observer_motion(const Rec& rec, const double* Rv, const double* wo, double* s) {
  double rp[3];
  mat3_vec(Rv, wo + 3, rp);
  const double n2 = Rv[9];
  s[0] = n2 * (rec.p(1) * wo[2] - rec.p(2) * wo[1]) - rp[0];
  s[1] = n2 * (rec.p(2) * wo[0] - rec.p(0) * wo[2]) - rp[1];
  s[2] = n2 * (rec.p(0) * wo[1] - rec.p(1) * wo[0]) - rp[2];
}

template <bool kF32>
__global__ __launch_bounds__(kObsTile) void k_back_substitute(DevTopology t, const int32_t* __restrict__ tile_begin,
                                                              const double* __restrict__ vR,
                                                              const double* __restrict__ lm,
                                                              const void* __restrict__ obs_rec,
                                                              const double* __restrict__ lm_acc,
                                                              const double* __restrict__ lm_z,
                                                              const double* __restrict__ w, double* __restrict__ u_out,
                                                              double* __restrict__ part) {
  __shared__ double red[kObsTile * 3];
  __shared__ double ush[kObsTile * 6];  // u, and R_B_M' (u + M w_a), at each segment head
  __shared__ int32_t seg[kObsTile];
  __shared__ double lds4[4];
  const int tid = threadIdx.x;
  const int b = tile_begin[blockIdx.x], e = tile_begin[blockIdx.x + 1];
  if (t.lm_flags[t.obs_landmark[b]] & kLmSplit) {  // whole tile belongs to a split landmark
    if (tid == 0) part[2 * blockIdx.x] = part[2 * blockIdx.x + 1] = 0.0;
    return;
  }
  const int o = b + tid;
  int32_t l = -1, v = 0, type = kTypeKeyframe;
  uint32_t flags = 0;
  double K[6], s[3] = {0, 0, 0}, c[3] = {0, 0, 0}, r[2] = {0, 0};
  const double* Rv = vR;
  // The observation itself says whether its landmark was active when the
  // structure was built, and brings its observer's variable (obs_col): no load
  // waits for the landmark's flags. Values of a landmark deactivated since are
  // left out below. 500 keyframes, all active / 60 % inactive / three quarters of
  // the tiles inactive: 98 / 64 / 32 us; loaded whatever the landmark's state 97 /
  // 79 / 47, after its flags 102 / 66 / 33.
  if (o < e) {
    l = t.obs_landmark[o];
    const int32_t meta = t.obs_meta[o], col = t.obs_col[o];
    v = t.obs_vertex[o];
    if (obs_built_active(meta)) {
      const RecView<kF32> rec(obs_rec, o);
      flags = t.lm_flags[l];
      type = obs_type(meta);
      for (int k = 0; k < 6; ++k) K[k] = rec.K(k);
      r[0] = rec.r(0);
      r[1] = rec.r(1);
      if (type != kTypeKeyframe) {
        Rv = vR + 12 * v;
        if (col >= 0) {
          observer_motion(rec, Rv, w + 6 * col, s);
          const double j0 = K[0] * s[0] + K[1] * s[1] + K[2] * s[2], j1 = K[3] * s[0] + K[4] * s[1] + K[5] * s[2];
          const double kj[3] = {-(K[0] * j0 + K[3] * j1), -(K[1] * j0 + K[4] * j1), -(K[2] * j0 + K[5] * j1)};
          rotate_observer(t, type, l, v, Rv, false, kj, c);
        }
      }
    }
  }
  const bool active = o < e && (flags & kLmActive);
  for (int k = 0; k < 3; ++k) red[tid * 3 + k] = c[k];
  seg[tid] = active ? l : -1;
  __syncthreads();
  double uu = 0.0;
  if (active && (tid == 0 || seg[tid - 1] != l)) {
    const double* acc = lm_acc + (size_t)kLmAcc * l;
    const double* Ra = vR + 12 * t.lm_anchor[l];
    double sum[3] = {0, 0, 0}, tv[3];
    for (int k = tid; k < kObsTile && seg[k] == l; ++k)
      for (int a = 0; a < 3; ++a) sum[a] += red[k * 3 + a];
    mat3_vec(Ra, sum, tv);
    for (int a = 0; a < 3; ++a) tv[a] += acc[12 + a];
    double u[3], Mwa[3], um[3];
    landmark_step(t, l, vR, lm, lm_acc, lm_z, w, tv, u, Mwa);
    uu = u[0] * u[0] + u[1] * u[1] + u[2] * u[2];
    for (int a = 0; a < 3; ++a) {
      u_out[3 * l + a] = u[a];
      ush[tid * 6 + a] = u[a];
      Mwa[a] += u[a];
    }
    mat3t_vec(Ra, Mwa, um);
    for (int a = 0; a < 3; ++a) ush[tid * 6 + 3 + a] = um[a];
  }
  __syncthreads();
  double mcc = 0.0;
  if (active) {
    const int h = t.lm_begin[l] - b;
    double y[3];
    if (type == kTypeKeyframe) {
      for (int a = 0; a < 3; ++a) y[a] = ush[h * 6 + a];
    } else {
      rotate_observer(t, type, l, v, Rv, true, &ush[h * 6 + 3], y);
      for (int a = 0; a < 3; ++a) y[a] += s[a];
    }
    const double j0 = K[0] * y[0] + K[1] * y[1] + K[2] * y[2], j1 = K[3] * y[0] + K[4] * y[1] + K[5] * y[2];
    mcc = j0 * r[0] + j1 * r[1] - 0.5 * (j0 * j0 + j1 * j1);
  }
  const double s1 = block_sum256(mcc, lds4);
  const double s2 = block_sum256(uu, lds4);
  if (tid == 0) {
    part[2 * blockIdx.x] = s1;
    part[2 * blockIdx.x + 1] = s2;
  }
}

// The same for the landmarks split over several tiles, one thread each.
template <bool kF32>
__global__ __launch_bounds__(256) void k_back_substitute_split(DevTopology t, int32_t n_split,
                                                               const int32_t* __restrict__ split_ids,
                                                               const double* __restrict__ vR,
                                                               const double* __restrict__ lm,
                                                               const void* __restrict__ obs_rec,
                                                               const double* __restrict__ lm_acc,
                                                               const double* __restrict__ lm_z,
                                                               const double* __restrict__ w,
                                                               double* __restrict__ u_out, double* __restrict__ part) {
  __shared__ double lds4[4];
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  double mcc = 0.0, uu = 0.0;
  if (k < n_split && (t.lm_flags[split_ids[k]] & kLmActive)) {
    const int l = split_ids[k];
    const int lb = t.lm_begin[l], le = t.lm_begin[l + 1];
    const double* acc = lm_acc + (size_t)kLmAcc * l;
    const double* Ra = vR + 12 * t.lm_anchor[l];
    double sum[3] = {0, 0, 0}, tv[3];
    for (int o = lb; o < le; ++o) {
      const int32_t meta = t.obs_meta[o], type = obs_type(meta);
      if (type == kTypeKeyframe || !obs_observer_var(meta)) continue;
      const RecView<kF32> rec(obs_rec, o);
      const int v = t.obs_vertex[o];
      double s[3], c[3];
      observer_motion(rec, vR + 12 * v, w + 6 * t.vertex_var[v], s);
      const double j0 = rec.K(0) * s[0] + rec.K(1) * s[1] + rec.K(2) * s[2];
      const double j1 = rec.K(3) * s[0] + rec.K(4) * s[1] + rec.K(5) * s[2];
      const double kj[3] = {-(rec.K(0) * j0 + rec.K(3) * j1), -(rec.K(1) * j0 + rec.K(4) * j1),
                            -(rec.K(2) * j0 + rec.K(5) * j1)};
      rotate_observer(t, type, l, v, vR + 12 * v, false, kj, c);
      for (int a = 0; a < 3; ++a) sum[a] += c[a];
    }
    mat3_vec(Ra, sum, tv);
    for (int a = 0; a < 3; ++a) tv[a] += acc[12 + a];
    double u[3], Mwa[3], um[3];
    landmark_step(t, l, vR, lm, lm_acc, lm_z, w, tv, u, Mwa);
    uu = u[0] * u[0] + u[1] * u[1] + u[2] * u[2];
    for (int a = 0; a < 3; ++a) {
      u_out[3 * l + a] = u[a];
      Mwa[a] += u[a];
    }
    mat3t_vec(Ra, Mwa, um);
    for (int o = lb; o < le; ++o) {
      const int32_t meta = t.obs_meta[o], type = obs_type(meta);
      const RecView<kF32> rec(obs_rec, o);
      double y[3] = {u[0], u[1], u[2]};
      if (type != kTypeKeyframe) {
        const int v = t.obs_vertex[o];
        const double* Rv = vR + 12 * v;
        rotate_observer(t, type, l, v, Rv, true, um, y);
        if (obs_observer_var(meta)) {
          double s[3];
          observer_motion(rec, Rv, w + 6 * t.vertex_var[v], s);
          for (int a = 0; a < 3; ++a) y[a] += s[a];
        }
      }
      const double j0 = rec.K(0) * y[0] + rec.K(1) * y[1] + rec.K(2) * y[2];
      const double j1 = rec.K(3) * y[0] + rec.K(4) * y[1] + rec.K(5) * y[2];
      mcc += j0 * rec.r(0) + j1 * rec.r(1) - 0.5 * (j0 * j0 + j1 * j1);
    }
  }
  const double s1 = block_sum256(mcc, lds4);
  const double s2 = block_sum256(uu, lds4);
  if (threadIdx.x == 0) { part[2 * blockIdx.x] = s1; part[2 * blockIdx.x + 1] = s2; }
}

// Vertex step w = C_p y_p, candidate vertices x [+] (-w) (JPL Plus) and their
// rotation records (as k_vertex_prep); partials of |w|^2 and of |x|^2 over
// variable vertices.
__global__ __launch_bounds__(256) void k_step_vertices(DevTopology t, const double* __restrict__ vert,
                                                       const double* __restrict__ y,
                                                       const double* __restrict__ pose_scale, double* __restrict__ w,
                                                       double* __restrict__ cand, double* __restrict__ cand_vR,
                                                       double* __restrict__ part_w, double* __restrict__ part_x) {
  __shared__ double lds4[4];
  const int v = blockIdx.x * blockDim.x + threadIdx.x;
  double xx = 0.0, ww = 0.0;
  if (v < t.P) {
    const double* x = vert + 7 * v;
    double c[7];
    const int32_t j = t.vertex_var[v];
    if (j >= 0) {
      double wv[6];
      for (int k = 0; k < 6; ++k) {
        wv[k] = y[6 * j + k] * pose_scale[6 * j + k];
        w[6 * j + k] = wv[k];
        ww += wv[k] * wv[k];
      }
      const double d[3] = {-wv[0], -wv[1], -wv[2]};
      quat_plus_jpl(x, d, c);
      c[4] = x[4] - wv[3];
      c[5] = x[5] - wv[4];
      c[6] = x[6] - wv[5];
      for (int k = 0; k < 7; ++k) xx += x[k] * x[k];
    } else {
      for (int k = 0; k < 7; ++k) c[k] = x[k];
    }
    double* out = cand + 7 * v;
    for (int k = 0; k < 7; ++k) out[k] = c[k];
    vertex_rotation(c, cand_vR + 12 * v);
  }
  const double sw = block_sum256(ww, lds4);
  const double sx = block_sum256(xx, lds4);
  if (threadIdx.x == 0) {
    part_w[blockIdx.x] = sw;
    part_x[blockIdx.x] = sx;
  }
}

// Candidate landmarks x - u; partials of |x|^2 over variable landmarks.
__global__ __launch_bounds__(256) void k_candidate_landmarks(DevTopology t, const double* __restrict__ lm,
                                                             const double* __restrict__ u,
                                                             double* __restrict__ cand, double* __restrict__ part) {
  __shared__ double lds4[4];
  const int l = blockIdx.x * blockDim.x + threadIdx.x;
  double xx = 0.0;
  if (l < t.L) {
    const uint32_t f = t.lm_flags[l];
    const bool var = (f & kLmActive) && !(f & kLmConstant);
    for (int k = 0; k < 3; ++k) {
      const double x = lm[3 * l + k];
      cand[3 * l + k] = var ? x - u[3 * l + k] : x;
      if (var) xx += x * x;
    }
  }
  const double s = block_sum256(xx, lds4);
  if (threadIdx.x == 0) part[blockIdx.x] = s;
}

// max |x - Plus(x, -g)| over variable blocks (ceres gradient_max_norm).
__global__ __launch_bounds__(256) void k_gradient_norm(DevTopology t, const double* __restrict__ vert,
                                                       const double* __restrict__ pose_grad,
                                                       const double* __restrict__ lm_acc,
                                                       double* __restrict__ part) {
  __shared__ double red[4];
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  double m = 0.0;
  if (k < t.Pvar) {
    const double* x = vert + 7 * t.var_vertex[k];
    const double* g = pose_grad + 6 * k;
    const double d[3] = {-g[0], -g[1], -g[2]};
    double q[4];
    quat_plus_jpl(x, d, q);
    for (int c = 0; c < 4; ++c) m = fmax(m, fabs(x[c] - q[c]));
    for (int c = 0; c < 3; ++c) m = fmax(m, fabs(g[3 + c]));
  } else if (k - t.Pvar < t.L) {
    const int l = k - t.Pvar;
    const uint32_t f = t.lm_flags[l];
    if ((f & kLmActive) && !(f & kLmConstant)) {
      const double* g = lm_acc + (size_t)kLmAcc * l + 12;
      for (int c = 0; c < 3; ++c) m = fmax(m, fabs(g[c]));
    }
  }
  m = wave_max(m);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
  __syncthreads();
  if (threadIdx.x == 0) part[blockIdx.x] = fmax(fmax(red[0], red[1]), fmax(red[2], red[3]));
}

// Fixed-order final reduction of partial arrays: out[k] = sum (or max) of
// parts[k] (stride `stride`, n entries). One block per output.
__device__ inline void reduce_parts(int32_t n, int32_t stride, int32_t offset, int32_t is_max,
                                    const double* __restrict__ parts, double* __restrict__ out) {
  __shared__ double lds4[4];
  double s = 0.0;
  for (int k = threadIdx.x; k < n; k += blockDim.x) {
    const double v = parts[(size_t)k * stride + offset];
    s = is_max ? fmax(s, v) : s + v;
  }
  if (is_max) {
    s = wave_max(s);
    __shared__ double red[4];
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) *out = fmax(fmax(red[0], red[1]), fmax(red[2], red[3]));
  } else {
    s = block_sum256(s, lds4);
    if (threadIdx.x == 0) *out = s;
  }
}

__global__ void k_reduce(int32_t n, int32_t stride, int32_t offset, int32_t is_max, const double* __restrict__ parts,
                         double* __restrict__ out) {
  reduce_parts(n, stride, offset, is_max, parts, out);
}

// Several independent reductions in one launch, work-group b computing
// reduction b exactly as k_reduce does; the step's failure counter is handed
// over and cleared with them.
__global__ void k_reduce_many(ReduceBatch batch) {
  const ReduceDesc& d = batch.d[blockIdx.x];
  reduce_parts(d.n, d.stride, d.offset, d.is_max, d.parts, d.out);
  if (batch.fail && blockIdx.x == 0 && threadIdx.x == 0) {
    *batch.fail_out = (double)*batch.fail;
    *batch.fail = 0;
  }
}

// ------------------------------------------------------------ Evaluate API

// Every Jacobian block of VisualReprojectionError::Evaluate
// (visual-error-term-inl.h:184-367), in the caller's order, ambient or
// tangent. Observation index is in the original (caller) order via perm. Each
// block goes to an array of its own, as the caller has it, so that it is
// copied out as it is.
__global__ __launch_bounds__(256) void k_evaluate_full(DevTopology t, const double* __restrict__ vert,
                                                       const double* __restrict__ vR,
                                                       const double* __restrict__ lm,
                                                       const double* __restrict__ baseframes,
                                                       const double* __restrict__ cam_q, int32_t tangent,
                                                       const int32_t* __restrict__ perm, double* __restrict__ res,
                                                       EvalOut jout, int32_t want_jac) {
  const int o = blockIdx.x * blockDim.x + threadIdx.x;
  if (o >= t.N) return;
  const int32_t meta = t.obs_meta[o];
  const int32_t type = obs_type(meta);
  const int32_t ci = obs_camera(meta);
  const DevCamera& cam = t.cams[ci];
  const int32_t l = t.obs_landmark[o];
  const int32_t v = t.obs_vertex[o];
  const int32_t a = t.lm_anchor[l];
  const double* pB = lm + 3 * l;
  const double* Rv = vR + 12 * v;
  const double* Ra = vR + 12 * a;
  // Frame chain with all intermediate rotations.
  double pI[3], pG[3] = {0, 0, 0};
  double D_pI_pB[9], D_pI_pa[9], D_pI_pGLM[9], D_pI_pGM[9], D_pI_pv[9];
  double D_pI_qa[9], D_pI_qGLM[9], D_pI_qGM[9], D_pI_qv[9];
  for (int k = 0; k < 9; ++k) {
    D_pI_pB[k] = D_pI_pa[k] = D_pI_pGLM[k] = D_pI_pGM[k] = D_pI_pv[k] = 0.0;
    D_pI_qa[k] = D_pI_qGLM[k] = D_pI_qGM[k] = D_pI_qv[k] = 0.0;
  }
  auto skew_right = [](const double* A, const double* p, double* out) {  // A [p]x
    for (int r = 0; r < 3; ++r) {
      out[r * 3 + 0] = A[r * 3 + 1] * p[2] - A[r * 3 + 2] * p[1];
      out[r * 3 + 1] = A[r * 3 + 2] * p[0] - A[r * 3 + 0] * p[2];
      out[r * 3 + 2] = A[r * 3 + 0] * p[1] - A[r * 3 + 1] * p[0];
    }
  };
  if (type == kTypeKeyframe) {
    for (int k = 0; k < 3; ++k) pI[k] = pB[k];
    for (int k = 0; k < 9; ++k) D_pI_pB[k] = (k % 4 == 0) ? 1.0 : 0.0;
  } else {
    double pM[3];
    mat3t_vec(Ra, pB, pM);
    const double* pa = vert + 7 * a + 4;
    for (int k = 0; k < 3; ++k) pM[k] += pa[k];
    double A[9];  // d p_I / d p_M
    for (int k = 0; k < 9; ++k) A[k] = Rv[k];
    double P_M_LM[9];  // d p_M / d p_LM
    for (int k = 0; k < 9; ++k) P_M_LM[k] = (k % 4 == 0) ? 1.0 : 0.0;
    if (type == kTypeGlobal) {
      const double* TL = t.mission_T + 12 * t.vertex_mission[a];
      const double* TM = t.mission_T + 12 * t.vertex_mission[v];
      double pLM[3] = {pM[0], pM[1], pM[2]};
      mat3_vec(TL, pLM, pG);
      for (int k = 0; k < 3; ++k) pG[k] += TL[9 + k];
      double d[3] = {pG[0] - TM[9], pG[1] - TM[10], pG[2] - TM[11]};
      mat3t_vec(TM, d, pM);
      // d p_M / d p_LM = R_M_G R_G_LM
      for (int r = 0; r < 3; ++r)
        for (int c = 0; c < 3; ++c)
          P_M_LM[r * 3 + c] = TM[r] * TL[c] + TM[3 + r] * TL[3 + c] + TM[6 + r] * TL[6 + c];
      double AR[9];  // d p_I / d p_G = R_I_M R_M_G
      for (int r = 0; r < 3; ++r)
        for (int c = 0; c < 3; ++c) AR[r * 3 + c] = A[r * 3] * TM[c * 3] + A[r * 3 + 1] * TM[c * 3 + 1] + A[r * 3 + 2] * TM[c * 3 + 2];
      for (int k = 0; k < 9; ++k) { D_pI_pGLM[k] = AR[k]; D_pI_pGM[k] = -AR[k]; }
      // Reference forms (visual-error-term-inl.h:208-209) use [p_G]x for both baseframes.
      skew_right(D_pI_pGLM, pG, D_pI_qGLM);
      skew_right(D_pI_pGM, pG, D_pI_qGM);
    }
    const double* pv = vert + 7 * v + 4;
    const double dm[3] = {pM[0] - pv[0], pM[1] - pv[1], pM[2] - pv[2]};
    mat3_vec(Rv, dm, pI);
    for (int k = 0; k < 9; ++k) D_pI_pv[k] = -A[k];
    double T1[9];
    mat3_mul(A, P_M_LM, T1);  // d p_I / d p_LM
    for (int k = 0; k < 9; ++k) D_pI_pa[k] = T1[k];
    mat3_mul_bt(T1, Ra, D_pI_pB);  // * R_LM_B
    skew_right(D_pI_pB, pB, D_pI_qa);
    for (int k = 0; k < 9; ++k) D_pI_qa[k] = -D_pI_qa[k];
    double I3[9] = {1, 0, 0, 0, 1, 0, 0, 0, 1};
    skew_right(I3, pI, D_pI_qv);  // [p_I]x
  }
  double pC[3];
  mat3_vec(cam.R_C_I, pI, pC);
  for (int k = 0; k < 3; ++k) pC[k] += cam.p_C_I[k];
  double kp[2], jp[6];
  const int32_t status = project_camera(cam.model, cam.xi, cam.dist_type, cam.intr, cam.dist, cam.width, cam.height, pC, kp, jp);
  const bool failed = projection_failed(status, pC, kp);
  const double sinv = t.obs_sinv[o];
  const int32_t oo = perm[o];
  if (res) {
    res[2 * oo] = failed ? 0.0 : (kp[0] - t.obs_kp[2 * o]) * sinv;
    res[2 * oo + 1] = failed ? 0.0 : (kp[1] - t.obs_kp[2 * o + 1]) * sinv;
  }
  if (!want_jac) return;
  // K = d r / d p_I = jp sinv R_C_I; Kc = jp sinv (d r / d p_C).
  double Kc[6], K[6];
  for (int k = 0; k < 6; ++k) Kc[k] = failed ? 0.0 : jp[k] * sinv;
  for (int r = 0; r < 2; ++r)
    for (int c = 0; c < 3; ++c)
      K[r * 3 + c] = Kc[r * 3] * cam.R_C_I[c] + Kc[r * 3 + 1] * cam.R_C_I[3 + c] + Kc[r * 3 + 2] * cam.R_C_I[6 + c];
  // Block 9 (requested only with the xi flag) is d r / d xi of a
  // unified-projection camera.
  const int amb[10] = {3, 7, 7, 7, 7, 4, 3, 4, 4, 1};
  const int tng[10] = {3, 6, 6, 6, 6, 3, 3, 4, 4, 1};
  auto at = [&](int b) { return jout.block[b] + (size_t)oo * jout.stride[b]; };
  auto zero_block = [&](int b) {
    const int n = 2 * (tangent ? tng[b] : amb[b]);
    double* J = at(b);
    for (int k = 0; k < n; ++k) J[k] = 0.0;
  };
  // Write J = Kx * D (2x3) into columns [c0, c0+3) of a block of width w.
  auto put3 = [&](int b, int c0, const double* Kx, const double* D, double scale) {
    const int w = tangent ? tng[b] : amb[b];
    double* J = at(b);
    for (int r = 0; r < 2; ++r)
      for (int c = 0; c < 3; ++c)
        J[r * w + c0 + c] =
            scale * (Kx[r * 3] * D[c] + Kx[r * 3 + 1] * D[3 + c] + Kx[r * 3 + 2] * D[6 + c]);
  };
  // Rotation block: tangent = J_q |q|^2 ; ambient = J_q * 4 Jq(q)^T.
  auto put_rot = [&](int b, const double* Kx, const double* D, const double* q) {
    double Jr[6];
    for (int r = 0; r < 2; ++r)
      for (int c = 0; c < 3; ++c) Jr[r * 3 + c] = Kx[r * 3] * D[c] + Kx[r * 3 + 1] * D[3 + c] + Kx[r * 3 + 2] * D[6 + c];
    const int w = tangent ? tng[b] : amb[b];
    double* J = at(b);
    if (tangent) {
      const double n2 = q[0] * q[0] + q[1] * q[1] + q[2] * q[2] + q[3] * q[3];
      for (int r = 0; r < 2; ++r)
        for (int c = 0; c < 3; ++c) J[r * w + c] = Jr[r * 3 + c] * n2;
    } else {
      // 4 * 0.5 * [[w,-z,y],[z,w,-x],[-y,x,w],[-x,-y,-z]]^T (quaternion-param-jpl.cc:8-32)
      const double x = q[0], y = q[1], z = q[2], w4 = q[3];
      const double JqT[12] = {w4, z, -y, -x, -z, w4, x, -y, y, -x, w4, -z};  // 3x4
      for (int r = 0; r < 2; ++r)
        for (int c = 0; c < 4; ++c)
          J[r * w + c] =
              2.0 * (Jr[r * 3] * JqT[c] + Jr[r * 3 + 1] * JqT[4 + c] + Jr[r * 3 + 2] * JqT[8 + c]);
    }
  };
  const double* qa = vert + 7 * a;
  const double* qv = vert + 7 * v;
  const double* qGLM = baseframes + 7 * t.vertex_mission[a];
  const double* qGM = baseframes + 7 * t.vertex_mission[v];
  const double* qCI = cam_q + 7 * ci;
  for (int b = 0; b < 10; ++b) {
    if (!jout.block[b]) continue;
    const bool used = (b == 0) || (b == 5) || (b == 6) || (b == 7) || (b == 8) ||
                      (b == 9 && cam.model == kCameraUnifiedProjection) ||
                      ((b == 1 || b == 4) && type != kTypeKeyframe) || ((b == 2 || b == 3) && type == kTypeGlobal);
    if (failed || !used) {
      zero_block(b);
      continue;
    }
    const int pc0 = tangent ? 3 : 4;  // column of the position part of a pose block
    switch (b) {
      case 0: put3(0, 0, K, D_pI_pB, 1.0); break;
      case 1: put_rot(1, K, D_pI_qa, qa); put3(1, pc0, K, D_pI_pa, 1.0); break;
      case 2: put_rot(2, K, D_pI_qGLM, qGLM); put3(2, pc0, K, D_pI_pGLM, 1.0); break;
      case 3: put_rot(3, K, D_pI_qGM, qGM); put3(3, pc0, K, D_pI_pGM, 1.0); break;
      case 4: put_rot(4, K, D_pI_qv, qv); put3(4, pc0, K, D_pI_pv, 1.0); break;
      case 5: {
        // d p_C / d q_CI = [R_C_I p_I]x (visual-error-term-inl.h:186)
        double rp[3];
        mat3_vec(cam.R_C_I, pI, rp);
        double I3[9] = {1, 0, 0, 0, 1, 0, 0, 0, 1}, Sk[9];
        skew_right(I3, rp, Sk);
        put_rot(5, Kc, Sk, qCI);
        break;
      }
      case 6: {
        double I3[9] = {1, 0, 0, 0, 1, 0, 0, 0, 1};
        put3(6, 0, Kc, I3, 1.0);
        break;
      }
      case 7: {
        // d kp / d (fu fv cu cv) at the distorted normalized point.
        const double u = (kp[0] - cam.intr[2]) / cam.intr[0], vv = (kp[1] - cam.intr[3]) / cam.intr[1];
        double* J = at(7);
        J[0] = u * sinv; J[1] = 0.0; J[2] = sinv; J[3] = 0.0;
        J[4] = 0.0; J[5] = vv * sinv; J[6] = 0.0; J[7] = sinv;
        break;
      }
      case 8: {
        // d kp / d distortion at the undistorted normalized point (the
        // model's projection before distortion), rows x f.
        double* J = at(8);
        double den = pC[2];
        if (cam.model == kCameraUnifiedProjection)
          den += cam.xi * sqrt(pC[0] * pC[0] + pC[1] * pC[1] + pC[2] * pC[2]);
        const double x = pC[0] / den, y = pC[1] / den;
        double d[8];
        distortion_parameter_jacobian(cam.dist_type, cam.dist, x, y, d);
        for (int k = 0; k < 4; ++k) {
          J[k] = d[k] * cam.intr[0] * sinv;
          J[4 + k] = d[4 + k] * cam.intr[1] * sinv;
        }
        break;
      }
      case 9: {
        // d kp / d xi (camera-unified-projection.cc:176-189).
        double kx[2], jx[6], jxi[2];
        project_unified(cam.xi, cam.dist_type, cam.intr, cam.dist, cam.width, cam.height, pC, kx, jx, jxi);
        at(9)[0] = jxi[0] * sinv;
        at(9)[1] = jxi[1] * sinv;
        break;
      }
    }
  }
}

// ------------------------------------------------------------ launchers

// One launch; with `stop`, that event completes with the kernel. An event tied
// to its kernel's own completion costs a launch under 1 us, one recorded by
// itself 3 us (a packet of its own in the queue).
template <class... P, class... A>
static void launch(hipStream_t s, hipEvent_t stop, void (*kernel)(P...), int grid, int block, A... args) {
  if (stop)
    hipExtLaunchKernelGGL(kernel, dim3(grid), dim3(block), 0, s, nullptr, stop, 0, static_cast<P>(args)...);
  else
    kernel<<<grid, block, 0, s>>>(static_cast<P>(args)...);
}
// The stop event of a launcher that has nothing to launch.
static void launch_nothing(hipStream_t s, hipEvent_t stop) {
  if (stop) (void)hipEventRecord(stop, s);
}

void launch_vertex_prep(hipStream_t s, int32_t P, const double* vert, double* vR) {
  if (P > 0) k_vertex_prep<<<(P + 255) / 256, 256, 0, s>>>(P, vert, vR);
}
void launch_linearize(hipStream_t s, bool jac, int32_t tiles, const DevTopology& t, const double* vert,
                      const double* vR, const double* lm, DevLoss loss, const int32_t* tile_begin, double* obs_rec,
                      double* lm_acc, double* split_part, double* tile_cost, bool f32, hipEvent_t stop) {
  if (tiles <= 0) return launch_nothing(s, stop);
  const auto kernel = jac ? (f32 ? &k_linearize<true, true> : &k_linearize<true, false>) : &k_linearize<false, false>;
  launch(s, stop, kernel, tiles, kObsTile, t, vert, vR, lm, loss, tile_begin, obs_rec, lm_acc, split_part, tile_cost);
}
void launch_split_sum(hipStream_t s, int32_t n, const int32_t* ids, const int32_t* split_tiles,
                      const double* split_part, double* lm_acc) {
  if (n > 0) k_split_sum<<<(n * kLmAcc + 255) / 256, 256, 0, s>>>(n, ids, split_tiles, split_part, lm_acc);
}
void launch_pose_rows(hipStream_t s, const DevTopology& t, const double* vert, const double* vR, const double* lm,
                      const double* obs_rec, const double* lm_acc, double* pose_grad, double* pose_diag,
                      double* pose_jtj, bool f32, hipEvent_t stop) {
  if (t.Pvar <= 0) return launch_nothing(s, stop);
  launch(s, stop, f32 ? &k_pose_rows<true> : &k_pose_rows<false>, t.Pvar, kRowThreads, t, vert, vR, lm, obs_rec,
         lm_acc, pose_grad, pose_diag, pose_jtj);
}
void launch_jacobi_scaling(hipStream_t s, int32_t Pvar, int32_t L, int32_t use, const double* pose_diag,
                           const double* lm_acc, double* pose_scale, double* lm_scale) {
  const int n = std::max(6 * Pvar, 3 * L);
  if (n > 0) k_jacobi_scaling<<<(n + 255) / 256, 256, 0, s>>>(Pvar, L, use, pose_diag, lm_acc, pose_scale, lm_scale);
}
void launch_landmark_prep(hipStream_t s, const DevTopology& t, const double* lm_acc, const double* lm_scale,
                          double inv_mu, double min_diag, double max_diag, double* lm_z, double* lm_anc,
                          int32_t* fail, hipEvent_t stop) {
  if (t.L <= 0) return launch_nothing(s, stop);
  launch(s, stop, &k_landmark_prep, (t.L + 255) / 256, 256, t, lm_acc, lm_scale, inv_mu, min_diag, max_diag, lm_z,
         lm_anc, fail);
}
void launch_schur_factors(hipStream_t s, const DevTopology& t, int32_t n_g, const int32_t* g_row,
                          const int32_t* g_inc_ptr, const int32_t* g_inc, const double* vR, const double* lm,
                          const double* obs_rec, double* gf, double* gk, bool f32, hipEvent_t stop) {
  if (t.Pvar <= 0 || n_g <= 0) return launch_nothing(s, stop);
  launch(s, stop, f32 ? &k_schur_factors<true> : &k_schur_factors<false>, (n_g + 255) / 256, 256, t, n_g, g_row,
         g_inc_ptr, g_inc, vR, lm, obs_rec, gf, gk);
}
bool schur_items_per_wg_supported(int32_t n) { return n == 1 || n == 2 || n == 4 || n == 8; }
void launch_schur_tiles(hipStream_t s, const SchurTilesDev& d, const double* gf, const double* gk,
                        const double* lm_z, const double* lm_anc, double* partial, int32_t items_per_wg,
                        int32_t xcd_map) {
  if (d.n_segs <= 0) return;
  const int wgs = (d.n_segs + items_per_wg - 1) / items_per_wg;
  const int per_xcd = (wgs + 7) / 8;
  const TileArgs ta{d.batches, d.slots, d.batch_off, reinterpret_cast<const uint32_t*>(d.pairs), gf, gk, lm_z, lm_anc};
  k_schur_tiles<<<8 * per_xcd, kTileBlocks, 0, s>>>(d.n_segs, items_per_wg, xcd_map, d.seg_order, d.segs,
                                                     d.seg_thread, ta, partial);
}
void launch_schur_blocks(hipStream_t s, const DevTopology& t, const SchurTilesDev& d, int32_t nub, const int4* ublk,
                         const double* gf, const double* gk, const double* lm_z, const double* lm_anc,
                         const double* vR, const double* pose_scale, const double* pose_diag, const double* pose_jtj,
                         double inv_mu, double min_diag, double max_diag, double* partial, double* S, double* rhs,
                         int32_t items_per_wg, int32_t xcd_map, hipEvent_t stop) {
  if (t.Pvar <= 0 || nub <= 0) return launch_nothing(s, stop);
  launch_schur_tiles(s, d, gf, gk, lm_z, lm_anc, partial, items_per_wg, xcd_map);
  // kWide from 24 slots a block on (MI355X, tiles and this kernel, seven blocks a
  // work-group against one): 165 slots a block 62 and 24 us, 64 slots 107 and 58,
  // 28 slots 114 and 86, 19 slots 145 and 129, 13 slots 166 and 162, 8 slots 232
  // and 240. The two meet near 12; between there and the line the wide form would
  // save up to a tenth.
  const bool wide = d.n_uslot >= 24 * (int64_t)nub;
  launch(s, stop, wide ? &k_schur_finalize<true> : &k_schur_finalize<false>,
         wide ? nub : (nub + kFinalizeGroups - 1) / kFinalizeGroups, 252, t, nub, ublk, d.uslot_ptr, d.uslot, partial,
         vR, pose_scale, pose_diag, pose_jtj, inv_mu, min_diag, max_diag, S, rhs);
}
void launch_landmark_quality(hipStream_t s, const DevTopology& t, const double* vert, const double* vR,
                             const double* lm, int32_t min_observers, double min_angle_deg, double max_dist,
                             double min_dist, double max_reproj_px, uint8_t* good) {
  if (t.L <= 0) return;
  QualityArgs q;
  q.min_observers = min_observers;
  q.pad = 0;
  q.min_angle_deg = min_angle_deg;
  q.max_dist = max_dist;
  q.min_dist = min_dist;
  q.max_reproj2 = max_reproj_px > 0.0 ? max_reproj_px * max_reproj_px : 0.0;
  const int per = 4 * kQualityWaves;
  if (q.max_reproj2 > 0.0)
    k_landmark_quality<true><<<(t.L + per - 1) / per, 64 * kQualityWaves, 0, s>>>(t, vert, vR, lm, q, good);
  else
    k_landmark_quality<false><<<(t.L + per - 1) / per, 64 * kQualityWaves, 0, s>>>(t, vert, vR, lm, q, good);
}
void launch_block_inverse(hipStream_t s, int32_t Pvar, const int32_t* diag_pos, const double* S, double* Minv,
                          int32_t* fail, hipEvent_t stop) {
  if (Pvar <= 0) return launch_nothing(s, stop);
  launch(s, stop, &k_block_inverse, (Pvar + 63) / 64, 64, Pvar, diag_pos, S, Minv, fail);
}

// Part entries: 2 per tile, then 2 per block of 256 split landmarks; returns
// their count.
int32_t launch_back_substitute(hipStream_t s, const DevTopology& t, int32_t tiles, const int32_t* tile_begin,
                               int32_t n_split, const int32_t* split_ids, const double* vR, const double* lm,
                               const double* obs_rec, const double* lm_acc, const double* lm_z, const double* w,
                               double* u, double* part, bool f32, hipEvent_t stop) {
  const int sb = (n_split + 255) / 256;
  double* part_split = part + 2 * (size_t)std::max(tiles, 0);
  if (tiles <= 0 && sb <= 0) launch_nothing(s, stop);
  if (tiles > 0)
    launch(s, sb > 0 ? nullptr : stop, f32 ? &k_back_substitute<true> : &k_back_substitute<false>, tiles, kObsTile, t,
           tile_begin, vR, lm, obs_rec, lm_acc, lm_z, w, u, part);
  if (sb > 0)
    launch(s, stop, f32 ? &k_back_substitute_split<true> : &k_back_substitute_split<false>, sb, 256, t, n_split,
           split_ids, vR, lm, obs_rec, lm_acc, lm_z, w, u, part_split);
  return std::max(tiles, 0) + sb;
}
void launch_step_vertices(hipStream_t s, const DevTopology& t, const double* vert, const double* y,
                          const double* pose_scale, double* w, double* cand_v, double* cand_vR, double* part_w,
                          double* part_x, hipEvent_t stop) {
  if (t.P <= 0) return launch_nothing(s, stop);
  launch(s, stop, &k_step_vertices, (t.P + 255) / 256, 256, t, vert, y, pose_scale, w, cand_v, cand_vR, part_w, part_x);
}
void launch_candidate_landmarks(hipStream_t s, const DevTopology& t, const double* lm, const double* u, double* cand_l,
                                double* part_l, hipEvent_t stop) {
  if (t.L <= 0) return launch_nothing(s, stop);
  launch(s, stop, &k_candidate_landmarks, (t.L + 255) / 256, 256, t, lm, u, cand_l, part_l);
}
void launch_gradient_norm(hipStream_t s, const DevTopology& t, const double* vert, const double* pose_grad,
                          const double* lm_acc, double* part) {
  const int n = t.Pvar + t.L;
  if (n > 0) k_gradient_norm<<<(n + 255) / 256, 256, 0, s>>>(t, vert, pose_grad, lm_acc, part);
}
void launch_reduce(hipStream_t s, int32_t n, int32_t stride, int32_t offset, bool is_max, const double* parts,
                   double* out) {
  k_reduce<<<1, 256, 0, s>>>(n, stride, offset, is_max ? 1 : 0, parts, out);
}
bool launch_reduce_many(hipStream_t s, const ReduceBatch& batch, hipEvent_t stop) {
  if (batch.count < 1 || batch.count > kMaxReduceBatch) return false;  // caller reports it; nothing launched
  launch(s, stop, &k_reduce_many, batch.count, 256, batch);
  return true;
}
// ------------------------------------------------------------ calibration

// Normal equations of the camera calibration blocks when vertices and
// landmarks are constant. Per camera, over the 15 tangent columns
// [q_CI (3) | C_p_CI (3) | fu fv cu cv | distortion (4) | xi], of the
// robust-corrected residuals (ceres Corrector, as k_linearize):
//   entries 0..119  J'J upper triangle (row-major over a <= b),
//   entries 120..134 J'r, entry 135 the cost 0.5 rho.
// One work-group per tile of 256 observations (landmark-sorted order) writes
// its partial sums per camera; k_calib_sum adds the tiles in order.
// `rec` is the tangent k_evaluate_full record of every observation (caller
// order, stride kCalibStride) and `res` its residuals (caller order).
constexpr int kCalibEntries = 136;
constexpr int kCalibStride = 84;  // 2 x (3 + 6 + 6 + 6 + 6 + 3 + 3 + 4 + 4 + 1)

__global__ __launch_bounds__(256) void k_calib_partials(DevTopology t, const int32_t* __restrict__ perm,
                                                        const double* __restrict__ res,
                                                        const double* __restrict__ rec, DevLoss loss,
                                                        int32_t cost_only, double* __restrict__ partial) {
  __shared__ double lds4[4];
  const int o = blockIdx.x * 256 + threadIdx.x;
  int cam = -1;
  double J[30], r[2] = {0.0, 0.0}, cost = 0.0;
  for (int k = 0; k < 30; ++k) J[k] = 0.0;
  if (o < t.N) {
    const int32_t meta = t.obs_meta[o];
    const int32_t l = t.obs_landmark[o];
    if (t.lm_flags[l] & kLmActive) {
      cam = obs_camera(meta);
      const int32_t oo = perm[o];
      const double r0 = res[2 * oo], r1 = res[2 * oo + 1];
      const double s2 = r0 * r0 + r1 * r1;
      double rho[3];
      robust_loss(loss.type, loss_scale(loss, obs_type(meta), t.obs_sinv[o]), s2, rho);
      cost = 0.5 * rho[0];
      if (!cost_only) {
        // Tangent blocks 5 (q_CI), 6 (p_CI), 7 (intrinsics), 8 (distortion), 9 (xi).
        const double* R = rec + (size_t)oo * kCalibStride;
        const int off[5] = {54, 60, 66, 74, 82}, wid[5] = {3, 3, 4, 4, 1}, col[5] = {0, 3, 6, 10, 14};
        for (int b = 0; b < 5; ++b)
          for (int c = 0; c < wid[b]; ++c) {
            J[col[b] + c] = R[off[b] + c];
            J[15 + col[b] + c] = R[off[b] + wid[b] + c];
          }
        const double sq1 = sqrt(rho[1]);
        double rs = sq1, asq = 0.0;
        if (s2 > 0.0 && rho[2] > 0.0) {
          const double alpha = 1.0 - sqrt(1.0 + 2.0 * s2 * rho[2] / rho[1]);
          rs = sq1 / (1.0 - alpha);
          asq = alpha / s2;
        }
        for (int c = 0; c < 15; ++c) {
          const double rtj = J[c] * r0 + J[15 + c] * r1;
          J[c] = sq1 * (J[c] - asq * r0 * rtj);
          J[15 + c] = sq1 * (J[15 + c] - asq * r1 * rtj);
        }
        r[0] = r0 * rs;
        r[1] = r1 * rs;
      }
    }
  }
  for (int c = 0; c < t.C; ++c) {
    double* out = partial + ((size_t)blockIdx.x * t.C + c) * kCalibEntries;
    const bool mine = cam == c;
    if (!cost_only) {
      // Fully unrolled so that J stays in registers.
#pragma unroll
      for (int a = 0; a < 15; ++a)
#pragma unroll
        for (int b = a; b < 15; ++b) {
          const double v = block_sum256(mine ? J[a] * J[b] + J[15 + a] * J[15 + b] : 0.0, lds4);
          if (threadIdx.x == 0) out[a * 15 - a * (a - 1) / 2 + (b - a)] = v;
        }
#pragma unroll
      for (int a = 0; a < 15; ++a) {
        const double v = block_sum256(mine ? J[a] * r[0] + J[15 + a] * r[1] : 0.0, lds4);
        if (threadIdx.x == 0) out[120 + a] = v;
      }
    }
    const double v = block_sum256(mine ? cost : 0.0, lds4);
    if (threadIdx.x == 0) out[135] = v;
  }
}

// out[c][e] = sum over tiles of the partials, in tile order.
__global__ void k_calib_sum(int32_t tiles, int32_t C, const double* __restrict__ partial, double* __restrict__ out) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= C * kCalibEntries) return;
  const int c = k / kCalibEntries, e = k % kCalibEntries;
  double v = 0.0;
  for (int tile = 0; tile < tiles; ++tile) v += partial[((size_t)tile * C + c) * kCalibEntries + e];
  out[k] = v;
}

int32_t calib_entries() { return kCalibEntries; }
int32_t calib_record_stride() { return kCalibStride; }
void launch_calib_normal(hipStream_t s, const DevTopology& t, const int32_t* perm, const double* res,
                         const double* rec, DevLoss loss, bool cost_only, double* partial, double* out) {
  if (t.N <= 0 || t.C <= 0) return;
  const int tiles = (t.N + 255) / 256;
  k_calib_partials<<<tiles, 256, 0, s>>>(t, perm, res, rec, loss, cost_only ? 1 : 0, partial);
  const int n = t.C * kCalibEntries;
  k_calib_sum<<<(n + 255) / 256, 256, 0, s>>>(tiles, t.C, partial, out);
}

void launch_evaluate_full(hipStream_t s, const DevTopology& t, const double* vert, const double* vR, const double* lm,
                          const double* baseframes, const double* cam_q, bool tangent, const int32_t* perm,
                          double* res, const EvalOut& jout, bool want_jac) {
  if (t.N > 0)
    k_evaluate_full<<<(t.N + 255) / 256, 256, 0, s>>>(t, vert, vR, lm, baseframes, cam_q, tangent ? 1 : 0, perm, res,
                                                      jout, want_jac ? 1 : 0);
}

// ------------------------------------------------------------ outlier rejection

// p_C of observation o at the current state: the frame chain of
// eval_observation without the Jacobians.
__device__ inline void obs_point_camera(const DevTopology& t, int o, const double* __restrict__ vert,
                                        const double* __restrict__ vR, const double* __restrict__ lm,
                                        double* pC) {
  const int32_t meta = t.obs_meta[o];
  const int32_t type = obs_type(meta);
  const DevCamera& cam = t.cams[obs_camera(meta)];
  const int32_t l = t.obs_landmark[o];
  const int32_t v = t.obs_vertex[o];
  const double* pB = lm + 3 * l;
  double pI[3];
  if (type == kTypeKeyframe) {
    pI[0] = pB[0]; pI[1] = pB[1]; pI[2] = pB[2];
  } else {
    const int32_t a = t.lm_anchor[l];
    double pM[3];
    mat3t_vec(vR + 12 * a, pB, pM);
    for (int i = 0; i < 3; ++i) pM[i] += vert[7 * a + 4 + i];
    if (type == kTypeGlobal) {
      const double* TL = t.mission_T + 12 * t.vertex_mission[a];
      const double* TM = t.mission_T + 12 * t.vertex_mission[v];
      double pG[3], d[3];
      mat3_vec(TL, pM, pG);
      for (int i = 0; i < 3; ++i) d[i] = pG[i] + TL[9 + i] - TM[9 + i];
      mat3t_vec(TM, d, pM);
    }
    const double dm[3] = {pM[0] - vert[7 * v + 4], pM[1] - vert[7 * v + 5], pM[2] - vert[7 * v + 6]};
    mat3_vec(vR + 12 * v, dm, pI);
  }
  mat3_vec(cam.R_C_I, pI, pC);
  for (int i = 0; i < 3; ++i) pC[i] += cam.p_C_I[i];
}

// findOutlierLandmarks (outlier-rejection-solver.cc:28-103) over the active
// landmarks, one wave per landmark: outlier when any observation has
// p_C.z <= 0, or (use_reproj) a squared pixel error above max_reproj2, statuses
// other than visible / outside the image counting as infinite
// (landmark-quality-metrics.cc:57-73). An outlier is deactivated in place
// (kLmActive cleared: its observations then contribute nothing to the cost,
// the landmark sums, S or the step) and bad[l] = 1.
__global__ __launch_bounds__(64) void k_find_outliers(DevTopology t, const double* __restrict__ vert,
                                                      const double* __restrict__ vR, const double* __restrict__ lm,
                                                      int32_t use_reproj, double max_reproj2,
                                                      uint32_t* __restrict__ lm_flags, uint8_t* __restrict__ bad) {
  const int l = blockIdx.x, lane = threadIdx.x;
  const uint32_t flags = lm_flags[l];
  int out = 0;
  if (flags & kLmActive) {
    for (int o = t.lm_begin[l] + lane; o < t.lm_begin[l + 1]; o += 64) {
      double pC[3];
      obs_point_camera(t, o, vert, vR, lm, pC);
      if (pC[2] <= 0.0) { out = 1; continue; }
      if (use_reproj) {
        const DevCamera& cam = t.cams[obs_camera(t.obs_meta[o])];
        double kp[2], jp[6];
        const int st = project_camera(cam.model, cam.xi, cam.dist_type, cam.intr, cam.dist, cam.width, cam.height,
                                      pC, kp, jp);
        double e2 = 1.7976931348623157e308;
        if (st == kVisible || st == kOutsideImage) {
          const double du = kp[0] - t.obs_kp[2 * o], dv = kp[1] - t.obs_kp[2 * o + 1];
          e2 = du * du + dv * dv;
        }
        if (e2 > max_reproj2) out = 1;
      }
    }
  }
  out = __any(out);
  if (lane == 0) {
    bad[l] = (uint8_t)out;
    if (out) lm_flags[l] = flags & ~kLmActive;
  }
}
void launch_find_outliers(hipStream_t s, const DevTopology& t, const double* vert, const double* vR, const double* lm,
                          int32_t use_reproj, double max_reproj2, uint32_t* lm_flags, uint8_t* bad) {
  if (t.L > 0) k_find_outliers<<<t.L, 64, 0, s>>>(t, vert, vR, lm, use_reproj, max_reproj2, lm_flags, bad);
}

// ------------------------------------------------------------ measurement

// Copy of n 16-byte words (the bandwidth reference): each thread moves four
// words of one 4 x 256-word chunk per step (four loads in flight), chunks
// assigned grid-stride; the tail (n % 1024) word by word.
__global__ __launch_bounds__(256) void k_stream_copy(int64_t n, const int4* __restrict__ src, int4* __restrict__ dst) {
  const int64_t chunks = n / 1024;
  for (int64_t c = blockIdx.x; c < chunks; c += gridDim.x) {
    const int64_t b = c * 1024 + threadIdx.x;
    const int4 v0 = src[b], v1 = src[b + 256], v2 = src[b + 512], v3 = src[b + 768];
    dst[b] = v0; dst[b + 256] = v1; dst[b + 512] = v2; dst[b + 768] = v3;
  }
  for (int64_t i = chunks * 1024 + (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    dst[i] = src[i];
}
void launch_stream_copy(hipStream_t s, int64_t words, const void* src, void* dst) {
  if (words > 0)
    k_stream_copy<<<2048, 256, 0, s>>>(words, static_cast<const int4*>(src), static_cast<int4*>(dst));
}

}  // namespace mlba
