// ba_host.hip -- C ABI of libmaplab_ba.so: problem upload and topology, the
// Levenberg-Marquardt trust-region loop over the device kernels, the chunked
// outlier-rejection driver, and the batched Evaluate entry point.
//
// The LM loop restates ceres::TrustRegionMinimizer with the
// LevenbergMarquardtStrategy as configured by maplab
// (algorithms/map-optimization/include/map-optimization/solver-options.h:26-74):
// Jacobi column scaling fixed at the first linearization, LM diagonal
// clamp(diag(J'J)) / radius, step acceptance at relative decrease > 1e-3,
// radius update radius / max(1/3, 1 - (2 rho - 1)^3) on success and
// radius / decrease_factor (doubling) on failure, and the function,
// parameter, gradient and radius tolerances.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <array>
#include <chrono>
#include <cmath>
#include <cstring>
#include <new>
#include <atomic>
#include <mutex>
#include <string>
#include <thread>
#include <vector>

#include "../../include/maplab_ba.h"
#include "ba_pcg.h"
#include "ba_learned.h"
#include "ba_ritz.h"
#include "ba_tiles.h"
#include "../../include/maplab_ba_learned.h"
#include "ba_device.h"
#include "ba_math.h"

namespace mlba {
void launch_vertex_prep(hipStream_t s, int32_t P, const double* vert, double* vR);
void launch_linearize(hipStream_t s, bool jac, int32_t tiles, const DevTopology& t, const double* vert,
                      const double* vR, const double* lm, DevLoss loss, const int32_t* tile_begin, double* obs_rec,
                      double* lm_acc, double* split_part, double* tile_cost, bool f32 = false,
                      hipEvent_t stop = nullptr);
void launch_split_sum(hipStream_t s, int32_t n, const int32_t* ids, const int32_t* split_tiles,
                      const double* split_part, double* lm_acc);
void launch_pose_rows(hipStream_t s, const DevTopology& t, const double* vert, const double* vR, const double* lm,
                      const double* obs_rec, const double* lm_acc, double* pose_grad, double* pose_diag,
                      double* pose_jtj, bool f32 = false, hipEvent_t stop = nullptr);
void launch_jacobi_scaling(hipStream_t s, int32_t Pvar, int32_t L, int32_t use, const double* pose_diag,
                           const double* lm_acc, double* pose_scale, double* lm_scale);
void launch_landmark_prep(hipStream_t s, const DevTopology& t, const double* lm_acc, const double* lm_scale,
                          double inv_mu, double min_diag, double max_diag, double* lm_z, double* lm_anc,
                          int32_t* fail, hipEvent_t stop = nullptr);
void launch_schur_factors(hipStream_t s, const DevTopology& t, int32_t n_g, const int32_t* g_row,
                          const int32_t* g_inc_ptr, const int32_t* g_inc, const double* vR, const double* lm,
                          const double* obs_rec, double* gf, double* gk, bool f32 = false, hipEvent_t stop = nullptr);
void launch_schur_blocks(hipStream_t s, const DevTopology& t, const SchurTilesDev& d, int32_t nub, const int4* ublk,
                         const double* gf, const double* gk, const double* lm_z, const double* lm_anc,
                         const double* vR, const double* pose_scale, const double* pose_diag, const double* pose_jtj,
                         double inv_mu, double min_diag, double max_diag, double* partial, double* S, double* rhs,
                         int32_t items_per_wg, int32_t xcd_map, hipEvent_t stop = nullptr);
void launch_schur_tiles(hipStream_t s, const SchurTilesDev& d, const double* gf, const double* gk,
                        const double* lm_z, const double* lm_anc, double* partial, int32_t items_per_wg,
                        int32_t xcd_map);
bool schur_items_per_wg_supported(int32_t n);
int32_t calib_entries();
int32_t calib_record_stride();
void launch_calib_normal(hipStream_t s, const DevTopology& t, const int32_t* perm, const double* res,
                         const double* rec, DevLoss loss, bool cost_only, double* partial, double* out);
void launch_landmark_quality(hipStream_t s, const DevTopology& t, const double* vert, const double* vR,
                             const double* lm, int32_t min_observers, double min_angle_deg, double max_dist,
                             double min_dist, double max_reproj_px, uint8_t* good);
void launch_block_inverse(hipStream_t s, int32_t Pvar, const int32_t* diag_pos, const double* S, double* Minv,
                          int32_t* fail, hipEvent_t stop = nullptr);
int32_t pcg_max_lanczos();
int32_t launch_back_substitute(hipStream_t s, const DevTopology& t, int32_t tiles, const int32_t* tile_begin,
                               int32_t n_split, const int32_t* split_ids, const double* vR, const double* lm,
                               const double* obs_rec, const double* lm_acc, const double* lm_z, const double* w,
                               double* u, double* part, bool f32 = false, hipEvent_t stop = nullptr);
void launch_step_vertices(hipStream_t s, const DevTopology& t, const double* vert, const double* y,
                          const double* pose_scale, double* w, double* cand_v, double* cand_vR, double* part_w,
                          double* part_x, hipEvent_t stop = nullptr);
void launch_candidate_landmarks(hipStream_t s, const DevTopology& t, const double* lm, const double* u, double* cand_l,
                                double* part_l, hipEvent_t stop = nullptr);
void launch_gradient_norm(hipStream_t s, const DevTopology& t, const double* vert, const double* pose_grad,
                          const double* lm_acc, double* part);
bool launch_reduce_many(hipStream_t s, const ReduceBatch& batch, hipEvent_t stop = nullptr);
void launch_stream_copy(hipStream_t s, int64_t words, const void* src, void* dst);
void launch_find_outliers(hipStream_t s, const DevTopology& t, const double* vert, const double* vR, const double* lm,
                          int32_t use_reproj, double max_reproj2, uint32_t* lm_flags, uint8_t* bad);
void launch_reduce(hipStream_t s, int32_t n, int32_t stride, int32_t offset, bool is_max, const double* parts,
                   double* out);
void launch_evaluate_full(hipStream_t s, const DevTopology& t, const double* vert, const double* vR, const double* lm,
                          const double* baseframes, const double* cam_q, bool tangent, const int32_t* perm,
                          double* res, const EvalOut& jout, bool want_jac);
}  // namespace mlba

using namespace mlba;

namespace {

thread_local std::string g_create_error;

// PCG iterations between host convergence polls. A solve's first poll comes
// after the last similar solve's iteration count (with or without recycled
// columns), then every kPcgPollAfter iterations: successive LM solves take
// similar counts, a poll costs a host round trip (≈20 µs) and an iteration
// past convergence two early-exit launches (≈10 µs).
constexpr int32_t kPcgPoll = 16, kPcgPollAfter = 4;

// Default Schur dispatch schedule: largest segments first, one segment per
// work-group, no XCD remapping.
constexpr int kItemBandRows = 0, kItemsPerWg = 1, kItemXcd = 0;

// Pinned host buffer of the recycling (R = kPcgMaxRitz): the solve's
// coefficients (2 x 64), the tridiagonal's eigenvectors (64 x R), the Gram
// matrices (2 x 2R x 2R) and the merge coefficients (2R x R).
constexpr size_t kRitzCoefOff = 2 * 64, kRitzGramOff = kRitzCoefOff + 64 * kPcgMaxRitz;
constexpr size_t kRitzMergeOff = kRitzGramOff + 2 * (2 * kPcgMaxRitz) * (2 * kPcgMaxRitz);
constexpr size_t kRitzPinned = kRitzMergeOff + 2 * kPcgMaxRitz * kPcgMaxRitz;

double now_s() {
  return std::chrono::duration<double>(std::chrono::steady_clock::now().time_since_epoch()).count();
}

// A device allocation that frees itself.
template <typename T>
struct DBuf {
  T* p = nullptr;
  size_t n = 0;
  DBuf() = default;
  DBuf(const DBuf&) = delete;
  DBuf& operator=(const DBuf&) = delete;
  ~DBuf() { release(); }
  void release() {
    if (p) (void)hipFree(p);
    p = nullptr;
    n = 0;
  }
  bool alloc(size_t count) {
    if (count <= n && p) return true;
    release();
    const size_t bytes = std::max<size_t>(1, count) * sizeof(T);
    if (hipMalloc(&p, bytes) != hipSuccess) { p = nullptr; return false; }
    n = std::max<size_t>(1, count);
    return true;
  }
};

// Scalar slots of the reduction output array.
enum Slot { kCost = 0, kFixed, kMcc, kUU, kWW, kXV, kXL, kCandCost, kCandFixed, kGradMax, kFail, kPcgIters, kNumSlots };

}  // namespace

struct mlba_handle {
  std::string err;
  hipStream_t stream = nullptr;
  int device = 0;                       // device current at mlba_create (the stream's)
  int N = 0, L = 0, P = 0, C = 0, M = 0;
  // Host topology.
  std::vector<int32_t> perm;            // sorted -> caller observation index
  std::vector<int32_t> s_landmark, s_vertex, s_camera, s_type;
  std::vector<int32_t> lm_begin, lm_anchor, vertex_mission;
  std::vector<uint8_t> lm_active, lm_const, vertex_const;
  std::vector<double> h_baseframes, h_cam_q;
  std::vector<DevCamera> h_cams;        // host mirror of the device cameras
  // Derived per topology build.
  int32_t Pvar = 0, tiles = 0, nnzb = 0, n_inc = 0, n_split = 0, max_row_blocks = 0;
  int64_t schur_pairs = 0;              // incidence pairs summed into the upper blocks
  int32_t n_upper = 0;                  // upper-triangle blocks of S
  int32_t n_g = 0, n_segs = 0, nbands = 0;  // factor blocks, Schur work items (tile segments), tile bands
  int64_t n_visits = 0, n_batches = 0, n_tpairs = 0, n_staged = 0;
  // Device memory.
  DBuf<double> obs_kp, obs_sinv, obs_rec;
  DBuf<int32_t> obs_vertex, obs_meta, obs_landmark, perm_d;
  DBuf<int32_t> lm_begin_d, lm_anchor_d, split_ids, split_tiles;  // split landmarks: id; first tile, tile count
  DBuf<double> split_part;                                         // per-tile sums of split landmarks
  // Learned preconditioner (ba_learned.h): per block position of S its row,
  // transposed position and shared observation pairs; set-up, network and
  // PCG buffers (allocated on first use).
  DBuf<int32_t> lp_pos_row, lp_tpos, lp_shared;
  int32_t lp_max_lower_deg = 0;
  DBuf<double> lp_linv, lp_t, lp_u, lp_part;
  DBuf<float> lp_shat, lp_snorm, lp_kmat, lp_t2, lp_trace, lp_nf, lp_ef, lp_theta;
  DBuf<char> lp_state;
  void* lp_state_host = nullptr;
  DBuf<float> lp_params, lp_norm;       // network parameters and feature (mean, std)
  bool lp_model = false;
  GnnWorkspace* lp_ws = nullptr;
  int32_t lp_ws_nodes = -1, lp_ws_slots = -1;
  mlba_preconditioner_stats lp_stats{};
  DBuf<uint32_t> lm_flags;
  DBuf<uint8_t> lm_bad;                 // outlier flags of the last rejection pass
  DBuf<double> lm, lm_cand, lm_acc, lm_scale, lm_z, lm_anc, lm_u;
  DBuf<double> vert, vert_cand, vR, vR_cand;
  DBuf<int32_t> vertex_mission_d, vertex_var, var_vertex;
  DBuf<DevCamera> cams, cams_cand;
  DBuf<double> cam_q_cand, calib_res, calib_rec, calib_part, calib_out;
  DBuf<double> mission_T, baseframes, cam_q;
  DBuf<int32_t> tile_begin;
  DBuf<double> tile_cost, tile_cost2;
  DBuf<int32_t> row_ptr, col_var, diag_pos, inc_ptr, inc, obs_col;
  DBuf<int4> ublk;                      // upper block (position of S_ij, of S_ji, i, j)
  DBuf<int32_t> g_row, g_inc_ptr, g_inc;  // factor blocks (ba_tiles.h)
  DBuf<int4> t_batches, t_segs;
  DBuf<int2> t_slots;
  DBuf<uint32_t> t_seg_thread;
  DBuf<uint16_t> t_batch_off, t_pairs;
  DBuf<int32_t> t_uslot_ptr, t_uslot;   // partial slots of every upper block
  DBuf<int32_t> t_seg_order;            // segments in dispatch order
  DBuf<double> gf, gk;                  // per-linearization factor blocks (P, p) and their k
  DBuf<double> schur_partial;           // kTilePartial per segment
  std::vector<int4> h_segs;             // host copy of the segments (dispatch order)
  // Dispatch schedule of k_schur_tiles (mlba_autotune): tile rows per band of
  // the dispatch order (0: tile order), segments (work items) per
  // work-group, XCD-contiguous work-group mapping. It changes no result.
  int32_t sched_band = kItemBandRows, sched_waves = kItemsPerWg, sched_xcd = kItemXcd, sched_pcg = 0;
  // Jacobian storage of the observation records for the current solve
  // (mlba_options.jacobian_fp32): FP32 Jacobians, FP64 residuals.
  bool f32_jac = false;
  DBuf<int32_t> hat_node, node_range, grp_lo, blk_hat, blk_rng;
  std::vector<int32_t> h_row_ptr, h_col_var;  // host copy of the S block structure
  int32_t grp_width = 0;                // hat columns of the per-group SW window
  DBuf<double> hat_w, blk_w, defl_SR, defl_E, defl_Einv, defl_y, defl_cden, pcg_part2, pcg_step;
  int32_t hat_K = -1;  // coarse nodes of the current hat basis
  // Iterations of the last solve without and with recycled columns: the
  // length of the next such solve's first batch.
  int32_t pcg_last_iters[2] = {0, 0};
  // Recycled deflation columns: ritz[ritz_cur] holds ritz_nr of them; the
  // other buffer receives the merged set. ritz_Zh / ritz_coef keep the
  // Lanczos vectors and coefficients of the last solve.
  DBuf<double> ritz[2], ritz_new, ritz_snew, ritz_Zh, ritz_coef, ritz_small;
  int32_t ritz_cur = 0, ritz_nr = 0, ritz_zcap = 0;
  // Recycling runs in three phases that overlap device work: after a solve
  // the coefficients are copied (stage 1); while the step's back-substitution
  // and cost run, the host takes the tridiagonal's eigenvectors and queues
  // the Ritz kernels and the Gram download (stage 2); before the next solve
  // the host solves the small merge problem and queues the merge (stage 0).
  int32_t ritz_stage = 0, ritz_m = 0, ritz_r = 0;
  double* ritz_pinned = nullptr;  // pinned: coefficients, Y, Gram matrices, merge coefficients
  hipEvent_t ritz_ev_coef = nullptr, ritz_ev_ab = nullptr;
  DBuf<double> S, rhs, pose_grad, pose_diag, pose_jtj, pose_scale, w, Minv;
  DBuf<double> px, pr, pz, pp, pp2, pq, pcg_part, parts_a, parts_b, parts_c, parts_l, parts_v, parts_w, parts_g;
  DBuf<double> scal;
  DBuf<int32_t> fail;
  DBuf<char> pcg_state;
  void* pcg_host = nullptr;
  double* scal_host = nullptr;  // pinned: kNumSlots scalars
  hipEvent_t scal_ev = nullptr;
  DevTopology topo{};
  SchurTilesDev tdev{};
  bool topology_ok = false;  // topo and tdev describe the current active landmarks
  // Event pairs bracketing kernels inside the LM loop (kernel id, start, end).
  std::vector<hipEvent_t> ev_pool;
  std::vector<std::pair<int, std::pair<hipEvent_t, hipEvent_t>>> ev_pending;
  size_t ev_next = 0;
  mlba_summary* ev_summary = nullptr;

  ~mlba_handle() {
    if (ritz_pinned) (void)hipHostFree(ritz_pinned);
    if (ritz_ev_coef) (void)hipEventDestroy(ritz_ev_coef);
    if (ritz_ev_ab) (void)hipEventDestroy(ritz_ev_ab);
    for (hipEvent_t e : ev_pool) (void)hipEventDestroy(e);
    if (pcg_host) (void)hipHostFree(pcg_host);
    if (lp_state_host) (void)hipHostFree(lp_state_host);
    if (lp_ws) gnn_workspace_destroy(lp_ws);
    if (scal_host) (void)hipHostFree(scal_host);
    if (scal_ev) (void)hipEventDestroy(scal_ev);
    if (stream) (void)hipStreamDestroy(stream);
  }
};

namespace {

int set_err(mlba_handle* h, int code, const std::string& msg) {
  if (h) h->err = msg; else g_create_error = msg;
  return code;
}

// For the catch blocks of the C entry points: host memory ran out, so the
// message may not fit either.
int host_out_of_memory(mlba_handle* h) noexcept {
  try {
    return set_err(h, MLBA_ENOMEM, "host allocation failed");
  } catch (...) {
    return MLBA_ENOMEM;
  }
}

#define HIP_OK(expr)                                                                  \
  do {                                                                                \
    hipError_t e_ = (expr);                                                           \
    if (e_ != hipSuccess)                                                             \
      return set_err(h, MLBA_EDEVICE, std::string(#expr) + ": " + hipGetErrorString(e_)); \
  } while (0)

template <typename T>
int upload(mlba_handle* h, DBuf<T>& b, const T* src, size_t count) {
  if (!b.alloc(count)) return set_err(h, MLBA_ENOMEM, "device allocation failed");
  if (count) HIP_OK(hipMemcpyAsync(b.p, src, count * sizeof(T), hipMemcpyHostToDevice, h->stream));
  return MLBA_OK;
}

bool valid_quaternion(const double* q) {
  const double n2 = q[0] * q[0] + q[1] * q[1] + q[2] * q[2] + q[3] * q[3];
  return std::isfinite(n2) && std::fabs(n2 - 1.0) < 2e-5 && q[3] >= 0.0;
}

// Upload the Schur work items (tile segments) in the dispatch order of the
// current schedule: bands of sched_band tile rows, each band swept by tile
// column J, so that the band's factor blocks (staged again by every tile of
// the band) are reused from L2; sched_band 0: the segments with the most
// batches first (the short ones fill the end of the launch). Partial slots
// are the segment indices; the order changes no result.
int upload_item_order(mlba_handle* h) {
  std::vector<int32_t> ord(h->h_segs.size());
  for (size_t k = 0; k < ord.size(); ++k) ord[k] = (int32_t)k;
  const int band = h->sched_band;
  if (band == 0)
    std::stable_sort(ord.begin(), ord.end(), [&](int32_t a, int32_t b) {
      return h->h_segs[a].y - h->h_segs[a].x > h->h_segs[b].y - h->h_segs[b].x;
    });
  if (band > 0)
    std::stable_sort(ord.begin(), ord.end(), [&](int32_t a, int32_t b) {
      const int4 ra = h->h_segs[a], rb = h->h_segs[b];
      const int ba = ra.z / band, bb = rb.z / band;
      if (ba != bb) return ba < bb;
      if (ra.w != rb.w) return ra.w < rb.w;
      return ra.z < rb.z;
    });
  int rc = upload(h, h->t_seg_order, ord.data(), ord.size());
  if (rc) return rc;
  // The host vector is released when the call returns: wait for the copy.
  HIP_OK(hipStreamSynchronize(h->stream));
  return MLBA_OK;
}

// Build the observation / landmark / vertex topology and the reduced camera
// system structure for the current active landmark set, and upload it. A
// handle whose last build failed holds a part of each of two structures and
// runs nothing (check_topology) until a build succeeds.
int build_topology(mlba_handle* h) {
  h->topology_ok = false;
  const int N = h->N, L = h->L, P = h->P;
  // Error type per sorted observation (optimization-terms-addition.cc:68-78).
  // Variable vertices: non-constant and in an active pose-coupled residual.
  std::vector<uint8_t> used(P, 0), lm_coupled(L, 0);
  for (int o = 0; o < N; ++o) {
    const int l = h->s_landmark[o];
    if (!h->lm_active[l] || h->s_type[o] == kTypeKeyframe) continue;
    used[h->s_vertex[o]] = 1;
    used[h->lm_anchor[l]] = 1;
    lm_coupled[l] = 1;
  }
  std::vector<int32_t> vertex_var(P, -1), var_vertex;
  for (int v = 0; v < P; ++v)
    if (used[v] && !h->vertex_const[v]) { vertex_var[v] = (int32_t)var_vertex.size(); var_vertex.push_back(v); }
  const int Pvar = (int)var_vertex.size();
  h->Pvar = Pvar;
  // Tiles of whole landmarks, <= kObsTile observations each.
  std::vector<int32_t> tile_begin{0}, split;
  std::vector<uint32_t> flags(L, 0);
  {
    int cur = 0;
    for (int l = 0; l < L; ++l) {
      const int n = h->lm_begin[l + 1] - h->lm_begin[l];
      if (n > kObsTile) {
        if (h->lm_begin[l] > cur) tile_begin.push_back(h->lm_begin[l]);
        for (int k = kObsTile; k < n; k += kObsTile) tile_begin.push_back(h->lm_begin[l] + k);
        tile_begin.push_back(h->lm_begin[l + 1]);
        cur = h->lm_begin[l + 1];
        flags[l] |= kLmSplit;
        split.push_back(l);
      } else if (h->lm_begin[l + 1] - cur > kObsTile) {
        tile_begin.push_back(h->lm_begin[l]);
        cur = h->lm_begin[l];
      }
    }
    if (tile_begin.back() != N) tile_begin.push_back(N);
    // Remove empty tiles.
    tile_begin.erase(std::unique(tile_begin.begin(), tile_begin.end()), tile_begin.end());
  }
  // The tiles of a split landmark: consecutive, the first starting at its
  // first observation.
  std::vector<int32_t> split_tiles;
  for (int l : split) {
    const auto it = std::lower_bound(tile_begin.begin(), tile_begin.end(), h->lm_begin[l]);
    const int n = h->lm_begin[l + 1] - h->lm_begin[l];
    split_tiles.push_back((int32_t)(it - tile_begin.begin()));
    split_tiles.push_back((n + kObsTile - 1) / kObsTile);
  }
  h->tiles = (int32_t)tile_begin.size() - 1;
  h->n_split = (int32_t)split.size();
  for (int l = 0; l < L; ++l) {
    if (h->lm_active[l]) flags[l] |= kLmActive;
    if (h->lm_const[l]) flags[l] |= kLmConstant;
    if (h->lm_active[l] && lm_coupled[l] && vertex_var[h->lm_anchor[l]] >= 0) flags[l] |= kLmAnchorVar;
  }
  std::vector<int32_t> meta(N);
  for (int o = 0; o < N; ++o) {
    const int type = h->s_type[o];
    const bool ov = type != kTypeKeyframe && vertex_var[h->s_vertex[o]] >= 0;
    meta[o] = type | (ov ? 4 : 0) | (h->lm_active[h->s_landmark[o]] ? 8 : 0) | (h->s_camera[o] << 8);
  }
  // Incidences of each variable vertex row.
  std::vector<int32_t> inc_ptr(Pvar + 1, 0), inc;
  {
    std::vector<int32_t> cnt(Pvar, 0);
    for (int o = 0; o < N; ++o) {
      const int l = h->s_landmark[o];
      if (!h->lm_active[l] || !(meta[o] & 4)) continue;
      cnt[vertex_var[h->s_vertex[o]]]++;
    }
    for (int l = 0; l < L; ++l)
      if (flags[l] & kLmAnchorVar) cnt[vertex_var[h->lm_anchor[l]]]++;
    for (int i = 0; i < Pvar; ++i) inc_ptr[i + 1] = inc_ptr[i] + cnt[i];
    inc.resize(inc_ptr[Pvar]);
    std::vector<int32_t> fill(inc_ptr.begin(), inc_ptr.end() - 1);
    for (int o = 0; o < N; ++o) {
      const int l = h->s_landmark[o];
      if (!h->lm_active[l] || !(meta[o] & 4)) continue;
      inc[fill[vertex_var[h->s_vertex[o]]]++] = o;
    }
    for (int l = 0; l < L; ++l)
      if (flags[l] & kLmAnchorVar) inc[fill[vertex_var[h->lm_anchor[l]]]++] = -1 - l;
  }
  h->n_inc = (int32_t)inc.size();
  // Factor blocks and the work decomposition of the sums of S (ba_tiles.h).
  SchurTiles st;
  {
    std::string terr;
    if (!build_schur_tiles(Pvar, L, inc_ptr.data(), inc.data(), h->s_landmark.data(), &st, &terr))
      return set_err(h, MLBA_ENOMEM, terr);
  }
  // Block structure of S, the incidence pairs of every upper block.
  SchurRows sr;
  {
    std::string terr;
    if (!build_schur_rows(Pvar, L, st, &sr, &terr)) return set_err(h, MLBA_ENOMEM, terr);
  }
  const std::vector<int32_t>&row_ptr = sr.row_ptr, &col_var = sr.col, &diag_pos = sr.diag_pos, &upair = sr.upper_pairs;
  h->max_row_blocks = sr.max_row_blocks;
  h->nnzb = (int32_t)col_var.size();
  h->hat_K = -1;
  h->pcg_last_iters[0] = h->pcg_last_iters[1] = 0;
  h->ritz_nr = 0;
  h->ritz_stage = 0;
  h->h_row_ptr = row_ptr;
  h->h_col_var = col_var;
  // Upper blocks of S (row i, column j >= i, in row order).
  std::vector<int4> ublk;
  ublk.reserve(upair.size());
  for (int i = 0; i < Pvar; ++i)
    for (int k = diag_pos[i]; k < row_ptr[i + 1]; ++k) {
      const int j = col_var[k];
      int kt = k;
      if (j != i) {
        const int32_t* b = col_var.data() + row_ptr[j];
        const int32_t* e = col_var.data() + row_ptr[j + 1];
        kt = (int32_t)(std::lower_bound(b, e, i) - col_var.data());
      }
      ublk.push_back(make_int4(k, kt, i, j));
    }
  h->n_upper = (int32_t)ublk.size();
  h->schur_pairs = sr.pairs;
  h->n_g = (int32_t)st.g_row.size();
  h->nbands = st.nbands;
  h->n_segs = (int32_t)(st.segs.size() / 4);
  h->n_visits = st.visits;
  h->n_batches = (int64_t)(st.batches.size() / 4);
  h->n_tpairs = (int64_t)st.pairs.size();
  h->n_staged = st.staged;
  h->h_segs.assign(reinterpret_cast<const int4*>(st.segs.data()),
                   reinterpret_cast<const int4*>(st.segs.data()) + h->n_segs);
  // Partial slots of each upper block: its tile's segments in order, each
  // segment's parts of the block in order.
  std::vector<int32_t> uslot_ptr(ublk.size() + 1, 0), uslot;
  for (size_t u = 0; u < ublk.size(); ++u) {
    const int i = ublk[u].z, j = ublk[u].w;
    const int64_t key = (int64_t)(i / kTileBand) * st.nbands + j / kTileBand;
    const auto it = std::lower_bound(st.tile_key.begin(), st.tile_key.end(), key);
    if (it == st.tile_key.end() || *it != key) {
      uslot_ptr[u + 1] = (int32_t)uslot.size();  // a block no landmark couples (diagonal only)
      continue;
    }
    const size_t t = (size_t)(it - st.tile_key.begin());
    const int blk = (i % kTileBand) * kTileBand + j % kTileBand;
    for (int sg = st.tile_seg[2 * t]; sg < st.tile_seg[2 * t + 1]; ++sg) {
      const uint16_t bw = st.seg_block[(size_t)sg * kTileBlocks + blk];
      for (int q = 0; q < (bw >> 8); ++q) uslot.push_back(sg * kTileBlocks + (bw & 255) + q);
    }
    uslot_ptr[u + 1] = (int32_t)uslot.size();
  }
  // Learned preconditioner structure: row and transposed position of every
  // block of S, and the landmark pairs summed into it (shared observations).
  std::vector<int32_t> lp_pos_row(h->nnzb), lp_tpos(h->nnzb), lp_shared(h->nnzb, 0);
  h->lp_max_lower_deg = 0;
  for (int i = 0; i < Pvar; ++i) {
    for (int k = row_ptr[i]; k < row_ptr[i + 1]; ++k) lp_pos_row[k] = i;
    h->lp_max_lower_deg = std::max(h->lp_max_lower_deg, diag_pos[i] - row_ptr[i]);
  }
  for (int u = 0; u < h->n_upper; ++u) {
    const int4 b = ublk[u];
    lp_tpos[b.x] = b.y;
    lp_tpos[b.y] = b.x;
    lp_shared[b.x] = lp_shared[b.y] = upair[u];
  }
  std::vector<int32_t> obs_col(N, -1);
  for (int o = 0; o < N; ++o)
    if ((meta[o] & 4) && h->lm_active[h->s_landmark[o]]) obs_col[o] = vertex_var[h->s_vertex[o]];
  int rc;
  if ((rc = upload(h, h->lm_flags, flags.data(), flags.size()))) return rc;
  if ((rc = upload(h, h->obs_meta, meta.data(), meta.size()))) return rc;
  if ((rc = upload(h, h->vertex_var, vertex_var.data(), vertex_var.size()))) return rc;
  if ((rc = upload(h, h->var_vertex, var_vertex.data(), var_vertex.size()))) return rc;
  if ((rc = upload(h, h->tile_begin, tile_begin.data(), tile_begin.size()))) return rc;
  if ((rc = upload(h, h->split_ids, split.data(), split.size()))) return rc;
  if ((rc = upload(h, h->split_tiles, split_tiles.data(), split_tiles.size()))) return rc;
  if ((rc = upload(h, h->lp_pos_row, lp_pos_row.data(), lp_pos_row.size()))) return rc;
  if ((rc = upload(h, h->lp_tpos, lp_tpos.data(), lp_tpos.size()))) return rc;
  if ((rc = upload(h, h->lp_shared, lp_shared.data(), lp_shared.size()))) return rc;
  if ((rc = upload(h, h->inc_ptr, inc_ptr.data(), inc_ptr.size()))) return rc;
  if ((rc = upload(h, h->inc, inc.data(), inc.size()))) return rc;
  if ((rc = upload(h, h->row_ptr, row_ptr.data(), row_ptr.size()))) return rc;
  if ((rc = upload(h, h->col_var, col_var.data(), col_var.size()))) return rc;
  if ((rc = upload(h, h->diag_pos, diag_pos.data(), diag_pos.size()))) return rc;
  if ((rc = upload(h, h->ublk, ublk.data(), ublk.size()))) return rc;
  if ((rc = upload(h, h->g_row, st.g_row.data(), st.g_row.size()))) return rc;
  if ((rc = upload(h, h->g_inc_ptr, st.g_inc_ptr.data(), st.g_inc_ptr.size()))) return rc;
  if ((rc = upload(h, h->g_inc, st.g_inc.data(), st.g_inc.size()))) return rc;
  if ((rc = upload(h, h->t_slots, reinterpret_cast<const int2*>(st.slots.data()), st.slots.size() / 2))) return rc;
  if ((rc = upload(h, h->t_seg_thread, st.seg_thread.data(), st.seg_thread.size()))) return rc;
  if ((rc = upload(h, h->t_uslot_ptr, uslot_ptr.data(), uslot_ptr.size()))) return rc;
  if ((rc = upload(h, h->t_uslot, uslot.data(), uslot.size()))) return rc;
  if ((rc = upload(h, h->t_batches, reinterpret_cast<const int4*>(st.batches.data()), st.batches.size() / 4)))
    return rc;
  if ((rc = upload(h, h->t_segs, reinterpret_cast<const int4*>(st.segs.data()), st.segs.size() / 4))) return rc;
  if ((rc = upload(h, h->t_batch_off, st.batch_off.data(), st.batch_off.size()))) return rc;
  if ((rc = upload(h, h->t_pairs, st.pairs.data(), st.pairs.size()))) return rc;
  if ((rc = upload_item_order(h))) return rc;
  if ((rc = upload(h, h->obs_col, obs_col.data(), obs_col.size()))) return rc;
  const size_t T = h->tiles, V6 = 6 * (size_t)std::max(Pvar, 1);
  const size_t vb = (Pvar + 255) / 256 + 1;
  bool ok = h->tile_cost.alloc(2 * T) && h->tile_cost2.alloc(2 * T) && h->S.alloc(36 * (size_t)h->nnzb) &&
            h->split_part.alloc(h->n_split ? kLmAcc * T : 1) &&
            h->gf.alloc(kFactor * std::max<size_t>(st.g_row.size(), 1)) &&
            h->gk.alloc(3 * std::max<size_t>(st.g_row.size(), 1)) &&
            h->schur_partial.alloc((size_t)kTilePartial * std::max(h->n_segs, 1)) &&
            h->pose_jtj.alloc(36 * (size_t)std::max(Pvar, 1)) &&
            h->rhs.alloc(V6) && h->pose_grad.alloc(V6) && h->pose_diag.alloc(V6) && h->pose_scale.alloc(V6) &&
            h->w.alloc(V6) && h->Minv.alloc(36 * (size_t)std::max(Pvar, 1)) && h->px.alloc(V6) &&
            h->pr.alloc(V6) && h->pz.alloc(V6) && h->pp.alloc(V6) && h->pp2.alloc(V6) && h->pq.alloc(V6) &&
            h->pcg_part.alloc(3 * (size_t)std::max(Pvar, 1) + 3) &&
            h->parts_a.alloc(std::max<size_t>(Pvar, 2 * vb) + 1) && h->parts_b.alloc(2 * vb + 2) &&
            h->parts_l.alloc(2 * ((size_t)h->tiles + (size_t)(h->n_split + 255) / 256 + 1)) &&
            h->parts_c.alloc((size_t)(h->L + 255) / 256 + 1) &&
            h->parts_v.alloc((size_t)(h->P + 255) / 256 + 1) && h->parts_w.alloc((size_t)(h->P + 255) / 256 + 1) &&
            h->parts_g.alloc(((size_t)Pvar + h->L + 255) / 256 + 1);
  if (!ok) return set_err(h, MLBA_ENOMEM, "device allocation failed");
  // The landmark step of inactive or observation-less landmarks stays zero.
  if (h->L > 0) HIP_OK(hipMemsetAsync(h->lm_u.p, 0, 3 * (size_t)h->L * sizeof(double), h->stream));
  DevTopology& t = h->topo;
  t.N = h->N; t.L = h->L; t.P = h->P; t.Pvar = Pvar; t.M = h->M; t.C = h->C;
  t.obs_kp = h->obs_kp.p; t.obs_sinv = h->obs_sinv.p; t.obs_vertex = h->obs_vertex.p; t.obs_meta = h->obs_meta.p;
  t.obs_landmark = h->obs_landmark.p; t.obs_col = h->obs_col.p; t.lm_begin = h->lm_begin_d.p; t.lm_anchor = h->lm_anchor_d.p;
  t.lm_flags = h->lm_flags.p; t.cams = h->cams.p; t.mission_T = h->mission_T.p;
  t.vertex_mission = h->vertex_mission_d.p; t.vertex_var = h->vertex_var.p; t.var_vertex = h->var_vertex.p;
  t.row_ptr = h->row_ptr.p; t.col_var = h->col_var.p; t.diag_pos = h->diag_pos.p; t.inc_ptr = h->inc_ptr.p;
  t.inc = h->inc.p; t.max_row_blocks = h->max_row_blocks;
  SchurTilesDev& d = h->tdev;
  d.n_segs = h->n_segs; d.seg_order = h->t_seg_order.p; d.segs = h->t_segs.p; d.seg_thread = h->t_seg_thread.p;
  d.batches = h->t_batches.p; d.slots = h->t_slots.p; d.batch_off = h->t_batch_off.p; d.pairs = h->t_pairs.p;
  d.uslot_ptr = h->t_uslot_ptr.p; d.uslot = h->t_uslot.p; d.n_uslot = (int32_t)uslot.size();
  HIP_OK(hipStreamSynchronize(h->stream));
  h->topology_ok = true;
  return MLBA_OK;
}
int check_topology(mlba_handle* h) {
  if (!h->topology_ok) return set_err(h, MLBA_ESTATE, "the last change of the active landmarks failed");
  return MLBA_OK;
}

// Kernel timing inside the LM loop, only with a summary to fill: a timed span
// runs from one event to the next, most of them stop events of the kernels
// themselves (see launch in ba_kernels.hip); collect_events (after a stream
// synchronization) adds the elapsed times to the summary. With a recorded pair
// of events around every span, 10 LM iterations of a 10-keyframe map took 2.65
// ms against 2.03 without any.
hipEvent_t next_event(mlba_handle* h) {
  if (h->ev_next == h->ev_pool.size()) {
    hipEvent_t e;
    if (hipEventCreate(&e) != hipSuccess) return nullptr;
    h->ev_pool.push_back(e);
  }
  return h->ev_pool[h->ev_next++];
}
// An event for a launch's stop argument (null without a summary).
hipEvent_t stop_event(mlba_handle* h) { return h->ev_summary ? next_event(h) : nullptr; }
// An event recorded here.
hipEvent_t mark_event(mlba_handle* h) {
  hipEvent_t e = stop_event(h);
  if (e) (void)hipEventRecord(e, h->stream);
  return e;
}
void time_span(mlba_handle* h, int id, hipEvent_t begin, hipEvent_t end) {
  if (begin && end) h->ev_pending.push_back({id, {begin, end}});
}
void collect_events(mlba_handle* h) {
  if (h->ev_summary) {
    for (auto& p : h->ev_pending) {
      float ms = 0.f;
      if (hipEventElapsedTime(&ms, p.second.first, p.second.second) == hipSuccess) {
        h->ev_summary->kernel_ms[p.first] += ms;
        h->ev_summary->kernel_launches[p.first] += 1;
      }
    }
  }
  h->ev_pending.clear();
  h->ev_next = 0;
}

// Hat-function coarse basis over the variable-vertex order for the deflated
// PCG: K nodes spread evenly; vertex i has weights (1 - t, t) on nodes
// (n0, n0 + 1). K = 0 disables deflation.
int ensure_coarse_basis(mlba_handle* h, int32_t requested) {
  const int Pvar = h->Pvar;
  int K = requested > 0 ? requested : (requested < 0 ? 0 : std::min(pcg_max_hat_nodes(), Pvar / 16));
  K = std::min(K, pcg_max_hat_nodes());
  if (K < 2 || Pvar < 2 * K) K = 0;
  if (K == h->hat_K && h->hat_node.p) return MLBA_OK;
  std::vector<int32_t> node(std::max(Pvar, 1), 0), range(2 * std::max(K, 1), 0);
  std::vector<double> wts(2 * (size_t)std::max(Pvar, 1), 0.0);
  if (K > 0) {
    for (int k = 0; k < K; ++k) { range[2 * k] = Pvar; range[2 * k + 1] = -1; }
    for (int i = 0; i < Pvar; ++i) {
      const double sp = (double)i * (K - 1) / (Pvar - 1);
      const int n0 = std::min((int)sp, K - 2);
      const double t = sp - n0;
      node[i] = n0;
      wts[2 * i] = 1.0 - t;
      wts[2 * i + 1] = t;
      for (int k : {n0, n0 + 1}) {
        range[2 * k] = std::min(range[2 * k], i);
        range[2 * k + 1] = std::max(range[2 * k + 1], i);
      }
    }
  }
  // Window of hat nodes that the rows of each PCG row group touch in S W:
  // nodes of their block columns.
  const int gr = pcg_group_rows();
  const int ngroups = (std::max(Pvar, 1) + gr - 1) / gr;
  std::vector<int32_t> lo(ngroups, 0);
  int width = 1;
  if (K > 0) {
    for (int g = 0; g < ngroups; ++g) {
      int a = K, b = -1;
      for (int i = g * gr; i < std::min(Pvar, (g + 1) * gr); ++i)
        for (int k = h->h_row_ptr[i]; k < h->h_row_ptr[i + 1]; ++k) {
          const int n0 = node[h->h_col_var[k]];
          a = std::min(a, n0);
          b = std::max(b, std::min(n0 + 1, K - 1));
        }
      if (b < a) a = b = 0;
      lo[g] = a;
      width = std::max(width, b - a + 1);
    }
  }
  h->grp_width = 6 * width;
  // Hat node and weights of each block's column vertex.
  std::vector<int32_t> bh(std::max<size_t>(h->h_col_var.size(), 1), 0);
  std::vector<double> bw(2 * bh.size(), 0.0);
  for (size_t kb = 0; kb < h->h_col_var.size(); ++kb) {
    const int j = h->h_col_var[kb];
    bh[kb] = node[j];
    bw[2 * kb] = wts[2 * j];
    bw[2 * kb + 1] = wts[2 * j + 1];
  }
  // Blocks of each row in the support of each hat (columns are sorted, the
  // support is a vertex range, so they are contiguous).
  std::vector<int32_t> br(2 * (size_t)std::max(Pvar, 1) * std::max(K, 1), 0);
  for (int i = 0; i < Pvar && K > 0; ++i) {
    const int32_t* b = h->h_col_var.data() + h->h_row_ptr[i];
    const int32_t* e = h->h_col_var.data() + h->h_row_ptr[i + 1];
    for (int k = 0; k < K; ++k) {
      br[2 * ((size_t)i * K + k)] = (int32_t)(std::lower_bound(b, e, range[2 * k]) - h->h_col_var.data());
      br[2 * ((size_t)i * K + k) + 1] = (int32_t)(std::upper_bound(b, e, range[2 * k + 1]) - h->h_col_var.data());
    }
  }
  int rc;
  if ((rc = upload(h, h->blk_hat, bh.data(), bh.size())) || (rc = upload(h, h->blk_w, bw.data(), bw.size())) ||
      (rc = upload(h, h->blk_rng, br.data(), br.size())))
    return rc;
  if ((rc = upload(h, h->hat_node, node.data(), node.size())) || (rc = upload(h, h->hat_w, wts.data(), wts.size())) ||
      (rc = upload(h, h->node_range, range.data(), range.size())) || (rc = upload(h, h->grp_lo, lo.data(), lo.size())))
    return rc;
  // Room for the recycled dense columns beside the hat columns.
  const size_t nr = K > 0 ? (size_t)pcg_max_ritz() : 0;
  const size_t ne = 6 * (size_t)K + nr, gw = (size_t)h->grp_width + nr;
  const size_t groups = pcg_update_groups(std::max(Pvar, 1));
  if (!h->defl_SR.alloc(groups * gw * (size_t)(6 * gr)) ||
      !h->defl_E.alloc(std::max<size_t>(ne * ne, 1)) || !h->defl_Einv.alloc(std::max<size_t>(ne * ne + groups * gw * ne, 1)) ||
      !h->defl_y.alloc(std::max<size_t>(ne, 1)) || !h->defl_cden.alloc(std::max<size_t>(nr, 1)) ||
      !h->pcg_part2.alloc((groups + 1) * (3 + ne)) || !h->pcg_step.alloc(std::max<size_t>(pcg_step_doubles(Pvar, h->nnzb), 1)))
    return set_err(h, MLBA_ENOMEM, "device allocation failed");
  if (nr > 0) {
    const size_t n6 = 6 * (size_t)Pvar, zc = (size_t)pcg_max_lanczos();
    if (!h->ritz[0].alloc(nr * n6) || !h->ritz[1].alloc(nr * n6) || !h->ritz_new.alloc(nr * n6) ||
        !h->ritz_snew.alloc(nr * n6) || !h->ritz_Zh.alloc(zc * n6) || !h->ritz_coef.alloc(2 * zc) ||
        !h->ritz_small.alloc(2 * (2 * nr) * (2 * nr) + zc * nr + 2 * nr * nr))
      return set_err(h, MLBA_ENOMEM, "device allocation failed");
    h->ritz_zcap = (int32_t)zc;
    if (!h->ritz_pinned) {
      HIP_OK(hipHostMalloc(reinterpret_cast<void**>(&h->ritz_pinned), kRitzPinned * sizeof(double), hipHostMallocDefault));
      HIP_OK(hipEventCreateWithFlags(&h->ritz_ev_coef, hipEventDisableTiming));
      HIP_OK(hipEventCreateWithFlags(&h->ritz_ev_ab, hipEventDisableTiming));
    }
  } else {
    h->ritz_zcap = 0;
  }
  h->ritz_nr = 0;
  h->ritz_stage = 0;
  // Entries of the last group past the last row stay zero.
  HIP_OK(hipMemsetAsync(h->defl_SR.p, 0, h->defl_SR.n * sizeof(double), h->stream));
  h->hat_K = K;
  HIP_OK(hipStreamSynchronize(h->stream));
  return MLBA_OK;
}

// Recycled Ritz columns requested by the options (0 = automatic).
int32_t ritz_count(const mlba_options* o) {
  if (o->pcg_ritz_vectors < 0) return 0;
  return o->pcg_ritz_vectors == 0 ? pcg_max_ritz() : std::min(o->pcg_ritz_vectors, pcg_max_ritz());
}

// Device buffers of a PCG solve with the handle's coarse basis and nr
// recycled columns; Lanczos vectors are kept when `keep_lanczos`.
PcgBuffers pcg_buffers(mlba_handle* h, int32_t nr, bool keep_lanczos) {
  PcgBuffers B{};
  B.Pvar = h->Pvar;
  B.nnzb = h->nnzb;
  B.K = std::max(h->hat_K, 0);
  B.nr = B.K > 0 ? nr : 0;
  B.gwh = h->grp_width;
  B.zcap = keep_lanczos && B.K > 0 ? h->ritz_zcap : 0;
  B.partials = h->sched_pcg;
  B.row_ptr = h->row_ptr.p; B.col_var = h->col_var.p; B.S = h->S.p; B.Minv = h->Minv.p; B.b = h->rhs.p;
  B.hat_node = h->hat_node.p; B.hat_w = h->hat_w.p; B.node_range = h->node_range.p; B.grp_lo = h->grp_lo.p;
  B.R = h->ritz[h->ritz_cur].p;
  B.blk_hat = h->blk_hat.p; B.blk_w = h->blk_w.p; B.blk_rng = h->blk_rng.p;
  B.SR = h->defl_SR.p; B.E = h->defl_E.p; B.Einv = h->defl_Einv.p; B.y = h->defl_y.p; B.cden = h->defl_cden.p;
  B.x = h->px.p; B.r = h->pr.p; B.z = h->pz.p; B.p0 = h->pp.p; B.p1 = h->pp2.p; B.q = h->pq.p;
  B.part = h->pcg_part.p; B.part2 = h->pcg_part2.p; B.step = h->pcg_step.p; B.Zh = h->ritz_Zh.p; B.coef = h->ritz_coef.p;
  B.state_dev = h->pcg_state.p; B.state_host = h->pcg_host;
  return B;
}

// Recycled deflation columns from the solve just finished (its Lanczos
// vectors and coefficients, its S and SW): the r Ritz vectors of the solve's
// tridiagonal for its smallest eigenvalues, merged with the current columns
// by a Rayleigh-Ritz step on span[R, Rn] w.r.t. (S, M) that keeps the r best.
// A solve whose deflation was not applied (E not positive definite) clears
// the columns; one too short to resolve r Ritz vectors, or whose
// coefficients are not usable, keeps them.
//
// Stage 1, right after the solve: queue the coefficient download.
void ritz_after_solve(mlba_handle* h, int32_t r, int32_t iters) {
  h->ritz_stage = 0;
  if (r <= 0 || h->hat_K <= 0 || h->ritz_zcap <= 0 || !pcg_deflation_applied(h->pcg_host)) {
    h->ritz_nr = 0;
    return;
  }
  const int m = std::min<int>(iters, h->ritz_zcap);
  if (m < r + 2) return;
  if (hipMemcpyAsync(h->ritz_pinned, h->ritz_coef.p, 2 * (size_t)m * sizeof(double), hipMemcpyDeviceToHost,
                     h->stream) != hipSuccess ||
      hipEventRecord(h->ritz_ev_coef, h->stream) != hipSuccess)
    return;
  h->ritz_m = m;
  h->ritz_r = r;
  h->ritz_stage = 1;
}

// Stage 2, while the step's back-substitution and cost run: the
// tridiagonal's eigenvectors on the host, then Rn, S Rn and the Gram
// matrices queued on the device, and their download.
int ritz_queue_vectors(mlba_handle* h) {
  if (h->ritz_stage != 1) return MLBA_OK;
  h->ritz_stage = 0;
  hipStream_t s = h->stream;
  HIP_OK(hipEventSynchronize(h->ritz_ev_coef));
  const int m = h->ritz_m, r = h->ritz_r;
  const double* coef = h->ritz_pinned;
  // Lanczos tridiagonal of the deflated preconditioned operator:
  // T_jj = 1 / alpha_j + beta_{j-1} / alpha_{j-1}, T_j,j+1 = -sqrt(beta_j) / alpha_j,
  // beta_j = rz_{j+1} / rz_j.
  std::vector<double> d(m), e(std::max(m - 1, 1)), vals(r), Y((size_t)m * r);
  for (int j = 0; j < m; ++j) {
    const double rz = coef[2 * j], al = coef[2 * j + 1];
    if (!(rz > 0.0) || !(al > 0.0) || !std::isfinite(rz) || !std::isfinite(al)) return MLBA_OK;
    // A one-launch iteration's r'z is a difference: too few digits are left.
    if (j > 0 && rz <= 1e-12 * coef[2 * (j - 1)]) return MLBA_OK;
    d[j] = 1.0 / al + (j > 0 ? (rz / coef[2 * (j - 1)]) / coef[2 * (j - 1) + 1] : 0.0);
    if (j + 1 < m) e[j] = -std::sqrt(coef[2 * (j + 1)] / rz) / al;
  }
  if (tridiag_smallest_eigenpairs(m, d.data(), e.data(), r, vals.data(), Y.data())) return MLBA_OK;
  const int rmax = pcg_max_ritz();
  double* hY = h->ritz_pinned + kRitzCoefOff;
  for (int j = 0; j < m; ++j)
    for (int c = 0; c < r; ++c) hY[(size_t)j * r + c] = Y[(size_t)j * r + c] / std::sqrt(coef[2 * j]);
  double* dAB = h->ritz_small.p;
  double* dY = dAB + 2 * (2 * rmax) * (2 * rmax);
  const size_t n6 = 6 * (size_t)h->Pvar;
  HIP_OK(hipMemcpyAsync(dY, hY, (size_t)m * r * sizeof(double), hipMemcpyHostToDevice, s));
  launch_ritz_form(s, h->Pvar, m, r, h->ritz_Zh.p, dY, h->ritz_new.p);
  const int nr_old = h->ritz_nr;
  if (nr_old == 0) {
    HIP_OK(hipMemcpyAsync(h->ritz[h->ritz_cur].p, h->ritz_new.p, (size_t)r * n6 * sizeof(double),
                          hipMemcpyDeviceToDevice, s));
    HIP_OK(hipGetLastError());
    h->ritz_nr = r;
    return MLBA_OK;
  }
  launch_ritz_spmv(s, h->Pvar, r, h->row_ptr.p, h->col_var.p, h->S.p, h->ritz_new.p, h->ritz_snew.p);
  launch_ritz_gram(s, pcg_buffers(h, nr_old, false), r, h->ritz_new.p, h->ritz_snew.p, h->diag_pos.p, dAB);
  const int nb = nr_old + r;
  HIP_OK(hipMemcpyAsync(h->ritz_pinned + kRitzGramOff, dAB, 2 * (size_t)nb * nb * sizeof(double),
                        hipMemcpyDeviceToHost, s));
  HIP_OK(hipEventRecord(h->ritz_ev_ab, s));
  HIP_OK(hipGetLastError());
  h->ritz_stage = 2;
  return MLBA_OK;
}

// Stage 3, before the next solve: the small generalized eigenproblem of the
// merge on the host and the merged columns queued on the device.
int ritz_merge(mlba_handle* h) {
  if (h->ritz_stage != 2) return MLBA_OK;
  h->ritz_stage = 0;
  hipStream_t s = h->stream;
  HIP_OK(hipEventSynchronize(h->ritz_ev_ab));
  const int nr_old = h->ritz_nr, r = h->ritz_r, nb = nr_old + r, rmax = pcg_max_ritz();
  const double* AB = h->ritz_pinned + kRitzGramOff;
  std::vector<double> A((size_t)nb * nb), B((size_t)nb * nb), C((size_t)nb * r), vals(r);
  for (int i = 0; i < nb; ++i)
    for (int j = 0; j < nb; ++j) {
      A[(size_t)i * nb + j] = 0.5 * (AB[(size_t)i * nb + j] + AB[(size_t)j * nb + i]);
      B[(size_t)i * nb + j] = 0.5 * (AB[(size_t)nb * nb + (size_t)i * nb + j] + AB[(size_t)nb * nb + (size_t)j * nb + i]);
    }
  const size_t n6 = 6 * (size_t)h->Pvar;
  if (generalized_smallest_eigenpairs(nb, A.data(), B.data(), r, vals.data(), C.data())) {
    // The merged Gram matrix is singular: start over from the new vectors.
    HIP_OK(hipMemcpyAsync(h->ritz[h->ritz_cur].p, h->ritz_new.p, (size_t)r * n6 * sizeof(double),
                          hipMemcpyDeviceToDevice, s));
    h->ritz_nr = r;
    return MLBA_OK;
  }
  double* hC = h->ritz_pinned + kRitzMergeOff;
  std::copy(C.begin(), C.end(), hC);
  double* dC = h->ritz_small.p + 2 * (2 * rmax) * (2 * rmax) + (size_t)h->ritz_zcap * rmax;
  HIP_OK(hipMemcpyAsync(dC, hC, C.size() * sizeof(double), hipMemcpyHostToDevice, s));
  launch_ritz_merge(s, h->Pvar, h->ritz[h->ritz_cur].p, nr_old, h->ritz_new.p, r, dC, r,
                    h->ritz[h->ritz_cur ^ 1].p);
  HIP_OK(hipGetLastError());
  h->ritz_cur ^= 1;
  h->ritz_nr = r;
  return MLBA_OK;
}

DevLoss make_loss(const mlba_options* o) {
  DevLoss l;
  l.type = o ? o->loss_type : MLBA_LOSS_MAPLAB_HUBER;
  l.scale_px = o ? o->loss_scale_px : 1.0;
  return l;
}

// Linearize at the current state: residual records, landmark reductions,
// vertex-row gradient and diag(F'F). Leaves cost / fixed cost / gradient
// max norm in the scalar slots (device).
// Per-linearization Schur factors (P, p and k of every factor block).
void schur_factors(mlba_handle* h, hipEvent_t stop = nullptr) {
  launch_schur_factors(h->stream, h->topo, h->n_g, h->g_row.p, h->g_inc_ptr.p, h->g_inc.p, h->vR.p, h->lm.p,
                       h->obs_rec.p, h->gf.p, h->gk.p, h->f32_jac, stop);
}

// With `rotations`, the rotation records of the current vertices are formed
// first (an accepted candidate brings its own). Returns the last event of the
// linearization through `end`.
int linearize(mlba_handle* h, const mlba_options* o, bool rotations = true, hipEvent_t* end = nullptr) {
  hipStream_t s = h->stream;
  if (rotations) launch_vertex_prep(s, h->P, h->vert.p, h->vR.p);
  const hipEvent_t e0 = mark_event(h), e1 = stop_event(h), e2 = stop_event(h), e3 = stop_event(h);
  launch_linearize(s, true, h->tiles, h->topo, h->vert.p, h->vR.p, h->lm.p, make_loss(o), h->tile_begin.p,
                   h->obs_rec.p, h->lm_acc.p, h->split_part.p, h->tile_cost.p, h->f32_jac, e1);
  time_span(h, MLBA_KERNEL_LINEARIZE, e0, e1);
  launch_split_sum(s, h->n_split, h->split_ids.p, h->split_tiles.p, h->split_part.p, h->lm_acc.p);
  launch_pose_rows(s, h->topo, h->vert.p, h->vR.p, h->lm.p, h->obs_rec.p, h->lm_acc.p, h->pose_grad.p,
                   h->pose_diag.p, h->pose_jtj.p, h->f32_jac, e2);
  time_span(h, MLBA_KERNEL_POSE_ROWS, e1, e2);
  const int gb = (h->Pvar + h->L + 255) / 256;
  launch_gradient_norm(s, h->topo, h->vert.p, h->pose_grad.p, h->lm_acc.p, h->parts_g.p);
  ReduceBatch rb{};
  rb.d[0] = {h->tiles, 2, 0, 0, h->tile_cost.p, h->scal.p + kCost};
  rb.d[1] = {h->tiles, 2, 1, 0, h->tile_cost.p, h->scal.p + kFixed};
  rb.d[2] = {gb, 1, 0, 1, h->parts_g.p, h->scal.p + kGradMax};
  rb.count = 3;
  if (!launch_reduce_many(s, rb, e3)) return set_err(h, MLBA_EINVAL, "internal: scalar reduction batch size");
  if (end) *end = e3;
  HIP_OK(hipGetLastError());
  return MLBA_OK;
}

int read_scalars(mlba_handle* h) {
  HIP_OK(hipMemcpyAsync(h->scal_host, h->scal.p, kNumSlots * sizeof(double), hipMemcpyDeviceToHost, h->stream));
  HIP_OK(hipStreamSynchronize(h->stream));
  collect_events(h);
  return MLBA_OK;
}

void push_iteration(mlba_summary* sm, const mlba_iteration_summary& it) {
  if (!sm) return;
  if (sm->iterations && sm->num_iterations < sm->iterations_capacity) sm->iterations[sm->num_iterations] = it;
  sm->num_iterations++;
}

// One ceres::Solve (TrustRegionMinimizer + LevenbergMarquardtStrategy).
// ------------------------------------------------------------ learned preconditioner

LpSystem lp_system(const mlba_handle* h) {
  LpSystem sys{};
  sys.Pvar = h->Pvar;
  sys.nnzb = h->nnzb;
  sys.row_ptr = h->row_ptr.p;
  sys.col_var = h->col_var.p;
  sys.diag_pos = h->diag_pos.p;
  sys.pos_row = h->lp_pos_row.p;
  sys.tpos = h->lp_tpos.p;
  sys.S = h->S.p;
  return sys;
}

// Buffers of the preconditioner (network ones with `network`, T2 with `t2`).
int lp_ensure(mlba_handle* h, bool network, bool t2) {
  const size_t P = std::max(h->Pvar, 1), Z = std::max(h->nnzb, 1);
  bool ok = h->lp_linv.alloc(36 * P) && h->lp_t.alloc(6 * P) && h->lp_u.alloc(6 * P) && h->lp_part.alloc(2 * P) &&
            h->lp_shat.alloc(36 * Z) && h->lp_snorm.alloc(Z) && h->lp_kmat.alloc(36 * Z) &&
            h->lp_state.alloc(lp_pcg_state_bytes());
  if (network) ok = ok && h->lp_nf.alloc(kLpNodeFeatures * P) && h->lp_ef.alloc(kLpEdgeFeatures * Z) &&
                    h->lp_theta.alloc(kLpTerms * P);
  if (t2) ok = ok && h->lp_t2.alloc(36 * Z) && h->lp_trace.alloc(4 * P);
  if (!ok) return set_err(h, MLBA_ENOMEM, "device allocation failed");
  if (!h->lp_state_host && hipHostMalloc(&h->lp_state_host, lp_pcg_state_bytes(), hipHostMallocDefault) != hipSuccess) {
    h->lp_state_host = nullptr;
    return set_err(h, MLBA_ENOMEM, "pinned allocation failed");
  }
  if (network && h->lp_model && (h->lp_ws_nodes != h->Pvar || h->lp_ws_slots != h->nnzb)) {
    if (h->lp_ws) gnn_workspace_destroy(h->lp_ws);
    h->lp_ws = gnn_workspace_create(h->stream, h->Pvar, h->nnzb, false);
    if (!h->lp_ws) { h->lp_ws_nodes = -1; return set_err(h, MLBA_ENOMEM, "network workspace allocation failed"); }
    h->lp_ws_nodes = h->Pvar;
    h->lp_ws_slots = h->nnzb;
  }
  return MLBA_OK;
}

LpPcgBuffers lp_buffers(mlba_handle* h, bool use_k) {
  LpPcgBuffers B{};
  B.sys = lp_system(h);
  B.linv = h->lp_linv.p;
  B.kmat = use_k ? h->lp_kmat.p : nullptr;
  B.b = h->rhs.p;
  B.x = h->px.p; B.r = h->pr.p; B.t = h->lp_t.p; B.u = h->lp_u.p; B.z = h->pz.p;
  B.p0 = h->pp.p; B.p1 = h->pp2.p; B.q = h->pq.p; B.part = h->lp_part.p;
  B.state_dev = h->lp_state.p;
  B.state_host = h->lp_state_host;
  return B;
}

GnnGraph lp_graph(const mlba_handle* h) {
  GnnGraph g{};
  g.nodes = h->Pvar;
  g.slots = h->nnzb;
  g.row_ptr = h->row_ptr.p;
  g.col = h->col_var.p;
  g.rev = h->lp_tpos.p;
  g.node_feat = h->lp_nf.p;
  g.edge_feat = h->lp_ef.p;
  return g;
}

// Set-up of the preconditioner of the current S (factors into the step's
// failure counter). With `learned`: normalized blocks, features, the
// network's theta and K; *use_k = false when a row does not fit the
// neighbourhood kernel (block-Jacobi is used then).
int lp_setup(mlba_handle* h, bool learned, bool* use_k) {
  hipStream_t s = h->stream;
  const LpSystem sys = lp_system(h);
  launch_lp_factor(s, sys, h->lp_linv.p, h->fail.p);
  *use_k = false;
  if (learned) {
    launch_lp_normalize(s, sys, h->lp_linv.p, h->lp_shat.p, h->lp_snorm.p);
    launch_lp_features(s, sys, h->pose_jtj.p, h->pose_scale.p, h->lp_snorm.p, h->lp_shared.p, h->lp_norm.p,
                       h->lp_nf.p, h->lp_ef.p);
    if (!gnn_forward(s, h->lp_ws, lp_graph(h), h->lp_params.p, h->lp_theta.p))
      return set_err(h, MLBA_EDEVICE, "network launch failed");
    *use_k = launch_lp_terms(s, sys, h->lp_max_lower_deg, kLpAssemble, h->lp_shat.p, h->lp_theta.p, h->lp_kmat.p,
                             nullptr, nullptr);
  }
  HIP_OK(hipGetLastError());
  return MLBA_OK;
}

// PCG on the current S with the learned preconditioner (block-Jacobi when not
// `learned`), the block-Jacobi repeat when it does not converge.
int lp_solve(mlba_handle* h, const mlba_options* o, bool learned, int* iters) {
  int rc = lp_ensure(h, learned, false);
  if (rc) return rc;
  bool use_k = false;
  if ((rc = lp_setup(h, learned, &use_k))) return rc;
  int32_t conv = 0;
  int it = launch_lp_pcg(h->stream, lp_buffers(h, use_k), o->pcg_relative_tolerance, o->pcg_max_iterations,
                         kPcgPoll, &conv);
  if (it < 0) return set_err(h, MLBA_EDEVICE, "PCG launch failed");
  if (use_k) {
    h->lp_stats.solves++;
    h->lp_stats.iterations += it;
    if (!conv) {
      const int it2 = launch_lp_pcg(h->stream, lp_buffers(h, false), o->pcg_relative_tolerance,
                                    o->pcg_max_iterations, kPcgPoll, &conv);
      if (it2 < 0) return set_err(h, MLBA_EDEVICE, "PCG launch failed");
      h->lp_stats.fallbacks++;
      h->lp_stats.fallback_iterations += it2;
      it += it2;
    }
  }
  *iters = it;
  return MLBA_OK;
}

// The hat-deflated PCG with the learned preconditioner G'G (set up by
// lp_setup with `learned`); no recycled columns.
PcgBuffers lp_deflated_buffers(mlba_handle* h) {
  PcgBuffers B = pcg_buffers(h, 0, false);
  B.linv = h->lp_linv.p;
  B.kmat = h->lp_kmat.p;
  B.diag_pos = h->diag_pos.p;
  B.tpos = h->lp_tpos.p;
  B.t = h->lp_t.p;
  B.u = h->lp_u.p;
  return B;
}

// PCG on the current S with G'G inside the hat deflation; a solve that does
// not converge (or a row that does not fit the neighbourhood kernel) is
// repeated (run) with the deflated block-Jacobi PCG, which needs Minv.
int lp_deflated_solve(mlba_handle* h, const mlba_options* o, int* iters) {
  int rc = lp_ensure(h, true, false);
  if (rc) return rc;
  bool use_k = false;
  if ((rc = lp_setup(h, true, &use_k))) return rc;
  // The recycled columns come from block-Jacobi solves; they start again
  // when that solver is selected next.
  h->ritz_nr = 0;
  h->ritz_stage = 0;
  const int32_t maxit = o->pcg_max_iterations;
  int it = 0;
  if (use_k) {
    it = launch_pcg_deflated(h->stream, lp_deflated_buffers(h), o->pcg_relative_tolerance, maxit, kPcgPoll, kPcgPoll,
                             nullptr, 0);
    if (it < 0) return set_err(h, MLBA_EDEVICE, "PCG launch failed");
    h->lp_stats.solves++;
    h->lp_stats.iterations += it;
    if (it < maxit) {
      *iters = it;
      return MLBA_OK;
    }
  }
  const int it2 = launch_pcg_deflated(h->stream, pcg_buffers(h, 0, false), o->pcg_relative_tolerance, maxit, kPcgPoll,
                                      kPcgPoll, nullptr, 0);
  if (it2 < 0) return set_err(h, MLBA_EDEVICE, "PCG launch failed");
  if (use_k) {
    h->lp_stats.fallbacks++;
    h->lp_stats.fallback_iterations += it2;
  }
  *iters = it + it2;
  return MLBA_OK;
}

int minimize(mlba_handle* h, const mlba_options* o, double initial_radius, mlba_summary* sm, double* last_radius,
             int* termination) {
  hipStream_t s = h->stream;
  const double t_start = now_s();
  double radius = initial_radius, decrease_factor = 2.0;
  int rc;
  h->f32_jac = o->jacobian_fp32 != 0;
  if ((rc = ensure_coarse_basis(h, o->pcg_coarse_nodes))) return rc;
  const double t_ev0 = now_s();
  HIP_OK(hipMemsetAsync(h->fail.p, 0, sizeof(int32_t), s));  // each step hands it over and clears it
  if ((rc = linearize(h, o))) return rc;
  launch_jacobi_scaling(s, h->Pvar, h->L, o->use_jacobi_scaling, h->pose_diag.p, h->lm_acc.p, h->pose_scale.p,
                        h->lm_scale.p);
  {
    const hipEvent_t e0 = mark_event(h), e1 = stop_event(h);
    schur_factors(h, e1);
    time_span(h, MLBA_KERNEL_SCHUR_FACTORS, e0, e1);
  }
  if ((rc = read_scalars(h))) return rc;
  if (sm) sm->evaluate_seconds += now_s() - t_ev0;
  double x_cost = h->scal_host[kCost];
  const double fixed_cost = h->scal_host[kFixed];
  double grad_max = h->scal_host[kGradMax];
  if (sm) { sm->initial_cost = x_cost + fixed_cost; sm->fixed_cost = fixed_cost; }
  mlba_iteration_summary it{};
  it.iteration = 0;
  it.step_is_valid = 1;
  it.step_is_successful = 1;
  it.cost = x_cost + fixed_cost;
  it.gradient_max_norm = grad_max;
  it.trust_region_radius = radius;
  it.cumulative_time_in_seconds = it.iteration_time_in_seconds = now_s() - t_start;
  push_iteration(sm, it);
  *termination = MLBA_NO_CONVERGENCE;
  if (grad_max <= o->gradient_tolerance) { *termination = MLBA_CONVERGENCE; *last_radius = radius; goto done; }
  if (o->max_num_iterations <= 0) { *last_radius = radius; goto done; }
  {
    int consecutive_invalid = 0, iteration = 0;
    const int lb = (h->L + 255) / 256;
    const int pb = (h->P + 255) / 256;
    while (true) {
      const double t_iter = now_s();
      ++iteration;
      mlba_iteration_summary cur{};
      cur.iteration = iteration;
      const double inv_mu = 1.0 / radius;
      // Linear solve: Schur elimination + PCG on the reduced camera system.
      const double t_ls = now_s();
      const hipEvent_t e0 = mark_event(h), e_prep = stop_event(h), e_schur = stop_event(h), e_inv = stop_event(h);
      launch_landmark_prep(s, h->topo, h->lm_acc.p, h->lm_scale.p, inv_mu, o->min_lm_diagonal, o->max_lm_diagonal,
                           h->lm_z.p, h->lm_anc.p, h->fail.p, e_prep);
      time_span(h, MLBA_KERNEL_LANDMARK_PREP, e0, e_prep);
      launch_schur_blocks(s, h->topo, h->tdev, h->n_upper, h->ublk.p, h->gf.p, h->gk.p, h->lm_z.p, h->lm_anc.p,
                          h->vR.p, h->pose_scale.p, h->pose_diag.p, h->pose_jtj.p, inv_mu, o->min_lm_diagonal,
                          o->max_lm_diagonal, h->schur_partial.p, h->S.p, h->rhs.p, h->sched_waves, h->sched_xcd,
                          e_schur);
      time_span(h, MLBA_KERNEL_SCHUR_BLOCKS, e_prep, e_schur);
      launch_block_inverse(s, h->Pvar, h->diag_pos.p, h->S.p, h->Minv.p, h->fail.p, e_inv);
      HIP_OK(hipGetLastError());
      int pcg_iters = 0;
      bool pcg_small = false;  // iteration count read with the step's scalars
      if (h->Pvar > 0 && (o->pcg_preconditioner == MLBA_PRECOND_BLOCK_JACOBI ||
                          o->pcg_preconditioner == MLBA_PRECOND_LEARNED)) {
        if ((rc = lp_solve(h, o, o->pcg_preconditioner == MLBA_PRECOND_LEARNED, &pcg_iters))) return rc;
      } else if (h->Pvar > 0 && o->pcg_preconditioner == MLBA_PRECOND_LEARNED_DEFLATED) {
        if ((rc = lp_deflated_solve(h, o, &pcg_iters))) return rc;
      } else if (h->Pvar > 0) {
        const int32_t nritz = ritz_count(o);
        if ((rc = ritz_merge(h))) return rc;
        const int32_t nr_used = nritz > 0 ? h->ritz_nr : 0;
        const PcgBuffers B = pcg_buffers(h, nr_used, nritz > 0);
        if ((pcg_small = pcg_small_applies(B, o->pcg_max_iterations))) {
          if (!launch_pcg_small(s, B, o->pcg_relative_tolerance, o->pcg_max_iterations, h->scal.p + kPcgIters))
            return set_err(h, MLBA_EDEVICE, "PCG launch failed");
          h->ritz_nr = h->ritz_stage = 0;  // no coarse space to recycle columns for
        } else {
          int32_t& est = h->pcg_last_iters[nr_used > 0 ? 1 : 0];
          pcg_iters = launch_pcg_deflated(s, B, o->pcg_relative_tolerance, o->pcg_max_iterations,
                                          est > 0 ? est : kPcgPoll, est > 0 ? kPcgPollAfter : kPcgPoll, nullptr, 0);
          if (pcg_iters < 0) return set_err(h, MLBA_EDEVICE, "PCG launch failed");
          est = pcg_iters;
          ritz_after_solve(h, nritz, pcg_iters);
        }
      }
      const hipEvent_t e_pcg = mark_event(h);
      if (h->Pvar > 0) time_span(h, MLBA_KERNEL_PCG, e_inv, e_pcg);
      // Candidate point and its cost; the step's scalars (model cost change,
      // step and state norms) and the cost in one batch of reductions.
      const hipEvent_t e_vert = stop_event(h), e_back = stop_event(h), e_cand = stop_event(h), e_cost = stop_event(h);
      launch_step_vertices(s, h->topo, h->vert.p, h->px.p, h->pose_scale.p, h->w.p, h->vert_cand.p, h->vR_cand.p,
                           h->parts_w.p, h->parts_v.p, e_vert);
      const int32_t nbs = launch_back_substitute(s, h->topo, h->tiles, h->tile_begin.p, h->n_split, h->split_ids.p,
                                                 h->vR.p, h->lm.p, h->obs_rec.p, h->lm_acc.p, h->lm_z.p, h->w.p,
                                                 h->lm_u.p, h->parts_l.p, h->f32_jac, e_back);
      time_span(h, MLBA_KERNEL_BACK_SUBSTITUTE, e_vert, e_back);
      launch_candidate_landmarks(s, h->topo, h->lm.p, h->lm_u.p, h->lm_cand.p, h->parts_c.p, e_cand);
      launch_linearize(s, false, h->tiles, h->topo, h->vert_cand.p, h->vR_cand.p, h->lm_cand.p, make_loss(o),
                       h->tile_begin.p, nullptr, nullptr, nullptr, h->tile_cost2.p, false, e_cost);
      time_span(h, MLBA_KERNEL_COST, e_cand, e_cost);
      // The step's scalars and the candidate cost in one launch.
      ReduceBatch rb{};
      rb.d[0] = {nbs, 2, 0, 0, h->parts_l.p, h->scal.p + kMcc};
      rb.d[1] = {nbs, 2, 1, 0, h->parts_l.p, h->scal.p + kUU};
      rb.d[2] = {pb, 1, 0, 0, h->parts_w.p, h->scal.p + kWW};
      rb.d[3] = {pb, 1, 0, 0, h->parts_v.p, h->scal.p + kXV};
      rb.d[4] = {lb, 1, 0, 0, h->parts_c.p, h->scal.p + kXL};
      rb.d[5] = {h->tiles, 2, 0, 0, h->tile_cost2.p, h->scal.p + kCandCost};
      rb.count = 6;
      rb.fail = h->fail.p;
      rb.fail_out = h->scal.p + kFail;
      if (!launch_reduce_many(s, rb)) return set_err(h, MLBA_EINVAL, "internal: scalar reduction batch size");
      HIP_OK(hipGetLastError());
      HIP_OK(hipMemcpyAsync(h->scal_host, h->scal.p, kNumSlots * sizeof(double), hipMemcpyDeviceToHost, s));
      HIP_OK(hipEventRecord(h->scal_ev, s));
      // The recycling's host work and kernels go behind the step's cost.
      if ((rc = ritz_queue_vectors(h))) return rc;
      HIP_OK(hipEventSynchronize(h->scal_ev));
      collect_events(h);
      if (pcg_small) pcg_iters = (int)h->scal_host[kPcgIters];
      if (sm) sm->linear_solver_seconds += now_s() - t_ls;
      const double* sc = h->scal_host;
      const double mcc = sc[kMcc];
      bool step_valid = sc[kFail] == 0.0 && std::isfinite(mcc) && mcc > 0.0;
      cur.linear_solver_iterations = pcg_iters;
      if (sm) sm->total_linear_solver_iterations += pcg_iters;
      cur.step_is_valid = step_valid;
      if (!step_valid) {
        if (++consecutive_invalid >= o->max_num_consecutive_invalid_steps) {
          *termination = MLBA_FAILURE;
          break;
        }
        radius /= decrease_factor;
        decrease_factor *= 2.0;
        cur.cost = x_cost + fixed_cost;
        cur.gradient_max_norm = grad_max;
        cur.trust_region_radius = radius;
        cur.iteration_time_in_seconds = now_s() - t_iter;
        cur.cumulative_time_in_seconds = now_s() - t_start;
        push_iteration(sm, cur);
        if (sm) sm->num_unsuccessful_steps++;
      } else {
        consecutive_invalid = 0;
        const double candidate_cost = sc[kCandCost];
        const double x_norm = std::sqrt(sc[kXV] + sc[kXL]);
        const double step_norm = std::sqrt(sc[kWW] + sc[kUU]);
        cur.step_norm = step_norm;  // tangent step norm
        if (step_norm <= o->parameter_tolerance * (x_norm + o->parameter_tolerance)) {
          *termination = MLBA_CONVERGENCE;
          break;
        }
        cur.cost_change = x_cost - candidate_cost;
        if (std::fabs(cur.cost_change) <= o->function_tolerance * x_cost) {
          *termination = MLBA_CONVERGENCE;
          break;
        }
        cur.relative_decrease = (x_cost - candidate_cost) / mcc;
        if (cur.relative_decrease > o->min_relative_decrease) {
          std::swap(h->vert.p, h->vert_cand.p);
          std::swap(h->lm.p, h->lm_cand.p);
          std::swap(h->vR.p, h->vR_cand.p);
          const double t_ev = now_s();
          hipEvent_t e_lin = nullptr;
          if ((rc = linearize(h, o, false, &e_lin))) return rc;
          const hipEvent_t e_fac = stop_event(h);
          schur_factors(h, e_fac);
          time_span(h, MLBA_KERNEL_SCHUR_FACTORS, e_lin, e_fac);
          if ((rc = read_scalars(h))) return rc;
          if (sm) sm->evaluate_seconds += now_s() - t_ev;
          x_cost = h->scal_host[kCost];
          grad_max = h->scal_host[kGradMax];
          cur.step_is_successful = 1;
          cur.cost = x_cost + fixed_cost;
          cur.gradient_max_norm = grad_max;
          const double q = 2.0 * cur.relative_decrease - 1.0;
          radius = std::min(o->max_trust_region_radius, radius / std::max(1.0 / 3.0, 1.0 - q * q * q));
          decrease_factor = 2.0;
          if (sm) sm->num_successful_steps++;
        } else {
          radius /= decrease_factor;
          decrease_factor *= 2.0;
          cur.cost = candidate_cost + fixed_cost;
          cur.gradient_max_norm = grad_max;
          if (sm) sm->num_unsuccessful_steps++;
        }
        cur.trust_region_radius = radius;
        cur.iteration_time_in_seconds = now_s() - t_iter;
        cur.cumulative_time_in_seconds = now_s() - t_start;
        push_iteration(sm, cur);
      }
      if (now_s() - t_start > o->max_solver_time_in_seconds) { *termination = MLBA_NO_CONVERGENCE; break; }
      if (iteration >= o->max_num_iterations) { *termination = MLBA_NO_CONVERGENCE; break; }
      if (cur.step_is_successful && cur.gradient_max_norm <= o->gradient_tolerance) {
        *termination = MLBA_CONVERGENCE;
        break;
      }
      if (radius <= o->min_trust_region_radius) { *termination = MLBA_CONVERGENCE; break; }
    }
  }
  *last_radius = radius;
done:
  if (sm) {
    sm->final_cost = x_cost + fixed_cost;
    sm->lm_loop_seconds += now_s() - t_start;
  }
  return MLBA_OK;
}

void reset_summary(mlba_summary* sm) {
  if (!sm) return;
  for (int k = 0; k < MLBA_NUM_KERNELS; ++k) { sm->kernel_ms[k] = 0.0; sm->kernel_launches[k] = 0; }
  sm->num_iterations = 0;
  sm->num_successful_steps = sm->num_unsuccessful_steps = 0;
  sm->num_removed_landmarks = 0;
  sm->lm_loop_seconds = sm->evaluate_seconds = sm->linear_solver_seconds = 0.0;
  sm->total_linear_solver_iterations = 0;
  sm->initial_cost = sm->final_cost = sm->fixed_cost = 0.0;
}

int validate_options(mlba_handle* h, const mlba_options* o) {
  if (!o) return set_err(h, MLBA_EINVAL, "options is NULL");
  if (o->loss_type < 0 || o->loss_type > 2) return set_err(h, MLBA_EINVAL, "unknown loss_type");
  if (o->linear_solver_type != MLBA_SOLVER_SCHUR_PCG) return set_err(h, MLBA_EINVAL, "unknown linear_solver_type");
  if (o->jacobian_fp32 != 0 && o->jacobian_fp32 != 1) return set_err(h, MLBA_EINVAL, "jacobian_fp32 must be 0 or 1");
  if (o->pcg_preconditioner < MLBA_PRECOND_DEFLATED || o->pcg_preconditioner > MLBA_PRECOND_LEARNED_DEFLATED)
    return set_err(h, MLBA_EINVAL, "unknown pcg_preconditioner");
  if ((o->pcg_preconditioner == MLBA_PRECOND_LEARNED || o->pcg_preconditioner == MLBA_PRECOND_LEARNED_DEFLATED) &&
      !h->lp_model)
    return set_err(h, MLBA_ESTATE, "learned preconditioner without a model (mlba_set_preconditioner_model)");
  if (!(o->initial_trust_region_radius > 0.0)) return set_err(h, MLBA_EINVAL, "initial_trust_region_radius <= 0");
  if (o->loss_type == MLBA_LOSS_CAUCHY && !(o->loss_scale_px > 0.0)) return set_err(h, MLBA_EINVAL, "loss_scale_px <= 0");
  return check_topology(h);
}

int count_active_obs(const mlba_handle* h) {
  int n = 0;
  for (int o = 0; o < h->N; ++o) n += h->lm_active[h->s_landmark[o]] ? 1 : 0;
  return n;
}

}  // namespace

// =================================================================== C ABI

extern "C" {

int32_t mlba_abi_version(void) { return MLBA_ABI_VERSION; }

void mlba_options_init(mlba_options* o) {
  if (!o) return;
  std::memset(o, 0, sizeof(*o));
  o->max_num_iterations = 30;
  o->use_jacobi_scaling = 1;
  o->max_solver_time_in_seconds = 1e6;
  o->function_tolerance = 1e-12;
  o->gradient_tolerance = 1e-10;
  o->parameter_tolerance = 1e-8;
  o->initial_trust_region_radius = 1e5;
  o->max_trust_region_radius = 1e20;
  o->min_trust_region_radius = 1e-32;
  o->min_relative_decrease = 1e-3;
  o->min_lm_diagonal = 1e-6;
  o->max_lm_diagonal = 1e32;
  o->max_num_consecutive_invalid_steps = 5;
  o->loss_type = MLBA_LOSS_MAPLAB_HUBER;
  o->loss_scale_px = 1.0;
  o->linear_solver_type = MLBA_SOLVER_SCHUR_PCG;
  o->pcg_max_iterations = 500;
  o->pcg_relative_tolerance = 1e-10;
  o->reject_outliers_every_n_iters = 3;
  o->use_reprojection_error = 0;
  o->max_reprojection_error_px = 50.0;
}

const char* mlba_last_error(const mlba_handle* h) { return h ? h->err.c_str() : g_create_error.c_str(); }

// h is the caller's, who deletes it if this throws.
static int32_t create_handle(const mlba_problem_desc* d, mlba_handle** out, mlba_handle*& h) {
  if (!d || !out) return set_err(h, MLBA_EINVAL, "NULL argument");
  *out = nullptr;
  const int N = d->num_observations, L = d->num_landmarks, P = d->num_vertices, C = d->num_cameras,
            M = d->num_missions;
  if (N < 0 || L < 0 || P < 0 || C < 0 || M < 0) return set_err(h, MLBA_EINVAL, "negative size");
  if ((N > 0 && (!d->obs_vertex || !d->obs_landmark || !d->obs_camera || !d->obs_keypoint || !d->obs_sigma)) ||
      (P > 0 && (!d->vertex_q_IM__M_p_MI || !d->vertex_mission)) ||
      (L > 0 && (!d->landmark_p_B || !d->landmark_store_vertex)) ||
      (C > 0 && (!d->camera_q_CI__C_p_CI || !d->camera_intrinsics || !d->camera_distortion ||
                 !d->camera_distortion_type || !d->camera_resolution)) ||
      (M > 0 && !d->baseframe_q_GM__G_p_GM))
    return set_err(h, MLBA_EINVAL, "NULL array in problem description");
  if ((int64_t)C >= (1 << 23)) return set_err(h, MLBA_EINVAL, "too many cameras");
  for (int o = 0; o < N; ++o) {
    if (d->obs_vertex[o] < 0 || d->obs_vertex[o] >= P) return set_err(h, MLBA_EINVAL, "obs_vertex out of range");
    if (d->obs_landmark[o] < 0 || d->obs_landmark[o] >= L) return set_err(h, MLBA_EINVAL, "obs_landmark out of range");
    if (d->obs_camera[o] < 0 || d->obs_camera[o] >= C) return set_err(h, MLBA_EINVAL, "obs_camera out of range");
    if (!(d->obs_sigma[o] > 0.0)) return set_err(h, MLBA_EINVAL, "pixel sigma must be > 0");
    if (!std::isfinite(d->obs_keypoint[2 * o]) || !std::isfinite(d->obs_keypoint[2 * o + 1]))
      return set_err(h, MLBA_EINVAL, "non-finite keypoint");
  }
  for (int l = 0; l < L; ++l)
    if (d->landmark_store_vertex[l] < 0 || d->landmark_store_vertex[l] >= P)
      return set_err(h, MLBA_EINVAL, "landmark_store_vertex out of range");
  for (int v = 0; v < P; ++v) {
    if (d->vertex_mission[v] < 0 || d->vertex_mission[v] >= M) return set_err(h, MLBA_EINVAL, "vertex_mission out of range");
    if (!valid_quaternion(d->vertex_q_IM__M_p_MI + 7 * v)) return set_err(h, MLBA_ESTATE, "vertex quaternion not unit or w < 0");
  }
  for (int c = 0; c < C; ++c) {
    const int dt = d->camera_distortion_type[c];
    if (dt < 0 || dt > 3) return set_err(h, MLBA_EINVAL, "unknown distortion type");
    if (dt == kDistFisheye) {
      // FisheyeDistortion::areParametersValid (distortion-fisheye.cc:145-156).
      const double w = d->camera_distortion[4 * c];
      if (!(std::fabs(w) < 1e-16 || (w >= 0.5 && w <= 1.5)))
        return set_err(h, MLBA_EINVAL, "fisheye distortion w outside [0.5, 1.5]");
    }
    if (!valid_quaternion(d->camera_q_CI__C_p_CI + 7 * c)) return set_err(h, MLBA_ESTATE, "camera quaternion invalid");
    const int model = d->camera_model ? d->camera_model[c] : MLBA_CAMERA_PINHOLE;
    if (model != MLBA_CAMERA_PINHOLE && model != MLBA_CAMERA_UNIFIED_PROJECTION)
      return set_err(h, MLBA_EINVAL, "unknown camera model");
    if (model == MLBA_CAMERA_UNIFIED_PROJECTION) {
      // UnifiedProjectionCamera::areParametersValid (camera-unified-projection.cc:294-301).
      const double xi = d->camera_xi ? d->camera_xi[c] : 0.0;
      const double* in = d->camera_intrinsics + 4 * c;
      if (!(std::isfinite(xi) && xi >= 0.0 && in[0] > 0.0 && in[1] > 0.0 && in[2] > 0.0 && in[3] > 0.0))
        return set_err(h, MLBA_EINVAL, "unified-projection camera needs xi >= 0 and positive fu fv cu cv");
    }
  }
  for (int m = 0; m < M; ++m)
    if (!valid_quaternion(d->baseframe_q_GM__G_p_GM + 7 * m)) return set_err(h, MLBA_ESTATE, "baseframe quaternion invalid");

  h = new (std::nothrow) mlba_handle();
  if (!h) return set_err(nullptr, MLBA_ENOMEM, "host allocation failed");
  auto fail_out = [&](int code) {
    g_create_error = h->err;
    delete h;
    return code;
  };
  if (hipGetDevice(&h->device) != hipSuccess) h->device = 0;
  if (hipStreamCreateWithFlags(&h->stream, hipStreamNonBlocking) != hipSuccess) {
    h->err = "hipStreamCreate failed";
    return fail_out(MLBA_EDEVICE);
  }
  h->N = N; h->L = L; h->P = P; h->C = C; h->M = M;
  // Sort observations by (landmark, vertex, caller index).
  h->perm.resize(N);
  for (int o = 0; o < N; ++o) h->perm[o] = o;
  std::stable_sort(h->perm.begin(), h->perm.end(), [&](int a, int b) {
    if (d->obs_landmark[a] != d->obs_landmark[b]) return d->obs_landmark[a] < d->obs_landmark[b];
    return d->obs_vertex[a] < d->obs_vertex[b];
  });
  h->s_landmark.resize(N); h->s_vertex.resize(N); h->s_camera.resize(N); h->s_type.resize(N);
  std::vector<double> kp(2 * (size_t)N), sinv(N);
  h->lm_begin.assign(L + 1, 0);
  for (int k = 0; k < N; ++k) {
    const int o = h->perm[k];
    const int l = d->obs_landmark[o], v = d->obs_vertex[o];
    const int s = d->landmark_store_vertex[l];
    h->s_landmark[k] = l;
    h->s_vertex[k] = v;
    h->s_camera[k] = d->obs_camera[o];
    h->s_type[k] = v == s ? kTypeKeyframe : (d->vertex_mission[v] == d->vertex_mission[s] ? kTypeMission : kTypeGlobal);
    kp[2 * k] = d->obs_keypoint[2 * o];
    kp[2 * k + 1] = d->obs_keypoint[2 * o + 1];
    sinv[k] = 1.0 / d->obs_sigma[o];
    h->lm_begin[l + 1]++;
  }
  for (int l = 0; l < L; ++l) h->lm_begin[l + 1] += h->lm_begin[l];
  h->lm_anchor.assign(d->landmark_store_vertex, d->landmark_store_vertex + L);
  h->vertex_mission.assign(d->vertex_mission, d->vertex_mission + P);
  h->lm_active.assign(L, 1);
  h->lm_const.assign(L, 0);
  h->vertex_const.assign(P, 0);
  if (d->landmark_constant) for (int l = 0; l < L; ++l) h->lm_const[l] = d->landmark_constant[l] ? 1 : 0;
  if (d->vertex_constant) for (int v = 0; v < P; ++v) h->vertex_const[v] = d->vertex_constant[v] ? 1 : 0;
  h->h_baseframes.assign(d->baseframe_q_GM__G_p_GM, d->baseframe_q_GM__G_p_GM + 7 * (size_t)M);
  h->h_cam_q.assign(d->camera_q_CI__C_p_CI, d->camera_q_CI__C_p_CI + 7 * (size_t)C);
  std::vector<DevCamera> cams(C);
  for (int c = 0; c < C; ++c) {
    DevCamera& k = cams[c];
    std::memset(&k, 0, sizeof(k));
    rot_jpl(d->camera_q_CI__C_p_CI + 7 * c, k.R_C_I);
    for (int i = 0; i < 3; ++i) k.p_C_I[i] = d->camera_q_CI__C_p_CI[7 * c + 4 + i];
    for (int i = 0; i < 4; ++i) { k.intr[i] = d->camera_intrinsics[4 * c + i]; k.dist[i] = d->camera_distortion[4 * c + i]; }
    k.width = d->camera_resolution[2 * c];
    k.height = d->camera_resolution[2 * c + 1];
    k.dist_type = d->camera_distortion_type[c];
    k.model = d->camera_model ? d->camera_model[c] : MLBA_CAMERA_PINHOLE;
    k.xi = (k.model == MLBA_CAMERA_UNIFIED_PROJECTION && d->camera_xi) ? d->camera_xi[c] : 0.0;
  }
  std::vector<double> mT(12 * (size_t)M);
  for (int m = 0; m < M; ++m) {
    rot_jpl(d->baseframe_q_GM__G_p_GM + 7 * m, &mT[12 * m]);  // R_G_M
    for (int i = 0; i < 3; ++i) mT[12 * m + 9 + i] = d->baseframe_q_GM__G_p_GM[7 * m + 4 + i];
  }
  int rc;
  if ((rc = upload(h, h->obs_kp, kp.data(), kp.size())) || (rc = upload(h, h->obs_sinv, sinv.data(), sinv.size())) ||
      (rc = upload(h, h->obs_vertex, h->s_vertex.data(), (size_t)N)) ||
      (rc = upload(h, h->obs_landmark, h->s_landmark.data(), (size_t)N)) ||
      (rc = upload(h, h->perm_d, h->perm.data(), (size_t)N)) ||
      (rc = upload(h, h->lm_begin_d, h->lm_begin.data(), h->lm_begin.size())) ||
      (rc = upload(h, h->lm_anchor_d, h->lm_anchor.data(), (size_t)L)) ||
      (rc = upload(h, h->vertex_mission_d, h->vertex_mission.data(), (size_t)P)) ||
      (rc = upload(h, h->cams, (h->h_cams = cams).data(), cams.size())) ||
      (rc = upload(h, h->mission_T, mT.data(), mT.size())) ||
      (rc = upload(h, h->baseframes, h->h_baseframes.data(), h->h_baseframes.size())) ||
      (rc = upload(h, h->cam_q, h->h_cam_q.data(), h->h_cam_q.size())) ||
      (rc = upload(h, h->vert, d->vertex_q_IM__M_p_MI, 7 * (size_t)P)) ||
      (rc = upload(h, h->lm, d->landmark_p_B, 3 * (size_t)L)))
    return fail_out(rc);
  const bool ok = h->obs_rec.alloc((size_t)kObsRecord * N) && h->vert_cand.alloc(7 * (size_t)P) &&
                  h->vR.alloc(12 * (size_t)P) && h->vR_cand.alloc(12 * (size_t)P) && h->lm_cand.alloc(3 * (size_t)L) &&
                  h->lm_acc.alloc((size_t)kLmAcc * L) && h->lm_anc.alloc((size_t)kLmAnchor * L) && h->lm_scale.alloc(3 * (size_t)L) &&
                  h->lm_z.alloc(kLmZ * (size_t)L) && h->lm_u.alloc(3 * (size_t)L) && h->scal.alloc(kNumSlots) &&
                  h->fail.alloc(1) && h->pcg_state.alloc(pcg_state_bytes());
  if (!ok) { h->err = "device allocation failed"; return fail_out(MLBA_ENOMEM); }
  if (hipHostMalloc(&h->pcg_host, pcg_state_bytes(), hipHostMallocDefault) != hipSuccess ||
      hipHostMalloc((void**)&h->scal_host, kNumSlots * sizeof(double), hipHostMallocDefault) != hipSuccess ||
      hipEventCreateWithFlags(&h->scal_ev, hipEventDisableTiming) != hipSuccess) {
    h->err = "pinned host allocation failed";
    return fail_out(MLBA_ENOMEM);
  }
  if ((rc = build_topology(h))) return fail_out(rc);
  *out = h;
  return MLBA_OK;
}

int32_t mlba_create(const mlba_problem_desc* d, mlba_handle** out) {
  mlba_handle* h = nullptr;
  try {
    return create_handle(d, out, h);
  } catch (...) {
    delete h;
    return host_out_of_memory(nullptr);
  }
}

int32_t mlba_destroy(mlba_handle* h) {
  if (!h) return MLBA_EINVAL;
  if (h->stream) (void)hipStreamSynchronize(h->stream);
  delete h;
  return MLBA_OK;
}

int32_t mlba_upload_state(mlba_handle* h, const double* vertices, const double* landmarks) {
  if (!h) return MLBA_EINVAL;
  if (vertices)
    for (int v = 0; v < h->P; ++v)
      if (!valid_quaternion(vertices + 7 * v)) return set_err(h, MLBA_ESTATE, "vertex quaternion not unit or w < 0");
  if (vertices) HIP_OK(hipMemcpyAsync(h->vert.p, vertices, 7 * sizeof(double) * h->P, hipMemcpyHostToDevice, h->stream));
  if (landmarks) HIP_OK(hipMemcpyAsync(h->lm.p, landmarks, 3 * sizeof(double) * h->L, hipMemcpyHostToDevice, h->stream));
  HIP_OK(hipStreamSynchronize(h->stream));
  // A new state starts the linear solver afresh: no recycled deflation
  // columns or iteration estimate carried over from earlier solves, so that
  // a solve from an uploaded state repeats bit for bit.
  h->ritz_nr = 0;
  h->ritz_stage = 0;
  h->pcg_last_iters[0] = h->pcg_last_iters[1] = 0;
  return MLBA_OK;
}

int32_t mlba_download_state(const mlba_handle* hc, double* vertices, double* landmarks) {
  mlba_handle* h = const_cast<mlba_handle*>(hc);
  if (!h) return MLBA_EINVAL;
  if (vertices) HIP_OK(hipMemcpyAsync(vertices, h->vert.p, 7 * sizeof(double) * h->P, hipMemcpyDeviceToHost, h->stream));
  if (landmarks) HIP_OK(hipMemcpyAsync(landmarks, h->lm.p, 3 * sizeof(double) * h->L, hipMemcpyDeviceToHost, h->stream));
  HIP_OK(hipStreamSynchronize(h->stream));
  return MLBA_OK;
}

int32_t mlba_set_landmark_active(mlba_handle* h, const uint8_t* mask) {
  if (!h || !mask) return MLBA_EINVAL;
  try {
    for (int l = 0; l < h->L; ++l) h->lm_active[l] = mask[l] ? 1 : 0;
    return build_topology(h);
  } catch (...) {
    return host_out_of_memory(h);
  }
}

int32_t mlba_get_landmark_active(const mlba_handle* h, uint8_t* mask) {
  if (!h || !mask) return MLBA_EINVAL;
  for (int l = 0; l < h->L; ++l) mask[l] = h->lm_active[l];
  return MLBA_OK;
}

void mlba_quality_options_init(mlba_quality_options* o) {
  if (!o) return;
  o->min_observers = 4;
  o->reserved0 = 0;
  o->min_observation_angle_deg = 5.0;
  o->max_distance_from_closest_observer = 40.0;
  o->min_distance_from_closest_observer = 0.05;
  o->max_reprojection_error_px = -1.0;
}

int32_t mlba_landmark_quality(mlba_handle* h, const mlba_quality_options* o, uint8_t* good) {
  if (!h || !o || !good) return h ? set_err(h, MLBA_EINVAL, "null argument") : MLBA_EINVAL;
  if (const int rc = check_topology(h)) return rc;
  if (o->min_observers < 0) return set_err(h, MLBA_EINVAL, "min_observers must be >= 0");
  if (h->L == 0) return MLBA_OK;
  hipStream_t s = h->stream;
  DBuf<uint8_t> d;
  if (!d.alloc(h->L)) return set_err(h, MLBA_ENOMEM, "device allocation failed");
  launch_vertex_prep(s, h->P, h->vert.p, h->vR.p);
  launch_landmark_quality(s, h->topo, h->vert.p, h->vR.p, h->lm.p, o->min_observers, o->min_observation_angle_deg,
                          o->max_distance_from_closest_observer, o->min_distance_from_closest_observer,
                          o->max_reprojection_error_px, d.p);
  HIP_OK(hipGetLastError());
  HIP_OK(hipMemcpyAsync(good, d.p, h->L, hipMemcpyDeviceToHost, s));
  HIP_OK(hipStreamSynchronize(s));
  return MLBA_OK;
}

// Jacobian blocks as the caller's arrays hold them: the wanted ones one after
// the other from base, N x 2 x size each.
static EvalOut eval_blocks(double* base, size_t N, const int* sizes, int nblocks, double* const* jacobians) {
  EvalOut out{};
  for (int b = 0; b < nblocks; ++b) {
    if (!jacobians || !jacobians[b]) continue;
    out.block[b] = base;
    out.stride[b] = 2 * sizes[b];
    base += N * (size_t)out.stride[b];
  }
  return out;
}

// Queues the copies of the wanted blocks into the caller's arrays.
static int copy_eval_blocks(mlba_handle* h, const EvalOut& out, int nblocks, double* const* jacobians) {
  for (int b = 0; b < nblocks; ++b)
    if (out.block[b] && h->N)
      HIP_OK(hipMemcpyAsync(jacobians[b], out.block[b], sizeof(double) * out.stride[b] * (size_t)h->N,
                            hipMemcpyDeviceToHost, h->stream));
  return MLBA_OK;
}

int32_t mlba_evaluate(mlba_handle* h, int32_t flags, const mlba_options* options, double* residuals,
                      double* const* jacobians, double* cost) {
  if (!h) return MLBA_EINVAL;
  if (flags & ~(MLBA_EVAL_TANGENT | MLBA_EVAL_WITH_XI)) return set_err(h, MLBA_EINVAL, "unknown flags");
  if (const int rc = check_topology(h)) return rc;
  const bool tangent = (flags & MLBA_EVAL_TANGENT) != 0;
  const int nblocks = (flags & MLBA_EVAL_WITH_XI) ? 10 : 9;
  static const int amb[10] = {3, 7, 7, 7, 7, 4, 3, 4, 4, 1};
  static const int tng[10] = {3, 6, 6, 6, 6, 3, 3, 4, 4, 1};
  const int* sz = tangent ? tng : amb;
  size_t width = 0;  // doubles of the wanted blocks of one observation
  for (int b = 0; b < nblocks; ++b)
    if (jacobians && jacobians[b]) width += 2 * (size_t)sz[b];
  hipStream_t s = h->stream;
  launch_vertex_prep(s, h->P, h->vert.p, h->vR.p);
  DBuf<double> res_d, jac_d;
  if (residuals && !res_d.alloc(2 * (size_t)h->N)) return set_err(h, MLBA_ENOMEM, "device allocation failed");
  if (width && !jac_d.alloc(width * h->N)) return set_err(h, MLBA_ENOMEM, "device allocation failed");
  const EvalOut out = eval_blocks(jac_d.p, h->N, sz, nblocks, jacobians);
  launch_evaluate_full(s, h->topo, h->vert.p, h->vR.p, h->lm.p, h->baseframes.p, h->cam_q.p, tangent, h->perm_d.p,
                       residuals ? res_d.p : nullptr, out, width != 0);
  if (cost) {
    mlba_options defaults;
    mlba_options_init(&defaults);
    const mlba_options* o = options ? options : &defaults;
    launch_linearize(s, false, h->tiles, h->topo, h->vert.p, h->vR.p, h->lm.p, make_loss(o), h->tile_begin.p,
                     nullptr, nullptr, nullptr, h->tile_cost2.p);
    launch_reduce(s, h->tiles, 2, 0, false, h->tile_cost2.p, h->scal.p + kCandCost);
    launch_reduce(s, h->tiles, 2, 1, false, h->tile_cost2.p, h->scal.p + kCandFixed);
  }
  HIP_OK(hipGetLastError());
  if (residuals)
    HIP_OK(hipMemcpyAsync(residuals, res_d.p, 2 * sizeof(double) * h->N, hipMemcpyDeviceToHost, s));
  int rc = copy_eval_blocks(h, out, nblocks, jacobians);
  if (rc) return rc;
  if (cost) {
    if ((rc = read_scalars(h))) return rc;
    *cost = h->scal_host[kCandCost] + h->scal_host[kCandFixed];
  }
  HIP_OK(hipStreamSynchronize(s));
  return MLBA_OK;
}

// ------------------------------------------------------------ evaluate without allocation

// Staging of mlba_evaluate_noalloc: one array per device for the whole
// process (residuals, then the Jacobian records of every observation).
// Host code never uses its name as an address: the device address comes
// from hipGetSymbolAddress, once per device, with that device current.
static __device__ __align__(256) double scratch[MLBA_NOALLOC_SCRATCH_BYTES / sizeof(double)];

constexpr int kMaxDevices = 64;
static std::mutex g_scratch_mu[kMaxDevices];   // one call at a time per device holds its array
static double* g_scratch_ptr[kMaxDevices] = {};

int32_t mlba_evaluate_noalloc(mlba_handle* h, int32_t flags, const mlba_options* options, double* residuals,
                              double* const* jacobians, double* cost) {
  if (!h) return MLBA_EINVAL;
  if (flags & ~(MLBA_EVAL_TANGENT | MLBA_EVAL_WITH_XI)) return set_err(h, MLBA_EINVAL, "unknown flags");
  if (const int rc = check_topology(h)) return rc;
  if (h->device < 0 || h->device >= kMaxDevices) return set_err(h, MLBA_EINVAL, "device index out of range");
  const bool tangent = (flags & MLBA_EVAL_TANGENT) != 0;
  const int nblocks = (flags & MLBA_EVAL_WITH_XI) ? 10 : 9;
  static const int amb[10] = {3, 7, 7, 7, 7, 4, 3, 4, 4, 1};
  static const int tng[10] = {3, 6, 6, 6, 6, 3, 3, 4, 4, 1};
  const int* sz = tangent ? tng : amb;
  int stride = 0;
  uint32_t mask = 0;
  for (int b = 0; b < 10; ++b) {
    stride += 2 * sz[b];
    if (b < nblocks && jacobians && jacobians[b]) mask |= 1u << b;
  }
  const size_t res_n = residuals ? 2 * (size_t)h->N : 0;
  const size_t need = sizeof(double) * (res_n + (mask ? (size_t)stride * h->N : 0));
  if (need > MLBA_NOALLOC_SCRATCH_BYTES)
    return set_err(h, MLBA_EINVAL, "mlba_evaluate_noalloc: " + std::to_string(need) +
                                       " bytes of staging exceed the fixed " +
                                       std::to_string((size_t)MLBA_NOALLOC_SCRATCH_BYTES) + "-byte array");
  std::lock_guard<std::mutex> lock(g_scratch_mu[h->device]);
  int prev = 0;
  HIP_OK(hipGetDevice(&prev));
  if (prev != h->device) HIP_OK(hipSetDevice(h->device));
  // On every return the stream's work on the array has finished before the
  // lock is released, and the caller's device is current again.
  struct Restore {
    int dev, prev;
    hipStream_t s;
    ~Restore() {
      (void)hipStreamSynchronize(s);
      if (prev != dev) (void)hipSetDevice(prev);
    }
  } restore{h->device, prev, h->stream};
  if (!g_scratch_ptr[h->device]) {
    void* ptr = nullptr;
    HIP_OK(hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)));
    g_scratch_ptr[h->device] = static_cast<double*>(ptr);
  }
  double* res_d = g_scratch_ptr[h->device];
  double* jac_d = res_d + res_n;
  hipStream_t s = h->stream;
  launch_vertex_prep(s, h->P, h->vert.p, h->vR.p);
  // The wanted blocks take no more than the room asked for.
  const EvalOut out = eval_blocks(jac_d, h->N, sz, nblocks, jacobians);
  launch_evaluate_full(s, h->topo, h->vert.p, h->vR.p, h->lm.p, h->baseframes.p, h->cam_q.p, tangent, h->perm_d.p,
                       residuals ? res_d : nullptr, out, mask != 0);
  if (cost) {
    mlba_options defaults;
    mlba_options_init(&defaults);
    const mlba_options* o = options ? options : &defaults;
    launch_linearize(s, false, h->tiles, h->topo, h->vert.p, h->vR.p, h->lm.p, make_loss(o), h->tile_begin.p,
                     nullptr, nullptr, nullptr, h->tile_cost2.p);
    launch_reduce(s, h->tiles, 2, 0, false, h->tile_cost2.p, h->scal.p + kCandCost);
    launch_reduce(s, h->tiles, 2, 1, false, h->tile_cost2.p, h->scal.p + kCandFixed);
  }
  HIP_OK(hipGetLastError());
  if (residuals && h->N)
    HIP_OK(hipMemcpyAsync(residuals, res_d, 2 * sizeof(double) * h->N, hipMemcpyDeviceToHost, s));
  if (const int rc = copy_eval_blocks(h, out, nblocks, jacobians)) return rc;
  if (cost) {
    int rc = read_scalars(h);
    if (rc) return rc;
    *cost = h->scal_host[kCandCost] + h->scal_host[kCandFixed];
  }
  HIP_OK(hipStreamSynchronize(s));
  return MLBA_OK;
}

// ------------------------------------------------------------ learned preconditioner (C ABI)

int32_t mlba_set_preconditioner_model(mlba_handle* h, const float* params, const float* norm) {
  if (!h || !params || !norm) return MLBA_EINVAL;
  for (int k = 0; k < kGnnNormFloats; ++k)
    if (!std::isfinite(norm[k]) || (((k / kLpNodeFeatures == 1 && k < 2 * kLpNodeFeatures) ||
                                     k >= 2 * kLpNodeFeatures + kLpEdgeFeatures) && !(norm[k] > 0.0f)))
      return set_err(h, MLBA_EINVAL, "feature normalization: non-finite value or std <= 0");
  for (int k = 0; k < kGnnParams; ++k)
    if (!std::isfinite(params[k])) return set_err(h, MLBA_EINVAL, "non-finite network parameter");
  int rc;
  if ((rc = upload(h, h->lp_params, params, kGnnParams))) return rc;
  if ((rc = upload(h, h->lp_norm, norm, kGnnNormFloats))) return rc;
  HIP_OK(hipStreamSynchronize(h->stream));
  h->lp_model = true;
  return MLBA_OK;
}

int32_t mlba_get_preconditioner_stats(const mlba_handle* h, mlba_preconditioner_stats* st) {
  if (!h || !st) return MLBA_EINVAL;
  *st = h->lp_stats;
  return MLBA_OK;
}

int32_t mlba_reset_preconditioner_stats(mlba_handle* h) {
  if (!h) return MLBA_EINVAL;
  h->lp_stats = mlba_preconditioner_stats{};
  return MLBA_OK;
}

int32_t mlba_rcs_size(const mlba_handle* h, int32_t* rows, int32_t* slots) {
  if (!h || !rows || !slots) return MLBA_EINVAL;
  *rows = h->Pvar;
  *slots = h->nnzb;
  return MLBA_OK;
}

}  // extern "C"

namespace {

// S and its right-hand side at the current state with damping diag / radius
// (the linear system of an LM iteration), the state unchanged.
int build_rcs(mlba_handle* h, const mlba_options* o, double radius) {
  hipStream_t s = h->stream;
  int rc;
  if (!(radius > 0.0)) return set_err(h, MLBA_EINVAL, "radius <= 0");
  h->f32_jac = o->jacobian_fp32 != 0;
  if ((rc = linearize(h, o))) return rc;
  launch_jacobi_scaling(s, h->Pvar, h->L, o->use_jacobi_scaling, h->pose_diag.p, h->lm_acc.p, h->pose_scale.p,
                        h->lm_scale.p);
  schur_factors(h);
  HIP_OK(hipMemsetAsync(h->fail.p, 0, sizeof(int32_t), s));
  const double inv_mu = 1.0 / radius;
  launch_landmark_prep(s, h->topo, h->lm_acc.p, h->lm_scale.p, inv_mu, o->min_lm_diagonal, o->max_lm_diagonal,
                       h->lm_z.p, h->lm_anc.p, h->fail.p);
  launch_schur_blocks(s, h->topo, h->tdev, h->n_upper, h->ublk.p, h->gf.p, h->gk.p, h->lm_z.p, h->lm_anc.p,
                      h->vR.p, h->pose_scale.p, h->pose_diag.p, h->pose_jtj.p, inv_mu, o->min_lm_diagonal,
                      o->max_lm_diagonal, h->schur_partial.p, h->S.p, h->rhs.p, h->sched_waves, h->sched_xcd);
  HIP_OK(hipGetLastError());
  return MLBA_OK;
}

int read_fail(mlba_handle* h, int32_t* fail) {
  HIP_OK(hipMemcpyAsync(fail, h->fail.p, sizeof(int32_t), hipMemcpyDeviceToHost, h->stream));
  HIP_OK(hipStreamSynchronize(h->stream));
  return MLBA_OK;
}

}  // namespace

extern "C" {

int32_t mlba_rcs_system(mlba_handle* h, const mlba_options* o, double radius, int32_t* row_ptr, int32_t* col,
                        double* blocks, double* rhs) {
  if (!h) return MLBA_EINVAL;
  if (!row_ptr || !col || !blocks || !rhs) return set_err(h, MLBA_EINVAL, "NULL output");
  int rc = validate_options(h, o);
  if (rc) return rc;
  if ((rc = build_rcs(h, o, radius))) return rc;
  hipStream_t s = h->stream;
  if (h->nnzb > 0)
    HIP_OK(hipMemcpyAsync(blocks, h->S.p, sizeof(double) * 36 * (size_t)h->nnzb, hipMemcpyDeviceToHost, s));
  if (h->Pvar > 0) HIP_OK(hipMemcpyAsync(rhs, h->rhs.p, sizeof(double) * 6 * (size_t)h->Pvar, hipMemcpyDeviceToHost, s));
  HIP_OK(hipStreamSynchronize(s));
  std::memcpy(row_ptr, h->h_row_ptr.data(), sizeof(int32_t) * h->h_row_ptr.size());
  std::memcpy(col, h->h_col_var.data(), sizeof(int32_t) * h->h_col_var.size());
  return MLBA_OK;
}

int32_t mlba_rcs_records(mlba_handle* h, const mlba_options* o, double radius, int32_t* row_ptr, int32_t* col,
                         int32_t* rev, float* node_features, float* edge_features, float* qc) {
  if (!h) return MLBA_EINVAL;
  if (!row_ptr || !col || !rev || !node_features || !edge_features || !qc)
    return set_err(h, MLBA_EINVAL, "NULL output");
  int rc = validate_options(h, o);
  if (rc) return rc;
  if ((rc = build_rcs(h, o, radius))) return rc;
  if ((rc = lp_ensure(h, true, true))) return rc;
  hipStream_t s = h->stream;
  const LpSystem sys = lp_system(h);
  launch_lp_factor(s, sys, h->lp_linv.p, h->fail.p);
  int32_t fail = 0;
  if ((rc = read_fail(h, &fail))) return rc;
  if (fail) return set_err(h, MLBA_ESTATE, "a landmark or vertex block of the system is not positive definite");
  launch_lp_normalize(s, sys, h->lp_linv.p, h->lp_shat.p, h->lp_snorm.p);
  std::vector<float> ident(kGnnNormFloats, 0.0f);
  for (int k = kLpNodeFeatures; k < 2 * kLpNodeFeatures; ++k) ident[k] = 1.0f;
  for (int k = 2 * kLpNodeFeatures + kLpEdgeFeatures; k < kGnnNormFloats; ++k) ident[k] = 1.0f;
  DBuf<float> norm;
  if ((rc = upload(h, norm, ident.data(), ident.size()))) return rc;
  launch_lp_features(s, sys, h->pose_jtj.p, h->pose_scale.p, h->lp_snorm.p, h->lp_shared.p, norm.p, h->lp_nf.p,
                     h->lp_ef.p);
  if (!launch_lp_terms(s, sys, h->lp_max_lower_deg, kLpStoreT2, h->lp_shat.p, nullptr, nullptr, h->lp_t2.p,
                       h->lp_trace.p) ||
      !launch_lp_terms(s, sys, h->lp_max_lower_deg, kLpTraceT3, h->lp_shat.p, nullptr, nullptr, h->lp_t2.p,
                       h->lp_trace.p))
    return set_err(h, MLBA_EINVAL, "a row's lower neighbourhood does not fit the neighbourhood kernel");
  HIP_OK(hipGetLastError());
  const int P = h->Pvar, Z = h->nnzb;
  std::vector<float> tr(4 * (size_t)P);
  if (P) {
    HIP_OK(hipMemcpyAsync(node_features, h->lp_nf.p, sizeof(float) * kLpNodeFeatures * P, hipMemcpyDeviceToHost, s));
    HIP_OK(hipMemcpyAsync(tr.data(), h->lp_trace.p, sizeof(float) * 4 * P, hipMemcpyDeviceToHost, s));
  }
  if (Z) HIP_OK(hipMemcpyAsync(edge_features, h->lp_ef.p, sizeof(float) * kLpEdgeFeatures * Z, hipMemcpyDeviceToHost, s));
  HIP_OK(hipStreamSynchronize(s));
  std::memcpy(row_ptr, h->h_row_ptr.data(), sizeof(int32_t) * (P + 1));
  std::memcpy(col, h->h_col_var.data(), sizeof(int32_t) * Z);
  HIP_OK(hipMemcpy(rev, h->lp_tpos.p, sizeof(int32_t) * Z, hipMemcpyDeviceToHost));
  for (int i = 0; i < P; ++i) {
    const bool has = h->h_row_ptr[i] < Z && h->h_col_var[h->h_row_ptr[i]] < i;
    for (int k = 0; k < 4; ++k) qc[5 * (size_t)i + k] = has ? tr[4 * (size_t)i + k] : 0.0f;
    qc[5 * (size_t)i + 4] = has ? 1.0f : 0.0f;
  }
  return MLBA_OK;
}

int32_t mlba_rcs_pcg_iterations(mlba_handle* h, const mlba_options* o, double radius, int32_t preconditioner,
                                double tolerance, int32_t max_iterations, int32_t* iterations) {
  if (!h || !iterations) return MLBA_EINVAL;
  int rc = validate_options(h, o);
  if (rc) return rc;
  if (preconditioner < MLBA_PRECOND_DEFLATED || preconditioner > MLBA_PRECOND_LEARNED_DEFLATED ||
      !(tolerance > 0.0) || max_iterations <= 0)
    return set_err(h, MLBA_EINVAL, "preconditioner, tolerance or iteration cap");
  if ((preconditioner == MLBA_PRECOND_LEARNED || preconditioner == MLBA_PRECOND_LEARNED_DEFLATED) && !h->lp_model)
    return set_err(h, MLBA_ESTATE, "no preconditioner model");
  if ((rc = build_rcs(h, o, radius))) return rc;
  hipStream_t s = h->stream;
  *iterations = -1;
  if (h->Pvar == 0) { *iterations = 0; return MLBA_OK; }
  if (preconditioner == MLBA_PRECOND_DEFLATED) {
    launch_block_inverse(s, h->Pvar, h->diag_pos.p, h->S.p, h->Minv.p, h->fail.p);
    if ((rc = ensure_coarse_basis(h, o->pcg_coarse_nodes))) return rc;
    const int it = launch_pcg_deflated(s, pcg_buffers(h, 0, false), tolerance, max_iterations, kPcgPoll, kPcgPoll,
                                       nullptr, 0);
    if (it < 0) return set_err(h, MLBA_EDEVICE, "PCG launch failed");
    *iterations = it < max_iterations ? it : -1;
    return MLBA_OK;
  }
  if (preconditioner == MLBA_PRECOND_LEARNED_DEFLATED) {
    if ((rc = lp_ensure(h, true, false))) return rc;
    bool use_k = false;
    if ((rc = lp_setup(h, true, &use_k))) return rc;
    if (!use_k) return set_err(h, MLBA_EINVAL, "a row's lower neighbourhood does not fit the neighbourhood kernel");
    if ((rc = ensure_coarse_basis(h, o->pcg_coarse_nodes))) return rc;
    // No recycled columns and no Lanczos vectors: the recycling state is
    // left as it is.
    const int it = launch_pcg_deflated(s, lp_deflated_buffers(h), tolerance, max_iterations, kPcgPoll, kPcgPoll,
                                       nullptr, 0);
    if (it < 0) return set_err(h, MLBA_EDEVICE, "PCG launch failed");
    *iterations = it < max_iterations ? it : -1;
    return MLBA_OK;
  }
  const bool learned = preconditioner == MLBA_PRECOND_LEARNED;
  if ((rc = lp_ensure(h, learned, false))) return rc;
  bool use_k = false;
  if ((rc = lp_setup(h, learned, &use_k))) return rc;
  if (learned && !use_k) return set_err(h, MLBA_EINVAL, "a row's lower neighbourhood does not fit the neighbourhood kernel");
  int32_t conv = 0;
  const int it = launch_lp_pcg(s, lp_buffers(h, use_k), tolerance, max_iterations, kPcgPoll, &conv);
  if (it < 0) return set_err(h, MLBA_EDEVICE, "PCG launch failed");
  *iterations = conv ? it : -1;
  return MLBA_OK;
}

int32_t mlba_solve(mlba_handle* h, const mlba_options* o, mlba_summary* sm) {
  if (!h) return MLBA_EINVAL;
  int rc = validate_options(h, o);
  if (rc) return rc;
  reset_summary(sm);
  if (sm) sm->num_residual_blocks = count_active_obs(h);
  double radius = 0.0;
  int term = MLBA_NO_CONVERGENCE;
  h->ev_summary = sm;
  rc = minimize(h, o, o->initial_trust_region_radius, sm, &radius, &term);
  collect_events(h);
  h->ev_summary = nullptr;
  if (rc) return rc;
  if (sm) sm->termination_type = term;
  return MLBA_OK;
}

// outlier-rejection-solver.cc:28-103 and :142-182 on the device: every active
// landmark with an observation at p_C.z <= 0 (optionally a pixel
// reprojection error above the threshold) is deactivated in the device
// flags, which removes its observations from the cost, the landmark sums, S
// and the step without rebuilding the topology; the host reads back which
// landmarks were removed.
static int reject_outliers(mlba_handle* h, const mlba_options* o, int* removed) {
  hipStream_t s = h->stream;
  *removed = 0;
  if (h->L == 0) return MLBA_OK;
  if (!h->lm_bad.alloc(h->L)) return set_err(h, MLBA_ENOMEM, "device allocation failed");
  launch_vertex_prep(s, h->P, h->vert.p, h->vR.p);
  const double m = o->max_reprojection_error_px;
  launch_find_outliers(s, h->topo, h->vert.p, h->vR.p, h->lm.p, o->use_reprojection_error ? 1 : 0, m * m,
                       h->lm_flags.p, h->lm_bad.p);
  HIP_OK(hipGetLastError());
  std::vector<uint8_t> bad(h->L);
  HIP_OK(hipMemcpyAsync(bad.data(), h->lm_bad.p, h->L, hipMemcpyDeviceToHost, s));
  HIP_OK(hipStreamSynchronize(s));
  int n = 0;
  for (int l = 0; l < h->L; ++l)
    if (bad[l]) { h->lm_active[l] = 0; ++n; }
  *removed = n;
  // The recycled deflation columns are kept: the next solve rebuilds E from
  // the new S (and drops the deflation if E is not positive definite), so
  // any columns are valid, and the slow modes of a map with a few landmarks
  // removed are still close to them.
  return MLBA_OK;
}

int32_t mlba_solve_many(mlba_handle* const* handles, const mlba_options* const* options,
                        mlba_summary* const* summaries, int32_t* statuses, int32_t n, int32_t threads,
                        int32_t outlier_rejection) {
  if (n < 0 || (n > 0 && (!handles || !options))) return MLBA_EINVAL;
  for (int i = 0; i < n; ++i) {
    if (!handles[i] || !options[i]) return MLBA_EINVAL;
    for (int j = 0; j < i; ++j)
      if (handles[j] == handles[i]) return MLBA_EINVAL;
  }
  std::vector<int32_t> st(n, MLBA_OK);
  std::atomic<int> next{0};
  auto worker = [&]() {
    for (int i = next.fetch_add(1); i < n; i = next.fetch_add(1)) {
      mlba_summary* sm = summaries ? summaries[i] : nullptr;
      st[i] = outlier_rejection ? mlba_solve_with_outlier_rejection(handles[i], options[i], sm)
                                : mlba_solve(handles[i], options[i], sm);
    }
  };
  const int nt = std::max(1, std::min(n, threads > 0 ? threads : 8));
  std::vector<std::thread> pool;
  pool.reserve(nt - 1);
  for (int t = 1; t < nt; ++t) pool.emplace_back(worker);
  worker();
  for (std::thread& t : pool) t.join();
  int32_t rc = MLBA_OK;
  for (int i = 0; i < n; ++i) {
    if (statuses) statuses[i] = st[i];
    if (rc == MLBA_OK && st[i] != MLBA_OK) rc = st[i];
  }
  return rc;
}

int32_t mlba_solve_with_outlier_rejection(mlba_handle* h, const mlba_options* o, mlba_summary* sm) {
  if (!h) return MLBA_EINVAL;
  int rc = validate_options(h, o);
  if (rc) return rc;
  reset_summary(sm);
  if (o->reject_outliers_every_n_iters <= 0 || o->max_num_iterations <= 0) {
    if (sm) sm->termination_type = MLBA_FAILURE;  // outlier-rejection-solver.cc:214-218
    return MLBA_OK;
  }
  int remaining = o->max_num_iterations;
  double radius = o->initial_trust_region_radius;
  double budget = o->max_solver_time_in_seconds;
  int term = MLBA_NO_CONVERGENCE;
  bool first = true;
  double initial_cost = 0.0;
  while (remaining > 0 && budget > 0) {
    const double t0 = now_s();
    const int step_iters = std::min(remaining, o->reject_outliers_every_n_iters);
    mlba_options local = *o;
    local.max_num_iterations = step_iters;
    h->ev_summary = sm;
    rc = minimize(h, &local, radius, sm, &radius, &term);
    collect_events(h);
    h->ev_summary = nullptr;
    if (rc) return rc;
    if (first && sm) initial_cost = sm->initial_cost;
    first = false;
    int removed = 0;
    if ((rc = reject_outliers(h, o, &removed))) return rc;
    if (sm) sm->num_removed_landmarks += removed;
    if (term != MLBA_NO_CONVERGENCE) break;
    budget -= now_s() - t0;
    remaining -= step_iters;
  }
  if (sm) {
    sm->termination_type = term;
    sm->initial_cost = initial_cost;
    sm->num_residual_blocks = count_active_obs(h);
  }
  return MLBA_OK;
}

void mlba_calibration_options_init(mlba_calibration_options* c) {
  if (!c) return;
  c->fix_intrinsics = 1;
  c->fix_distortion = 1;
  c->fix_extrinsics_rotation = 1;
  c->fix_extrinsics_translation = 1;
}

int32_t mlba_download_cameras(const mlba_handle* h, double* q_CI__C_p_CI, double* intrinsics, double* distortion,
                              double* xi) {
  if (!h) return MLBA_EINVAL;
  for (int c = 0; c < h->C; ++c) {
    const DevCamera& k = h->h_cams[c];
    if (q_CI__C_p_CI)
      for (int i = 0; i < 7; ++i) q_CI__C_p_CI[7 * c + i] = h->h_cam_q[7 * c + i];
    if (intrinsics)
      for (int i = 0; i < 4; ++i) intrinsics[4 * c + i] = k.intr[i];
    if (distortion)
      for (int i = 0; i < 4; ++i) distortion[4 * c + i] = k.dist[i];
    if (xi) xi[c] = k.xi;
  }
  return MLBA_OK;
}

namespace {

// Free tangent columns of one camera: q_CI (0..2), C_p_CI (3..5), fu fv cu
// cv (6..9), distortion (10..13, as many as the model has), xi (14).
struct CalibLayout {
  std::vector<std::array<int32_t, 15>> col;  // per camera: global column or -1
  int32_t n = 0;
};

int distortion_parameter_count(int32_t type) {
  return type == kDistRadtan || type == kDistEquidistant ? 4 : (type == kDistFisheye ? 1 : 0);
}

// Host LM of the camera calibration blocks with the map held constant:
// dense normal equations over the free columns (at most 15 per camera),
// the Ceres rules of minimize() (Jacobi scaling, LM diagonal, gain ratio,
// radius update, tolerances).
class CalibSolver {
 public:
  CalibSolver(mlba_handle* h, const mlba_options* o, const CalibLayout& lay) : h_(h), o_(o), lay_(lay) {}

  // Cost (cameras with free columns), fixed cost, and with `jac` the normal
  // equations A, g at the cameras `cams` (device) / `cam_q`.
  int evaluate(const DevCamera* cams, const double* cam_q, bool jac, double* cost, double* fixed,
               std::vector<double>* A, std::vector<double>* g) {
    mlba_handle* h = h_;
    hipStream_t s = h->stream;
    DevTopology tt = h->topo;
    tt.cams = cams;
    const int E = calib_entries();
    // The calibration blocks 5 .. 9 inside one record per observation.
    static const int kTangent[10] = {3, 6, 6, 6, 6, 3, 3, 4, 4, 1};
    EvalOut rec{};
    for (int b = 0, off = 0; b < 10; off += 2 * kTangent[b], ++b) {
      if (!jac || b < 5) continue;
      rec.block[b] = h->calib_rec.p + off;
      rec.stride[b] = calib_record_stride();
    }
    launch_evaluate_full(s, tt, h->vert.p, h->vR.p, h->lm.p, h->baseframes.p, cam_q, true, h->perm_d.p,
                         h->calib_res.p, rec, jac);
    launch_calib_normal(s, tt, h->perm_d.p, h->calib_res.p, h->calib_rec.p, make_loss(o_), !jac, h->calib_part.p,
                        h->calib_out.p);
    HIP_OK(hipGetLastError());
    std::vector<double> out((size_t)E * h->C);
    HIP_OK(hipMemcpyAsync(out.data(), h->calib_out.p, out.size() * sizeof(double), hipMemcpyDeviceToHost, s));
    HIP_OK(hipStreamSynchronize(s));
    *cost = *fixed = 0.0;
    const int n = lay_.n;
    if (jac) { A->assign((size_t)n * n, 0.0); g->assign(n, 0.0); }
    for (int c = 0; c < h->C; ++c) {
      const double* oc = out.data() + (size_t)E * c;
      bool any = false;
      for (int k = 0; k < 15; ++k) any = any || lay_.col[c][k] >= 0;
      (any ? *cost : *fixed) += oc[135];
      if (!jac || !any) continue;
      for (int a = 0; a < 15; ++a) {
        const int ga = lay_.col[c][a];
        if (ga < 0) continue;
        (*g)[ga] = oc[120 + a];
        for (int b = a; b < 15; ++b) {
          const int gb = lay_.col[c][b];
          if (gb < 0) continue;
          const double v = oc[a * 15 - a * (a - 1) / 2 + (b - a)];
          (*A)[(size_t)ga * n + gb] = v;
          (*A)[(size_t)gb * n + ga] = v;
        }
      }
    }
    return MLBA_OK;
  }

  // max |x - Plus(x, -g)| over the free parameters.
  double gradient_max(const std::vector<double>& g) const {
    double m = 0.0;
    for (int c = 0; c < h_->C; ++c)
      for (int k = 0; k < 15; ++k) {
        const int j = lay_.col[c][k];
        if (j < 0) continue;
        if (k < 3) {
          if (k > 0) continue;
          const double* q = &h_->h_cam_q[7 * c];
          const double d[3] = {-g[j], -g[lay_.col[c][1]], -g[lay_.col[c][2]]};
          double qq[4];
          quat_plus_jpl(q, d, qq);
          for (int i = 0; i < 4; ++i) m = std::max(m, std::fabs(q[i] - qq[i]));
        } else {
          m = std::max(m, std::fabs(g[j]));
        }
      }
    return m;
  }

  // Candidate cameras x [+] (-w) into cand / cand_q, and the ambient norm of x.
  double candidate(const std::vector<double>& w, std::vector<DevCamera>* cand, std::vector<double>* cand_q) const {
    *cand = h_->h_cams;
    *cand_q = h_->h_cam_q;
    double xx = 0.0;
    for (int c = 0; c < h_->C; ++c) {
      const auto& col = lay_.col[c];
      DevCamera& k = (*cand)[c];
      double* q = &(*cand_q)[7 * c];
      const double* q0 = &h_->h_cam_q[7 * c];
      const DevCamera& k0 = h_->h_cams[c];
      if (col[0] >= 0) {
        const double d[3] = {-w[col[0]], -w[col[1]], -w[col[2]]};
        quat_plus_jpl(q0, d, q);
        rot_jpl(q, k.R_C_I);
        for (int i = 0; i < 4; ++i) xx += q0[i] * q0[i];
      }
      if (col[3] >= 0)
        for (int i = 0; i < 3; ++i) {
          q[4 + i] = q0[4 + i] - w[col[3 + i]];
          k.p_C_I[i] = q[4 + i];
          xx += q0[4 + i] * q0[4 + i];
        }
      if (col[6] >= 0)
        for (int i = 0; i < 4; ++i) {
          k.intr[i] = k0.intr[i] - w[col[6 + i]];
          xx += k0.intr[i] * k0.intr[i];
        }
      for (int i = 0; i < 4; ++i)
        if (col[10 + i] >= 0) {
          k.dist[i] = k0.dist[i] - w[col[10 + i]];
          xx += k0.dist[i] * k0.dist[i];
        }
      if (col[14] >= 0) {
        k.xi = k0.xi - w[col[14]];
        xx += k0.xi * k0.xi;
      }
    }
    return std::sqrt(xx);
  }

 private:
  mlba_handle* h_;
  const mlba_options* o_;
  const CalibLayout& lay_;
};

// Cholesky solve of the symmetric positive definite n x n system; false
// when not positive definite.
bool cholesky_solve(int n, std::vector<double> A, const std::vector<double>& b, std::vector<double>* x) {
  for (int j = 0; j < n; ++j) {
    double d = A[(size_t)j * n + j];
    for (int k = 0; k < j; ++k) d -= A[(size_t)j * n + k] * A[(size_t)j * n + k];
    if (!(d > 0.0) || !std::isfinite(d)) return false;
    const double l = std::sqrt(d);
    A[(size_t)j * n + j] = l;
    for (int i = j + 1; i < n; ++i) {
      double v = A[(size_t)i * n + j];
      for (int k = 0; k < j; ++k) v -= A[(size_t)i * n + k] * A[(size_t)j * n + k];
      A[(size_t)i * n + j] = v / l;
    }
  }
  x->assign(b.begin(), b.end());
  for (int i = 0; i < n; ++i) {
    double v = (*x)[i];
    for (int k = 0; k < i; ++k) v -= A[(size_t)i * n + k] * (*x)[k];
    (*x)[i] = v / A[(size_t)i * n + i];
  }
  for (int i = n - 1; i >= 0; --i) {
    double v = (*x)[i];
    for (int k = i + 1; k < n; ++k) v -= A[(size_t)k * n + i] * (*x)[k];
    (*x)[i] = v / A[(size_t)i * n + i];
  }
  return true;
}

}  // namespace

int32_t mlba_solve_calibration(mlba_handle* h, const mlba_options* o, const mlba_calibration_options* co,
                               mlba_summary* sm) {
  if (!h) return MLBA_EINVAL;
  int rc = validate_options(h, o);
  if (rc) return rc;
  if (!co) return set_err(h, MLBA_EINVAL, "calibration options are NULL");
  reset_summary(sm);
  // The map is held constant: every active observation's landmark, observer
  // and (for the mission and global types) landmark store vertex.
  std::vector<uint8_t> cam_used(h->C, 0);
  int n_active = 0;
  for (int k = 0; k < h->N; ++k) {
    const int l = h->s_landmark[k];
    if (!h->lm_active[l]) continue;
    ++n_active;
    cam_used[h->s_camera[k]] = 1;
    if (!h->lm_const[l] || !h->vertex_const[h->s_vertex[k]] ||
        (h->s_type[k] != kTypeKeyframe && !h->vertex_const[h->lm_anchor[l]]))
      return set_err(h, MLBA_EINVAL,
                     "calibration is solved with the map's vertices and landmarks held constant; "
                     "a variable vertex or landmark is in the problem");
  }
  CalibLayout lay;
  lay.col.assign(h->C, {});
  for (int c = 0; c < h->C; ++c) {
    auto& col = lay.col[c];
    col.fill(-1);
    if (!cam_used[c]) continue;
    const DevCamera& k = h->h_cams[c];
    auto take = [&](int first, int count) {
      for (int i = 0; i < count; ++i) col[first + i] = lay.n++;
    };
    if (!co->fix_extrinsics_rotation) take(0, 3);
    if (!co->fix_extrinsics_translation) take(3, 3);
    if (!co->fix_intrinsics) take(6, 4);
    if (!co->fix_distortion) take(10, distortion_parameter_count(k.dist_type));
    if (!co->fix_intrinsics && k.model == kCameraUnifiedProjection) take(14, 1);
  }
  if (lay.n == 0) return set_err(h, MLBA_EINVAL, "no calibration block is free");
  if (sm) sm->num_residual_blocks = n_active;
  const int n = lay.n;
  const int E = calib_entries();
  const int tiles = (h->N + 255) / 256;
  if (!h->calib_res.alloc(2 * (size_t)std::max(h->N, 1)) ||
      !h->calib_rec.alloc((size_t)calib_record_stride() * std::max(h->N, 1)) ||
      !h->calib_part.alloc((size_t)E * h->C * std::max(tiles, 1)) || !h->calib_out.alloc((size_t)E * h->C) ||
      !h->cams_cand.alloc(h->C) || !h->cam_q_cand.alloc(7 * (size_t)h->C))
    return set_err(h, MLBA_ENOMEM, "device allocation failed");
  hipStream_t s = h->stream;
  launch_vertex_prep(s, h->P, h->vert.p, h->vR.p);
  CalibSolver cs(h, o, lay);
  const double t_start = now_s();
  std::vector<double> A, g;
  double x_cost = 0.0, fixed_cost = 0.0;
  if ((rc = cs.evaluate(h->cams.p, h->cam_q.p, true, &x_cost, &fixed_cost, &A, &g))) return rc;
  double grad_max = cs.gradient_max(g);
  if (sm) { sm->initial_cost = x_cost + fixed_cost; sm->fixed_cost = fixed_cost; }
  mlba_iteration_summary it{};
  it.step_is_valid = it.step_is_successful = 1;
  it.cost = x_cost + fixed_cost;
  it.gradient_max_norm = grad_max;
  double radius = o->initial_trust_region_radius, decrease_factor = 2.0;
  it.trust_region_radius = radius;
  it.cumulative_time_in_seconds = it.iteration_time_in_seconds = now_s() - t_start;
  push_iteration(sm, it);
  int termination = MLBA_NO_CONVERGENCE;
  if (grad_max <= o->gradient_tolerance) termination = MLBA_CONVERGENCE;
  int consecutive_invalid = 0, iteration = 0;
  std::vector<DevCamera> cand;
  std::vector<double> cand_q, w, Ad, gd, scale(n, 1.0);
  while (termination == MLBA_NO_CONVERGENCE && o->max_num_iterations > 0) {
    const double t_iter = now_s();
    ++iteration;
    mlba_iteration_summary cur{};
    cur.iteration = iteration;
    // Jacobi scaling and the LM diagonal on the scaled system.
    for (int j = 0; j < n; ++j)
      scale[j] = o->use_jacobi_scaling ? 1.0 / (1.0 + std::sqrt(A[(size_t)j * n + j])) : 1.0;
    Ad.assign((size_t)n * n, 0.0);
    gd.assign(n, 0.0);
    for (int i = 0; i < n; ++i) {
      gd[i] = scale[i] * g[i];
      for (int j = 0; j < n; ++j) Ad[(size_t)i * n + j] = scale[i] * A[(size_t)i * n + j] * scale[j];
    }
    for (int j = 0; j < n; ++j)
      Ad[(size_t)j * n + j] += std::min(std::max(Ad[(size_t)j * n + j], o->min_lm_diagonal), o->max_lm_diagonal) / radius;
    const double t_ls = now_s();
    bool step_valid = cholesky_solve(n, Ad, gd, &w);
    double mcc = 0.0;
    if (step_valid) {
      for (int j = 0; j < n; ++j) w[j] *= scale[j];
      // Model cost change of the step -w: g'w - w'Aw / 2.
      double gw = 0.0, wAw = 0.0;
      for (int i = 0; i < n; ++i) {
        gw += g[i] * w[i];
        double aw = 0.0;
        for (int j = 0; j < n; ++j) aw += A[(size_t)i * n + j] * w[j];
        wAw += w[i] * aw;
      }
      mcc = gw - 0.5 * wAw;
      step_valid = std::isfinite(mcc) && mcc > 0.0;
    }
    if (sm) sm->linear_solver_seconds += now_s() - t_ls;
    cur.linear_solver_iterations = 1;
    cur.step_is_valid = step_valid;
    if (!step_valid) {
      if (++consecutive_invalid >= o->max_num_consecutive_invalid_steps) { termination = MLBA_FAILURE; break; }
      radius /= decrease_factor;
      decrease_factor *= 2.0;
      cur.cost = x_cost + fixed_cost;
      cur.gradient_max_norm = grad_max;
      cur.trust_region_radius = radius;
      if (sm) sm->num_unsuccessful_steps++;
    } else {
      consecutive_invalid = 0;
      double step_norm = 0.0;
      for (int j = 0; j < n; ++j) step_norm += w[j] * w[j];
      step_norm = std::sqrt(step_norm);
      const double x_norm = cs.candidate(w, &cand, &cand_q);
      cur.step_norm = step_norm;
      if (step_norm <= o->parameter_tolerance * (x_norm + o->parameter_tolerance)) {
        termination = MLBA_CONVERGENCE;
        break;
      }
      HIP_OK(hipMemcpyAsync(h->cams_cand.p, cand.data(), sizeof(DevCamera) * h->C, hipMemcpyHostToDevice, s));
      HIP_OK(hipMemcpyAsync(h->cam_q_cand.p, cand_q.data(), sizeof(double) * 7 * h->C, hipMemcpyHostToDevice, s));
      double cand_cost = 0.0, cand_fixed = 0.0;
      if ((rc = cs.evaluate(h->cams_cand.p, h->cam_q_cand.p, false, &cand_cost, &cand_fixed, nullptr, nullptr)))
        return rc;
      cur.cost_change = x_cost - cand_cost;
      if (std::fabs(cur.cost_change) <= o->function_tolerance * x_cost) {
        termination = MLBA_CONVERGENCE;
        break;
      }
      cur.relative_decrease = (x_cost - cand_cost) / mcc;
      if (cur.relative_decrease > o->min_relative_decrease) {
        h->h_cams = cand;
        h->h_cam_q = cand_q;
        HIP_OK(hipMemcpyAsync(h->cams.p, cand.data(), sizeof(DevCamera) * h->C, hipMemcpyHostToDevice, s));
        HIP_OK(hipMemcpyAsync(h->cam_q.p, cand_q.data(), sizeof(double) * 7 * h->C, hipMemcpyHostToDevice, s));
        const double t_ev = now_s();
        if ((rc = cs.evaluate(h->cams.p, h->cam_q.p, true, &x_cost, &fixed_cost, &A, &g))) return rc;
        if (sm) sm->evaluate_seconds += now_s() - t_ev;
        grad_max = cs.gradient_max(g);
        cur.step_is_successful = 1;
        cur.cost = x_cost + fixed_cost;
        cur.gradient_max_norm = grad_max;
        const double q = 2.0 * cur.relative_decrease - 1.0;
        radius = std::min(o->max_trust_region_radius, radius / std::max(1.0 / 3.0, 1.0 - q * q * q));
        decrease_factor = 2.0;
        if (sm) sm->num_successful_steps++;
      } else {
        radius /= decrease_factor;
        decrease_factor *= 2.0;
        cur.cost = cand_cost + fixed_cost;
        cur.gradient_max_norm = grad_max;
        if (sm) sm->num_unsuccessful_steps++;
      }
      cur.trust_region_radius = radius;
    }
    cur.iteration_time_in_seconds = now_s() - t_iter;
    cur.cumulative_time_in_seconds = now_s() - t_start;
    push_iteration(sm, cur);
    if (now_s() - t_start > o->max_solver_time_in_seconds) { termination = MLBA_NO_CONVERGENCE; break; }
    if (iteration >= o->max_num_iterations) break;
    if (cur.step_is_successful && cur.gradient_max_norm <= o->gradient_tolerance) { termination = MLBA_CONVERGENCE; break; }
    if (radius <= o->min_trust_region_radius) { termination = MLBA_CONVERGENCE; break; }
  }
  if (sm) {
    sm->termination_type = termination;
    sm->final_cost = x_cost + fixed_cost;
    sm->lm_loop_seconds += now_s() - t_start;
  }
  return MLBA_OK;
}

int32_t mlba_get_schedule(const mlba_handle* h, mlba_schedule* sc) {
  if (!h || !sc) return MLBA_EINVAL;
  std::memset(sc, 0, sizeof(*sc));
  sc->item_band_rows = h->sched_band;
  sc->item_waves = h->sched_waves;
  sc->xcd_mapping = h->sched_xcd;
  sc->pcg_partials = h->sched_pcg;
  return MLBA_OK;
}

int32_t mlba_set_schedule(mlba_handle* h, const mlba_schedule* sc) {
  if (!h) return MLBA_EINVAL;
  if (!sc) return set_err(h, MLBA_EINVAL, "schedule is NULL");
  if (sc->item_band_rows < 0 || sc->item_band_rows > 4096) return set_err(h, MLBA_EINVAL, "item_band_rows out of range");
  if (!schur_items_per_wg_supported(sc->item_waves)) return set_err(h, MLBA_EINVAL, "item_waves must be 1, 2, 4 or 8");
  if (sc->xcd_mapping != 0 && sc->xcd_mapping != 1) return set_err(h, MLBA_EINVAL, "xcd_mapping must be 0 or 1");
  if (sc->pcg_partials < 0 || sc->pcg_partials > 2) return set_err(h, MLBA_EINVAL, "pcg_partials must be 0, 1 or 2");
  const bool reorder = sc->item_band_rows != h->sched_band;
  h->sched_band = sc->item_band_rows;
  h->sched_waves = sc->item_waves;
  h->sched_xcd = sc->xcd_mapping;
  h->sched_pcg = sc->pcg_partials;
  // A build that is still to come orders its segments itself.
  return reorder && h->topology_ok ? upload_item_order(h) : MLBA_OK;
}

int32_t mlba_autotune(mlba_handle* h, const mlba_options* o, int32_t repeats, mlba_schedule* out) {
  if (!h) return MLBA_EINVAL;
  if (!out || repeats <= 0) return set_err(h, MLBA_EINVAL, "autotune needs a schedule output and repeats > 0");
  int rc = validate_options(h, o);
  if (rc) return rc;
  std::memset(out, 0, sizeof(*out));
  hipStream_t s = h->stream;
  if (h->n_segs > 0) {
    // The Schur factors of the first LM iteration at the current state.
    if ((rc = linearize(h, o))) return rc;
    launch_jacobi_scaling(s, h->Pvar, h->L, o->use_jacobi_scaling, h->pose_diag.p, h->lm_acc.p, h->pose_scale.p,
                          h->lm_scale.p);
    schur_factors(h);
    HIP_OK(hipMemsetAsync(h->fail.p, 0, sizeof(int32_t), s));
    launch_landmark_prep(s, h->topo, h->lm_acc.p, h->lm_scale.p, 1.0 / o->initial_trust_region_radius,
                         o->min_lm_diagonal, o->max_lm_diagonal, h->lm_z.p, h->lm_anc.p, h->fail.p);
    HIP_OK(hipGetLastError());
    hipEvent_t e0, e1;
    HIP_OK(hipEventCreate(&e0));
    if (hipEventCreate(&e1) != hipSuccess) {
      (void)hipEventDestroy(e0);
      return set_err(h, MLBA_EDEVICE, "hipEventCreate failed");
    }
    auto time_items = [&]() -> double {
      launch_schur_tiles(s, h->tdev, h->gf.p, h->gk.p, h->lm_z.p, h->lm_anc.p, h->schur_partial.p, h->sched_waves,
                         h->sched_xcd);  // warm
      (void)hipEventRecord(e0, s);
      for (int k = 0; k < repeats; ++k)
        launch_schur_tiles(s, h->tdev, h->gf.p, h->gk.p, h->lm_z.p, h->lm_anc.p, h->schur_partial.p,
                           h->sched_waves, h->sched_xcd);
      (void)hipEventRecord(e1, s);
      (void)hipEventSynchronize(e1);
      float ms = 0.f;
      (void)hipEventElapsedTime(&ms, e0, e1);
      return (double)ms / repeats;
    };
    static const int32_t kBands[] = {0, 1, 2, 4, 8, 16, 32}, kWaves[] = {1, 2, 4, 8};
    mlba_schedule best{kItemBandRows, kItemsPerWg, kItemXcd, 0, 0.0, 0.0, h->sched_pcg, 0};
    double best_ms = -1.0, default_ms = -1.0;
    for (int32_t band : kBands) {
      h->sched_band = band;
      if ((rc = upload_item_order(h))) break;
      for (int32_t waves : kWaves)
        for (int32_t xcd = 0; xcd < 2; ++xcd) {
          h->sched_waves = waves;
          h->sched_xcd = xcd;
          const double ms = time_items();
          ++out->schedules_tried;
          if (band == kItemBandRows && waves == kItemsPerWg && xcd == kItemXcd) default_ms = ms;
          if (best_ms < 0.0 || ms < best_ms) {
            best_ms = ms;
            best.item_band_rows = band;
            best.item_waves = waves;
            best.xcd_mapping = xcd;
          }
        }
    }
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    HIP_OK(hipGetLastError());
    if (rc) return rc;
    h->sched_band = -1;  // force the reorder
    if ((rc = mlba_set_schedule(h, &best))) return rc;
    out->default_ms = default_ms;
    out->tuned_ms = best_ms;
  }
  out->item_band_rows = h->sched_band;
  out->item_waves = h->sched_waves;
  out->xcd_mapping = h->sched_xcd;
  out->pcg_partials = h->sched_pcg;
  return MLBA_OK;
}

int32_t mlba_measure_copy(int64_t bytes, int32_t repeats, double* ms_per_copy) {
  if (bytes < 16 || bytes % 16 != 0 || repeats <= 0 || !ms_per_copy) return MLBA_EINVAL;
  void *a = nullptr, *b = nullptr;
  hipStream_t s = nullptr;
  hipEvent_t e0 = nullptr, e1 = nullptr;
  int32_t rc = MLBA_EDEVICE;
  if (hipMalloc(&a, bytes) == hipSuccess && hipMalloc(&b, bytes) == hipSuccess &&
      hipMemset(a, 1, bytes) == hipSuccess && hipStreamCreateWithFlags(&s, hipStreamNonBlocking) == hipSuccess &&
      hipEventCreate(&e0) == hipSuccess && hipEventCreate(&e1) == hipSuccess) {
    launch_stream_copy(s, bytes / 16, a, b);  // warm-up
    (void)hipEventRecord(e0, s);
    for (int r = 0; r < repeats; ++r) launch_stream_copy(s, bytes / 16, a, b);
    (void)hipEventRecord(e1, s);
    float ms = 0.f;
    if (hipEventSynchronize(e1) == hipSuccess && hipEventElapsedTime(&ms, e0, e1) == hipSuccess &&
        hipGetLastError() == hipSuccess) {
      *ms_per_copy = (double)ms / repeats;
      rc = MLBA_OK;
    }
  }
  if (e0) (void)hipEventDestroy(e0);
  if (e1) (void)hipEventDestroy(e1);
  if (s) (void)hipStreamDestroy(s);
  if (a) (void)hipFree(a);
  if (b) (void)hipFree(b);
  return rc;
}

int32_t mlba_time_kernels(mlba_handle* h, const mlba_options* o, int32_t repeats, mlba_kernel_times* t) {
  if (!h || !t || repeats <= 0) return MLBA_EINVAL;
  int rc = validate_options(h, o);
  if (rc) return rc;
  hipStream_t s = h->stream;
  std::memset(t, 0, sizeof(*t));
  hipEvent_t e0, e1;
  HIP_OK(hipEventCreate(&e0));
  HIP_OK(hipEventCreate(&e1));
  auto timed = [&](auto&& launch) -> double {
    launch();  // warm
    (void)hipEventRecord(e0, s);
    for (int k = 0; k < repeats; ++k) launch();
    (void)hipEventRecord(e1, s);
    (void)hipEventSynchronize(e1);
    float ms = 0.f;
    (void)hipEventElapsedTime(&ms, e0, e1);
    return (double)ms / repeats;
  };
  const DevLoss loss = make_loss(o);
  const double inv_mu = 1.0 / o->initial_trust_region_radius;
  h->f32_jac = o->jacobian_fp32 != 0;
  if ((rc = linearize(h, o))) return rc;
  launch_jacobi_scaling(s, h->Pvar, h->L, o->use_jacobi_scaling, h->pose_diag.p, h->lm_acc.p, h->pose_scale.p,
                        h->lm_scale.p);
  t->schur_factors_ms = timed([&] { schur_factors(h); });
  launch_vertex_prep(s, h->P, h->vert.p, h->vR.p);
  t->linearize_ms = timed([&] {
    launch_linearize(s, true, h->tiles, h->topo, h->vert.p, h->vR.p, h->lm.p, loss, h->tile_begin.p, h->obs_rec.p,
                     h->lm_acc.p, h->split_part.p, h->tile_cost.p, h->f32_jac);
    launch_split_sum(s, h->n_split, h->split_ids.p, h->split_tiles.p, h->split_part.p, h->lm_acc.p);
  });
  t->cost_ms = timed([&] {
    launch_linearize(s, false, h->tiles, h->topo, h->vert.p, h->vR.p, h->lm.p, loss, h->tile_begin.p, nullptr,
                     nullptr, nullptr, h->tile_cost2.p);
  });
  t->pose_rows_ms = timed([&] {
    launch_pose_rows(s, h->topo, h->vert.p, h->vR.p, h->lm.p, h->obs_rec.p, h->lm_acc.p, h->pose_grad.p,
                     h->pose_diag.p, h->pose_jtj.p, h->f32_jac);
  });
  HIP_OK(hipMemsetAsync(h->fail.p, 0, sizeof(int32_t), s));
  t->landmark_prep_ms = timed([&] {
    launch_landmark_prep(s, h->topo, h->lm_acc.p, h->lm_scale.p, inv_mu, o->min_lm_diagonal, o->max_lm_diagonal,
                         h->lm_z.p, h->lm_anc.p, h->fail.p);
  });
  t->schur_blocks_ms = timed([&] {
    launch_schur_blocks(s, h->topo, h->tdev, h->n_upper, h->ublk.p, h->gf.p, h->gk.p, h->lm_z.p, h->lm_anc.p,
                        h->vR.p, h->pose_scale.p, h->pose_diag.p, h->pose_jtj.p, inv_mu, o->min_lm_diagonal,
                        o->max_lm_diagonal, h->schur_partial.p, h->S.p, h->rhs.p, h->sched_waves, h->sched_xcd);
  });
  t->block_inverse_ms = timed([&] { launch_block_inverse(s, h->Pvar, h->diag_pos.p, h->S.p, h->Minv.p, h->fail.p); });
  if (h->Pvar > 0) {
    if ((rc = ensure_coarse_basis(h, o->pcg_coarse_nodes))) return rc;
    int32_t iters = 0;
    const PcgBuffers B = pcg_buffers(h, ritz_count(o) > 0 ? h->ritz_nr : 0, false);
    const bool small = pcg_small_applies(B, o->pcg_max_iterations);
    t->pcg_solve_ms = timed([&] {
      if (small)
        iters = launch_pcg_small(s, B, o->pcg_relative_tolerance, o->pcg_max_iterations, h->scal.p + kPcgIters) ? 0 : -1;
      else
        iters = launch_pcg_deflated(s, B, o->pcg_relative_tolerance, o->pcg_max_iterations, kPcgPoll, kPcgPoll, nullptr,
                                    0);
    });
    if (iters < 0) return set_err(h, MLBA_EDEVICE, "PCG launch failed");
    if (small) {
      if ((rc = read_scalars(h))) return rc;
      iters = (int32_t)h->scal_host[kPcgIters];
    }
    t->pcg_iterations = iters;
    // One more iteration: each of its kernels (one: pcg_spmv, or two) launched
    // repeats x 8 times back to back between events (launch gaps included),
    // averaged.
    hipEvent_t pe[3];
    for (auto& e : pe) HIP_OK(hipEventCreate(&e));
    const int reps = std::max(1, repeats) * 8;
    if (iters > 0 && !small) {
      const int it = launch_pcg_deflated(s, B, o->pcg_relative_tolerance, std::min<int32_t>(o->pcg_max_iterations, 4),
                                         kPcgPoll, kPcgPoll, pe, reps);
      if (it < 0) return set_err(h, MLBA_EDEVICE, "PCG launch failed");
      HIP_OK(hipEventSynchronize(pe[2]));
      float a = 0.f, b = 0.f;
      HIP_OK(hipEventElapsedTime(&a, pe[0], pe[1]));
      HIP_OK(hipEventElapsedTime(&b, pe[1], pe[2]));
      t->pcg_spmv_ms = a / reps;
      t->pcg_update_ms = pcg_step_applies(B) ? 0.0 : b / reps;
    }
    for (auto& e : pe) (void)hipEventDestroy(e);
    const int32_t nr_used = h->hat_K > 0 && ritz_count(o) > 0 ? h->ritz_nr : 0;
    t->pcg_coarse_columns = 6 * (int64_t)std::max(h->hat_K, 0) + nr_used;
    t->pcg_window_columns = h->grp_width + nr_used;
  }
  launch_step_vertices(s, h->topo, h->vert.p, h->px.p, h->pose_scale.p, h->w.p, h->vert_cand.p, h->vR_cand.p,
                       h->parts_w.p, h->parts_v.p);
  t->back_substitute_ms = timed([&] {
    (void)launch_back_substitute(s, h->topo, h->tiles, h->tile_begin.p, h->n_split, h->split_ids.p, h->vR.p,
                                 h->lm.p, h->obs_rec.p, h->lm_acc.p, h->lm_z.p, h->w.p, h->lm_u.p, h->parts_l.p,
                                 h->f32_jac);
  });
  HIP_OK(hipGetLastError());
  HIP_OK(hipStreamSynchronize(s));
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  t->num_observations = h->N;
  t->num_landmarks = h->L;
  t->num_variable_vertices = h->Pvar;
  t->schur_blocks = h->nnzb;
  t->schur_upper_blocks = h->n_upper;
  t->schur_pairs = h->schur_pairs;
  t->incidences = h->n_inc;
  t->linearize_tiles = h->tiles;
  t->schur_factor_blocks = h->n_g;
  t->schur_staged_blocks = h->n_staged;
  t->schur_visits = h->n_visits;
  t->schur_batches = h->n_batches;
  t->schur_segments = h->n_segs;
  t->schur_tile_pairs = h->n_tpairs;
  return MLBA_OK;
}

}  // extern "C"
