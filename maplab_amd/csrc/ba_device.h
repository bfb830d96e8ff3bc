// ba_device.h -- device-side data layout of the visual BA problem in HBM and
// the kernel entry points (ba_kernels.hip). Everything here is internal to
// libmaplab_ba.so; the public ABI is include/maplab_ba.h.
#ifndef MAPLAB_AMD_BA_DEVICE_H_
#define MAPLAB_AMD_BA_DEVICE_H_

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace mlba {

constexpr int kObsTile = 256;        // observations per linearization tile
// Observation record (96 bytes): the robust-corrected residual r (2), its
// Jacobian K = d r / d p_I (2x3) with respect to the landmark in the observer's
// IMU frame, and p_I. The Jacobians of the residual's blocks follow from them
// and the vertex: J_landmark = K G with G = d p_I / d p_B (landmark_to_imu),
// J_observer = K [|q|^2 [p_I]x | -R_I_M].
constexpr int kObsRecord = 12;       // doubles: r K p_I, one unused

// The record with the Jacobian in FP32 and the remainder of the rounding in
// BF16 (32 significant bits together): 80 bytes. K alone carries what J_landmark
// and J_observer used to round separately, 18 entries whose roundings partly
// cancelled; with K in FP32 only, solves ended 1.3 times as far from the FP64
// ones as those did.
struct Rec32 {
  double r[2];
  double p[3];
  float K[6];
  uint16_t lo[6];
  uint32_t unused;
};
__host__ __device__ inline float bf16_value(uint16_t b) {
  union { uint32_t u; float f; } v;
  v.u = (uint32_t)b << 16;
  return v.f;
}
// The nearest BF16 (ties to even) of a finite value.
__host__ __device__ inline uint16_t bf16_round(float x) {
  union { float f; uint32_t u; } v;
  v.f = x;
  return (uint16_t)((v.u + 0x7FFFu + ((v.u >> 16) & 1u)) >> 16);
}

template <bool kF32>
struct RecView;
template <>
struct RecView<false> {
  const double* q;
  __host__ __device__ RecView(const void* base, size_t x) : q(static_cast<const double*>(base) + kObsRecord * x) {}
  __host__ __device__ double r(int k) const { return q[k]; }
  __host__ __device__ double K(int k) const { return q[2 + k]; }
  __host__ __device__ double p(int k) const { return q[8 + k]; }
};
template <>
struct RecView<true> {
  const Rec32* q;
  __host__ __device__ RecView(const void* base, size_t x) : q(static_cast<const Rec32*>(base) + x) {}
  __host__ __device__ double r(int k) const { return q->r[k]; }
  __host__ __device__ double K(int k) const { return static_cast<double>(q->K[k]) + static_cast<double>(bf16_value(q->lo[k])); }
  __host__ __device__ double p(int k) const { return q->p[k]; }
};
constexpr int kLmAcc = 18;           // V_own(6) V_mission(6) g(3) g_mission(3); V = V_own + V_mission
constexpr int kLmZ = 10;             // T(6, lower triangle, Z = T'T), T g(3), one unused
constexpr int kLmAnchor = 18;        // anchor's factor: U(9), the negated self product(6), rhs(3)
constexpr int kFactor = 12;          // factor block: P(3x3), p_I(3)

// A batch of independent scalar reductions (k_reduce_many), 1..kMaxReduceBatch
// of them.
struct ReduceDesc {
  int32_t n, stride, offset, is_max;
  const double* parts;
  double* out;
};
constexpr int kMaxReduceBatch = 8;
struct ReduceBatch {
  ReduceDesc d[kMaxReduceBatch];
  int32_t count;
  int32_t* fail;     // nullable: failure counter, copied to fail_out and cleared
  double* fail_out;
};
constexpr int kRowThreads = 256;     // threads of a reduced-camera-system row block

// Landmark flags.
constexpr uint32_t kLmActive = 1u;
constexpr uint32_t kLmConstant = 2u;
constexpr uint32_t kLmAnchorVar = 4u;   // anchor vertex variable and landmark has pose-coupled obs
constexpr uint32_t kLmSplit = 8u;       // observations span several linearization tiles

// Observation meta word: bits 0-1 error type, bit 2 observer variable, bit 3
// landmark active, bits 8.. camera index.
__host__ __device__ inline int32_t obs_type(int32_t meta) { return meta & 3; }
__host__ __device__ inline bool obs_observer_var(int32_t meta) { return (meta >> 2) & 1; }
// The landmark was active when the topology was built (outlier rejection may
// have cleared kLmActive since).
__host__ __device__ inline bool obs_built_active(int32_t meta) { return (meta >> 3) & 1; }
__host__ __device__ inline int32_t obs_camera(int32_t meta) { return meta >> 8; }

struct DevCamera {
  double R_C_I[9];
  double p_C_I[3];
  double intr[4];
  double dist[4];
  double width, height;
  double xi;          // unified-projection mirror parameter (0 for pinhole)
  int32_t dist_type;
  int32_t model;      // kCameraPinhole / kCameraUnifiedProjection
};

// Read-only problem topology (observation order = landmark-sorted).
struct DevTopology {
  int32_t N, L, P, Pvar, M, C;
  const double* obs_kp;        // 2N
  const double* obs_sinv;      // N
  const int32_t* obs_vertex;   // N
  const int32_t* obs_meta;     // N
  const int32_t* obs_landmark; // N
  const int32_t* obs_col;      // N: variable index of the observer when the observation couples it, else -1
  const int32_t* lm_begin;     // L+1
  const int32_t* lm_anchor;    // L
  const uint32_t* lm_flags;    // L
  const DevCamera* cams;       // C
  const double* mission_T;     // 12M: R_G_M (JPL matrix of q_GM) and p_G_M
  const int32_t* vertex_mission; // P
  const int32_t* vertex_var;   // P: variable index or -1
  const int32_t* var_vertex;   // Pvar
  // reduced camera system
  const int32_t* row_ptr;      // Pvar+1 block row pointers of S
  const int32_t* col_var;      // nnzb: column variable index
  const int32_t* diag_pos;     // Pvar: position of the diagonal block
  const int32_t* inc_ptr;      // Pvar+1 incidence lists of each row
  const int32_t* inc;          // >=0: observation index, <0: -1-landmark (anchor)
  int32_t max_row_blocks;
};

// Device copy of the reduced camera system's work decomposition (ba_tiles.h):
// segments (in dispatch order through seg_order) with their thread parts,
// batches with their slot and pair lists, and for every upper block of S
// the partial slots (segment * kTileBlocks + thread) summed into it, in order.
struct SchurTilesDev {
  int32_t n_segs, n_uslot;
  const int32_t* seg_order;
  const int4* segs;
  const uint32_t* seg_thread;
  const int4* batches;
  const int2* slots;
  const uint16_t* batch_off;
  const uint16_t* pairs;
  const int32_t* uslot_ptr;
  const int32_t* uslot;
};

// Where k_evaluate_full writes the Jacobian blocks: block b of observation o
// (2 x size, row-major) at block[b] + o * stride[b]; null: not wanted.
struct EvalOut {
  double* block[10];
  int32_t stride[10];
};

// Loss of the whitened residual.
struct DevLoss {
  int32_t type;      // 0 Huber (maplab), 1 Cauchy, 2 trivial
  double scale_px;   // Cauchy scale in pixels
};

}  // namespace mlba

#endif  // MAPLAB_AMD_BA_DEVICE_H_
