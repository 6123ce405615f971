// Learned per-vertex surrogate for large springy steps: shared constants, device-visible structs
// and the launchers of surrogate_kernels.hip.
//
// The network maps 72 features of a vertex (its up-to-12 strut neighbours, 6 values each) through
// three hidden layers of 128 GELU units (a piecewise-quadratic GELU, see surrogate_kernels.hip) to a
// 3-vector, the correction acceleration for a step of H = ratio * dt.  Weights and activations
// are bf16, products accumulate in f32 (MFMA).
#pragma once

#include "kernels.hpp"

namespace fp {

constexpr int kSlots = 12;
constexpr int kFeat = 6 * kSlots;  // 72
constexpr int kHid = 128;
constexpr int kOut = 3;
constexpr uint32_t kNoSlot = 0xffffffffu;

// Parameter vector (f32), each matrix row-major [out][in] (z = W x + b)
constexpr int kOffW1 = 0;
constexpr int kOffB1 = kOffW1 + kHid * kFeat;
constexpr int kOffW2 = kOffB1 + kHid;
constexpr int kOffB2 = kOffW2 + kHid * kHid;
constexpr int kOffW3 = kOffB2 + kHid;
constexpr int kOffB3 = kOffW3 + kHid * kHid;
constexpr int kOffW4 = kOffB3 + kHid;
constexpr int kOffB4 = kOffW4 + kOut * kHid;
constexpr int kParams = kOffB4 + kOut;  // 42,755

// LDS image of the inference kernel: bf16 weight matrices with the K index permuted to the MFMA
// operand layout and rows padded (104 / 136 elements) so that the 16 rows one MFMA operand read
// touches fall in distinct LDS banks; then the f32 biases.
constexpr int kLd1 = 104, kLd = 136;
constexpr int kImgW1 = 0;                              // [128][104]
constexpr int kImgW2 = kImgW1 + kHid * kLd1 * 2;       // [128][136]
constexpr int kImgW3 = kImgW2 + kHid * kLd * 2;        // [128][136]
constexpr int kImgW4 = kImgW3 + kHid * kLd * 2;        // [16][136], rows 3..15 zero
constexpr int kImgB = kImgW4 + 16 * kLd * 2;           // f32 b1[128] b2[128] b3[128] b4[16]
constexpr int kImgBytes = kImgB + (3 * kHid + 16) * 4;  // 102,208
static_assert(kImgBytes % 16 == 0, "image is copied in 16-byte units");

// One feature slot of a vertex: the strut neighbour and the strut's rest length.
struct SlotEnt {
  uint32_t nbr;  // global vertex id, kNoSlot when the slot is empty
  float rest;
};

// Where slot j of vertex i stands: the vertices in slices of 64, each slot's 64 entries together, so
// that one load of a wavefront over consecutive vertices reads consecutive entries (an array of 12
// entries a vertex spread each load over as many lines as lanes).
__host__ __device__ inline size_t slot_at(uint32_t i, int j) {
  return (size_t)(i / 64) * (64 * kSlots) + (size_t)(64 * j) + i % 64;
}
inline size_t slot_count(uint64_t n) { return (n + 63) / 64 * (64 * kSlots); }

struct FeatParams {
  float H;             // big step (s)
  float strain_scale;  // position features: strain_scale * (|d| - L) / L * d / |d|
};

// Per-block diagnostics of a big step: the largest strut-strain change; the energy (kinetic +
// spring + gravity potential) before, and after minus the work of the face forces; and the
// mechanical energy (kinetic + spring) before plus after, the scale of the energy residual.
struct DiagOut {
  float max_dstrain, e_old, e_new, emech_old;
};

// The same of a whole mesh, summed in double.
struct MeshDiag {
  double e_old, e_new, emech_old;
  float max_dstrain, pad;
};
// A mesh's blocks, and the number of slots that a vertex of it has at most.
struct MeshSlots {
  uint32_t blk_begin, blk_end, n_slots, pad;
};

// variant: vertices per wave / 16 (2: 1024-thread workgroups, the default; 4: 512 threads)
hipError_t launch_sur_mlp(const SoA& st, const SlotEnt* slots, uint32_t n, const void* image, FeatParams fp,
                          float out_scale, float* da, int grid, int variant, hipStream_t s);
// Big-step update of the vertices in `blocks` from `a.in` to `a.out` with acceleration
// F_ext / m + da (F_ext: gravity and face forces, plus strut forces when `struts`); `work` gets
// each vertex's face-force work over the step.
hipError_t launch_sur_integrate(const StepArgs& a, const CsrView& t, const BlockRange* blocks, uint32_t n_blocks,
                                const float* da, float* work, bool struts, hipStream_t s);
// Diagnostics of the big step from `in` to `out`: per block in `diag`, then per mesh in `per_mesh`.
hipError_t launch_sur_diag(const SoA& in, const SoA& out, const SlotEnt* slots, const float* slot_k,
                           const StepParams* params, const float* mass, const float* work, const BlockRange* blocks,
                           uint32_t n_blocks, const MeshSlots* meshes, uint32_t n_meshes, DiagOut* diag,
                           MeshDiag* per_mesh, hipStream_t s);
// Per block of `blocks`: max over its vertices of |v| / vmax and |strain| / smax (+inf when any
// value is not finite).
hipError_t launch_sur_health(const SoA& st, const SlotEnt* slots, const BlockRange* blocks, uint32_t n_blocks,
                             float vmax, float smax, float* out, hipStream_t s);
// Features (natural order: slot * 6 + component, f32) of the vertices `ids`.
hipError_t launch_sur_features(const SoA& st, const SlotEnt* slots, const uint32_t* ids, uint32_t n, FeatParams fp,
                               float* out, hipStream_t s);

// Training samples at big step b from positions x_b (cur) and x_{b+1} (next) of the plain solver.
// noise: `noisy` = positions x_b + e1 and velocities ((x_b + e1) - (x_{b-1} + e2)) / H with e1, e2
// normal(0, sigma) per component (zero for pinned vertices).
struct Pos3 {
  const float *x, *y, *z;
};
hipError_t launch_sur_noise(Pos3 prev, Pos3 cur, SoA noisy, const uint32_t* pins, uint32_t n, float H, float sigma,
                            uint64_t seed, hipStream_t s);
// For the vertices `ids` (mesh ids in `mesh_of`): features of the noisy state a.in (bf16 row of
// 72) and the normalised target ((x_{b+1} - x~_b) / H^2 - v~ / H - F_ext / m) / out_scale, which is
// ((x_{b+1} - 2 x~_b + x~_{b-1}) / H^2 - F_ext / m) / out_scale.
hipError_t launch_sur_samples(const StepArgs& a, const CsrView& t, const uint32_t* ids, const uint32_t* mesh_of,
                              uint32_t n, Pos3 next, const SlotEnt* slots, FeatParams fp, float out_scale, bool struts,
                              __bf16* X, float* T, hipStream_t s);

// Training (surrogate_train.hip).  One optimiser step is three launches: the chain kernel takes
// every batch row through the network and back, the weight kernel forms the weight gradients over
// slices of the batch, the update kernel sums the slices and applies Adam.
constexpr int kTrainTile = 128;    // workspace rows are padded to this
constexpr int kTrainSlices = 64;   // most batch slices of the weight gradients
// Transposed workspace, [row of the operand][batch row], each operand row `pitch` bf16 long: the
// batch's features (80 rows, 72..79 zero), the hidden activations, what the backward pass sends to
// each layer's sums, and the output error (16 rows, 3..15 zero).
constexpr int kTrX = 0, kTrH1 = 80, kTrH2 = kTrH1 + kHid, kTrH3 = kTrH2 + kHid, kTrZ1 = kTrH3 + kHid,
              kTrZ2 = kTrZ1 + kHid, kTrZ3 = kTrZ2 + kHid, kTrY = kTrZ3 + kHid, kTrRows = kTrY + 16;
struct TrainBatch {
  const __bf16* X;  // bf16 rows of 72 and f32 targets of 3
  const float* T;
  uint64_t count, seed;  // rows drawn from `count` by a hash of (seed, j); count 0: batch row j is row j
  int rows, pitch;       // batch rows, and the workspace's row length (a multiple of kTrainTile)
  const float* P;        // f32 parameters (biases)
  const __bf16* wb;      // bf16 parameters, and the transposes [in][out] of W2 and W3
  const __bf16* wbt;
  __bf16* tr;            // transposed workspace (kTrRows * pitch)
  float* Y;              // outputs [rows][3], or nullptr
  float* loss_part;      // squared-error sum of each workgroup
};
struct AdamArgs {
  float *p, *m, *v;  // nullptr p: gradient only
  float lr, b1, b2, eps, c1, c2;
};
inline int train_waves(int pitch) { return pitch <= 64 * 256 ? 4 : 8; }
inline int train_groups(int pitch) { return pitch / (16 * train_waves(pitch)); }
inline int train_slices(int pitch) { return pitch / 256 < 1 ? 1 : pitch / 256 > kTrainSlices ? kTrainSlices : pitch / 256; }
hipError_t launch_train_chain(const TrainBatch& b, hipStream_t s);
// Weight and bias gradients of each of train_slices(pitch) batch slices: part[slice][kParams].
hipError_t launch_train_weights(const __bf16* tr, int pitch, float* part, hipStream_t s);
// g = sum of the slices, *loss = scale * sum of the n_loss partial losses, then Adam and the bf16 copies
// (a.p != nullptr) of the updated parameters.
hipError_t launch_train_update(const float* part, int slices, float* g, const float* loss_part, int n_loss,
                               float scale, float* loss, const AdamArgs& a, __bf16* wb, __bf16* wbt, hipStream_t s);
// The bf16 copies of the parameters.
hipError_t launch_train_weights_bf16(const float* p, __bf16* wb, __bf16* wbt, hipStream_t s);
hipError_t launch_to_bf16(const float* in, __bf16* out, long n, hipStream_t s);

}  // namespace fp
