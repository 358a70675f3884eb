// Chemistry surrogate: a 12 -> 4x128 (GELU or hard swish) -> 10 MLP with BF16 weights and FP32 accumulation on the
// gfx950 matrix cores.  A training step is three kernels (32 rows through all layers and back, the weight gradients, Adam);
// inference runs as one persistent kernel holding every weight in LDS, fused with the feature scaling, the
// element-conserving projection, the temperature recovery and the fallback gate.
#pragma once

#include <vector>

#include <hip/hip_runtime.h>

#include "chem.hpp"
#include "chem_kernels.hpp"

namespace corefl {

constexpr int kMlpLayers = 5, kMlpIn = 12, kMlpOut = 10, kMlpHidden = 128;
constexpr int kMlpK[kMlpLayers] = {12, 128, 128, 128, 128};
constexpr int kMlpN[kMlpLayers] = {128, 128, 128, 128, 10};
constexpr int kMlpKp[kMlpLayers] = {16, 128, 128, 128, 128}; // K padded to the 16-deep MFMA step
constexpr int kMlpNp[kMlpLayers] = {128, 128, 128, 128, 32}; // N padded to the 32-wide MFMA tile

// Device weights: BF16 W^T, [Np][Kp] row-major (k contiguous), zero padded; FP32 biases [N].
// Hidden activation: GELU in its tanh form (the network the specification names) or hard swish.
constexpr int kActGelu = 0, kActHardSwish = 1;

// Flat parameter layout: W_0 (K_0 x N_0, row-major), b_0, W_1, b_1, ..., W_4, b_4.
constexpr int mlp_offset(int layer, bool bias) {
  int o = 0;
  for (int l = 0; l < layer; ++l) o += kMlpK[l] * kMlpN[l] + kMlpN[l];
  return bias ? o + kMlpK[layer] * kMlpN[layer] : o;
}
constexpr int kMlpParams = mlp_offset(4, true) + kMlpOut;
constexpr int kMlpBackN[kMlpLayers] = {0, 128, 128, 128, 16}; // depth of the layers' backward products

struct MlpDev {
  const unsigned short *wt[kMlpLayers];
  const float *bias[kMlpLayers];
  int act; // kActGelu or kActHardSwish
};

// Feature and target scaling.  Features (T, ln p, Y_1^a..Y_9^a, ln dt) -> (f - mu) / sig, with a = y_power
// (1: plain mass fractions; a < 1 spreads the small radical fractions).  Targets: s = out * sig + mu is the
// signed logarithm of the rate, rate = sign(s) r0 (exp|s| - 1) for (dY_k/dt, dT/dt); r0 <= 0 means
// rate = s (no transform).
struct SurrogateScaling {
  float in_mu[kMlpIn], in_sig[kMlpIn];
  double out_mu[kMlpOut], out_sig[kMlpOut], out_r0[kMlpOut];
  double y_power;
};

// A cell uses the network only inside this input box, when the network's own temperature change agrees
// with the one recovered from energy conservation to within dT_max, and when its temperature changes by at
// most dT_step over the sub-step (fast-reacting cells go to the exact integrator).
struct SurrogateGate {
  double t_min, t_max, p_min, p_max, dt_min, dt_max, dT_max, dT_step;
};

// Element conservation: E[e][k] = (atoms of element e in species k) / MW_k, at most 4 elements; rows
// e >= ne are zero.
struct ElementMatrix {
  int ne;
  double E[4][kMaxSpec];
  // inverse of the projection's normal matrix E E^T (rows e >= ne: identity) when no species is held at
  // zero, the common case
  double M0inv[4][4];
  // the same for every set of species held at zero (bit k: species k): 512 entries of 17 doubles, the 4 x 4
  // inverse of the normal matrix over the other species and 1 + m (0 where that matrix is singular), m the
  // bit set of the elements no free species carries (their rows and columns are the identity's)
  const double *inv_table;
};

constexpr int kProjTableEntries = 512, kProjTableStride = 17;
// E, M0inv and the held-species inverse table of a mechanism (host); false if it has more than 4 elements or
// E E^T is singular.
bool projection_tables(const ChemMech &mech, ElementMatrix &em, std::vector<double> &table);

// One training step (or gradient, or forward pass) of a mini-batch.  Rows are handled 32 at a time; the arrays that the
// weight gradients contract over the batch are stored with eight consecutive rows of a neuron together, as the MFMA
// takes them (blocks of 32 neurons x 16 rows; ld rows in all, a multiple of 64).
constexpr int kTrainRows = 32;                       // rows of a work-group of the forward / backward kernel
// parts of a batch of B rows whose weight gradients are summed apart, at most
inline int train_max_chunks(int B) { return B <= 16384 ? 16 : 64; }
// BF16 copies of the weights: W^T [Np][Kp] for inference, and in blocks of one MFMA operand each the rows of W^T for the
// forward pass of the training and the rows of W (layers 1..4, N padded to 16 in layer 4) for its backward pass.
struct WeightCopies {
  unsigned short *wt[kMlpLayers], *wf[kMlpLayers], *wb[kMlpLayers];
};

struct TrainArgs {
  int B;                                             // rows of the mini-batch
  const float *X, *Y;                                // data set [n][12], [n][10]; Y null: forward only
  long n;                                            // rows of the data set
  unsigned long long seed;                           // row i of the batch is data row i (0), or hash(seed, step, i) mod n
  long step;
  const unsigned short *wf[kMlpLayers], *wb[kMlpLayers]; // as in WeightCopies
  const float *bias[kMlpLayers];
  unsigned short *HT[kMlpLayers];                    // inputs of layer l, 32 or 128 neurons x ld
  unsigned short *GT[kMlpLayers];                    // gradients of layer l's pre-activations, 128 or 32 neurons x ld
  long ld;
  float *loss_part;                                  // one partial loss per work-group
  float *out;                                        // forward only: [B][10]
  int act;
};
// The forward pass, and with Y the loss and the backward pass down to every layer's pre-activation gradient.
hipError_t launch_train_tile(const TrainArgs &a, hipStream_t s);
// Weight and bias gradients from HT and GT, chunk by chunk of the batch: part[chunk][flat parameter].
int train_chunks(int B);
hipError_t launch_train_grad(const TrainArgs &a, float *part, hipStream_t s);
// Sums the chunks and the partial losses (loss null: not); grads non-null: the gradient goes there and nothing is
// updated; else Adam on the flat parameters, with the BF16 copies of the weights.
struct AdamArgs {
  const float *part, *loss_part;
  int chunks, loss_parts;
  float *loss, *grads;
  float *p, *m, *v;
  WeightCopies w;
  float lr, b1, b2, eps, c1, c2;
};
hipError_t launch_train_adam(const AdamArgs &a, hipStream_t s);
// FP32 weights (flat parameters p) -> the BF16 copies.
hipError_t launch_pack_weights(const float *p, const WeightCopies &w, hipStream_t s);

// Work arrays of a surrogate chemistry step for n cells: BF16 features [n][16], FP32 outputs [n][10] and
// the input-range flags [n].
struct SurrogateWork {
  unsigned short *feat;
  float *out;
  unsigned char *flag;
};

// FP32 feature rows X [n][12] -> BF16 rows [n][16] (zero padded).
hipError_t launch_rows_to_feat(const float *X, long n, unsigned short *feat, hipStream_t s);
// Inference.  Raw mode: BF16 feature rows feat [n][16] (as launch_rows_to_feat writes them) -> outputs y [n][10].
hipError_t launch_mlp_raw(const MlpDev &net, long n, const unsigned short *feat, float *y, int blocks,
                          hipStream_t s);
// Chemistry mode: every cell of b (n cells) is advanced by dt (b.dtc per cell if set) with the network
// (features, network, projection / temperature / gate kernels); cells that fail the gate are appended to
// fb_list (count in *fb_count, zeroed by the launch) and left unchanged for the exact integrator.
hipError_t launch_mlp_chem(const MlpDev &net, const ChemMech *mech_dev, const ChemBatch &b, double dt,
                           const SurrogateScaling &sc, const SurrogateGate &gate, const ElementMatrix &em,
                           const SurrogateWork &w, int *fb_list, int *fb_count, int blocks, hipStream_t s);

} // namespace corefl
