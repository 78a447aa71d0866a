// Radiance MLP on MFMA: BF16 operands, FP32 accumulation.
//
// Network: 9 features (position, shading normal, albedo) -> 12-frequency
// encoding (9 raw + 9 x 12 x {sin, cos} = 225, zero-padded to 256) -> 6
// hidden layers of width 256 with ReLU -> 3 outputs (padded to 16). Weights
// are [out][in] row-major; no biases.
#pragma once

#include <hip/hip_runtime.h>
#include <hip/hip_bf16.h>

#include <cstdint>

namespace pt {
namespace mlp {

using bf16 = __hip_bfloat16;

constexpr uint32_t kFeatures = 9;
constexpr uint32_t kFrequencies = 12;
constexpr uint32_t kEncoded = kFeatures * (1 + 2 * kFrequencies); // 225
constexpr uint32_t kInPad = 256;
constexpr uint32_t kWidth = 256;
constexpr uint32_t kHidden = 6;
constexpr uint32_t kOut = 3;
constexpr uint32_t kOutPad = 16;
constexpr uint32_t kLayers = kHidden + 1; // 7 weight matrices
constexpr uint32_t kRowAlign = 128;       // batch rows are a multiple of this

inline uint32_t layer_in(uint32_t l) { return l == 0 ? kInPad : kWidth; }
inline uint32_t layer_out(uint32_t l) { return l + 1 == kLayers ? kOutPad : kWidth; }
inline uint64_t layer_offset(uint32_t l) {
  uint64_t o = 0;
  for (uint32_t i = 0; i < l; ++i)
    o += uint64_t(layer_in(i)) * layer_out(i);
  return o;
}
inline uint64_t param_count() { return layer_offset(kLayers); }

enum Epilogue : int {
  kEpiReluBf16 = 0, // C = bf16(max(acc, 0))
  kEpiF32 = 1,      // C = acc (fp32)
};

// C[M x N] = sum_k A[m * lda + k] B[n * ldb + k].
// Requirements: M, N, K, lda, ldb multiples of 8.
struct GemmArgs {
  const bf16 *A;
  const bf16 *B;
  uint32_t lda, ldb;
  uint32_t M, N, K;
  void *C;
  uint32_t ldc;
};

hipError_t launch_gemm(const GemmArgs &g, int epilogue, hipStream_t s);
// features [n x 9] fp32 -> encoded [rows_pad x 256] bf16 in the kernels'
// column order (mlp_encode.h); rows from n on encode zero features
hipError_t launch_encode(const float *features, uint32_t n, uint32_t rows_pad, bf16 *out,
                         hipStream_t s);

// Weights in the fragment orders of mlp_fused.hip. Forward: the hidden layers
// and the output layer padded to 32 outputs; backward: layers 1 .. 5, then the
// output layer's one step of 16.
constexpr size_t kWFragElems = size_t(kHidden) * kWidth * kWidth + 32 * kWidth;
constexpr size_t kWtFragElems = size_t(kHidden - 1) * kWidth * kWidth + 16 * kWidth;

// Operands of the fused forward (and, for training, loss and data gradients)
// of a batch of n rows in tiles of mlp_tile_rows(rows_pad).
struct MlpTileArgs {
  const float *feat, *targ; // [n x 9], [n x 3], or the whole training set
  uint64_t set_rows;        // != 0: row i is row random(seed, i) of that many
  uint64_t seed;
  uint32_t n;
  const uint16_t *w_frag, *wt_frag;
  float *pred;              // inference: [rows_pad x 3]
  // training
  uint16_t *a_frag, *g_frag; // layer l's input / output gradient at l * layer_stride
  size_t layer_stride;       // rows_pad * 256
  uint32_t *masks;           // rows_pad * 48 words
  float *out_part;           // [tiles][3][256]: output layer's weight gradient
  float *loss_part;          // [tiles]
};
// Rows per tile: 128, or 64 or 32 for batches that would leave the chip idle.
uint32_t mlp_tile_rows(uint32_t rows_pad);
hipError_t launch_mlp_tile(const MlpTileArgs &a, uint32_t rows_pad, bool train, hipStream_t s);

// Weight gradients of the hidden layers (split over the rows, fp32 partials)
// and the sums of the tiles' output-layer gradients and losses.
struct MlpWgradArgs {
  const uint16_t *a_frag, *g_frag;
  size_t layer_stride;
  uint32_t rows_pad, splits, tiles;
  float *part; // [6][splits][256][256]
  const float *out_part, *loss_part;
  float *out_grad; // [3][256]
  float *loss;     // one float on the device
};
uint32_t mlp_wgrad_splits(uint32_t rows_pad);
hipError_t launch_mlp_wgrad(const MlpWgradArgs &a, hipStream_t s);

enum MlpUpdate : int {
  kUpdatePack = 0,     // only the bf16 copies of w
  kUpdateGradient = 1, // the summed gradient to grad
  kUpdateAdam = 2,     // Adam (bias corrections c1, c2) on w, then its copies
};
struct MlpUpdateArgs {
  const float *part, *out_grad; // k_mlp_wgrad's
  uint32_t splits;
  float *grad, *w, *m, *v;             // parameter order
  uint16_t *w_rows, *w_frag, *wt_frag; // bf16 copies
  float lr, beta1, beta2, eps, c1, c2;
};
hipError_t launch_mlp_update(const MlpUpdateArgs &a, int mode, hipStream_t s);

// out[i][c] = pred[i][c] for c < 3 (rows of 16 -> rows of 3)
hipError_t launch_compact_pred(const float *pred, uint32_t n, float *out, hipStream_t s);

} // namespace mlp
} // namespace pt
