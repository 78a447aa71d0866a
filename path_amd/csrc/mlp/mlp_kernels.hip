// The layer-by-layer forward of the radiance MLP (encoding, one MFMA GEMM per
// layer), against which the fused kernels are checked and timed.
#include "mlp_encode.h"

namespace pt {
namespace mlp {

// ---------------------------------------------------------------------------
// GEMM: 128 x 128 block tile, K step 64, 4 waves in a 2 x 2 grid, each wave a
// 64 x 64 tile of 2 x 2 v_mfma_f32_32x32x16_bf16. Operands are staged in LDS
// as [row][k] (k contiguous, row stride 72 bf16 = 144 B). The next K step's
// global loads are issued into registers before the current step's MFMAs, so
// their latency overlaps the math.
// MFMA lane layout (32x32x16): lane l holds A[l % 32][8 (l / 32) .. +8],
// B[8 (l / 32) .. +8][l % 32]; accumulator r of lane l is
// C[8 (r / 4) + 4 (l / 32) + r % 4][l % 32].
// ---------------------------------------------------------------------------
constexpr uint32_t kBM = 128, kBN = 128, kBK = 64, kLdsStride = 72;
constexpr uint32_t kChunks = kBM * kBK / 8 / 256; // 16-byte chunks per thread per operand

// Global -> registers: chunk c of the tile (8 bf16 along k), zero outside
// [0, rows) x [k0, k_end).
__device__ __forceinline__ void fetch_tile(const uint16_t *__restrict__ src, uint32_t ld,
                                           uint32_t r0, uint32_t rows, uint32_t k0,
                                           uint32_t k_end, uint4 (&v)[kChunks]) {
#pragma unroll
  for (uint32_t i = 0; i < kChunks; ++i) {
    const uint32_t c = threadIdx.x + 256u * i;
    v[i] = make_uint4(0, 0, 0, 0);
    const uint32_t row = c / (kBK / 8), kc = (c % (kBK / 8)) * 8u;
    const uint32_t gr = r0 + row, gk = k0 + kc;
    if (gr < rows && gk < k_end)
      v[i] = *reinterpret_cast<const uint4 *>(src + size_t(gr) * ld + gk);
  }
}

__device__ __forceinline__ void store_tile(const uint4 (&v)[kChunks], uint16_t *__restrict__ dst) {
#pragma unroll
  for (uint32_t i = 0; i < kChunks; ++i) {
    const uint32_t c = threadIdx.x + 256u * i;
    const uint32_t row = c / (kBK / 8), kc = (c % (kBK / 8)) * 8u;
    *reinterpret_cast<uint4 *>(dst + row * kLdsStride + kc) = v[i];
  }
}

// XCD-aware tile order. Workgroups go to the 8 XCDs round-robin by linear
// id, and each XCD has its own L2. The N tiles of one row block share its
// operand tile and get consecutive slots on one XCD, so it is fetched into one
// L2 once. Identity when the row blocks do not fill the XCDs evenly.
struct TileId {
  uint32_t x, y;
};

__device__ __forceinline__ TileId gemm_tile() {
  const uint32_t gx = gridDim.x, gy = gridDim.y;
  if (gx % 8u != 0)
    return {blockIdx.x, blockIdx.y};
  const uint32_t b = blockIdx.x + gx * blockIdx.y;
  const uint32_t xcd = b % 8u, slot = b / 8u;
  return {(slot / gy) * 8u + xcd, slot % gy};
}

template <int kEpi>
__global__ __launch_bounds__(256) void k_gemm(GemmArgs g) {
  __shared__ __attribute__((aligned(16))) uint16_t As[kBM * kLdsStride];
  __shared__ __attribute__((aligned(16))) uint16_t Bs[kBN * kLdsStride];
  const TileId tile = gemm_tile();
  const uint32_t m0 = tile.x * kBM, n0 = tile.y * kBN;
  const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
  const uint32_t wm = wave >> 1, wn = wave & 1u;
  const uint16_t *A = reinterpret_cast<const uint16_t *>(g.A);
  const uint16_t *B = reinterpret_cast<const uint16_t *>(g.B);
  f32x16_t acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r)
        acc[i][j][r] = 0.f;
  uint4 va[kChunks], vb[kChunks];
  fetch_tile(A, g.lda, m0, g.M, 0, g.K, va);
  fetch_tile(B, g.ldb, n0, g.N, 0, g.K, vb);
  for (uint32_t k0 = 0; k0 < g.K; k0 += kBK) {
    store_tile(va, As);
    store_tile(vb, Bs);
    __syncthreads();
    if (k0 + kBK < g.K) {
      fetch_tile(A, g.lda, m0, g.M, k0 + kBK, g.K, va);
      fetch_tile(B, g.ldb, n0, g.N, k0 + kBK, g.K, vb);
    }
#pragma unroll
    for (uint32_t kk = 0; kk < kBK; kk += 16) {
      bf16x8_t a[2], b[2];
      const uint32_t ko = kk + (lane >> 5) * 8u;
#pragma unroll
      for (int i = 0; i < 2; ++i)
        a[i] = *reinterpret_cast<const bf16x8_t *>(
            As + (wm * 64u + i * 32u + (lane & 31u)) * kLdsStride + ko);
#pragma unroll
      for (int j = 0; j < 2; ++j)
        b[j] = *reinterpret_cast<const bf16x8_t *>(
            Bs + (wn * 64u + j * 32u + (lane & 31u)) * kLdsStride + ko);
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[i], b[j], acc[i][j], 0, 0, 0);
    }
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const uint32_t row = m0 + wm * 64u + i * 32u + (r / 4) * 8u + (lane >> 5) * 4u + (r % 4);
        const uint32_t col = n0 + wn * 64u + j * 32u + (lane & 31u);
        if (row >= g.M || col >= g.N)
          continue;
        const float v = acc[i][j][r];
        const size_t o = size_t(row) * g.ldc + col;
        if constexpr (kEpi == kEpiF32)
          reinterpret_cast<float *>(g.C)[o] = v;
        else
          reinterpret_cast<uint16_t *>(g.C)[o] = f2bf(v > 0.f ? v : 0.f);
      }
}

hipError_t launch_gemm(const GemmArgs &g, int epilogue, hipStream_t s) {
  if (g.M % 8 || g.N % 8 || g.K % 8 || g.lda % 8 || g.ldb % 8)
    return hipErrorInvalidValue;
  dim3 grid((g.M + kBM - 1) / kBM, (g.N + kBN - 1) / kBN);
  if (epilogue == kEpiReluBf16)
    hipLaunchKernelGGL(k_gemm<kEpiReluBf16>, grid, dim3(256), 0, s, g);
  else
    hipLaunchKernelGGL(k_gemm<kEpiF32>, grid, dim3(256), 0, s, g);
  return hipGetLastError();
}

// 28 rows per block: thread t < 252 encodes feature t % 9 of row t / 9, then
// the block zeroes the padding columns of its rows.
constexpr uint32_t kEncRows = 256 / kFeatures;

__global__ __launch_bounds__(256) void k_encode(const float *__restrict__ f, uint32_t n,
                                                uint32_t rows_pad, uint16_t *__restrict__ out) {
  const size_t row0 = size_t(blockIdx.x) * kEncRows;
  const uint32_t t = threadIdx.x;
  if (t < kEncRows * kFeatures) {
    const size_t row = row0 + t / kFeatures;
    if (row < rows_pad)
      encode_feature(row < n ? f[row * kFeatures + t % kFeatures] : 0.f, t % kFeatures,
                     out + row * kInPad);
  }
  for (uint32_t i = t; i < kEncRows * (kInPad - kEncoded); i += 256u) {
    const size_t row = row0 + i / (kInPad - kEncoded);
    if (row < rows_pad)
      out[row * kInPad + kEncoded + i % (kInPad - kEncoded)] = 0;
  }
}

hipError_t launch_encode(const float *features, uint32_t n, uint32_t rows_pad, bf16 *out,
                         hipStream_t s) {
  if (rows_pad == 0)
    return hipSuccess;
  hipLaunchKernelGGL(k_encode, dim3((rows_pad + kEncRows - 1) / kEncRows), dim3(256), 0, s,
                     features, n, rows_pad, reinterpret_cast<uint16_t *>(out));
  return hipGetLastError();
}

__global__ void k_compact_pred(const float *__restrict__ pred, uint32_t n,
                               float *__restrict__ out) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= 3 * n)
    return;
  out[i] = pred[size_t(i / 3) * kOutPad + i % 3];
}

hipError_t launch_compact_pred(const float *pred, uint32_t n, float *out, hipStream_t s) {
  if (n == 0)
    return hipSuccess;
  hipLaunchKernelGGL(k_compact_pred, dim3((3 * n + 255) / 256), dim3(256), 0, s, pred, n, out);
  return hipGetLastError();
}

} // namespace mlp
} // namespace pt
