// gemm.hpp — the matrix products of the prefill projections, called by
// ikv_mul_mat_f32 for more than one token: on F32 MFMA (gemm.hip) and, where
// it is faster, on bf16 MFMA with every float split into three exact pieces
// (gemm_bf16x3.hip).
#pragma once

#include <hip/hip_runtime.h>

#include <climits>
#include <cstdint>

namespace ikv {

// Whether gemm_nt_f32 takes the shape: n_out % 64 == 0, k % 64 == 0.
bool gemm_nt_supported(int64_t n_out, int64_t k, int64_t m);

// Tile shape (a gemm_nt_tile code) and number of K splits for a product.
struct GemmPlan {
  int tile;
  int split;
};
// The F32 MFMA kernel's plan and its estimated time, and the choice between it
// and the bf16-piece kernel.
GemmPlan gemm_f32_plan(int64_t n_out, int64_t k, int64_t m, bool may_split, double *us);
GemmPlan gemm_plan(int64_t n_out, int64_t k, int64_t m, bool may_split);

// One launch on tile shape `tile` (tokens x outputs; F32 MFMA: 0 128 x 128
// (n_out % 128 == 0), 1 64 x 64, 2 64 x 32, 3 32 x 64, 4 32 x 32; bf16 pieces:
// 5 128 x 256, 6 128 x 128, 7 64 x 128, 8 64 x 64) with K cut into
// n_split ranges (1 <= n_split <= k / 64); for n_split > 1, counters (one
// per tile, all 0; 0 again after the launch) and part (n_split partial
// tiles per tile).
int gemm_nt_tile(int tile, int n_split, const float *w, const float *x, float *out,
                 const float *residual, int n_out, int k, int m, float *part, int *counters,
                 hipStream_t s);

// The bf16-piece kernel's tile shapes (code = tile - 5 above). A tile's 256
// weight rows of k floats are one buffer range, hence the bound on k.
constexpr int kBf16x3MaxRows = 256;
inline bool gemm_bf16x3_supported(int64_t n_out, int64_t k, int64_t m) {
  return gemm_nt_supported(n_out, k, m) && k <= INT_MAX / (kBf16x3MaxRows * 4);
}
int gemm_bf16x3_tile(int code, int n_split, const float *w, const float *x, float *out,
                     const float *residual, int n_out, int k, int m, float *part, int *counters,
                     hipStream_t s);

// out[m][n_out] = x[m][k] w[n_out][k]^T (+ residual[m][n_out], which may be
// out itself); w and x 16-byte aligned. With may_split, a product whose tiles
// do not fill the CUs splits K, on a workspace of the stream (allocated on
// the first such call for the device and stream, 8 MiB, kept until exit).
// 0, or -ENOTSUP / -EINVAL / -EOVERFLOW / -ENOMEM before any launch, or the
// hipError_t of the allocation or launch.
int gemm_nt_f32(const float *w, const float *x, float *out, const float *residual, int64_t n_out,
                int64_t k, int64_t m, bool may_split, hipStream_t s);

}  // namespace ikv
