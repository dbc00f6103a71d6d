// The f32 projections of the Qwen3 runner (gemm_f32.hip).
#pragma once

#include "inl_common.hpp"

namespace inl {

enum : int32_t {
  GF_STORE = 0,    // y = product
  GF_PART = 1,     // y[s] = product over part s of k, m * ys elements apart
  GF_SWIGLU = 2,   // y = silu(gate) * up; w holds n gate rows, then n up rows
};

// Whether a layer's four projections have the widths the kernels take.
bool gemm_f32_fits(int32_t hidden, int32_t qkv_rows, int32_t attn_width, int32_t intermediate);
// Whether a batch of m rows is faster here than on hipBLASLt. The tiles' k loops
// are serial, so few of them leave CUs idle: at least 128 tiles of the q/k/v
// projection, and more rows than 464, below which the fourth row of tiles is half
// empty. us per encode, own / hipBLASLt. 0.6B shape (32 tiles a row): 400 rows
// 5,109 / 4,993, 466 rows 5,319 / 5,845, 512 rows 5,354 / 6,353, 800 6,986 / 7,811,
// 1,024 7,505 / 11,350, 2,048 12,408 / 15,582. 4 layers of hidden 512, q/k/v 3,072
// (24 a row): 480 rows 491 / 438, 700 523 / 558, 1,024 583 / 726, 4,096 1,538 /
// 1,922. 4 layers of hidden 256, q/k/v 1,024 (8 a row): 480 rows 397 / 319, 2,000
// 466 / 470, 4,096 643 / 714.
bool gemm_f32_pays(int64_t m, int32_t qkv_rows);
// Parts of k for an m x n output, within part_bytes of workspace.
int gemm_f32_splits(int64_t m, int32_t n, int32_t k, int cus, size_t part_bytes);
// y[m, n] = x[m, k] . w[n, k]^T; w contiguous, x and y rows xs and ys apart,
// everything 16-byte aligned.
int gemm_f32_launch(int64_t m, int32_t n, int32_t k, const float* x, int64_t xs, const float* w, int32_t epi,
                    int32_t splits, float* y, int64_t ys, hipStream_t st);
// h += the sum of `parts` arrays [rows, dim]; x = rms_norm(h) * gamma unless
// gamma is NULL. Contiguous rows.
int add_norm_launch(int64_t rows, int32_t dim, float* h, const float* part, int32_t parts, const float* gamma, float eps,
                    float* x, hipStream_t st);

}  // namespace inl
