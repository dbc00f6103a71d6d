// An encoder layer on a few token rows (skinny.hip), as the Qwen3 runner
// issues it.
#pragma once

#include "inl_common.hpp"

namespace inl {

enum : int32_t {
  SKINNY_STORE = 0,     // y = product, in the model dtype
  SKINNY_ADD_F32 = 1,   // f32 rows y += product; yf: their fragments
  SKINNY_SWIGLU = 2,    // yf = fragments of silu(gate) * up; w holds n gate rows, then n up rows
};

// The weights the launch after this one starts on: `consumers` workgroups of
// `bytes` each (16 rows), and with `second` the same again that far behind.
struct SkinnyNext {
  const char* w = nullptr;   // nullptr: nothing to prefetch
  int64_t bytes = 0, second = 0;
  int32_t consumers = 0;
  int32_t cus = 0;           // of the device: a workgroup on each that the launch itself leaves idle
};
inline SkinnyNext skinny_next(int32_t dtype, const void* w, int32_t n, int32_t k, bool swiglu, int32_t cus) {
  const int64_t row = (int64_t)k * dtype_size(dtype);
  return {(const char*)w, 16 * row, swiglu ? n * row : 0, n / 16, cus};
}

// y[m, n] from x[m, k] . w[n, k]^T, x in fragments xf. gamma != NULL: xf
// holds f32 h rows, RMS-normalised here, times gamma, rounded to dtype (epi
// STORE or SWIGLU); gamma == NULL: xf holds dtype, epi ADD_F32.
int skinny_launch(int32_t dtype, int64_t m, int32_t n, int32_t k, const void* xf, const void* gamma, float eps,
                  const void* w, int32_t epi, void* y, int64_t ys, void* yf, const SkinnyNext& next,
                  hipStream_t st);

// Token rows up to which a layer runs this way. Measured against the general
// path, us per encode of the 0.6B shape: bf16 897 / 2,066 at 17 rows, 1,184 /
// 2,205 at 64, 1,719 / 2,154 at 128 (there every projection is two workgroup
// rows, and 256 rows would be four); f32 1,575 / 2,412 at 17, 2,261 / 2,825 at
// 64, 3,298 / 2,648 at 128: f32 MFMAs take 16 times as long.
constexpr int64_t FEW_ROWS_BF16 = 128, FEW_ROWS_F32 = 64;

// Whether the launches prefetch: while one row of workgroups covers all n rows (64
// in bf16, 32 in f32). The workgroups of a second row would wait behind the
// prefetchers. us per encode of the 0.6B shape, with / without: bf16 17 rows 914 /
// 994, 64 rows 1,287 / 1,379, 128 rows (two rows of workgroups) 1,742 / 1,725; f32
// 8 rows 1,161 / 1,303, 32 rows 1,590 / 1,701, 48 rows (two) 2,415 / 1,983, 64
// rows (two) 2,710 / 2,261.
bool few_prefetch(int32_t dtype, int64_t n);

// Whether a batch (n rows, longest text) of a model of this shape can.
bool few_fits(int32_t dtype, int64_t n, int32_t longest, int32_t hidden, int32_t heads, int32_t kv_heads,
              int32_t head_dim, int32_t intermediate);

// Bytes of the fragments of f32 h rows, and of dtype rows of `width`.
size_t few_h_bytes(int64_t n, int32_t hidden);
size_t few_x_bytes(int32_t dtype, int64_t n, int64_t width);

// h rows (f32 [n, hidden]) and their fragments from the embedding table.
int few_embed(int32_t dtype, int64_t n, const int32_t* ids, const void* table, int64_t vocab, int32_t hidden, float* h,
              void* hf, hipStream_t st);

// Causal attention (scale 1 / sqrt(128)) of the texts at device offsets cu,
// q/k norms and RoPE included, from q/k/v rows of qs elements to fragments of.
int few_attn(int32_t dtype, int32_t n_texts, int64_t n, int32_t longest, const int32_t* cu, const void* qkv, int64_t qs,
             int32_t heads, int32_t kv_heads, const void* qw, const void* kw, float eps, const float* cos,
             const float* sin, void* of, const SkinnyNext& next, hipStream_t st);

}  // namespace inl
