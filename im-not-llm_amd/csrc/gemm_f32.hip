// f32 GEMM on the bf16 matrix cores (gfx950): y[m, n] = x[m, k] . w[n, k]^T
// with f32 operands, results and accuracy, for the f32 encoder's projections.
//
// The f32 MFMA does 256 multiply-adds per clock and CU, the bf16 one 2,048. A
// f32 value is the sum of three bf16 values (8 + 8 + 8 significand bits, each
// rounded to nearest), and of the nine products of two such sums three are
// below 2^-26 of the whole: six bf16 products give what one f32 product gives,
// in three quarters of the time. They are exact, and are summed in f32 by the
// MFMA, the leading ones and the small ones apart, so that a small product
// rounds at its own size. Against f64 the error is below that of an f32 MFMA
// chain (k / 16 roundings instead of k / 4): a 28-layer encode of 800 rows is
// 4.9e-7 off, with f32 MFMA GEMMs it was 1.7e-6. What has no such parts (an
// infinity, or a value above 3.39e38, which rounds to one in bf16: the remainder
// is inf - inf) makes every product it enters NaN. A wave that finds a NaN among
// its results therefore multiplies its block again, on the f32 MFMA.
//
// Kernel: 128 x 128 tiles, 8 waves as 2 (w rows) x 4 (x rows), each 64 x 32 =
// 2 blocks of v_mfma_f32_32x32x16_bf16. A stage of 32 k goes from memory to
// registers (f32, coalesced, two stages ahead), is split once per workgroup
// (11 instructions per two values) and lies in LDS as three planes in operand
// order; two stages of LDS, one barrier per stage. Splitting costs about as
// many issue slots as multiplying, so the two waves of a SIMD (w and w + 4)
// take the two halves of a stage in opposite order: one multiplies stage s
// while the other splits stage s + 1. Splitting first in both, with 128 x 64
// tiles and two workgroups per CU, took 62 us for the 0.6B shape's q/k/v
// projection of 778 rows, this 50.
//
// Narrow outputs (o and down projections) leave CUs idle; their k is cut into
// up to 8 parts whose products go to a workspace, and the kernel that follows
// anyway, the residual add and row norm, adds them up in a fixed order.
//
// Tile order: workgroup b runs on XCD b % 8. When the w tiles divide by 8 an
// XCD takes a contiguous eighth of them for all x rows: w comes from HBM once,
// and x (a few MB) is shared in each L2.
#include <algorithm>
#include <cmath>

#include "attn_stream.hpp"
#include "gemm_f32.hpp"
#include "lanes.hpp"

namespace inl {

namespace {

constexpr int GF_BN = 128, GF_BM = 128, GF_BK = 32;
constexpr int GF_THREADS = 512;
constexpr int GF_FRAG = 1024;                                // 32 rows x 16 k of one plane
constexpr int GF_BLOCKS = (GF_BN + GF_BM) / 32;              // 4 of w, 4 of x
constexpr int GF_STAGE = GF_BLOCKS * 2 * 3 * GF_FRAG;        // 48 KiB
constexpr int GF_LDS = 2 * GF_STAGE;
constexpr int GF_LOADS = (GF_BN + GF_BM) * GF_BK / 4 / GF_THREADS;  // 16-byte loads per thread and stage

struct GemmF32Params {
  const char* x;
  const char* w;
  char* y;
  int64_t xs, ws, ys;       // elements between rows
  int32_t m, n, k;          // n: output columns
  int32_t nt, mt, splits;   // tiles
  int64_t part;             // elements between the outputs of two k parts
};

// Slot of (row, half of 8 k) in a fragment of k step s: 16 bytes per slot,
// rows swizzled so that the 4 rows x 4 quarters of k that half a wave writes
// at a time cover all banks.
__device__ __forceinline__ int gf_slot(int row, int hf, int s) { return hf * 32 + (row ^ ((2 * s + hf) << 2)); }

template <int EPI>
__global__ __launch_bounds__(GF_THREADS) void gemm_f32_kernel(GemmF32Params p) {
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wn = wave >> 2, wm = wave & 3;
  const int l32 = lane & 31, hf = lane >> 5;
  int nt, mt, sp;
  {
    const int per = p.mt * p.splits;   // workgroups of one w tile
    int id = blockIdx.x;
    if (p.nt % 8 == 0) id = (id % 8) * (p.nt / 8 * per) + id / 8;
    nt = id / per;
    id -= nt * per;
    sp = id / p.mt;
    mt = id - sp * p.mt;
  }
  const int kp = p.k / p.splits;       // k of this part
  const int stages = kp / GF_BK;
  // w tile: rows n0 .., or (SwiGLU) 32 gate rows, their 32 up rows, and again:
  // a wave's two blocks are then the two factors of the same outputs
  constexpr int BNO = EPI == GF_SWIGLU ? GF_BN / 2 : GF_BN;
  const int n0 = nt * BNO, m0 = mt * GF_BM;

  // this thread's loads: row r of the stage (w rows, then x rows), k chunk c
  const int c = tid & 7;
  uint32_t off[GF_LOADS];
  int dst[GF_LOADS];
  const char* wb = p.w + ((int64_t)n0 * p.ws + (int64_t)sp * kp) * 4;
  const char* xb = p.x + ((int64_t)m0 * p.xs + (int64_t)sp * kp) * 4;
  const int64_t w_span = EPI == GF_SWIGLU ? (int64_t)p.n + BNO : GF_BN;   // rows the w buffer covers
  const __amdgpu_buffer_rsrc_t wr = pp_rsrc(wb, (uint32_t)(((w_span - 1) * p.ws + kp) * 4));
  const int xrows = min(GF_BM, p.m - m0);
  const __amdgpu_buffer_rsrc_t xr = pp_rsrc(xb, (uint32_t)(((int64_t)(xrows - 1) * p.xs + kp) * 4));
#pragma unroll
  for (int i = 0; i < GF_LOADS; ++i) {
    const int r = (GF_THREADS / 8) * i + (tid >> 3), blk = r >> 5;
    uint32_t row;
    int64_t stride;
    const bool is_w = i < GF_BN * 8 / GF_THREADS;
    if (is_w) {
      row = EPI == GF_SWIGLU ? (uint32_t)((blk >> 1) * 32 + (r & 31) + ((blk & 1) ? p.n : 0)) : (uint32_t)r;
      stride = p.ws;
    } else {
      row = (uint32_t)(r - GF_BN);
      stride = p.xs;
    }
    const bool dead = !is_w && (int)row >= xrows;   // reads zeros past the buffer's end
    off[i] = dead ? 0x80000000u : (uint32_t)(row * stride * 4) + c * 16;
    const int s = c >> 2, h = c & 1;             // k = 16 s + 8 half + 4 h
    dst[i] = (blk * 2 + s) * 3 * GF_FRAG + gf_slot(r & 31, (c >> 1) & 1, s) * 16 + h * 8;
  }
  // Loads past a part's last stage read the next part's k, or zeros: they are
  // never multiplied.
  auto fetch = [&](f32x4 (&raw)[GF_LOADS], int stage) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < GF_LOADS; ++i)
      raw[i] = __builtin_bit_cast(
          f32x4, __builtin_amdgcn_raw_buffer_load_b128(i < GF_BN * 8 / GF_THREADS ? wr : xr, off[i], stage * GF_BK * 4, 0));
  };
  // three bf16 parts of each value, to the stage's planes
  auto split = [&](const f32x4 (&raw)[GF_LOADS], int buf) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < GF_LOADS; ++i) {
      u32x2 o[3];
      bf16_parts4(raw[i], o);
#pragma unroll
      for (int n = 0; n < 3; ++n) *reinterpret_cast<u32x2*>(smem + buf * GF_STAGE + dst[i] + n * GF_FRAG) = o[n];
    }
  };
  const f32x16 zero = {};
  f32x16 hi[2] = {zero, zero}, lo[2] = {zero, zero};
  auto multiply = [&](int buf) __attribute__((always_inline)) {
    const char* st = smem + buf * GF_STAGE;
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const int slot = gf_slot(l32, hf, t) * 16;
      bf16x8 b[3], a[2][3];
#pragma unroll
      for (int n = 2; n >= 0; --n) {
        b[n] = *reinterpret_cast<const bf16x8*>(st + (((GF_BN / 32 + wm) * 2 + t) * 3 + n) * GF_FRAG + slot);
#pragma unroll
        for (int q = 0; q < 2; ++q)
          a[q][n] = *reinterpret_cast<const bf16x8*>(st + (((wn * 2 + q) * 2 + t) * 3 + n) * GF_FRAG + slot);
      }
#pragma unroll
      for (int d = 2; d >= 0; --d)
#pragma unroll
        for (int i = 0; i <= d; ++i)
#pragma unroll
          for (int q = 0; q < 2; ++q) {
            f32x16& acc = d ? lo[q] : hi[q];
            acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[q][i], b[d - i], acc, 0, 0, 0);
          }
    }
  };
  // One stage: multiply it and split the next (`raw`), whose registers then
  // take the loads of the stage after that one's successor. The order of the
  // halves is the wave's.
  auto stage = [&](int s, int buf, f32x4 (&raw)[GF_LOADS]) __attribute__((always_inline)) {
    if (wave < 4) {
      multiply(buf);
      __builtin_amdgcn_sched_barrier(0);
      split(raw, buf ^ 1);
      fetch(raw, s + 3);
    } else {
      split(raw, buf ^ 1);
      fetch(raw, s + 3);
      __builtin_amdgcn_sched_barrier(0);
      multiply(buf);
    }
    __builtin_amdgcn_sched_barrier(0);
    lds_barrier();
  };

  f32x4 r0[GF_LOADS], r1[GF_LOADS];
  fetch(r0, 0);
  fetch(r1, 1);
  split(r0, 0);
  fetch(r0, 2);
  lds_barrier();
  int s = 0;
  for (; s + 2 <= stages; s += 2) {
    stage(s, 0, r1);
    stage(s + 1, 1, r0);
  }
  if (s < stages) stage(s, 0, r1);

  {
    float s = 0.f;   // NaN if a result is NaN (or infinite)
#pragma unroll
    for (int q = 0; q < 2; ++q)
#pragma unroll
      for (int r = 0; r < 16; ++r) s = __builtin_fmaf(hi[q][r] + lo[q][r], 0.f, s);
    if (__any(s != s)) {
      // lane half hf takes 4 k of each 8, of w row l32 of a block and x row l32
      const int xrow = wm * 32 + l32;
      const uint32_t xo = xrow < xrows ? (uint32_t)(xrow * p.xs * 4) + hf * 16 : 0x80000000u;
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        const int wrow = EPI == GF_SWIGLU ? wn * 32 + l32 + q * p.n : (wn * 2 + q) * 32 + l32;
        const uint32_t wo = (uint32_t)(wrow * p.ws * 4) + hf * 16;
        hi[q] = lo[q] = zero;
#pragma nounroll
        for (int k = 0; k < kp; k += 8) {
          const f32x4 a = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(wr, wo, k * 4, 0));
          const f32x4 b = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(xr, xo, k * 4, 0));
#pragma unroll
          for (int e = 0; e < 4; ++e) hi[q] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[e], b[e], hi[q], 0, 0, 0);
        }
      }
    }
  }

  // Epilogue: lane holds x row l32 of its wave's 32, w rows 8 g + 4 hf + e of
  // each block. Through LDS (32 rows x 272 bytes per wave), so that a store
  // instruction writes 4 rows x 256 bytes (SwiGLU: 8 x 128).
  constexpr int ROWB = 64 * 4 + 16;
  char* stg = smem + wave * (32 * ROWB);
  constexpr int NQ = EPI == GF_SWIGLU ? 1 : 2;
#pragma unroll
  for (int q = 0; q < NQ; ++q)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      f32x4 v;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float a = hi[q][4 * g + e] + lo[q][4 * g + e];
        if constexpr (EPI == GF_SWIGLU) {
          const float u = hi[1][4 * g + e] + lo[1][4 * g + e];
          v[e] = a / (1.0f + expf(-a)) * u;
        } else {
          v[e] = a;
        }
      }
      *reinterpret_cast<f32x4*>(stg + l32 * ROWB + (q * 32 + 8 * g + 4 * hf) * 4) = v;
    }
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // this wave's own staging
  constexpr int CH = NQ * 8;   // 16-byte chunks per row
  float* y = reinterpret_cast<float*>(p.y) + (EPI == GF_PART ? sp * p.part : 0);
#pragma unroll
  for (int j = 0; j < 32 * CH / 64; ++j) {
    const int r = (j * 64 + lane) / CH, ch = lane % CH;
    const f32x4 v = *reinterpret_cast<const f32x4*>(stg + r * ROWB + ch * 16);
    const int row = m0 + wm * 32 + r;
    if (row < p.m) *reinterpret_cast<f32x4*>(y + row * p.ys + n0 + wn * (NQ * 32) + ch * 4) = v;
  }
}

// ---- h += the parts; x = rms_norm(h) * gamma (gamma NULL: h alone) ----
// One wave per row of at most 2,048 values, held in registers.
template <int K>
__global__ __launch_bounds__(256) void add_norm_kernel(float* h, const float* part, int64_t part_stride, int32_t parts,
                                                       const float* gamma, float eps, int64_t rows, int32_t dim,
                                                       float* x) {
  const int64_t r = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (r >= rows) return;
  f32x4 v[K];
  float ss = 0.f;
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const int i = lane * 4 + 256 * k;
    const int64_t at = r * dim + (i < dim ? i : 0);
    f32x4 t = *reinterpret_cast<const f32x4*>(part + at);
    for (int s = 1; s < parts; ++s) t += *reinterpret_cast<const f32x4*>(part + s * part_stride + at);
    v[k] = *reinterpret_cast<const f32x4*>(h + at) + t;
    if (i >= dim) v[k] = (f32x4){0.f, 0.f, 0.f, 0.f};
    ss += (v[k][0] * v[k][0] + v[k][1] * v[k][1]) + (v[k][2] * v[k][2] + v[k][3] * v[k][3]);
  }
  const float inv = 1.0f / sqrtf(wave_sum(ss) / (float)dim + eps);
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const int i = lane * 4 + 256 * k;
    if (i >= dim) continue;
    *reinterpret_cast<f32x4*>(h + r * dim + i) = v[k];
    if (gamma) *reinterpret_cast<f32x4*>(x + r * dim + i) = v[k] * inv * *reinterpret_cast<const f32x4*>(gamma + i);
  }
}

}  // namespace

bool gemm_f32_fits(int32_t hidden, int32_t qkv_rows, int32_t attn_width, int32_t intermediate) {
  return hidden % GF_BN == 0 && hidden <= 2048 && qkv_rows % GF_BN == 0 && attn_width % GF_BK == 0 &&
         intermediate % GF_BN == 0 && (int64_t)(2 * (int64_t)intermediate) * hidden * 4 < ((int64_t)1 << 31) &&
         (int64_t)GF_BN * std::max(attn_width, intermediate) * 4 < ((int64_t)1 << 31);
}

bool gemm_f32_pays(int64_t m, int32_t qkv_rows) {
  const int64_t tiles = (m + GF_BM - 1) / GF_BM * (qkv_rows / GF_BN);
  return m > 464 && tiles >= 128;
}

int gemm_f32_splits(int64_t m, int32_t n, int32_t k, int cus, size_t part_bytes) {
  // parts until every CU has a workgroup, while a part keeps 8 stages
  const int64_t tiles = (m + GF_BM - 1) / GF_BM * (n / GF_BN);
  int s = 1;
  while (s < 8 && tiles * s * 2 <= (int64_t)cus && k % (s * 2 * GF_BK) == 0 && k / (s * 2) >= 8 * GF_BK &&
         (size_t)(s * 2) * m * n * 4 <= part_bytes)
    s *= 2;
  return s;
}

int gemm_f32_launch(int64_t m, int32_t n, int32_t k, const float* x, int64_t xs, const float* w, int32_t epi,
                    int32_t splits, float* y, int64_t ys, hipStream_t st) {
  GemmF32Params p{};
  p.x = (const char*)x;
  p.w = (const char*)w;
  p.y = (char*)y;
  p.xs = xs;
  p.ws = k;
  p.ys = ys;
  p.m = (int32_t)m;
  p.n = n;
  p.k = k;
  p.nt = n / (epi == GF_SWIGLU ? GF_BN / 2 : GF_BN);
  p.mt = (int32_t)((m + GF_BM - 1) / GF_BM);
  p.splits = splits;
  p.part = m * ys;
  const dim3 grid((unsigned)(p.nt * p.mt * splits));
  const void* fn = epi == GF_STORE ? (const void*)gemm_f32_kernel<GF_STORE>
                   : epi == GF_PART ? (const void*)gemm_f32_kernel<GF_PART> : (const void*)gemm_f32_kernel<GF_SWIGLU>;
  const int rc = set_max_dynamic_lds(fn, GF_LDS);
  if (rc) return rc;
  void* args[] = {&p};
  INL_HIP_TRY(hipLaunchKernel(fn, grid, dim3(GF_THREADS), args, GF_LDS, st));
  return INL_OK;
}

int add_norm_launch(int64_t rows, int32_t dim, float* h, const float* part, int32_t parts, const float* gamma, float eps,
                    float* x, hipStream_t st) {
  const dim3 grid((unsigned)((rows + 3) / 4));
  if (dim <= 1024)
    hipLaunchKernelGGL(add_norm_kernel<4>, grid, dim3(256), 0, st, h, part, rows * dim, parts, gamma, eps, rows, dim, x);
  else
    hipLaunchKernelGGL(add_norm_kernel<8>, grid, dim3(256), 0, st, h, part, rows * dim, parts, gamma, eps, rows, dim, x);
  INL_HIP_TRY(hipGetLastError());
  return INL_OK;
}

}  // namespace inl
