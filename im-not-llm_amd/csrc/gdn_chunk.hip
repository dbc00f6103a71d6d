// The gated delta rule in chunks, on the matrix cores (gfx950).
//
// The per-token recurrence (gdn.hip) is bound by vector FMAs and by its
// serial chain: 0.59 us per token of the longest text at 16 heads, whatever
// else the chip has to do. Over a chunk of C tokens the same recurrence is
// (the reference's own chunked form, crates/inl-late/src/qwen3_5.rs:607-728):
//
//   A_ij = beta_i (k_i . k_j) e^(c_i - c_j), j < i        c = running sum of g
//   T    = (I + A)^-1 diag(beta)
//   R    = V - e^c K S          (rows scaled)             S: the state [dk, dv]
//   U    = T R
//   O    = e^c Q S + P U,       P_ij = (q_i . k_j) e^(c_i - c_j), j <= i
//   S   <- e^(c_C) S + K^T (e^(c_C - c) U)
//
// Measured against the per-token kernel, rule alone, 16 heads, bf16: 16 texts
// of 80 to 1,453 tokens 861 -> 243 us, 16 texts of 2,048 1,216 -> 462 us.
//
// What a product cannot do: 0 times inf or NaN is NaN, so a token's inf or NaN
// would reach earlier tokens of its chunk, and unnormalised K and Q overflow
// where k / |k| does not. Each of these leaves a chunk's results not finite, so a
// wave that finds such results takes its columns from that chunk's first token on
// by the recurrence itself, once its loop is over (S waits in its registers).
//
// Two kernels. gdn_chunk_prep computes T and P of every chunk of every text
// at once (one wave per chunk and head) and leaves them in the rows of `out`
// that the chunk's results will replace: 2 C values of the row's 128, so no
// workspace is needed. gdn_chunk_rule walks a text's chunks, one workgroup of
// 8 waves per (text, head), wave w holding columns 16 w .. 16 w + 15 of S, U
// and O in registers; only what all columns share (K, Q, K^T, T, P) is in LDS,
// in operand order, so a chunk costs two barriers.
//
// Precision. State, R, U, T and P are f32 and enter the products as three
// bf16 parts each (8 + 8 + 8 significand bits, rounded to nearest: the parts
// add up to the f32 value), of whose nine products the six above 2^-27 are
// summed in f32 by the MFMAs. bf16 K and Q are taken raw, as the one exact
// part they are (three products), and their norms scale rows of the results.
// The running sum of g is kept in f64 and takes no g below -1,000 (e^g is 0 in
// f32 from -104 on): it stays within 64,000 of zero, where an ulp is 7e-12, so
// that e^(c_i - c_j) is exact to f32 after any reset, -inf included. Against
// the f64 recurrence the error is no larger than the per-token kernel's.
//
// An MFMA contraction of 32 takes its terms in any order that both operands
// share. Here lane group g = lane / 16, element e = 4 h + r holds term 16 h +
// 4 g + r: that is how a product's own registers lie (row 4 g + r of block h),
// so S, R and U feed the next product without leaving their lane.
#include "gdn_chunk.hpp"
#include "attn_stream.hpp"
#include "lanes.hpp"

namespace inl {

namespace {

constexpr int GC_D = 128;     // key and value dim
constexpr int GC_WAVES = 8;

template <typename T>
constexpr int gc_len() { return sizeof(T) == 2 ? 64 : 32; }   // f32: three parts of K, Q, K^T fit LDS at 32
template <typename T>
constexpr int gc_parts() { return sizeof(T) == 2 ? 1 : 3; }

// An operand's values as N bf16 parts.
template <int N>
__device__ __forceinline__ void gc_split(const float (&x)[8], bf16x8 (&p)[N]) {
  u32x4 w[N];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    uint32_t u[N];
    bf16_parts<N>((f32x2){x[2 * j], x[2 * j + 1]}, u);
#pragma unroll
    for (int n = 0; n < N; ++n) w[n][j] = u[n];
  }
#pragma unroll
  for (int n = 0; n < N; ++n) p[n] = __builtin_bit_cast(bf16x8, w[n]);
}
// hi + lo += a . b over 32 terms: the leading parts' product in hi, the smaller
// ones in lo (their sum rounds at its own size), those below 2^-26 dropped.
template <int NA, int NB>
__device__ __forceinline__ void gc_mm(const bf16x8 (&a)[NA], const bf16x8 (&b)[NB], f32x4& hi, f32x4& lo) {
#pragma unroll
  for (int s = 2; s > 0; --s)
#pragma unroll
    for (int i = 0; i < NA; ++i)
      if (s - i >= 0 && s - i < NB) lo = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i], b[s - i], lo, 0, 0, 0);
  hi = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[0], b[0], hi, 0, 0, 0);
}

// Eight values of T as loaded, and as bf16 parts.
template <typename T>
struct Raw;
template <>
struct Raw<bf16> {
  bf16x8 v;
  __device__ __forceinline__ float squares() const {
    float s = 0.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) s += (float)v[e] * (float)v[e];
    return s;
  }
  __device__ __forceinline__ void parts(bf16x8 (&p)[1]) const { p[0] = v; }
};
template <>
struct Raw<float> {
  float v[8];
  __device__ __forceinline__ float squares() const {
    float s = 0.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) s += v[e] * v[e];
    return s;
  }
  __device__ __forceinline__ void parts(bf16x8 (&p)[3]) const { gc_split<3>(v, p); }
};
// Loads at byte offset `off` of a buffer that starts at a chunk's first row and
// ends with the text: rows past the end read as zeros, without a clamp or a
// mask. The 8 terms of one operand and step: 4 at off, 4 at off + 16 terms.
template <typename T>
__device__ __forceinline__ void gc_load(Raw<T>& x, __amdgpu_buffer_rsrc_t r, uint32_t off) {
  if constexpr (sizeof(T) == 2) {
    const u32x2 a = __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(r, off, 0, 0));
    const u32x2 b = __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(r, off + 32, 0, 0));
    const u32x4 w = {a[0], a[1], b[0], b[1]};
    x.v = __builtin_bit_cast(bf16x8, w);
  } else {
    const f32x4 a = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0));
    const f32x4 b = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(r, off + 64, 0, 0));
#pragma unroll
    for (int e = 0; e < 4; ++e) { x.v[e] = a[e]; x.v[4 + e] = b[e]; }
  }
}
__device__ __forceinline__ float gc_load_f32(__amdgpu_buffer_rsrc_t r, uint32_t off) {
  return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, off, 0, 0));
}

// Clamped bounds of text b (a malformed table gives wrong rows, never an
// access outside the tensors).
__device__ __forceinline__ void gc_bounds(const int32_t* cu, int b, int64_t n, int64_t* begin, int64_t* end) {
  const int64_t c0 = cu[b], c1 = cu[b + 1];
  *begin = c0 < 0 ? 0 : (c0 > n ? n : c0);
  *end = c1 < *begin ? *begin : (c1 > n ? n : c1);
}

// Inclusive sum over the wave's lanes, in f64.
__device__ __forceinline__ double gc_scan(double x, int lane) {
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const double y = __shfl_up(x, d, 64);
    if (lane >= d) x += y;
  }
  return x;
}

// The buffers of the chunk at row t0: `rows` rows of a tensor of f32 or T.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t gc_rows_of(const void* base, int64_t t0, int64_t stride,
                                                              int rows, int64_t width, int esize) {
  return pp_rsrc(static_cast<const char*>(base) + t0 * stride * esize,
                 (uint32_t)(((rows - 1) * stride + width) * esize));
}

// One wave per (chunk, value head). The chunks of text b are numbered from
// cu[b] / C + b on: a device-side numbering without a prefix sum, with at most
// one unused number per text.
//
// The inverse is taken by 16 x 16 blocks: the four diagonal blocks by forward
// substitution side by side (lane = 16 block + column, 120 FMAs each), then
// X_rc = -D_r sum_k A_rk X_kc on the f32 MFMAs, whose D registers (rows 4 g +
// r) are the next product's B operand. One column of 64 per lane, 2,016 FMAs
// in a chain of 64 rows, made the kernel 60 us at 138 chunks x 16 heads; this
// form takes 45.
template <typename T>
__global__ __launch_bounds__(256) void gdn_chunk_prep(GdnChunkParams p) {
  constexpr int C = gc_len<T>(), RB = C / 16, NP = gc_parts<T>(), AS = C + 4;
  __shared__ __attribute__((aligned(16))) float s_a[4][C][AS];
  __shared__ __attribute__((aligned(16))) float s_d[4][RB][16][20];
  __shared__ __attribute__((aligned(16))) float s_ki[4][C], s_beta[4][C], s_qi[4][C];
  __shared__ __attribute__((aligned(16))) double s_cum[4][C];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int i16 = lane & 15, g = lane >> 4;
  const int h = blockIdx.y * 4 + wave;
  if (h >= p.nv) return;   // no workgroup barrier below
  int lo = 0, hi = p.n_texts - 1;   // the last text whose numbers start at or before this one
  const int64_t slot = blockIdx.x;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    int64_t b0, b1;
    gc_bounds(p.cu, mid, p.n, &b0, &b1);
    if (b0 / C + mid <= slot) lo = mid;
    else hi = mid - 1;
  }
  int64_t begin, end;
  gc_bounds(p.cu, lo, p.n, &begin, &end);
  const int64_t t0 = begin + (slot - begin / C - lo) * C;
  if (t0 < begin || t0 >= end) return;
  const int rows = (int)min((int64_t)C, end - t0);
  const int kh = h / (p.nv / p.nk);
  const int ES = (int)sizeof(T);
  const int64_t width = (int64_t)2 * p.nk * GC_D + (int64_t)p.nv * GC_D;
  const __amdgpu_buffer_rsrc_t mr = gc_rows_of(p.mixed, t0, p.ms, rows, width, ES);
  const __amdgpu_buffer_rsrc_t gr = gc_rows_of(p.g, t0, p.gs, rows, p.nv, 4);
  const __amdgpu_buffer_rsrc_t br = gc_rows_of(p.beta, t0, p.gs, rows, p.nv, 4);
  const __amdgpu_buffer_rsrc_t orr = gc_rows_of(p.out, t0, p.os, rows, (int64_t)p.nv * GC_D, 4);
  auto sync = [] __attribute__((always_inline)) () {   // this wave's LDS writes, read by its other lanes
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  };

  // 16 rows as operands; returns their sums of squares
  auto load_rows = [&](int64_t off, int rb, bf16x8 (&f)[4][NP]) __attribute__((always_inline)) {
    const uint32_t at = (uint32_t)((16 * rb + i16) * p.ms + off + 4 * g) * ES;
    Raw<T> x[4];
#pragma unroll
    for (int s = 0; s < 4; ++s) gc_load<T>(x[s], mr, at + 32 * s * ES);
    float ss = 0.f;
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      ss += x[s].squares();
      x[s].parts(f[s]);
    }
    return rows4_sum(ss);
  };
  auto dot = [&](const bf16x8 (&a)[4][NP], const bf16x8 (&b)[4][NP]) __attribute__((always_inline)) {
    f32x4 hi = {0.f, 0.f, 0.f, 0.f}, lo = hi;
#pragma unroll
    for (int s = 0; s < 4; ++s) gc_mm<NP, NP>(a[s], b[s], hi, lo);
    if constexpr (NP > 1) hi += lo;
    return hi;
  };
  const int64_t q_off = (int64_t)kh * GC_D, k_off = (int64_t)(p.nk + kh) * GC_D;
  float gv = lane < C ? gc_load_f32(gr, (uint32_t)(lane * p.gs + h) * 4) : 0.f;
  gv = gv < -1000.f ? -1000.f : gv;   // (a NaN stays)
  const float bv = lane < C ? gc_load_f32(br, (uint32_t)(lane * p.gs + h) * 4) : 0.f;
  bf16x8 kf[RB][4][NP];
#pragma unroll
  for (int rb = 0; rb < RB; ++rb) {
    const float ss = load_rows(k_off, rb, kf[rb]);
    if (lane < 16) s_ki[wave][16 * rb + lane] = 1.0f / sqrtf(ss + 1e-6f);
  }
  const double cum = gc_scan((double)gv, lane);
  {
    if (lane < C) {
      s_cum[wave][lane] = cum;
      s_beta[wave][lane] = bv;
    }
  }
  const float dk_scale = 1.0f / sqrtf((float)GC_D);
  auto put = [&](int i, int c, float v) __attribute__((always_inline)) {   // rows past the end are dropped
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, v), orr,
                                          (uint32_t)(i * p.os + (int64_t)h * GC_D + c) * 4, 0, 0);
  };
#pragma unroll
  for (int rb = 0; rb < RB; ++rb) {
    bf16x8 qf[4][NP];
    const float qs = load_rows(q_off, rb, qf);
    if (lane < 16) s_qi[wave][16 * rb + lane] = dk_scale / sqrtf(qs + 1e-6f);
    sync();
    const f32x4 ki = *reinterpret_cast<const f32x4*>(&s_ki[wave][16 * rb + 4 * g]);
    const f32x4 bi = *reinterpret_cast<const f32x4*>(&s_beta[wave][16 * rb + 4 * g]);
    const f32x4 qi = *reinterpret_cast<const f32x4*>(&s_qi[wave][16 * rb + 4 * g]);
    double ci[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) ci[r] = s_cum[wave][16 * rb + 4 * g + r];
#pragma unroll
    for (int cb = 0; cb <= rb; ++cb) {
      const f32x4 kk = dot(kf[rb], kf[cb]), qk = dot(qf, kf[cb]);
      const int j = 16 * cb + i16;
      const float kj = s_ki[wave][j];
      const double cj = s_cum[wave][j];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int i = 16 * rb + 4 * g + r;
        const float dec = i >= j ? expf((float)(ci[r] - cj)) * kj : 0.f;
        s_a[wave][i][j] = kk[r] * ki[r] * dec * bi[r];
        put(i, 64 + j, i >= j ? qk[r] * qi[r] * dec : 0.f);
      }
    }
    if (rb % 2 == 0)   // the other half of the operand's 32 columns
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        put(16 * rb + 4 * g + r, 64 + 16 * (rb + 1) + i16, 0.f);
        put(16 * rb + 4 * g + r, 16 * (rb + 1) + i16, 0.f);
      }
  }
  sync();
  if (lane < rows) {
    // The chunk's row scales, in columns of T that no operand reads (those of
    // rows 0 .. 31 past the first step): token t in row t % 32.
    const double all = s_cum[wave][rows - 1];
    const float ec = expf((float)cum);
    const int c = 32 + 4 * (lane >> 5);
    put(lane & 31, c, ec * s_ki[wave][lane]);
    put(lane & 31, c + 1, ec * s_qi[wave][lane]);
    put(lane & 31, c + 2, expf((float)(all - cum)) * s_ki[wave][lane]);
    if (lane == 0) put(0, 35, expf((float)all));
  }
  {   // diagonal blocks: lane holds column i16 of block g
    const int blk = g < RB ? g : 0;
    float x[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      float s0 = 0.f, s1 = 0.f;
#pragma unroll
      for (int k = 0; k < i; k += 4) {
        const f32x4 a = *reinterpret_cast<const f32x4*>(&s_a[wave][16 * blk + i][16 * blk + k]);
        s0 = __builtin_fmaf(a[0], x[k], s0);
        if (k + 1 < i) s1 = __builtin_fmaf(a[1], x[k + 1], s1);
        if (k + 2 < i) s0 = __builtin_fmaf(a[2], x[k + 2], s0);
        if (k + 3 < i) s1 = __builtin_fmaf(a[3], x[k + 3], s1);
      }
      x[i] = i16 == i ? 1.0f : -(s0 + s1);
      if (g < RB) s_d[wave][blk][i][i16] = x[i];
    }
  }
  sync();
  f32x4 X[RB][RB];   // X[rb][cb]: rows 16 rb + 4 g + r, column 16 cb + i16
  auto mm16 = [&](const f32x4& a, const f32x4& b, f32x4 acc) __attribute__((always_inline)) {
#pragma unroll
    for (int r = 0; r < 4; ++r) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a[r], b[r], acc, 0, 0, 0);
    return acc;
  };
#pragma unroll
  for (int rb = 0; rb < RB; ++rb) {
    const f32x4 d = *reinterpret_cast<const f32x4*>(&s_d[wave][rb][i16][4 * g]);
#pragma unroll
    for (int r = 0; r < 4; ++r) X[rb][rb][r] = s_d[wave][rb][4 * g + r][i16];
#pragma unroll
    for (int cb = 0; cb < rb; ++cb) {
      f32x4 y = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int kb = cb; kb < rb; ++kb)
        y = mm16(*reinterpret_cast<const f32x4*>(&s_a[wave][16 * rb + i16][16 * kb + 4 * g]), X[kb][cb], y);
      X[rb][cb] = -mm16(d, y, (f32x4){0.f, 0.f, 0.f, 0.f});
    }
#pragma unroll
    for (int cb = 0; cb <= rb; ++cb) {
      const float bj = s_beta[wave][16 * cb + i16];
#pragma unroll
      for (int r = 0; r < 4; ++r) put(16 * rb + 4 * g + r, 16 * cb + i16, X[rb][cb][r] * bj);
    }
  }
}

// LDS of gdn_chunk_rule: fragments of 1 KiB, 16 bytes per lane. Row i of lane
// group g sits at slot 16 g + (i ^ x); x, a constant of the fragment and lane
// group, spreads what a wave writes at a time over the banks: it loads whole
// rows (a load of 16 bytes per lane from 16 rows runs at a quarter of the rate
// of one from 4), so its lanes write one or two rows of many fragments. Against
// loads in operand order: gdn_chunk_rule 219 -> 197 us at 16 texts of 80 to
// 1,453 tokens, 16 heads, bf16. f32 still loads K, Q and K^T in operand order;
// whole rows were not tried there.
__device__ __forceinline__ int gc_slot(int g, int i, int x) { return (16 * g + (i ^ x)) * 16; }
template <typename T>
struct GcLds {
  static constexpr int C = gc_len<T>(), RB = C / 16, TS = C / 32, NP = gc_parts<T>();
  static constexpr int KF = 0;                        // [RB][4][NP]
  static constexpr int QF = KF + RB * 4 * NP * 1024;
  static constexpr int KT = QF + RB * 4 * NP * 1024;  // [8][TS][NP]
  static constexpr int TF = KT + 8 * TS * NP * 1024;  // [RB][TS][3]
  static constexpr int PF = TF + RB * TS * 3 * 1024;
  static constexpr int VEC = PF + RB * TS * 3 * 1024; // row scales [3][C] f32, e^(c_C)
  static constexpr int TOTAL = VEC + 3 * C * 4 + 16;
};

template <typename T>
__global__ __launch_bounds__(64 * GC_WAVES) void gdn_chunk_rule(GdnChunkParams p) {
  using L = GcLds<T>;
  constexpr int C = L::C, RB = L::RB, TS = L::TS, NP = L::NP;
  constexpr int FK = RB * 4 / GC_WAVES;   // KiB of K (and Q) a wave stages
  constexpr int FT = 8 * TS / GC_WAVES;   // K^T fragments
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  const int h = blockIdx.x, b = blockIdx.y;
  int64_t begin, end;
  gc_bounds(p.cu, b, p.n, &begin, &end);
  if (end <= begin) return;
  const int kh = h / (p.nv / p.nk);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int i16 = lane & 15, g = lane >> 4;
  const int ES = (int)sizeof(T);
  const int64_t width = (int64_t)2 * p.nk * GC_D + (int64_t)p.nv * GC_D;
  const uint32_t q_off = (uint32_t)kh * GC_D, k_off = (uint32_t)(p.nk + kh) * GC_D;
  const uint32_t v_off = (uint32_t)2 * p.nk * GC_D + (uint32_t)h * GC_D + 16 * wave + i16;
  const uint32_t ms = (uint32_t)p.ms, os = (uint32_t)p.os;
  // fragment i of an array, this lane's 16 bytes
  auto frag = [&](int base, int i, int x) __attribute__((always_inline)) {
    return reinterpret_cast<bf16x8*>(smem + base + i * 1024 + gc_slot(g, i16, x));
  };
  // the swizzles: K and Q of step s, K^T of block db, T and P of step ts
  auto x_k = [](int s) __attribute__((always_inline)) { return 4 * s; };
  auto x_t = [](int db) __attribute__((always_inline)) { return 2 * db; };
  auto x_l = [](int grp, int ts) __attribute__((always_inline)) { return 2 * grp | 8 * ts; };

  // registers of the chunk to come
  // bf16: 2 x 4 whole rows of K and Q; f32: operands. T and P: RT x 2 rows.
  constexpr int RT = C / 2 / GC_WAVES;
  Raw<T> rk[FK], rq[FK], rt[FT];
  f32x4 rl[RT];
  float rs[4];
  T rv[RB][4];
  auto load_t = [&](__amdgpu_buffer_rsrc_t r, uint32_t off) __attribute__((always_inline)) {
    if constexpr (sizeof(T) == 2)
      return __builtin_bit_cast(bf16, (unsigned short)__builtin_amdgcn_raw_buffer_load_b16(r, off, 0, 0));
    else return gc_load_f32(r, off);
  };
  auto fetch = [&](int64_t t0) __attribute__((always_inline)) {
    const int rows = (int)min((int64_t)C, end - t0);
    const __amdgpu_buffer_rsrc_t mr = gc_rows_of(p.mixed, t0, p.ms, rows, width, ES);
    const __amdgpu_buffer_rsrc_t orr = gc_rows_of(p.out, t0, p.os, rows, (int64_t)p.nv * GC_D, 4);
    if constexpr (NP == 1) {
#pragma unroll
      for (int f = 0; f < FK; ++f) {   // row 8 wave + 4 f + lane / 16, dims 8 (lane % 16) ..
        const uint32_t at = (8 * wave + 4 * f + g) * ms + 8 * i16;
        rk[f].v = __builtin_bit_cast(bf16x8, __builtin_amdgcn_raw_buffer_load_b128(mr, (at + k_off) * ES, 0, 0));
        rq[f].v = __builtin_bit_cast(bf16x8, __builtin_amdgcn_raw_buffer_load_b128(mr, (at + q_off) * ES, 0, 0));
      }
    } else {
#pragma unroll
      for (int f = 0; f < FK; ++f) {
        const int id = wave * FK + f, rb = id >> 2, s = id & 3;
        const uint32_t at = (16 * rb + i16) * ms + 32 * s + 4 * g;
        gc_load<T>(rk[f], mr, (at + k_off) * ES);
        gc_load<T>(rq[f], mr, (at + q_off) * ES);
      }
#pragma unroll
      for (int f = 0; f < FT; ++f) {
        const int id = wave * FT + f, db = id / TS, ts = id % TS;
#pragma unroll
        for (int e = 0; e < 8; ++e)
          rt[f].v[e] = load_t(mr, ((32 * ts + 16 * (e >> 2) + 4 * g + (e & 3)) * ms + k_off + 16 * db + i16) * ES);
      }
    }
#pragma unroll
    for (int f = 0; f < RT; ++f)   // row 2 (RT wave + f) + lane / 32, columns 4 (lane % 32) ..: T, then P
      rl[f] = __builtin_bit_cast(
          f32x4, __builtin_amdgcn_raw_buffer_load_b128(
                     orr, ((2 * (RT * wave + f) + (lane >> 5)) * os + (uint32_t)h * GC_D + 4 * (lane & 31)) * 4, 0, 0));
#pragma unroll
    for (int rb = 0; rb < RB; ++rb)
#pragma unroll
      for (int r = 0; r < 4; ++r) rv[rb][r] = load_t(mr, ((16 * rb + 4 * g + r) * ms + v_off) * ES);
    if (wave == GC_WAVES - 1) {   // row scales, one token per lane
#pragma unroll
      for (int n = 0; n < 4; ++n)
        rs[n] = gc_load_f32(orr, ((lane & 31) * os + (uint32_t)h * GC_D + 32 + 4 * (lane >> 5) + n) * 4);
    }
  };

  f32x4 S[8];   // rows 16 b + 4 g + r of column 16 wave + i16
#pragma unroll
  for (int i = 0; i < 8; ++i) S[i] = (f32x4){0.f, 0.f, 0.f, 0.f};
  float* vec = reinterpret_cast<float*>(smem + L::VEC);

  // The rows of the chunk at t0 by the recurrence itself, for this wave's 16
  // columns: lane (g, i16) holds rows 16 b + 4 g .. + 3 of its column.
  auto walk = [&](int64_t t0) __attribute__((always_inline)) {
    const int rows = (int)min((int64_t)C, end - t0);
    const __amdgpu_buffer_rsrc_t mr = gc_rows_of(p.mixed, t0, p.ms, rows, width, ES);
    const __amdgpu_buffer_rsrc_t orr = gc_rows_of(p.out, t0, p.os, rows, (int64_t)p.nv * GC_D, 4);
    const __amdgpu_buffer_rsrc_t gr = gc_rows_of(p.g, t0, p.gs, rows, p.nv, 4);
    const __amdgpu_buffer_rsrc_t br = gc_rows_of(p.beta, t0, p.gs, rows, p.nv, 4);
    // a token's values, loaded while the one before it is worked on
    Raw<T> kr[4], qr[4];
    float dec, bet, vt;
    auto load_row = [&](Raw<T> (&x)[4], uint32_t off, int t) __attribute__((always_inline)) {
#pragma unroll
      for (int b = 0; b < 4; ++b) gc_load<T>(x[b], mr, (t * ms + off + 32 * b + 4 * g) * ES);
    };
    auto load_rest = [&](int t) __attribute__((always_inline)) {
      dec = gc_load_f32(gr, (uint32_t)(t * p.gs + h) * 4);
      bet = gc_load_f32(br, (uint32_t)(t * p.gs + h) * 4);
      vt = (float)load_t(mr, (t * ms + v_off) * ES);
    };
    f32x4 x[8];   // 32 of a row's 128 values, times 1 / sqrt(|row|^2 + 1e-6)
    auto normed = [&](const Raw<T> (&r)[4]) __attribute__((always_inline)) {
      float ss = 0.f;
#pragma unroll
      for (int b = 0; b < 4; ++b) ss += r[b].squares();
      const float inv = 1.0f / sqrtf(rows4_sum(ss) + 1e-6f);
#pragma unroll
      for (int b = 0; b < 4; ++b)
#pragma unroll
        for (int e = 0; e < 8; ++e) x[2 * b + (e >> 2)][e & 3] = (float)r[b].v[e] * inv;
    };
    auto dot_s = [&]() __attribute__((always_inline)) {
      float s[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int b = 0; b < 8; ++b)
#pragma unroll
        for (int r = 0; r < 4; ++r) s[r] = __builtin_fmaf(S[b][r], x[b][r], s[r]);
      return rows4_sum((s[0] + s[1]) + (s[2] + s[3]));
    };
    load_row(kr, k_off, 0);
    load_row(qr, q_off, 0);
    load_rest(0);
#pragma nounroll
    for (int t = 0; t < rows; ++t) {
      normed(kr);
      load_row(kr, k_off, t + 1);
      const float d = expf(dec);
#pragma unroll
      for (int b = 0; b < 8; ++b) S[b] *= d;
      const float u = (vt - dot_s()) * bet;
      load_rest(t + 1);
#pragma unroll
      for (int b = 0; b < 8; ++b)
#pragma unroll
        for (int r = 0; r < 4; ++r) S[b][r] = __builtin_fmaf(x[b][r], u, S[b][r]);
      normed(qr);
      load_row(qr, q_off, t + 1);
      const float o = dot_s() * (1.0f / sqrtf((float)GC_D));
      if (g == 0)
        __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, o), orr,
                                              (t * os + (uint32_t)h * GC_D + 16 * wave + i16) * 4, 0, 0);
    }
  };
  int64_t by_token = end;   // the recurrence takes over at this token

  // The two waves of a SIMD leave each barrier together; with equal priority
  // both split (VALU), then both multiply. Favouring one lets it run ahead into
  // its MFMAs while the other splits.
  if (wave < GC_WAVES / 2) __builtin_amdgcn_s_setprio(2);
  fetch(begin);
  for (int64_t t0 = begin; t0 < end; t0 += C) {
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");   // the last chunk's readers are done
    {
      // an opaque copy of the lane: the addresses below are made here for each
      // chunk; kept over the loop they cost the registers that are not there
      int ln = lane;
      asm volatile("" : "+v"(ln));
      if constexpr (NP == 1) {
#pragma unroll
        for (int f = 0; f < FK; ++f) {
          const int t = 8 * wave + 4 * f + (ln >> 4), c = ln & 15;   // token, chunk of 8 dims
          const int step = c >> 2, hh = (c >> 1) & 1;
          const u32x4 kw = __builtin_bit_cast(u32x4, rk[f].v), qw = __builtin_bit_cast(u32x4, rq[f].v);
#pragma unroll
          for (int half = 0; half < 2; ++half) {   // dims 4 half .. of the chunk: lane group 2 (c % 2) + half
            const int at = ((t >> 4) * 4 + step) * 1024 + gc_slot(2 * (c & 1) + half, t & 15, x_k(step)) + 8 * hh;
            *reinterpret_cast<u32x2*>(smem + L::KF + at) = (u32x2){kw[2 * half], kw[2 * half + 1]};
            *reinterpret_cast<u32x2*>(smem + L::QF + at) = (u32x2){qw[2 * half], qw[2 * half + 1]};
          }
#pragma unroll
          for (int e = 0; e < 8; ++e) {   // K^T: token t is term 4 h + r of lane group (t % 16) / 4
            const int db = c >> 1, i = 8 * (c & 1) + e;
            *reinterpret_cast<bf16*>(smem + L::KT + (db * TS + (t >> 5)) * 1024 +
                                     gc_slot((t & 15) >> 2, i, x_t(db)) + (4 * ((t >> 4) & 1) + (t & 3)) * 2) = rk[f].v[e];
          }
        }
      } else {
#pragma unroll
        for (int f = 0; f < FK; ++f) {
          const int id = wave * FK + f;
          bf16x8 a[NP], q[NP];
          rk[f].parts(a);
          rq[f].parts(q);
#pragma unroll
          for (int n = 0; n < NP; ++n) {
            *frag(L::KF, id * NP + n, x_k(id & 3)) = a[n];
            *frag(L::QF, id * NP + n, x_k(id & 3)) = q[n];
          }
        }
#pragma unroll
        for (int f = 0; f < FT; ++f) {
          const int id = wave * FT + f;
          bf16x8 a[NP];
          rt[f].parts(a);
#pragma unroll
          for (int n = 0; n < NP; ++n) *frag(L::KT, id * NP + n, x_t(id / TS)) = a[n];
        }
      }
#pragma unroll
      for (int f = 0; f < RT; ++f) {
        const int t = 2 * (RT * wave + f) + (ln >> 5), c = ln & 15;   // row, chunk of 4 columns of T or P
        const int ts = c >> 3, hh = (c >> 2) & 1, grp = c & 3;
        if (TS == 1 && ts) continue;   // f32 chunks have 32 columns
        u32x2 o[3];
        bf16_parts4(rl[f], o);
        char* at = smem + ((ln & 16) ? L::PF : L::TF) + ((t >> 4) * TS + ts) * 3 * 1024 +
                   gc_slot(grp, t & 15, x_l(grp, ts)) + 8 * hh;
#pragma unroll
        for (int n = 0; n < 3; ++n) *reinterpret_cast<u32x2*>(at + n * 1024) = o[n];
      }
      if (wave == GC_WAVES - 1) {
        if (lane < C) {
#pragma unroll
          for (int n = 0; n < 3; ++n) vec[n * C + lane] = t0 + lane < end ? rs[n] : 0.f;
        }
        if (lane == 0) vec[3 * C] = rs[3];
      }
    }
    f32x4 v[RB], o[RB];
#pragma unroll
    for (int rb = 0; rb < RB; ++rb)
#pragma unroll
      for (int r = 0; r < 4; ++r) v[rb][r] = (float)rv[rb][r];
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    if (t0 + C < end) fetch(t0 + C);
    if (by_token < end) continue;

    const float eall = vec[3 * C];
    auto scale = [&](int which, int rb) __attribute__((always_inline)) {
      return *reinterpret_cast<const f32x4*>(vec + which * C + 16 * rb + 4 * g);
    };
    const f32x4 zero = {0.f, 0.f, 0.f, 0.f};

    {   // R = V - e^c K S, O = e^c Q S
      bf16x8 sp[4][3];
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        float x[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) x[e] = S[2 * s + (e >> 2)][e & 3];
        gc_split<3>(x, sp[s]);
      }
#pragma unroll
      for (int rb = 0; rb < RB; ++rb) {
        f32x4 kh_ = zero, kl = zero, qh = zero, ql = zero;
#pragma unroll
        for (int s = 0; s < 4; ++s) {
          bf16x8 a[NP], q[NP];
#pragma unroll
          for (int n = 0; n < NP; ++n) {
            a[n] = *frag(L::KF, (rb * 4 + s) * NP + n, x_k(s));
            q[n] = *frag(L::QF, (rb * 4 + s) * NP + n, x_k(s));
          }
          gc_mm<NP, 3>(a, sp[s], kh_, kl);
          gc_mm<NP, 3>(q, sp[s], qh, ql);
        }
        v[rb] -= scale(0, rb) * (kh_ + kl);
        o[rb] = scale(1, rb) * (qh + ql);
      }
    }
    bf16x8 up[TS][3];
    auto split_rows = [&](const f32x4 (&m)[RB]) __attribute__((always_inline)) {
#pragma unroll
      for (int ts = 0; ts < TS; ++ts) {
        float x[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) x[e] = m[2 * ts + (e >> 2)][e & 3];
        gc_split<3>(x, up[ts]);
      }
    };
    split_rows(v);   // R
    // U = T R and O += P U: block row rb of the lower triangles ends in step rb / 2
    auto lower = [&](int base, f32x4 (&m)[RB]) __attribute__((always_inline)) {
#pragma unroll
      for (int rb = 0; rb < RB; ++rb) {
        f32x4 lo = zero;
#pragma unroll
        for (int ts = 0; ts <= rb / 2; ++ts) {
          bf16x8 a[3];
#pragma unroll
          for (int n = 0; n < 3; ++n) a[n] = *frag(base, (rb * TS + ts) * 3 + n, x_l(g, ts));
          gc_mm<3, 3>(a, up[ts], m[rb], lo);
        }
        m[rb] += lo;
      }
    };
    f32x4 u[RB];
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) u[rb] = zero;
    lower(L::TF, u);
    split_rows(u);
    lower(L::PF, o);
    float nan = 0.f;   // unless a result is not finite
#pragma unroll
    for (int rb = 0; rb < RB; ++rb)
#pragma unroll
      for (int r = 0; r < 4; ++r) nan = __builtin_fmaf(o[rb][r], 0.f, nan);
    if (__any(nan != nan)) {
      by_token = t0;
      continue;
    }
    {
      const int rows = (int)min((int64_t)C, end - t0);
      const __amdgpu_buffer_rsrc_t orr = gc_rows_of(p.out, t0, p.os, rows, (int64_t)p.nv * GC_D, 4);
#pragma unroll
      for (int rb = 0; rb < RB; ++rb)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float x = o[rb][r];
          __builtin_amdgcn_raw_buffer_store_b32(
              __builtin_bit_cast(uint32_t, x), orr,
              ((16 * rb + 4 * g + r) * os + (uint32_t)h * GC_D + 16 * wave + i16) * 4, 0, 0);
        }
    }
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) u[rb] *= scale(2, rb);
    split_rows(u);
#pragma unroll
    for (int db = 0; db < 8; ++db) {
      f32x4 lo = zero;
      S[db] *= eall;
#pragma unroll
      for (int ts = 0; ts < TS; ++ts) {
        bf16x8 a[NP];
#pragma unroll
        for (int n = 0; n < NP; ++n) a[n] = *frag(L::KT, (db * TS + ts) * NP + n, x_t(db));
        gc_mm<NP, 3>(a, up[ts], S[db], lo);
      }
      S[db] += lo;
    }
  }
  for (int64_t t0 = by_token; t0 < end; t0 += C) walk(t0);
}

template <typename T>
int gdn_chunk_go(const GdnChunkParams& p, hipStream_t st) {
  constexpr int C = gc_len<T>();
  const int64_t slots = p.n / C + p.n_texts;
  if (slots > 0x7fffffff) return fail(INL_E_UNSUPPORTED, "gdn_rule: too many tokens");
  const int rc = set_max_dynamic_lds(reinterpret_cast<const void*>(&gdn_chunk_rule<T>), GcLds<T>::TOTAL);
  if (rc) return rc;
  hipLaunchKernelGGL(gdn_chunk_prep<T>, dim3((unsigned)slots, (unsigned)((p.nv + 3) / 4)), dim3(256), 0, st, p);
  INL_HIP_TRY(hipGetLastError());
  hipLaunchKernelGGL(gdn_chunk_rule<T>, dim3((unsigned)p.nv, (unsigned)p.n_texts), dim3(64 * GC_WAVES),
                     GcLds<T>::TOTAL, st, p);
  INL_HIP_TRY(hipGetLastError());
  return INL_OK;
}

}  // namespace

bool gdn_chunk_fits(const GdnChunkParams& p, int32_t dtype) {
  // both dims 128 (a row of `out` holds 2 x 64 values of T and P), rows that
  // take the vector loads
  const int64_t esize = dtype_size(dtype);
  return p.dk == GC_D && p.dv == GC_D && p.ms % 4 == 0 && ((uintptr_t)p.mixed % (4 * esize)) == 0 && p.os % 4 == 0 &&
         ((uintptr_t)p.out & 15) == 0 && p.ms <= (1 << 22) && p.os <= (1 << 22) && p.gs <= (1 << 22) &&   // a chunk's offsets fit 32 bits
         (p.nv + 3) / 4 <= 65535 &&
         // Short texts leave most of a chunk empty and still pay two launches:
         // one text of 32 tokens took 23 us here and 21 per token, one of 64
         // 25 and 39, 128 texts of 40 121 and 201. The lengths are on the
         // device, so the line is drawn at their mean.
         p.n >= 40 * (int64_t)p.n_texts;
}

int gdn_chunk_launch(const GdnChunkParams& p, int32_t dtype, hipStream_t st) {
  return dtype == INL_BF16 ? gdn_chunk_go<bf16>(p, st) : gdn_chunk_go<float>(p, st);
}

}  // namespace inl
