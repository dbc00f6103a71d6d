// An encoder layer on a few token rows (gfx950, MFMA): one search query or a
// handful of short texts. Five launches a layer:
//
//   q/k/v rows        = rms_norm(h) * gamma . Wqkv^T           skinny_kernel, NORM
//   attention         = q/k norm + RoPE + causal softmax . V   few_attn_kernel
//   h                += attention . Wo^T                       skinny_kernel, ADD
//   act               = silu(gate) * up of rms_norm(h) * gamma skinny_kernel, NORM, SWIGLU
//   h                += act . Wdown^T                          skinny_kernel, ADD
//
// What bounds it: at a few dozen rows the weights are read once and used once
// per row, so a projection's floor is its weight bytes over HBM (8.4 MB of
// q/k/v weights of the 0.6B shape: 1.7 us at 4.9 TB/s) plus the ~1.6 us of a
// launch; everything else is latency, and address processing in the vector
// memory path. A load of 16 bytes per lane runs at 64 bytes per clock when
// neighbouring lanes read neighbouring bytes and at 16 when they read 16
// different rows, which is what an MFMA operand wants (lane l: row l % 16).
// At 64 rows the strided x loads alone took 7.5 of the o projection's 12 us.
// Hence:
//  - the rows between these kernels are kept in operand order ("fragments",
//    below): a wave reads an operand as one contiguous KiB. h is kept both
//    ways, f32 in both; the fragments of one kernel's output are written by
//    its epilogue, 16 bytes per lane;
//  - weights go from memory to LDS (direct loads, contiguous) and from there
//    into operands, swizzled so that 16 rows of a read cover all banks;
//  - the 8 waves of a workgroup split k, not rows: each wave loads its own
//    slice of x and w, all of it before anything waits, and the waves meet
//    only to add 8 partial tiles;
//  - the row norm is computed from the wave's slices and one exchange of
//    partial sums while the weights are on their way: reading a few f32 rows
//    in every workgroup costs less than a launch of its own;
//  - the gate and up rows of the same outputs belong to one workgroup.
//
// Fragments of rows [m, k] of type T: step s covers 32 k, block b 16 rows;
// lane l of (s, b) holds row 16 b + l % 16 and, with g = l / 16,
//   bf16: k = 32 s + 8 g .. + 7       (one plane of 16 bytes per lane)
//   f32:  k = 32 s + 16 h + 4 g .. + 3, plane h = 0, 1
// and the f32 h rows behind bf16 operands: k = 32 s + 8 g + 4 h .. + 3, plane h.
// Plane p of (s, b) is the KiB at ((s * blocks + b) * planes + p) * 1024.
// Rows past m in the last block hold anything: a row of x only reaches its own
// column of the product, which is not stored.
#include "skinny.hpp"
#include "lanes.hpp"

namespace inl {

namespace {

constexpr int SK_WAVES = 8;
constexpr int SK_STEP = 32;   // k per step: one MFMA in bf16, eight in f32

struct SkinnyParams {
  const char* xf;       // fragments of T, or of the f32 h (NORM)
  const char* w;        // T [n (or 2n), k]
  const char* gamma;    // T [k] (NORM)
  char* y;              // STORE: T rows of ys elements; ADD: f32 rows; SWIGLU: unused
  char* yf;             // ADD: fragments of h; SWIGLU: fragments of T
  int64_t ys;
  int32_t m, n, k;
  int32_t blocks;       // blocks of 16 rows
  float eps;
  SkinnyNext next;
};

// Workgroups past a kernel's own read the next projection's weights into the
// L2 of the XCD that will run them (workgroup b runs on XCD b % 8) and drop
// them. A kernel of this chain leaves CUs idle (the o and down projections
// use 64 workgroups, the attention of one text 8) and the memory bus idle
// while it waits for its first loads, adds up partials and drains; the next
// kernel then starts on weights that are already on the chip.
constexpr int XCDS = 8;

__device__ __forceinline__ void prefetch_next(const SkinnyNext& q, int first, int wgs) {
  // workgroup id `first` .. of the grid's `wgs`: the ones of this XCD take its consumers in turn
  const int id = blockIdx.x, xcd = id % XCDS;
  const int f0 = first + (xcd - first % XCDS + XCDS) % XCDS;   // this XCD's first prefetcher
  const int step = (wgs - f0 + XCDS - 1) / XCDS, mine = (id - f0) / XCDS;
  const int threads = blockDim.x;
  const int64_t piece = (int64_t)threads * 64;   // 4 loads per lane
  const int per = (int)((q.bytes + piece - 1) / piece) * (q.second ? 2 : 1);   // pieces per consumer
  const int consumers = (q.consumers - xcd + XCDS - 1) / XCDS;
  for (int j = mine; j < consumers * per; j += step) {
    const int b = xcd + XCDS * (j / per), r = j % per;
    const int half = q.second ? r & 1 : 0, at = q.second ? r >> 1 : r;
    const char* src = q.w + (half ? q.second : 0) + (int64_t)b * q.bytes + at * piece;
    const int64_t left = q.bytes - at * piece;
    u32x4 v[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int64_t off = ((int64_t)i * threads + threadIdx.x) * 16;
      v[i] = *reinterpret_cast<const u32x4*>(src + (off < left ? off : 0));
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) asm volatile("" ::"v"(v[i]));
  }
}

template <typename T>
struct Frag;   // a lane's 8 k values of one step
template <>
struct Frag<bf16> {
  u32x4 v;
};
template <>
struct Frag<float> {
  f32x4 v[2];
};

// acc += a . b over one step of 32 k (a: 16 weight rows, b: 16 token rows).
// f32: v_mfma_f32_16x16x4_f32 takes one k per lane group; element e of a
// plane pairs the same k of a and b.
__device__ __forceinline__ f32x4 mfma_step(const Frag<bf16>& a, const Frag<bf16>& b, f32x4 acc) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a.v), __builtin_bit_cast(bf16x8, b.v),
                                                 acc, 0, 0, 0);
}
__device__ __forceinline__ f32x4 mfma_step(const Frag<float>& a, const Frag<float>& b, f32x4 acc) {
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int e = 0; e < 4; ++e) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a.v[h][e], b.v[h][e], acc, 0, 0, 0);
  return acc;
}

template <typename T>
constexpr int planes() { return sizeof(T) == 2 ? 1 : 2; }

// Byte offset, in fragments with h planes of f32 for T operands, of the 16
// bytes that hold columns c .. c + 3 (c % 4 == 0) of a row.
template <typename T>
__device__ __forceinline__ int64_t hfrag_off(int row, int c, int blocks) {
  const int s = c >> 5, i = c & 31;
  const int g = sizeof(T) == 2 ? i >> 3 : (i & 15) >> 2;
  const int h = sizeof(T) == 2 ? (i >> 2) & 1 : i >> 4;
  return (((int64_t)s * blocks + (row >> 4)) * 2 + h) * 1024 + (g * 16 + (row & 15)) * 16;
}
// The same in fragments of T (4 values: 8 bytes of bf16, 16 of f32).
template <typename T>
__device__ __forceinline__ int64_t xfrag_off(int row, int c, int blocks) {
  if constexpr (sizeof(T) == 4) {
    return hfrag_off<float>(row, c, blocks);
  } else {
    const int s = c >> 5, i = c & 31;
    return ((int64_t)s * blocks + (row >> 4)) * 1024 + ((i >> 3) * 16 + (row & 15)) * 16 + (i & 7) * 2;
  }
}
template <typename T>
__device__ __forceinline__ void store4(char* p, const f32x4& v) {
  if constexpr (sizeof(T) == 2) {
    bf16x4 r;
#pragma unroll
    for (int e = 0; e < 4; ++e) r[e] = (bf16)v[e];
    *reinterpret_cast<bf16x4*>(p) = r;
  } else {
    *reinterpret_cast<f32x4*>(p) = v;
  }
}

// Maximum over the four lanes that share lane & 15, in all of them.
__device__ __forceinline__ float rows4_max(float x) {
  float a = x, b = x;
  asm volatile("s_nop 1\n\tv_permlane16_swap_b32 %0, %1" : "+v"(a), "+v"(b));
  a = b = fmaxf(a, b);
  asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %1" : "+v"(a), "+v"(b));
  return fmaxf(a, b);
}

// The f32 row values behind one Frag<T> of normalised x, in the same k order.
template <typename T>
struct HFrag {
  f32x4 v[2];
  __device__ __forceinline__ float squares() const {
    float s = 0.f;
#pragma unroll
    for (int h = 0; h < 2; ++h)
      s += (v[h][0] * v[h][0] + v[h][1] * v[h][1]) + (v[h][2] * v[h][2] + v[h][3] * v[h][3]);
    return s;
  }
  // (v * inv * gamma) rounded to T, the row norm's own order of products
  __device__ __forceinline__ Frag<T> normed(float inv, const Frag<T>& g) const {
    Frag<T> o;
    if constexpr (sizeof(T) == 2) {
      bf16x8 r;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const uint32_t gw = g.v[j];
        r[2 * j] = (bf16)(v[j >> 1][2 * (j & 1)] * inv * __builtin_bit_cast(float, gw << 16));
        r[2 * j + 1] = (bf16)(v[j >> 1][2 * (j & 1) + 1] * inv * __builtin_bit_cast(float, gw & 0xffff0000u));
      }
      o.v = __builtin_bit_cast(u32x4, r);
    } else {
#pragma unroll
      for (int h = 0; h < 2; ++h) o.v[h] = v[h] * inv * g.v[h];
    }
    return o;
  }
};

typedef __attribute__((address_space(1))) const void* gptr_t;
typedef __attribute__((address_space(3))) void* lptr_t;

// Weight panels in LDS: 16 rows x 128 bytes; 16-byte chunk c of row r sits at
// r * 128 + ((c ^ ((r >> 1) & 7)) << 4), so the 16 rows of one ds_read_b128
// pass cover all 64 banks. The direct load writes LDS in lane order, so the
// swizzle is in which chunk a lane fetches.
__device__ __forceinline__ void load_panel(const char* w, int64_t row_bytes, char* lds, int lane) {
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int r = 8 * i + (lane >> 3);
    const char* src = w + r * row_bytes + (((lane & 7) ^ ((r >> 1) & 7)) << 4);
    __builtin_amdgcn_global_load_lds((gptr_t)src, (lptr_t)(lds + i * 1024), 16, 0, 0);
  }
}
__device__ __forceinline__ u32x4 panel_chunk(const char* lds, int r, int c) {
  return *reinterpret_cast<const u32x4*>(lds + r * 128 + ((c ^ ((r >> 1) & 7)) << 4));
}

// The wave's direct loads have written their panels (the compiler does not
// order LDS reads behind them).
__device__ __forceinline__ void panels_landed() {
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
}

// This lane's weight operand of step s of a wave's slice (panels of 64 k in
// bf16, 32 in f32).
template <typename T>
__device__ __forceinline__ Frag<T> w_frag(const char* lds, int s, int lane) {
  const int r = lane & 15, g = lane >> 4;
  Frag<T> f;
  if constexpr (sizeof(T) == 2) {
    f.v = panel_chunk(lds + (s >> 1) * 2048, r, 4 * (s & 1) + g);
  } else {
    f.v[0] = __builtin_bit_cast(f32x4, panel_chunk(lds + s * 2048, r, g));
    f.v[1] = __builtin_bit_cast(f32x4, panel_chunk(lds + s * 2048, r, 4 + g));
  }
  return f;
}

// MB: blocks of 16 token rows a workgroup owns; EPI: what becomes of the
// product; NS: steps of one pass over a wave's slice (with NORM the only one):
// all of a pass's loads are issued before its first wait.
template <typename T, int MB, bool NORM, int EPI, int NS>
__global__ __launch_bounds__(64 * SK_WAVES) void skinny_kernel(SkinnyParams p) {
  constexpr int CB = EPI == SKINNY_SWIGLU ? 2 : 1;             // blocks of 16 weight rows
  constexpr int PANELS = NS * SK_STEP * (int)sizeof(T) / 128;  // per block of weight rows and pass
  // A wave's weight panels, and afterwards its partial tiles.
  constexpr int OWN = CB * (PANELS * 2048 > MB * 1024 ? PANELS * 2048 : MB * 1024);
  __shared__ __attribute__((aligned(1024))) char own[SK_WAVES][OWN];
  __shared__ float ssum[SK_WAVES][MB * 16];
  if ((int)blockIdx.x >= p.n / 16) {
    prefetch_next(p.next, p.n / 16, gridDim.x);   // (only launched beside one row of workgroups)
    return;
  }
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n0 = blockIdx.x * 16, b0 = blockIdx.y * MB;
  const int kw = p.k / SK_WAVES, k0 = wave * kw, steps = kw / SK_STEP;
  const int64_t row_bytes = (int64_t)p.k * (int)sizeof(T);
  const char* wrow = p.w + n0 * row_bytes + (int64_t)k0 * (int)sizeof(T);
  const int nb = min(MB, p.blocks - b0);   // uniform
  // fragment (step s of this wave, block b, plane h) of x
  constexpr int XP = NORM ? 2 : planes<T>();
  auto xptr = [&](int s, int b, int h) __attribute__((always_inline)) {
    const int bc = b0 + (b < nb ? b : nb - 1);   // blocks past the last repeat it
    return p.xf + (((int64_t)(k0 / SK_STEP + s) * p.blocks + bc) * XP + h) * 1024 + lane * 16;
  };
  // the output this lane finishes: 4 neighbouring columns of one token row
  const int fb = wave, frow = 16 * (b0 + fb) + (lane & 15), fcol = n0 + (lane >> 4) * 4;
  const bool fin = fb < MB && frow < p.m;
  f32x4 before = {0.f, 0.f, 0.f, 0.f};
  if (EPI == SKINNY_ADD_F32 && fin)
    before = *reinterpret_cast<const f32x4*>(p.y + ((int64_t)frow * p.ys + fcol) * 4);
  f32x4 acc[CB][MB];
#pragma unroll
  for (int c = 0; c < CB; ++c)
#pragma unroll
    for (int b = 0; b < MB; ++b) acc[c][b] = (f32x4){0.f, 0.f, 0.f, 0.f};
  auto load_w = [&](int s0) __attribute__((always_inline)) {
#pragma unroll
    for (int c = 0; c < CB; ++c)
#pragma unroll
      for (int i = 0; i < PANELS; ++i)
        load_panel(wrow + (int64_t)c * p.n * row_bytes + s0 * SK_STEP * (int)sizeof(T) + i * 128, row_bytes,
                   own[wave] + (c * PANELS + i) * 2048, lane);
  };

  if constexpr (NORM) {
    // The rows come from the L2, the weights from HBM: rows first, so that the
    // norm runs while the weights are on their way.
    HFrag<T> hf[MB][NS];
    Frag<T> gf[NS];
#pragma unroll
    for (int b = 0; b < MB; ++b)
#pragma unroll
      for (int s = 0; s < NS; ++s)
#pragma unroll
        for (int h = 0; h < 2; ++h) hf[b][s].v[h] = *reinterpret_cast<const f32x4*>(xptr(s, b, h));
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      const char* gp = p.gamma + (int64_t)(k0 + s * SK_STEP) * (int)sizeof(T) + (lane >> 4) * 16;
      if constexpr (sizeof(T) == 2) {
        gf[s].v = *reinterpret_cast<const u32x4*>(gp);
      } else {
        gf[s].v[0] = *reinterpret_cast<const f32x4*>(gp);
        gf[s].v[1] = *reinterpret_cast<const f32x4*>(gp + 64);
      }
    }
    load_w(0);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int b = 0; b < MB; ++b) {
      float ss = 0.f;
#pragma unroll
      for (int s = 0; s < NS; ++s) ss += hf[b][s].squares();
      ss = rows4_sum(ss);
      if (lane < 16) ssum[wave][16 * b + lane] = ss;
    }
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");   // not the weights in flight
    Frag<T> xf[MB][NS];
#pragma unroll
    for (int b = 0; b < MB; ++b) {
      float t = 0.f;
#pragma unroll
      for (int v = 0; v < SK_WAVES; ++v) t += ssum[v][16 * b + (lane & 15)];
      const float inv = 1.0f / sqrtf(t / (float)p.k + p.eps);
#pragma unroll
      for (int s = 0; s < NS; ++s) xf[b][s] = hf[b][s].normed(inv, gf[s]);
    }
    panels_landed();
#pragma unroll
    for (int s = 0; s < NS; ++s)
#pragma unroll
      for (int c = 0; c < CB; ++c) {
        const Frag<T> wf = w_frag<T>(own[wave] + c * PANELS * 2048, s, lane);
#pragma unroll
        for (int b = 0; b < MB; ++b) acc[c][b] = mfma_step(wf, xf[b][s], acc[c][b]);
      }
  } else {
    for (int s0 = 0; s0 < steps; s0 += NS) {
      if (s0) asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // the last pass's panel reads are done
      load_w(s0);
      Frag<T> xf[MB][NS];
#pragma unroll
      for (int s = 0; s < NS; ++s)
#pragma unroll
        for (int b = 0; b < MB; ++b)
          if constexpr (sizeof(T) == 2) {
            xf[b][s].v = *reinterpret_cast<const u32x4*>(xptr(s0 + s, b, 0));
          } else {
            xf[b][s].v[0] = *reinterpret_cast<const f32x4*>(xptr(s0 + s, b, 0));
            xf[b][s].v[1] = *reinterpret_cast<const f32x4*>(xptr(s0 + s, b, 1));
          }
      panels_landed();
#pragma unroll
      for (int s = 0; s < NS; ++s) {
        const Frag<T> wf = w_frag<T>(own[wave], s, lane);
#pragma unroll
        for (int b = 0; b < MB; ++b) acc[0][b] = mfma_step(wf, xf[b][s], acc[0][b]);
      }
    }
  }

#pragma unroll
  for (int c = 0; c < CB; ++c)
#pragma unroll
    for (int b = 0; b < MB; ++b)
      *reinterpret_cast<f32x4*>(own[wave] + ((c * MB + b) * 64 + lane) * 16) = acc[c][b];
  __syncthreads();
  // The wave partials are added in wave order: the result does not depend on
  // timing.
  if (!fin) return;
  f32x4 sum[CB];
#pragma unroll
  for (int c = 0; c < CB; ++c) {
    const int off = ((c * MB + fb) * 64 + lane) * 16;
    sum[c] = *reinterpret_cast<const f32x4*>(own[0] + off);
#pragma unroll
    for (int w = 1; w < SK_WAVES; ++w) sum[c] += *reinterpret_cast<const f32x4*>(own[w] + off);
  }
  if constexpr (EPI == SKINNY_ADD_F32) {
    const f32x4 h = before + sum[0];
    *reinterpret_cast<f32x4*>(p.y + ((int64_t)frow * p.ys + fcol) * 4) = h;
    *reinterpret_cast<f32x4*>(p.yf + hfrag_off<T>(frow, fcol, p.blocks)) = h;
  } else if constexpr (EPI == SKINNY_SWIGLU) {
    f32x4 o;
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e] = sum[0][e] / (1.0f + expf(-sum[0][e])) * sum[CB - 1][e];
    store4<T>(p.yf + xfrag_off<T>(frow, fcol, p.blocks), o);
  } else {
    store4<T>(p.y + ((int64_t)frow * p.ys + fcol) * (int)sizeof(T), sum[0]);
  }
}

// Prefetching workgroups beside `own` working ones: the CUs left over.
int prefetchers(const SkinnyNext& q, int own) { return q.w && own < q.cus ? q.cus - own : 0; }

// ---- embedding: h[t, :] = f32(table[ids[t], :]), as rows and as fragments ----
// One workgroup per token row; an id outside [0, vocab) gives a NaN row.
template <typename T>
__global__ __launch_bounds__(256) void few_embed_kernel(const int32_t* ids, const char* table, int64_t vocab,
                                                        int32_t hidden, int32_t blocks, float* h, char* hf) {
  const int t = blockIdx.x;
  const int32_t id = ids[t];
  const bool ok = id >= 0 && id < vocab;
  const T* row = reinterpret_cast<const T*>(table) + (int64_t)(ok ? id : 0) * hidden;
  for (int c = threadIdx.x * 4; c < hidden; c += 1024) {
    f32x4 v;
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = ok ? (float)row[c + e] : __builtin_nanf("");
    *reinterpret_cast<f32x4*>(h + (int64_t)t * hidden + c) = v;
    *reinterpret_cast<f32x4*>(hf + hfrag_off<T>(t, c, blocks)) = v;
  }
}

// ---- attention of short texts, with the q/k norms and RoPE ----
// One workgroup of 4 or 8 waves per (text, K/V head); head_dim 128, at most 8
// blocks of 16 keys. Nothing here is large enough to be bound by
// anything but latency, so the whole prologue is folded in: what a launch of
// its own costs (4.5-5 us) is more than all of its work.
//  1. K: a wave takes one key block, as MFMA operands (a lane holds 8
//     consecutive dims per step of 32, and the RoPE partner, 64 dims away, is
//     its own operand two steps on), norms, rotates, rounds as the prologue
//     kernel does and leaves them in LDS in operand order.
//  2. A wave takes 16-query blocks NW apart: Q the same way, S^T = K Q^T, the
//     causal softmax of a column over registers and one exchange between the
//     four lanes of a query; P (f16, or f32) goes to LDS in operand order.
//  3. A wave takes its share of the 128 dims: O^T = V^T P^T for every query block,
//     its V^T operands loaded from global memory at the kernel's start. Keys
//     pair up in the order the P registers hold: step s, e = 4 h + r is key
//     32 s + 16 h + 4 g + r.
// O leaves in fragment order, the o projection's operand.
constexpr int FEW_D = 128;
constexpr int FEW_LDS_MAX = 160 * 1024;

struct FewAttnParams {
  const char* qkv;      // T rows [m, qs]: q heads, k heads, v heads
  const char* qw;       // T [128] q and k norm weights
  const char* kw;
  const float* cos;     // [positions, 64]
  const float* sin;
  const int32_t* cu;    // device offsets
  char* of;             // fragments of T [m, heads * 128]
  int64_t qs;
  int32_t n_texts, heads, kv_heads, blocks;
  float eps, scale_log2;
  SkinnyNext next;
};

__device__ __forceinline__ float few_round(float v, bf16) { return (float)(bf16)v; }
__device__ __forceinline__ float few_round(float v, float) { return v; }

// 8 dims per step of one head row in operand order, as f32.
template <typename T>
__device__ __forceinline__ void few_load(const char* row, int g, float (&v)[4][8]) {
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    if constexpr (sizeof(T) == 2) {
      const u32x4 w = *reinterpret_cast<const u32x4*>(row + (s * 32 + g * 8) * 2);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const uint32_t u = w[j];
        v[s][2 * j] = __builtin_bit_cast(float, u << 16);
        v[s][2 * j + 1] = __builtin_bit_cast(float, u & 0xffff0000u);
      }
    } else {
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const f32x4 w = *reinterpret_cast<const f32x4*>(row + (s * 32 + h * 16 + g * 4) * 4);
#pragma unroll
        for (int e = 0; e < 4; ++e) v[s][4 * h + e] = w[e];
      }
    }
  }
}

// The cos and sin columns of position `pos` that this lane rotates with, in
// operand order (steps 0 and 1; steps 2 and 3 are their partners).
struct FewTable {
  f32x4 c[2][2], s[2][2];
  template <typename T>
  __device__ __forceinline__ void load(const FewAttnParams& p, int pos, int g) {
#pragma unroll
    for (int st = 0; st < 2; ++st)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int col = st * 32 + (sizeof(T) == 2 ? g * 8 + h * 4 : h * 16 + g * 4);
        c[st][h] = *reinterpret_cast<const f32x4*>(p.cos + (int64_t)pos * 64 + col);
        s[st][h] = *reinterpret_cast<const f32x4*>(p.sin + (int64_t)pos * 64 + col);
      }
  }
};

// RMSNorm, weight, rounding and half-split RoPE of one row (the prologue's
// own order of operations).
template <typename T>
__device__ __forceinline__ void few_norm_rope(float (&v)[4][8], const float (&w)[4][8], const FewTable& tab, float eps) {
  float ss = 0.f;
#pragma unroll
  for (int s = 0; s < 4; ++s)
#pragma unroll
    for (int e = 0; e < 8; ++e) ss += v[s][e] * v[s][e];
  const float inv = 1.0f / sqrtf(rows4_sum(ss) / (float)FEW_D + eps);
#pragma unroll
  for (int s = 0; s < 4; ++s)
#pragma unroll
    for (int e = 0; e < 8; ++e) v[s][e] = few_round(v[s][e] * inv * w[s][e], T{});
#pragma unroll
  for (int s = 0; s < 2; ++s)
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float a = v[s][e], b = v[s + 2][e];
      const float c = few_round(tab.c[s][e >> 2][e & 3], T{}), sn = few_round(tab.s[s][e >> 2][e & 3], T{});
      v[s][e] = a * c - b * sn;
      v[s + 2][e] = b * c + a * sn;
    }
}

template <typename T>
__device__ __forceinline__ Frag<T> few_pack(const float (&v)[8]) {
  Frag<T> f;
  if constexpr (sizeof(T) == 2) {
    bf16x8 r;
#pragma unroll
    for (int e = 0; e < 8; ++e) r[e] = (bf16)v[e];
    f.v = __builtin_bit_cast(u32x4, r);
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e) { f.v[0][e] = v[e]; f.v[1][e] = v[4 + e]; }
  }
  return f;
}
// Fragment i of an LDS array of them: planes of 16 bytes per lane.
template <typename T>
__device__ __forceinline__ void lds_put(char* base, int i, int lane, const Frag<T>& f) {
  char* q = base + (i * planes<T>() * 64 + lane) * 16;
  if constexpr (sizeof(T) == 2) {
    *reinterpret_cast<u32x4*>(q) = f.v;
  } else {
    *reinterpret_cast<f32x4*>(q) = f.v[0];
    *reinterpret_cast<f32x4*>(q + 1024) = f.v[1];
  }
}
template <typename T>
__device__ __forceinline__ Frag<T> lds_get(const char* base, int i, int lane) {
  const char* q = base + (i * planes<T>() * 64 + lane) * 16;
  Frag<T> f;
  if constexpr (sizeof(T) == 2) {
    f.v = *reinterpret_cast<const u32x4*>(q);
  } else {
    f.v[0] = *reinterpret_cast<const f32x4*>(q);
    f.v[1] = *reinterpret_cast<const f32x4*>(q + 1024);
  }
  return f;
}
// acc += V^T . P^T over 32 keys
__device__ __forceinline__ f32x4 pv_step(const Frag<bf16>& a, const Frag<bf16>& b, f32x4 acc) {
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a.v), __builtin_bit_cast(f16x8, b.v), acc,
                                                0, 0, 0);
}
__device__ __forceinline__ f32x4 pv_step(const Frag<float>& a, const Frag<float>& b, f32x4 acc) {
  return mfma_step(a, b, acc);
}
template <typename T>
__device__ __forceinline__ Frag<T> pv_pack(const float (&v)[8]) {   // Frag<bf16> carries f16 bits here
  if constexpr (sizeof(T) == 2) {
    f16x8 r;
#pragma unroll
    for (int e = 0; e < 8; ++e) r[e] = (f16)v[e];
    Frag<bf16> f;
    f.v = __builtin_bit_cast(u32x4, r);
    return f;
  } else {
    return few_pack<float>(v);
  }
}

constexpr int few_waves(int kb) { return kb == 2 ? 4 : 8; }
// KB: blocks of 16 keys the registers and LDS hold (2, 4 or 8); NW: waves.
template <typename T, int KB>
__global__ __launch_bounds__(64 * few_waves(KB), 1) void few_attn_kernel(FewAttnParams p) {
  constexpr int NW = few_waves(KB);
  constexpr int DB = 8 / NW;                  // blocks of 16 dims a wave's PV covers
  constexpr int ES = (int)sizeof(T);
  constexpr int KS = KB / 2;                  // steps of 32 keys
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int i16 = lane & 15, g = lane >> 4;
  const int group = p.heads / p.kv_heads;
  if ((int)blockIdx.x >= p.n_texts * p.kv_heads) {
    prefetch_next(p.next, p.n_texts * p.kv_heads, gridDim.x);
    return;
  }
  const int text = blockIdx.x / p.kv_heads, kvh = blockIdx.x - text * p.kv_heads;
  const int r0 = p.cu[text], T_ = p.cu[text + 1] - r0;
  const int nkb = (T_ + 15) >> 4;             // <= KB (the launcher's choice)
  const int nqb = group * nkb;                // query blocks: (head of the group, block)
  char* kf = smem;                                              // [KB][4] fragments
  char* pf = smem + KB * 4 * planes<T>() * 1024;                // [group * KB][KS] fragments
  float* li = reinterpret_cast<float*>(pf + (size_t)group * KB * KS * planes<T>() * 1024);   // [group * KB][16]
  const char* base = p.qkv + (int64_t)r0 * p.qs * ES;

  // Every load a wave's first blocks need goes out here, before anything
  // waits: its key block, its first query block, their tables, its V^T.
  const int t_k = min(16 * wave + i16, T_ - 1);
  const int hq0 = wave / nkb, t_q = min(16 * (wave - hq0 * nkb) + i16, T_ - 1);
  float w[4][8], qw[4][8], k0[4][8], q0[4][8];
  FewTable ktab, qtab;
  const char* krow = base + (int64_t)(p.heads + kvh) * FEW_D * ES;
  few_load<T>(krow + (int64_t)t_k * p.qs * ES, g, k0);
  few_load<T>(p.kw, g, w);
  ktab.load<T>(p, t_k, g);
  few_load<T>(base + (int64_t)t_q * p.qs * ES + (int64_t)(kvh * group + min(hq0, group - 1)) * FEW_D * ES, g, q0);
  few_load<T>(p.qw, g, qw);
  qtab.load<T>(p, t_q, g);
  // V^T operands of dims 16 DB w .. of this wave, for step 3
  float vv[DB][KS][8];
  {
    const char* vp = base + ((int64_t)(p.heads + p.kv_heads + kvh) * FEW_D + wave * 16 * DB + i16) * ES;
#pragma unroll
    for (int d = 0; d < DB; ++d)
#pragma unroll
      for (int s = 0; s < KS; ++s)
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const int key = 32 * s + 16 * (e >> 2) + 4 * g + (e & 3);   // keys past the end: P is 0 there
          vv[d][s][e] = (float)*reinterpret_cast<const T*>(vp + (int64_t)min(key, T_ - 1) * p.qs * ES + d * 16 * ES);
        }
  }
  __builtin_amdgcn_sched_barrier(0);
  if (wave < nkb) {   // KB <= NW: one key block a wave
    few_norm_rope<T>(k0, w, ktab, p.eps);
#pragma unroll
    for (int s = 0; s < 4; ++s) lds_put<T>(kf, wave * 4 + s, lane, few_pack<T>(k0[s]));
  }
  few_norm_rope<T>(q0, qw, qtab, p.eps);
  __syncthreads();
  for (int qb = wave; qb < nqb; qb += NW) {
    const int hh = qb / nkb, tb = qb - hh * nkb;
    const int t = 16 * tb + i16, tc = min(t, T_ - 1);
    if (qb != wave) {
      few_load<T>(base + (int64_t)tc * p.qs * ES + (int64_t)(kvh * group + hh) * FEW_D * ES, g, q0);
      qtab.load<T>(p, tc, g);
      few_norm_rope<T>(q0, qw, qtab, p.eps);
    }
    Frag<T> qf[4];
#pragma unroll
    for (int s = 0; s < 4; ++s) qf[s] = few_pack<T>(q0[s]);
    f32x4 st[KB];   // S^T: keys 16 kb + 4 g + r of query t
    float mx = -__builtin_inff();
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) {
      st[kb] = (f32x4){0.f, 0.f, 0.f, 0.f};
      if (kb <= tb) {   // uniform
#pragma unroll
        for (int s = 0; s < 4; ++s) st[kb] = mfma_step(lds_get<T>(kf, kb * 4 + s, lane), qf[s], st[kb]);
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const bool see = kb <= tb && 16 * kb + 4 * g + r <= tc;
        st[kb][r] = see ? st[kb][r] * p.scale_log2 : -__builtin_inff();
        mx = fmaxf(mx, st[kb][r]);
      }
    }
    mx = rows4_max(mx);   // finite: a query sees itself
    float l = 0.f;
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      float pv[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float x = exp2f(st[2 * s + (e >> 2)][e & 3] - mx);
        pv[e] = sizeof(T) == 2 ? (float)(f16)x : x;   // the sum takes the weights as PV takes them
        l += pv[e];
      }
      lds_put<T>(pf, qb * KS + s, lane, pv_pack<T>(pv));
    }
    l = rows4_sum(l);
    if (g == 0) li[qb * 16 + i16] = l;
  }
  __syncthreads();
  Frag<T> vf[DB][KS];
#pragma unroll
  for (int d = 0; d < DB; ++d)
#pragma unroll
    for (int s = 0; s < KS; ++s) vf[d][s] = pv_pack<T>(vv[d][s]);
  for (int qb = 0; qb < nqb; ++qb) {
    const int hh = qb / nkb, tb = qb - hh * nkb;
    f32x4 o[DB];
#pragma unroll
    for (int d = 0; d < DB; ++d) o[d] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < KS; ++s)
      if (2 * s <= tb) {   // uniform: later steps hold no key a query of this block sees
        const Frag<T> f = lds_get<T>(pf, qb * KS + s, lane);
#pragma unroll
        for (int d = 0; d < DB; ++d) o[d] = pv_step(vf[d][s], f, o[d]);
      }
    const float inv = 1.0f / li[qb * 16 + i16];
    const int t = 16 * tb + i16;
    if (t >= T_) continue;
#pragma unroll
    for (int d = 0; d < DB; ++d) {
      const int col = (kvh * group + hh) * FEW_D + (wave * DB + d) * 16 + g * 4;
      store4<T>(p.of + xfrag_off<T>(r0 + t, col, p.blocks), o[d] * inv);
    }
  }
}

template <typename T, int KB>
int few_lds(int group) {
  return KB * 4 * planes<T>() * 1024 + group * KB * (KB / 2) * planes<T>() * 1024 + group * KB * 64;
}

template <typename T, int KB>
int few_attn_go(const FewAttnParams& p, hipStream_t st) {
  const int lds = few_lds<T, KB>(p.heads / p.kv_heads);
  if (lds > 64 * 1024) {
    const int rc = set_max_dynamic_lds(reinterpret_cast<const void*>(&few_attn_kernel<T, KB>), FEW_LDS_MAX);
    if (rc) return rc;
  }
  const int own = p.n_texts * p.kv_heads;
  hipLaunchKernelGGL((few_attn_kernel<T, KB>), dim3(own + prefetchers(p.next, own)), dim3(64 * few_waves(KB)), lds, st, p);
  INL_HIP_TRY(hipGetLastError());
  return INL_OK;
}

template <typename T>
int few_attn_by_len(const FewAttnParams& p, int longest, hipStream_t st) {
  if (longest <= 32) return few_attn_go<T, 2>(p, st);
  if constexpr (sizeof(T) == 2)
    if (longest > 64) return few_attn_go<T, 8>(p, st);
  return few_attn_go<T, 4>(p, st);
}

template <typename T, int MB, bool NORM, int EPI, int NS>
void go(const SkinnyParams& p, hipStream_t st) {
  const dim3 grid(p.n / 16 + prefetchers(p.next, p.n / 16), (p.blocks + MB - 1) / MB);
  hipLaunchKernelGGL((skinny_kernel<T, MB, NORM, EPI, NS>), grid, dim3(64 * SK_WAVES), 0, st, p);
}

template <typename T, bool NORM, int EPI, int NS>
void by_rows(const SkinnyParams& p, hipStream_t st) {
  if (p.blocks == 1) go<T, 1, NORM, EPI, NS>(p, st);
  else if (p.blocks == 2 || sizeof(T) == 4) go<T, 2, NORM, EPI, NS>(p, st);
  else if constexpr (sizeof(T) == 2) go<T, 4, NORM, EPI, NS>(p, st);
}

template <typename T, bool NORM, int EPI>
void by_steps(const SkinnyParams& p, hipStream_t st) {
  const int steps = p.k / (SK_WAVES * SK_STEP);
  if constexpr (NORM) {
    if (steps == 4) by_rows<T, NORM, EPI, 4>(p, st);
    else by_rows<T, NORM, EPI, 2>(p, st);
  } else {
    if (steps % 12 == 0 && sizeof(T) == 2) by_rows<T, NORM, EPI, sizeof(T) == 2 ? 12 : 4>(p, st);
    else if (steps % 8 == 0 && sizeof(T) == 2) by_rows<T, NORM, EPI, sizeof(T) == 2 ? 8 : 4>(p, st);
    else by_rows<T, NORM, EPI, 4>(p, st);
  }
}

template <typename T>
void by_kind(const SkinnyParams& p, bool norm, int epi, hipStream_t st) {
  if (norm && epi == SKINNY_STORE) by_steps<T, true, SKINNY_STORE>(p, st);
  else if (norm) by_steps<T, true, SKINNY_SWIGLU>(p, st);
  else by_steps<T, false, SKINNY_ADD_F32>(p, st);
}

}  // namespace

bool few_prefetch(int32_t dtype, int64_t n) { return n <= (dtype == INL_BF16 ? 64 : 32); }

bool few_fits(int32_t dtype, int64_t n, int32_t longest, int32_t hidden, int32_t heads, int32_t kv_heads,
              int32_t head_dim, int32_t intermediate) {
  constexpr int KQ = SK_WAVES * SK_STEP;   // 256: every wave a whole number of steps
  if (n > (dtype == INL_BF16 ? FEW_ROWS_BF16 : FEW_ROWS_F32) || longest > 128 || head_dim != FEW_D) return false;
  // hidden: a wave's slice of the h rows is held in registers across the
  // norm's exchange, 2 or 4 steps of it; the others walk their slice by 4 steps
  if ((hidden != 2 * KQ && hidden != 4 * KQ) || (heads * FEW_D) % (4 * KQ) || intermediate % (4 * KQ)) return false;
  const int group = heads / kv_heads;
  const int lds = dtype == INL_BF16
                      ? (longest <= 32 ? few_lds<bf16, 2>(group) : longest <= 64 ? few_lds<bf16, 4>(group) : few_lds<bf16, 8>(group))
                      : (longest <= 32 ? few_lds<float, 2>(group) : few_lds<float, 4>(group));
  return lds <= FEW_LDS_MAX;
}

size_t few_h_bytes(int64_t n, int32_t hidden) { return (size_t)((n + 15) / 16) * 16 * hidden * 4; }
size_t few_x_bytes(int32_t dtype, int64_t n, int64_t width) {
  return (size_t)((n + 15) / 16) * 16 * width * dtype_size(dtype);
}

int few_embed(int32_t dtype, int64_t n, const int32_t* ids, const void* table, int64_t vocab, int32_t hidden, float* h,
              void* hf, hipStream_t st) {
  const int32_t blocks = (int32_t)((n + 15) / 16);
  if (dtype == INL_BF16)
    hipLaunchKernelGGL(few_embed_kernel<bf16>, dim3((unsigned)n), dim3(256), 0, st, ids, (const char*)table, vocab,
                       hidden, blocks, h, (char*)hf);
  else
    hipLaunchKernelGGL(few_embed_kernel<float>, dim3((unsigned)n), dim3(256), 0, st, ids, (const char*)table, vocab,
                       hidden, blocks, h, (char*)hf);
  INL_HIP_TRY(hipGetLastError());
  return INL_OK;
}

int few_attn(int32_t dtype, int32_t n_texts, int64_t n, int32_t longest, const int32_t* cu, const void* qkv, int64_t qs,
             int32_t heads, int32_t kv_heads, const void* qw, const void* kw, float eps, const float* cos,
             const float* sin, void* of, const SkinnyNext& next, hipStream_t st) {
  FewAttnParams p{};
  p.next = next;
  p.n_texts = n_texts;
  p.qkv = (const char*)qkv;
  p.qw = (const char*)qw;
  p.kw = (const char*)kw;
  p.cos = cos;
  p.sin = sin;
  p.cu = cu;
  p.of = (char*)of;
  p.qs = qs;
  p.heads = heads;
  p.kv_heads = kv_heads;
  p.blocks = (int32_t)((n + 15) / 16);
  p.eps = eps;
  p.scale_log2 = 1.4426950408889634f / sqrtf((float)FEW_D);
  return dtype == INL_BF16 ? few_attn_by_len<bf16>(p, longest, st)
                           : few_attn_by_len<float>(p, longest, st);
}

int skinny_launch(int32_t dtype, int64_t m, int32_t n, int32_t k, const void* xf, const void* gamma, float eps,
                  const void* w, int32_t epi, void* y, int64_t ys, void* yf, const SkinnyNext& next,
                  hipStream_t st) {
  SkinnyParams p{};
  p.next = next;
  p.xf = (const char*)xf;
  p.w = (const char*)w;
  p.gamma = (const char*)gamma;
  p.y = (char*)y;
  p.yf = (char*)yf;
  p.ys = ys;
  p.m = (int32_t)m;
  p.n = n;
  p.k = k;
  p.blocks = (int32_t)((m + 15) / 16);
  p.eps = eps;
  if (dtype == INL_BF16) by_kind<bf16>(p, gamma != nullptr, epi, st);
  else by_kind<float>(p, gamma != nullptr, epi, st);
  INL_HIP_TRY(hipGetLastError());
  return INL_OK;
}

}  // namespace inl
