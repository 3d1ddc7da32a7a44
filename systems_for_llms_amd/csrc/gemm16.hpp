// 16-bit MFMA GEMM building blocks shared by the prefill GEMM kernels (gemm.hip,
// gemm_small.hip): arguments, the swizzled LDS stage layout, the XCD-aware tile
// order and the fused epilogues.
#pragma once
#include "attn_mfma.hpp"
#include "lds_dma.hpp"

namespace sfl {

typedef float f32x4 __attribute__((ext_vector_type(4)));

enum GemmEpi { G_PLAIN = 0, G_QKV = 1, G_SWIGLU = 2 };

struct GemmArgs {
  const uint16_t* a;   // [M, K]
  const uint16_t* w;   // [N, K]
  int m, n, k;
  // PLAIN
  void* c;             // [M, N] (ldc = N)
  int c_f32, accumulate;
  // QKV
  const float* cos_t;
  const float* sin_t;
  int seq, heads, head_dim, d_model, cap;
  uint16_t* q_out;     // [B, H, T, dk]
  uint16_t* k_cache;   // [B, H, cap, dk]
  uint16_t* v_cache;
  // SWIGLU
  uint16_t* h_out;     // [M, N/2]
  // PLAIN residual (fp32 C += A W^T) that also prepares the next RMSNorm
  // (norm_gain null: not): norm_act = bf16(C * gain), and per token and part
  // of norm_part features the sum of C^2 in norm_ss [ceil(N / norm_part)][M].
  // norm_part is norm_part_of(tile): 32 for the K-split tiles, else 128; 128
  // asked for by the caller keeps the launch off the K-split tiles.
  const uint16_t* norm_gain;
  uint16_t* norm_act;
  float* norm_ss;
  int norm_part;
  // QKV / SWIGLU fed by such an input: the products are scaled by 1 / rms of
  // token m, given as row_scale[m] or formed from the ss_parts sums of squares
  // ss[part][M] a residual GEMM left (both null: not scaled).
  const float* row_scale;
  const float* ss;
  int ss_parts;
  // Every bf16 output base is 16-byte aligned: the 32x32 kernel then stores
  // 8 consecutive outputs per lane (lane pairs exchange halves first).
  int vec16;
};

template <typename T>
__device__ __forceinline__ f32x4 mfma16(const u32x4& a, const u32x4& b, f32x4 c);
template <>
__device__ __forceinline__ f32x4 mfma16<bf16_t>(const u32x4& a, const u32x4& b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}
template <>
__device__ __forceinline__ f32x4 mfma16<f16_t>(const u32x4& a, const u32x4& b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
}

// One value rounded to T (round to nearest even), as raw bits.
template <typename T> __device__ __forceinline__ uint16_t bits16(float v);
template <> __device__ __forceinline__ uint16_t bits16<bf16_t>(float v) { return f32_to_bf16_bits(v); }
template <> __device__ __forceinline__ uint16_t bits16<f16_t>(float v) { return f32_to_f16_bits(v); }

// The low and high T values of a packed pair, as fp32.
template <typename T> __device__ __forceinline__ float lo16(uint32_t w);
template <typename T> __device__ __forceinline__ float hi16(uint32_t w);
template <> __device__ __forceinline__ float lo16<bf16_t>(uint32_t w) { return bf16_lo(w); }
template <> __device__ __forceinline__ float hi16<bf16_t>(uint32_t w) { return bf16_hi(w); }
template <> __device__ __forceinline__ float lo16<f16_t>(uint32_t w) { return f16_bits_to_f32(uint16_t(w & 0xffffu)); }
template <> __device__ __forceinline__ float hi16<f16_t>(uint32_t w) { return f16_bits_to_f32(uint16_t(w >> 16)); }

// v, or zeros when !keep. Selected per component: a select of whole uint4
// structs is lowered through scratch memory.
__device__ __forceinline__ uint4 keep16(const uint4& v, bool keep) {
  return make_uint4(keep ? v.x : 0u, keep ? v.y : 0u, keep ? v.z : 0u, keep ? v.w : 0u);
}


// Where a lane's 4 QKV features and its token go: section (0 q, 1 k, 2 v),
// head, dim of the first feature; batch row and position of the token.
// Computed once per feature tile / token tile by the caller (integer
// divisions by runtime sizes are long instruction sequences).
struct QkvFeat { int section, head, dim; };
struct QkvTok { int b, t; };

__device__ __forceinline__ QkvFeat qkv_feat(const GemmArgs& g, int n) {
  const int section = n / g.d_model;
  const int f = n - section * g.d_model;
  const int head = f / g.head_dim;
  return QkvFeat{section, head, f - head * g.head_dim};
}
// qkv_feat of feature nt + off from base = qkv_feat(nt), 0 <= off < 32: the
// head changes at most twice within 32 features (head dims >= 16), so two
// compare-and-wrap steps replace the two integer divisions.
__device__ __forceinline__ QkvFeat qkv_feat_at(const GemmArgs& g, const QkvFeat& base, int off) {
  QkvFeat f{base.section, base.head, base.dim + off};
#pragma unroll
  for (int w = 0; w < 2; ++w) {
    if (f.dim >= g.head_dim) {
      f.dim -= g.head_dim;
      if (++f.head == g.heads) {
        f.head = 0;
        ++f.section;
      }
    }
  }
  return f;
}
__device__ __forceinline__ QkvTok qkv_tok(const GemmArgs& g, int m) {
  const int b = m / g.seq;
  return QkvTok{b, m - b * g.seq};
}

// RoPE (attention.py:44-58) of 4 consecutive q or k features (dims dim ..
// dim+3 of one head: two rotation pairs) of token qt; v features pass through.
__device__ __forceinline__ void rope4(const GemmArgs& g, float (&y)[4], const QkvFeat& qf, const QkvTok& qt) {
  if (qf.section >= 2) return;
  // Feature-major tables [head_dim / 2][cap]: the 32 lanes of a group hold 32
  // consecutive tokens, so each load reads consecutive floats (row-major
  // tables put the 32 tokens on 32 cache lines: 345 -> 330 us on the 324M
  // q/k/v shape, same values).
  const long r0 = long(qf.dim / 2) * g.cap + qt.t;
  const float2 c = make_float2(g.cos_t[r0], g.cos_t[r0 + g.cap]);
  const float2 s = make_float2(g.sin_t[r0], g.sin_t[r0 + g.cap]);
  const float e0 = y[0], o0 = y[1], e1 = y[2], o1 = y[3];
  y[0] = e0 * c.x - o0 * s.x;
  y[1] = e0 * s.x + o0 * c.x;
  y[2] = e1 * c.y - o1 * s.y;
  y[3] = e1 * s.y + o1 * c.y;
}

// Destination of feature qf of token qt: q [B, H, T, dk] or the k / v cache [B, H, cap, dk].
__device__ __forceinline__ uint16_t* qkv_dst(const GemmArgs& g, const QkvFeat& qf, const QkvTok& qt) {
  if (qf.section == 0) return g.q_out + ((long(qt.b) * g.heads + qf.head) * g.seq + qt.t) * g.head_dim + qf.dim;
  uint16_t* cache = qf.section == 1 ? g.k_cache : g.v_cache;
  return cache + ((long(qt.b) * g.heads + qf.head) * g.cap + qt.t) * g.head_dim + qf.dim;
}

// silu(a) * c = a * c / (1 + e^-a) with the hardware base-2 exponential and
// reciprocal (e^-a = 2^(-a log2 e); each ~1 ulp): the bf16 rounding of the
// result dominates their error. a -> -inf gives 2^+inf = inf and a zero
// reciprocal (a signed zero), as the exact form does.
__device__ __forceinline__ float silu_mul(float a, float c) {
  const float e = __builtin_amdgcn_exp2f(a * -1.4426950408889634f);
  return a * c * __builtin_amdgcn_rcpf(1.f + e);
}

// Two packed groups of 4 bf16 outputs, A (lane-local features f .. f+3) and
// B (f+8 .. f+11), where lane l ^ 32 holds f+4 .. f+7 and f+12 .. f+15: one
// v_permlane32_swap per dword gives lanes 0..31 features f .. f+7 (own A,
// partner's A) and lanes 32..63 features f+8 .. f+15 (partner's B, own B),
// one 16-byte store each instead of two 8-byte stores.
__device__ __forceinline__ uint4 pair8(const uint32_t (&a)[2], const uint32_t (&b)[2]) {
  const auto s0 = __builtin_amdgcn_permlane32_swap(a[0], b[0], false, false);
  const auto s1 = __builtin_amdgcn_permlane32_swap(a[1], b[1], false, false);
  return make_uint4(s0[0], s1[0], s0[1], s1[1]);
}

// Epilogue of one 16x16 MFMA tile: v holds features nt + 4*grp + (0..3) of
// token m. Every lane must call it (the SwiGLU pairing shuffles).
template <typename T, int E>
__device__ __forceinline__ void store_tile(const GemmArgs& g, const f32x4& v, int nt, int grp, int m,
                                           QkvFeat qf = QkvFeat{}, QkvTok qt = QkvTok{}) {
  const int n = nt + 4 * grp;
  float y[4] = {v[0], v[1], v[2], v[3]};
  if constexpr (E == G_SWIGLU) {
    // Rows 0..7 of the 16-row tile are W1 features, rows 8..15 the
    // matching W3 features: lane groups 0,1 pair with groups 2,3.
    float c3[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) c3[e] = lane_xor(y[e], 32);
    if (grp >= 2 || m >= g.m) return;
    const int f = nt / 2 + 4 * grp;  // hidden feature index
    if (f >= g.n / 2) return;
    float h[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) h[e] = silu_mul(y[e], c3[e]);
    *reinterpret_cast<uint2*>(g.h_out + long(m) * (g.n / 2) + f) = make_uint2(pack2<T>(h[0], h[1]), pack2<T>(h[2], h[3]));
  } else {
    if (m >= g.m || n >= g.n) return;
    if constexpr (E == G_PLAIN) {
      if (g.c_f32) {
        float* c = static_cast<float*>(g.c) + long(m) * g.n + n;
        if (n + 3 < g.n && (g.n & 3) == 0) {
          float4 old = g.accumulate ? *reinterpret_cast<const float4*>(c) : make_float4(0.f, 0.f, 0.f, 0.f);
          *reinterpret_cast<float4*>(c) = make_float4(old.x + y[0], old.y + y[1], old.z + y[2], old.w + y[3]);
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (n + e < g.n) c[e] = (g.accumulate ? c[e] : 0.f) + y[e];
        }
      } else {
        uint16_t* c = static_cast<uint16_t*>(g.c) + long(m) * g.n + n;
        if (n + 3 < g.n && (g.n & 3) == 0) {
          *reinterpret_cast<uint2*>(c) = make_uint2(pack2<T>(y[0], y[1]), pack2<T>(y[2], y[3]));
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (n + e < g.n) c[e] = bits16<T>(y[e]);
        }
      }
    } else {  // G_QKV
      rope4(g, y, qf, qt);
      *reinterpret_cast<uint2*>(qkv_dst(g, qf, qt)) = make_uint2(pack2<T>(y[0], y[1]), pack2<T>(y[2], y[3]));
    }
  }
}

constexpr int K2 = 64;     // K step


template <int TN_, int TM_, int SL_>
struct Stage32 {
  uint4 w[TN_][SL_];  // [row][swizzled 16-byte slot]
  uint4 a[TM_][SL_];
};

// Physical 16-byte slot offset of row r in a stage of SL slots per row: the
// XOR under which the MFMA operand reads (16 consecutive lanes reading rows r
// .. r+15 at one logical slot, 256 bytes per LDS cycle) touch every bank
// once. Rows of 128 bytes already alternate bank halves, rows of 64 bytes
// cycle through bank quarters, so the swizzle only has to separate rows that
// share a half / quarter.
template <int SL>
__device__ __forceinline__ int stage_swizzle(int r) {
  return SL == 8 ? (r >> 1) & 7 : (r >> 2) & 3;
}

// Tile of workgroup b in a 1-D grid of tn x tm tiles, XCD-aware: workgroups
// are dealt to the 8 XCDs round-robin (b % 8) and each XCD has its own L2, so
// XCD x is given a contiguous range of the tile order, and that order walks
// groups of gm token tiles across the feature tiles. The workgroups an
// XCD runs at once then cover about 4 token tiles x 8 feature tiles, whose
// operands stay in (or near) its 4 MB L2 (for 256 x 384 tiles, 448 KB of the
// 2.5 MB a K step requests are distinct).
constexpr int kGroupM = 4;

__device__ __forceinline__ int2 xcd_tile(int b, int tn, int tm, int gm = kGroupM) {
  const int total = tn * tm;
  const int x = b % kXcds, idx = b / kXcds;
  const int base = total / kXcds, extra = total % kXcds;  // XCD x gets base + (x < extra) tiles
  const int t = x * base + min(x, extra) + idx;
  const int group = t / (gm * tn);
  const int gm0 = group * gm;
  const int gsize = min(gm, tm - gm0);
  const int r = t - group * gm * tn;
  return make_int2(r / gsize, gm0 + r % gsize);  // (feature tile, token tile)
}


// Epilogue of one 32x32 MFMA block that is not a residual update: acc[4q + e]
// holds feature nt + 8q + 4hf + e of token m (hf: the lane's half), scaled by
// rsc. Every lane of the wave must call it (lane pairs exchange halves).
template <typename T, int E>
__device__ __forceinline__ void store_block(const GemmArgs& g, const f32x16& acc, int nt, int m, const QkvTok& tok,
                                            float rsc, int hf) {
  // One division pair per 32-feature block; the lane's features derive from
  // it. With head dims that are multiples of 32 the block is one head of one
  // section: its features share the destination row.
  const QkvFeat fb = E == G_QKV ? qkv_feat(g, nt) : QkvFeat{};
  const bool blk = E == G_QKV && g.head_dim % 32 == 0;
  uint16_t* const base = blk ? qkv_dst(g, fb, tok) : nullptr;
  if constexpr (E == G_SWIGLU) {
    // W1/W3 interleaved in blocks of 8 rows: groups q = 0, 2 are W1 features,
    // q + 1 the matching W3 features, all in this lane. Hidden features
    // nt/2 + 4q + 4hf .. +3; with vec16 the two groups go out as one
    // 16-byte store per lane at nt/2 + 8hf (d_ff % 8 == 0: a group of 8 is
    // wholly inside or outside d_ff).
    uint32_t pk[2][2];
#pragma unroll
    for (int q = 0; q < 4; q += 2) {
      float h[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float a1 = acc[4 * q + e] * rsc, a3 = acc[4 * q + 4 + e] * rsc;
        h[e] = silu_mul(a1, a3);
      }
      pk[q / 2][0] = pack2<T>(h[0], h[1]);
      pk[q / 2][1] = pack2<T>(h[2], h[3]);
    }
    if (g.vec16) {
      const uint4 v8 = pair8(pk[0], pk[1]);
      const int f = nt / 2 + 8 * hf;
      if (m < g.m && f < g.n / 2) *reinterpret_cast<uint4*>(g.h_out + long(m) * (g.n / 2) + f) = v8;
    } else if (m < g.m) {
#pragma unroll
      for (int q = 0; q < 4; q += 2) {
        const int f = nt / 2 + 4 * q + 4 * hf;  // hidden feature index
        if (f < g.n / 2)
          *reinterpret_cast<uint2*>(g.h_out + long(m) * (g.n / 2) + f) = make_uint2(pk[q / 2][0], pk[q / 2][1]);
      }
    }
  } else if (E != G_PLAIN || (!g.c_f32 && !g.accumulate)) {
    // bf16 outputs (q/k/v, plain bf16): feature groups q and q + 1 of the
    // lane pair go out as 16-byte stores (vec16; whole 32-feature blocks
    // inside N), else 8 bytes per group.
    const bool wide = g.vec16 && nt + 32 <= g.n && (E == G_QKV || g.n % 8 == 0);
#pragma unroll
    for (int q = 0; q < 4; q += 2) {
      uint32_t pk[2][2];
      QkvFeat feat[2];
#pragma unroll
      for (int r = 0; r < 2; ++r) {
        float y[4] = {acc[4 * (q + r)] * rsc, acc[4 * (q + r) + 1] * rsc,
                      acc[4 * (q + r) + 2] * rsc, acc[4 * (q + r) + 3] * rsc};
        feat[r] = E != G_QKV ? QkvFeat{}
                  : blk ? QkvFeat{fb.section, fb.head, fb.dim + 8 * (q + r) + 4 * hf}
                        : qkv_feat_at(g, fb, 8 * (q + r) + 4 * hf);
        if constexpr (E == G_QKV) rope4(g, y, feat[r], tok);
        pk[r][0] = pack2<T>(y[0], y[1]);
        pk[r][1] = pack2<T>(y[2], y[3]);
      }
      if (wide) {
        const uint4 v8 = pair8(pk[0], pk[1]);
        if (m < g.m) {
          const int f = nt + 8 * q + 8 * hf;  // first of this lane's 8 features
          uint16_t* dst = E == G_QKV ? (blk ? base + 8 * q + 8 * hf : qkv_dst(g, qkv_feat_at(g, fb, 8 * q + 8 * hf), tok))
                                     : static_cast<uint16_t*>(g.c) + long(m) * g.n + f;
          *reinterpret_cast<uint4*>(dst) = v8;
        }
      } else if (m < g.m) {
#pragma unroll
        for (int r = 0; r < 2; ++r) {
          const int n = nt + 8 * (q + r) + 4 * hf;
          if (E == G_QKV) {
            if (n < g.n) *reinterpret_cast<uint2*>(qkv_dst(g, feat[r], tok)) = make_uint2(pk[r][0], pk[r][1]);
          } else if (n + 3 < g.n && (g.n & 3) == 0) {
            *reinterpret_cast<uint2*>(static_cast<uint16_t*>(g.c) + long(m) * g.n + n) =
                make_uint2(pk[r][0], pk[r][1]);
          } else {
            uint16_t* c = static_cast<uint16_t*>(g.c) + long(m) * g.n + n;
            const uint32_t w[2] = {pk[r][0], pk[r][1]};
#pragma unroll
            for (int e = 0; e < 4; ++e)
              if (n + e < g.n) c[e] = uint16_t(w[e / 2] >> (16 * (e % 2)));
          }
        }
      }
    }
  } else {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const f32x4 v = {acc[4 * q] * rsc, acc[4 * q + 1] * rsc, acc[4 * q + 2] * rsc,
                       acc[4 * q + 3] * rsc};
      // store_tile's feature index is nt + 4 * grp: grp = 2q + hf.
      const QkvFeat feat = E == G_QKV ? qkv_feat_at(g, fb, 8 * q + 4 * hf) : QkvFeat{};
      store_tile<T, E>(g, v, nt, 2 * q + hf, m, feat, tok);
    }
  }
}

// Epilogue of one 32x32 block of a residual update (fp32 C, N % 4 == 0): acc
// already holds the updated C values of features nt + 8q + 4hf + (0..3) of
// token m. With norm, T(x * gain) (gw: this lane's gains) goes to norm_act and
// the lane's sum of x^2 is added to ssq. Every lane of the wave must call it.
template <typename T>
__device__ __forceinline__ void residual_block(const GemmArgs& g, const f32x16& acc, int nt, int m, int hf, bool norm,
                                               const uint2 (&gw)[4], float& ssq) {
  float* const c = static_cast<float*>(g.c);
  uint32_t pk[4][2];  // T(x * gain) of features nt + 8q + 4hf + (0..3)
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int n = nt + 8 * q + 4 * hf;
    const float4 v = make_float4(acc[4 * q], acc[4 * q + 1], acc[4 * q + 2],
                                 acc[4 * q + 3]);
    const bool in = m < g.m && n < g.n;
    if (in) *reinterpret_cast<float4*>(c + long(m) * g.n + n) = v;
    if (norm) {
      pk[q][0] = pack2<T>(v.x * lo16<T>(gw[q].x), v.y * hi16<T>(gw[q].x));
      pk[q][1] = pack2<T>(v.z * lo16<T>(gw[q].y), v.w * hi16<T>(gw[q].y));
      if (in) ssq += (v.x * v.x + v.y * v.y) + (v.z * v.z + v.w * v.w);
    }
  }
  if (norm) {
    if (g.vec16) {  // 8 consecutive features per lane (every lane swaps)
#pragma unroll
      for (int q = 0; q < 4; q += 2) {
        const uint4 o = pair8(pk[q], pk[q + 1]);
        const int n = nt + 8 * q + 8 * hf;
        if (m < g.m && n < g.n) *reinterpret_cast<uint4*>(g.norm_act + long(m) * g.n + n) = o;
      }
    } else {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int n = nt + 8 * q + 4 * hf;
        if (m < g.m && n < g.n)
          *reinterpret_cast<uint2*>(g.norm_act + long(m) * g.n + n) = make_uint2(pk[q][0], pk[q][1]);
      }
    }
  }
}

// 1 / rms of token m from the parts of its sum of squares: in their order, the
// sum norm_scale_kernel forms, so a consumer that reads them itself gives the
// same bits and saves that launch.
__device__ __forceinline__ float parts_scale(const GemmArgs& g, int m) {
  float t = 0.f;
#pragma unroll 8
  for (int p = 0; p < g.ss_parts; ++p) t += g.ss[long(p) * g.m + m];
  return 1.f / sqrtf(t / float(g.k) + 1e-5f);
}

// Output tile (features x tokens) of a launch. S*: K split over the waves
// (gemm_small.hip); T*: K in LDS steps shared by the waves (gemm.hip).
enum Tile16 { S32x32, S64x32, S64x64, S128x64, T128x64, T128x128, T256x256, T256x384 };

// The tile for an [M, K] x [N, K]^T product with epilogue `epi`; see gemm.hip.
Tile16 tile16_for(long m, long n, long k, int epi);
inline int norm_part_of(Tile16 t) { return t <= S128x64 ? 32 : 128; }

// Explicitly instantiated in gemm_small.hip for bf16/fp16 and every epilogue
// (t: one of S*). Preconditions: K % 64 == 0 and operands under 2^30 elements.
template <typename T, int E>
int launch_gemm_small(const GemmArgs& g, Tile16 t, hipStream_t s, const char* what);

}  // namespace sfl
