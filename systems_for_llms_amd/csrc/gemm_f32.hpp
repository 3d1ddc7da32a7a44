// fp32 prefill GEMMs (prefill_f32.hip): the arguments the 16-bit GEMM entry
// points (gemm.hip) pass through when their dtype is SFL_DTYPE_F32.
#pragma once
#include <math.h>

#include "attn_mfma.hpp"

namespace sfl {

enum F32Epi { F32_PLAIN = 0, F32_QKV = 1, F32_SWIGLU = 2 };

struct F32GemmArgs {
  const float* a;  // [M, K]
  const float* w;  // [N, K]
  int m, n, k;
  // PLAIN: C [M, N] fp32, stored or (accumulate) added to
  float* c;
  int accumulate;
  // QKV: RoPE from the feature-major tables [head_dim / 2, cap]; q to
  // [B, H, T, dk], k / v to the [B, H, cap, dk] cache at positions 0..T-1
  const float* cos_t;
  const float* sin_t;
  int seq, heads, head_dim, d_model, cap;
  float* q_out;
  float* k_cache;
  float* v_cache;
  // SWIGLU: W is W1/W3 interleaved in blocks of 8 rows; h [M, N / 2]
  float* h_out;
};

// silu(a) * c with an IEEE exponential (layers.py:102-104,114-115).
__device__ __forceinline__ float silu_mul_f32(float a, float c) { return a / (1.f + expf(-a)) * c; }

// Epilogue of one 32x32 block: acc[4q + e] holds feature nt + 8q + 4hf + e of token m.
template <int E>
__device__ __forceinline__ void store_block_f32(const F32GemmArgs& g, const f32x16& acc, int nt, int m, int hf) {
  if (m >= g.m) return;
  if constexpr (E == F32_SWIGLU) {
    // Groups q = 0, 2 are W1 rows, q + 1 the W3 rows of the same hidden features
    // nt/2 + 4q + 4hf .. +3.
#pragma unroll
    for (int q = 0; q < 4; q += 2) {
      const int f = nt / 2 + 4 * q + 4 * hf;
      if (f >= g.n / 2) continue;
      float h[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) h[e] = silu_mul_f32(acc[4 * q + e], acc[4 * q + 4 + e]);
      *reinterpret_cast<float4*>(g.h_out + long(m) * (g.n / 2) + f) = make_float4(h[0], h[1], h[2], h[3]);
    }
  } else if constexpr (E == F32_QKV) {
    const int b = m / g.seq, t = m - (m / g.seq) * g.seq;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int n = nt + 8 * q + 4 * hf;
      if (n >= g.n) continue;
      const int section = n / g.d_model;
      const int fi = n - section * g.d_model;
      const int head = fi / g.head_dim, dim = fi - (fi / g.head_dim) * g.head_dim;
      float y[4] = {acc[4 * q], acc[4 * q + 1], acc[4 * q + 2], acc[4 * q + 3]};
      if (section < 2) {  // RoPE pairs (dim, dim+1), (dim+2, dim+3) (attention.py:44-58)
        const long r0 = long(dim / 2) * g.cap + t;
        const float c0 = g.cos_t[r0], c1 = g.cos_t[r0 + g.cap];
        const float s0 = g.sin_t[r0], s1 = g.sin_t[r0 + g.cap];
        const float e0 = y[0], o0 = y[1], e1 = y[2], o1 = y[3];
        y[0] = e0 * c0 - o0 * s0;
        y[1] = e0 * s0 + o0 * c0;
        y[2] = e1 * c1 - o1 * s1;
        y[3] = e1 * s1 + o1 * c1;
      }
      float* dst = section == 0 ? g.q_out + ((long(b) * g.heads + head) * g.seq + t) * g.head_dim + dim
                                : (section == 1 ? g.k_cache : g.v_cache) +
                                      ((long(b) * g.heads + head) * g.cap + t) * g.head_dim + dim;
      *reinterpret_cast<float4*>(dst) = make_float4(y[0], y[1], y[2], y[3]);
    }
  } else {  // F32_PLAIN
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int n = nt + 8 * q + 4 * hf;
      float* c = g.c + long(m) * g.n + n;
      if (n + 3 < g.n && (g.n & 3) == 0) {
        float4 v = make_float4(acc[4 * q], acc[4 * q + 1], acc[4 * q + 2], acc[4 * q + 3]);
        if (g.accumulate) {
          const float4 old = *reinterpret_cast<const float4*>(c);
          v = make_float4(old.x + v.x, old.y + v.y, old.z + v.z, old.w + v.w);
        }
        *reinterpret_cast<float4*>(c) = v;
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (n + e < g.n) c[e] = (g.accumulate ? c[e] : 0.f) + acc[4 * q + e];
      }
    }
  }
}

// Launches the fp32 GEMM with epilogue `epi` (argument checks done by the caller).
int launch_gemm_f32(const F32GemmArgs& g, int epi, hipStream_t stream, const char* what);

}  // namespace sfl
