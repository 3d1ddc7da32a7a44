// The launches of a whole prefill in one host call. A prompt of a few hundred
// tokens is 5 launches of 5-13 us per layer; issued one ctypes call at a time
// they cost the host 7-25 us each, so the 100M model's short prompts waited on
// Python (forward of 2 x 205 tokens: 830 us of host time, ~450 of kernels).
#include <algorithm>

#include "common.hpp"

using namespace sfl;

namespace sfl {
namespace {

// State of the session and embedding of the prompt: x[r] = emb[given[r]] in
// fp32, one workgroup per prompt position r < rows; the [batch, capacity] token
// arrays are dealt over the whole grid, which has workgroups of its own for
// them where the prompt is short and the capacity long (begin_grid). Bound by the launch (5 us for 2048 rows of
// 512): one kernel where fills, copies and the gather were six, each 1.5-5 us
// with 10-25 us of host time ahead of the first layer. Every prefill is ~25 us
// shorter for this and the last position's kernel below: 24 tokens of 3
// sequences on the 100M model 501 -> 437 us, 2048 on the fp32 pilot 748 -> 721.
template <typename T>
__global__ __launch_bounds__(128) void prefill_begin_kernel(
    const int64_t* __restrict__ given, const T* __restrict__ emb, float* __restrict__ x, int d, int seq, int given_len,
    int batch, int cap, int64_t* __restrict__ tokens, int64_t* __restrict__ predicted, int32_t* __restrict__ prompt_len) {
  constexpr int V = vec_elems<T>();
  const unsigned m = blockIdx.x;
  if (m < unsigned(batch) * unsigned(seq)) {
    const unsigned b = m / unsigned(seq), t = m - b * unsigned(seq);
    const T* src = emb + given[long(b) * given_len + t] * d;
    float* xr = x + long(m) * d;
    const bool wide = reinterpret_cast<uintptr_t>(emb) % 16 == 0;  // rows are multiples of 32 bytes
    for (int i = V * threadIdx.x; i < d; i += V * 128) {
      float v[V];
      if (wide) {
        unpack16<T>(load16(src + i), v);
      } else {
#pragma unroll
        for (int j = 0; j < V; ++j) v[j] = load_scalar<T>(src + i + j);
      }
#pragma unroll
      for (int j = 0; j < V; j += 4)
        *reinterpret_cast<float4*>(xr + i + j) = make_float4(v[j], v[j + 1], v[j + 2], v[j + 3]);
    }
  }
  const long all = long(batch) * cap;
  for (long i = long(m) * 128 + threadIdx.x; i < all; i += long(gridDim.x) * 128) {
    const long row = i / cap, col = i - row * cap;
    tokens[i] = col < given_len ? given[row * given_len + col] : 0;
    predicted[i] = -1;
    if (col == 0) prompt_len[row] = given_len;
  }
}

// The last position's rows, where the decode step's lm_head reads them.
__global__ __launch_bounds__(256) void prefill_end_kernel(const float* __restrict__ x, float* __restrict__ x_last,
                                                          int d, int seq, int32_t* __restrict__ pos,
                                                          int32_t* __restrict__ lengths) {
  const long b = blockIdx.x;
  const float4* src = reinterpret_cast<const float4*>(x + ((b + 1) * seq - 1) * d);
  float4* dst = reinterpret_cast<float4*>(x_last + b * d);
  for (int i = threadIdx.x; i < d / 4; i += 256) dst[i] = src[i];
  if (threadIdx.x == 0) {
    pos[b] = seq - 1;
    lengths[b] = seq;
  }
}

// Workgroups of prefill_begin_kernel: one per prompt position, and enough that
// a thread fills about 4 entries of the token arrays (up to 8 per CU; with the
// prompt's alone, one token at a capacity of 131072 filled them on one CU:
// 174 us, now 4.7; 4096 7.2 -> 4.6).
inline unsigned begin_grid(long rows, long entries) {
  return unsigned(std::max(rows, std::min(2048L, (entries + 511) / 512)));
}

template <typename T>
int launch_begin(const sfl_prefill_args* p, hipStream_t s) {
  const dim3 grid(begin_grid(long(p->batch) * p->seq, long(p->batch) * p->capacity));
  hipLaunchKernelGGL(prefill_begin_kernel<T>, grid, dim3(128), 0, s, p->given,
                     static_cast<const T*>(p->emb), p->x, p->d_model, p->seq, p->given_len, p->batch, p->capacity,
                     p->tokens, p->predicted, p->prompt_len);
  return check_launch("prefill_layers");
}

}  // namespace
}  // namespace sfl

namespace sfl {
namespace {

// Whatever an entry point of the sequence would refuse, refused before the
// first launch: a call that fails leaves the session as it was.
int check_prefill(const sfl_prefill_args* p, const char* what) {
  if (!p || !p->given || !p->tokens || !p->predicted || !p->prompt_len || !p->pos || !p->lengths || !p->x_last ||
      !p->emb || !p->attn_norm || !p->w_qkv || !p->w_out || !p->ffn_norm || !p->w13 || !p->w2 || !p->k_cache ||
      !p->v_cache || !p->cos_t || !p->sin_t || !p->x || !p->act || !p->q || !p->attn || !p->hidden ||
      (p->fold && (!p->ss || !p->rscale)))
    return set_error(SFL_ERR_INVALID, "%s: null pointer argument", what);
  if (p->layers < 1 || p->batch < 1 || p->seq < 1 || p->d_model < 1 || p->heads < 1 || p->d_ff < 1 ||
      p->d_model % p->heads || p->d_model % 16 || p->given_len < p->seq || p->capacity < p->given_len ||
      long(p->batch) * p->seq > (1L << 31) - 1)
    return set_error(SFL_ERR_INVALID, "%s: bad sizes", what);
  if (p->dtype != SFL_DTYPE_F32 && p->dtype != SFL_DTYPE_BF16 && p->dtype != SFL_DTYPE_F16)
    return set_error(SFL_ERR_UNSUPPORTED, "%s: model dtype must be F32, BF16 or F16", what);
  if (!(p->scale > 0.f) || !__builtin_isfinite(p->scale))
    return set_error(SFL_ERR_INVALID, "%s: scale must be finite and positive", what);
  const bool f32 = p->dtype == SFL_DTYPE_F32;
  const long m = long(p->batch) * p->seq, d = p->d_model, f = p->d_ff, dk = d / p->heads;
  if (dk != 32 && dk != 64 && dk != 128 && !(f32 && dk == 16))
    return set_error(SFL_ERR_UNSUPPORTED, "%s: head dim must be 32, 64 or 128 (F32: or 16)", what);
  if (f % 8) return set_error(SFL_ERR_UNSUPPORTED, "%s: d_ff must be a multiple of 8", what);
  if ((p->seq + 63L) / 64 * p->batch * p->heads > (1L << 31) - 1)
    return set_error(SFL_ERR_UNSUPPORTED, "%s: too many query tiles", what);
  // [m, k] x [n, k]^T: 32-bit operand offsets, or the kernel for any size with its grid of up to 65535 token tiles.
  const auto gemm_ok = [&](long n, long k) {
    const long limit = f32 ? 1L << 29 : 1L << 30;
    return (k % (f32 ? 32 : 64) == 0 && m * k < limit && n * k < limit) || m <= 65535L * (f32 ? 64 : 128);
  };
  if (!gemm_ok(3 * d, d) || !gemm_ok(d, d) || !gemm_ok(2 * f, d) || !gemm_ok(d, f))
    return set_error(SFL_ERR_UNSUPPORTED, "%s: too many rows", what);
  if (p->fold && (f32 || d % 64 || f % 64 || d > 2048 || m * d >= 1L << 30 || m * f >= 1L << 30 ||
                  3 * d * d >= 1L << 30 || 2 * f * d >= 1L << 30))
    return set_error(SFL_ERR_UNSUPPORTED, "%s: folded norms need 16-bit weights, d_model and d_ff multiples of 64, "
                     "d_model at most 2048 and operands under 2^30 elements", what);
  const auto off = [](const void* q, unsigned n) { return reinterpret_cast<uintptr_t>(q) % n != 0; };
  bool bad = off(p->x, 16) || off(p->x_last, 16) || (p->fold && off(p->act, 8));
  if (f32) bad = bad || off(p->act, 16) || off(p->q, 16) || off(p->attn, 16) || off(p->hidden, 16);
  for (int l = 0; l < p->layers; ++l) {
    if (!p->attn_norm[l] || !p->w_qkv[l] || !p->w_out[l] || !p->ffn_norm[l] || !p->w13[l] || !p->w2[l] ||
        !p->k_cache[l] || !p->v_cache[l])
      return set_error(SFL_ERR_INVALID, "%s: null pointer argument (layer %d)", what, l);
    if (p->fold) bad = bad || off(p->ffn_norm[l], 8) || (l > 0 && off(p->attn_norm[l], 8));
    if (f32)
      bad = bad || off(p->w_qkv[l], 16) || off(p->w_out[l], 16) || off(p->w13[l], 16) || off(p->w2[l], 16) ||
            off(p->k_cache[l], 16) || off(p->v_cache[l], 16);
  }
  if (bad)
    return set_error(SFL_ERR_INVALID, "%s: x and x_last must be 16-byte aligned, folded norms' act and gains 8-byte, "
                     "F32 operands and outputs 16-byte", what);
  return SFL_OK;
}

}  // namespace
}  // namespace sfl

extern "C" int sfl_prefill_layers(const sfl_prefill_args* p, void* stream) {
  const char* what = "prefill_layers";
  if (int rc = check_prefill(p, what)) return rc;
  const hipStream_t s = static_cast<hipStream_t>(stream);
  const int m = p->batch * p->seq, t = p->seq, d = p->d_model, f = p->d_ff, h = p->heads, dk = d / h, dt = p->dtype;
  const int F32 = SFL_DTYPE_F32;
  // Strides (batch, head, position) of q, the caches and the [B, T, H, dk] attention output.
  const long qs[3] = {long(h) * t * dk, long(t) * dk, dk};
  const long cs[3] = {long(h) * p->capacity * dk, long(p->capacity) * dk, dk};
  const long os[3] = {long(t) * h * dk, dk, long(h) * dk};
  const int part_o = sfl_gemm_norm_part(m, d, d), part_f = sfl_gemm_norm_part(m, d, f);
  const int parts_o = (d + part_o - 1) / part_o, parts_f = (d + part_f - 1) / part_f;
#define SFL_TRY(call)               \
  do {                              \
    if (int rc = (call)) return rc; \
  } while (0)
  SFL_TRY(dt == F32              ? launch_begin<float>(p, s)
          : dt == SFL_DTYPE_BF16 ? launch_begin<bf16_t>(p, s)
                                 : launch_begin<f16_t>(p, s));
  if (p->fold)
    SFL_TRY(sfl_rmsnorm_rows_scaled(p->x, p->attn_norm[0], p->act, p->rscale, m, d, dt, stream));
  for (int l = 0; l < p->layers; ++l) {
    if (!p->fold) {
      SFL_TRY(sfl_rmsnorm_rows(p->x, p->attn_norm[l], p->act, m, d, dt, dt, stream));
      SFL_TRY(sfl_gemm_qkv_rope(p->act, p->w_qkv[l], m, t, d, h, p->cos_t, p->sin_t, p->q, p->k_cache[l],
                                p->v_cache[l], p->capacity, dt, stream));
    } else if (l == 0) {
      SFL_TRY(sfl_gemm_qkv_rope_scaled(p->act, p->w_qkv[l], p->rscale, m, t, d, h, p->cos_t, p->sin_t, p->q,
                                       p->k_cache[l], p->v_cache[l], p->capacity, dt, stream));
    } else {
      SFL_TRY(sfl_gemm_qkv_rope_normed(p->act, p->w_qkv[l], p->ss, parts_f, m, t, d, h, p->cos_t, p->sin_t, p->q,
                                       p->k_cache[l], p->v_cache[l], p->capacity, dt, stream));
    }
    if (dt == F32)
      SFL_TRY(sfl_causal_attention_f32(static_cast<const float*>(p->q), static_cast<const float*>(p->k_cache[l]),
                                       static_cast<const float*>(p->v_cache[l]), static_cast<float*>(p->attn),
                                       p->batch, h, t, dk, qs, cs, cs, os, p->scale, stream));
    else
      SFL_TRY(sfl_masked_attention(p->q, p->k_cache[l], p->v_cache[l], p->attn, nullptr, p->batch, h, t, dk, qs, cs,
                                   cs, os, p->scale, 1, -1, -1, 0, nullptr, 0, nullptr, nullptr, nullptr, 1, dt,
                                   stream));
    if (p->fold) {
      SFL_TRY(sfl_gemm_residual_norm_parts(p->attn, p->w_out[l], p->x, m, d, d, p->ffn_norm[l], p->act, p->ss, part_o,
                                           dt, stream));
      SFL_TRY(sfl_gemm_swiglu_normed(p->act, p->w13[l], p->ss, parts_o, p->hidden, m, f, d, dt, stream));
    } else {
      SFL_TRY(sfl_gemm(p->attn, p->w_out[l], p->x, m, d, d, dt, F32, 1, stream));
      SFL_TRY(sfl_rmsnorm_rows(p->x, p->ffn_norm[l], p->act, m, d, dt, dt, stream));
      SFL_TRY(sfl_gemm_swiglu(p->act, p->w13[l], p->hidden, m, f, d, dt, stream));
    }
    if (p->fold && l + 1 < p->layers)
      SFL_TRY(sfl_gemm_residual_norm_parts(p->hidden, p->w2[l], p->x, m, d, f, p->attn_norm[l + 1], p->act, p->ss,
                                           part_f, dt, stream));
    else
      SFL_TRY(sfl_gemm(p->hidden, p->w2[l], p->x, m, d, f, dt, F32, 1, stream));
  }
#undef SFL_TRY
  hipLaunchKernelGGL(prefill_end_kernel, dim3(p->batch), dim3(256), 0, s, p->x, p->x_last, d, t, p->pos, p->lengths);
  return check_launch(what);
}
