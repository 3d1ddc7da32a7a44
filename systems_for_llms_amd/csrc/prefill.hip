// The launches of a whole prefill in one host call. A prompt of a few hundred
// tokens is 5 launches of 5-13 us per layer; issued one ctypes call at a time
// they cost the host 7-25 us each, so the 100M model's short prompts waited on
// Python (forward of 2 x 205 tokens: 830 us of host time, ~450 of kernels).
#include "common.hpp"

using namespace sfl;

extern "C" int sfl_prefill_layers(const sfl_prefill_args* p, void* stream) {
  const char* what = "prefill_layers";
  if (!p || !p->ids || !p->emb || !p->attn_norm || !p->w_qkv || !p->w_out || !p->ffn_norm || !p->w13 || !p->w2 ||
      !p->k_cache || !p->v_cache || !p->x || !p->act || !p->q || !p->attn || !p->hidden ||
      (p->fold && (!p->ss || !p->rscale)))
    return set_error(SFL_ERR_INVALID, "%s: null pointer argument", what);
  if (p->layers < 1 || p->batch < 1 || p->seq < 1 || p->d_model < 1 || p->heads < 1 || p->d_ff < 1 ||
      p->d_model % p->heads || long(p->batch) * p->seq > (1L << 31) - 1)
    return set_error(SFL_ERR_INVALID, "%s: bad sizes", what);
  const int m = p->batch * p->seq, t = p->seq, d = p->d_model, f = p->d_ff, h = p->heads, dk = d / h, dt = p->dtype;
  const int F32 = SFL_DTYPE_F32;
  // Strides (batch, head, position) of q, the caches and the [B, T, H, dk] attention output.
  const long qs[3] = {long(h) * t * dk, long(t) * dk, dk};
  const long cs[3] = {long(h) * p->capacity * dk, long(p->capacity) * dk, dk};
  const long os[3] = {long(t) * h * dk, dk, long(h) * dk};
  const int part_o = sfl_gemm_norm_part(m, d, d), part_f = sfl_gemm_norm_part(m, d, f);
  const int parts_o = (d + part_o - 1) / part_o, parts_f = (d + part_f - 1) / part_f;
#define SFL_TRY(call)           \
  do {                          \
    if (int rc = (call)) return rc; \
  } while (0)
  SFL_TRY(sfl_embed_rows(p->ids, p->emb, p->x, m, d, dt, stream));
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
  return SFL_OK;
}
