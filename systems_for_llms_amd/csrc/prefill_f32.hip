// Prefill of float32 models: the Linear layers as fp32 MFMA GEMMs and causal
// attention in fp32, so a float32 forward over T positions is one pass.
//
// The reference's float32 TransformerLM.forward (src/llmlab/model/
// transformer.py:121-139) runs every Linear (layers.py:34-35) and the
// attention (attention.py:61-98,187-197) in fp32; these kernels form every
// product of fp32 values to within an fp32 rounding and sum in fp32, so they
// differ from it by the order of fp32 additions.
//
// GEMM: K a multiple of 32 and operands under 2 GiB run gemm_split_kernel
// (gemm_split.hpp: K split over the waves, each operand as three exact bf16
// pieces, eight of whose nine products are summed on the bf16 matrix cores;
// the ninth is below 2^-30 of the product). Its tiles with an infinity, a NaN
// or an operand under 2^-110 are computed again on fp32 MFMAs. Other shapes run
// gemm_f32_kernel: C^T[n][m] = sum_k W[n][k] A[m][k] on v_mfma_f32_32x32x2_f32
// (fp32 operands, fp32 accumulation). A workgroup of 4 waves (2 x 2) computes 64
// features x 64 tokens, a wave one 32 x 32 block; K advances by 32 through two
// LDS stages (rows padded to 36 floats), the next stage's global loads in
// registers while the current one computes. A lane reads 16 bytes -- 4
// consecutive k of its row -- per operand and feeds them to 4 MFMAs: lane
// half h takes k = 8 kq + 4 h + s in step s for both operands, so each
// product pairs equal k (the contraction is exact in any shared order). The
// output layout of the 32x32 MFMA puts features 8q + 4h .. +3 of one token in
// a lane, so the epilogues of the 16-bit GEMMs carry over: RoPE pairs in-lane,
// W1/W3 interleaved in blocks of 8 rows paired in-lane, 16-byte stores.
//
// Attention: one workgroup of 4 waves per 64 queries of one (batch, head), the
// same pieces on the matrix cores, an exact fp32 online softmax (base 2, the
// scale folded into q).
#include <math.h>

#include "gemm_split.hpp"

namespace sfl {
namespace {

constexpr int FT = 64;        // features and tokens per workgroup
constexpr int FK = 32;        // K per LDS stage
constexpr int FLD = FK + 4;   // LDS row stride (floats)
constexpr int kF32Threads = 256;

__device__ __forceinline__ f32x16 mfma32f(float a, float b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
}

template <int E>
__global__ __launch_bounds__(kF32Threads) void gemm_f32_kernel(F32GemmArgs g) {
  __shared__ __align__(16) float ws[2][FT * FLD];
  __shared__ __align__(16) float as[2][FT * FLD];
  const int tid = threadIdx.x;
  const int wave = tid / kWave, lane = tid % kWave;
  const int wn = wave / 2, wm = wave % 2;
  const int l32 = lane % 32, hf = lane / 32;
  const int n0 = blockIdx.x * FT;
  const int m0 = blockIdx.y * FT;
  const int ksteps = (g.k + FK - 1) / FK;

  // Thread tid moves row r = idx / 8, floats 4 c4 .. +3 of a stage, idx = tid + 256 i.
  // Loads are unconditional from clamped rows; columns past K are zeroed per
  // component (a select of whole float4 values is lowered through scratch).
  float4 wr[2], ar[2];
#define SFL_F32_GLOAD(kt)                                                                   \
  _Pragma("unroll") for (int i = 0; i < 2; ++i) {                                           \
    const int idx = tid + i * kF32Threads;                                                  \
    const int r = idx / (FK / 4), c4 = idx % (FK / 4);                                      \
    const int kk = (kt) * FK + 4 * c4;                                                      \
    const bool in = kk < g.k;                                                               \
    const int kc = in ? kk : 0;                                                             \
    const float4 w_ = *reinterpret_cast<const float4*>(g.w + long(min(n0 + r, g.n - 1)) * g.k + kc); \
    const float4 a_ = *reinterpret_cast<const float4*>(g.a + long(min(m0 + r, g.m - 1)) * g.k + kc); \
    wr[i] = make_float4(in ? w_.x : 0.f, in ? w_.y : 0.f, in ? w_.z : 0.f, in ? w_.w : 0.f);  \
    ar[i] = make_float4(in ? a_.x : 0.f, in ? a_.y : 0.f, in ? a_.z : 0.f, in ? a_.w : 0.f);  \
  }
#define SFL_F32_SSTORE(buf)                                                                 \
  _Pragma("unroll") for (int i = 0; i < 2; ++i) {                                           \
    const int idx = tid + i * kF32Threads;                                                  \
    const int r = idx / (FK / 4), c4 = idx % (FK / 4);                                      \
    *reinterpret_cast<float4*>(&ws[buf][r * FLD + 4 * c4]) = wr[i];                         \
    *reinterpret_cast<float4*>(&as[buf][r * FLD + 4 * c4]) = ar[i];                         \
  }

  f32x16 acc;
#pragma unroll
  for (int e = 0; e < 16; ++e) acc[e] = 0.f;
  SFL_F32_GLOAD(0)
  SFL_F32_SSTORE(0)
  __syncthreads();
  for (int kt = 0; kt < ksteps; ++kt) {
    const int buf = kt & 1;
    if (kt + 1 < ksteps) { SFL_F32_GLOAD(kt + 1) }
    const float* wrow = &ws[buf][(32 * wn + l32) * FLD + 4 * hf];
    const float* arow = &as[buf][(32 * wm + l32) * FLD + 4 * hf];
#pragma unroll
    for (int kq = 0; kq < FK / 8; ++kq) {
      const float4 av = *reinterpret_cast<const float4*>(wrow + 8 * kq);
      const float4 bv = *reinterpret_cast<const float4*>(arow + 8 * kq);
      acc = mfma32f(av.x, bv.x, acc);
      acc = mfma32f(av.y, bv.y, acc);
      acc = mfma32f(av.z, bv.z, acc);
      acc = mfma32f(av.w, bv.w, acc);
    }
    if (kt + 1 < ksteps) {
      SFL_F32_SSTORE(buf ^ 1)
      __syncthreads();
    }
  }
#undef SFL_F32_GLOAD
#undef SFL_F32_SSTORE

  store_block_f32<E>(g, acc, n0 + 32 * wn, m0 + 32 * wm + l32, hf);
}

struct F32AttnArgs {
  const float *q, *k, *v;
  float* o;
  long qs[3], ks[3], vs[3], os[3];  // strides (elements) of batch, head, sequence
  int batch, heads, n;
  float scale_log2;
};

constexpr int kAttnQ = 64;   // queries per workgroup
constexpr int kAttnK = 64;   // keys per staged tile
constexpr int kValuK = 32;   // keys per tile of causal_rows_valu

// The 64 query rows from qb * 64 of one (batch, head) on the VALU: four
// threads per query, each with a quarter of the head dim; a key above a
// query's row is never read by it. smem: 2 * kValuK * D floats.
template <int D>
__device__ __forceinline__ void causal_rows_valu(const F32AttnArgs& a, int qb, int b, int h, float* smem) {
  constexpr int DQ = D / 4;  // head-dim quarter of a thread
  float (*kt)[D] = reinterpret_cast<float (*)[D]>(smem);
  float (*vt)[D] = kt + kValuK;
  const int tid = threadIdx.x;
  const int qrow = qb * kAttnQ + tid / 4, part = tid % 4;
  const float* qp = a.q + b * a.qs[0] + h * a.qs[1] + long(min(qrow, a.n - 1)) * a.qs[2] + part * DQ;
  float qv[DQ], o[DQ];
#pragma unroll
  for (int d = 0; d < DQ; ++d) {
    qv[d] = qp[d] * a.scale_log2;
    o[d] = 0.f;
  }
  float m_run = -INFINITY, l_run = 0.f;
  const int kend = min(a.n, qb * kAttnQ + kAttnQ);  // keys 0 .. kend-1 cover every row of the block
  const float* kb = a.k + b * a.ks[0] + h * a.ks[1];
  const float* vb = a.v + b * a.vs[0] + h * a.vs[1];
  for (int k0 = 0; k0 < kend; k0 += kValuK) {
    __syncthreads();
    for (int idx = tid; idx < kValuK * D / 4; idx += kF32Threads) {
      const int r = idx / (D / 4), c4 = idx % (D / 4);
      const long key = min(k0 + r, a.n - 1);
      *reinterpret_cast<float4*>(&kt[r][4 * c4]) = *reinterpret_cast<const float4*>(kb + key * a.ks[2] + 4 * c4);
      *reinterpret_cast<float4*>(&vt[r][4 * c4]) = *reinterpret_cast<const float4*>(vb + key * a.vs[2] + 4 * c4);
    }
    __syncthreads();
    const int jn = min(kValuK, kend - k0);  // uniform over the workgroup
    for (int j = 0; j < jn; ++j) {
      float s = 0.f;
#pragma unroll
      for (int d = 0; d < DQ; ++d) s = fmaf(qv[d], kt[j][part * DQ + d], s);
      s += lane_xor(s, 1);
      s += lane_xor(s, 2);
      if (k0 + j <= qrow) {  // causal (attention.py:187-197)
        if (s > m_run) {
          const float alpha = exp2f(m_run - s);  // 0 for the first key
          l_run *= alpha;
#pragma unroll
          for (int d = 0; d < DQ; ++d) o[d] *= alpha;
          m_run = s;
        }
        const float p = exp2f(s - m_run);
        l_run += p;
#pragma unroll
        for (int d = 0; d < DQ; ++d) o[d] = fmaf(p, vt[j][part * DQ + d], o[d]);
      }
    }
  }
  if (qrow >= a.n) return;
  const float inv = 1.f / l_run;  // key 0 is always admissible: l_run >= 1
  float* op = a.o + b * a.os[0] + h * a.os[1] + long(qrow) * a.os[2] + part * DQ;
#pragma unroll
  for (int d = 0; d < DQ; d += 4)
    *reinterpret_cast<float4*>(op + d) = make_float4(o[d] * inv, o[d + 1] * inv, o[d + 2] * inv, o[d + 3] * inv);
}

// Causal attention of 64 queries per workgroup on the bf16 matrix cores, every
// fp32 operand as three exact bf16 pieces, eight products each (split3): S^T =
// K Q^T and O^T += V^T P^T with the layouts of the 16-bit masked attention
// (k_swizzle, vt_slot, transpose reads), K and V split once per tile into
// three LDS planes. Waves 0 and 1 take the first 32 keys of each 64-key tile
// for queries 0..31 and 32..63, waves 2 and 3 the other 32 keys: a wave's
// chain -- the longest row bounds a short launch -- is half as long, and the
// two halves of a row merge through LDS at the end. The softmax is fp32, the
// row sum over the fp32 probabilities (v_exp_f32 gives 0 for one below 2^-126
// of the row's largest, and its pieces keep what is at least 2^-133). Against
// causal_rows_valu for every row (one key at a time, 21 TFLOP/s), causal us:
// 4x12x1000 D 64 272 -> 62, 2x16x4096 D 64 2220 -> 509, 8x16x256 D 32
// 50 -> 12.5, 2x4x2048 D 128 758 -> 166; relative error to float64 (2-norm)
// 3.3e-7 -> 1.3e-7 at 4x12x1000, 2.0e-7 -> 1.0e-7 at 8x16x256. Bound by the
// split and softmax VALU work beside ~2000 MFMA cycles per 32 x 32 block at
// D 64; 3 waves per SIMD there do not fit its 230 registers. A row that comes
// out NaN (an infinity or NaN in q, k or v, which the pieces do not carry, or
// which a masked key's zero probability would multiply) or an operand its
// pieces do not hold sends its workgroup to causal_rows_valu.
template <int D>
__global__ __launch_bounds__(kF32Threads) __attribute__((amdgpu_waves_per_eu(D < 64 ? 3 : D == 64 ? 2 : 1)))
void causal_attention_f32_kernel(F32AttnArgs a) {
  constexpr int DL = D < 64 ? 64 : D;          // LDS row width (values)
  constexpr int RS = DL / 8;                   // 16-byte slots per LDS row
  constexpr int SL = D / 8;                    // of which used
  constexpr int KS = D / 16;                   // MFMA steps over the head dim
  constexpr int DT = D < 32 ? 1 : D / 32;      // 32-wide dim tiles of O^T
  constexpr int NLD = (kAttnK * SL + kF32Threads - 1) / kF32Threads;  // slots a thread stages per operand
  struct Lds {
    uint4 k[3][kAttnK][RS];
    uint4 v[3][kAttnK][RS];
  };
  __shared__ __align__(16) Lds st;
  static_assert(sizeof(Lds) >= sizeof(float) * 2 * kValuK * D, "the VALU rows fit");
  static_assert(sizeof(Lds) >= sizeof(float) * 2 * kWave * (16 * DT + 2), "the merge rows fit");
  const int2 tile = attn_tile((a.n + kAttnQ - 1) / kAttnQ, a.batch * a.heads);
  const int qb = __builtin_amdgcn_readfirstlane(tile.x), bh = __builtin_amdgcn_readfirstlane(tile.y);
  const int b = bh / a.heads, hd = bh % a.heads;
  const int tid = threadIdx.x, lane = tid % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int qsub = wave & 1, grp = wave >> 1;  // 32-query half, 32-key half of each tile
  const int c = lane % 32, h = lane / 32;
  const int qrow = qb * kAttnQ + 32 * qsub + c;

  // Q^T operand pieces of step ks: dims (D/2) h + 8 ks .. +7, scaled.
  u32x4 qreg[KS][3];
  uint32_t lost = 0;
  {
    const float* qp = a.q + b * a.qs[0] + hd * a.qs[1] + long(min(qrow, a.n - 1)) * a.qs[2] + (D / 2) * h;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      uint32_t x[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) x[e] = __float_as_uint(qp[8 * ks + e] * a.scale_log2);
      split3(make_uint4(x[0], x[1], x[2], x[3]), make_uint4(x[4], x[5], x[6], x[7]), qreg[ks], lost);
    }
  }
  const float* kb = a.k + b * a.ks[0] + hd * a.ks[1];
  const float* vb = a.v + b * a.vs[0] + hd * a.vs[1];
  uint4 kr[NLD][2], vr[NLD][2];
  auto load = [&](int t) {
#pragma unroll
    for (int i = 0; i < NLD; ++i) {
      const int idx = min(tid + i * kF32Threads, kAttnK * SL - 1);
      const long key = min(t * kAttnK + idx / SL, a.n - 1);
      const float* kp = kb + key * a.ks[2] + 8 * (idx % SL);
      const float* vp = vb + key * a.vs[2] + 8 * (idx % SL);
      kr[i][0] = load16(kp);
      kr[i][1] = load16(kp + 4);
      vr[i][0] = load16(vp);
      vr[i][1] = load16(vp + 4);
    }
  };
  unsigned vlane[DT];
#pragma unroll
  for (int t = 0; t < DT; ++t) vlane[t] = vt_lane_offset<DL>(lane, t) + unsigned(grp) * 32u * 2u * DL;

  float m_run = -INFINITY, l_run = 0.f;
  // The products beside p0 p0 of one dim tile: a running sum of their own, or,
  // of several dim tiles, one per step (registers).
  constexpr bool kLowKept = DT == 1;
  f32x16 o[DT], o_low, zero;
#pragma unroll
  for (int j = 0; j < 16; ++j) o_low[j] = zero[j] = 0.f;
#pragma unroll
  for (int t = 0; t < DT; ++t)
#pragma unroll
    for (int j = 0; j < 16; ++j) o[t][j] = 0.f;
  load(0);
  for (int t = 0; t <= qb; ++t) {
    __syncthreads();  // the previous tile is no longer read
#pragma unroll
    for (int i = 0; i < NLD; ++i) {
      const int idx = tid + i * kF32Threads;
      if (kAttnK * SL % kF32Threads == 0 || idx < kAttnK * SL) {
        const int r = idx / SL, s = idx % SL;
        u32x4 pk[3], pv[3];
        split3(kr[i][0], kr[i][1], pk, lost);
        split3(vr[i][0], vr[i][1], pv, lost);
#pragma unroll
        for (int p = 0; p < 3; ++p) {
          st.k[p][r][s ^ k_swizzle<DL>(r)] = make_uint4(pk[p][0], pk[p][1], pk[p][2], pk[p][3]);
          st.v[p][r][vt_slot(s, r)] = make_uint4(pv[p][0], pv[p][1], pv[p][2], pv[p][3]);
        }
      }
    }
    __syncthreads();
    if (t < qb) load(t + 1);
    if (t == qb && grp > qsub) continue;  // keys above every query of the wave
    f32x16 s, s_low;
#pragma unroll
    for (int j = 0; j < 16; ++j) s[j] = s_low[j] = 0.f;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      u32x4 kp[3];
#pragma unroll
      for (int p = 0; p < 3; ++p) {
        const uint4 r = st.k[p][32 * grp + c][(KS * h + ks) ^ k_swizzle<DL>(c)];
        kp[p] = u32x4{r.x, r.y, r.z, r.w};
      }
#pragma unroll
      for (int p = 0; p < kLowProducts; ++p) s_low = mfma32<bf16_t>(kp[kLowA[p]], qreg[ks][kLowB[p]], s_low);
      s = mfma32<bf16_t>(kp[0], qreg[ks][0], s);
    }
    s += s_low;
    if (t == qb && grp == qsub) {  // the diagonal block (attention.py:187-197)
#pragma unroll
      for (int j = 0; j < 16; ++j) s[j] = 8 * (j / 4) + 4 * h + j % 4 <= c ? s[j] : -INFINITY;
    }
    float mx = s[0];
#pragma unroll
    for (int j = 1; j < 16; ++j) mx = fmaxf(mx, s[j]);
    mx = fmaxf(mx, lane_xor(mx, 32));
    const float m_new = fmaxf(m_run, mx);
    const float alpha = __builtin_amdgcn_exp2f(m_run - m_new);
    m_run = m_new;
    float sum = 0.f;
#pragma unroll
    for (int j = 0; j < 16; ++j) {
      s[j] = __builtin_amdgcn_exp2f(s[j] - m_new);
      sum += s[j];
    }
    l_run = l_run * alpha + sum;
    if (__ballot(alpha != 1.f)) {
#pragma unroll
      for (int d = 0; d < DT; ++d) o[d] *= alpha;
      if (kLowKept) o_low *= alpha;
    }
#pragma unroll
    for (int s2 = 0; s2 < 2; ++s2) {
      uint32_t x[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) x[e] = __float_as_uint(s[8 * s2 + e]);
      u32x4 pp[3];
      uint32_t below = 0;  // of a probability, only what is under 2^-133 of the row's largest
      split3(make_uint4(x[0], x[1], x[2], x[3]), make_uint4(x[4], x[5], x[6], x[7]), pp, below);
#pragma unroll
      for (int d = 0; d < DT; ++d) {
        u32x4 vp[3];
#pragma unroll
        for (int p = 0; p < 3; ++p) {
          const unsigned off = lds_offset(&st.v[p][0][0]) + vlane[d] + 32u * DL * s2;
          const i16x4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4_t*)(size_t)(off));
          const i16x4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4_t*)(size_t)(off + 16u * DL));
          const uint2 l2 = __builtin_bit_cast(uint2, lo), h2 = __builtin_bit_cast(uint2, hi);
          vp[p] = u32x4{l2.x, l2.y, h2.x, h2.y};
        }
#pragma unroll
        for (int p = 0; p < kLowProducts; ++p)
          o_low = mfma32<bf16_t>(vp[kLowA[p]], pp[kLowB[p]], kLowKept || p ? o_low : zero);
        o[d] = mfma32<bf16_t>(vp[0], pp[0], o[d]);
        if (!kLowKept) o[d] += o_low;
      }
    }
  }

  // Waves 2 and 3 hand their half of each row to waves 0 and 1.
  l_run += lane_xor(l_run, 32);
  if (kLowKept) o[0] += o_low;
  float* const red = reinterpret_cast<float*>(&st) + (qsub * (16 * DT + 2)) * kWave + lane;
  __syncthreads();
  if (grp == 1) {
#pragma unroll
    for (int d = 0; d < DT; ++d)
#pragma unroll
      for (int j = 0; j < 16; ++j) red[(16 * d + j) * kWave] = o[d][j];
    red[16 * DT * kWave] = m_run;
    red[(16 * DT + 1) * kWave] = l_run;
  }
  __syncthreads();
  bool redo = (lost & 0xffffu) != 0;
  if (grp == 0) {
    const float m1 = red[16 * DT * kWave], l1 = red[(16 * DT + 1) * kWave];
    const float top = fmaxf(m_run, m1);
    const float w0 = __builtin_amdgcn_exp2f(m_run - top), w1 = __builtin_amdgcn_exp2f(m1 - top);
    const float inv = 1.f / (l_run * w0 + l1 * w1);  // key 0 is always admissible: the sum is at least 1
#pragma unroll
    for (int d = 0; d < DT; ++d)
#pragma unroll
      for (int j = 0; j < 16; ++j) {
        o[d][j] = (o[d][j] * w0 + red[(16 * d + j) * kWave] * w1) * inv;
        if (D >= 32 || j < 8) redo |= qrow < a.n && o[d][j] != o[d][j];
      }
  }
  if (__syncthreads_or(redo)) return causal_rows_valu<D>(a, qb, b, hd, reinterpret_cast<float*>(&st));
  if (grp == 1 || qrow >= a.n) return;
  float* op = a.o + b * a.os[0] + hd * a.os[1] + long(qrow) * a.os[2];
#pragma unroll
  for (int d = 0; d < DT; ++d)
#pragma unroll
    for (int q = 0; q < (D < 32 ? 2 : 4); ++q)
      *reinterpret_cast<float4*>(op + 32 * d + 8 * q + 4 * h) =
          make_float4(o[d][4 * q], o[d][4 * q + 1], o[d][4 * q + 2], o[d][4 * q + 3]);
}

template <int E, int TBN, int TBM, int KS, int NW, int NS>
int launch_tile(const F32GemmArgs& g, hipStream_t s, const char* what) {
  const long tiles = long((g.n + TBN - 1) / TBN) * ((g.m + TBM - 1) / TBM);
  if (tiles > (1L << 31) - 1) return set_error(SFL_ERR_UNSUPPORTED, "%s: too many tiles", what);
  hipLaunchKernelGGL((gemm_split_kernel<float, E, TBN, TBM, KS, NW, NS>), dim3(unsigned(tiles)), dim3(NW * kWave), 0,
                     s, g);
  return check_launch(what);
}

// Tile of an fp32 GEMM. 32 x 32 runs two workgroups per CU, and while that
// covers the grid no larger tile is faster; 64 x 64 on 8 waves fills a CU
// alone; beyond, 64 x 64 (two per CU) or 64 x 32 (three), whichever leaves the
// fullest CU less to do (a 64 x 32 tile costs 1.12 halves of a 64 x 64 one).
// us, gemm_f32_kernel -> this: M 1000 N 512 K 512 18.0 -> 8.7 (32 x 32);
// M 2048 N 512 K 1344 61 -> 25 (64 x 64, 8 waves); M 1000 N 2304 K 768
// 56 -> 37 (64 x 32); M 4000 N 2304 K 768 155 -> 111, M 12000 N 4096 K 768
// 730 -> 559 (64 x 64: 135 TFLOP/s). Relative error to float64 (2-norm) at
// K 64 / 512 / 768 / 2752: 1.5 / 4.1 / 5.0 / 9.4e-7 -> 0.5 / 0.8 / 0.9 / 1.5e-7;
// of a row with one non-zero value, 2.5e-8 rms and 6.0e-8 at most either way.
template <int E>
int launch_split(const F32GemmArgs& g, hipStream_t s, const char* what) {
  constexpr long kCus = 256;
  const auto count = [&](long tn, long tm) { return ((g.n + tn - 1) / tn) * ((g.m + tm - 1) / tm); };
  if (count(32, 32) <= 2 * kCus) return launch_tile<E, 32, 32, 32, 4, 2>(g, s, what);
  const long t64 = count(64, 64);
  if (t64 <= kCus) return launch_tile<E, 64, 64, 16, 8, 1>(g, s, what);
  const double most64 = 2. * double((t64 + kCus - 1) / kCus);
  const double most32 = 1.12 * double((count(64, 32) + kCus - 1) / kCus);
  if (most32 < most64) return launch_tile<E, 64, 32, 16, 4, 2>(g, s, what);
  return launch_tile<E, 64, 64, 16, 4, 2>(g, s, what);
}

}  // namespace

int launch_gemm_f32(const F32GemmArgs& g, int epi, hipStream_t stream, const char* what) {
  if (g.m < 1 || g.n < 1 || g.k < 1) return set_error(SFL_ERR_INVALID, "%s: sizes must be positive", what);
  if (g.k % 4) return set_error(SFL_ERR_UNSUPPORTED, "%s: fp32 K must be a multiple of 4", what);
  const auto a16 = [](const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; };
  if (!a16(g.a) || !a16(g.w))
    return set_error(SFL_ERR_INVALID, "%s: fp32 operands must be 16-byte aligned", what);
  // 32-bit byte offsets and whole 128-byte K chunks: the split kernel.
  if (g.k % 32 == 0 && long(g.m) * g.k < (1L << 29) && long(g.n) * g.k < (1L << 29)) {
    switch (epi) {
      case F32_QKV: return launch_split<F32_QKV>(g, stream, what);
      case F32_SWIGLU: return launch_split<F32_SWIGLU>(g, stream, what);
      default: return launch_split<F32_PLAIN>(g, stream, what);
    }
  }
  const dim3 grid(unsigned((g.n + FT - 1) / FT), unsigned((g.m + FT - 1) / FT));
  if (grid.y > 65535) return set_error(SFL_ERR_UNSUPPORTED, "%s: M too large", what);
  switch (epi) {
    case F32_QKV: hipLaunchKernelGGL(gemm_f32_kernel<F32_QKV>, grid, dim3(kF32Threads), 0, stream, g); break;
    case F32_SWIGLU: hipLaunchKernelGGL(gemm_f32_kernel<F32_SWIGLU>, grid, dim3(kF32Threads), 0, stream, g); break;
    default: hipLaunchKernelGGL(gemm_f32_kernel<F32_PLAIN>, grid, dim3(kF32Threads), 0, stream, g); break;
  }
  return check_launch(what);
}

}  // namespace sfl

using namespace sfl;

extern "C" int sfl_causal_attention_f32(const float* q, const float* k, const float* v, float* o, int batch,
                                        int heads, int n, int head_dim, const long* q_strides,
                                        const long* k_strides, const long* v_strides, const long* o_strides,
                                        float scale, void* stream) {
  const char* what = "causal_attention_f32";
  if (!q || !k || !v || !o || !q_strides || !k_strides || !v_strides || !o_strides)
    return set_error(SFL_ERR_INVALID, "%s: null pointer argument", what);
  if (batch < 1 || heads < 1 || n < 1) return set_error(SFL_ERR_INVALID, "%s: sizes must be positive", what);
  if (!(scale > 0.f) || !__builtin_isfinite(scale))
    return set_error(SFL_ERR_INVALID, "%s: scale must be finite and positive", what);
  for (int i = 0; i < 3; ++i)
    if (q_strides[i] < 0 || k_strides[i] < 0 || v_strides[i] < 0 || o_strides[i] < 0)
      return set_error(SFL_ERR_INVALID, "%s: strides must be non-negative", what);
  const auto a16 = [](const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; };
  bool aligned = a16(k) && a16(v) && a16(o);
  for (int i = 0; i < 3; ++i) aligned = aligned && k_strides[i] % 4 == 0 && v_strides[i] % 4 == 0 && o_strides[i] % 4 == 0;
  if (!aligned) return set_error(SFL_ERR_INVALID, "%s: k, v and o rows must be 16-byte aligned", what);
  if (long((n + kAttnQ - 1) / kAttnQ) * batch * heads > (1L << 31) - 1)
    return set_error(SFL_ERR_UNSUPPORTED, "%s: too many query blocks", what);
  F32AttnArgs a{};
  a.q = q; a.k = k; a.v = v; a.o = o;
  for (int i = 0; i < 3; ++i) {
    a.qs[i] = q_strides[i]; a.ks[i] = k_strides[i]; a.vs[i] = v_strides[i]; a.os[i] = o_strides[i];
  }
  a.batch = batch; a.heads = heads; a.n = n; a.scale_log2 = scale * kLog2e;
  const dim3 grid(unsigned((n + kAttnQ - 1) / kAttnQ) * unsigned(batch * heads));
  const hipStream_t s = static_cast<hipStream_t>(stream);
  switch (head_dim) {
    case 16: hipLaunchKernelGGL(causal_attention_f32_kernel<16>, grid, dim3(kF32Threads), 0, s, a); break;
    case 32: hipLaunchKernelGGL(causal_attention_f32_kernel<32>, grid, dim3(kF32Threads), 0, s, a); break;
    case 64: hipLaunchKernelGGL(causal_attention_f32_kernel<64>, grid, dim3(kF32Threads), 0, s, a); break;
    case 128: hipLaunchKernelGGL(causal_attention_f32_kernel<128>, grid, dim3(kF32Threads), 0, s, a); break;
    default: return set_error(SFL_ERR_UNSUPPORTED, "%s: head dim must be 16, 32, 64 or 128", what);
  }
  return check_launch(what);
}
