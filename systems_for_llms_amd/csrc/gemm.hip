// Prefill projections as 16-bit MFMA GEMMs with fused epilogues, plus the
// row-wise prefill helpers (embedding gather, RMSNorm).
//
// Every GEMM computes C^T[n][m] = sum_k W[n][k] * A[m][k] for A [M, K]
// activations (one row per token) and W [N, K] weights, both K-contiguous as
// the reference's Linear stores them (src/llmlab/model/layers.py:34-35), in
// the model's 16-bit type T (bf16 or fp16; the kernels are templates on T,
// whose 16-bit outputs are stored in T too).
// Features are the MFMA rows, so each lane ends with 4 consecutive features
// of one token: RoPE pairs and SwiGLU pairs are in-lane or one shuffle away
// and stores are 8/16-byte vectors.
//
// Tiling: a workgroup of 4 waves computes a 128-feature x 128-token tile;
// wave (wn, wm) owns 64 x 64 = 4 x 4 MFMA tiles of 16x16x32. K advances in
// steps of 64 through double-buffered LDS tiles (rows padded by 8 elements);
// the next step's global loads are in registers while the current step runs.
// Epilogues:
//   PLAIN     C[m][n] stored as fp32 or bf16 (optionally accumulated into fp32).
//   QKV       RoPE on q and k (attention.py:44-58) from the host fp32 table at
//             position m % T, q to [B, H, T, dk] bf16, k/v to the KV cache.
//   SWIGLU    W is W1/W3 interleaved in blocks of 8 rows; h = silu(a) * c
//             (layers.py:114-115) as bf16 [M, d_ff].
#include <algorithm>
#include <initializer_list>

#include "gemm16.hpp"
#include "gemm_f32.hpp"

namespace sfl {
namespace {

constexpr int TN = 128, TM = 128, TK = 64;
constexpr int LDT = TK + 8;      // LDS row stride (elements)
constexpr int kThreads = 256;

template <typename T, int E>
__global__ __launch_bounds__(kThreads) void gemm_kernel(GemmArgs g) {
  __shared__ __align__(16) uint16_t ws[2][TN * LDT];
  __shared__ __align__(16) uint16_t as[2][TM * LDT];
  const int tid = threadIdx.x;
  const int wave = tid / kWave, lane = tid % kWave;
  const int wn = wave / 2, wm = wave % 2;
  const int col = lane % 16, grp = lane / 16;
  const int n0 = blockIdx.x * TN;
  const int m0 = blockIdx.y * TM;
  const int ksteps = (g.k + TK - 1) / TK;

  // Each thread moves 4 x 16 bytes of W and of A per K step: row r, 8-element
  // group cg. Loads are unconditional from clamped addresses; the K tail is
  // zeroed when the registers go to LDS, so no load waits inside its guard.
  uint4 wr[4], ar[4];
  bool kin[4];
#define SFL_GEMM_GLOAD(kt)                                                   \
  _Pragma("unroll") for (int i = 0; i < 4; ++i) {                            \
    const int idx = tid + i * kThreads;                                      \
    const int r = idx / (TK / 8), cg = idx % (TK / 8);                       \
    const int kk = (kt) * TK + cg * 8;                                       \
    kin[i] = kk < g.k;                                                       \
    const int kc = kin[i] ? kk : 0;                                          \
    wr[i] = load16(g.w + long(min(n0 + r, g.n - 1)) * g.k + kc);             \
    ar[i] = load16(g.a + long(min(m0 + r, g.m - 1)) * g.k + kc);             \
  }
#define SFL_GEMM_SSTORE(buf)                                                 \
  _Pragma("unroll") for (int i = 0; i < 4; ++i) {                            \
    const int idx = tid + i * kThreads;                                      \
    const int r = idx / (TK / 8), cg = idx % (TK / 8);                       \
    *reinterpret_cast<uint4*>(&ws[buf][r * LDT + cg * 8]) = keep16(wr[i], kin[i]); \
    *reinterpret_cast<uint4*>(&as[buf][r * LDT + cg * 8]) = keep16(ar[i], kin[i]); \
  }

  f32x4 acc[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  SFL_GEMM_GLOAD(0)
  SFL_GEMM_SSTORE(0)
  __syncthreads();
  for (int kt = 0; kt < ksteps; ++kt) {
    const int buf = kt & 1;
    if (kt + 1 < ksteps) { SFL_GEMM_GLOAD(kt + 1) }
#pragma unroll
    for (int ks = 0; ks < TK / 32; ++ks) {
      u32x4 af[4], bfr[4];
#pragma unroll
      for (int i = 0; i < 4; ++i)
        af[i] = *reinterpret_cast<const u32x4*>(&ws[buf][(wn * 64 + i * 16 + col) * LDT + ks * 32 + grp * 8]);
#pragma unroll
      for (int j = 0; j < 4; ++j)
        bfr[j] = *reinterpret_cast<const u32x4*>(&as[buf][(wm * 64 + j * 16 + col) * LDT + ks * 32 + grp * 8]);
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = mfma16<T>(af[i], bfr[j], acc[i][j]);
    }
    if (kt + 1 < ksteps) {
      SFL_GEMM_SSTORE(buf ^ 1)
      __syncthreads();
    }
  }
#undef SFL_GEMM_GLOAD
#undef SFL_GEMM_SSTORE

  // Epilogue: acc[i][j] holds features n0 + wn*64 + 16i + 4grp + (0..3) of token m0 + wm*64 + 16j + col.
  QkvTok tok[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) tok[j] = E == G_QKV ? qkv_tok(g, m0 + wm * 64 + j * 16 + col) : QkvTok{};
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const QkvFeat feat = E == G_QKV ? qkv_feat(g, n0 + wn * 64 + i * 16 + 4 * grp) : QkvFeat{};
#pragma unroll
    for (int j = 0; j < 4; ++j)
      store_tile<T, E>(g, acc[i][j], n0 + wn * 64 + i * 16, grp, m0 + wm * 64 + j * 16 + col, feat, tok[j]);
  }
}

// GEMM for K % 64 == 0 on v_mfma_f32_32x32x16_{bf16,f16} (on gfx950 the 32x32
// form sustains about twice the bf16 rate of the 16x16x32 form used above).
// A workgroup of 4 waves (2 x 2) computes 128 features x 128 tokens; wave
// (wn, wm) owns 2 x 2 MFMA tiles of 32x32. Operands reach LDS through buffer
// loads with an LDS destination (no register staging). A K step stores each
// operand tile row-major, 128 bytes (64 k values) per row in 8 slots of 16
// bytes, slot = (16-byte column) ^ ((row >> 1) & 7): a load instruction moves
// 8 whole rows (1 KB, full cache lines, the lanes of a row in swizzled order)
// and every MFMA operand read -- 32 rows x 2 columns per instruction -- is
// free of bank conflicts. Rows past the matrix read as zeros through the
// buffer range check. K advances by 64 through two LDS stages, the loads of
// the next step in flight while a step computes.
// TBN x TBM tiles (features x tokens) per workgroup of WN x WM waves; a wave
// owns (TBN/WN) x (TBM/WM) as blocks of 32 x 32. 128 x 128 with 2 x 2 waves:
// two workgroups per CU (64 KB of LDS each), 64 x 64 per wave. 256 x 384 with
// 4 x 2 waves: one workgroup of 8 waves per CU using all 160 KB of LDS (two
// stages of 80 KB), 64 x 192 per wave (12 accumulator blocks, ~236 VGPRs, no
// spills); per MFMA it stages 5/8 of the bytes of the 128 x 128 tile through
// LDS and reads 2/3 of its LDS operand bytes.
template <typename T, int E, int TBN, int TBM, int WN, int WM, int KS, int NS>
__global__ __launch_bounds__(64 * WN * WM) __attribute__((amdgpu_waves_per_eu(2)))
void gemm32_kernel(GemmArgs g) {
  constexpr int NW = WN * WM;              // waves
  constexpr int NBN = TBN / WN / 32;       // 32x32 blocks per wave along features
  constexpr int NBM = TBM / WM / 32;       // and along tokens
  constexpr int SL = KS / 8;               // 16-byte slots per row of a stage
  constexpr int RPL = kWave / SL;          // rows one 1 KB load instruction moves
  // NS LDS stages of KS k values each; see lds_load16 for why the loads are
  // counted by hand.
  __shared__ Stage32<TBN, TBM, SL> st[NS];
  const int tid = threadIdx.x;
  // readfirstlane: the wave index is uniform, so the LDS destinations live in scalar registers.
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave), lane = tid % kWave;
  const int wn = wave / WM, wm = wave % WM;
  const int l32 = lane % 32, hf = lane / 32;
  const int2 tile = xcd_tile(blockIdx.x, (g.n + TBN - 1) / TBN, (g.m + TBM - 1) / TBM);
  const int n0 = tile.x * TBN;
  const int m0 = tile.y * TBM;
  const int ksteps = g.k / KS;

  // Loads: the TBN + TBM rows of a step are chunks of RPL rows; wave w takes
  // chunks w, w + NW, ... Lane i of a chunk moves row RPL c + i/SL into slot
  // i%SL, i.e. column (i%SL) ^ stage_swizzle(row); the swizzle depends on the
  // chunk's parity at most, so two byte offsets per lane cover every chunk.
  const i32x4_t rw = buffer_rsrc(g.w, unsigned(g.n * g.k * 2));
  const i32x4_t ra = buffer_rsrc(g.a, unsigned(g.m * g.k * 2));
  const int rr = lane / SL, pos = lane % SL;
  unsigned voff[2];
#pragma unroll
  for (int par = 0; par < 2; ++par)
    voff[par] = unsigned((rr * g.k + 8 * (pos ^ stage_swizzle<SL>(RPL * par + rr))) * 2);
  constexpr int CHN = TBN / RPL, CHM = TBM / RPL;  // chunks per operand
  constexpr int CPW = (CHN + CHM) / NW;            // load instructions per wave and stage
  static_assert((CHN + CHM) % NW == 0 && CHN % 2 == 0, "chunks per wave");

#define SFL_G32_ISSUE(stage, kt)                                                            \
  {                                                                                         \
    _Pragma("unroll") for (int c0 = 0; c0 < CHN + CHM; c0 += NW) {                          \
      const int c = c0 + wave;                                                              \
      if (c < CHN)                                                                          \
        lds_load16(rw, lds_offset(&stage.w[RPL * c][0]), voff[c & 1],                       \
                   unsigned(((n0 + RPL * c) * g.k + (kt) * KS) * 2));                       \
      else                                                                                  \
        lds_load16(ra, lds_offset(&stage.a[RPL * (c - CHN)][0]), voff[(c - CHN) & 1],       \
                   unsigned(((m0 + RPL * (c - CHN)) * g.k + (kt) * KS) * 2));               \
    }                                                                                       \
  }
  // Operand reads: lane (l32, hf) takes row 32t + l32, column 2kk + hf.
  const int sw = stage_swizzle<SL>(l32);
#define SFL_G32_COMPUTE(stage)                                                              \
  _Pragma("unroll") for (int kk = 0; kk < KS / 16; ++kk) {                                  \
    const int slot = (2 * kk + hf) ^ sw;                                                    \
    u32x4 af[NBN], bfr[NBM];                                                                \
    _Pragma("unroll") for (int t = 0; t < NBN; ++t) {                                       \
      const uint4 ra_ = stage.w[32 * (NBN * wn + t) + l32][slot];                           \
      af[t] = u32x4{ra_.x, ra_.y, ra_.z, ra_.w};                                            \
    }                                                                                       \
    _Pragma("unroll") for (int t = 0; t < NBM; ++t) {                                       \
      const uint4 rb_ = stage.a[32 * (NBM * wm + t) + l32][slot];                           \
      bfr[t] = u32x4{rb_.x, rb_.y, rb_.z, rb_.w};                                           \
    }                                                                                       \
    _Pragma("unroll") for (int i = 0; i < NBN; ++i)                                         \
      _Pragma("unroll") for (int j = 0; j < NBM; ++j) acc[i][j] = mfma32<T>(af[i], bfr[j], acc[i][j]); \
  }

  f32x16 acc[NBN][NBM];
#pragma unroll
  for (int i = 0; i < NBN; ++i)
#pragma unroll
    for (int j = 0; j < NBM; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;
  // Residual accumulation into fp32 C (x += A W^T): the accumulators start
  // from the old C values, loaded now, while the first stages are in flight,
  // so the epilogue only stores. (Unconditional loads from clamped addresses;
  // the values of rows / columns past C are never stored.)
  const bool acc_c = E == G_PLAIN && g.c_f32 && g.accumulate && (g.n & 3) == 0;
  if constexpr (E == G_PLAIN) {
    if (acc_c) {
      const float* c = static_cast<const float*>(g.c);
#pragma unroll
      for (int j = 0; j < NBM; ++j) {
        const long mr = min(m0 + (TBM / WM) * wm + 32 * j + l32, g.m - 1);
#pragma unroll
        for (int i = 0; i < NBN; ++i) {
          const int nt = n0 + (TBN / WN) * wn + 32 * i;
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const float4 o = *reinterpret_cast<const float4*>(c + mr * g.n + min(nt + 8 * q + 4 * hf, g.n - 4));
            acc[i][j][4 * q] = o.x;
            acc[i][j][4 * q + 1] = o.y;
            acc[i][j][4 * q + 2] = o.z;
            acc[i][j][4 * q + 3] = o.w;
          }
        }
      }
    }
  }

  // Row scales of the normalized input (q/k/v, SwiGLU), loaded while the
  // first stages are in flight.
  float rsc[NBM];
#pragma unroll
  for (int j = 0; j < NBM; ++j) rsc[j] = 1.f;
  if constexpr (E != G_PLAIN) {
    if (g.row_scale) {
#pragma unroll
      for (int j = 0; j < NBM; ++j) rsc[j] = g.row_scale[min(m0 + (TBM / WM) * wm + 32 * j + l32, g.m - 1)];
    }
  }

  // NS LDS stages in a ring: step kt computes from stage kt % NS while the
  // loads of the next NS - 1 steps are in flight. At step kt the wave waits
  // only for stage kt's loads (the younger stages' CPW each may stay
  // outstanding), the barrier then covers every wave's share, and stage
  // (kt - 1) % NS, last read before that barrier, is refilled with step
  // kt + NS - 1. One loop body, so every accumulator keeps its registers.
#pragma unroll
  for (int p = 0; p < NS - 1; ++p)
    if (p < ksteps) SFL_G32_ISSUE(st[p], p)
  if constexpr (E != G_PLAIN) {
    if (g.ss) {
#pragma unroll
      for (int j = 0; j < NBM; ++j) rsc[j] = parts_scale(g, min(m0 + (TBM / WM) * wm + 32 * j + l32, g.m - 1));
    }
  }
  for (int kt = 0; kt < ksteps; ++kt) {
    wait_younger<NS - 2, CPW>(min(NS - 2, ksteps - 1 - kt));  // stages issued after stage kt
    __syncthreads();  // every wave's loads of this stage landed; stage (kt - 1) % NS is no longer read
    if (kt + NS - 1 < ksteps) SFL_G32_ISSUE(st[(kt + NS - 1) % NS], kt + NS - 1)
    SFL_G32_COMPUTE(st[kt % NS])
  }
#undef SFL_G32_COMPUTE
#undef SFL_G32_ISSUE

  if constexpr (E == G_PLAIN) {
    if (acc_c) {
      const bool norm = g.norm_gain != nullptr;  // uniform
      // The next norm's gains for this lane's features (one batch of loads,
      // before any store).
      uint2 gw[NBN][4];
      if (norm) {
#pragma unroll
        for (int i = 0; i < NBN; ++i)
#pragma unroll
          for (int q = 0; q < 4; ++q)
            gw[i][q] = *reinterpret_cast<const uint2*>(
                g.norm_gain + min(n0 + (TBN / WN) * wn + 32 * i + 8 * q + 4 * hf, g.n - 4));
      }
      float ssq[NBM];
#pragma unroll
      for (int j = 0; j < NBM; ++j) {
        const int m = m0 + (TBM / WM) * wm + 32 * j + l32;
        ssq[j] = 0.f;
#pragma unroll
        for (int i = 0; i < NBN; ++i)
          residual_block<T>(g, acc[i][j], n0 + (TBN / WN) * wn + 32 * i, m, hf, norm, gw[i], ssq[j]);
      }
      if (norm) {
        // Sum of squares per token over each 128-feature part: this lane's 32
        // features, its partner lane's (l ^ 32: the other 4 of each 8), then
        // the wave pair (wn, wn ^ 1) covering the part, in that order.
        float* const part_s = reinterpret_cast<float*>(&st[0]);  // [WN][TBM] (the stages are free now)
        __syncthreads();  // every wave has read the last stage
#pragma unroll
        for (int j = 0; j < NBM; ++j) {
          const float t = ssq[j] + lane_xor(ssq[j], 32);
          if (hf == 0) part_s[wn * TBM + (TBM / WM) * wm + 32 * j + l32] = t;
        }
        __syncthreads();
        static_assert(TBN / WN == 64, "two waves per 128-feature part");
        const int part = (n0 + (TBN / WN) * wn) / 128;
        if ((wn & 1) == 0 && part * 128 < g.n) {
          for (int r = lane; r < TBM / WM; r += kWave) {
            const int row = (TBM / WM) * wm + r;
            const int m = m0 + row;
            if (m < g.m) g.norm_ss[long(part) * g.m + m] = part_s[wn * TBM + row] + part_s[(wn + 1) * TBM + row];
          }
        }
      }
      return;
    }
  }

  // acc[i][j][4q + e] holds feature n0 + (TBN/WN)wn + 32i + 8q + 4hf + e of
  // token m0 + (TBM/WM)wm + 32j + l32.
#pragma unroll
  for (int j = 0; j < NBM; ++j) {
    const int m = m0 + (TBM / WM) * wm + 32 * j + l32;
    const QkvTok tok = E == G_QKV ? qkv_tok(g, m) : QkvTok{};
#pragma unroll
    for (int i = 0; i < NBN; ++i)
      store_block<T, E>(g, acc[i][j], n0 + (TBN / WN) * wn + 32 * i, m, tok, rsc[j], hf);
  }
}

inline bool aligned16(const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; }

template <typename T, int E>
int launch_gemm_t(const GemmArgs& g, hipStream_t s, const char* what) {
  if (g.m < 1 || g.n < 1 || g.k < 1) return set_error(SFL_ERR_INVALID, "%s: sizes must be positive", what);
  if (g.k % 8) return set_error(SFL_ERR_UNSUPPORTED, "%s: K must be a multiple of 8", what);
  if (g.k % K2 == 0 && long(g.m) * g.k < (1L << 30) && long(g.n) * g.k < (1L << 30)) {
    Tile16 t = tile16_for(g.m, g.n, g.k, E);
    if (t <= S128x64 && g.norm_gain && g.norm_part == 128) t = T128x64;
    if (t <= S128x64) return launch_gemm_small<T, E>(g, t, s, what);
    const int tn = t == T256x384 || t == T256x256 ? 256 : 128;
    const int tm = t == T256x384 ? 384 : t == T256x256 ? 256 : t == T128x128 ? 128 : 64;
    const long tiles = long((g.n + tn - 1) / tn) * ((g.m + tm - 1) / tm);
    if (tiles > (1L << 31) - 1) return set_error(SFL_ERR_UNSUPPORTED, "%s: too many tiles", what);
    const dim3 grid{unsigned(tiles)};
    switch (t) {
      case T256x384: hipLaunchKernelGGL((gemm32_kernel<T, E, 256, 384, 4, 2, 64, 2>), grid, dim3(512), 0, s, g); break;
      case T256x256: hipLaunchKernelGGL((gemm32_kernel<T, E, 256, 256, 4, 2, 64, 2>), grid, dim3(512), 0, s, g); break;
      case T128x128: hipLaunchKernelGGL((gemm32_kernel<T, E, 128, 128, 2, 2, 64, 2>), grid, dim3(256), 0, s, g); break;
      default: hipLaunchKernelGGL((gemm32_kernel<T, E, 128, 64, 2, 2, 64, 2>), grid, dim3(256), 0, s, g); break;
    }
    return check_launch(what);
  }
  dim3 grid((g.n + TN - 1) / TN, (g.m + TM - 1) / TM);
  if (grid.y > 65535) return set_error(SFL_ERR_UNSUPPORTED, "%s: M too large", what);
  hipLaunchKernelGGL((gemm_kernel<T, E>), grid, dim3(kThreads), 0, s, g);
  return check_launch(what);
}

// The GEMMs' 16-bit element type: SFL_DTYPE_BF16 or SFL_DTYPE_F16.
template <int E>
int launch_gemm(const GemmArgs& g, int dtype, hipStream_t s, const char* what) {
  if (dtype == SFL_DTYPE_BF16) return launch_gemm_t<bf16_t, E>(g, s, what);
  if (dtype == SFL_DTYPE_F16) return launch_gemm_t<f16_t, E>(g, s, what);
  return set_error(SFL_ERR_UNSUPPORTED, "%s: dtype must be BF16 or F16", what);
}

// Prefill embedding gather: x[m] = emb[ids[m]] in fp32.
template <typename T>
__global__ __launch_bounds__(256) void embed_rows_kernel(const int64_t* ids, const T* emb, float* x, int d) {
  const long m = blockIdx.x;
  const T* src = emb + ids[m] * d;
  for (int i = threadIdx.x; i < d; i += blockDim.x) x[m * d + i] = load_scalar<T>(src + i);
}

// Prefill RMSNorm: out[m] = O(x[m] / sqrt(mean(x[m]^2) + eps) * w) (layers.py:133-141),
// O the GEMMs' 16-bit type.
template <typename T, typename O>
__global__ __launch_bounds__(256) void rmsnorm_rows_kernel(const float* x, const T* w, O* out, int d) {
  __shared__ float part[4];
  const long m = blockIdx.x;
  const float* xr = x + m * d;
  float ss = 0.f;
  for (int i = threadIdx.x; i < d; i += 256) ss = fmaf(xr[i], xr[i], ss);
  ss = wave_sum(ss);
  if (threadIdx.x % kWave == 0) part[threadIdx.x / kWave] = ss;
  __syncthreads();
  const float total = part[0] + part[1] + part[2] + part[3];
  const float inv = 1.f / sqrtf(total / float(d) + 1e-5f);
  for (int i = threadIdx.x; i < d; i += 256) store_scalar<O>(out + m * d + i, (xr[i] * inv) * load_scalar<T>(w + i));
}

// The same for rows of d % 4 == 0 and d <= 4 * 64 * kNormVec with one wave per
// row: the row is read once with 16-byte loads and kept in registers, the sum
// of squares is a wave reduction (no LDS, no barrier), and each lane stores
// four 16-bit values at a time.
constexpr int kNormVec = 8;
// kScaled: out = O(x * w) and rscale[row] = 1 / rms(x), for a consumer GEMM
// that applies the scale to its products.
template <typename T, typename O, bool kScaled = false>
__global__ __launch_bounds__(256) void rmsnorm_rows_wave_kernel(const float* x, const T* w, O* out, int m,
                                                               int d, float* rscale = nullptr) {
  const long row = long(blockIdx.x) * 4 + threadIdx.x / kWave;
  const int lane = threadIdx.x % kWave;
  if (row >= m) return;
  const float* xr = x + row * d;
  float4 v[kNormVec];
  float ss = 0.f;
#pragma unroll
  for (int j = 0; j < kNormVec; ++j) {
    const int i = 4 * (j * kWave + lane);
    v[j] = i < d ? *reinterpret_cast<const float4*>(xr + i) : make_float4(0.f, 0.f, 0.f, 0.f);
    ss = fmaf(v[j].x, v[j].x, ss);
    ss = fmaf(v[j].y, v[j].y, ss);
    ss = fmaf(v[j].z, v[j].z, ss);
    ss = fmaf(v[j].w, v[j].w, ss);
  }
  const float inv = 1.f / sqrtf(wave_sum(ss) / float(d) + 1e-5f);
  if (kScaled && lane == 0) rscale[row] = inv;
  const float sc = kScaled ? 1.f : inv;
#pragma unroll
  for (int j = 0; j < kNormVec; ++j) {
    const int i = 4 * (j * kWave + lane);
    if (i < d) {
      float y0 = v[j].x, y1 = v[j].y, y2 = v[j].z, y3 = v[j].w;
      if (!kScaled) {
        y0 *= sc; y1 *= sc; y2 *= sc; y3 *= sc;
      }
      y0 *= load_scalar<T>(w + i); y1 *= load_scalar<T>(w + i + 1);
      y2 *= load_scalar<T>(w + i + 2); y3 *= load_scalar<T>(w + i + 3);
      if constexpr (sizeof(O) == 4)
        *reinterpret_cast<float4*>(out + row * d + i) = make_float4(y0, y1, y2, y3);
      else
        *reinterpret_cast<uint2*>(out + row * d + i) = make_uint2(pack2<O>(y0, y1), pack2<O>(y2, y3));
    }
  }
}

// rscale[m] = 1 / sqrt(sum_p ss[p][m] / d + eps): the inverse RMS from the
// per-part sums of squares a residual GEMM left (parts in a fixed order).
__global__ __launch_bounds__(256) void norm_scale_kernel(const float* __restrict__ ss, int parts, int m, int d,
                                                         float* __restrict__ rscale) {
  const long row = long(blockIdx.x) * 256 + threadIdx.x;
  if (row >= m) return;
  float t = 0.f;
  for (int p = 0; p < parts; ++p) t += ss[long(p) * m + row];
  rscale[row] = 1.f / sqrtf(t / float(d) + 1e-5f);
}

}  // namespace

// Which tile a shape runs on. Up to one tile per CU the smallest that still
// gives every workgroup its own CU wins (K-split tiles, gemm_small.hip), except
// that 128 x 64 splits K only from K = 1024 on: below, too few chunks per wave
// repay its reduction (SwiGLU N 2688 K 512 M 512: 7.4 us shared, 8.3 split;
// residual N 1024 K 2752 M 2048: 31.3 shared, 24.3 split). Beyond, the shapes
// differ mostly by how their last round of workgroups fills the chip, so the
// time is estimated from rounds: 128 x 64 runs 3 workgroups per CU, 128 x 128
// two, the larger ones one, and a round costs (in units of a full round of
// 128 x 128, 18-33 us at K = 1024 by epilogue) what the tables below hold,
// measured over N 512..5504, K 512..2752, M 512..49152 with each epilogue.
// Against the former rule (256 x 384 from 320 such tiles on, else 128 x 128),
// same outputs: q/k/v N 2304 K 768 M 2048 19.4 -> 16.0 us, SwiGLU N 5504
// K 1024 M 4096 55.5 -> 45.3, M 4734 62.7 -> 59.3, residual N 1024 K 2752
// M 16384 110 -> 98; M 49152 unchanged (256 x 384).
Tile16 tile16_for(long m, long n, long k, int epi) {
  constexpr long kCus = 256;
  const auto count = [&](long tn, long tm) { return ((n + tn - 1) / tn) * ((m + tm - 1) / tm); };
  if (count(32, 32) <= kCus) return S32x32;
  if (count(64, 32) <= kCus) return S64x32;
  if (count(64, 64) <= kCus) return S64x64;
  if (count(128, 64) <= kCus) return k >= 1024 ? S128x64 : T128x64;
  // Rounds of up to `per` workgroups per CU: whole rounds at part[per - 1]
  // plus the last one by how many per CU it needs; past 3 rounds the
  // workgroups no longer run in step and the fraction counts.
  const auto cost = [&](long tiles, long per, std::initializer_list<double> part) {
    const double full = part.begin()[per - 1];
    const long slots = per * kCus, rem = tiles % slots;
    if (tiles > 3 * slots) return full * (double(tiles) / double(slots) + 0.25);
    return full * double(tiles / slots) + (rem == 0 ? 0. : part.begin()[(rem - 1) / kCus]);
  };
  const double c64 = cost(count(128, 64), 3, {0.58, 0.70, 0.83});
  const double c128 = cost(count(128, 128), 2, {0.72, 1.0});
  const double c256 = cost(count(256, 256), 1, {epi == G_QKV ? 1.8 : 1.6});
  const double c384 = cost(count(256, 384), 1, {epi == G_QKV ? 2.6 : 2.2});
  const double best = std::min(std::min(c64, c128), std::min(c256, c384));
  return best == c384 ? T256x384 : best == c256 ? T256x256 : best == c128 ? T128x128 : T128x64;
}

}  // namespace sfl

using namespace sfl;

// The GEMMs' 16-bit element type (A, W and 16-bit outputs).
static bool gemm_dtype_ok(int dtype) { return dtype == SFL_DTYPE_BF16 || dtype == SFL_DTYPE_F16; }

extern "C" int sfl_gemm(const void* a, const void* w, void* c, int m, int n, int k, int dtype, int c_dtype,
                        int accumulate, void* stream) {
  const char* what = "gemm";
  if (!a || !w || !c) return set_error(SFL_ERR_INVALID, "%s: null pointer argument", what);
  if (dtype == SFL_DTYPE_F32) {  // the fp32 MFMA GEMM (prefill_f32.hip)
    if (c_dtype != SFL_DTYPE_F32) return set_error(SFL_ERR_UNSUPPORTED, "%s: F32 inputs need an F32 output", what);
    F32GemmArgs f{};
    f.a = static_cast<const float*>(a); f.w = static_cast<const float*>(w);
    f.m = m; f.n = n; f.k = k; f.c = static_cast<float*>(c); f.accumulate = accumulate;
    return launch_gemm_f32(f, F32_PLAIN, static_cast<hipStream_t>(stream), what);
  }
  if (!gemm_dtype_ok(dtype)) return set_error(SFL_ERR_UNSUPPORTED, "%s: dtype must be F32, BF16 or F16", what);
  if (c_dtype != SFL_DTYPE_F32 && c_dtype != dtype)
    return set_error(SFL_ERR_UNSUPPORTED, "%s: output dtype must be F32 or the input dtype", what);
  if (accumulate && c_dtype != SFL_DTYPE_F32)
    return set_error(SFL_ERR_UNSUPPORTED, "%s: accumulation needs an F32 output", what);
  GemmArgs g{};
  g.a = static_cast<const uint16_t*>(a); g.w = static_cast<const uint16_t*>(w);
  g.m = m; g.n = n; g.k = k; g.c = c; g.c_f32 = c_dtype == SFL_DTYPE_F32; g.accumulate = accumulate;
  g.vec16 = aligned16(c);
  return launch_gemm<G_PLAIN>(g, dtype, static_cast<hipStream_t>(stream), what);
}

extern "C" int sfl_gemm_qkv_rope(const void* a, const void* w_qkv, int m, int seq, int d_model, int heads,
                                 const float* cos_t, const float* sin_t, void* q_out, void* k_cache,
                                 void* v_cache, int capacity, int dtype, void* stream) {
  const char* what = "gemm_qkv_rope";
  if (!a || !w_qkv || !cos_t || !sin_t || !q_out || !k_cache || !v_cache)
    return set_error(SFL_ERR_INVALID, "%s: null pointer argument", what);
  if (seq < 1 || m % seq) return set_error(SFL_ERR_INVALID, "%s: rows must be batch * seq", what);
  if (heads < 1 || d_model % heads || (d_model / heads) % 16)
    return set_error(SFL_ERR_UNSUPPORTED, "%s: head dim must be a multiple of 16", what);
  if (seq > capacity) return set_error(SFL_ERR_INVALID, "%s: seq exceeds the cache capacity", what);
  if (dtype == SFL_DTYPE_F32) {
    if (!aligned16(q_out) || !aligned16(k_cache) || !aligned16(v_cache))
      return set_error(SFL_ERR_INVALID, "%s: fp32 q and caches must be 16-byte aligned", what);
    F32GemmArgs f{};
    f.a = static_cast<const float*>(a); f.w = static_cast<const float*>(w_qkv);
    f.m = m; f.n = 3 * d_model; f.k = d_model;
    f.cos_t = cos_t; f.sin_t = sin_t; f.seq = seq; f.heads = heads; f.head_dim = d_model / heads;
    f.d_model = d_model; f.cap = capacity;
    f.q_out = static_cast<float*>(q_out); f.k_cache = static_cast<float*>(k_cache);
    f.v_cache = static_cast<float*>(v_cache);
    return launch_gemm_f32(f, F32_QKV, static_cast<hipStream_t>(stream), what);
  }
  GemmArgs g{};
  g.a = static_cast<const uint16_t*>(a); g.w = static_cast<const uint16_t*>(w_qkv);
  g.m = m; g.n = 3 * d_model; g.k = d_model;
  g.cos_t = cos_t; g.sin_t = sin_t; g.seq = seq; g.heads = heads; g.head_dim = d_model / heads;
  g.d_model = d_model; g.cap = capacity;
  g.q_out = static_cast<uint16_t*>(q_out); g.k_cache = static_cast<uint16_t*>(k_cache);
  g.v_cache = static_cast<uint16_t*>(v_cache);
  g.vec16 = aligned16(q_out) && aligned16(k_cache) && aligned16(v_cache);
  return launch_gemm<G_QKV>(g, dtype, static_cast<hipStream_t>(stream), what);
}

// The fused-norm entry points need the 32x32 kernels (K % 64 == 0, 32-bit offsets).
static bool gemm32_path(int m, int n, int k) {
  return k % K2 == 0 && long(m) * k < (1L << 30) && long(n) * k < (1L << 30);
}

// q/k/v of a normalized input scaled by rscale[r], or by the ss_parts sums of squares ss.
static int gemm_qkv_normed(const char* what, const void* a_xg, const void* w_qkv, const float* rscale,
                           const float* ss, int ss_parts, int m, int seq, int d_model, int heads,
                           const float* cos_t, const float* sin_t, void* q_out, void* k_cache, void* v_cache,
                           int capacity, int dtype, void* stream) {
  if (!gemm32_path(m, 3 * d_model, d_model))
    return set_error(SFL_ERR_UNSUPPORTED, "%s: d_model must be a multiple of %d", what, K2);
  if (!a_xg || !w_qkv || !cos_t || !sin_t || !q_out || !k_cache || !v_cache)
    return set_error(SFL_ERR_INVALID, "%s: null pointer argument", what);
  if (seq < 1 || m % seq) return set_error(SFL_ERR_INVALID, "%s: rows must be batch * seq", what);
  if (heads < 1 || d_model % heads || (d_model / heads) % 16)
    return set_error(SFL_ERR_UNSUPPORTED, "%s: head dim must be a multiple of 16", what);
  if (seq > capacity) return set_error(SFL_ERR_INVALID, "%s: seq exceeds the cache capacity", what);
  GemmArgs g{};
  g.a = static_cast<const uint16_t*>(a_xg); g.w = static_cast<const uint16_t*>(w_qkv);
  g.m = m; g.n = 3 * d_model; g.k = d_model;
  g.cos_t = cos_t; g.sin_t = sin_t; g.seq = seq; g.heads = heads; g.head_dim = d_model / heads;
  g.d_model = d_model; g.cap = capacity;
  g.q_out = static_cast<uint16_t*>(q_out); g.k_cache = static_cast<uint16_t*>(k_cache);
  g.v_cache = static_cast<uint16_t*>(v_cache);
  g.vec16 = aligned16(q_out) && aligned16(k_cache) && aligned16(v_cache);
  g.row_scale = rscale; g.ss = ss; g.ss_parts = ss_parts;
  return launch_gemm<G_QKV>(g, dtype, static_cast<hipStream_t>(stream), what);
}

extern "C" int sfl_gemm_qkv_rope_scaled(const void* a_xg, const void* w_qkv, const float* rscale, int m, int seq,
                                        int d_model, int heads, const float* cos_t, const float* sin_t,
                                        void* q_out, void* k_cache, void* v_cache, int capacity, int dtype,
                                        void* stream) {
  const char* what = "gemm_qkv_rope_scaled";
  if (!rscale) return set_error(SFL_ERR_INVALID, "%s: null pointer argument", what);
  return gemm_qkv_normed(what, a_xg, w_qkv, rscale, nullptr, 0, m, seq, d_model, heads, cos_t, sin_t, q_out, k_cache,
                         v_cache, capacity, dtype, stream);
}

extern "C" int sfl_gemm_qkv_rope_normed(const void* a_xg, const void* w_qkv, const float* ss_parts, int parts, int m,
                                        int seq, int d_model, int heads, const float* cos_t, const float* sin_t,
                                        void* q_out, void* k_cache, void* v_cache, int capacity, int dtype,
                                        void* stream) {
  const char* what = "gemm_qkv_rope_normed";
  if (!ss_parts) return set_error(SFL_ERR_INVALID, "%s: null pointer argument", what);
  if (parts < 1) return set_error(SFL_ERR_INVALID, "%s: parts must be positive", what);
  return gemm_qkv_normed(what, a_xg, w_qkv, nullptr, ss_parts, parts, m, seq, d_model, heads, cos_t, sin_t, q_out,
                         k_cache, v_cache, capacity, dtype, stream);
}

static int gemm_swiglu_normed(const char* what, const void* a_xg, const void* w13_interleaved, const float* rscale,
                              const float* ss, int ss_parts, void* h_out, int m, int d_ff, int k, int dtype,
                              void* stream) {
  if (!a_xg || !w13_interleaved || !h_out) return set_error(SFL_ERR_INVALID, "%s: null pointer argument", what);
  if (d_ff % 8) return set_error(SFL_ERR_UNSUPPORTED, "%s: d_ff must be a multiple of 8", what);
  if (!gemm32_path(m, 2 * d_ff, k)) return set_error(SFL_ERR_UNSUPPORTED, "%s: K must be a multiple of %d", what, K2);
  GemmArgs g{};
  g.a = static_cast<const uint16_t*>(a_xg); g.w = static_cast<const uint16_t*>(w13_interleaved);
  g.m = m; g.n = 2 * d_ff; g.k = k; g.h_out = static_cast<uint16_t*>(h_out);
  g.vec16 = aligned16(h_out);
  g.row_scale = rscale; g.ss = ss; g.ss_parts = ss_parts;
  return launch_gemm<G_SWIGLU>(g, dtype, static_cast<hipStream_t>(stream), what);
}

extern "C" int sfl_gemm_swiglu_scaled(const void* a_xg, const void* w13_interleaved, const float* rscale,
                                      void* h_out, int m, int d_ff, int k, int dtype, void* stream) {
  const char* what = "gemm_swiglu_scaled";
  if (!rscale) return set_error(SFL_ERR_INVALID, "%s: null pointer argument", what);
  return gemm_swiglu_normed(what, a_xg, w13_interleaved, rscale, nullptr, 0, h_out, m, d_ff, k, dtype, stream);
}

extern "C" int sfl_gemm_swiglu_normed(const void* a_xg, const void* w13_interleaved, const float* ss_parts, int parts,
                                      void* h_out, int m, int d_ff, int k, int dtype, void* stream) {
  const char* what = "gemm_swiglu_normed";
  if (!ss_parts) return set_error(SFL_ERR_INVALID, "%s: null pointer argument", what);
  if (parts < 1) return set_error(SFL_ERR_INVALID, "%s: parts must be positive", what);
  return gemm_swiglu_normed(what, a_xg, w13_interleaved, nullptr, ss_parts, parts, h_out, m, d_ff, k, dtype, stream);
}

static int gemm_residual_norm(const char* what, const void* a, const void* w, float* x, int m, int n, int k,
                              const void* gain_next, void* act_xg, float* ss_parts, int part, int dtype,
                              void* stream) {
  if (!a || !w || !x || !gain_next || !act_xg || !ss_parts)
    return set_error(SFL_ERR_INVALID, "%s: null pointer argument", what);
  if (m < 1 || n < 1 || k < 1) return set_error(SFL_ERR_INVALID, "%s: sizes must be positive", what);
  if (n % 4) return set_error(SFL_ERR_UNSUPPORTED, "%s: N must be a multiple of 4", what);
  if (!gemm32_path(m, n, k)) return set_error(SFL_ERR_UNSUPPORTED, "%s: K must be a multiple of %d", what, K2);
  if (reinterpret_cast<uintptr_t>(x) % 16 || reinterpret_cast<uintptr_t>(act_xg) % 8 ||
      reinterpret_cast<uintptr_t>(gain_next) % 8)
    return set_error(SFL_ERR_INVALID, "%s: x must be 16-byte and act / gain 8-byte aligned", what);
  GemmArgs g{};
  g.a = static_cast<const uint16_t*>(a); g.w = static_cast<const uint16_t*>(w);
  g.m = m; g.n = n; g.k = k; g.c = x; g.c_f32 = 1; g.accumulate = 1;
  g.norm_gain = static_cast<const uint16_t*>(gain_next);
  g.norm_act = static_cast<uint16_t*>(act_xg);
  g.norm_ss = ss_parts;
  g.norm_part = part;
  g.vec16 = aligned16(act_xg) && n % 8 == 0;  // rows of act start 16-byte aligned
  return launch_gemm<G_PLAIN>(g, dtype, static_cast<hipStream_t>(stream), what);
}

extern "C" int sfl_gemm_residual_norm(const void* a, const void* w, float* x, int m, int n, int k,
                                      const void* gain_next, void* act_xg, float* ss_parts, int dtype,
                                      void* stream) {
  return gemm_residual_norm("gemm_residual_norm", a, w, x, m, n, k, gain_next, act_xg, ss_parts, 128, dtype, stream);
}

extern "C" int sfl_gemm_tile(int m, int n, int k, int epilogue, int* features, int* tokens, int* k_split) {
  const char* what = "gemm_tile";
  if (!features || !tokens || !k_split) return set_error(SFL_ERR_INVALID, "%s: null pointer argument", what);
  if (m < 1 || n < 1 || k < 1 || epilogue < G_PLAIN || epilogue > G_SWIGLU)
    return set_error(SFL_ERR_INVALID, "%s: bad sizes or epilogue", what);
  if (!gemm32_path(m, n, k)) return set_error(SFL_ERR_UNSUPPORTED, "%s: K must be a multiple of %d", what, K2);
  const Tile16 t = tile16_for(m, n, k, epilogue);
  *features = t == S32x32 ? 32 : t <= S64x64 ? 64 : t <= T128x128 ? 128 : 256;
  *tokens = t <= S64x32 ? 32 : t <= T128x64 ? 64 : t == T128x128 ? 128 : t == T256x256 ? 256 : 384;
  *k_split = t <= S128x64;
  return SFL_OK;
}

extern "C" int sfl_gemm_norm_part(int m, int n, int k) { return norm_part_of(tile16_for(m, n, k, G_PLAIN)); }

extern "C" int sfl_gemm_residual_norm_parts(const void* a, const void* w, float* x, int m, int n, int k,
                                            const void* gain_next, void* act_xg, float* ss_parts, int part,
                                            int dtype, void* stream) {
  const char* what = "gemm_residual_norm_parts";
  if (part != 128 && (m < 1 || n < 1 || part != sfl_gemm_norm_part(m, n, k)))
    return set_error(SFL_ERR_INVALID, "%s: part must be 128 or sfl_gemm_norm_part(m, n, k)", what);
  return gemm_residual_norm(what, a, w, x, m, n, k, gain_next, act_xg, ss_parts, part, dtype, stream);
}

extern "C" int sfl_norm_scale(const float* ss_parts, int parts, int m, int d_model, float* rscale, void* stream) {
  if (!ss_parts || !rscale) return set_error(SFL_ERR_INVALID, "norm_scale: null pointer argument");
  if (parts < 1 || m < 1 || d_model < 1) return set_error(SFL_ERR_INVALID, "norm_scale: sizes must be positive");
  hipLaunchKernelGGL(norm_scale_kernel, dim3(unsigned((m + 255) / 256)), dim3(256), 0,
                     static_cast<hipStream_t>(stream), ss_parts, parts, m, d_model, rscale);
  return check_launch("norm_scale");
}

extern "C" int sfl_rmsnorm_rows_scaled(const float* x, const void* w, void* act_xg, float* rscale, int m,
                                       int d_model, int dtype, void* stream) {
  const char* what = "rmsnorm_rows_scaled";
  if (!x || !w || !act_xg || !rscale) return set_error(SFL_ERR_INVALID, "%s: null pointer argument", what);
  if (m < 1 || d_model < 1) return set_error(SFL_ERR_INVALID, "%s: sizes must be positive", what);
  if (!gemm_dtype_ok(dtype)) return set_error(SFL_ERR_UNSUPPORTED, "%s: dtype must be BF16 or F16", what);
  if (d_model % 4 || d_model > 4 * kWave * kNormVec || reinterpret_cast<uintptr_t>(x) % 16 ||
      reinterpret_cast<uintptr_t>(act_xg) % 8)
    return set_error(SFL_ERR_UNSUPPORTED, "%s: d_model must be a multiple of 4 and at most %d, x 16-byte and "
                     "act 8-byte aligned", what, 4 * kWave * kNormVec);
  const hipStream_t s = static_cast<hipStream_t>(stream);
  if (dtype == SFL_DTYPE_BF16)
    hipLaunchKernelGGL((rmsnorm_rows_wave_kernel<bf16_t, bf16_t, true>), dim3((m + 3) / 4), dim3(256), 0, s, x,
                       static_cast<const bf16_t*>(w), static_cast<bf16_t*>(act_xg), m, d_model, rscale);
  else
    hipLaunchKernelGGL((rmsnorm_rows_wave_kernel<f16_t, f16_t, true>), dim3((m + 3) / 4), dim3(256), 0, s, x,
                       static_cast<const f16_t*>(w), static_cast<f16_t*>(act_xg), m, d_model, rscale);
  return check_launch(what);
}

extern "C" int sfl_gemm_swiglu(const void* a, const void* w13_interleaved, void* h_out, int m, int d_ff,
                               int k, int dtype, void* stream) {
  const char* what = "gemm_swiglu";
  if (!a || !w13_interleaved || !h_out) return set_error(SFL_ERR_INVALID, "%s: null pointer argument", what);
  if (d_ff % 8) return set_error(SFL_ERR_UNSUPPORTED, "%s: d_ff must be a multiple of 8", what);
  if (dtype == SFL_DTYPE_F32) {
    if (!aligned16(h_out)) return set_error(SFL_ERR_INVALID, "%s: fp32 h must be 16-byte aligned", what);
    F32GemmArgs f{};
    f.a = static_cast<const float*>(a); f.w = static_cast<const float*>(w13_interleaved);
    f.m = m; f.n = 2 * d_ff; f.k = k; f.h_out = static_cast<float*>(h_out);
    return launch_gemm_f32(f, F32_SWIGLU, static_cast<hipStream_t>(stream), what);
  }
  GemmArgs g{};
  g.a = static_cast<const uint16_t*>(a); g.w = static_cast<const uint16_t*>(w13_interleaved);
  g.m = m; g.n = 2 * d_ff; g.k = k; g.h_out = static_cast<uint16_t*>(h_out);
  g.vec16 = aligned16(h_out);
  return launch_gemm<G_SWIGLU>(g, dtype, static_cast<hipStream_t>(stream), what);
}

extern "C" int sfl_embed_rows(const int64_t* ids, const void* emb, float* x, int m, int d_model, int dtype,
                              void* stream) {
  if (!ids || !emb || !x) return set_error(SFL_ERR_INVALID, "embed_rows: null pointer argument");
  if (m < 1 || d_model < 1) return set_error(SFL_ERR_INVALID, "embed_rows: sizes must be positive");
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (dtype == SFL_DTYPE_BF16)
    hipLaunchKernelGGL(embed_rows_kernel<bf16_t>, dim3(m), dim3(256), 0, s, ids, static_cast<const bf16_t*>(emb), x, d_model);
  else if (dtype == SFL_DTYPE_F16)
    hipLaunchKernelGGL(embed_rows_kernel<f16_t>, dim3(m), dim3(256), 0, s, ids, static_cast<const f16_t*>(emb), x, d_model);
  else if (dtype == SFL_DTYPE_F32)
    hipLaunchKernelGGL(embed_rows_kernel<float>, dim3(m), dim3(256), 0, s, ids, static_cast<const float*>(emb), x, d_model);
  else
    return set_error(SFL_ERR_UNSUPPORTED, "embed_rows: dtype must be F32, BF16 or F16");
  return check_launch("embed_rows");
}

template <typename T, typename O>
static void launch_rmsnorm_rows(const float* x, const void* w, void* out, int m, int d, bool wave_rows, hipStream_t s) {
  if (wave_rows)
    hipLaunchKernelGGL((rmsnorm_rows_wave_kernel<T, O>), dim3((m + 3) / 4), dim3(256), 0, s, x,
                       static_cast<const T*>(w), static_cast<O*>(out), m, d, nullptr);
  else
    hipLaunchKernelGGL((rmsnorm_rows_kernel<T, O>), dim3(m), dim3(256), 0, s, x, static_cast<const T*>(w),
                       static_cast<O*>(out), d);
}

extern "C" int sfl_rmsnorm_rows(const float* x, const void* w, void* out, int m, int d_model, int dtype,
                                int out_dtype, void* stream) {
  const char* what = "rmsnorm_rows";
  if (!x || !w || !out) return set_error(SFL_ERR_INVALID, "%s: null pointer argument", what);
  if (m < 1 || d_model < 1) return set_error(SFL_ERR_INVALID, "%s: sizes must be positive", what);
  if (dtype != SFL_DTYPE_BF16 && dtype != SFL_DTYPE_F16 && dtype != SFL_DTYPE_F32)
    return set_error(SFL_ERR_UNSUPPORTED, "%s: dtype must be F32, BF16 or F16", what);
  if (out_dtype != SFL_DTYPE_BF16 && out_dtype != SFL_DTYPE_F16 && out_dtype != SFL_DTYPE_F32)
    return set_error(SFL_ERR_UNSUPPORTED, "%s: out dtype must be F32, BF16 or F16", what);
  hipStream_t s = static_cast<hipStream_t>(stream);
  const bool wave_rows = d_model % 4 == 0 && d_model <= 4 * kWave * kNormVec &&
                         reinterpret_cast<uintptr_t>(x) % 16 == 0 &&
                         reinterpret_cast<uintptr_t>(out) % (out_dtype == SFL_DTYPE_F32 ? 16 : 8) == 0;
  const int key = dtype * 8 + out_dtype;
  switch (key) {
    case SFL_DTYPE_BF16 * 8 + SFL_DTYPE_BF16: launch_rmsnorm_rows<bf16_t, bf16_t>(x, w, out, m, d_model, wave_rows, s); break;
    case SFL_DTYPE_F32 * 8 + SFL_DTYPE_BF16: launch_rmsnorm_rows<float, bf16_t>(x, w, out, m, d_model, wave_rows, s); break;
    case SFL_DTYPE_F16 * 8 + SFL_DTYPE_F16: launch_rmsnorm_rows<f16_t, f16_t>(x, w, out, m, d_model, wave_rows, s); break;
    case SFL_DTYPE_F32 * 8 + SFL_DTYPE_F32: launch_rmsnorm_rows<float, float>(x, w, out, m, d_model, wave_rows, s); break;
    default: return set_error(SFL_ERR_UNSUPPORTED, "%s: unsupported weight / output dtype pair", what);
  }
  return check_launch(what);
}
