// 16-bit prefill GEMMs of few tiles (prompts of up to ~1000 tokens): K split
// over the waves of a workgroup.
//
// A prompt of 301 tokens gives the residual GEMMs of d_model 1024 only 24
// tiles of 128 x 128, and each of those workgroups walks its K steps with a
// barrier and one step of loads in flight: 0.55 us per step, 14 us at K = 1024
// and 29 us at K = 2752 whatever M is. What bounds such a launch is that chain
// and how fast one CU can pull its operands (~30 bytes per cycle measured with
// the weights coming from HBM), so here (a) tiles are as small as it takes to
// give every CU one, and (b) each wave computes the whole tile over its own
// share of K: a wave has its own LDS stages and waits only for its own loads,
// so no barrier stands in the K loop, and a tile's MFMA operands are read from
// LDS once per (features + tokens) instead of once per wave pair. The partial
// tiles are added through LDS in wave order, so results do not vary from call
// to call. Measured (graph replays, weights rotating through 400 MB; launch
// gap of ~2 us included), 128 x 128 tiles -> these:
//   M 301 N 1024 K 1024   14.2 ->  6.0 us (64 x 32)
//   M 301 N 1024 K 2752   28.8 ->  8.9    (64 x 32)
//   M 301 N 3072 K 1024   14.6 ->  7.8    (64 x 64)
//   M 301 N 5504 K 1024   19.7 -> 13.2    (128 x 64)
//   M 16  N 1024 K 1024   12.6 ->  4.9    (32 x 32)
//   M 2048 N 1024 K 2752  32.4 -> 19.9    (128 x 64)
// 8 waves, other stage counts, K chunks of 32 and a 128 x 128 tile per wave
// were no faster at the tile each grid size uses.
#include "gemm16.hpp"

namespace sfl {
namespace {

// TBN features x TBM tokens per workgroup of NW waves; wave w takes the KS-wide
// K chunks w, w + NW, ... of the whole tile through a private ring of NS LDS
// stages (the layout, swizzle and operand reads of gemm32_kernel's stages).
template <typename T, int E, int TBN, int TBM, int KS, int NW, int NS>
__global__ __launch_bounds__(NW * kWave) void gemm_small_kernel(GemmArgs g) {
  constexpr int NBN = TBN / 32, NBM = TBM / 32, NB = NBN * NBM;  // 32x32 blocks of the tile
  constexpr int SL = KS / 8;                    // 16-byte slots per row of a stage
  constexpr int RPL = kWave / SL;               // rows one 1 KB load instruction moves
  constexpr int LPS = (TBN + TBM) / RPL;        // load instructions per stage
  using Stage = Stage32<TBN, TBM, SL>;
  // Blocks whose partials (4 KB per wave) fit the stages at once; each pass
  // over that many blocks, a wave finishes OPB of them.
  constexpr int kFit = int(sizeof(Stage)) * NS / 4096;
  constexpr int RB = kFit >= NB ? NB : NB / 2;
  constexpr int OPB = RB >= NW ? RB / NW : 1;
  static_assert(kFit >= RB && NB % RB == 0 && (RB % NW == 0 || RB < NW), "reduction passes");
  __shared__ Stage st[NW][NS];
  const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x) / kWave), lane = threadIdx.x % kWave;
  const int l32 = lane % 32, hf = lane / 32;
  const int2 tile = xcd_tile(blockIdx.x, (g.n + TBN - 1) / TBN, (g.m + TBM - 1) / TBM, 16);
  const int n0 = tile.x * TBN, m0 = tile.y * TBM;
  const int chunks = g.k / KS;

  const i32x4_t rw = buffer_rsrc(g.w, unsigned(g.n * g.k * 2));
  const i32x4_t ra = buffer_rsrc(g.a, unsigned(g.m * g.k * 2));
  const int rr = lane / SL, pos = lane % SL;
  unsigned voff[2];
#pragma unroll
  for (int par = 0; par < 2; ++par)
    voff[par] = unsigned((rr * g.k + 8 * (pos ^ stage_swizzle<SL>(RPL * par + rr))) * 2);
  auto issue = [&](Stage& s, int c) {
#pragma unroll
    for (int r = 0; r < TBN / RPL; ++r)
      lds_load16(rw, lds_offset(&s.w[RPL * r][0]), voff[r & 1], unsigned(((n0 + RPL * r) * g.k + c * KS) * 2));
#pragma unroll
    for (int r = 0; r < TBM / RPL; ++r)
      lds_load16(ra, lds_offset(&s.a[RPL * r][0]), voff[r & 1], unsigned(((m0 + RPL * r) * g.k + c * KS) * 2));
  };

  f32x16 acc[NBN][NBM];
#pragma unroll
  for (int i = 0; i < NBN; ++i)
#pragma unroll
    for (int j = 0; j < NBM; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;
  const int mine = (chunks - wave + NW - 1) / NW;  // this wave's chunks
#pragma unroll
  for (int s = 0; s < NS; ++s)
    if (s < mine) issue(st[wave][s], wave + s * NW);
  const int sw = stage_swizzle<SL>(l32);
  int cur = 0;
  for (int t = 0; t < mine; ++t) {
    wait_younger<NS - 1, LPS>(min(NS - 1, mine - 1 - t));
    const Stage& s = st[wave][cur];
#pragma unroll
    for (int kk = 0; kk < KS / 16; ++kk) {
      const int slot = (2 * kk + hf) ^ sw;
      u32x4 af[NBN], bf[NBM];
#pragma unroll
      for (int i = 0; i < NBN; ++i) {
        const uint4 v = s.w[32 * i + l32][slot];
        af[i] = u32x4{v.x, v.y, v.z, v.w};
      }
#pragma unroll
      for (int j = 0; j < NBM; ++j) {
        const uint4 v = s.a[32 * j + l32][slot];
        bf[j] = u32x4{v.x, v.y, v.z, v.w};
      }
#pragma unroll
      for (int i = 0; i < NBN; ++i)
#pragma unroll
        for (int j = 0; j < NBM; ++j) acc[i][j] = mfma32<T>(af[i], bf[j], acc[i][j]);
    }
    if (t + NS < mine) issue(st[wave][cur], wave + (t + NS) * NW);
    cur = cur + 1 == NS ? 0 : cur + 1;
  }

  // Partial tiles to LDS, RB blocks at a time; each block is summed in wave
  // order by the wave that finishes it. A residual update adds the sum to the
  // old C, loaded before the barriers.
  const bool acc_c = E == G_PLAIN && g.c_f32 && g.accumulate && (g.n & 3) == 0;
  const bool norm = E == G_PLAIN && g.norm_gain != nullptr;
  float4* const red = reinterpret_cast<float4*>(&st[0][0]);  // [wave][RB][4][lane]
#pragma unroll
  for (int b0 = 0; b0 < NB; b0 += RB) {
    f32x16 own[OPB];
    float rsc[OPB];
#pragma unroll
    for (int o = 0; o < OPB; ++o) {
      const int blk = b0 + min(wave * OPB + o, RB - 1);
      const int mr = min(m0 + 32 * (blk % NBM) + l32, g.m - 1);
      rsc[o] = 1.f;
#pragma unroll
      for (int e = 0; e < 16; ++e) own[o][e] = 0.f;
      if constexpr (E == G_PLAIN) {
        if (acc_c) {
          const float* c = static_cast<const float*>(g.c) + long(mr) * g.n;
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const float4 v = *reinterpret_cast<const float4*>(c + min(n0 + 32 * (blk / NBM) + 8 * q + 4 * hf, g.n - 4));
            own[o][4 * q] = v.x;
            own[o][4 * q + 1] = v.y;
            own[o][4 * q + 2] = v.z;
            own[o][4 * q + 3] = v.w;
          }
        }
      } else {
        if (g.ss) rsc[o] = parts_scale(g, mr);
        else if (g.row_scale) rsc[o] = g.row_scale[mr];
      }
    }
    __syncthreads();  // the stages (or the previous pass's partials) are no longer read
#pragma unroll
    for (int b = 0; b < RB; ++b)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const f32x16& v = acc[(b0 + b) / NBM][(b0 + b) % NBM];
        red[((wave * RB + b) * 4 + q) * kWave + lane] = make_float4(v[4 * q], v[4 * q + 1], v[4 * q + 2], v[4 * q + 3]);
      }
    __syncthreads();
    if (wave * OPB < RB) {
#pragma unroll
      for (int o = 0; o < OPB; ++o) {
        const int lb = wave * OPB + o, blk = b0 + lb;
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
          for (int w = 0; w < NW; ++w) {
            const float4 v = red[((w * RB + lb) * 4 + q) * kWave + lane];
            own[o][4 * q] += v.x;
            own[o][4 * q + 1] += v.y;
            own[o][4 * q + 2] += v.z;
            own[o][4 * q + 3] += v.w;
          }
        const int nt = n0 + 32 * (blk / NBM), m = m0 + 32 * (blk % NBM) + l32;
        if constexpr (E == G_PLAIN) {
          if (acc_c) {
            uint2 gw[4] = {};
            if (norm) {
#pragma unroll
              for (int q = 0; q < 4; ++q)
                gw[q] = *reinterpret_cast<const uint2*>(g.norm_gain + min(nt + 8 * q + 4 * hf, g.n - 4));
            }
            float ssq = 0.f;
            residual_block<T>(g, own[o], nt, m, hf, norm, gw, ssq);
            if (norm) {  // parts of 32 features: this block's
              const float t = ssq + lane_xor(ssq, 32);
              if (hf == 0 && m < g.m && nt < g.n) g.norm_ss[long(nt / 32) * g.m + m] = t;
            }
            continue;
          }
        }
        const QkvTok tok = E == G_QKV ? qkv_tok(g, m) : QkvTok{};
        store_block<T, E>(g, own[o], nt, m, tok, rsc[o], hf);
      }
    }
  }
}

template <typename T, int E, int TBN, int TBM, int KS, int NW, int NS>
int launch_tile(const GemmArgs& g, hipStream_t s, const char* what) {
  const long tiles = long((g.n + TBN - 1) / TBN) * ((g.m + TBM - 1) / TBM);
  hipLaunchKernelGGL((gemm_small_kernel<T, E, TBN, TBM, KS, NW, NS>), dim3(unsigned(tiles)), dim3(NW * kWave), 0, s, g);
  return check_launch(what);
}

}  // namespace

template <typename T, int E>
int launch_gemm_small(const GemmArgs& g, Tile16 t, hipStream_t s, const char* what) {
  switch (t) {
    case S32x32: return launch_tile<T, E, 32, 32, 64, 4, 2>(g, s, what);
    case S64x32: return launch_tile<T, E, 64, 32, 64, 4, 3>(g, s, what);
    case S64x64: return launch_tile<T, E, 64, 64, 64, 4, 2>(g, s, what);
    default: return launch_tile<T, E, 128, 64, 64, 6, 1>(g, s, what);
  }
}

template int launch_gemm_small<bf16_t, G_PLAIN>(const GemmArgs&, Tile16, hipStream_t, const char*);
template int launch_gemm_small<bf16_t, G_QKV>(const GemmArgs&, Tile16, hipStream_t, const char*);
template int launch_gemm_small<bf16_t, G_SWIGLU>(const GemmArgs&, Tile16, hipStream_t, const char*);
template int launch_gemm_small<f16_t, G_PLAIN>(const GemmArgs&, Tile16, hipStream_t, const char*);
template int launch_gemm_small<f16_t, G_QKV>(const GemmArgs&, Tile16, hipStream_t, const char*);
template int launch_gemm_small<f16_t, G_SWIGLU>(const GemmArgs&, Tile16, hipStream_t, const char*);

}  // namespace sfl
