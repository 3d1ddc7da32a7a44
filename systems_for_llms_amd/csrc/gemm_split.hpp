// Prefill GEMM tiles with K split over the waves of a workgroup, for 16-bit
// operands (gemm_small.hip) and fp32 ones (prefill_f32.hip).
#pragma once
#include <type_traits>

#include "gemm16.hpp"
#include "gemm_f32.hpp"

namespace sfl {

template <typename T> struct SplitArgs { using type = GemmArgs; };
template <> struct SplitArgs<float> { using type = F32GemmArgs; };

// acc += the products of one 16-byte slot per lane of both operands: 8 16-bit
// values, one 32x32x16 MFMA; or 4 floats, four 32x32x2 ones (lane half h holds
// k = 8 kk + 4 h + s in step s for both operands, so each product pairs equal k).
template <typename T>
__device__ __forceinline__ f32x16 mma_slot(const u32x4& a, const u32x4& b, f32x16 acc) {
  if constexpr (std::is_same<T, float>::value) {
#pragma unroll
    for (int s = 0; s < 4; ++s)
      acc = __builtin_amdgcn_mfma_f32_32x32x2f32(__uint_as_float(a[s]), __uint_as_float(b[s]), acc, 0, 0, 0);
    return acc;
  } else {
    return mfma32<T>(a, b, acc);
  }
}


// fp32 products on the bf16 matrix cores, by the published method of splitting
// an fp32 operand into three bf16 ones (Henry, Tang, Heinecke, "Leveraging the
// bfloat16 Artificial Intelligence Datatype For Higher-Precision Computations",
// ARITH 2019): x = p0 + p1 + p2 exactly, 8 significant bits apiece by
// truncation, all of x's sign. Of the nine products of two operands' pieces the
// eight without p2 p2 are summed in fp32; the one left out is below 2^-30 of
// the operands' product, under the 2^-24 that an fp32 product rounds by. p0 p0
// has a sum of its own: the other seven, about 2^-6 of it at most, then cost it
// one rounding in all and not one per product, so a sum of few terms is as exact
// as one of fp32 products.
// `lost` collects the bits no piece holds in its low half: none for operands
// of at least 2^-110, some below, where p2 would need values under bf16's
// smallest subnormal (the MFMAs keep subnormal operands and results); the
// callers compute such a tile again on fp32 products. (No contraction: the
// remainder is that of x, not of a product x was rounded from.)
// An MFMA takes 16 k values at 32 cycles, eight of them 256, where eight
// 32x32x2 fp32 ones take 512.
__device__ __forceinline__ void split3(const uint4& lo, const uint4& hi, u32x4 (&p)[3], uint32_t& lost) {
#pragma clang fp contract(off)
  const uint32_t x[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    uint32_t a = x[2 * i], b = x[2 * i + 1];
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      p[j][i] = __builtin_amdgcn_perm(b, a, 0x07060302u);
      if (j < 2) {
        a = __float_as_uint(__uint_as_float(a) - __uint_as_float(a & 0xffff0000u));
        b = __float_as_uint(__uint_as_float(b) - __uint_as_float(b & 0xffff0000u));
      }
    }
    lost |= a | b;
  }
}

// The products beside p0 p0, smallest first: piece kLowA[i] of one operand with
// piece kLowB[i] of the other.
constexpr int kLowProducts = 7;
constexpr int kLowA[kLowProducts] = {2, 1, 2, 1, 0, 1, 0};
constexpr int kLowB[kLowProducts] = {1, 2, 0, 1, 2, 0, 1};

// TBN features x TBM tokens per workgroup of NW waves; wave w takes the KS-wide
// K chunks w, w + NW, ... of the whole tile through a private ring of NS LDS
// stages (the layout, swizzle and operand reads of gemm32_kernel's stages).
template <typename T, int E, int TBN, int TBM, int KS, int NW, int NS>
__global__ __launch_bounds__(NW * kWave) __attribute__((amdgpu_waves_per_eu(std::is_same<T, float>::value ? 2 : 1)))
void gemm_split_kernel(typename SplitArgs<T>::type g) {
  constexpr bool kF32 = std::is_same<T, float>::value;
  constexpr int EB = Elem<T>::bytes;            // bytes per operand element
  constexpr int NBN = TBN / 32, NBM = TBM / 32, NB = NBN * NBM;  // 32x32 blocks of the tile
  constexpr int SL = KS * EB / 16;              // 16-byte slots per row of a stage
  constexpr int RPL = kWave / SL;               // rows one 1 KB load instruction moves
  constexpr int LPS = (TBN + TBM) / RPL;        // load instructions per stage
  using Stage = Stage32<TBN, TBM, SL>;
  // Blocks whose partials (4 KB per wave) fit the stages at once; each pass
  // over that many blocks, a wave finishes OPB of them.
  constexpr int kFit = int(sizeof(Stage)) * NS / 4096;
  constexpr int RB = kFit >= NB ? NB : kFit >= NB / 2 ? NB / 2 : NB / 4;
  constexpr int OPB = RB >= NW ? RB / NW : 1;
  static_assert(kFit >= RB && NB % RB == 0 && (RB % NW == 0 || RB < NW), "reduction passes");
  __shared__ Stage st[NW][NS];
  const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x) / kWave), lane = threadIdx.x % kWave;
  const int l32 = lane % 32, hf = lane / 32;
  const int2 tile = xcd_tile(blockIdx.x, (g.n + TBN - 1) / TBN, (g.m + TBM - 1) / TBM, 16);
  const int n0 = tile.x * TBN, m0 = tile.y * TBM;
  const int chunks = g.k / KS;

  const i32x4_t rw = buffer_rsrc(g.w, unsigned(g.n * g.k * EB));
  const i32x4_t ra = buffer_rsrc(g.a, unsigned(g.m * g.k * EB));
  const int rr = lane / SL, pos = lane % SL;
  unsigned voff[2];
#pragma unroll
  for (int par = 0; par < 2; ++par)
    voff[par] = unsigned(rr * g.k * EB + 16 * (pos ^ stage_swizzle<SL>(RPL * par + rr)));
  auto issue = [&](Stage& s, int c) {
#pragma unroll
    for (int r = 0; r < TBN / RPL; ++r)
      lds_load16(rw, lds_offset(&s.w[RPL * r][0]), voff[r & 1], unsigned(((n0 + RPL * r) * g.k + c * KS) * EB));
#pragma unroll
    for (int r = 0; r < TBM / RPL; ++r)
      lds_load16(ra, lds_offset(&s.a[RPL * r][0]), voff[r & 1], unsigned(((m0 + RPL * r) * g.k + c * KS) * EB));
  };

  f32x16 acc[NBN][NBM];
  f32x16 low[kF32 ? NBN : 1][kF32 ? NBM : 1];  // fp32: the products beside p0 p0
  const int mine = (chunks - wave + NW - 1) / NW;  // this wave's chunks
  const int sw = stage_swizzle<SL>(l32);
  uint32_t lost = 0;
  if constexpr (kF32) {
#pragma unroll
    for (int i = 0; i < NBN; ++i)
#pragma unroll
      for (int j = 0; j < NBM; ++j)
#pragma unroll
        for (int e = 0; e < 16; ++e) low[i][j][e] = 0.f;
  }
  const auto k_loop = [&](auto pieces) {
#pragma unroll
    for (int i = 0; i < NBN; ++i)
#pragma unroll
      for (int j = 0; j < NBM; ++j)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;
#pragma unroll
    for (int s = 0; s < NS; ++s)
      if (s < mine) issue(st[wave][s], wave + s * NW);
    int cur = 0;
    for (int t = 0; t < mine; ++t) {
      wait_younger<NS - 1, LPS>(min(NS - 1, mine - 1 - t));
      const Stage& s = st[wave][cur];
      if constexpr (decltype(pieces)::value) {
        // 16 k values per step: lane half h takes k = 16 kk + 8 h .. + 7 of both operands.
#pragma unroll
        for (int kk = 0; kk < SL / 4; ++kk) {
          const int slot = 4 * kk + 2 * hf;
          u32x4 af[NBN][3], bf[NBM][3];
#pragma unroll
          for (int i = 0; i < NBN; ++i) split3(s.w[32 * i + l32][slot ^ sw], s.w[32 * i + l32][(slot + 1) ^ sw], af[i], lost);
#pragma unroll
          for (int j = 0; j < NBM; ++j) split3(s.a[32 * j + l32][slot ^ sw], s.a[32 * j + l32][(slot + 1) ^ sw], bf[j], lost);
#pragma unroll
          for (int p = 0; p < kLowProducts; ++p)
#pragma unroll
            for (int i = 0; i < NBN; ++i)
#pragma unroll
              for (int j = 0; j < NBM; ++j) low[i][j] = mfma32<bf16_t>(af[i][kLowA[p]], bf[j][kLowB[p]], low[i][j]);
#pragma unroll
          for (int i = 0; i < NBN; ++i)
#pragma unroll
            for (int j = 0; j < NBM; ++j) acc[i][j] = mfma32<bf16_t>(af[i][0], bf[j][0], acc[i][j]);
        }
      } else {
#pragma unroll
        for (int kk = 0; kk < SL / 2; ++kk) {
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
            for (int j = 0; j < NBM; ++j) acc[i][j] = mma_slot<T>(af[i], bf[j], acc[i][j]);
        }
      }
      if (t + NS < mine) {
        wait_lds_reads();
        issue(st[wave][cur], wave + (t + NS) * NW);
      }
      cur = cur + 1 == NS ? 0 : cur + 1;
    }
  };
  if constexpr (kF32) {
    k_loop(std::true_type{});
    // An infinite or NaN operand leaves a NaN remainder, so every sum it
    // enters is NaN: such a tile is computed again on fp32 products, whose
    // infinities and NaNs are those of the operation, and so is one with an
    // operand its pieces do not hold.
    bool redo = (lost & 0xffffu) != 0;
#pragma unroll
    for (int i = 0; i < NBN; ++i)
#pragma unroll
      for (int j = 0; j < NBM; ++j)
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          acc[i][j][e] += low[i][j][e];
          redo |= acc[i][j][e] != acc[i][j][e];
        }
    if (__syncthreads_or(redo)) k_loop(std::false_type{});
  } else {
    k_loop(std::false_type{});
  }

  // Partial tiles to LDS, RB blocks at a time; each block is summed in wave
  // order by the wave that finishes it. A residual update adds the sum to the
  // old C, loaded before the barriers.
  bool acc_c = false, norm = false;
  if constexpr (E == G_PLAIN && !kF32) {
    acc_c = g.c_f32 && g.accumulate && (g.n & 3) == 0;
    norm = g.norm_gain != nullptr;
  }
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
      if constexpr (kF32) {
        // (fp32 adds the whole sum to the old C in its epilogue)
      } else if constexpr (E == G_PLAIN) {
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
        if constexpr (kF32) {
          store_block_f32<E>(g, own[o], nt, m, hf);
          continue;
        } else if constexpr (E == G_PLAIN) {
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
        if constexpr (!kF32) {
          const QkvTok tok = E == G_QKV ? qkv_tok(g, m) : QkvTok{};
          store_block<T, E>(g, own[o], nt, m, tok, rsc[o], hf);
        }
      }
    }
  }
}

}  // namespace sfl
