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
// (One product alone, again and again. Between the other launches of a prompt,
// at M 301: q/k/v 10.7, SwiGLU 13.7, output projection and w2 9.3 on average.)
// 8 waves, other stage counts, K chunks of 32 and a 128 x 128 tile per wave
// were no faster at the tile each grid size uses.
#include "gemm_split.hpp"

namespace sfl {
namespace {

template <typename T, int E, int TBN, int TBM, int KS, int NW, int NS>
int launch_tile(const GemmArgs& g, hipStream_t s, const char* what) {
  const long tiles = long((g.n + TBN - 1) / TBN) * ((g.m + TBM - 1) / TBM);
  hipLaunchKernelGGL((gemm_split_kernel<T, E, TBN, TBM, KS, NW, NS>), dim3(unsigned(tiles)), dim3(NW * kWave), 0, s, g);
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
