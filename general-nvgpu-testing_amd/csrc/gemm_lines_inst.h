// The tiles of gemm_kernel.h whose fills take whole 128-byte lines, and their launcher, for one element type (BEAM_T).
#include "kernel_set.h"

namespace beam {

template <int EPI, int BM, int BN, int WVM, int WVN, int AST, int BST, bool B_KMAJOR, int KG, int FORM>
static hipError_t launch_lines_t(const GemmParams& p, dim3 grid, hipStream_t stream) {
  using Tile = GemmTile<BEAM_T, BM, BN, WVM, WVN, EPI, AST, BST, B_KMAJOR, KG, FORM>;
  auto kern = gemmrc_kernel<BEAM_T, BM, BN, WVM, WVN, EPI, AST, BST, B_KMAJOR, KG, FORM>;
  static std::atomic<unsigned long long> configured{0};
  constexpr int LDS = Tile::GROUPS * Tile::LDS_BYTES;
  if (hipError_t e = allow_lds_once(configured, reinterpret_cast<const void*>(kern), LDS); e != hipSuccess) return e;
  hipLaunchKernelGGL(kern, grid, dim3(KG * Tile::NT), LDS, stream, p);
  return hipGetLastError();
}

template <int EPI>
static hipError_t launch_lines_tile(int block_m, int block_n, const GemmParams& p, dim3 grid, hipStream_t stream) {
  // (LayerNorm never comes here with 64 x 64 tiles: gemm_kwave.h has them up to 256, and 96 x 64 is ahead beyond)
#define BEAM_LINES(BM, BN, S, KG, FORM)                                \
  if constexpr (EPI != kEpiLnFused || BM * BN > 64 * 64)               \
    if (block_m == BM && block_n == BN) return launch_lines_t<EPI, BM, BN, 2, 2, S, S, false, KG, FORM>(p, grid, stream);
  BEAM_FOR_EACH_LINES_TILE(BEAM_LINES)
#undef BEAM_LINES
  return hipErrorInvalidValue;
}

template <>
hipError_t launch_gemm_lines<BEAM_T>(int block_m, int block_n, const GemmParams& p, dim3 grid, hipStream_t stream) {
  return launch_lines_tile<kEpiStore>(block_m, block_n, p, grid, stream);
}

template <>
hipError_t launch_gemm_lines_kmajor<BEAM_T>(int block_m, int block_n, const GemmParams& p, dim3 grid, hipStream_t stream) {
#define BEAM_LINES(BM, BN, WVM, WVN, S, KG, FORM) \
  if (block_m == BM && block_n == BN) return launch_lines_t<kEpiStore, BM, BN, WVM, WVN, S + 1, S, true, KG, FORM>(p, grid, stream);
  BEAM_FOR_EACH_KMAJOR_LINES_TILE(BEAM_LINES)
#undef BEAM_LINES
  return hipErrorInvalidValue;
}

template <>
hipError_t launch_gemm_lines_ln<BEAM_T>(int block_m, int block_n, const GemmParams& p, dim3 grid, hipStream_t stream) {
  return launch_lines_tile<kEpiLnFused>(block_m, block_n, p, grid, stream);
}

}  // namespace beam
