// Instances of the kernel of gemm_kwave.h for one element type (KW_T), and the choice among them.  Included by
// gemm_kwave_{fp16,bf16}.hip.
#include "gemm_kwave.h"
#include "kernel_set.h"

namespace beam {

namespace {

template <int AG, int CB, int NW, int S, KwRows MODE, bool KMAJOR>
hipError_t launch_plain(const KwParams& p, hipStream_t stream) {
  using Tile = KwTile<KW_T, AG, CB, NW, S, MODE, KMAJOR>;
  auto kern = gemm_kwave_kernel<KW_T, AG, CB, NW, S, MODE, KMAJOR>;
  static std::atomic<unsigned long long> configured{0};
  if (hipError_t e = allow_lds_once(configured, reinterpret_cast<const void*>(kern), Tile::LDS_BYTES); e != hipSuccess) return e;
  hipLaunchKernelGGL(kern, dim3((unsigned)(p.tiles_m * p.tiles_n)), dim3(NW * 64), Tile::LDS_BYTES, stream, p);
  return hipGetLastError();
}

template <int AG, int CB, int NW, int S, KwRows MODE>
hipError_t launch_ln(const KwLnParams& p, hipStream_t stream) {
  using Tile = KwTile<KW_T, AG, CB, NW, S, MODE, false>;
  auto kern = gemm_kwave_ln_kernel<KW_T, AG, CB, NW, S, MODE>;
  static std::atomic<unsigned long long> configured{0};
  if (hipError_t e = allow_lds_once(configured, reinterpret_cast<const void*>(kern), Tile::LDS_BYTES); e != hipSuccess) return e;
  hipLaunchKernelGGL(kern, dim3((unsigned)(p.tiles_m * p.tiles_n)), dim3(NW * 64), Tile::LDS_BYTES, stream, p);
  return hipGetLastError();
}

// Whole-line fills are for tiles above 8 rows whose K tiles x (rows + columns) are 1200 and more (kw_plan): with 16 x 16 that is
// from K = 2400 on, where a workgroup has eight wavefronts.
template <int AG, int CB, int NW>
constexpr bool kShifts = AG > 1 && !(AG == 2 && CB == 1 && NW == 4);

template <int AG, int CB, int NW>
hipError_t launch_tile(const KwPlan& plan, const KwParams& p, bool b_kmajor, hipStream_t stream) {
  if (plan.shift) {
    if constexpr (kShifts<AG, CB, NW>)
      return b_kmajor ? launch_plain<AG, CB, NW, 2, kKwShift, true>(p, stream) : launch_plain<AG, CB, NW, 2, kKwShift, false>(p, stream);
    else
      return hipErrorInvalidValue;
  }
  if (b_kmajor) {
    if constexpr (AG > 1)
      return launch_plain<AG, CB, NW, 2, kKwStraight, true>(p, stream);
    else
      return hipErrorInvalidValue;
  }
  return launch_plain<AG, CB, NW, 2, kKwStraight, false>(p, stream);
}

template <int AG, int CB, int NW, KwRows MODE>
hipError_t launch_side(const KwSideParams& p, int side_workgroups, hipStream_t stream) {
  using Tile = KwTile<KW_T, AG, CB, NW, 2, MODE, false>;
  auto kern = gemm_kwave_side_kernel<KW_T, AG, CB, NW, 2, MODE>;
  static std::atomic<unsigned long long> configured{0};
  if (hipError_t e = allow_lds_once(configured, reinterpret_cast<const void*>(kern), Tile::LDS_BYTES); e != hipSuccess) return e;
  hipLaunchKernelGGL(kern, dim3((unsigned)(p.tiles_m * p.tiles_n + side_workgroups)), dim3(NW * 64), Tile::LDS_BYTES, stream, p);
  return hipGetLastError();
}

template <int AG, int CB, int NW>
hipError_t launch_tile_side(const KwPlan& plan, const KwSideParams& p, int side_workgroups, hipStream_t stream) {
  if (plan.shift) {
    if constexpr (kShifts<AG, CB, NW>)
      return launch_side<AG, CB, NW, kKwShift>(p, side_workgroups, stream);
    else
      return hipErrorInvalidValue;
  }
  return launch_side<AG, CB, NW, kKwStraight>(p, side_workgroups, stream);
}

template <int AG, int CB>
hipError_t launch_tile_ln(const KwPlan& plan, const KwLnParams& p, hipStream_t stream) {
  return plan.shift ? launch_ln<AG, CB, 4, 2, kKwShift>(p, stream) : launch_ln<AG, CB, 4, 2, kKwStraight>(p, stream);
}

}  // namespace

template <>
hipError_t launch_gemm_kwave<KW_T>(const KwPlan& plan, const KwParams& p, bool b_kmajor, hipStream_t stream) {
  switch (plan.rows * 256 + plan.cols) {
    case 8 * 256 + 16: return plan.waves == 8 ? launch_tile<1, 1, 8>(plan, p, b_kmajor, stream) : launch_tile<1, 1, 4>(plan, p, b_kmajor, stream);
    case 16 * 256 + 16: return plan.waves == 8 ? launch_tile<2, 1, 8>(plan, p, b_kmajor, stream) : launch_tile<2, 1, 4>(plan, p, b_kmajor, stream);
    case 8 * 256 + 64: return launch_tile<1, 4, 4>(plan, p, b_kmajor, stream);
    case 16 * 256 + 64: return launch_tile<2, 4, 4>(plan, p, b_kmajor, stream);
    case 16 * 256 + 32: return launch_tile<2, 2, 4>(plan, p, b_kmajor, stream);
    case 32 * 256 + 16: return launch_tile<4, 1, 4>(plan, p, b_kmajor, stream);
    case 32 * 256 + 32: return launch_tile<4, 2, 4>(plan, p, b_kmajor, stream);
    case 32 * 256 + 64: return launch_tile<4, 4, 4>(plan, p, b_kmajor, stream);
    case 64 * 256 + 32: return launch_tile<8, 2, 4>(plan, p, b_kmajor, stream);
    case 64 * 256 + 64: return launch_tile<8, 4, 4>(plan, p, b_kmajor, stream);
  }
  return hipErrorInvalidValue;
}

template <>
hipError_t launch_gemm_kwave_side<KW_T>(const KwPlan& plan, const KwSideParams& p, int side_workgroups, hipStream_t stream) {
  const int n = side_workgroups;
  switch (plan.rows * 256 + plan.cols) {
    case 8 * 256 + 16: return plan.waves == 8 ? launch_tile_side<1, 1, 8>(plan, p, n, stream) : launch_tile_side<1, 1, 4>(plan, p, n, stream);
    case 16 * 256 + 16: return plan.waves == 8 ? launch_tile_side<2, 1, 8>(plan, p, n, stream) : launch_tile_side<2, 1, 4>(plan, p, n, stream);
    case 8 * 256 + 64: return launch_tile_side<1, 4, 4>(plan, p, n, stream);
    case 16 * 256 + 64: return launch_tile_side<2, 4, 4>(plan, p, n, stream);
    case 16 * 256 + 32: return launch_tile_side<2, 2, 4>(plan, p, n, stream);
    case 32 * 256 + 16: return launch_tile_side<4, 1, 4>(plan, p, n, stream);
    case 32 * 256 + 32: return launch_tile_side<4, 2, 4>(plan, p, n, stream);
    case 32 * 256 + 64: return launch_tile_side<4, 4, 4>(plan, p, n, stream);
    case 64 * 256 + 32: return launch_tile_side<8, 2, 4>(plan, p, n, stream);
    case 64 * 256 + 64: return launch_tile_side<8, 4, 4>(plan, p, n, stream);
  }
  return hipErrorInvalidValue;
}

template <>
hipError_t launch_gemm_kwave_ln<KW_T>(const KwPlan& plan, const KwLnParams& p, hipStream_t stream) {
  switch (plan.rows * 256 + plan.cols) {
    case 16 * 256 + 16: return launch_tile_ln<2, 1>(plan, p, stream);
    case 16 * 256 + 32: return launch_tile_ln<2, 2>(plan, p, stream);
    case 32 * 256 + 16: return launch_tile_ln<4, 1>(plan, p, stream);
    case 32 * 256 + 32: return launch_tile_ln<4, 2>(plan, p, stream);
    case 16 * 256 + 64: return launch_tile_ln<2, 4>(plan, p, stream);
    case 32 * 256 + 64: return launch_tile_ln<4, 4>(plan, p, stream);
    case 64 * 256 + 32: return launch_tile_ln<8, 2>(plan, p, stream);
    case 64 * 256 + 64: return launch_tile_ln<8, 4>(plan, p, stream);
  }
  return hipErrorInvalidValue;
}

}  // namespace beam
