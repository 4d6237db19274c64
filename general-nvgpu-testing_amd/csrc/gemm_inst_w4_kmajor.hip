// The 256x256 tile of four 128x128 wavefronts (gemm_w4.h) with B stored [K][N], fp16 and bf16.
#include "gemm_w4.h"
#include "kernel_set.h"

namespace beam {

template <typename T, int STORE>
static hipError_t launch_w4_kmajor_t(const GemmParams& p, dim3 grid, hipStream_t stream) {
  using Tile = GemmW4<T, STORE, false, 4, 8, 2, true>;
  auto kern = gemmrc_w4_kernel<T, STORE, false, 4, 8, 2, true>;
  static std::atomic<unsigned long long> configured{0};
  if (hipError_t e = allow_lds_once(configured, reinterpret_cast<const void*>(kern), Tile::LDS_BYTES); e != hipSuccess) return e;
  hipLaunchKernelGGL(kern, grid, dim3(Tile::NT), Tile::LDS_BYTES, stream, p);
  return hipGetLastError();
}

template <typename T>
static hipError_t launch_w4_kmajor_kind(const GemmParams& p, dim3 grid, hipStream_t stream) {
  if (p.c_store == kStoreStreaming) return launch_w4_kmajor_t<T, kStoreStreaming>(p, grid, stream);
  return p.c_store == kStoreCached ? launch_w4_kmajor_t<T, kStoreCached>(p, grid, stream) : launch_w4_kmajor_t<T, kStoreThrough>(p, grid, stream);
}

hipError_t launch_gemm_w4_kmajor(const GemmParams& p, int dtype, dim3 grid, hipStream_t stream) {
  return dtype == BEAM_BF16 ? launch_w4_kmajor_kind<__bf16>(p, grid, stream) : launch_w4_kmajor_kind<_Float16>(p, grid, stream);
}

}  // namespace beam
