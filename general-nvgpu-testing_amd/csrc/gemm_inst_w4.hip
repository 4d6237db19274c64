// The 256x256 tile of four 128x128 wavefronts (gemm_w4.h), fp16 and bf16.
#include "gemm_w4.h"
#include "kernel_set.h"

namespace beam {

template <typename T, int STORE, bool LN = false>
static hipError_t launch_w4_t(const GemmParams& p, dim3 grid, hipStream_t stream) {
  auto kern = gemmrc_w4_kernel<T, STORE, LN>;
  static std::atomic<unsigned long long> configured{0};
  if (hipError_t e = allow_lds_once(configured, reinterpret_cast<const void*>(kern), GemmW4<T>::LDS_BYTES); e != hipSuccess) return e;
  hipLaunchKernelGGL(kern, grid, dim3(GemmW4<T>::NT), GemmW4<T>::LDS_BYTES, stream, p);
  return hipGetLastError();
}

template <typename T>
static hipError_t launch_w4_kind(const GemmParams& p, dim3 grid, hipStream_t stream) {
  if (p.c_store == kStoreStreaming) return launch_w4_t<T, kStoreStreaming>(p, grid, stream);
  return p.c_store == kStoreCached ? launch_w4_t<T, kStoreCached>(p, grid, stream) : launch_w4_t<T, kStoreThrough>(p, grid, stream);
}

hipError_t launch_gemm_w4(const GemmParams& p, int dtype, dim3 grid, hipStream_t stream) {
  return dtype == BEAM_BF16 ? launch_w4_kind<__bf16>(p, grid, stream) : launch_w4_kind<_Float16>(p, grid, stream);
}

static_assert(kW4LnCompactTiles == GemmW4<_Float16, kStoreThrough, true>::kLnCompactTiles, "the host's bound is the kernel's");

template <typename T>
static hipError_t launch_w4_ln_kind(const GemmParams& p, dim3 grid, hipStream_t stream) {
  return p.c_store == kStoreCached ? launch_w4_t<T, kStoreCached, true>(p, grid, stream) : launch_w4_t<T, kStoreThrough, true>(p, grid, stream);
}

hipError_t launch_gemm_w4_ln(const GemmParams& p, int dtype, dim3 grid, hipStream_t stream) {
  return dtype == BEAM_BF16 ? launch_w4_ln_kind<__bf16>(p, grid, stream) : launch_w4_ln_kind<_Float16>(p, grid, stream);
}

}  // namespace beam
