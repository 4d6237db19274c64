// Instances of the few-row kernel (gemm_rows.h) and the choice among them.
#include "gemm_rows.h"
#include "kernel_set.h"

namespace beam {

namespace {

template <typename T, int AG, int CB, int NW, int S>
hipError_t launch_rows(const void* A, const void* B, void* C, int M, int N, int K, hipStream_t stream) {
  using Tile = RowsTile<T, AG, CB, NW, S>;
  auto kern = gemm_rows_kernel<T, AG, CB, NW, S>;
  static std::atomic<unsigned long long> configured{0};
  if (hipError_t e = allow_lds_once(configured, reinterpret_cast<const void*>(kern), Tile::LDS_BYTES); e != hipSuccess) return e;
  hipLaunchKernelGGL(kern, dim3((unsigned)((N + Tile::COLS - 1) / Tile::COLS)), dim3(NW * 64), Tile::LDS_BYTES, stream, A, B, C, M, N, K);
  return hipGetLastError();
}

// The fewest row groups that hold M: every one more is fetched with each workgroup's columns of B.
template <typename T>
hipError_t launch_typed(RowsPlan plan, const void* A, const void* B, void* C, int M, int N, int K, hipStream_t stream) {
  switch (plan) {
    case kRowsNone: break;
    case kRowsNarrow:
      if (M <= 8) return launch_rows<T, 1, 1, 8, 2>(A, B, C, M, N, K, stream);
      if (M <= 16) return launch_rows<T, 2, 1, 8, 2>(A, B, C, M, N, K, stream);
      if (M <= 32) return launch_rows<T, 4, 1, 4, 3>(A, B, C, M, N, K, stream);
      if (M <= 64) return launch_rows<T, 8, 1, 4, 2>(A, B, C, M, N, K, stream);
      break;
    case kRowsDeep:
      if (M <= 8) return launch_rows<T, 1, 1, 4, 2>(A, B, C, M, N, K, stream);
      if (M <= 16) return launch_rows<T, 2, 1, 4, 2>(A, B, C, M, N, K, stream);
      break;
    case kRowsWide:
      if (M <= 8) return launch_rows<T, 1, 4, 4, 2>(A, B, C, M, N, K, stream);
      if (M <= 16) return launch_rows<T, 2, 4, 4, 2>(A, B, C, M, N, K, stream);
      if (M <= 32) return launch_rows<T, 4, 2, 4, 2>(A, B, C, M, N, K, stream);
      break;
  }
  return hipErrorInvalidValue;
}

}  // namespace

hipError_t launch_gemm_rows(RowsPlan plan, const void* A, const void* B, void* C, int M, int N, int K, int dtype, hipStream_t stream) {
  if (M < 1 || N < 1 || K < 8 || K % 8 != 0 || K > kRowsMaxK) return hipErrorInvalidValue;
  return dtype == 0 ? launch_typed<_Float16>(plan, A, B, C, M, N, K, stream) : launch_typed<__bf16>(plan, A, B, C, M, N, K, stream);
}

}  // namespace beam
