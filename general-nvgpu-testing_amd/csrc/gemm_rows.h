// c = a @ b^T where a has at most 64 rows (decoding: a handful of tokens through a wide projection).
//
// Bound: reading B once, from HBM or the last-level cache; and inside a CU the fills of LDS, 122 GB/s for whole lines.
// The tiled kernels leave both idle: 64 columns per workgroup make too few workgroups, and each pays a serial chain
// (barrier, LDS reads, MFMAs) of 145-190 ns per K tile.  Here a workgroup owns only 16 columns, its wavefronts deal the K
// tiles out among themselves, and each has a ring of LDS slots that nobody else reads: no barrier until the sums meet.
// A is fetched again by every workgroup (from L2), in groups of 8 rows so that a single token costs half as much as 16.
// Fragments straight from memory into registers were 2-3 times slower: 16 neighbouring lanes then touch 16 lines.
// Two slots per wavefront and several workgroups per CU beat one workgroup with long rings (4 x 4096 x 4096: 4.1 us with 8
// wavefronts of 2 slots, 4.6 with 5), as do 16 columns against 32 (5.0) or 64 (8.3).
//   bf16, us, tiled kernel -> this: 1 x 1024 x 9480 23.1 -> 5.3, 4 x 4096 x 4096 11.8 -> 4.1, 16 x 1024 x 16384
//   36.8 -> 11.5, 32 x 4096 x 4096 12.0 -> 7.4, 64 x 512 x 8192 20.1 -> 11.3, 64 x 64 x 512 3.6 -> 3.3.  Where B comes from
//   memory in every call: fp16 16 x 11008 x 4096 21.2 -> 19.7 (4.6 TB/s); out of the last-level cache 15.6 either way.
#pragma once

#include "gemm_kernel.h"

namespace beam {

// AG groups of 8 rows of A, CB blocks of 16 columns, NW wavefronts, S LDS slots of one K tile for each.
template <typename T, int AG, int CB, int NW, int S>
struct RowsTile {
  static constexpr int COLS = 16 * CB;
  static constexpr int MB = AG < 2 ? 1 : AG / 2;  // blocks of 16 rows
  static constexpr int LOADS = AG + 2 * CB;       // buffer loads (1 KiB: 8 rows of one 128-byte line) per K tile
  static constexpr int A_BYTES = MB * 16 * kRowBytes;  // (AG == 1: rows 8 .. 15 are never filled, and never stored)
  static constexpr int SLOT = A_BYTES + COLS * kRowBytes;
  static constexpr int LDS_BYTES = NW * S * SLOT;
  static constexpr int OUTS = MB * 16 * COLS;
  static_assert(AG == 1 || AG % 2 == 0, "rows in blocks of 16");
  static_assert(S >= 2 && (S - 1) * LOADS < 64, "vmcnt range");
  static_assert(2 * LDS_BYTES <= 160 * 1024 && OUTS * 4 <= S * SLOT, "two workgroups per CU; the sums reuse the ring");

  static __device__ __forceinline__ void run(const void* A, const void* B, void* C, int M, int N, int K, char* smem) {
    using Traits = ElemTraits<T>;
    using vec8 = typename Traits::vec8;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int col0 = (int)blockIdx.x * COLS;
    const int rows_b = N - col0 < COLS ? N - col0 : COLS;
    const __amdgpu_buffer_rsrc_t ra = make_rsrc(A, (unsigned)M * (unsigned)K * 2u);
    const __amdgpu_buffer_rsrc_t rb = make_rsrc((const T*)B + (size_t)col0 * K, (unsigned)rows_b * (unsigned)K * 2u);
    char* const ring = smem + wave * (S * SLOT);
    const int n_all = (K + kBK - 1) / kBK;
    const int n_tiles = (n_all - wave + NW - 1) / NW;  // tile t of this wavefront is tile t * NW + wave; may be 0

    // Lane l fetches chunk position l % 8 of row l / 8 of a group; the position holds chunk position ^ swizzle_of_row(row).
    int chunk[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) chunk[i] = ((lane & 7) ^ swizzle_of_row(i * 8 + (lane >> 3))) * 8;
    auto load_tile = [&](int t, int slot) __attribute__((always_inline)) {
      const int k0 = (t * NW + wave) * kBK;
      char* const dst = ring + slot * SLOT;
#pragma unroll
      for (int i = 0; i < (AG > 2 * CB ? AG : 2 * CB); ++i) {
        const int k = k0 + chunk[i & 1];
        // K % 8 == 0: a chunk exists whole or not at all.  Rows and chunks past the end arrive as zeros and touch no memory.
        const unsigned off = k < K ? ((unsigned)(i * 8 + (lane >> 3)) * (unsigned)K + (unsigned)k) * 2u : kOobOffset;
        if (i < 2 * CB)
          __builtin_amdgcn_raw_ptr_buffer_load_lds(rb, (__attribute__((address_space(3))) void*)(dst + A_BYTES + i * 1024), 16, (int)off, 0, 0, 0);
        if (i < AG)
          __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, (__attribute__((address_space(3))) void*)(dst + i * 1024), 16, (int)off, 0, 0, 0);
      }
    };
#pragma unroll
    for (int s = 0; s < S; ++s) load_tile(s, s);

    f32x4 acc[MB][CB];
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
      for (int j = 0; j < CB; ++j) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    int frag_off[2];
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) frag_off[kk] = lds_offset(lane & 15, 4 * kk + (lane >> 4));
    int slot = 0;
    for (int t = 0; t < n_tiles; ++t) {
      asm volatile("" ::: "memory");
      wait_vm_and_lds<(S - 1) * LOADS>();  // my fills of this tile have landed
      asm volatile("" ::: "memory");
      const char* const sa = ring + slot * SLOT;
      vec8 fa[2][MB], fb[2][CB];
#pragma unroll
      for (int kk = 0; kk < 2; ++kk) {
#pragma unroll
        for (int j = 0; j < CB; ++j) fb[kk][j] = *(const vec8*)(sa + A_BYTES + j * 16 * kRowBytes + frag_off[kk]);
#pragma unroll
        for (int i = 0; i < MB; ++i) fa[kk][i] = *(const vec8*)(sa + i * 16 * kRowBytes + frag_off[kk]);
      }
      asm volatile("" ::: "memory");
      wait_lds<0>();  // ... and are read: the slot is free
      __builtin_amdgcn_sched_barrier(0);
      load_tile(t + S, slot);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int kk = 0; kk < 2; ++kk)
#pragma unroll
        for (int i = 0; i < MB; ++i)
#pragma unroll
          for (int j = 0; j < CB; ++j) acc[i][j] = Traits::mfma(fb[kk][j], fa[kk][i], acc[i][j]);
      slot = slot + 1 == S ? 0 : slot + 1;
    }
    wait_vm_and_lds<0>();  // the empty fills of the last iterations must be gone before the ring is reused

    // Lane l of a block holds columns 4 * (l >> 4) .. + 3 of row l & 15.  The sums are added in the order of the wavefronts.
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
      for (int j = 0; j < CB; ++j) *(f32x4*)(ring + ((i * CB + j) * 64 + lane) * 16) = acc[i][j];
    __syncthreads();
    for (int o = threadIdx.x; o < OUTS; o += NW * 64) {
      const int c = o % COLS, m = o / COLS;
      const int n = col0 + c;
      if (m >= M || n >= N) continue;
      const int at = ((m >> 4) * CB + (c >> 4)) * 256 + ((m & 15) + 16 * ((c & 15) >> 2)) * 4 + (c & 3);
      float part[NW];
#pragma unroll
      for (int w = 0; w < NW; ++w) part[w] = ((const float*)(smem + w * (S * SLOT)))[at];
      float v = part[0];
#pragma unroll
      for (int w = 1; w < NW; ++w) v += part[w];
      ((T*)C)[(size_t)m * N + n] = (T)v;
    }
  }
};

template <typename T, int AG, int CB, int NW, int S>
__global__ void __launch_bounds__(NW * 64, 2) gemm_rows_kernel(const void* A, const void* B, void* C, int M, int N, int K) {
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  RowsTile<T, AG, CB, NW, S>::run(A, B, C, M, N, K, smem);
}

}  // namespace beam
