// c = a @ b^T (or a @ b with B stored [K][N]) in small workgroup tiles whose K range is dealt out to the wavefronts.
//
// What a problem of few output tiles pays in the tiled kernels (gemm_kernel.h) is a serial chain per K tile -- barrier, LDS
// reads, MFMAs: 145-190 ns -- on the few CUs that have a tile at all.  Here a workgroup owns at most 64 x 64 outputs, so that
// there are many workgroups, and every wavefront multiplies a part of K for the whole tile with a ring of LDS slots that
// nobody else reads: no barrier until the fp32 sums meet in LDS, added in the wavefronts' order.
//
// Bound: LDS fills, (rows + columns) x K of a CU's tile at up to 122 GB/s.  That rate is one 128-byte line per two clocks,
// whether a fill uses the whole line or a part of it.  A row whose K elements do not start on a line (K % 64 != 0) has every
// 128-byte K tile in two lines, half the rate.  So for a long K a fill takes whole lines of memory, whatever K elements those
// are (kKwShift): in slot t a row's chunks c < 8 - phase (phase: 16-byte chunks between the line's start and the row's K tile)
// belong to K tile t and the others, which sit in the same line in front of them, to K tile t - 1.  A chunk keeps its place in
// the slot; a fragment of K tile t - 1 is then slot t's in the lanes that read a late chunk and slot t - 1's, kept in
// registers, in the others: one select per register, between MFMAs that leave the vector unit idle three quarters of the time.
// Any phase gives the right result; the right one gives one line per row and K tile.  Same machine, us, straight -> shifted:
// 1000 x 1000 x 8184 43.7 -> 32.7, 466 x 864 x 1032 6.6 -> 6.1; 466 x 864 x 520 5.0 -> 5.1 (each wavefront has one fill more).
//
// us, the tiled kernels -> this: 256 x 256 x 4096 12.8 -> 5.7, x 8184 21.8 -> 7.6, 233 x 1416 x 1832 10.7 -> 7.4, 1284 x 80 x
// 5464 25.8 -> 8.6, 1024 x 1024 x 4088 19.5 -> 16.7; [K][N] 512 x 768 x 4096 16.6 -> 11.4, 16 x 4096 x 4096
// 16.2 -> 11.2, 1284 x 80 x 5464 22.0 -> 12.5.  A handful of rows (which had a kernel of this kind for themselves, 16 columns,
// straight): 4 x 4096 x 4096 7.9 -> 6.9, 64 x 4096 x 4096 10.4 -> 8.3, 16 x 8192 x 8192 33.0 -> 27.5.
// Two slots and four wavefronts are the best of 1-4 slots and 2-16 wavefronts nearly everywhere (466 x 864 x 600: 5.2 us, 5.5
// with 3 slots, 5.7 with 8 wavefronts of one); fragments straight from memory into registers were 2-3 times slower, since
// 16 neighbouring lanes then touch 16 lines.
#pragma once

#include "gemm_kernel.h"

namespace beam {

struct KwParams {
  const void* A;
  const void* B;
  void* C;
  int M, N, K;
  int tiles_m, tiles_n, group_m;
  TileDivs divs;
};

// How the fills take K elements.
enum KwRows : int {
  kKwStraight = 0,  // a K tile's 128 bytes of a row as they lie
  kKwShift = 1,     // whole lines of memory
};

// With an elementwise job y[i] = silu(x[i]) for the workgroups behind the tiles' in the same grid.
struct KwSideParams : KwParams {
  const void* side_x;
  void* side_y;
  long long side_count;
};

// GEMM+LayerNorm: the exchange of gemm_kernel.h, workgroups in one of the orders without padding.
struct KwLnParams : KwParams {
  float* stats;  // 8-byte words [tiles_m][tiles_n][ROWS] = (mean, tag)
  float* next_stats;  // ... = (M2, ~tag)
  int* timeout_flag;
  unsigned* host_timeout;
  const void* gamma;
  const void* beta;
  unsigned ln_nonce;
  float eps;
  int spin_limit;
};

// Column tiles of a band that stays together on an XCD.  A launch that shares the device and gets s of an XCD's 32 CUs still
// finishes band by band if s is at least this many: XCD 0 starts with a whole band, and each XCD's last band is what
// the next one's first workgroups wait for.  (Longer bands, and groups of bands, are up to 64 workgroups in id order: room for 8
// of them on every XCD does, and 64 CUs of some XCDs do not.)  Two launches that wait may each hold the XCDs that the other one
// needs, since the XCDs start launches independently: 512 x 1024 x 256 and 64 x 4096 x 136 have 256 workgroups each, of 96 and
// 80 KiB of LDS.  The waits' bound then ends it.
constexpr int kKwLnShortBand = 8;

// Sum over W (4, 8 or 16) neighbouring lanes, the same bits in each of them.
template <int W>
__device__ __forceinline__ float lanes_sum(float x) {
  static_assert(W == 4 || W == 8 || W == 16, "a row of 16 lanes at most");
  auto add = [](float v, auto ctrl) __attribute__((always_inline)) {
    return v + __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), decltype(ctrl)::value, 0xf, 0xf, true));
  };
  x = add(x, std::integral_constant<int, 0xB1>{});                           // quad_perm 1 0 3 2
  x = add(x, std::integral_constant<int, 0x4E>{});                           // quad_perm 2 3 0 1
  if constexpr (W >= 8) x = add(x, std::integral_constant<int, 0x141>{});   // row_half_mirror
  if constexpr (W >= 16) x = add(x, std::integral_constant<int, 0x140>{});  // row_mirror
  return x;
}

// K-major B slots (64 rows of k, COLS columns): the 16-byte chunk position of chunk c of row k, for conflict-free transposing
// reads (tile_map.h: kmajor_swizzle).  64 columns: that layout.  32 columns: four rows to a bank sweep, the segment XORed
// with bit 3 of k.  16 columns: eight rows to a sweep, and rows 4 .. 7 and 8 .. 11 of every 16 change places.
BEAM_HD int kw_kmajor_row(int k, int cols) { return cols == 16 ? (k & ~12) | ((k & 4) << 1) | ((k & 8) >> 1) : k; }
BEAM_HD int kw_kmajor_swizzle(int k, int cols) { return cols == 64 ? kmajor_swizzle(k, 64) : (cols == 32 ? ((k >> 3) & 1) << 1 : 0); }
BEAM_HD int kw_kmajor_offset(int k, int n, int cols) {
  return kw_kmajor_row(k, cols) * cols * 2 + (((n >> 3) ^ kw_kmajor_swizzle(k, cols)) << 4) + ((n & 7) << 1);
}

// AG groups of 8 rows of A, CB blocks of 16 columns, NW wavefronts, S LDS slots of one K tile for each.
template <typename T, int AG, int CB, int NW, int S, KwRows MODE, bool KMAJOR>
struct KwTile {
  using Traits = ElemTraits<T>;
  using vec8 = typename Traits::vec8;
  using vec4 = typename Traits::vec4;
  static constexpr bool SHIFT = MODE == kKwShift;
  static constexpr int MB = AG < 2 ? 1 : AG / 2;  // blocks of 16 rows
  static constexpr int ROWS = AG * 8;
  static constexpr int COLS = 16 * CB;
  static constexpr int NT = NW * 64;
  static constexpr int LB = 2 * CB;
  static constexpr int LOADS = AG + LB;                // buffer loads of 1 KiB per K tile
  static constexpr int A_BYTES = MB * 16 * kRowBytes;  // (AG == 1: rows 8 .. 15 are never filled, and never stored)
  static constexpr int SLOT = A_BYTES + COLS * kRowBytes;
  static constexpr int LDS_BYTES = NW * S * SLOT;
  static constexpr int CG = COLS / 4;            // groups of 4 columns in a row
  static constexpr int QUADS = MB * 16 * CG;     // of the tile
  static constexpr int SUM_BYTES = QUADS * 16;   // one wavefront's fp32 sums
  static_assert(AG == 1 || AG % 2 == 0, "rows in blocks of 16");
  static_assert(S >= 1 && (S - 1) * LOADS < 64, "vmcnt range");
  static_assert(LDS_BYTES <= 160 * 1024 && SUM_BYTES <= S * SLOT, "LDS; the sums reuse the ring");
  static_assert(CG == 4 || CG == 8 || CG == 16, "sum layout");

  // Where the four sums of (row, column group) lie: 16 rows of one column group (what a store of a block writes) and 16
  // neighbouring column groups or rows (what a thread's neighbours read) are 16 different 16-byte slots of a bank sweep.
  static __device__ __forceinline__ int sum_slot(int row, int cg) { return row * CG + (cg ^ ((row / (16 / CG)) & (CG - 1))); }

  // The K loop: this wavefront's share of the tile at (row0, col0), added up in acc.
  static __device__ __forceinline__ void multiply(const KwParams& p, int row0, int col0, int wave, int lane, char* ring, f32x4 (&acc)[MB][CB]) {
    const int M = p.M, N = p.N, K = p.K;
    const int rows_a = M - row0 < ROWS ? M - row0 : ROWS;
    const int rows_b = N - col0 < COLS ? N - col0 : COLS;
    // Whole chunks of 8 elements, and up to 8 that come last.  K-major rows that are not whole chunks: the very last row is
    // always among those, so that every row that is fetched has another one behind it and may be read past its end.
    const bool n_odd = KMAJOR && (N & 7) != 0;
    const int k8 = (K - (n_odd ? 1 : 0)) >> 3, rem = K - 8 * k8;
    const int n_all = (k8 + 7) >> 3;       // K tiles
    // This wavefront's K tiles are t0, t0 + EVERY, ...; may be none.  Shifted, a part of K in one piece (K tile t + 1's line
    // holds chunks of K tile t); straight, every NW-th.
    constexpr int EVERY = SHIFT ? 1 : NW;
    const int t0 = SHIFT ? wave * n_all / NW : wave;
    const int n = SHIFT ? (wave + 1) * n_all / NW - t0 : (n_all - wave + NW - 1) / NW;
    const T* const a_base = (const T*)p.A + (size_t)row0 * K;
    const T* const b_base = KMAJOR ? (const T*)p.B + col0 : (const T*)p.B + (size_t)col0 * K;
    // The shifted fills count from one line in front of the rows, so that no chunk's offset is negative.
    constexpr int LEAD = SHIFT ? kRowBytes : 0;
    const __amdgpu_buffer_rsrc_t ra = make_rsrc((const char*)a_base - LEAD, (unsigned)rows_a * (unsigned)K * 2u + LEAD);
    const __amdgpu_buffer_rsrc_t rb = make_rsrc((const char*)b_base - LEAD, KMAJOR ? 0u : (unsigned)rows_b * (unsigned)K * 2u + LEAD);
    const unsigned row_bytes = (unsigned)K * 2u;
    // chunks between the start of row r's first line and the row (rows 16 apart share it: exact for K % 4 == 0)
    auto phase_of = [&](const T* base, int r) __attribute__((always_inline)) {
      return SHIFT ? (int)(((unsigned)(size_t)base + (unsigned)r * row_bytes) & 127u) >> 4 : 0;
    };

    // Lane l fetches chunk position l % 8 of row l / 8 of a group; the position holds chunk position ^ swizzle_of_row(row).
    // For each of the two groups of a block: the chunk's offset in K tile 0, and the fills that bring one that exists.
    struct Lane {
      unsigned off;
      int first;       // the first fill with a chunk of this wavefront
      unsigned count;  // ... and how many there are
    };
    auto lane_of = [&](const T* base, int cls) __attribute__((always_inline)) {
      Lane f;
      const int r = cls * 8 + (lane >> 3);
      const int c = (lane & 7) ^ swizzle_of_row(r);
      const bool late = SHIFT && c + phase_of(base, r) >= 8;
      f.off = LEAD + (unsigned)r * row_bytes + (unsigned)(c - (late ? 8 : 0)) * 16u;
      f.first = late ? 1 : 0;
      int cnt = (k8 - 8 * t0 - c + 8 * EVERY - 1) / (8 * EVERY);
      cnt = cnt < n ? cnt : n;
      f.count = (unsigned)(cnt > 0 ? cnt : 0);
      return f;
    };
    const Lane la0 = lane_of(a_base, 0), la1 = lane_of(a_base, 1);
    const Lane lb0 = lane_of(b_base, 0), lb1 = lane_of(b_base, 1);
    // K-major B: chunk position q of a slot is row k = q / CPR (after kw_kmajor_row, its own inverse), chunk q % CPR ^ swizzle
    constexpr int CPR = COLS / 8;
    unsigned voff_b[LB];
    if constexpr (KMAJOR) {
#pragma unroll
      for (int i = 0; i < LB; ++i) {
        const int q = i * 64 + lane;
        const int k = kw_kmajor_row(q / CPR, COLS);
        voff_b[i] = ((unsigned)k * (unsigned)N + (unsigned)((q % CPR) ^ kw_kmajor_swizzle(k, COLS)) * 8u) * 2u;
      }
    }
    auto fill = [&](int t, int slot) __attribute__((always_inline)) {
      char* const dst = ring + slot * SLOT;
      const unsigned k_off = (unsigned)(t0 + t * EVERY) * kRowBytes;
      auto off_of = [&](const Lane& f, int i) __attribute__((always_inline)) {
        const unsigned off = f.off + (k_off + (unsigned)(i >> 1) * 16u * row_bytes);
        return (int)((unsigned)(t - f.first) < f.count ? off : kOobOffset);
      };
      if constexpr (KMAJOR) {
        // with shifted rows of A, K tile t - 1 is multiplied when fill t has arrived
        const int koff = (t0 + (SHIFT ? t - 1 : t * EVERY)) * kBK;
        const bool exists = SHIFT ? t >= 1 && t <= n : t < n;
        // (not the rows behind the whole chunks: those of A are zeros there, and zero times infinity is not)
        const int rows = 8 * k8 - koff < kBK ? 8 * k8 - koff : kBK;
        // (columns past N in the rows in front of the last read the next row's data and feed outputs that do not exist)
        // The range check works on whole dwords from a lane's own offset: an odd last column needs the element behind it in range,
        // and that one alone is no whole dword of the row behind, which starts there.  (Telling the lanes of that row instead, by
        // selects or by a branch in the loop, cost 0.5-1.4%: 288 x 448 x 4432 9.54 -> 9.67 and 9.59 us.)
        const __amdgpu_buffer_rsrc_t rk = make_rsrc(b_base + (exists ? (size_t)koff * N : 0), exists ? ((unsigned)(rows - 1) * (unsigned)N + (unsigned)(N - col0) + (unsigned)(N & 1)) * 2u : 0u);
#pragma unroll
        for (int i = 0; i < LB; ++i)
          __builtin_amdgcn_raw_ptr_buffer_load_lds(rk, (__attribute__((address_space(3))) void*)(dst + A_BYTES + i * 1024), 16, (int)voff_b[i], 0, 0, 0);
      } else {
#pragma unroll
        for (int i = 0; i < LB; ++i)
          __builtin_amdgcn_raw_ptr_buffer_load_lds(rb, (__attribute__((address_space(3))) void*)(dst + A_BYTES + i * 1024), 16, off_of(i & 1 ? lb1 : lb0, i), 0, 0, 0);
      }
#pragma unroll
      for (int i = 0; i < AG; ++i)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, (__attribute__((address_space(3))) void*)(dst + i * 1024), 16, off_of(i & 1 ? la1 : la0, i), 0, 0, 0);
    };

    const int fills = n > 0 ? (SHIFT ? n + 1 : n) : 0;
    if (fills > 0) {
#pragma unroll
      for (int s = 0; s < S; ++s) fill(s, s);
    }

    // Fragments: lane l reads row l & 15, chunk 4 * kk + (l >> 4) of a block.
    int frag_off[2];
    bool late_a[2], late_b[2];
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      const int c = 4 * kk + (lane >> 4);
      frag_off[kk] = lds_offset(lane & 15, c);
      late_a[kk] = SHIFT && c + phase_of(a_base, lane & 15) >= 8;
      late_b[kk] = SHIFT && !KMAJOR && c + phase_of(b_base, lane & 15) >= 8;
    }
    int bfrag_off[CB];
    if constexpr (KMAJOR) {
#pragma unroll
      for (int j = 0; j < CB; ++j)
        bfrag_off[j] = A_BYTES + kw_kmajor_offset(8 * (lane >> 4) + ((lane >> 2) & 3), j * 16 + 4 * (lane & 3), COLS);
    }
    struct Frags {
      vec8 a[2][MB], b[2][CB];
    };
    // Waits for fill t, reads its fragments and hands the slot on to fill t + S.
    auto take = [&](Frags& f, int t, int slot) __attribute__((always_inline)) {
      asm volatile("" ::: "memory");
      wait_vm_and_lds<(S - 1) * LOADS>();
      asm volatile("" ::: "memory");
      const char* const sa = ring + slot * SLOT;
#pragma unroll
      for (int kk = 0; kk < 2; ++kk) {
#pragma unroll
        for (int j = 0; j < CB; ++j) {
          if constexpr (KMAJOR) {
            // (inline assembly, waited for below: through the intrinsic the compiler orders such reads behind every fill)
            const unsigned addr = (unsigned)(size_t)(__attribute__((address_space(3))) const char*)(sa + bfrag_off[j]);
            constexpr int FOUR_ROWS = (COLS == 16 ? 8 : 4) * COLS * 2, HALF = 32 * COLS * 2;
            vec4 lo, hi;
            if (kk == 0) {
              asm volatile("ds_read_b64_tr_b16 %0, %1" : "=v"(lo) : "v"(addr));
              asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(hi) : "v"(addr), "n"(FOUR_ROWS));
            } else {
              asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(lo) : "v"(addr), "n"(HALF));
              asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(hi) : "v"(addr), "n"(HALF + FOUR_ROWS));
            }
            f.b[kk][j] = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
          } else {
            f.b[kk][j] = *(const vec8*)(sa + A_BYTES + j * 16 * kRowBytes + frag_off[kk]);
          }
        }
#pragma unroll
        for (int i = 0; i < MB; ++i) f.a[kk][i] = *(const vec8*)(sa + i * 16 * kRowBytes + frag_off[kk]);
      }
      asm volatile("" ::: "memory");
      wait_lds<0>();  // ... and they are read: the slot is free
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (KMAJOR) {
#pragma unroll
        for (int kk = 0; kk < 2; ++kk)
#pragma unroll
          for (int j = 0; j < CB; ++j) asm volatile("" : "+v"(f.b[kk][j]));
      }
      fill(t + S, slot);
      __builtin_amdgcn_sched_barrier(0);
    };
    auto mfmas = [&](const Frags& f) __attribute__((always_inline)) {
#pragma unroll
      for (int kk = 0; kk < 2; ++kk)
#pragma unroll
        for (int i = 0; i < MB; ++i)
#pragma unroll
          for (int j = 0; j < CB; ++j) acc[i][j] = Traits::mfma(f.b[kk][j], f.a[kk][i], acc[i][j]);
    };
    auto pick = [](bool late, vec8 now, vec8 before) __attribute__((always_inline)) {
      const i32x4 x = __builtin_bit_cast(i32x4, now), y = __builtin_bit_cast(i32x4, before);
      return __builtin_bit_cast(vec8, i32x4{late ? x[0] : y[0], late ? x[1] : y[1], late ? x[2] : y[2], late ? x[3] : y[3]});
    };
    // K tile t - 1: `before` holds fill t - 1, `now` fill t
    auto shifted_mfmas = [&](Frags& before, const Frags& now) __attribute__((always_inline)) {
#pragma unroll
      for (int kk = 0; kk < 2; ++kk) {
#pragma unroll
        for (int j = 0; j < CB; ++j) before.b[kk][j] = KMAJOR ? now.b[kk][j] : pick(late_b[kk], now.b[kk][j], before.b[kk][j]);
#pragma unroll
        for (int i = 0; i < MB; ++i) {
          before.a[kk][i] = pick(late_a[kk], now.a[kk][i], before.a[kk][i]);
#pragma unroll
          for (int j = 0; j < CB; ++j) acc[i][j] = Traits::mfma(before.b[kk][j], before.a[kk][i], acc[i][j]);
        }
      }
    };
    int slot = 0;
    auto next_slot = [&]() __attribute__((always_inline)) { slot = slot + 1 == S ? 0 : slot + 1; };
    if constexpr (SHIFT) {
      Frags x, y;
      if (fills > 0) {
        take(x, 0, slot);
        next_slot();
      }
      int t = 1;
      for (; t + 1 < fills; t += 2) {
        take(y, t, slot);
        next_slot();
        shifted_mfmas(x, y);
        take(x, t + 1, slot);
        next_slot();
        shifted_mfmas(y, x);
      }
      if (t < fills) {
        take(y, t, slot);
        shifted_mfmas(x, y);
      }
    } else {
      for (int t = 0; t < fills; ++t) {
        Frags f;
        take(f, t, slot);
        mfmas(f);
        next_slot();
      }
    }
    wait_vm_and_lds<0>();  // the empty fills of the last iterations must be gone before the ring is reused

    // The elements behind the last whole chunk, straight from memory: lanes 0 .. 15 hold them as the first of an MFMA's
    // four groups of 8, the other lanes zeros.  A row's last 16 bytes are fetched as they stand and shifted down.
    if (rem != 0 && wave == NW - 1) {  // (uniform)
      const int r = lane & 15;
      auto row_end = [&](const T* base, int rows, int block) __attribute__((always_inline)) {
        typedef unsigned long long u64x2 __attribute__((ext_vector_type(2)));
        const __amdgpu_buffer_rsrc_t rs = make_rsrc(base, (unsigned)rows * row_bytes);
        const int row = block * 16 + r;
        const unsigned off = lane < 16 && row < rows ? (unsigned)row * row_bytes + row_bytes - 16u : kOobOffset;
        const u64x2 w = __builtin_bit_cast(u64x2, __builtin_amdgcn_raw_buffer_load_b128(rs, (int)off, 0, 0));
        const int bits = 128 - 16 * rem;
        if (bits == 0) return __builtin_bit_cast(vec8, w);
        u64x2 o;
        o[0] = bits >= 64 ? w[1] >> (bits - 64) : (w[0] >> bits) | (w[1] << (64 - bits));
        o[1] = bits >= 64 ? 0ull : w[1] >> bits;
        return __builtin_bit_cast(vec8, o);
      };
      vec8 fb[CB];
#pragma unroll
      for (int j = 0; j < CB; ++j) {
        if constexpr (KMAJOR) {
          const int nn = col0 + j * 16 + r;
#pragma unroll
          for (int e = 0; e < 8; ++e) fb[j][e] = lane < 16 && e < rem && nn < N ? ((const T*)p.B)[(size_t)(k8 * 8 + e) * N + nn] : (T)0.0f;
        } else {
          fb[j] = row_end(b_base, rows_b, j);
        }
      }
#pragma unroll
      for (int i = 0; i < MB; ++i) {
        const vec8 fa = row_end(a_base, rows_a, i);
#pragma unroll
        for (int j = 0; j < CB; ++j) acc[i][j] = Traits::mfma(fb[j], fa, acc[i][j]);
      }
    }
  }

  // Puts the wavefronts' sums into LDS; after the barrier inside, total(q) adds quad q = (row, column group) of the tile.
  static __device__ __forceinline__ void meet(int lane, char* ring, const f32x4 (&acc)[MB][CB]) {
    // Lane l of a block holds columns 4 * (l >> 4) .. + 3 of row l & 15.
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
      for (int j = 0; j < CB; ++j) *(f32x4*)(ring + sum_slot(i * 16 + (lane & 15), j * 4 + (lane >> 4)) * 16) = acc[i][j];
    __syncthreads();
  }
  static __device__ __forceinline__ f32x4 total(const char* smem, int q) {
    const char* at = smem + sum_slot(q / CG, q % CG) * 16;
    f32x4 part[NW];
#pragma unroll
    for (int w = 0; w < NW; ++w) part[w] = *(const f32x4*)(at + w * (S * SLOT));
    f32x4 v = part[0];
#pragma unroll
    for (int w = 1; w < NW; ++w) v += part[w];
    return v;
  }
  static __device__ __forceinline__ void store_quad(T* C, int m, int n, int N, vec4 v) {
    typedef T at_element __attribute__((ext_vector_type(4), aligned(2)));  // C lies at any element's address
    T* dst = C + (size_t)m * N + n;
    if (n + 3 < N) {
      *(at_element*)dst = v;
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (n + e < N) dst[e] = v[e];
    }
  }

  static __device__ __forceinline__ void run(const KwParams& p, char* smem) {
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const TileCoord tc = tile_of_workgroup(blockIdx.x, p.tiles_m, p.tiles_n, p.group_m, p.divs);
    const int row0 = tc.tm * ROWS, col0 = tc.tn * COLS;
    char* const ring = smem + wave * (S * SLOT);
    f32x4 acc[MB][CB];
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
      for (int j = 0; j < CB; ++j) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    multiply(p, row0, col0, wave, lane, ring, acc);
    meet(lane, ring, acc);
#pragma unroll
    for (int q0 = 0; q0 < QUADS; q0 += NT) {
      const int q = q0 + (int)threadIdx.x;
      const int m = row0 + q / CG, n = col0 + (q % CG) * 4;
      if (q >= QUADS || q / CG >= ROWS || m >= p.M || n >= p.N) continue;
      const f32x4 v = total(smem, q);
      vec4 o;
#pragma unroll
      for (int e = 0; e < 4; ++e) o[e] = (T)v[e];
      store_quad((T*)p.C, m, n, p.N, o);
    }
  }

  // The tile's share of y = LayerNorm(x) * gamma + beta.  A thread owns QT quads of the summed tile; a row's quads are
  // neighbouring lanes.  Beyond the product's time this is a chain of latencies: the tile's statistics to memory, the band's
  // back, 3 us.  us, the tiled kernel (one K group, tiles of 64 x 64 and more) -> this: 100 x 304 x 3896 26.9 -> 8.8,
  // 151 x 632 x 4384 32.0 -> 10.2, 512 x 1024 x 1000 12.0 -> 8.7, 1024 x 1024 x 3000 24.9 -> 18.2, 1298 x 312 x 7512 51.8 -> 21.4.
  static __device__ __forceinline__ void run_ln(const KwLnParams& p, char* smem) {
    constexpr int QT = (QUADS + NT - 1) / NT;
    constexpr int TPR = NT / ROWS < 16 ? NT / ROWS : 16;  // threads that merge a row's statistics
    static_assert(AG >= 2 && QUADS % 64 == 0 && (QUADS < NT || QUADS % NT == 0) && TPR * ROWS <= NT, "LayerNorm threads");
    static_assert((64 + 1) * ROWS * 8 <= LDS_BYTES, "statistics of 64 column tiles and the row results");
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // Short bands stay together on an XCD, which then fetches their rows once (1298 x 312 x 7512 28.7 -> 25.9 us); long ones
    // are spread (capi.hip: band_group).
    const int id = p.tiles_n <= kKwLnShortBand ? xcd_remap(blockIdx.x, p.tiles_m * p.tiles_n) : (int)blockIdx.x;
    const TileCoord tc = unpadded_band_tile(id, p.tiles_m, p.tiles_n, p.divs);
    const int tm = tc.tm, tn = tc.tn;
    const int row0 = tm * ROWS, col0 = tn * COLS;
    const int M = p.M, N = p.N;
    char* const ring = smem + wave * (S * SLOT);
    f32x4 acc[MB][CB];
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
      for (int j = 0; j < CB; ++j) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    multiply(p, row0, col0, wave, lane, ring, acc);
    // a thread's columns are the same for all its quads (NT is a multiple of CG)
    const int cg = tid % CG, n = col0 + cg * 4;
    vec4 g, b;
    if (N % 4 == 0 && n < N) {
      g = *(const vec4*)((const T*)p.gamma + n);
      b = *(const vec4*)((const T*)p.beta + n);
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int nn = n + e < N ? n + e : N - 1;
        g[e] = ((const T*)p.gamma)[nn];
        b[e] = ((const T*)p.beta)[nn];
      }
    }
    const unsigned tag = ln_launch_tag(p);
    ln_sign_header(p, tag);
    meet(lane, ring, acc);
    f32x4 v[QT];
#pragma unroll
    for (int u = 0; u < QT; ++u) v[u] = tid + u * NT < QUADS ? total(smem, tid + u * NT) : f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    __syncthreads();  // the sums have been read: LDS is free
    // the tile's (mean, M2) per row: about the tile's own mean first, so nothing cancels
    const int cols = N - col0 < COLS ? N - col0 : COLS;
    const size_t band = (size_t)tm * p.tiles_n * ROWS;
#pragma unroll
    for (int u = 0; u < QT; ++u) {
      float s = 0.0f, m2 = 0.0f;
#pragma unroll
      for (int e = 0; e < 4; ++e) s += n + e < N ? v[u][e] : 0.0f;
      const float mean = lanes_sum<CG>(s) / (float)cols;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float d = n + e < N ? v[u][e] - mean : 0.0f;
        m2 += d * d;
      }
      m2 = lanes_sum<CG>(m2);
      if (cg == 0 && tid + u * NT < QUADS) ln_publish(p, band + (size_t)tn * ROWS + (tid + u * NT) / CG, mean, m2, tag);
    }
    float* const red = (float*)smem;          // [ROWS][2]: (mean, 1 / standard deviation) of the whole row
    float* const gathered = red + ROWS * 2;   // [tiles_n][ROWS][2]
    ln_gather<NT>(p, tag, band, p.tiles_n * ROWS, tid, (unsigned long long*)gathered);
    __syncthreads();
    if (tid < ROWS * TPR) {
      const int r = tid / TPR, part = tid % TPR;
      float s = 0.0f, m2 = 0.0f;
      for (int t = part; t < p.tiles_n; t += TPR) {
        const int w = N - t * COLS < COLS ? N - t * COLS : COLS;
        s += (float)w * gathered[(t * ROWS + r) * 2];
      }
      const float mean = lanes_sum<TPR>(s) / (float)N;
      for (int t = part; t < p.tiles_n; t += TPR) {
        const int w = N - t * COLS < COLS ? N - t * COLS : COLS;
        const float d = gathered[(t * ROWS + r) * 2] - mean;
        m2 += gathered[(t * ROWS + r) * 2 + 1] + (float)w * d * d;
      }
      m2 = lanes_sum<TPR>(m2);
      if (part == 0) {
        red[r * 2] = mean;
        red[r * 2 + 1] = 1.0f / sqrtf(m2 / (float)N + p.eps);
      }
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < QT; ++u) {
      const int q = tid + u * NT, m = row0 + q / CG;
      if (q >= QUADS || m >= M || n >= N) continue;
      const float mean = red[q / CG * 2], rstd = red[q / CG * 2 + 1];
      vec4 o;
#pragma unroll
      for (int e = 0; e < 4; ++e) o[e] = (T)((v[u][e] - mean) * rstd * (float)g[e] + (float)b[e]);
      store_quad((T*)p.C, m, n, N, o);
    }
  }
};

template <typename T, int AG, int CB, int NW, int S, KwRows MODE, bool KMAJOR>
__global__ void __launch_bounds__(NW * 64, 2) gemm_kwave_kernel(const KwParams p) {
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  KwTile<T, AG, CB, NW, S, MODE, KMAJOR>::run(p, smem);
}

// A second launch costs 2.6 us and waits for the first one's last tile; here the array is streamed by the CUs that have no
// tile, or no tile any more.  Such a workgroup holds a tile's LDS, so a CU has only 4 to 20 wavefronts of them: rounds of 8
// accesses for every thread.  (In the tiles of up to 48 rows + columns and 32 x 32, not shifted, the compiler has two of a
// round in flight at a time and uses fewer registers; eight, held together by a scheduling barrier, are ahead at 32 x 32 with
// 2^24 elements, 19.2 -> 17.4 us, and behind in a long job, 256 x 256 x 128 with 2^26 51.9 -> 62.2.)
template <typename T, int AG, int CB, int NW, int S, KwRows MODE>
__global__ void __launch_bounds__(NW * 64, 2) gemm_kwave_side_kernel(const KwSideParams p) {
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  const unsigned tiles = (unsigned)(p.tiles_m * p.tiles_n);
  if (blockIdx.x >= tiles) {  // (uniform)
    silu_stream<T, 8>((const T*)p.side_x, (T*)p.side_y, (size_t)p.side_count, (size_t)(blockIdx.x - tiles) * (NW * 64) + threadIdx.x,
                      (size_t)(gridDim.x - tiles) * (NW * 64));
    return;
  }
  KwTile<T, AG, CB, NW, S, MODE, false>::run(p, smem);
}

template <typename T, int AG, int CB, int NW, int S, KwRows MODE>
__global__ void __launch_bounds__(NW * 64, 2) gemm_kwave_ln_kernel(const KwLnParams p) {
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  KwTile<T, AG, CB, NW, S, MODE, false>::run_ln(p, smem);
}

}  // namespace beam
