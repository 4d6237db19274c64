// Elementwise functions shared by the tiled kernel's side job and the standalone streaming kernel.
#pragma once

#include <hip/hip_runtime.h>

namespace beam {

// silu(x) = x / (1 + exp(-x)) in fp32 (hardware exp2 and reciprocal, about 1 ulp each: far inside
// the rounding of a 16-bit result).  Same formula as the reference's side job,
// cuda/cute_kernels/cute_gemm_ln.cu:191-192.
//
// WIDE_RANGE: the hardware reciprocal flushes denormal results, which 1 / (1 + exp(-x)) is for x below
// -87.3 although x times it is still a normal fp32 number down to x = -88.7 (where exp(-x) overflows
// and the formula gives -0).  bf16 can hold a result that small, so for bf16 numerator and
// denominator are scaled by 2^-64 in that range; an fp16 result is -0 there either way.
//
// The product passes through an empty asm so that it stays a plain fp32 multiply: a multiply that
// feeds the 16-bit conversion directly is selected as a mixed-precision fma with a +0 addend,
// which turns the -0 of silu(-0) into +0.
template <bool WIDE_RANGE>
__device__ __forceinline__ float silu_f32(float x) {
  const float d = 1.0f + __builtin_amdgcn_exp2f(x * -1.4426950408889634f);
  float r;
  if (WIDE_RANGE) {
    const bool big = d > 0x1p64f;
    const float ds = big ? d * 0x1p-64f : d;
    const float xs = big ? x * 0x1p-64f : x;
    r = xs * __builtin_amdgcn_rcpf(ds);
  } else {
    r = x * __builtin_amdgcn_rcpf(d);
  }
  asm("" : "+v"(r));
  return r;
}

template <typename T>
__device__ __forceinline__ T silu_16(T x) {
  return (T)silu_f32<sizeof(T) == 2 && !__is_same(T, _Float16)>((float)x);
}

// y[i] = silu(x[i]) by thread `id` of `threads` that share the array: 16 bytes per access, rounds of U accesses.
template <typename T, int U>
__device__ __forceinline__ void silu_stream(const T* __restrict__ x, T* __restrict__ y, size_t count, size_t id, size_t threads) {
  typedef T vec8 __attribute__((ext_vector_type(8)));
  const size_t vecs = count / 8;
  size_t v = id;
  for (; v + (U - 1) * threads < vecs; v += U * threads) {
    vec8 in[U];
#pragma unroll
    for (int u = 0; u < U; ++u) in[u] = *(const vec8*)(x + (v + u * threads) * 8);
#pragma unroll
    for (int u = 0; u < U; ++u) {
      vec8 out;
#pragma unroll
      for (int e = 0; e < 8; ++e) out[e] = silu_16<T>(in[u][e]);
      *(vec8*)(y + (v + u * threads) * 8) = out;
    }
  }
  // What is left of a thread's last round, fetched at once: up to U - 1 accesses one after the other are longer than a small
  // GEMM beside them (65 x 1072 x 160 with 174096 elements, U = 8: one by one 5.0 us, at once 4.3).
  if (v < vecs) {
    vec8 in[U];
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (v + u * threads < vecs) in[u] = *(const vec8*)(x + (v + u * threads) * 8);
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (v + u * threads >= vecs) break;
      vec8 out;
#pragma unroll
      for (int e = 0; e < 8; ++e) out[e] = silu_16<T>(in[u][e]);
      *(vec8*)(y + (v + u * threads) * 8) = out;
    }
  }
  const size_t i = vecs * 8 + id;
  if (i < count) y[i] = silu_16<T>(x[i]);
}

}  // namespace beam
