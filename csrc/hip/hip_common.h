// hip_common.h — shared device helpers for the gfx950 (CDNA4) kernels.
// Wave width is 64 on CDNA4; every cross-lane idiom below assumes that.
#pragma once
#include <hip/hip_runtime.h>
#include <hip/hip_bf16.h>
#include <cstdint>

#define WAVE 64

// vectorized bf16 access: 8 bf16 = 16 B per lane (coalescing sweet spot, guide G13)
typedef __attribute__((ext_vector_type(8))) short short8;
typedef __attribute__((ext_vector_type(4))) short short4v;
typedef __attribute__((ext_vector_type(4))) float float4v;
typedef __attribute__((ext_vector_type(2))) float float2v;

__device__ __forceinline__ float bf16_to_f32(short u) {
  union { float f; uint32_t i; } c;
  c.i = ((uint32_t)(uint16_t)u) << 16;
  return c.f;
}

__device__ __forceinline__ short f32_to_bf16(float f) {
  union { float f; uint32_t i; } c;
  c.f = f;
  // round-to-nearest-even
  uint32_t lsb = (c.i >> 16) & 1;
  uint32_t rounded = c.i + 0x7FFF + lsb;
  return (short)(uint16_t)(rounded >> 16);
}

// ---- fp8 (OCP e4m3) KV-cache element support ------------------------------
// gfx950 hardware converts: v_cvt_f32_fp8 unpacks one byte of a dword
// (constant byte select), v_cvt_pk_fp8_f32 packs two floats into half a
// dword. Cache element type CT is short (bf16) or unsigned char (fp8).
typedef __attribute__((ext_vector_type(8))) unsigned char uchar8;

// load 8 fp8 cache elements -> f32[8]
__device__ __forceinline__ void load_kv8(const unsigned char* p, float* f) {
  const uint32_t* w = (const uint32_t*)p;   // two dwords = 8 fp8
  uint32_t a = w[0], b = w[1];
  f[0] = __builtin_amdgcn_cvt_f32_fp8(a, 0);
  f[1] = __builtin_amdgcn_cvt_f32_fp8(a, 1);
  f[2] = __builtin_amdgcn_cvt_f32_fp8(a, 2);
  f[3] = __builtin_amdgcn_cvt_f32_fp8(a, 3);
  f[4] = __builtin_amdgcn_cvt_f32_fp8(b, 0);
  f[5] = __builtin_amdgcn_cvt_f32_fp8(b, 1);
  f[6] = __builtin_amdgcn_cvt_f32_fp8(b, 2);
  f[7] = __builtin_amdgcn_cvt_f32_fp8(b, 3);
}

// store 8 bf16 source elements as cache elements
__device__ __forceinline__ void store_kv8(short* p, short8 v) {
  *(short8*)p = v;
}

__device__ __forceinline__ void store_kv8(unsigned char* p, short8 v) {
  uint32_t lo = 0, hi = 0;
  lo = __builtin_amdgcn_cvt_pk_fp8_f32(bf16_to_f32(v[0]), bf16_to_f32(v[1]),
                                       lo, false);
  lo = __builtin_amdgcn_cvt_pk_fp8_f32(bf16_to_f32(v[2]), bf16_to_f32(v[3]),
                                       lo, true);
  hi = __builtin_amdgcn_cvt_pk_fp8_f32(bf16_to_f32(v[4]), bf16_to_f32(v[5]),
                                       hi, false);
  hi = __builtin_amdgcn_cvt_pk_fp8_f32(bf16_to_f32(v[6]), bf16_to_f32(v[7]),
                                       hi, true);
  uint32_t* w = (uint32_t*)p;
  w[0] = lo;
  w[1] = hi;
}

// full-wave f32 sum reduction (6 xor-shuffle steps over 64 lanes)
__device__ __forceinline__ float wave_reduce_sum(float v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, WAVE);
  return v;
}

__device__ __forceinline__ float wave_reduce_max(float v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v = fmaxf(v, __shfl_xor(v, off, WAVE));
  return v;
}

// block-level f32 sum reduction across NW waves (NW <= 16), via LDS scratch.
// `scratch` must hold NW floats; returns the total to all threads.
template <int NW>
__device__ __forceinline__ float block_reduce_sum(float v, float* scratch) {
  int wave = threadIdx.x / WAVE;
  int lane = threadIdx.x % WAVE;
  v = wave_reduce_sum(v);
  if (lane == 0) scratch[wave] = v;
  __syncthreads();
  float total = 0.f;
#pragma unroll
  for (int w = 0; w < NW; ++w) total += scratch[w];
  return total;
}

// The sums of `parts` 32-bit parts of a product that split K, of the 8 values at each
// src[i]; apart: float4s from part to part. Up to 8 parts of all N are under way
// together: summed one by one, or in a loop that the compiler unrolls by 4, each
// few of them cost the latency of a cache that another XCD wrote behind.
template <int N>
struct PartSums {
  float4v a[N][2];

  __device__ __forceinline__ PartSums(const float4v* const (&src)[N],
                                      int64_t apart, int parts) {
#pragma unroll
    for (int i = 0; i < N; ++i)          // -0 leaves what is added as it is
      a[i][0] = a[i][1] = (float4v){-0.f, -0.f, -0.f, -0.f};
    int k = 0;
    for (; k + 8 <= parts; k += 8) add<8>(src, apart, k);
    switch (parts - k) {
      case 7: add<7>(src, apart, k); break;
      case 6: add<6>(src, apart, k); break;
      case 5: add<5>(src, apart, k); break;
      case 4: add<4>(src, apart, k); break;
      case 3: add<3>(src, apart, k); break;
      case 2: add<2>(src, apart, k); break;
      case 1: add<1>(src, apart, k); break;
    }
  }
  template <int G>
  __device__ __forceinline__ void add(const float4v* const (&src)[N],
                                      int64_t apart, int first) {
    float4v g[G][N][2];
#pragma unroll
    for (int k = 0; k < G; ++k)
#pragma unroll
      for (int i = 0; i < N; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) g[k][i][j] = src[i][(first + k) * apart + j];
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int k = 0; k < G; ++k)
#pragma unroll
      for (int i = 0; i < N; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) a[i][j] += g[k][i][j];
  }
  __device__ __forceinline__ void get(int i, float* f) const {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      f[j] = a[i][0][j];
      f[4 + j] = a[i][1][j];
    }
  }
};

#define HIP_CHECK_LAST()                                              \
  do {                                                                 \
    hipError_t e_ = hipGetLastError();                                 \
    if (e_ != hipSuccess) {                                            \
      return e_;                                                       \
    }                                                                  \
  } while (0)

// Workgroup barrier that orders LDS accesses only: global loads issued before
// it stay in flight across it (__syncthreads waits for them)
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}
