// flash_core.h — the part that the prefill attention kernels share: a wave's
// 32 query rows against 32 or 64 keys in LDS, with an online softmax per query.
//
// S' = K Q' on 32x32x16 tiles leaves lane (column c, half h) with the scores
// of query c for keys (r & 3) + 8 (r >> 2) + 4 h, r = 0..15. The order of the
// keys inside a step of O' = V' P' is free, so the probabilities of registers
// 8 s .. 8 s + 7 are step s's operand as they are, and V' is read in the same
// order: rows 16 s + 4 h .. + 3 and + 8 .. + 11. Nothing crosses the wave but
// the maximum. Each score has one multiply-add, one exponential (the scale is in
// the multiply-add), half a pack, and its shares of the maximum and the sum: two
// thirds of the cycles that the matrix cores need, which the other wave of a SIMD
// fills. LDS reads run a fixed number of operands ahead of their instructions, in
// an order that is written out: left to the compiler, each operand of K was waited
// for before the next was asked for.
#pragma once
#include "hip_common.h"

namespace flash {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;
typedef __attribute__((ext_vector_type(16))) float f32x16;
typedef __attribute__((ext_vector_type(4))) unsigned int uint4v;

constexpr float LOG2E = 1.4426950408889634f;
constexpr float NEG = -1e30f;

// |scale| in log2 units. Not 0, which makes nothing of a masked -infinity: scores
// below 1e30 come out all alike by this one as well.
__device__ __forceinline__ float log2_scale(float scale) {
  return fmaxf(fabsf(scale) * LOG2E, 1e-37f);
}

__device__ __forceinline__ unsigned int pack2(float a, float b) {
  const float2v v = {a, b};
  return __builtin_bit_cast(unsigned int,
                            __builtin_convertvector(v, bf16x2));
}

// maximum over a lane and the one 32 apart
__device__ __forceinline__ float max_halves(float x) {
  const unsigned int a = __builtin_bit_cast(unsigned int, x);
  const auto r = __builtin_amdgcn_permlane32_swap(a, a, false, false);
  // not r[i] itself: a bit cast of a vector's element takes the first one
  const unsigned int lo = r[0], up = r[1];
  return fmaxf(__builtin_bit_cast(float, lo), __builtin_bit_cast(float, up));
}

// Bank swizzle of LDS rows of 128 channels (256 bytes; the 16-byte pieces of a
// row change places by XOR): the two 2-bit halves of row & 15 swapped. The
// 16-byte reads of K need any bijection on row & 15 (a group of 16 lanes
// covers all 16 values); the transposing reads of V (32 lanes: four rows in
// order, 64 bytes of each) need row & 3 in address bits 7 and 6.
__device__ __forceinline__ int swizzle(int row) {
  return (((row & 3) << 2) | ((row >> 2) & 3)) << 4;
}

// State of a lane's query: running maximum (log2 units) and, of the keys that
// this lane has seen, the sum. join() adds the halves' sums.
struct Softmax {
  float m = NEG, l = 0.f;
  __device__ __forceinline__ float join() const {
    return l + __shfl_xor(l, 32, WAVE);
  }
};

// the larger of three; a is known to come from a vector instruction (which the
// compiler keeps apart from the matrix instruction that gave b and c)
__device__ __forceinline__ float max3(float a, float b, float c) {
  asm("v_max3_f32 %0, %0, %1, %2" : "+v"(a) : "v"(b), "v"(c));
  return a;
}

// SUB x 32 keys. NK = key channels / 16, NV = value channels / 32.
//   key(u, kk)        16 bytes of key row 32 u + (lane & 31), channels 16 kk + 8
//                     half ..
//   value(u, row, t)  address of the lane's 8 bytes of value row 32 u + row:
//                     channels 32 t + 16 (lane / 16 & 1) + 4 (lane & 3) ..; row is
//                     this lane's of the four that a transposing read covers
//   FINE              probabilities as the sum of two bf16 (2^-17 of their size
//                     off, as good as the 32-bit ones of the decode kernel)
//   inside            every lane's query sees all keys; else those with
//                     first <= key <= last, relative to the tile
//   between(i)        what goes between the NK SUB matrix instructions of the
//                     scores: the caller's loads of later tiles, which in a row
//                     would hold the wave up
// scale_log2 > 0: log2_scale.
template <int NK, int NV, int SUB, bool FINE, class Key, class Value,
          class Between>
__device__ __forceinline__ void attend(Key key, Value value, const bf16x8* qf,
                                       float scale_log2, bool inside, int first,
                                       int last, Softmax& st, f32x16* acc,
                                       Between between) {
  const int lane = threadIdx.x % WAVE, hi = lane >> 5;
  // operands read ahead, as many as the registers hold
  constexpr int AHEAD = NK <= 8 && NV <= 4 ? 8 : 4;
  f32x16 s[SUB];
#pragma unroll
  for (int u = 0; u < SUB; ++u) s[u] = (f32x16)(0.f);
  {
    constexpr int N = NK * SUB;
    bf16x8 kf[AHEAD];
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < (N < AHEAD ? N : AHEAD); ++i)
      kf[i] = key(i % SUB, i / SUB);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < N; ++i) {
      s[i % SUB] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
          kf[i % AHEAD], qf[i / SUB], s[i % SUB], 0, 0, 0);
      if (i + AHEAD < N)
        kf[i % AHEAD] = key((i + AHEAD) % SUB, (i + AHEAD) / SUB);
      between(i);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  // operand (k, t) of V': step k of 16 keys, 32 channels
  const int row = 4 * hi + lane % 16 / 4;
  auto operand = [&](int i) {
    const int k = i / NV, t = i % NV;
    typedef __attribute__((address_space(3))) short4v lds4;
    const short4v lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
        (lds4*)value(k / 2, k % 2 * 16 + row, t));
    const short4v up = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
        (lds4*)value(k / 2, k % 2 * 16 + row + 8, t));
    const short8 v = {lo[0], lo[1], lo[2], lo[3], up[0], up[1], up[2], up[3]};
    return __builtin_bit_cast(bf16x8, v);
  };
  // half of the operands read ahead come in while the softmax runs, the others
  // once its registers are free
  constexpr int N = NV * 2 * SUB;
  bf16x8 vf[AHEAD];
#pragma unroll
  for (int i = 0; i < AHEAD / 2; ++i) vf[i] = operand(i);
  __builtin_amdgcn_sched_barrier(0);

  if (!inside) {
#pragma unroll
    for (int u = 0; u < SUB; ++u)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int t = u * 32 + (r & 3) + 8 * (r >> 2) + 4 * hi;
        if (t < first || t > last) s[u][r] = -INFINITY;
      }
  }
  float mx[SUB];
#pragma unroll
  for (int u = 0; u < SUB; ++u) {
    mx[u] = fmaxf(s[u][0], s[u][1]);
#pragma unroll
    for (int r = 2; r < 16; r += 2) mx[u] = max3(mx[u], s[u][r], s[u][r + 1]);
  }
  float largest = mx[0];
#pragma unroll
  for (int u = 1; u < SUB; ++u) largest = fmaxf(largest, mx[u]);
  largest = max_halves(largest);
  // without a key so far m stays at NEG and every exponent underflows to 0
  const float top = largest == -INFINITY ? NEG : largest * scale_log2;
  // The largest probability is exactly 1, which bf16 holds: to let the maximum
  // lag behind would spare rescaling and cost precision (5 % more error).
  if (__any(top > st.m)) {
    const float to = fmaxf(top, st.m);
    const float alpha = __builtin_amdgcn_exp2f(st.m - to);
    st.m = to;
    st.l *= alpha;
#pragma unroll
    for (int t = 0; t < NV; ++t)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[t][e] *= alpha;
  }
#pragma unroll
  for (int u = 0; u < SUB; ++u)
#pragma unroll
    for (int r = 0; r < 16; ++r)
      s[u][r] = __builtin_amdgcn_exp2f(fmaf(s[u][r], scale_log2, -st.m));
  float sum[SUB];
#pragma unroll
  for (int u = 0; u < SUB; ++u) {
    sum[u] = s[u][0] + s[u][1];
#pragma unroll
    for (int r = 2; r < 16; r += 2) sum[u] += s[u][r] + s[u][r + 1];
    st.l += sum[u];
  }
  bf16x8 pf[2 * SUB], pr[2 * SUB];
#pragma unroll
  for (int k = 0; k < 2 * SUB; ++k) {
    uint4v w, v;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float a = s[k / 2][k % 2 * 8 + 2 * i];
      const float b = s[k / 2][k % 2 * 8 + 2 * i + 1];
      const unsigned int ab = pack2(a, b);
      w[i] = ab;
      if (FINE) {
        const unsigned int lo = ab << 16, up = ab & 0xffff0000u;
        v[i] = pack2(a - __builtin_bit_cast(float, lo),
                     b - __builtin_bit_cast(float, up));
      }
    }
    pf[k] = __builtin_bit_cast(bf16x8, w);
    if (FINE) pr[k] = __builtin_bit_cast(bf16x8, v);
  }
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int i = AHEAD / 2; i < (N < AHEAD ? N : AHEAD); ++i) vf[i] = operand(i);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int i = 0; i < N; ++i) {
    const int k = i / NV, t = i % NV;
    acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[i % AHEAD], pf[k],
                                                     acc[t], 0, 0, 0);
    if constexpr (FINE)
      acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[i % AHEAD], pr[k],
                                                       acc[t], 0, 0, 0);
    if (i + AHEAD < N) vf[i % AHEAD] = operand(i + AHEAD);
    __builtin_amdgcn_sched_barrier(0);
  }
}

}  // namespace flash
