// linear_rows.hip — y = x w' for up to 128 rows of x (bf16, 32-bit sums).
//
// The weights' bytes are what counts, so they go straight from memory into
// matrix-core operands, once, with plain loads (marked non-temporal they come
// at three quarters of the rate). A workgroup owns 128 or 256 output channels
// (8 waves of 16 CT) and walks K in steps of 128; a wave reads 256 bytes of 16
// weight rows per step, two steps ahead. x goes through LDS: the waves share
// it, since a workgroup that reads x for each wave (or few channels for each
// x) spends as much of the caches' rate on x as on weights. Loads retire in
// order, so x of a step is asked for ahead of the weights of that step. The
// order of K inside a step is the same for both operands, and workgroups start
// at different steps: in step they would hit the same few memory channels
// where rows are a power of two apart.
//
// Measured, cold weights, without the sum of the parts (library call: its time
// on the device): 4096 -> 28672, 30 rows: 45 us, 5.3 TB/s (49); 14336 -> 4096,
// 30 rows: 24 us, 5.0 TB/s (31; 69 with weights stored [in, out]); 25600 ->
// 5120, 30 rows: 50 us, 5.2 TB/s (145); 4096 -> 4096, 1 row: 9 us (15).
#include "layered/elem.h"

namespace {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;

struct Rows {
  const short *x, *w;        // [M, K], [N, K] (GATED: [2 N, K], gate first)
  int64_t x_row, w_row;      // strides in elements
  void* y;                   // [M, N]; PARTS: [parts, M, N] 32-bit
  int M, N, K, k_part;       // k_part: K per part, a multiple of KS
  int act;
};

// what becomes of the sums: bf16, 32-bit (also of a part of K), or
// act(gate) * up as bf16
enum Out { BF16, F32, GATED };

constexpr int NW = 8, KS = 128, XS = KS + 8;   // XS: row of x in LDS

template <int CT, int MT, int OUT>
__global__ __launch_bounds__(NW * WAVE) void linear_rows_kernel(const Rows p) {
  __shared__ __align__(16) short xl[2][16 * MT * XS];
  constexpr int WI = KS / 32, XR = NW * WAVE / (KS / 8);
  constexpr int XT = (16 * MT + XR - 1) / XR;      // pieces of x per thread
  const int wave = threadIdx.x / WAVE, lane = threadIdx.x % WAVE;
  const int col = lane % 16, grp = lane / 16, M = p.M, N = p.N;
  const int k_lo = blockIdx.y * p.k_part, k_hi = min(p.K, k_lo + p.k_part);
  // GATED: waves 0 to 3 take gate's channels, 4 to 7 the same ones of up
  constexpr int NC = OUT == GATED ? NW / 2 : NW;
  const int n0 = (blockIdx.x * NC + wave % NC) * 16 * CT;
  // channels past N and rows past M repeat the last one and are dropped
  const short* wr[CT];
#pragma unroll
  for (int c = 0; c < CT; ++c)
    wr[c] = p.w + (min(n0 + c * 16 + col, N - 1) + wave / NC * N) * p.w_row +
            grp * 16;
  const int xr = threadIdx.x / (KS / 8), xp = threadIdx.x % (KS / 8);
  const short* xg[XT];
#pragma unroll
  for (int j = 0; j < XT; ++j)
    xg[j] = p.x + min(xr + j * XR, M - 1) * p.x_row + xp * 8;
  float4v acc[CT][MT];
#pragma unroll
  for (int c = 0; c < CT; ++c)
#pragma unroll
    for (int t = 0; t < MT; ++t) acc[c][t] = (float4v){0.f, 0.f, 0.f, 0.f};
  const short8 zero = {0, 0, 0, 0, 0, 0, 0, 0};
  short8 w0[CT][WI], w1[CT][WI], xn[XT];
  const int steps = (k_hi - k_lo + KS - 1) / KS;
  const int first = blockIdx.x * 3u % steps;   // 1 instead of 3: gate and up
                                               // of a wave pair collide, 60 us
                                               // for 44
  auto at = [&](int s) {
    s += first;
    return k_lo + (s >= steps ? s - steps : s) * KS;
  };
  auto fetch_w = [&](auto& r, int s) {
    const int k0 = at(s);
    const bool whole = k0 + KS <= k_hi;    // K is a multiple of 8
#pragma unroll
    for (int c = 0; c < CT; ++c)
#pragma unroll
      for (int i = 0; i < WI; ++i) {
        const int k = k0 + i / 2 * 64 + i % 2 * 8;
        r[c][i] = whole || k + grp * 16 < k_hi ? *(const short8*)(wr[c] + k)
                                               : zero;
      }
  };
  auto fetch_x = [&](int s) {
    const int k0 = at(s);
#pragma unroll
    for (int j = 0; j < XT; ++j)
      xn[j] = k0 + xp * 8 < k_hi ? *(const short8*)(xg[j] + k0) : zero;
  };
  auto put_x = [&](int b) {
#pragma unroll
    for (int j = 0; j < XT; ++j)
      if (16 * MT % XR == 0 || xr + j * XR < 16 * MT)
        *(short8*)(xl[b] + (xr + j * XR) * XS + xp * 8) = xn[j];
  };
  auto step = [&](auto& r, int b, int s) {
#pragma unroll
    for (int i = 0; i < WI; ++i) {
      bf16x8 xf[MT];
#pragma unroll
      for (int t = 0; t < MT; ++t)
        xf[t] = *(const bf16x8*)(xl[b] + (t * 16 + col) * XS + i / 2 * 64 +
                                 grp * 16 + i % 2 * 8);
#pragma unroll
      for (int c = 0; c < CT; ++c)
#pragma unroll
        for (int t = 0; t < MT; ++t)
          acc[c][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              __builtin_bit_cast(bf16x8, r[c][i]), xf[t], acc[c][t], 0, 0, 0);
    }
    if (s + 1 < steps) put_x(b ^ 1);
    if (s + 2 < steps) fetch_x(s + 2);
    __builtin_amdgcn_sched_barrier(0);     // x ahead of the weights
    if (s + 2 < steps) fetch_w(r, s + 2);
    __builtin_amdgcn_sched_barrier(0);
    lds_barrier();
  };
  fetch_x(0);
  fetch_w(w0, 0);
  put_x(0);
  if (1 < steps) fetch_x(1);
  if (1 < steps) fetch_w(w1, 1);
  lds_barrier();
  for (int s = 0; s < steps; s += 2) {
    step(w0, 0, s);
    if (s + 1 < steps) step(w1, 1, s + 1);
  }
  float4v* up = (float4v*)xl;              // no longer read: the loop's end
  if constexpr (OUT == GATED) {
    static_assert(sizeof(xl) >= NC * CT * MT * WAVE * sizeof(float4v));
    if (wave >= NC) {
#pragma unroll
      for (int c = 0; c < CT; ++c)
#pragma unroll
        for (int t = 0; t < MT; ++t)
          up[(((wave - NC) * CT + c) * MT + t) * WAVE + lane] = acc[c][t];
    }
    __syncthreads();
    if (wave >= NC) return;
  }
#pragma unroll
  for (int c = 0; c < CT; ++c)
#pragma unroll
    for (int t = 0; t < MT; ++t) {
      const int n = n0 + c * 16 + grp * 4, m = t * 16 + col;
      if (n >= N || m >= M) continue;      // N is a multiple of 4
      const float4v a = acc[c][t];
      const int64_t o = ((int64_t)blockIdx.y * M + m) * N + n;
      if constexpr (OUT == F32) {
        *(float4v*)((float*)p.y + o) = a;
      } else {
        short4v v;
        float4v u = a;
        if constexpr (OUT == GATED)
          u = up[((wave * CT + c) * MT + t) * WAVE + lane];
#pragma unroll
        for (int r = 0; r < 4; ++r)
          v[r] = f32_to_bf16(OUT == GATED ? activate(p.act, a[r]) * u[r]
                                          : a[r]);
        *(short4v*)((short*)p.y + o) = v;
      }
    }
}

// sum of the parts; n4: float4s of one
template <typename T>
__global__ __launch_bounds__(256) void sum_parts_kernel(
    const float4v* __restrict__ part, T* __restrict__ y, int64_t n4,
    int parts) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n4) return;
  float4v s = part[i];
#pragma unroll 8
  for (int k = 1; k < parts; ++k) s += part[k * n4 + i];
  if constexpr (sizeof(T) == 4)
    ((float4v*)y)[i] = s;
  else
    ((short4v*)y)[i] = (short4v){f32_to_bf16(s[0]), f32_to_bf16(s[1]),
                                 f32_to_bf16(s[2]), f32_to_bf16(s[3])};
}

// in [R, C] 32-bit -> out [C, R] bf16, tiles of 64 x 64: the layout of weights
// that are drawn as [in, out]. 4096 x 28672 in 136 us, where a strided copy
// takes 504 us.
__global__ __launch_bounds__(256) void lay_weights_kernel(
    const float* __restrict__ in, short* __restrict__ out, int R, int C) {
  __shared__ float tile[64][65];
  const int c0 = blockIdx.x * 64, r0 = blockIdx.y * 64, tid = threadIdx.x;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int r = tid / 16 + i * 16, c = tid % 16 * 4;
    if (r0 + r < R && c0 + c < C) {          // C is a multiple of 4
      const float4v v = *(const float4v*)(in + (int64_t)(r0 + r) * C + c0 + c);
#pragma unroll
      for (int j = 0; j < 4; ++j) tile[r][c + j] = v[j];
    }
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int c = tid / 8 + i * 32, r = tid % 8 * 8;
    if (r0 + r < R && c0 + c < C) {          // R is a multiple of 8
      short8 v;
#pragma unroll
      for (int j = 0; j < 8; ++j) v[j] = f32_to_bf16(tile[r + j][c]);
      *(short8*)(out + (int64_t)(c0 + c) * R + r0 + r) = v;
    }
  }
}

// 16-channel tiles per wave. 256 channels per workgroup halve what x costs
// beside the weights: from 33 rows on that is worth it, unless the output is
// so narrow that K falls into many parts (50 rows: 4096 -> 28672 45 us with
// 256 in two parts, 50 with 128; 14336 -> 4096 27 in 16 parts, 26 in 8), and
// where 128 would make more than one round of the 256 compute units.
int channel_tiles(int M, int weight_rows) {
  if (weight_rows > 128 * 256) return 2;
  return M > 32 && weight_rows > 4096 ? 2 : 1;
}

template <int CT, int MT, int OUT>
hipError_t go(const Rows& p, int parts, hipStream_t stream) {
  constexpr int width = NW * 16 * CT / (OUT == GATED ? 2 : 1);
  hipLaunchKernelGGL((linear_rows_kernel<CT, MT, OUT>),
                     dim3((p.N + width - 1) / width, parts), dim3(NW * WAVE),
                     0, stream, p);
  HIP_CHECK_LAST();
  return hipSuccess;
}

template <int CT, int OUT>
hipError_t go_rows(const Rows& p, int parts, hipStream_t stream) {
  if (p.M <= 16) return go<CT, 1, OUT>(p, parts, stream);
  if (p.M <= 32) return go<CT, 2, OUT>(p, parts, stream);
  if (OUT == GATED || p.M <= 64) return go<CT, 4, OUT>(p, parts, stream);
  if (p.M <= 96) return go<CT, 6, OUT>(p, parts, stream);
  return go<CT, 8, OUT>(p, parts, stream);
}

}  // namespace

extern "C" {

// Parts of K of a product: as many as make up one round of the 256 compute
// units, each with two steps of K at least. (4096 -> 4096, 1 row: 9 us in 8
// parts and 4 for their sum, 25 in one.)
int lds_linear_rows_parts(int M, int N, int K) {
  const int width = 128 * channel_tiles(M, N);
  int parts = 256 / ((N + width - 1) / width);
  if (parts > K / (2 * KS)) parts = K / (2 * KS);
  if (parts < 1) parts = 1;
  const int k_part = ((K + parts - 1) / parts + KS - 1) / KS * KS;
  return (K + k_part - 1) / k_part;
}

// Whether a product of M rows is faster here than in the library (device
// times, here / there, of 4096 -> 4096 W, 4096 -> 12576 I, 14336 -> 4096 D,
// 4096 -> 32768 H and 4096 -> [2 x 14336] G).
//   parts: the caller sums the parts itself: always. 1 row: W 9 / 15, I 21 /
//     28, D 22 / 26; 64 rows: W 11 / 15, I 26 / 26, D 28 / 39.
//   plain, in parts: their sum is a launch of 4.5 us. Up to 32 rows the call
//     is as fast or faster and costs the host half as much; above only where
//     the output is narrow: 50 rows W 15 / 14, I 30 / 25, D 31 / 36; 128 rows
//     D 43 / 75.
//   plain, in one: 96 rows H 62 / 63, 128 rows H 69 / 64.
//   gated: 64 rows G 52 / 53 (with its activation), 96 rows G 60 / 58. The
//     library is better in wide ones: 5120 -> [2 x 25600], 30 rows, 106 / 97.
int lds_linear_rows_takes(int M, int N, int K, int gated, int parts) {
  if (parts) return M <= 128;
  if (gated) return M <= 64 && 2 * N <= 128 * 256;
  if (lds_linear_rows_parts(M, N, K) == 1) return M <= 96;
  return M <= 32 || (M <= 128 && K >= 2 * N);
}

// x [M, K], w [N, K], rows x_row and w_row apart and 16-byte aligned; y [M, N]
// bf16 or (f32) 32-bit. part: [parts, M, N] floats if parts > 1; without y
// the result stays there.
hipError_t lds_linear_rows(const void* x, int64_t x_row, const void* w,
                           int64_t w_row, void* y, float* part, int parts,
                           int M, int N, int K, int f32, hipStream_t stream) {
  if (M < 1 || M > 128 || N < 1 || N % 4 || K < 8 || K % 8 || x_row % 8 ||
      w_row % 8 || parts < 1 || (!part && (parts > 1 || !y)))
    return hipErrorInvalidValue;
  Rows p{(const short*)x, (const short*)w, x_row, w_row, y, M, N, K, K, 0};
  p.k_part = ((K + parts - 1) / parts + KS - 1) / KS * KS;
  if (parts > 1 || !y) p.y = part;
  const bool two = channel_tiles(M, N) == 2;
  hipError_t e;
  if (f32 || p.y == part)
    e = two ? go_rows<2, F32>(p, parts, stream)
            : go_rows<1, F32>(p, parts, stream);
  else
    e = two ? go_rows<2, BF16>(p, 1, stream) : go_rows<1, BF16>(p, 1, stream);
  if (e != hipSuccess || p.y == y) return e;
  if (!y) return hipSuccess;
  const int64_t n4 = (int64_t)M * N / 4;
  const dim3 grid((uint32_t)((n4 + 255) / 256));
  if (f32)
    hipLaunchKernelGGL(sum_parts_kernel<float>, grid, dim3(256), 0, stream,
                       (const float4v*)part, (float*)y, n4, parts);
  else
    hipLaunchKernelGGL(sum_parts_kernel<short>, grid, dim3(256), 0, stream,
                       (const float4v*)part, (short*)y, n4, parts);
  HIP_CHECK_LAST();
  return hipSuccess;
}

// in [R, C] 32-bit -> out [C, R] bf16
hipError_t lds_lay_weights(const float* in, void* out, int R, int C,
                           hipStream_t stream) {
  if (R < 8 || R % 8 || C < 4 || C % 4) return hipErrorInvalidValue;
  const dim3 grid((C + 63) / 64, (R + 63) / 64);
  if (grid.y > 65535) return hipErrorInvalidValue;
  hipLaunchKernelGGL(lay_weights_kernel, grid, dim3(256), 0, stream, in,
                     (short*)out, R, C);
  HIP_CHECK_LAST();
  return hipSuccess;
}

// y [M, N] = act(x gate') * (x up'), w [2 N, K] = [gate; up]
hipError_t lds_gated_rows(const void* x, int64_t x_row, const void* w,
                          int64_t w_row, void* y, int M, int N, int K, int act,
                          hipStream_t stream) {
  if (M < 1 || M > 64 || N < 1 || N % 4 || K < 8 || K % 8 || x_row % 8 ||
      w_row % 8 || act < 0 || act >= ACTS)
    return hipErrorInvalidValue;
  // 64 channels per workgroup: 128 rows of weights
  const Rows p{(const short*)x, (const short*)w, x_row, w_row, y, M, N, K,
               (K + KS - 1) / KS * KS, act};
  return go_rows<1, GATED>(p, 1, stream);
}

}  // extern "C"
