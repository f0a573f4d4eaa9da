// linear_rows.hip — y = x w' for few rows of x (bf16, 32-bit sums): the kernel
// for up to 16 rows, and which product goes where. Products of up to 256 rows
// go to linear_tiles.hip.
//
// The weights' bytes are what counts, so they go straight from memory into
// matrix-core operands, once, with plain loads (marked non-temporal they come
// at three quarters of the rate). A workgroup owns 128 or 256 output channels
// (8 waves of 16 CT) and walks K in steps of 128; a wave reads 256 bytes of 16
// weight rows per step, two steps ahead. x goes through LDS: the waves share
// it, since a workgroup that reads x for each wave spends as much of the
// caches' rate on x as on weights. Loads retire in order, so x of a step is
// asked for ahead of the weights of that step. Workgroups start at different
// steps: in step they would hit the same few memory channels where rows are a
// power of two apart. linear_tiles.hip adds up in the same order, so a row
// comes out the same, to the bit, whichever of the two took it: as the one row
// of a decode step or within a short prompt.
//
// Measured, 1 row, cold weights, without the sum of the parts (library: its
// time on the device): 4096 -> 28672: 43 us, 5.5 TB/s (58); 14336 -> 4096 22 us
// (26); 25600 -> 5120: 47 us (134); 4096 -> 4096: 8.4 us (15).
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

template <int CT, int OUT>
__global__ __launch_bounds__(NW * WAVE) void linear_rows_kernel(const Rows p) {
  __shared__ __align__(16) short xl[2][16 * XS];
  constexpr int WI = KS / 32;
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
            grp * 8;
  // half of the threads bring 16 bytes of x each
  const int xr = threadIdx.x / (KS / 8), xp = threadIdx.x % (KS / 8);
  const bool x_mine = xr < 16;
  const short* xg = p.x + min(xr, M - 1) * p.x_row + xp * 8;
  float4v acc[CT];
#pragma unroll
  for (int c = 0; c < CT; ++c) acc[c] = (float4v){0.f, 0.f, 0.f, 0.f};
  const short8 zero = {0, 0, 0, 0, 0, 0, 0, 0};
  short8 w0[CT][WI], w1[CT][WI], xn = zero;
  const int steps = (k_hi - k_lo + KS - 1) / KS;
  // where rows are 8 KB apart, 1 of 4096 -> 28672: a start of 3 blockIdx.x 43
  // us, 1: 44, 2: 72, 6: 51, none: 52; gated, with twice the streams, 6: 42.5,
  // 3: 45, 1: 67, none: 52. Other sizes hardly mind.
  const int first = blockIdx.x * (OUT == GATED ? 6u : 3u) % steps;
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
        const int k = k0 + i * 32;
        r[c][i] = whole || k + grp * 8 < k_hi ? *(const short8*)(wr[c] + k)
                                               : zero;
      }
  };
  auto fetch_x = [&](int s) {
    const int k0 = at(s);
    if (x_mine) xn = k0 + xp * 8 < k_hi ? *(const short8*)(xg + k0) : zero;
  };
  auto put_x = [&](int b) {
    if (x_mine) *(short8*)(xl[b] + xr * XS + xp * 8) = xn;
  };
  auto step = [&](auto& r, int b, int s) {
#pragma unroll
    for (int i = 0; i < WI; ++i) {
      const bf16x8 xf =
          *(const bf16x8*)(xl[b] + col * XS + i * 32 + grp * 8);
#pragma unroll
      for (int c = 0; c < CT; ++c)
        acc[c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
            __builtin_bit_cast(bf16x8, r[c][i]), xf, acc[c], 0, 0, 0);
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
    static_assert(sizeof(xl) >= NC * CT * WAVE * sizeof(float4v));
    if (wave >= NC) {
#pragma unroll
      for (int c = 0; c < CT; ++c)
        up[((wave - NC) * CT + c) * WAVE + lane] = acc[c];
    }
    __syncthreads();
    if (wave >= NC) return;
  }
#pragma unroll
  for (int c = 0; c < CT; ++c) {
    const int n = n0 + c * 16 + grp * 4, m = col;
    if (n >= N || m >= M) continue;        // N is a multiple of 4
    const float4v a = acc[c];
    const int64_t o = ((int64_t)blockIdx.y * M + m) * N + n;
    if constexpr (OUT == F32) {
      *(float4v*)((float*)p.y + o) = a;
    } else {
      short4v v;
      float4v u = a;
      if constexpr (OUT == GATED) u = up[(wave * CT + c) * WAVE + lane];
#pragma unroll
      for (int r = 0; r < 4; ++r)
        v[r] = f32_to_bf16(OUT == GATED ? activate(p.act, a[r]) * u[r]
                                        : a[r]);
      *(short4v*)((short*)p.y + o) = v;
    }
  }
}

// sum of the parts, or (act >= 0) the activation of it; n4: float4s of one
template <typename T>
__global__ __launch_bounds__(256) void sum_parts_kernel(
    const float4v* __restrict__ part, T* __restrict__ y, int64_t n4,
    int parts, int act) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n4) return;
  float4v s = part[i];
#pragma unroll 8
  for (int k = 1; k < parts; ++k) s += part[k * n4 + i];
  if (act >= 0)
#pragma unroll
    for (int j = 0; j < 4; ++j) s[j] = activate(act, s[j]);
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

// 16-channel tiles per wave: two where 128 channels per workgroup would make
// more than one round of the 256 compute units
int channel_tiles(int weight_rows) { return weight_rows > 128 * 256 ? 2 : 1; }

template <int CT, int OUT>
hipError_t go(const Rows& p, int parts, hipStream_t stream) {
  constexpr int width = NW * 16 * CT / (OUT == GATED ? 2 : 1);
  hipLaunchKernelGGL((linear_rows_kernel<CT, OUT>),
                     dim3((p.N + width - 1) / width, parts), dim3(NW * WAVE),
                     0, stream, p);
  HIP_CHECK_LAST();
  return hipSuccess;
}

// up to 16 rows come here, more go to linear_tiles.hip
constexpr int ROWS = 16, TILE_ROWS = 256;

// of one part of K
int workgroups(int M, int N) {
  const int width = M <= ROWS ? 128 * channel_tiles(N) : 128;
  return (N + width - 1) / width;
}

}  // namespace

extern "C" {

hipError_t lds_linear_tiles(const void*, int64_t, const void*, int64_t, void*,
                            int, int, int, int, int, int, hipStream_t);

// Parts of K of a product: as many as make up one round of the 256 compute
// units, each with 256 of K at least. (4096 -> 4096, 1 row: 9 us in 8 parts
// and 4 for their sum, 25 in one; 150 rows: 14 us in 8 parts, 17 in 4, 18 in
// 16.)
int lds_linear_rows_parts(int M, int N, int K) {
  int parts = 256 / workgroups(M, N);
  if (parts > K / 256) parts = K / 256;
  if (parts < 1) parts = 1;
  const int k_part = ((K + parts - 1) / parts + KS - 1) / KS * KS;
  return (K + k_part - 1) / k_part;
}

// Whether a product of M rows is faster here than in the library. Device
// times, here / there, in us:
//   parts the caller sums itself: always. 4096 -> 4096: 1 row 8 / 15, 96 rows
//     12 / 22, 256 rows 18 / 23; 14336 -> 4096: 64 rows 23 / 40, 256 rows
//     41 / 63; 4096 -> 12576: 64 rows 24 / 25, 256 rows 42 / 50. (Above 128 rows
//     a K below 1600 takes up to 3 us more here, 688 -> 1680, 256 rows 13 / 10;
//     that it comes out as a single row does is worth it.)
//   one part, and gated ones (there with their activation): if the workgroups
//     fill at least 7/8 of their rounds, plain up to 128 rows. 4096 -> 32768: 32 rows
//     46 / 62, 128 rows 55 / 64, 160 rows 66 / 67; -> 128256 (98 %): 64 rows
//     182 / 208; 5120 -> 51200 (78 %): 64 rows 110 / 98. 4096 -> [2 x 14336]:
//     64 rows 44 / 58, 128 rows 53 / 60, 192 rows 65 / 67, 256 rows 69 / 75. From
//     193 rows on by linear_wide, for K from 1024 on in whole steps, where the
//     workgroups are one round and K is at most 8192: 1.01 to 1.25 times as fast
//     over 25 sizes (232 rows, 1024 -> [2 x 14624]: 28 / 35). In two or three
//     rounds it is 0.66 to 1.06 times (245 rows, 3584 -> [2 x 28744]: 132 / 118), by
//     longer K 0.74 to 1.07 (15872 -> [2 x 15456]: 367 / 271);
//     inside a 4-layer stack of about 180 rows the pass takes 790 / 835;
//     2048 -> [2 x 4096] (25 %): 32 rows 18 / 16.
//   parts and their sum (3 to 5 us): with full rounds (4096 -> 6144: 64 rows
//     16 / 18, 160 rows 23 / 28; 8192 -> 5120: 256 rows 40 / 74) unless K is
//     short (2048 -> 8192: 64 rows 13.3 / 14.0, 128 rows 17.7 / 16.8), else
//     narrow ones up to 64 rows (4096 -> 1024: 64 rows 11 / 15, 96 rows
//     13 / 12; 4096 -> 12576, 77 %: 64 rows 27 / 25).
int lds_linear_rows_takes(int M, int N, int K, int gated, int parts) {
  if (M > TILE_ROWS) return 0;
  const int n = gated ? 1 : lds_linear_rows_parts(M, N, K);
  if (parts && n > 1) return 1;
  const int groups = gated ? (N + 63) / 64 : workgroups(M, N) * n;
  const bool full = groups * 8 >= (groups + 255) / 256 * 256 * 7;
  if (gated)
    return full && (M <= 192 || (groups <= 256 && K >= 1024 && K <= 8192 &&
                                 K % KS == 0));
  if (N > 128 * 128) return full && M <= 128;
  if (full) return M <= 64 || K >= 4096;
  return M <= 64 && N <= 4096;
}

// y [n] = the sum of part [parts, n], or (act >= 0) its activation; 16-byte aligned, n
// a multiple of 4
hipError_t lds_sum_parts(const float* part, void* y, int64_t n, int parts,
                         int f32, int act, hipStream_t stream) {
  if (n < 0 || n % 4 || act >= ACTS) return hipErrorInvalidValue;
  if (n == 0) return hipSuccess;
  const int64_t n4 = n / 4;
  const dim3 grid((uint32_t)((n4 + 255) / 256));
  if (f32)
    hipLaunchKernelGGL(sum_parts_kernel<float>, grid, dim3(256), 0, stream,
                       (const float4v*)part, (float*)y, n4, parts, act);
  else
    hipLaunchKernelGGL(sum_parts_kernel<short>, grid, dim3(256), 0, stream,
                       (const float4v*)part, (short*)y, n4, parts, act);
  HIP_CHECK_LAST();
  return hipSuccess;
}

// x [M, K], w [N, K], rows x_row and w_row apart and 16-byte aligned; y [M, N]
// bf16 or (f32) 32-bit. part: [parts, M, N] floats if parts > 1; without y
// the result stays there.
hipError_t lds_linear_rows(const void* x, int64_t x_row, const void* w,
                           int64_t w_row, void* y, float* part, int parts,
                           int M, int N, int K, int f32, hipStream_t stream) {
  if (M < 1 || M > TILE_ROWS || N < 1 || N % 4 || K < 8 || K % 8 ||
      x_row % 8 || w_row % 8 || parts < 1 || (!part && (parts > 1 || !y)))
    return hipErrorInvalidValue;
  const bool in_part = parts > 1 || !y;
  hipError_t e;
  if (M > ROWS) {
    e = lds_linear_tiles(x, x_row, w, w_row, in_part ? part : y, parts, M, N,
                         K, in_part || f32, -1, stream);
  } else {
    Rows p{(const short*)x, (const short*)w, x_row, w_row,
           in_part ? part : y, M, N, K, K, 0};
    p.k_part = ((K + parts - 1) / parts + KS - 1) / KS * KS;
    const bool two = channel_tiles(N) == 2;
    if (in_part || f32)
      e = two ? go<2, F32>(p, parts, stream) : go<1, F32>(p, parts, stream);
    else
      e = two ? go<2, BF16>(p, 1, stream) : go<1, BF16>(p, 1, stream);
  }
  if (e != hipSuccess || !in_part || !y) return e;
  return lds_sum_parts(part, y, (int64_t)M * N, parts, f32, -1, stream);
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
  if (M < 1 || M > TILE_ROWS || N < 1 || N % 4 || K < 8 || K % 8 ||
      x_row % 8 || w_row % 8 || act < 0 || act >= ACTS)
    return hipErrorInvalidValue;
  if (M > ROWS)
    return lds_linear_tiles(x, x_row, w, w_row, y, 1, M, N, K, 0, act, stream);
  // 64 channels per workgroup: 128 rows of weights
  const Rows p{(const short*)x, (const short*)w, x_row, w_row, y, M, N, K,
               (K + KS - 1) / KS * KS, act};
  return go<1, GATED>(p, 1, stream);
}

}  // extern "C"
