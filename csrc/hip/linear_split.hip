// linear_split.hip — y = x w' for 257 to some thousand rows of x and long K (bf16,
// 32-bit sums): tiles of 256 weight rows by 192 or 256 rows of x by the loop of
// tile_core.h, K split until the tiles fill a round of the compute units.
//
// There are too few tiles for 256 compute units without the split, and the library
// fills them with smaller tiles, which read each operand more often, at 400 to 900
// TFLOP/s. Here the matrix cores bound it, and the parts, which are written once
// and read once in 32-bit: 12 to 20 us. us, library / here with the sum of the
// parts: 14336 -> 4096, 341 rows 77 / 50, 1000 rows 131 / 97, 1600 rows 331 / 160;
// 25600 -> 5120, 300 rows 180 / 92, 775 rows 332 / 194; 8192 -> 2048, 1063 rows 64
// / 48; 16384 -> 1024, 935 rows 68 / 44.
#include "tile_core.h"

namespace {

constexpr int BC = 256;        // weight rows of a tile

struct Product {
  const short *x, *w;          // [M, K], [N, K]
  int64_t x_row, w_row;        // strides in elements
  float* y;                    // [parts, M, N]
  int M, N, K, parts;
  uint32_t x_bytes, w_bytes;
};

template <int PT>
__global__ __launch_bounds__(256, 1) void linear_split_kernel(const Product p) {
  typedef TileCore<8, PT, 2> Core;
  constexpr int LW = Core::LW, LP = Core::LP, BR = Core::ROWS;
  static_assert(Core::CHANNELS == BC, "");
  extern __shared__ __align__(16) short split_lds[];
  // Workgroups go round the 8 XCDs in turn: each gets a contiguous share, in
  // which the tiles of all rows walk the channels of a part of K together.
  const int nx = (p.N + BC - 1) / BC, ny = (p.M + BR - 1) / BR;
  const int id = blockIdx.x % 8 * (gridDim.x / 8) + blockIdx.x / 8;
  if (id >= nx * ny * p.parts) return;
  const int m0 = id % ny * BR, n0 = id / ny % nx * BC, part = id / ny / nx;
  const int M = p.M, N = p.N, all = p.K / TILE_K;
  const int first = (int)((int64_t)all * part / p.parts);
  const int steps = (int)((int64_t)all * (part + 1) / p.parts) - first;
  Core core;
  // rows and channels past the end repeat the last one and are dropped
  uint32_t wsrc[2][LW], xsrc[2][LP];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
#pragma unroll
    for (int j = 0; j < LW; ++j) {
      const int n = n0 + h * Core::CH + core.template loaded<LW>(j);
      wsrc[h][j] = (uint32_t)(min(n, N - 1) * p.w_row +
                              core.template piece<LW>(j)) * 2;
    }
#pragma unroll
    for (int j = 0; j < LP; ++j) {
      const int m = m0 + h * Core::RH + core.template loaded<LP>(j);
      xsrc[h][j] = (uint32_t)(min(m, M - 1) * p.x_row +
                              core.template piece<LP>(j)) * 2;
    }
  }
  core.run(split_lds, p.w, p.w_bytes, wsrc, p.x, p.x_bytes, xsrc, steps,
           [&](int s) { return (first + s) * TILE_K * 2; });
#pragma unroll
  for (int t = 0; t < PT; ++t) {
    const int m = m0 + core.row(t) + core.col;
    if (m >= M) continue;
    const int64_t o = ((int64_t)part * M + m) * N;
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      const int n = n0 + core.channel(c) + core.grp * 4;
      if (n >= N) continue;            // N is a multiple of 4
      *(float4v*)(p.y + o + n) = core.acc[c][t];
    }
  }
}

template <int PT>
hipError_t go(const Product& p, hipStream_t stream) {
  typedef TileCore<8, PT, 2> Core;
  const int64_t n = (int64_t)((p.N + BC - 1) / BC) *
                    ((p.M + Core::ROWS - 1) / Core::ROWS) * p.parts;
  if (n > 1 << 24) return hipErrorInvalidValue;
  auto fn = linear_split_kernel<PT>;
  const hipError_t e = hipFuncSetAttribute(
      (const void*)fn, hipFuncAttributeMaxDynamicSharedMemorySize, Core::LDS);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(fn, dim3((uint32_t)((n + 7) / 8 * 8)), dim3(256), Core::LDS,
                     stream, p);
  HIP_CHECK_LAST();
  return hipSuccess;
}

}  // namespace

extern "C" {

// Rows of a tile | parts of K << 16 with the least time by this measure, 0 if one
// part is best, which the library does as well (0.9 to 1.2 times as fast). us: a
// step of 64 and round of the compute units takes 1.5 (192 rows: 1.12), two fifths
// of that for the power that all of them draw; parts are written and read at 4.5
// TB/s. Below 5120 of K parts gain nothing either (4096 -> 6144, 523 rows: library
// 41, here 42; 4096 -> 4096, 978 rows: 44 and 47). Over 140 draws of 10 sizes with K
// from there on and 257 to 2400 rows, where there are parts: 1.01 to 2.1 times as
// fast as the library. (More rows and narrower products were not compared.)
int lds_linear_split_plan(int64_t M, int64_t N, int64_t K) {
  if (M <= 256 || M > 2560 || N < 1024 || N > BC * 256 || N % 8 || K < 5120 ||
      K % TILE_K)
    return 0;
  const int64_t nx = (N + BC - 1) / BC, all = K / TILE_K;
  int best = 0;
  float least = 1e30f;
  for (int rows = 192; rows <= 256; rows += 64)
    for (int64_t parts = 1; parts <= 16; ++parts) {
      const int64_t tiles = nx * ((M + rows - 1) / rows) * parts;
      if (parts > 1 && tiles > 256) break;
      const int64_t rounds = (tiles + 255) / 256;
      const float busy = rounds > 1 ? 1.f : tiles / 256.f;
      const float step = (rows == 256 ? 1.5f : 1.12f) * (0.6f + 0.4f * busy);
      float us = rounds * ((all + parts - 1) / parts) * step;
      if (parts > 1) us += 3.f + parts * M * N * 8 / 4.5e6f;
      if (us < least) {
        least = us;
        best = parts > 1 ? rows | (int)parts << 16 : 0;
      }
    }
  return best;
}

hipError_t lds_sum_parts(const float* part, void* y, int64_t n, int parts,
                         int f32, int act, hipStream_t stream);

// x [M, K], w [N, K], rows x_row and w_row apart, 16-byte aligned, K a multiple of 64
// with 128 per part at least, N one of 4; plan: of the function above. part [parts,
// M, N] 32-bit and its sum y [M, N] in bf16; without y the result stays in part.
hipError_t lds_linear_split(const void* x, int64_t x_row, const void* w,
                            int64_t w_row, void* y, float* part, int plan,
                            int M, int N, int K, hipStream_t stream) {
  const int rows = plan & 0xffff, parts = plan >> 16;
  if (M < 1 || N < 4 || N % 4 || K % TILE_K || parts < 1 ||
      K / TILE_K / parts < 2 || x_row % 8 || w_row % 8 ||
      (rows != 192 && rows != 256))
    return hipErrorInvalidValue;
  const int64_t xb = ((M - 1) * x_row + K) * 2;
  const int64_t wb = (((int64_t)N - 1) * w_row + K) * 2;
  if (xb >= 1ll << 32 || wb >= 1ll << 32) return hipErrorInvalidValue;
  const Product p{(const short*)x, (const short*)w, x_row, w_row, part,
                  M, N, K, parts, (uint32_t)xb, (uint32_t)wb};
  const hipError_t e = rows == 192 ? go<6>(p, stream) : go<8>(p, stream);
  if (e != hipSuccess || !y) return e;
  return lds_sum_parts(part, y, (int64_t)M * N, parts, 0, -1, stream);
}

}  // extern "C"
