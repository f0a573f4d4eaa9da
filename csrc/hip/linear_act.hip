// linear_act.hip — y = act(x gate') * (x up') and y = act(x w') for many rows
// (bf16, 32-bit sums): tiles of 256 weight rows by 256 or 192 rows of x by the loop
// of tile_core.h, the activation in the sums' registers.
//
// The library's product of the same weights is 3 % faster, but its result, twice
// as wide where a gate is in it, goes to memory and comes back for the activation:
// a tenth of the product's time. A wave's channels of gate and up are the same ones,
// 64 of the first and of the second half of the tile's weight rows, so that both
// sums are in one lane.
#include "layered/elem.h"
#include "tile_core.h"

namespace {

template <int PT> using Whole = TileCore<8, PT, 2>;    // 32 PT rows
typedef TileCore<4, 8, 4> Half;       // the last tile, of up to 128
constexpr int BC = Whole<8>::CHANNELS;
static_assert(Half::CHANNELS == BC && Half::CH == Whole<8>::CH &&
                  Half::LDS_TURN <= Whole<6>::LDS_TURN,
              "");
constexpr int TG = 4;        // tiles of rows that walk the channels together

struct Product {
  const short *x, *w;        // [M, K], [N, K] (GATED: [2 N, K], gate first)
  int64_t x_row, w_row;      // strides in elements
  short* y;                  // [M, N]
  int M, N, K, act;
  uint32_t x_bytes, w_bytes;
  int whole;                 // tiles ahead of those that are cut in two
};

// As activate() of elem.h, by the exponential and the reciprocal of the hardware. The
// exponential's argument is rounded, so the error grows with it, to |a| 2^-24 (2^-18 at
// -80) and a few 2^-24: far below the 2^-8 of the bf16 result. Of 27468 sums in bf16 up
// to 200, one silu rounds the other way (5.9375). The reciprocal is taken of a value
// 2^-24 as large: past 2^126 it would be no normal number, 0 on this hardware, where
// the activation still is one (-9e-37 at -87.5).
__device__ __forceinline__ float times_sigmoid(float z, float a) {
  return z * 0x1p-24f * rcp_f(fmaf(__expf(-a), 0x1p-24f, 0x1p-24f));
}
template <int ACT>
__device__ __forceinline__ float act_f(float z) {
  if (ACT == ACT_RELU_SQUARED) return z > 0.f ? z * z : 0.f;
  if (ACT == ACT_SILU) return times_sigmoid(z, z);
  return times_sigmoid(z, 2.f * 0.7978845608028654f *
                              (z + 0.044715f * z * z * z));
}

template <int ACT, bool GATED, typename Core>
__device__ __forceinline__ void tile(const Product& p, short* lds, int m0, int blk) {
  Core core;
  constexpr int LW = Core::LW, LP = Core::LP, QC = Core::QC;
  constexpr int PT = Core::ROWS / 16 / Core::WP;
  const int M = p.M, N = p.N;
  // rows and channels past the end repeat the last one and are dropped
  uint32_t wsrc[2][LW], xsrc[2][LP];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
#pragma unroll
    for (int j = 0; j < LW; ++j) {
      const int r = core.template loaded<LW>(j);
      const int n = GATED ? h * N + min(blk * Core::CH + r, N - 1)
                          : min(blk * BC + h * Core::CH + r, N - 1);
      wsrc[h][j] = (uint32_t)(n * p.w_row + core.template piece<LW>(j)) * 2;
    }
#pragma unroll
    for (int j = 0; j < LP; ++j) {
      const int r = m0 + h * Core::RH + core.template loaded<LP>(j);
      xsrc[h][j] = (uint32_t)(min(r, M - 1) * p.x_row +
                              core.template piece<LP>(j)) * 2;
    }
  }
  core.run(lds, p.w, p.w_bytes, wsrc, p.x, p.x_bytes, xsrc, p.K / TILE_K,
           [](int s) { return s * TILE_K * 2; });
  const int n0 = blk * (GATED ? Core::CH : BC);
#pragma unroll
  for (int b = 0; b < PT / 2; ++b)
    core.template turn<GATED ? QC : 2 * QC>(
        lds, b,
        [&](int c, int t, int x) {
          const float z = act_f<ACT>(core.acc[c][t][x]);
          return GATED ? z * core.acc[GATED ? c + QC : c][t][x] : z;
        },
        [&](int, int r, int c, short8 v) {
          if (m0 + r < M && n0 + c < N)         // N is a multiple of 8
            *(short8*)(p.y + (int64_t)(m0 + r) * N + n0 + c) = v;
        });
}

template <int ACT, bool GATED, int PT>
__global__ __launch_bounds__(256, 1) void linear_act_kernel(const Product p) {
  extern __shared__ __align__(16) short act_lds[];
  constexpr int BR = Whole<PT>::ROWS;
  // Workgroups go round the 8 XCDs in turn: each gets a contiguous share of the
  // whole tiles, then one of the others, in which TG tiles of rows walk the channels
  // together.
  constexpr int width = GATED ? BC / 2 : BC;
  const int nx = (p.N + width - 1) / width, ny = (p.M + BR - 1) / BR;
  const bool cut = (int)blockIdx.x >= p.whole && p.whole > 0;
  const int b = cut || p.whole == 0 ? blockIdx.x - p.whole : blockIdx.x;
  const int share = (cut || p.whole == 0 ? gridDim.x - p.whole : p.whole) / 8;
  const int at = b % 8 * share + b / 8;
  const int id = cut ? p.whole + at / 2 : at;
  if (id >= nx * ny) return;
  const int g = id / (TG * nx), in = id % (TG * nx);
  const int side = min(TG, ny - g * TG);
  const int m0 = (g * TG + in % side) * BR + (cut ? at % 2 * Half::ROWS : 0);
  const int blk = in / side;
  if (m0 >= p.M) return;
  if (!cut && p.M - m0 > Half::ROWS)
    tile<ACT, GATED, Whole<PT>>(p, act_lds, m0, blk);
  else
    tile<ACT, GATED, Half>(p, act_lds, m0, blk);
}

constexpr int CUS = 256;
// Tiles behind whole rounds of the compute units, up to half a round of them, are cut
// in two by rows: a half takes 0.65 of a round (4096 -> 7168, K = 4096: 42 us for 70 to
// 88). us, whole / so: 4096 -> 7168, 5400 rows 248 / 226, 7000 334 / 307, 7821 343 / 325,
// 8190 344 / 329; 2048 -> [2 x 8192], 8195 rows 430 / 414. More than half a round would
// take two rounds of halves.
bool cut_in_two(int64_t tiles) {
  return tiles > CUS && tiles % CUS > 0 && tiles % CUS <= CUS / 2;
}

template <int ACT, bool GATED, int PT>
hipError_t go(Product p, hipStream_t stream) {
  constexpr int width = GATED ? BC / 2 : BC, BR = Whole<PT>::ROWS;
  constexpr int bytes = Whole<PT>::LDS_TURN;
  int64_t n = (int64_t)((p.N + width - 1) / width) * ((p.M + BR - 1) / BR);
  if (n > 1 << 24) return hipErrorInvalidValue;
  p.whole = 0;
  if (BR == 2 * Half::ROWS && cut_in_two(n)) {
    p.whole = (int)(n / CUS * CUS);
    n += n - p.whole;
  }
  auto fn = linear_act_kernel<ACT, GATED, PT>;
  const hipError_t e = hipFuncSetAttribute(
      (const void*)fn, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(fn, dim3((uint32_t)((n + 7) / 8 * 8)), dim3(256), bytes,
                     stream, p);
  HIP_CHECK_LAST();
  return hipSuccess;
}

}  // namespace

extern "C" {

// Rows of a tile with which a product of many rows and its activation are one
// kernel: 256, or 192 where these fill their rounds over the compute units better by
// 1.08 (they are that much slower per row); 0 below 11/20 of a round's work. us,
// library and activation / here, behind it rows of a tile and how full. 4096 -> [2 x
// 14336]: 283 rows 96 / 70 (192, 64 %), 391 123 / 99 (256, 67 %), 524 152 / 139 (192,
// 60 %), 744 176 / 144 (192, 85 %; 256, 64 %: 172), 1014 213 / 180 (256, 87 %), 8190
// 1415 / 1298. 2048 -> [2 x 8192]: 565 rows 50 / 37 (192, 74 %), 1232 92 / 75 (192, 80
// %). 5120 -> [2 x 25600]: 320 rows 205 / 176 (192, 65 %), 1005 528 / 429 (256, 77 %;
// 192, 82 %: 468). 4096 -> 7168: 732 rows 61 / 66 (192, 42 %), 1047 69 / 62 (192, 60 %),
// 8190 376 / 329 (256, the last 128 tiles cut). 2048 -> 4096: 925 rows 31 / 33 (30 %), 2809 57 / 40 (192, 91 %).
// 5120 -> 12800: 565 rows 89 / 87 (192, 57 %). Cut tiles count as 0.65 of a round: by
// 192 and by 256 rows, 4096 -> [2 x 14336] 2400 rows 418 / 405, 2900 504 / 487, 4700
// 798 / 782, 2048 -> [2 x 8192] 4400 rows 234 / 226, 5120 -> 12800 5400 rows 508 / 491.
int lds_linear_act_rows(int64_t M, int64_t N, int64_t K, int gated) {
  const int64_t width = gated ? BC / 2 : BC;
  if (M <= 256 || K < 2 * TILE_K || K % TILE_K || N < 8 || N % 8) return 0;
  auto cost = [&](int64_t rows) {
    const int64_t tiles = (M + rows - 1) / rows * ((N + width - 1) / width);
    const int64_t last = rows == 2 * Half::ROWS && cut_in_two(tiles) ? CUS * 13 / 20 : CUS;
    return (tiles / CUS * CUS + (tiles % CUS ? last : 0)) * rows * width;
  };
  const int rows = cost(192) * 108 < cost(256) * 100 ? 192 : 256;
  return M * N * 20 >= cost(rows) * 11 ? rows : 0;
}

// y [M, N] = act(x gate') * (x up') of w [2 N, K] = [gate; up], or (not gated)
// act(x w') of w [N, K]; rows x_row and w_row apart, 16-byte aligned; K a multiple
// of 64 from 128 on, N one of 8; tiles of `rows` rows (192 or 256).
hipError_t lds_linear_act(const void* x, int64_t x_row, const void* w,
                          int64_t w_row, void* y, int rows, int M, int N,
                          int K, int act, int gated, hipStream_t stream) {
  const int64_t xb = ((M - 1) * x_row + K) * 2;
  const int64_t wb = (((gated ? 2 : 1) * (int64_t)N - 1) * w_row + K) * 2;
  if (M < 1 || N < 8 || N % 8 || K < 2 * TILE_K || K % TILE_K || x_row % 8 ||
      w_row % 8 || act < 0 || act >= ACTS || (rows != 192 && rows != 256) ||
      xb >= 1ll << 32 || wb >= 1ll << 32)
    return hipErrorInvalidValue;
  const Product p{(const short*)x, (const short*)w, x_row, w_row, (short*)y,
              M, N, K, act, (uint32_t)xb, (uint32_t)wb, 0};
#define GO(A)                                                                \
  return rows == 192                                                         \
             ? gated ? go<A, true, 6>(p, stream) : go<A, false, 6>(p, stream) \
         : gated ? go<A, true, 8>(p, stream)                                 \
                 : go<A, false, 8>(p, stream)
  if (act == ACT_SILU) GO(ACT_SILU);
  if (act == ACT_RELU_SQUARED) GO(ACT_RELU_SQUARED);
  GO(ACT_GELU_TANH);
#undef GO
}

}  // extern "C"
