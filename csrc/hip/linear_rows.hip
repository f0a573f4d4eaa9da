// linear_rows.hip — y = x w' for few rows of x (bf16, 32-bit sums): the kernel
// for up to 64 rows, and which product goes where. Others of up to 256 rows go to
// linear_tiles.hip.
//
// The weights' bytes are what counts. A workgroup has all rows of x against 128 rows of
// w by the loop of rows_core.h, and K is split until the workgroups make up a round of
// the 256 compute units; or K is one part, and the rows of w are dealt out in even
// rounds, 16 to 128 to a workgroup. Where the parts are left to the caller, and in gated
// products by whole blocks of 128, linear_tiles.hip adds up in the same order, so a row
// comes out the same, to the bit, whichever of the two took it: as the one row of a decode
// step or within a short prompt. Elsewhere how K is shared out, over parts or over groups
// of waves, hangs on the number of rows, and so do a row's last bits.
//
// Measured, cold weights, without the sum of the parts; before: weights by way of the L2
// caches like x (and 128 bytes of a row at a time): 1 row, 4096 -> [2 x 14336] 38.3 us,
// 6.1 TB/s (41.8, 43.7; library 58 and the activation), 4096 -> 6144 10.4 (11.1, 11.4),
// 14336 -> 4096 20.2 (22.4, 22.4), 4096 -> 4096 7.5 (7.8, 8.4), 25600 -> 5120 42.1 (47.4,
// 47.6); 30 rows 39.3, 11.4, 21.5, 8.5, 44.2 (42.3, 12.0, 23.4, 8.7, 49.3).
#include "rows_core.h"

namespace {

using namespace rows_core;

struct Rows {
  const short *x, *w;        // [M, K], [N, K] (GATED: [2 N, K], gate first)
  int64_t x_row, w_row;      // strides in elements
  void* y;                   // [M, N]; F32: [parts, M, N] 32-bit
  int M, N, K, k_part;       // k_part: K per part, a multiple of KS
  int parts, act;
  int width;                 // rows of w of a workgroup, a multiple of UNIT
  int first;                 // blocks of the first of two products of one shape, or 0
  const short *x2, *w2;
  void* y2;
};

// what becomes of the sums: bf16, 32-bit (also of a part of K), act of them or
// act(gate) * up as bf16
enum Out { BF16, F32, ACT, GATED };

constexpr int ROUND = 256;       // compute units
constexpr int UNIT = 8;

// RT: rows of x / 16. BN rows of w; KG: groups of BN / 16 waves, each with its share of
// K, whose sums meet at the end. A wave has CT tiles of 16 channels by MT of 16 rows.
template <int RT, int BN, int KG, int OUT>
__global__ __launch_bounds__(BN / 16 * KG * WAVE) void linear_rows_kernel(
    const Rows p) {
  extern __shared__ __align__(16) char lds[];
  typedef RowsCore<RT, BN> Core;
  constexpr int NW = Core::NW, WC = Core::WC, CT = Core::CT, MT = Core::MT;
  constexpr int WL = Core::WL, XL = Core::XL;
  const int all = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
  const int group = all / NW, wave = all % NW;
  const int lane = threadIdx.x % WAVE, col = lane % 16, grp = lane / 16;
  const int M = p.M, N = p.N;
  const int part = blockIdx.x % p.parts;
  int blk = p.parts > 1 ? blockIdx.x / p.parts
                        : along_xcd(blockIdx.x, gridDim.x, ROUND);
  const short *x = p.x, *w = p.w;
  void* y = p.y;
  if (p.first && blk >= p.first) {
    blk -= p.first;
    x = p.x2;
    w = p.w2;
    y = p.y2;
  }
  const int width = p.width, n0 = OUT == GATED ? blk * (width / 2) : blk * width;
  if (n0 >= N) return;
  // this group's K: steps of KS, the last ones past the end where they do not go round
  const int p_lo = part * p.k_part, p_hi = min(p.K, p_lo + p.k_part);
  const int steps = ((p_hi - p_lo + KS - 1) / KS + KG - 1) / KG;
  const int k_lo = p_lo + group * steps * KS, k_hi = min(p_hi, k_lo + steps * KS);
  // by blocks of 128 rows of w, as in linear_tiles.hip
  const int first = (OUT == GATED    ? blk * width / 128 * 6
                     : N > 128 * 256 ? blk * width / 256 * 3
                                     : blk * width / 128 * 3) %
                    steps;
  // Rows that do not exist repeat the last one. GATED: of 16 rows of w 8 are of gate, 8
  // the same ones of up.
  const int n1 = min(N, n0 + (OUT == GATED ? width / 2 : width));
  const short *w_from[WL], *x_from[XL];
#pragma unroll
  for (int j = 0; j < WL; ++j) {
    const int r = Core::w_row(wave, j) + grp;          // row in LDS
    const int n = OUT == GATED ? r / 16 * 8 + r % 8 : r;
    const bool up = OUT == GATED && r % 16 >= 8;
    w_from[j] = w + (min(n0 + n, n1 - 1) + (up ? N : 0)) * p.w_row + Core::piece(r, lane);
  }
#pragma unroll
  for (int j = 0; j < XL; ++j) {
    const int r = Core::x_row(wave, j) + grp;
    x_from[j] = x + min(r, M - 1) * p.x_row + Core::piece(r, lane);
  }
  float4v acc[CT][MT];
  Core::run(lds + group * Core::RINGS, wave, lane, w_from, x_from, k_lo, k_hi, steps,
            first, wave * 16 < width, acc);
  const int wc = wave % WC, wm = wave / WC;      // its channels, its rows

  if constexpr (KG > 1) {                  // to the sums of the first group
    constexpr int ONE = CT * MT * NW * WAVE;
    static_assert((KG - 1) * ONE * 16 <= KG * Core::RINGS, "");
    float4v* other = (float4v*)lds;
    __syncthreads();                       // the rings are no longer read
#pragma unroll
    for (int c = 0; c < CT; ++c)
#pragma unroll
      for (int t = 0; t < MT; ++t)
        if (group > 0)
          other[(group - 1) * ONE + ((c * MT + t) * NW + wave) * WAVE + lane] =
              acc[c][t];
    __syncthreads();
    if (group > 0) return;
#pragma unroll
    for (int i = 0; i < KG - 1; ++i)
#pragma unroll
      for (int c = 0; c < CT; ++c)
#pragma unroll
        for (int t = 0; t < MT; ++t)
          acc[c][t] += other[i * ONE + ((c * MT + t) * NW + wave) * WAVE + lane];
  }
  // lane: row `col` of a tile, channels 4 grp ..; GATED: gate with the lower half of the
  // lanes, up with the other, and of two tiles each half takes one
#pragma unroll
  for (int t = 0; t < MT; ++t)
#pragma unroll
    for (int c = 0; c < CT; c += OUT == GATED ? 2 : 1) {
      const int m = (wm * MT + t) * 16 + col;
      int n = n0 + (wc * CT + c) * 16 + grp * 4;
      float4v s = acc[c][t];
      if constexpr (OUT == GATED) {
        n = n0 + (wc * CT + c + grp / 2) * 8 + grp % 2 * 4;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const auto both = __builtin_amdgcn_permlane32_swap(
              __float_as_uint(s[r]), __float_as_uint(acc[CT == 1 ? c : c + 1][t][r]),
              false, false);
          s[r] = activate(p.act, __uint_as_float(both[0])) * __uint_as_float(both[1]);
        }
        if (CT == 1 && grp >= 2) continue;
      }
      if (m >= M || n >= n1) continue;     // n1 - n0 is a multiple of 4
      const int64_t o = ((int64_t)part * M + m) * N + n;
      if constexpr (OUT == F32) {
        *(float4v*)((float*)y + o) = s;
      } else {
        short4v v;
#pragma unroll
        for (int r = 0; r < 4; ++r)
          v[r] = f32_to_bf16(OUT == ACT ? activate(p.act, s[r]) : s[r]);
        *(short4v*)((short*)y + o) = v;
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

// Rows of w of a workgroup where K is one part: as many rounds of the chip as by 128,
// each full, unless they nearly are by 128 (16 rows, by 128 / so: 8668 x 5640 gated 52.1 /
// 41.2 us, 17408 x 5120 87.4 / 69.0, 25600 x 5120 99.4 / 92.5, 20480 x 2048 37.7 / 33.4;
// 36864 x 4096 plain 66.1 / 54.5, 41000 x 3072 54.2 / 48.5; by 64 / so: 1960 x 6160 gated
// 27.5 / 17.6, 3072 x 1024 plain 5.8 / 4.8, 6720 x 6456 31.6 / 22.4).
int even_width(int rows) {
  const int blocks = (rows + 127) / 128, slots = (blocks + ROUND - 1) / ROUND * ROUND;
  if (blocks * 8 >= slots * 7) return 128;
  const int width = ((rows + slots - 1) / slots + UNIT - 1) / UNIT * UNIT;
  return width < 16 ? 16 : width;
}

template <int RT, int BN, int KG, int OUT>
hipError_t go(Rows p, hipStream_t stream) {
  constexpr int bytes = KG * RowsCore<RT, BN>::RINGS;
  auto fn = linear_rows_kernel<RT, BN, KG, OUT>;
  const hipError_t e = hipFuncSetAttribute(
      (const void*)fn, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
  if (e != hipSuccess) return e;
  const int rows = (OUT == GATED || p.x2 ? 2 : 1) * p.N;        // of w
  p.width = p.parts > 1 ? BN : even_width(rows);
  const int ch = OUT == GATED ? p.width / 2 : p.width;
  int groups = (p.N + ch - 1) / ch * p.parts;
  if (p.x2) {
    p.first = groups;
    groups *= 2;
  }
  if (p.parts == 1) groups = (groups + 7) / 8 * 8;     // equal shares of the XCDs
  hipLaunchKernelGGL(fn, dim3(groups), dim3(BN / 16 * KG * WAVE), bytes, stream,
                     p);
  HIP_CHECK_LAST();
  return hipSuccess;
}

// Where few rows of w come to a workgroup K is shared out inside it, as far as the rings
// fit, so that more is under way (1, 16 and 50 rows, in us: K whole by 64 rows of w; in
// halves by 64; as it is here):
//   4096 -> 1024           12.8, 13.6, 18.4    10.6, 10.8, 15.3     6.9,  7.6, 12.8
//   4096 -> 6144           16.4, 17.0, 21      14.0, 14.3, 18.1    11.9, 12.5, 16.6
//   8192 -> [2 x 2048]     30.1, 30.6, 42      21.7, 21.4, 30.4    15.2, 15.9, 25.2
//   4096 -> 10240          21.0, 21.2, 23.9    19.7, 19.7, 22.4    19.2, 19.6, 23.9
// Parts of a few steps are taken by 64 too, two workgroups per compute unit, whose ends
// overlap (4096 -> 4096, parts of 512: 7.4 us, 7.6 by 128, 30 rows 8.3, 8.5; parts of 896
// up: 22.1, 21.9).
template <int RT, int OUT>
hipError_t go_width(const Rows& p, hipStream_t stream) {
  const int rows = (OUT == GATED || p.x2 ? 2 : 1) * p.N;        // of w
  if (p.parts == 1 && rows <= 32 * ROUND)
    return go<RT, 32, RT == 1 ? 4 : 2, OUT>(p, stream);
  if (p.parts == 1 && rows <= 64 * ROUND)
    return go<RT, 64, RT == 4 ? 1 : 2, OUT>(p, stream);
  if constexpr (OUT == F32)
    if (p.parts > 1 && p.k_part <= 512) return go<RT, 64, 1, OUT>(p, stream);
  if constexpr (OUT == ACT) return hipErrorInvalidValue;
  else return go<RT, 128, 1, OUT>(p, stream);
}

template <int OUT>
hipError_t go_rows(const Rows& p, hipStream_t stream) {
  return p.M <= 16   ? go_width<1, OUT>(p, stream)
         : p.M <= 32 ? go_width<2, OUT>(p, stream)
                     : go_width<4, OUT>(p, stream);
}

// Up to 64 rows come here, up to 32 where K is split, more go to linear_tiles.hip (60
// rows, here / there: 4096 -> [2 x 14336] 44.0 us / 50.2, 4096 -> 6144 in 5 parts 13.4 /
// 12.7, 4096 -> 4096 in 8 11.4 / 10.1, 14336 -> 4096 in 8 24.8 / 24.7).
constexpr int ROWS = 64, SPLIT_ROWS = 32, TILE_ROWS = 256;

// Of one part of K, by which the split and the rule below are reckoned: of 256 rows
// of w for up to 16 of x where 128 are more than a round
int workgroups(int M, int N) {
  const int width = M <= 16 && N > 128 * 256 ? 256 : 128;
  return (N + width - 1) / width;
}

// Whether workgroups fill 7/8 of their rounds
bool fills(int groups) {
  return groups * 8 >= (groups + ROUND - 1) / ROUND * ROUND * 7;
}

// Whether a gated product that fills no round of the chip is faster here, up to 64 rows,
// than as a product and its activation, by the blocks of 64 channels that K takes: the
// more rows, the fewer groups of waves share K out. own: that product is one of this
// file, not the library's. Here / there:
//                  16 rows   17     32     33     64
//   2560 x  256     0.78    0.92   0.93   0.99   1.03
//   2800 x  192     0.79    0.87   0.86   0.86   0.97
//   3072 x  256     0.81    1.00   0.96   1.05   1.07
//   3392 x  520     0.81    1.09   1.05   1.14   1.10
//   3840 x 1296     0.82    0.83   0.84   1.03   0.94
//   4096 x   64     0.83    1.15   1.10   1.22   1.24
//   4096 x  768     0.80    0.92   0.87   1.05   1.00
//   4712 x 2336     0.89    0.53   0.57   0.67   0.70 (library)
//   5120 x 2048     0.87    0.84   0.86   1.00   1.06
//   5120 x 4096     0.90    0.90   0.89   0.94   0.94
//   7168 x 3072     0.92    0.91   0.92   1.00   1.03
//   8192 x 4096     0.98    1.10   1.06   1.04   1.03
bool enough_blocks(int M, int blocks, int K, bool own) {
  if (M <= 16)
    return K <= 4096 || (K <= 6144 && blocks >= 32) || (K <= 8192 && blocks >= 48);
  if (M <= 32)
    return K <= 3072 || (K <= 4096 && blocks >= 12) || (K <= 6144 && blocks >= 32) ||
           (K < 8192 && blocks >= 48);
  return K <= 2688 || (K < 3072 && blocks >= 2) || (K <= 3072 && blocks >= 8) ||
         (K <= 4096 && blocks >= 16) || (K <= 4736 && blocks >= 32) ||
         (K <= 6144 && ((blocks >= 48 && M <= 40) || (blocks >= 32 && !own))) ||
         (K < 8192 && blocks >= 64);
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

// The same where the sum of the parts is a launch of its own (3 to 5 us): one part of
// short K, or of many channels, the more of them the more rows there are. From 33 rows
// on three parts or four that make up their round are faster still where K is long, but
// four of a power of two, which begin at the same memory channels in every row. One part /
// parts and their sum, in us:
//                     1 row        16 rows      32 rows      50 rows
//   1536 -> 1024      4.4 /  6.2    4.8 /  6.8   5.7 /  7.1   6.6 /  8.2
//   2048 -> 4096      5.8 /  8.8    6.2 /  9.6   7.2 / 10.4   8.5 / 12.4
//   3072 -> 2048      6.1 /  7.8    6.8 /  8.5   8.8 /  9.2  10.4 / 10.2
//   4096 -> 1024      7.0 /  7.7    7.5 /  8.6  10.6 /  9.0  12.6 / 10.1
//   4096 -> 4096      8.7 / 11.6    9.3 / 12.2  11.6 / 12.5  13.8 / 13.6
//   4096 -> 8192     15.6 / 17.7   15.9 / 18.7  17.4 / 19.0  19.0 / 20.0
//   8192 -> 2048     11.5 / 12.1   12.6 / 12.9  18.7 / 13.6  22.5 / 14.6
//   8192 -> 8192     25.7 / 31.5   26.3 / 32.3  26.8 / 33.2  31.7 / 34.3
// and their ratio:    17 rows  32 rows            33 rows  48 rows  64 rows
//   4096 -> 2304       1.14     1.06    5120 ->  8192  1.06  1.08  1.05
//   3840 -> 2560       1.10     1.00    7680 ->  8192  1.04  1.14  1.13
//   4096 -> 3072       0.97     0.90    4096 -> 10240  1.07  1.07  1.09
//   3072 -> 2048       1.02     0.94    6144 -> 10240  1.10  1.04  1.03
// (8192 -> 9216, whose three parts do not fill their round, takes 42.4 us, 33 rows, the
// library 38.6.)
int lds_linear_plain_parts(int M, int N, int K) {
  const int parts = lds_linear_rows_parts(M, N, K);
  if (M > ROWS || N > 64 * ROUND || K > 8192) return parts;
  const bool round = K >= 4096 && (parts == 3 || (parts == 4 && K % 4096)) &&
                     (fills(workgroups(M, N) * parts) || (parts == 3 && K >= 8192));
  const bool one =
      K <= 2048 || (M <= 16   ? K <= 4096 || N >= 2048
                    : M <= 32 ? N >= (K <= 3072 ? 2048 : K <= 4096 ? 2816 : 6144)
                              : N >= (K <= 3072 ? 3072 : 8192) && !round);
  return one ? 1 : parts;
}

// Whether a product of M rows is faster here than in the library. Device
// times, here / there, in us:
//   parts the caller sums itself: always. 4096 -> 4096: 1 row 8 / 15, 96 rows
//     12 / 22, 256 rows 18 / 23; 14336 -> 4096: 64 rows 23 / 40, 256 rows
//     41 / 63; 4096 -> 12576: 64 rows 24 / 25, 256 rows 42 / 50. (Above 128 rows
//     a K below 1600 takes up to 3 us more here, 688 -> 1680, 256 rows 13 / 10;
//     that it comes out as a single row does is worth it.)
//   one part, and gated ones (there with their activation), up to 64 rows: if the
//     workgroups fill at least 7/8 of their rounds. 4096 -> 32768: 32 rows 46 / 62; ->
//     128256 (98 %): 64 rows 182 / 208; 5120 -> 51200 (78 %): 64 rows 110 / 98; 4096 ->
//     [2 x 14336]: 64 rows 44 / 58. Gated ones need not fill their round (enough_blocks;
//     16 rows, 256 -> [2 x 2304] 4.0 / 12).
//   the same of 65 rows and more, ratio of the times over 140 sizes:
//     one round, of which plain ones fill more than half: 0.63 to 1.0 but for three of
//     1.05 to 1.08 (143 blocks, 128 rows, K of 5248 the most). 0.95 to 1.0 from a K of
//     11392 on, so that longer ones stay away. Gated: from 5/8 of the round on 0.64 to
//     0.97, 105 to 128 blocks 0.9 to 1.25; above 192 rows K of 15872 1.13.
//     more rounds, 7/8 full: up to 128 rows 0.66 to 1.0, 192 rows 0.79 to 1.04 for K up to
//     4096 and 0.83 to 1.11 for more; 256 rows 1.07 to 1.22 in two rounds, in three to
//     five 0.85 to 1.02 for K up to 4224 (128256 x 4096 264 / 300 us), gated 0.88 to 1.13.
//     Less full ones 1.02 to 1.34.
//   parts and their sum (3 to 5 us): with full rounds (4096 -> 6144: 64 rows
//     16 / 18, 160 rows 23 / 28; 8192 -> 5120: 256 rows 40 / 74) unless K is
//     short (2048 -> 8192: 64 rows 13.3 / 14.0, 128 rows 17.7 / 16.8), else
//     narrow ones up to 64 rows (4096 -> 1024: 64 rows 11 / 15, 96 rows
//     13 / 12), or of one part (lds_linear_plain_parts; 2048 -> 8192: 50 rows 11.0 /
//     13.5; 4096 -> 8192: 16 rows 16.8 / 16.4, 50 rows 19.6 / 18.6, -> 10240 19.9 / 26.0,
//     22.1 / 27.5, -> 12576 23.4 / 28.4, 26.6 / 26.7; 8192 -> 8192 27.1 / 30.3).
//   more than 16384 rows of w, in even rounds (even_width): up to 64 rows, K from 512 to
//     10240. Over 76 sizes of 16384 to 130000 rows of w, gated and plain, 4 to 64 rows of
//     x, 1.3 times as fast at the median; slower by 3 and 6 % at two (51200 x 5120 and
//     49152 x 1024, plain, 64 rows), and past that range 53248 x 16384 649 / 622.
int lds_linear_rows_takes(int M, int N, int K, int gated, int parts) {
  if (M > TILE_ROWS) return 0;
  if (!gated && parts && lds_linear_rows_parts(M, N, K) > 1) return 1;
  const int n = gated ? 1 : lds_linear_plain_parts(M, N, K);
  const int groups = gated ? (N + 63) / 64 : workgroups(M, N) * n;
  const bool full = fills(groups);
  const bool one_round = M > ROWS && groups <= ROUND && groups * 8 >= ROUND * 5;
  if (M <= ROWS && (gated ? 2 : 1) * N > 128 * 128 && K >= 512 && K <= 10240) return 1;
  if (gated && M <= ROWS && groups <= 256 && K >= 256 &&
      enough_blocks(M, groups, K, lds_linear_rows_takes(M, 2 * N, K, 0, 0)))
    return 1;
  if (gated)
    return M <= 192 ? full || one_round
                    : one_round && K >= 1024 && K <= 8192 && K % KS == 0;
  if (N > 128 * 128)
    return M <= ROWS         ? full
           : groups <= ROUND
               ? K <= 12288
               : full && (M <= 128 || (K <= 4096 && (M <= 192 || (groups > 2 * ROUND &&
                                                                  K >= 1024))));
  if (full) return M <= 64 || K >= 4096;
  return M <= ROWS && (N <= 4096 || n == 1);
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

// x [M, K], w [N, K], rows x_row and w_row apart and 16-byte aligned, N a multiple of 8; y
// [M, N]
// bf16 or (f32) 32-bit. part: [parts, M, N] floats if parts > 1; without y
// the result stays there.
hipError_t lds_linear_rows(const void* x, int64_t x_row, const void* w,
                           int64_t w_row, void* y, float* part, int parts,
                           int M, int N, int K, int f32, hipStream_t stream) {
  if (M < 1 || M > TILE_ROWS || N < 1 || N % 8 || K < 8 || K % 8 ||
      x_row % 8 || w_row % 8 || parts < 1 || (!part && (parts > 1 || !y)))
    return hipErrorInvalidValue;
  const bool in_part = parts > 1 || !y;
  hipError_t e;
  if (M > ROWS || (M > SPLIT_ROWS && parts > 1)) {
    e = lds_linear_tiles(x, x_row, w, w_row, in_part ? part : y, parts, M, N,
                         K, in_part || f32, -1, stream);
  } else {
    Rows p{(const short*)x, (const short*)w, x_row, w_row,
           in_part ? part : y, M, N, K, K, parts, 0};
    p.k_part = ((K + parts - 1) / parts + KS - 1) / KS * KS;
    if ((K + p.k_part - 1) / p.k_part != parts) return hipErrorInvalidValue;
    e = in_part || f32 ? go_rows<F32>(p, stream) : go_rows<BF16>(p, stream);
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

// y [M, N] = act(x gate') * (x up'), w [2 N, K] = [gate; up], N a multiple of 8
hipError_t lds_gated_rows(const void* x, int64_t x_row, const void* w,
                          int64_t w_row, void* y, int M, int N, int K, int act,
                          hipStream_t stream) {
  if (M < 1 || M > TILE_ROWS || N < 1 || N % 8 || K < 8 || K % 8 ||
      x_row % 8 || w_row % 8 || act < 0 || act >= ACTS)
    return hipErrorInvalidValue;
  if (M > ROWS)
    return lds_linear_tiles(x, x_row, w, w_row, y, 1, M, N, K, 0, act, stream);
  const Rows p{(const short*)x, (const short*)w, x_row, w_row, y, M, N, K,
               (K + KS - 1) / KS * KS, 1, act};
  return go_rows<GATED>(p, stream);
}

// y [M, N] = act(x w') of one part, for up to 64 rows and 128 x 128 channels
hipError_t lds_activated_rows(const void* x, int64_t x_row, const void* w,
                              int64_t w_row, void* y, int M, int N, int K,
                              int act, hipStream_t stream) {
  if (M < 1 || M > ROWS || N < 1 || N % 4 || N > 128 * 128 || K < 8 || K % 8 ||
      x_row % 8 || w_row % 8 || act < 0 || act >= ACTS)
    return hipErrorInvalidValue;
  const Rows p{(const short*)x, (const short*)w, x_row, w_row, y, M, N, K,
               (K + KS - 1) / KS * KS, 1, act};
  return go_rows<ACT>(p, stream);
}

// Two products of one shape and one part, y = x w' and y2 = x2 w2', in a launch, for up to
// 64 rows (two of 128 -> 4096, 50 rows: 3.9 us each)
hipError_t lds_linear_pair(const void* x, const void* x2, int64_t x_row,
                           const void* w, const void* w2, int64_t w_row, void* y,
                           void* y2, int M, int N, int K, hipStream_t stream) {
  if (M < 1 || M > ROWS || N < 1 || N % 4 || N > 1 << 24 || K < 8 || K % 8 ||
      x_row % 8 || w_row % 8 || !x2)
    return hipErrorInvalidValue;
  const Rows p{(const short*)x, (const short*)w, x_row, w_row, y, M, N, K,
               (K + KS - 1) / KS * KS, 1, -1, 0, 0, (const short*)x2,
               (const short*)w2, y2};
  return go_rows<BF16>(p, stream);
}

}  // extern "C"
