// linear_tiles.hip — y = x w' for 65 to 256 rows of x, from 33 where K is split (bf16,
// 32-bit sums).
//
// The weights should be read from memory once, at its rate, so one workgroup
// has all rows of x (tiles of 64, up to four) against 128 rows of w, and K is
// split until the workgroups make up a round of the 256 compute units. Both
// operands go to LDS by direct loads, 64 of K at a time, into a ring of three
// or four steps, so that 64 to 96 KB per compute unit are under way. 8 waves
// of 64 channels by a quarter of the rows: operands of the next half of a step
// are read while the matrix cores work on this one, and the one barrier per
// step stands between the halves (without that overlap 4096 -> 28672, 256
// rows: 85 us for 75; 4 waves with twice the rows 99; two workgroups per
// compute unit of half the rows 87). Parts of K run fastest over the grid:
// with 8 of them each XCD's L2 holds one part of x. Workgroups start at
// different steps, as in linear_rows.hip.
//
// Measured, cold weights, without the sum of the parts (library): 4096 -> [2 x 14336]:
// 128 rows 53 us (60); 14336 -> 4096: 128 rows 28.4, 160 rows 35 (84), 256 rows 41
// (63); 25600 -> 5120: 256 rows 111 (260). Above 128 rows matrix cores and LDS bound it
// (with one row of x and of w repeated, nothing to fetch, 256 rows 64 of 75 us), and
// both operands' way to LDS: 4096 -> [2 x 14336], 178 rows 57 to 62 us, the loads alone
// 50, those of w 42, matrix cores and LDS without loads 30.
#include "layered/elem.h"
#include "tile_core.h"

namespace {

struct Tiles {
  const short *x, *w;        // [M, K], [N, K] (GATED: [2 N, K], gate first)
  int64_t x_row, w_row;      // strides in elements
  void* y;                   // [M, N]; F32: [parts, M, N] 32-bit
  int M, N, K, k_part;       // k_part: K per part, a multiple of 2 KS
  int parts, act;
  uint32_t x_bytes, w_bytes; // linear_wide
};

enum Out { BF16, F32, GATED };

constexpr int NW = 8, KS = 64, BN = 128;      // BN: rows of w per workgroup
constexpr int ROW = KS * 2;                   // bytes of a row in LDS

// The order of linear_rows.hip: steps of 128, starting at one by the channels.
template <int OUT>
__device__ __forceinline__ int start(int blk, int N, int steps) {
  return (OUT == GATED    ? blk * 6
          : N > 128 * 256 ? blk / 2 * 3
                          : blk * 3) %
         (steps / 2) * 2;
}

// 128 channels by 256 rows, a ring of three steps
typedef TileCore<4, 8, 2, 3> Wide;

// what is past the end of K
__device__ const float4v zeros = {0.f, 0.f, 0.f, 0.f};

// steps in the ring of 64 MT rows, and their LDS
constexpr int ring(int MT) { return MT <= 2 ? 4 : 3; }
constexpr int stage_bytes(int MT) { return (BN + 64 * MT) * ROW; }

template <int MT, int OUT>
__global__ __launch_bounds__(NW * WAVE, 2) void linear_tiles_kernel(
    const Tiles p) {
  extern __shared__ __align__(16) char lds[];
  constexpr int R = ring(MT), STAGE = stage_bytes(MT);
  constexpr int WL = BN * 8 / (NW * WAVE), XL = MT;    // loads of a thread
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
  const int lane = threadIdx.x % WAVE, col = lane % 16, grp = lane / 16;
  const int part = blockIdx.x % p.parts, blk = blockIdx.x / p.parts;
  const int k_lo = part * p.k_part, k_hi = min(p.K, k_lo + p.k_part);
  const int steps = (k_hi - k_lo + 2 * KS - 1) / (2 * KS) * 2;
  const int first = start<OUT>(blk, p.N, steps);
  const int M = p.M, N = p.N;

  // A load takes 8 rows of KS, 8 pieces of 16 bytes each; the pieces of a row
  // change places by XOR with its number halved, so that 16 lanes that read
  // one piece of 16 rows find 16 bank groups. Rows of w that do not exist
  // repeat the last one, as do rows of x.
  const int r8 = lane / 8;
  const short* from[WL + XL];
#pragma unroll
  for (int j = 0; j < WL; ++j) {
    const int r = (wave * WL + j) * 8 + r8;       // row in LDS
    int n;
    if (OUT == GATED)       // of 64 rows 32 gate, 32 up
      n = min(blk * (BN / 2) + r / 64 * 32 + r % 32, N - 1) +
          (r % 64 >= 32 ? N : 0);
    else
      n = min(blk * BN + r, N - 1);
    from[j] = p.w + n * p.w_row + (lane % 8 ^ (r / 2 % 8)) * 8;
  }
#pragma unroll
  for (int j = 0; j < XL; ++j) {
    const int r = (wave * XL + j) * 8 + r8;
    from[WL + j] =
        p.x + min(r, M - 1) * p.x_row + (lane % 8 ^ (r / 2 % 8)) * 8;
  }
  auto issue = [&](int s, int buf) {
    int k = s + first;
    k = k_lo + (k >= steps ? k - steps : k) * KS;
    char* b = lds + buf * STAGE;
    typedef const __attribute__((address_space(1))) unsigned int gmem;
    typedef __attribute__((address_space(3))) unsigned int smem;
#pragma unroll
    for (int j = 0; j < WL + XL; ++j) {
      const int r = j < WL ? wave * WL + j : BN / 8 + wave * XL + j - WL;
      const bool in = k + (lane % 8 ^ ((r * 8 + r8) / 2 % 8)) * 8 < k_hi;
      __builtin_amdgcn_global_load_lds(
          (gmem*)(in ? from[j] + k : (const short*)&zeros),
          (smem*)(b + r * 1024), 16, 0, 0);
    }
  };

  // wave: 64 channels, a quarter of the rows
  float4v acc[4][MT];
#pragma unroll
  for (int c = 0; c < 4; ++c)
#pragma unroll
    for (int t = 0; t < MT; ++t) acc[c][t] = (float4v){0.f, 0.f, 0.f, 0.f};
  const int wc = wave % 2, wm = wave / 2;
  struct Operands {
    bf16x8 w[4], x[MT];
  };
  // operands of 32 k
  const int w_at = (wc * 64 + col) * ROW;
  const int x_at = (BN + wm * 16 * MT + col) * ROW;
  const int piece0 = (grp ^ col / 2) * 16, piece1 = ((4 + grp) ^ col / 2) * 16;
  auto read = [&](Operands& o, int buf, int piece) {
    const char* b = lds + buf * STAGE + piece;
#pragma unroll
    for (int c = 0; c < 4; ++c)
      o.w[c] = *(const bf16x8*)(b + w_at + c * 16 * ROW);
#pragma unroll
    for (int t = 0; t < MT; ++t)
      o.x[t] = *(const bf16x8*)(b + x_at + t * 16 * ROW);
    __builtin_amdgcn_sched_barrier(0);    // all are under way before use
  };
  auto multiply = [&](const Operands& o) {
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
      for (int c = 0; c < 4; ++c)
        acc[c][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(o.x[t], o.w[c],
                                                            acc[c][t], 0, 0, 0);
    __builtin_amdgcn_sched_barrier(0);
  };
  // step s has landed, and so it has for the other waves, when only the loads
  // of later ones are under way
  constexpr int L = WL + XL;
  auto landed = [&](int s) {
    if (R > 3 && s + 2 < steps)
      asm volatile("s_waitcnt vmcnt(%0)" ::"i"((R - 2) * L) : "memory");
    else if (s + 1 < steps)
      asm volatile("s_waitcnt vmcnt(%0)" ::"i"(L) : "memory");
    else
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  auto after = [](int b) { return b + 1 == R ? 0 : b + 1; };

  // Operands are read one half of a step ahead of their products. At the
  // barrier in the middle of step s all of its operands are in registers: its
  // buffer takes step s + R.
#pragma unroll
  for (int s = 0; s < R - 1; ++s)
    if (s < steps) issue(s, s);
  Operands o0, o1;
  landed(0);
  if (R - 1 < steps) issue(R - 1, R - 1);
  read(o0, 0, piece0);
  int buf = 0;
  for (int s = 0; s < steps; ++s) {
    read(o1, buf, piece1);
    multiply(o0);
    if (s + 1 < steps) {
      landed(s + 1);
      if (s + R < steps) issue(s + R, buf);
      buf = after(buf);
      read(o0, buf, piece0);
    }
    multiply(o1);
  }

  // lane: channel `col` of a tile; register r: row 4 grp + r
#pragma unroll
  for (int t = 0; t < MT; ++t)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int m = (wm * MT + t) * 16 + grp * 4 + r;
      if (m >= M) continue;
      const int n = blk * (OUT == GATED ? BN / 2 : BN) +
                    wc * (OUT == GATED ? 32 : 64) + col;
      const int64_t o = ((int64_t)part * M + m) * N + n;
#pragma unroll
      for (int c = 0; c < (OUT == GATED ? 2 : 4); ++c)
        if (n + 16 * c < N) {
          const float a = acc[c][t][r];
          if constexpr (OUT == F32)
            ((float*)p.y)[o + 16 * c] = a;
          else
            ((short*)p.y)[o + 16 * c] = f32_to_bf16(
                OUT == GATED ? activate(p.act, a) * acc[OUT == GATED ? c + 2 : c][t][r] : a);
        }
    }
}

// From 193 rows on, K in parts of 1024 and more, multiples of 128: 128 rows of w by
// all of x in four waves, by the loop of tile_core.h. The matrix cores are 75 %
// busy, but they and the stream of weights together take the clock down to 1.25 to
// 1.9 GHz: 4096 -> [2 x 14336], 256 rows 69 us (78 above; library 65 to 69 and 6
// for the activation), 14336 -> 4096 37 (41), 4096 -> 12576 37 (42), of 5120 ->
// 10240 38 (42). Shorter parts end sooner in eight waves (4096 -> 4096, 512 each:
// 18 us for 20), as do 192 rows and fewer (a stack of 178: 795 us a pass for 814).
template <int OUT>
__global__ __launch_bounds__(256, 1) void linear_wide_kernel(const Tiles p) {
  extern __shared__ __align__(16) short wide_lds[];
  constexpr int LW = Wide::LW, LP = Wide::LP, QC = Wide::QC;
  Wide core;
  const int part = blockIdx.x % p.parts, blk = blockIdx.x / p.parts;
  const int k_lo = part * p.k_part, M = p.M, N = p.N;
  const int steps = (min(p.K, k_lo + p.k_part) - k_lo) / KS;
  const int first = start<OUT>(blk, N, steps);
  uint32_t wsrc[2][LW], xsrc[2][LP];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
#pragma unroll
    for (int j = 0; j < LW; ++j) {
      const int r = core.loaded<LW>(j);
      const int n = OUT == GATED ? h * N + min(blk * Wide::CH + r, N - 1)
                                 : min(blk * BN + h * Wide::CH + r, N - 1);
      wsrc[h][j] = (uint32_t)(n * p.w_row + core.piece<LW>(j)) * 2;
    }
#pragma unroll
    for (int j = 0; j < LP; ++j)
      xsrc[h][j] =
          (uint32_t)(min(h * Wide::RH + core.loaded<LP>(j), M - 1) *
                         p.x_row + core.piece<LP>(j)) * 2;
  }
  core.run(wide_lds, p.w, p.w_bytes, wsrc, p.x, p.x_bytes, xsrc, steps,
           [&](int s) {
             s += first;
             return (k_lo + (s >= steps ? s - steps : s) * KS) * 2;
           });
#pragma unroll
  for (int t = 0; t < Wide::ROWS / 32; ++t) {
    const int m = core.row(t) + core.col;
    if (m >= M) continue;
    const int64_t o = ((int64_t)part * M + m) * N;
#pragma unroll
    for (int c = 0; c < (OUT == GATED ? QC : 2 * QC); ++c) {
      const int n =
          blk * (OUT == GATED ? Wide::CH : BN) + core.channel(c) + core.grp * 4;
      if (n >= N) continue;           // N is a multiple of 4
      float4v v = core.acc[c][t];
      if constexpr (OUT == F32) {
        *(float4v*)((float*)p.y + o + n) = v;
      } else {
#pragma unroll
        for (int x = 0; x < 4; ++x)
          v[x] = activate(p.act, v[x]) * core.acc[c + QC][t][x];
        *(bf16x4*)((short*)p.y + o + n) = __builtin_convertvector(v, bf16x4);
      }
    }
  }
}

template <int OUT>
hipError_t go_wide(const Tiles& p, hipStream_t stream) {
  constexpr int width = OUT == GATED ? BN / 2 : BN;
  auto fn = linear_wide_kernel<OUT>;
  const hipError_t e = hipFuncSetAttribute(
      (const void*)fn, hipFuncAttributeMaxDynamicSharedMemorySize,
      Wide::LDS);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(fn, dim3((p.N + width - 1) / width * p.parts), dim3(256),
                     Wide::LDS, stream, p);
  HIP_CHECK_LAST();
  return hipSuccess;
}

template <int MT, int OUT>
hipError_t go(const Tiles& p, hipStream_t stream) {
  constexpr int width = OUT == GATED ? BN / 2 : BN;
  constexpr int bytes = ring(MT) * stage_bytes(MT);
  auto fn = linear_tiles_kernel<MT, OUT>;
  const hipError_t e = hipFuncSetAttribute(
      (const void*)fn, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(fn, dim3((p.N + width - 1) / width * p.parts),
                     dim3(NW * WAVE), bytes, stream, p);
  HIP_CHECK_LAST();
  return hipSuccess;
}

template <int OUT>
hipError_t go_rows(Tiles p, hipStream_t stream) {
  const int64_t xb = ((p.M - 1) * p.x_row + p.K) * 2;
  const int64_t wb =
      (((OUT == GATED ? 2 : 1) * (int64_t)p.N - 1) * p.w_row + p.K) * 2;
  // (products of one part that are not gated go to the library)
  if (OUT != BF16 && p.M > 192 && p.k_part >= 1024 && p.K % (2 * KS) == 0 &&
      xb < 1ll << 32 && wb < 1ll << 32) {
    p.x_bytes = (uint32_t)xb;
    p.w_bytes = (uint32_t)wb;
    if constexpr (OUT != BF16) return go_wide<OUT>(p, stream);
  }
  if (OUT == F32 && p.M <= 64) return go<OUT == F32 ? 1 : 2, OUT>(p, stream);
  if (p.M <= 128) return go<2, OUT>(p, stream);
  if (p.M <= 192) return go<3, OUT>(p, stream);
  if constexpr (OUT == GATED) return hipErrorInvalidValue;
  else return go<4, OUT>(p, stream);
}

}  // namespace

// x [M, K], w [N, K], rows x_row and w_row apart and 16-byte aligned, up
// to 256 rows; y [M, N] bf16, or (f32) [parts, M, N]
// 32-bit. act >= 0: y [M, N] = act(x gate') * (x up'), w [2 N, K]; of more than 192
// rows for K in whole steps of 128 from 1024 on and operands of less than 4 GiB.
extern "C" hipError_t lds_linear_tiles(const void* x, int64_t x_row,
                                       const void* w, int64_t w_row, void* y,
                                       int parts, int M, int N, int K, int f32,
                                       int act, hipStream_t stream) {
  if (M < 1 || M > 256 || N < 1 || K < 8 || K % 8 || x_row % 8 ||
      w_row % 8 || parts < 1 || (parts > 1 && !f32) || act >= ACTS ||
      (act >= 0 && f32))
    return hipErrorInvalidValue;
  Tiles p{(const short*)x, (const short*)w, x_row, w_row, y, M, N, K, K};
  p.k_part = ((K + parts - 1) / parts + 2 * KS - 1) / (2 * KS) * (2 * KS);
  p.parts = (K + p.k_part - 1) / p.k_part;
  p.act = act;
  if (p.parts != parts) return hipErrorInvalidValue;
  if (act >= 0) return go_rows<GATED>(p, stream);
  return f32 ? go_rows<F32>(p, stream) : go_rows<BF16>(p, stream);
}
