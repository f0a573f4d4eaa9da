// linear_tiles.hip — y = x w' for 65 to 256 rows of x, from 33 where K is split (bf16,
// 32-bit sums).
//
// The weights should be read from memory once, at its rate, so one workgroup has all
// rows of x (groups of 64, up to four) against 128 rows of w, and K is split until the
// workgroups make up a round of the 256 compute units. Both operands go to LDS by direct
// loads, those of w past the L2 caches (rows_core.h; 178 rows, 4096 -> [2 x 14336] 56 us
// by way of them, so 53; 5120 -> [2 x 25600] 138, 129). 8 waves of 64 channels by 16 rows
// of each group. Parts of K run fastest over the grid: with 8 of them each XCD's L2 holds
// one part of x. Workgroups start at different steps, as in linear_rows.hip.
//
// Two kernels, which add up in one order:
//   lines   256 bytes of a row by one load, as in rows_core.h; K in whole steps of 128.
//   short   64 of K at a time: 128 bytes of a row, but the first products and the last
//           ones are that much sooner, which counts where a part has few steps.
// Measured, cold weights, without the sum of the parts, lines / short (short before,
// weights by way of the L2 caches and other stores; library):
//   4096 -> [2 x 14336]   65 rows 44.5 / 48.6 us (51; 58), 128 46.2 / 50.4 (53; 60),
//                         192 51.9 / 59.4 (61; 73), 256 66.9 / 70.0 (72; 80)
//   5120 -> [2 x 25600]   180 rows 128.7 / 153.1 (160)
//   4096 -> 32768         128 rows 47.9 (59; 64), 192 52.9 (68), 256 63.7 (71)
//   14336 -> 4096, 8 parts of 1792     100 rows 24.6 / 24.4 (26.5), 178 27.5 / 29.6
//                         (31.2), 256 35.8 / 36.5 (37.5)
//   8192 -> 5120, 6 parts of 1408      100 rows 20.8 / 19.4 (20.7), 178 21.6 / 23.5
//                         (24.7), 256 27.9 / 30.9 (31.1)
//   4096 -> 6144, 5 parts of 896       100 rows 14.9 / 13.6 (14.9), 178 16.6 / 16.4
//                         (18.0), 256 21.9 / 21.6 (23.1)
//   4096 -> 4096, 8 parts of 512       50 rows 9.0 / 8.2 (9.3), 100 12.2 / 10.4 (11.6),
//                         178 13.4 / 13.0 (14.0), 256 19.1 / 17.2 (17.6)
// The loads bound it: with nothing but loads 4096 -> [2 x 14336] takes 44 us by lines
// at 128 rows and 49 at 178, of which w 40; parts of few steps, what they write besides
// (without stores 256 rows, 4096 -> 4096 12 us).
#include "rows_core.h"
#include "tile_core.h"

namespace {

struct Tiles {
  const short *x, *w;        // [M, K], [N, K] (GATED: [2 N, K], gate first)
  int64_t x_row, w_row;      // strides in elements
  void* y;                   // [M, N]; F32: [parts, M, N] 32-bit
  int M, N, K, k_part;       // k_part: K per part, a multiple of KS
  int parts, act;
  uint32_t x_bytes, w_bytes; // lines
};

enum Out { BF16, F32, GATED };

constexpr int NW = 8, KS = 128, BN = 128;      // BN: rows of w per workgroup
constexpr int ROW = KS * 2;                    // bytes of a row in LDS: lines
constexpr int HALF = TILE_K * 2;               // short
constexpr int LDS_BYTES = 160 * 1024;          // lines

// The order of linear_rows.hip: steps of 128, starting at one by the channels.
template <int OUT>
__device__ __forceinline__ int start(int blk, int N, int steps) {
  return (OUT == GATED    ? blk * 6
          : N > 128 * 256 ? blk / 2 * 3
                          : blk * 3) %
         steps;
}

// Results of the four waves by two leave by whole lines: turned round in LDS, where the
// 16-byte pieces of a row change places by XOR with its number. Past the caches: as other
// stores they take their time at the end of the kernel, when all of the parts are
// written back at once (4096 -> 6144, 178 rows 19.3 us, so 16.5; by whole lines only 17.9).
// Up to 64 rows they are few, and whoever sums them finds them in the caches (a pass of
// the delta design, 50 rows, 1372 us past them, 1356 so).
template <int MT, int OUT>
__device__ __forceinline__ void store(const Tiles& p, char* lds, int part, int blk,
                                      const float4v (&acc)[4][MT]) {
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
  const int lane = threadIdx.x % WAVE, col = lane % 16, grp = lane / 16;
  const int wc = wave % 2, wm = wave / 2, M = p.M, N = p.N;
  typedef std::conditional_t<OUT == F32, float, short> Elem;
  constexpr int CH = OUT == GATED ? BN / 2 : BN;       // channels of the workgroup
  constexpr int PIECES = CH * (int)sizeof(Elem) / 16, EACH = 16 / sizeof(Elem);
  __builtin_amdgcn_s_barrier();                        // the rings are no longer read
  asm volatile("" ::: "memory");
  // lane: row `col` of a tile, channels 4 grp ..
#pragma unroll
  for (int t = 0; t < MT; ++t) {
    const int m = t * 64 + wm * 16 + col;
#pragma unroll
    for (int c = 0; c < (OUT == GATED ? 2 : 4); ++c) {
      const int n = wc * (CH / 2) + c * 16 + grp * 4;
      char* to = lds + (m * PIECES + (n / EACH ^ m % PIECES)) * 16;
      float4v v = acc[c][t];
      if constexpr (OUT == F32) {
        *(float4v*)to = v;
      } else {
        if constexpr (OUT == GATED)
#pragma unroll
          for (int r = 0; r < 4; ++r) v[r] = activate(p.act, v[r]) * acc[c + 2][t][r];
        *(bf16x4*)(to + n % EACH * 2) = __builtin_convertvector(v, bf16x4);
      }
    }
  }
  __syncthreads();
  constexpr int ROWS = NW * WAVE / PIECES;             // of a store
  const int piece = threadIdx.x % PIECES, n = blk * CH + piece * EACH;
  if (n >= N) return;                                  // N is a multiple of 8
#pragma unroll
  for (int i = 0; i < 64 * MT; i += ROWS) {
    const int m = i + threadIdx.x / PIECES;
    if (m >= M) continue;
    const float4v v = *(const float4v*)(lds + (m * PIECES + (piece ^ m % PIECES)) * 16);
    float4v* const to = (float4v*)((Elem*)p.y + ((int64_t)part * M + m) * N + n);
    if (MT == 1)
      *to = v;
    else
      __builtin_nontemporal_store(v, to);
  }
}

// ---- short

// Operands of the next half of a step are read while the matrix cores work on this one,
// and the one barrier per step stands between the halves.

// steps in the ring of 64 MT rows, and their LDS
constexpr int ring(int MT) { return MT <= 2 ? 4 : 3; }
constexpr int stage_bytes(int MT) { return (BN + 64 * MT) * HALF; }
// (results are turned round in them)
static_assert(ring(1) * stage_bytes(1) >= 64 * BN * 4 &&
              ring(4) * stage_bytes(4) >= 256 * BN * 4, "");

template <int MT, int OUT>
__global__ __launch_bounds__(NW * WAVE, 2) void linear_short_kernel(
    const Tiles p) {
  extern __shared__ __align__(16) char lds[];
  constexpr int R = ring(MT), STAGE = stage_bytes(MT);
  constexpr int WL = 2, XL = MT;                       // loads of a wave
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
  const int lane = threadIdx.x % WAVE, col = lane % 16, grp = lane / 16;
  const int part = blockIdx.x % p.parts, blk = blockIdx.x / p.parts;
  const int k_lo = part * p.k_part, k_hi = min(p.K, k_lo + p.k_part);
  const int steps = (k_hi - k_lo + KS - 1) / KS * 2;
  const int first = start<OUT>(blk, p.N, steps / 2) * 2;
  const int M = p.M, N = p.N;

  // A load takes 8 rows of TILE_K, 8 pieces of 16 bytes each; the pieces of a row
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
    k = k_lo + (k >= steps ? k - steps : k) * TILE_K;
    char* b = lds + buf * STAGE;
    typedef const __attribute__((address_space(1))) unsigned int gmem;
    typedef __attribute__((address_space(3))) unsigned int smem;
#pragma unroll
    for (int j = 0; j < WL + XL; ++j) {
      const int r = j < WL ? wave * WL + j : BN / 8 + wave * XL + j - WL;
      const bool in = k + (lane % 8 ^ ((r * 8 + r8) / 2 % 8)) * 8 < k_hi;
      gmem* const at = (gmem*)(in ? from[j] + k : (const short*)&rows_core::zeros);
      smem* const to = (smem*)(b + r * 1024);
      if (j < WL)
        __builtin_amdgcn_global_load_lds(at, to, 16, 0, rows_core::ONCE);
      else
        __builtin_amdgcn_global_load_lds(at, to, 16, 0, 0);
    }
  };

  // wave: 64 channels, 16 rows of every group of 64
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
  const int w_at = (wc * 64 + col) * HALF;
  const int x_at = (BN + wm * 16 + col) * HALF;
  const int piece0 = (grp ^ col / 2) * 16, piece1 = ((4 + grp) ^ col / 2) * 16;
  auto read = [&](Operands& o, int buf, int piece) {
    const char* b = lds + buf * STAGE + piece;
#pragma unroll
    for (int c = 0; c < 4; ++c)
      o.w[c] = *(const bf16x8*)(b + w_at + c * 16 * HALF);
#pragma unroll
    for (int t = 0; t < MT; ++t)
      o.x[t] = *(const bf16x8*)(b + x_at + t * 64 * HALF);
    __builtin_amdgcn_sched_barrier(0);    // all are under way before use
  };
  auto multiply = [&](const Operands& o) {
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
      for (int c = 0; c < 4; ++c)
        acc[c][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(o.w[c], o.x[t],
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

  store<MT, OUT>(p, lds, part, blk, acc);
}

// ---- lines

// Rings of 64 MT rows, in steps of w (32 KB) and groups of x (16 KB): all of the LDS.
constexpr int w_ring(int MT) { return MT <= 2 ? 3 : 2; }
constexpr int x_ring(int MT) { return MT <= 2 ? 4 : 6; }
constexpr int WL = 4, XL = 2;        // loads of a wave for one of them
constexpr int W_STEP = BN * ROW, X_GROUP = 64 * ROW;

// Loads under way at the start of phase t when what it waits for has landed: the group
// of x after this one and, in the last phase, the next step's w. Phase p loads group p +
// x_ring, then, if it is the second of its step, w of step p / MT + w_ring.
constexpr int under_way(int MT, int t) {
  const int step = 64, p = step * MT + t;        // any step
  const int x = p + 1 - x_ring(MT), w = (step + 1 - w_ring(MT)) * MT + 1;
  int n = 0, m = 0;
  for (int j = p - 16; j < p; ++j) {
    const int loads_w = j % MT == 1 ? WL : 0;
    if (j >= x) n += (j > x ? XL : 0) + loads_w;
    if (j > w) m += XL + loads_w;
  }
  return t == MT - 1 && m < n ? m : n;
}

// s_waitcnt's operand for numbers of loads and LDS reads under way
constexpr int waits(int vm, int lgkm) {
  return (vm & 15) | 7 << 4 | lgkm << 8 | (vm >> 4) << 14;
}

// 16 bytes per lane to LDS, from byte `at` + k of a buffer of `bytes`; past its end
// nothing is fetched
template <int HINT>
__device__ __forceinline__ void to_lds(const short* buffer, uint32_t bytes,
                                       uint32_t at, int k, char* lds) {
  typedef __attribute__((address_space(3))) unsigned int smem;
  __builtin_amdgcn_raw_ptr_buffer_load_lds(
      __builtin_amdgcn_make_buffer_rsrc((void*)buffer, 0,
                                        __builtin_amdgcn_readfirstlane(bytes),
                                        BUFFER_BYTES),
      (smem*)lds, 16, at, __builtin_amdgcn_readfirstlane(k), 0, HINT);
}

// A step is MT phases, each of which multiplies a group of 64 rows of x: w of a step is
// in registers, and so is a group of x one phase ahead. So the rings give way 16 KB of x
// at a time, and all of the LDS holds what is under way: two or three steps of w, four to
// six groups of x. (Without matrix instructions 178 rows, 4096 -> [2 x 14336] take 50 us
// of 54.5, 128 rows 47 of 48.5; w in the first phase of its step no sooner.)
template <int MT, int OUT>
__global__ __launch_bounds__(NW * WAVE, 2) void linear_lines_kernel(
    const Tiles p) {
  extern __shared__ __align__(16) char lds[];
  constexpr int WR = w_ring(MT), XR = x_ring(MT);
  static_assert(WR * W_STEP + XR * X_GROUP <= LDS_BYTES && XR <= WR * MT, "");
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
  const int lane = threadIdx.x % WAVE, col = lane % 16, grp = lane / 16;
  const int part = blockIdx.x % p.parts;
  const int blk = p.parts > 1 ? blockIdx.x / p.parts
                              : rows_core::along_xcd(blockIdx.x, gridDim.x, 256);
  if (blk * (OUT == GATED ? BN / 2 : BN) >= p.N) return;
  const int k_lo = part * p.k_part, k_hi = min(p.K, k_lo + p.k_part);
  const int steps = (k_hi - k_lo + KS - 1) / KS;
  const int first = start<OUT>(blk, p.N, steps);
  const int M = p.M, N = p.N;
  char* const w_lds = lds;
  char* const x_lds = lds + WR * W_STEP;

  // A load takes 4 rows of KS, 16 pieces of 16 bytes each; the pieces of a row change
  // places by XOR with its number, so that 16 lanes that read one piece of 16 rows find
  // all banks. Rows of w that do not exist repeat the last one, as do rows of x.
  uint32_t w_from[WL], x_from[MT][XL];            // byte offsets
#pragma unroll
  for (int j = 0; j < WL; ++j) {
    const int r = (wave * WL + j) * 4 + grp;      // row in LDS
    int n;
    if (OUT == GATED)       // of 64 rows 32 gate, 32 up
      n = min(blk * (BN / 2) + r / 64 * 32 + r % 32, N - 1) +
          (r % 64 >= 32 ? N : 0);
    else
      n = min(blk * BN + r, N - 1);
    w_from[j] = (uint32_t)(n * p.w_row + (col ^ r % 16) * 8) * 2;
  }
#pragma unroll
  for (int t = 0; t < MT; ++t)
#pragma unroll
    for (int j = 0; j < XL; ++j) {
      const int r = (wave * XL + j) * 4 + grp;
      x_from[t][j] =
          (uint32_t)(min(t * 64 + r, M - 1) * p.x_row + (col ^ r % 16) * 8) * 2;
    }
  auto k_of = [&](int s) {                        // bytes
    s += first;
    return (k_lo + (s >= steps ? s - steps : s) * KS) * 2;
  };
  // Loads j0 .. of step s, of its group t of x. Past the last step the operands are
  // empty.
  auto load_w = [&](int s, int j0, int n, int place) {
#pragma unroll
    for (int j = j0; j < j0 + n; ++j)
      to_lds<rows_core::ONCE>(p.w, s < steps ? p.w_bytes : 0, w_from[j], s < steps ? k_of(s) : 0,
             w_lds + place * W_STEP + (wave * WL + j) * 1024);
  };
  auto load_x = [&](int s, int t, int place) {
#pragma unroll
    for (int j = 0; j < XL; ++j)
      to_lds<0>(p.x, s < steps ? p.x_bytes : 0, x_from[t][j], s < steps ? k_of(s) : 0,
             x_lds + place * X_GROUP + (wave * XL + j) * 1024);
  };
  // at the start of phase t
  auto landed = [&](auto t_) {
    constexpr int t = decltype(t_)::value;
    __builtin_amdgcn_s_waitcnt(waits(under_way(MT, t), t == 0 ? 4 : 0));
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  };

  // wave: 64 channels, 16 rows of every group of 64
  float4v acc[4][MT];
#pragma unroll
  for (int c = 0; c < 4; ++c)
#pragma unroll
    for (int t = 0; t < MT; ++t) acc[c][t] = (float4v){0.f, 0.f, 0.f, 0.f};
  const int wc = wave % 2, wm = wave / 2;
  bf16x8 wo[4][4], xo[2][4];       // operands of 32 of K each: a step's, a group's
  const char* const w_at = w_lds + (wc * 64 + col) * ROW;
  const char* const x_at = x_lds + (wm * 16 + col) * ROW;
  auto read_w = [&](int q, int place) {
    const char* b = w_at + place * W_STEP + ((q * 4 + grp) ^ col) * 16;
#pragma unroll
    for (int c = 0; c < 4; ++c) wo[q][c] = *(const bf16x8*)(b + c * 16 * ROW);
    __builtin_amdgcn_sched_barrier(0);
  };
  auto read_x = [&](int par, int place) {
    const char* b = x_at + place * X_GROUP;
#pragma unroll
    for (int q = 0; q < 4; ++q)
      xo[par][q] = *(const bf16x8*)(b + ((q * 4 + grp) ^ col) * 16);
    __builtin_amdgcn_sched_barrier(0);
  };
  int w_next = 0, x_next = 0, x_now = 0, w_now = 0;   // places to load, to read next
  auto after = [](int i, int n) { return i + 1 == n ? 0 : i + 1; };

  // Phase t of step s multiplies group t of x, in registers since the one before, and
  // reads the next; in the last one of a step the next step's w takes the registers of
  // this one's, 32 of K at a time. When its barrier is passed all waves have read this
  // group: the place takes the one x_ring groups on. (w's last reads may be under way
  // then, which only the barrier of the phase that loads w waits for.)
  auto phase = [&](auto t_, auto par_, int s) {
    constexpr int t = decltype(t_)::value, par = decltype(par_)::value;
    landed(t_);
    read_x(1 - par, x_now);
    x_now = after(x_now, XR);
    constexpr int xt = (t + XR) % MT, xs = (t + XR) / MT;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
#pragma unroll
      for (int c = 0; c < 4; ++c)
        acc[c][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wo[q][c], xo[par][q],
                                                            acc[c][t], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
      if (q == 0) {
        load_x(s + xs, xt, x_next);
        x_next = after(x_next, XR);
      }
      if (t == 1 && (q == 1 || q == 2)) {
        load_w(s + WR, 2 * q - 2, 2, w_next);
        if (q == 2) w_next = after(w_next, WR);
      }
      __builtin_amdgcn_sched_barrier(0);
      if (t == MT - 1) read_w(q, w_now);
    }
    if (t == MT - 1) w_now = after(w_now, WR);
  };
  // before the first step: the loads of the phases ahead of it in their order, and the
  // reads of the last of them
#pragma unroll
  for (int j = -WR * MT; j < 0; ++j) {
    if (j == -1) landed(std::integral_constant<int, MT - 1>{});
    if (j + XR >= 0) {
      load_x((j + XR) / MT, (j + XR) % MT, x_next);
      x_next = after(x_next, XR);
    }
    if ((j + WR * MT) % MT == 1) {
      load_w((j + WR * MT) / MT, 0, WL, w_next);
      w_next = after(w_next, WR);
    }
    __builtin_amdgcn_sched_barrier(0);
  }
  read_x(0, x_now);
  x_now = after(x_now, XR);
#pragma unroll
  for (int q = 0; q < 4; ++q) read_w(q, w_now);
  w_now = after(w_now, WR);

  auto step = [&](auto par_, int s) {
    constexpr int par = decltype(par_)::value;
    auto turn = [&](auto t_) {
      constexpr int t = decltype(t_)::value;
      if constexpr (t < MT)
        phase(t_, std::integral_constant<int, (par + t) % 2>{}, s);
    };
    turn(std::integral_constant<int, 0>{});
    turn(std::integral_constant<int, 1>{});
    turn(std::integral_constant<int, 2>{});
    turn(std::integral_constant<int, 3>{});
  };
  for (int s = 0; s < steps; ++s) {
    step(std::integral_constant<int, 0>{}, s);
    if constexpr (MT % 2)
      if (++s < steps) step(std::integral_constant<int, 1>{}, s);
  }
  // what was loaded past the end has landed
  __builtin_amdgcn_s_waitcnt(waits(0, 0));

  store<MT, OUT>(p, lds, part, blk, acc);
}

template <int MT, int OUT, bool LINES>
hipError_t go(const Tiles& p, hipStream_t stream) {
  constexpr int width = OUT == GATED ? BN / 2 : BN;
  constexpr int bytes = LINES ? LDS_BYTES : ring(MT) * stage_bytes(MT);
  void (*const fn)(Tiles) = [] {
    if constexpr (LINES) return linear_lines_kernel<MT, OUT>;
    else return linear_short_kernel<MT, OUT>;
  }();
  const hipError_t e = hipFuncSetAttribute(
      (const void*)fn, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
  if (e != hipSuccess) return e;
  int groups = (p.N + width - 1) / width * p.parts;
  if (LINES && p.parts == 1) groups = (groups + 7) / 8 * 8;   // equal shares of the XCDs
  hipLaunchKernelGGL(fn, dim3(groups), dim3(NW * WAVE), bytes, stream, p);
  HIP_CHECK_LAST();
  return hipSuccess;
}

template <int OUT>
hipError_t go_rows(Tiles p, hipStream_t stream) {
  const int64_t xb = ((p.M - 1) * p.x_row + p.K) * 2;
  const int64_t wb =
      (((OUT == GATED ? 2 : 1) * (int64_t)p.N - 1) * p.w_row + p.K) * 2;
  const bool whole = p.K % KS == 0 && xb < 1ll << 32 && wb < 1ll << 32;
  p.x_bytes = (uint32_t)xb;
  p.w_bytes = (uint32_t)wb;
  // by the sizes in the head of this file
  if (whole && p.M > 64 && p.k_part >= (OUT != F32 ? 1024 : p.M <= 128 ? 1792 : 1280))
    return p.M <= 128   ? go<2, OUT, true>(p, stream)
           : p.M <= 192 ? go<3, OUT, true>(p, stream)
                        : go<4, OUT, true>(p, stream);
  if constexpr (OUT == F32)
    if (p.M <= 64) return go<1, OUT, false>(p, stream);
  if (p.M <= 128) return go<2, OUT, false>(p, stream);
  if (p.M <= 192) return go<3, OUT, false>(p, stream);
  if constexpr (OUT == GATED) return hipErrorInvalidValue;
  else return go<4, OUT, false>(p, stream);
}

}  // namespace

// x [M, K], w [N, K], rows x_row and w_row apart and 16-byte aligned, up
// to 256 rows, N a multiple of 8; y [M, N] bf16, or (f32) [parts, M, N]
// 32-bit. act >= 0: y [M, N] = act(x gate') * (x up'), w [2 N, K]; of more than 192
// rows for K in whole steps of 128 from 1024 on and operands of less than 4 GiB.
extern "C" hipError_t lds_linear_tiles(const void* x, int64_t x_row,
                                       const void* w, int64_t w_row, void* y,
                                       int parts, int M, int N, int K, int f32,
                                       int act, hipStream_t stream) {
  if (M < 1 || M > 256 || N < 1 || N % 8 || K < 8 || K % 8 || x_row % 8 ||
      w_row % 8 || parts < 1 || (parts > 1 && !f32) || act >= ACTS ||
      (act >= 0 && f32))
    return hipErrorInvalidValue;
  Tiles p{(const short*)x, (const short*)w, x_row, w_row, y, M, N, K, K};
  p.k_part = ((K + parts - 1) / parts + KS - 1) / KS * KS;
  p.parts = (K + p.k_part - 1) / p.k_part;
  p.act = act;
  if (p.parts != parts) return hipErrorInvalidValue;
  if (act >= 0) return go_rows<GATED>(p, stream);
  return f32 ? go_rows<F32>(p, stream) : go_rows<BF16>(p, stream);
}
