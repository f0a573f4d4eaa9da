// tile_core.h — the inner loop of products of many rows: 256 channels of the
// weights by up to 256 rows, bf16 operands, 32-bit sums, one workgroup of four
// waves per tile and compute unit.
//
// What bounds it is power: with the matrix cores 90 % busy the clock falls to
// 1.55 to 1.7 GHz of 2.4, so what counts is energy per multiply as much as idle
// cycles. Hence
//  * 16x16x32 instructions: without any loads they run 2130 TFLOP/s at the power
//    limit where 32x32x16 run 1860 (twice the traffic of sums per multiply);
//  * 128 x 128 results per wave, the largest that the registers hold, for the
//    fewest LDS reads (half of what 128 x 64 take).
// The loop holds nothing but matrix instructions, LDS reads, loads to LDS and
// one barrier per half step, all in a fixed order: slots are known at compile
// time (two steps make up the ring), so every address is a register plus a
// constant. 8192 rows, 4096 -> 8192: 2260 cycles per step of 64 where the matrix
// instructions take 2048; address arithmetic in the loop 2440, instructions in
// the compiler's order (reads and loads in bursts) 2800.
//
// A step of 64 of K is four halves: 128 channels, 128 rows, the other rows, the
// other channels, and four phases, one per quarter of the products. Phase i
// multiplies with operands that are in registers, reads the half after next from
// LDS into the registers of the half that was done with before, and loads the
// half that takes the slot of half i, two steps ahead. Steps take their halves
// of rows in turn first, so that each phase needs one new half only.
#pragma once
#include "hip_common.h"

#include <type_traits>

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) __bf16 bf16x4;

// fourth word of a buffer: raw bytes
constexpr int BUFFER_BYTES = 0x00027000;

constexpr int TILE_C = 256;             // channels of a tile
constexpr int TILE_K = 64;              // K of a step
constexpr int TILE_SLOTS = 8;           // halves in LDS: two steps
constexpr int TILE_SLOT = 128 * TILE_K;
// results that a wave turns round at a time: 32 rows x 128 channels
constexpr int TILE_TURN = 32 * 128;
constexpr int TILE_LDS =
    (TILE_SLOTS * TILE_SLOT + 4 * TILE_TURN) * (int)sizeof(short);

// CT x PT results of 16 x 16 per wave, WC waves across the channels, the others
// across the rows: 8, 8, 2 for 256 rows, 4, 8, 4 for 128.
template <int CT, int PT, int WC>
struct TileCore {
  static_assert(16 * CT * WC == TILE_C && WC <= 4, "");
  static constexpr int QC = CT / 2, QP = PT / 2;   // of a quarter
  static constexpr int WP = 4 / WC;
  static constexpr int ROWS = 16 * PT * WP;
  // 8 rows per load; loads of a wave and half
  static constexpr int LW = 4, LP = QP * WP / 2;
  static constexpr int G = 2 * CT;       // pieces of 8 channels of a wave's row

  float4v acc[CT][PT];
  int wave, lane, col, grp, wc, wp;

  __device__ __forceinline__ TileCore() {
    wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
    lane = threadIdx.x % WAVE;
    col = lane % 16;
    grp = lane / 16;
    wc = wave % WC;
    wp = wave / WC;
  }
  // the row of the tile that load j (0 .. 2 LP) of the rows, or j (0 .. 2 LW) of
  // the channels, brings in by this lane
  template <int L>
  __device__ __forceinline__ int loaded(int j) const {
    return (j / L * 4 * L + wave * L + j % L) * 8 + lane / 8;
  }
  // A row of a step is 8 pieces of 8 values. Piece c of row r lies at place
  // c ^ (r / 2 % 8): the 16 rows that a read serves at once meet all 64 banks.
  __device__ __forceinline__ uint32_t piece(int j) const {
    return (lane % 8 ^ (lane / 16 + j % 2 * 4)) * 8;
  }
  // row of the wave -> row of the tile; piece of the wave -> channel of the tile
  __device__ __forceinline__ int row_of(int r) const {
    return r / (16 * QP) * (16 * QP * WP) + wp * 16 * QP + r % (16 * QP);
  }
  __device__ __forceinline__ int channel_of(int g) const {
    return g / (2 * QC) * 128 + wc * 16 * QC + g % (2 * QC) * 8;
  }
  // where the wave's results turn round: piece g of row r (of 32)
  __device__ __forceinline__ int turned(int r, int g) const {
    return (r * G + (g ^ (G == 16 ? r & 15 : r / 2 & 7))) * 8;
  }

  // acc = channels x rows. wres, ares: the operands' buffers; wsrc, asrc: byte
  // offsets of what each load brings in at the first step (row and piece), all
  // of whose rows hold 64 steps values; steps >= 2.
  __device__ __forceinline__ void run(short* lds, __amdgpu_buffer_rsrc_t wres,
                                      const uint32_t (&wsrc)[2 * LW],
                                      __amdgpu_buffer_rsrc_t ares,
                                      const uint32_t (&asrc)[2 * LP],
                                      int steps) {
    using std::integral_constant;
    typedef __attribute__((address_space(3))) unsigned int smem;
    short* const wdst = lds + wave * LW * 8 * TILE_K;
    short* const adst = lds + wave * LP * 8 * TILE_K;
    // load j of half i of a step of parity par, byte k of the rows
    auto load = [&](int k, int par, int i, int slot, int j) {
      if (i == 0 || i == 3)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(
            wres, (smem*)(wdst + slot * TILE_SLOT + j * 8 * TILE_K), 16,
            wsrc[i / 3 * LW + j], k, 0, 0);
      else
        __builtin_amdgcn_raw_ptr_buffer_load_lds(
            ares, (smem*)(adst + slot * TILE_SLOT + j * 8 * TILE_K), 16,
            asrc[(i == 1 ? par : 1 - par) * LP + j], k, 0, 0);
    };
#pragma unroll
    for (int n = 0; n < TILE_SLOTS; ++n)
#pragma unroll
      for (int j = 0; j < (n % 4 % 3 ? LP : LW); ++j)
        load(n / 4 * TILE_K * 2, n / 4, n % 4, n, j);

#pragma unroll
    for (int c = 0; c < CT; ++c)
#pragma unroll
      for (int t = 0; t < PT; ++t) acc[c][t] = (float4v){0.f, 0.f, 0.f, 0.f};
    bf16x8 wf[2][2][QC], af[2][2][QP];     // [half][32 of K][16 rows]
    // pieces 4 kk + grp; slots beyond the fourth from addresses of their own (an
    // LDS read has 16 bits of offset)
    const short *wl[2][2], *al[2][2];
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      const int at = ((kk * 4 + grp) ^ (col / 2 & 7)) * 8;
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        wl[u][kk] = lds + u * 4 * TILE_SLOT + (wc * 16 * QC + col) * TILE_K + at;
        al[u][kk] = lds + u * 4 * TILE_SLOT + (wp * 16 * QP + col) * TILE_K + at;
      }
    }
    // read i of a half
    auto read_w = [&](int h, int slot, int i) {
      wf[h][i / QC][i % QC] = *(const bf16x8*)(
          wl[slot / 4][i / QC] + slot % 4 * TILE_SLOT + i % QC * 16 * TILE_K);
    };
    auto read_a = [&](int h, int slot, int i) {
      af[h][i / QP][i % QP] = *(const bf16x8*)(
          al[slot / 4][i / QP] + slot % 4 * TILE_SLOT + i % QP * 16 * TILE_K);
    };
    // the first two halves into registers
    asm volatile("s_waitcnt vmcnt(%0)" ::"i"(3 * LW + 3 * LP) : "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
#pragma unroll
    for (int i = 0; i < 2 * QC; ++i) read_w(0, 0, i);
#pragma unroll
    for (int i = 0; i < 2 * QP; ++i) read_a(0, 1, i);

    auto phase = [&](auto par_, auto i_, int k) {
      constexpr int par = decltype(par_)::value, i = decltype(i_)::value;
      constexpr int r = i + 2, rs = (par * 4 + r) % TILE_SLOTS;    // read
      constexpr int reads = r == 3 || r == 4 ? 2 * QC : 2 * QP;
      constexpr int loads = i % 3 ? LP : LW;
      constexpr int hw = i / 2, ha = i % 3 ? 1 - par : par;
      constexpr int n = 2 * QC * QP;                   // matrix instructions
      // The barrier of phases 0 and 2 lets this and the next one read and load:
      // every wave has what the loads of halves i + 2 and i + 3 brought in (up
      // to i + 7 are on their way), and has read halves i and i + 1. It comes
      // after 8 instructions, which wait for the last reads piece by piece.
      constexpr int at = i % 2 ? 0 : 8;
      constexpr int every = (n - at) / reads < 4 ? (n - at) / reads : 4;
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int m = 0; m < n; ++m) {
        if (i % 2 == 0 && m == at) {
          asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"i"(2 * LW + 2 * LP)
                       : "memory");
          __builtin_amdgcn_s_barrier();
          asm volatile("" ::: "memory");
          __builtin_amdgcn_sched_barrier(0);
        }
        const int kk = m / (QC * QP), c = m / QP % QC, t = m % QP;
        // In asm because sums and products are one register there: the compiler
        // takes others and copies all 256 back in every pass. It does not see
        // that these are matrix instructions, so the waits that it would put
        // ahead of sums just set and behind sums to be read are written out.
        float4v& d = acc[hw * QC + c][ha * QP + t];
        const bf16x8 w = wf[hw][kk][c], a = af[ha][kk][t];
        if (i == 0 && m == 0)
          asm volatile("s_nop 4\n\tv_mfma_f32_16x16x32_bf16 %0, %1, %2, %0"
                       : "+a"(d) : "v"(w), "v"(a));
        else if (i == 3 && m == n - 1)
          asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0\n\t"
                       "s_nop 7\n\ts_nop 7"
                       : "+a"(d) : "v"(w), "v"(a));
        else
          asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0"
                       : "+a"(d) : "v"(w), "v"(a));
        const int x = m - at;
        if (x >= 0 && x % every == 0 && x / every < reads) {
          if (r == 3 || r == 4) read_w(r % 2, rs, x / every);
          else read_a(1 - par, rs, x / every);
        }
        constexpr int apart = (n - at) / loads;
        if (x >= 0 && x % apart == apart - 1 && x / apart < loads)
          load(k, par, i, par * 4 + i, x / apart);
        __builtin_amdgcn_sched_barrier(0);
      }
    };
    // what is loaded: the step after next; past the end the last one once more
    const int last = (steps - 1) * TILE_K * 2;
    int k = 2 * TILE_K * 2;
    auto step = [&](auto par) {
      const int kc = min(k, last);
      phase(par, integral_constant<int, 0>{}, kc);
      phase(par, integral_constant<int, 1>{}, kc);
      phase(par, integral_constant<int, 2>{}, kc);
      phase(par, integral_constant<int, 3>{}, kc);
      k += TILE_K * 2;
    };
    for (int s = 0; s + 1 < steps; s += 2) {
      step(integral_constant<int, 0>{});
      step(integral_constant<int, 1>{});
    }
    if (steps % 2) step(integral_constant<int, 0>{});
  }

  // The results of rows [32 b, 32 b + 32) of the wave as bf16, after f(sum, t)
  // for those of row 16 t + col. The wave's share of LDS behind the ring turns
  // them round so that they leave in whole lines: store(row of the 32, row of the
  // tile, channel of the tile, 8 values).
  template <typename F, typename S>
  __device__ __forceinline__ void turn(short* lds, int b, F f, S store) const {
    short* mine = lds + TILE_SLOTS * TILE_SLOT + wave * TILE_TURN;
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int c = 0; c < CT; ++c) {
        float4v v;
#pragma unroll
        for (int x = 0; x < 4; ++x) v[x] = f(acc[c][2 * b + t][x], 2 * b + t);
        *(bf16x4*)(mine + turned(t * 16 + col, c * 2 + grp / 2) + grp % 2 * 4) =
            __builtin_convertvector(v, bf16x4);
      }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
    for (int j = 0; j < 32; j += WAVE / G) {
      const int row = j + lane / G;
      store(row, row_of(32 * b + row), channel_of(lane % G),
            *(const short8*)(mine + turned(row, lane % G)));
    }
    asm volatile("" ::: "memory");
  }
};
