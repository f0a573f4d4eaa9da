// tile_core.h — the inner loop of products whose operands go through LDS: a tile
// of up to 256 channels of the weights by up to 256 rows, bf16 operands, 32-bit
// sums, one workgroup of four waves per tile and compute unit.
//
// With 256 x 256 tiles it is bound by power: with the matrix cores 90 % busy the
// clock falls to 1.55 to 1.7 GHz of 2.4, so what counts is energy per multiply as
// much as idle cycles. Hence
//  * 16x16x32 instructions: without any loads they run 2130 TFLOP/s at the power
//    limit where 32x32x16 run 1860 (twice the traffic of sums per multiply);
//  * 128 x 128 results per wave, the largest that the registers hold, for the
//    fewest LDS reads (half of what 128 x 64 take).
// The loop holds nothing but matrix instructions, LDS reads, loads to LDS and
// one barrier per half step, all in a fixed order: with a ring of two steps the
// slots are known at compile time, so every address is a register plus a
// constant. 8192 rows, 4096 -> 8192: 2260 cycles per step of 64 where the matrix
// instructions take 2048; address arithmetic in the loop 2440, instructions in
// the compiler's order (reads and loads in bursts) 2800.
//
// A step of 64 of K is four halves: half of the channels, half of the rows, the
// other rows, the other channels, and four phases, one per quarter of the
// products. Phase i multiplies with operands that are in registers, reads the
// half after next from LDS into the registers of the half that was done with
// before, and loads the half that takes the place of half i, a ring ahead. Steps
// take their halves of rows in turn first, so that each phase needs one new half
// only.
#pragma once
#include "hip_common.h"

#include <type_traits>

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) __bf16 bf16x4;

// fourth word of a buffer: raw bytes
constexpr int BUFFER_BYTES = 0x00027000;

constexpr int TILE_K = 64;              // K of a step

// CT x PT results of 16 x 16 per wave, WC waves across the channels, the others
// across the rows.
template <int CT, int PT, int WC>
struct TileCore {
  static constexpr int QC = CT / 2, QP = PT / 2;   // of a quarter
  static constexpr int WP = 4 / WC;
  static constexpr int CHANNELS = 16 * CT * WC, ROWS = 16 * PT * WP;
  static constexpr int CH = CHANNELS / 2, RH = ROWS / 2;   // of a half
  // 8 rows per load; loads of a wave and half
  static constexpr int LW = CH / 32, LP = RH / 32;
  static_assert(CH % 32 == 0 && RH % 32 == 0, "");
  static constexpr int STEP = (CHANNELS + ROWS) * TILE_K;
  static constexpr int RING = 2 * STEP;
  // results that a wave turns round at a time: 32 rows
  static constexpr int TURN = 32 * 16 * CT;
  static constexpr int LDS = RING * (int)sizeof(short);
  static constexpr int LDS_TURN = (RING + 4 * TURN) * (int)sizeof(short);

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
  // the row within its half that load j of a wave brings in by this lane
  template <int L>
  __device__ __forceinline__ int loaded(int j) const {
    return (wave * L + j) * 8 + lane / 8;
  }
  // A row of a step is 8 pieces of 8 values. Piece c of row r lies at place
  // c ^ (r / 2 % 8): the 16 rows that a read serves at once meet all 64 banks.
  template <int L>
  __device__ __forceinline__ uint32_t piece(int j) const {
    return (lane % 8 ^ loaded<L>(j) / 2 % 8) * 8;
  }
  // results acc[c][t]: channels from channel(c) + 4 grp on, row row(t) + col
  __device__ __forceinline__ int channel(int c) const {
    return c / QC * CH + (wc * QC + c % QC) * 16;
  }
  __device__ __forceinline__ int row(int t) const {
    return t / QP * RH + (wp * QP + t % QP) * 16;
  }

  // acc = channels x rows. wptr, aptr: the operands, wbytes and abytes long;
  // wsrc[h][j], asrc[h][j]: byte offsets of what load j of half h brings in (row
  // and piece), to which at(s) is added for step s.
  template <typename At>
  __device__ __forceinline__ void run(short* lds, const void* wptr,
                                      uint32_t wbytes,
                                      const uint32_t (&wsrc)[2][LW],
                                      const void* aptr, uint32_t abytes,
                                      const uint32_t (&asrc)[2][LP], int steps,
                                      At at) {
    using std::integral_constant;
    typedef __attribute__((address_space(3))) unsigned int smem;
    short* const wdst = lds + wave * LW * 8 * TILE_K;
    short* const adst = lds + wave * LP * 8 * TILE_K;
    // where half i lies in a step
    constexpr int place[4] = {0, CH * TILE_K, (CH + RH) * TILE_K,
                              (CH + 2 * RH) * TILE_K};
    struct Source {
      __amdgpu_buffer_rsrc_t w, a;
      int k;
    };
    // past the end the operands are empty: their loads fetch nothing
    auto source = [&](int s) {
      const bool in = s < steps;
      const int wb = __builtin_amdgcn_readfirstlane(in ? wbytes : 0);
      const int ab = __builtin_amdgcn_readfirstlane(in ? abytes : 0);
      return Source{__builtin_amdgcn_make_buffer_rsrc((void*)wptr, 0, wb,
                                                      BUFFER_BYTES),
                    __builtin_amdgcn_make_buffer_rsrc((void*)aptr, 0, ab,
                                                      BUFFER_BYTES),
                    __builtin_amdgcn_readfirstlane(in ? at(s) : 0)};
    };
    // load j of half i of a step of parity par
    auto load = [&](const Source& s, int par, int i, int j) {
      const int base = par * STEP;
      if (i % 3 == 0)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(
            s.w, (smem*)(wdst + base + place[i] + j * 8 * TILE_K), 16,
            wsrc[i / 3][j], s.k, 0, 0);
      else
        __builtin_amdgcn_raw_ptr_buffer_load_lds(
            s.a, (smem*)(adst + base + place[i] + j * 8 * TILE_K), 16,
            asrc[i == 1 ? par : 1 - par][j], s.k, 0, 0);
    };
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      const Source from = source(s);
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < (i % 3 ? LP : LW); ++j)
          load(from, s, i, j);
    }

#pragma unroll
    for (int c = 0; c < CT; ++c)
#pragma unroll
      for (int t = 0; t < PT; ++t) acc[c][t] = (float4v){0.f, 0.f, 0.f, 0.f};
    bf16x8 wf[2][2][QC], af[2][2][QP];     // [half][32 of K][16 rows]
    // pieces 4 kk + grp; the second step of the ring from addresses of its own (an
    // LDS read has 16 bits of offset)
    const short *wl[2][2], *al[2][2];
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      const int p = ((kk * 4 + grp) ^ (col / 2 & 7)) * 8;
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        wl[u][kk] = lds + u * STEP + (wc * 16 * QC + col) * TILE_K + p;
        al[u][kk] = lds + u * STEP + (wp * 16 * QP + col) * TILE_K + p;
      }
    }
    // read x of half i of step u of the ring
    auto read_w = [&](int h, int u, int x) {
      wf[h][x / QC][x % QC] = *(const bf16x8*)(
          wl[u][x / QC] + place[h * 3] + x % QC * 16 * TILE_K);
    };
    auto read_a = [&](int h, int i, int u, int x) {
      af[h][x / QP][x % QP] = *(const bf16x8*)(
          al[u][x / QP] + place[i] + x % QP * 16 * TILE_K);
    };
    // the first two halves into registers
    asm volatile("s_waitcnt vmcnt(%0)" ::"i"(3 * (LW + LP))
                 : "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
#pragma unroll
    for (int x = 0; x < 2 * QC; ++x) read_w(0, 0, x);
#pragma unroll
    for (int x = 0; x < 2 * QP; ++x) read_a(0, 1, 0, x);

    auto phase = [&](auto par_, auto i_, const Source& from) {
      constexpr int par = decltype(par_)::value, i = decltype(i_)::value;
      constexpr int hw = i / 2, ha = i % 3 ? 1 - par : par;
      constexpr int n = 2 * QC * QP;                   // matrix instructions
      constexpr bool channels = i == 1 || i == 2;      // what is read
      constexpr int reads = channels ? 2 * QC : 2 * QP;
      constexpr int loads = i % 3 ? LP : LW;
      // The barrier of phases 0 and 2 lets this and the next one read and load:
      // every wave has what the loads of halves i + 2 and i + 3 brought in (those
      // after them are on their way), and has read halves i and i + 1. It
      // comes after some instructions, which wait for the last reads piece by
      // piece.
      constexpr int ahead = i % 2 ? 0 : n / 4;
      constexpr int every = (n - ahead) / reads < 4 ? (n - ahead) / reads : 4;
      constexpr int apart = (n - ahead) / loads;
      static_assert(every > 0 && apart > 0, "");
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int m = 0; m < n; ++m) {
        if (i % 2 == 0 && m == ahead) {
          asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"i"(
                           2 * (LW + LP))
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
        const int x = m - ahead;
        if (x >= 0 && x % every == 0 && x / every < reads) {
          if (i == 0) read_a(1 - par, 2, par, x / every);
          if (i == 1) read_w(1, par, x / every);
          if (i == 2) read_w(0, 1 - par, x / every);
          if (i == 3) read_a(1 - par, 1, 1 - par, x / every);
        }
        if (x >= 0 && x % apart == apart - 1 && x / apart < loads)
          load(from, par, i, x / apart);
        __builtin_amdgcn_sched_barrier(0);
      }
    };
    int s = 0;
    auto step = [&](auto par) {
      const Source from = source(s + 2);
      phase(par, integral_constant<int, 0>{}, from);
      phase(par, integral_constant<int, 1>{}, from);
      phase(par, integral_constant<int, 2>{}, from);
      phase(par, integral_constant<int, 3>{}, from);
      ++s;
    };
    while (s + 1 < steps) {
      step(integral_constant<int, 0>{});
      step(integral_constant<int, 1>{});
    }
    if (s < steps) step(integral_constant<int, 0>{});
  }

  // Results of 16 rows from row(2 b), 16 from row(2 b + 1) and the first NC tiles of
  // channels, f(c, t, x) for what acc[c][t][x] stands for, as bf16. The wave's share
  // of LDS behind the ring turns them round so that they leave in whole lines:
  // store(row of the 32, row of the tile, channel of the tile, 8 values).
  template <int NC, typename F, typename S>
  __device__ __forceinline__ void turn(short* lds, int b, F f, S store) const {
    static_assert(PT % 2 == 0 && NC <= CT, "");
    constexpr int G = 2 * NC;            // pieces of 8 channels in a row
    static_assert(G == 16 || G == 8 || G == 4, "");
    short* mine = lds + RING + wave * TURN;
    auto place = [](int r, int g) {
      return (r * G + (g ^ (G == 16 ? r & 15 : G == 8 ? r / 2 & 7 : r / 4 & 3))) *
             8;
    };
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        float4v v;
#pragma unroll
        for (int x = 0; x < 4; ++x) v[x] = f(c, 2 * b + t, x);
        *(bf16x4*)(mine + place(t * 16 + col, c * 2 + grp / 2) + grp % 2 * 4) =
            __builtin_convertvector(v, bf16x4);
      }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    const int g = lane % G;
#pragma unroll
    for (int j = 0; j < 32; j += WAVE / G) {
      const int r = j + lane / G;
      store(r, (j < 16 ? row(2 * b) : row(2 * b + 1) - 16) + r,
            channel(g / 2) + g % 2 * 8,
            *(const short8*)(mine + place(r, g)));
    }
    asm volatile("" ::: "memory");
  }
};
