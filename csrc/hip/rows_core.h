// rows_core.h — few rows of x against a block of rows of w (bf16, 32-bit sums), both by
// way of LDS: the loop of linear_rows.hip and of the experts' products of few pairs.
//
// The weights' bytes are what counts. Both operands go to LDS by direct loads, 128 of K
// at a time, into a ring of three steps: 64 KB of w per compute unit are under way. What
// the rate hangs on is the length of what is read of a row at a time: 256 bytes of each
// by one instruction come at 5.9 TB/s, pieces of 128 take 10 to 20 % longer (14336 ->
// 4096 read and nothing else: 21.3 us, 23.8; 25600 -> 5120: 45, 54). Workgroups start at
// different steps: in step they would hit the same few memory channels where rows are a
// power of two apart (read and nothing else, 4096 -> [2 x 14336], a start of 6 blocks:
// 41.5 us, 1: 63, none: 48), and each XCD has blocks that follow each other (39.9).
#pragma once
#include "layered/elem.h"

namespace rows_core {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;

constexpr int KS = 128, ROW = KS * 2;          // ROW: bytes of a row in LDS
constexpr int RING = 3;          // 4 are no faster, 2 up to 15 % slower

// Cache policy (nt) of loads of weights that one workgroup reads. As other loads they push
// x and each other's lines on their way out of the L2 caches: 1 row, 4096 -> [2 x 14336]
// 41.8 us, so 38.3 (6.1 TB/s); 25600 -> 5120 47.4, 42.1; 30 rows 42.3 and 39.3, 49.3 and
// 44.2. (sc0, or sc0 and sc1, gain a third of that.) Weights that stay in the 256 MB
// cache from one pass to the next lose by it, which only those of a model of less than
// 100 million parameters do, and a matrix does not tell: 4096 -> 4096, 1 and 64 rows, of
// 64 MB in turn 4.7 and 7.9 us, so 5.1 and 8.6; of 700 MB 8.4 and 11.2, 7.7 and 10.0.
// Those that several workgroups read at a time are to be loaded without (experts.hip).
constexpr int ONCE = 2;

// what is past the end of K
__device__ const float4v zeros = {0.f, 0.f, 0.f, 0.f};

// The block that workgroup i of n has, a multiple of 8, where each round of workgroups
// over the chip is dealt out so that an XCD has blocks that follow each other (65536 x
// 2048: 52.4 us, 59.6 in the order of the grid; over the whole grid 49.3, but 128256 x
// 4096 171.6, 168.7 and 175.9: eight far ends of a large matrix).
__device__ __forceinline__ int along_xcd(int i, int n, int round) {
  const int first = i / round * round, at = i - first;
  return first + at % 8 * (min(round, n - first) / 8) + at / 8;
}

// RT: rows of x / 16. BN rows of w for BN / 16 waves. A wave has CT tiles of 16 channels
// by MT of 16 rows. HINT: cache policy of the loads of w.
template <int RT, int BN, int HINT = ONCE>
struct RowsCore {
  static constexpr int NW = BN / 16, WM = RT == 1 ? 1 : 2, WC = NW / WM;
  static constexpr int CT = BN / 16 / WC, MT = RT / WM;
  static constexpr int W_STEP = BN * ROW, X_STEP = 16 * RT * ROW;
  static constexpr int RINGS = RING * (W_STEP + X_STEP);
  // loads of a wave, 4 rows each (where x has fewer the last one is repeated)
  static constexpr int WL = BN / 4 / NW, XL = (4 * RT + NW - 1) / NW;

  // A load takes 4 rows of KS, 16 pieces of 16 bytes each; the pieces of a row change
  // places by XOR with its number, so that 16 lanes that read one piece of 16 rows find
  // all banks. The first of the rows of a wave's load j, and a lane's piece:
  static __device__ __forceinline__ int w_row(int wave, int j) {
    return (wave * WL + j) * 4;
  }
  static __device__ __forceinline__ int x_row(int wave, int j) {
    return min(wave * XL + j, 4 * RT - 1) * 4;
  }
  static __device__ __forceinline__ int piece(int row, int lane) {
    return (lane % 16 ^ row % 16) * 8;
  }

  // 4 rows of K from k on, rows 4 q .. of their kind
  template <int POLICY>
  static __device__ __forceinline__ void load(const short* from, char* to, int q,
                                              int lane, int k, int k_hi) {
    typedef const __attribute__((address_space(1))) unsigned int gmem;
    typedef __attribute__((address_space(3))) unsigned int smem;
    const bool in = k + piece(q * 4 + lane / 16, lane) < k_hi;
    __builtin_amdgcn_global_load_lds((gmem*)(in ? from + k : (const short*)&zeros),
                                     (smem*)(to + q * 1024), 16, 0, POLICY);
  }

  // K from k_lo to k_hi in `steps` of KS, from step `first` on and round; past k_hi it
  // counts as zero. w_from, x_from: the lane's piece at K = 0 of its row, w_row + lane /
  // 16 and x_row + lane / 16, of each load; rows that do not exist repeat others. A wave
  // without any of w (its 16 from w_row on) says so by `some`.
  static __device__ __forceinline__ void run(
      char* lds, int wave, int lane, const short* const (&w_from)[WL],
      const short* const (&x_from)[XL], int k_lo, int k_hi, int steps, int first,
      bool some, float4v (&acc)[CT][MT]) {
    char* const w_ring = lds;
    char* const x_ring = lds + RING * W_STEP;
    const int col = lane % 16, grp = lane / 16;
    auto k_of = [&](int s) {
      s += first;
      return k_lo + (s >= steps ? s - steps : s) * KS;
    };
    auto issue = [&](int s, int buf) {
      const int k = k_of(s);
      if (some)
#pragma unroll
        for (int j = 0; j < WL; ++j)
          load<HINT>(w_from[j], w_ring + buf * W_STEP, wave * WL + j, lane, k, k_hi);
#pragma unroll
      for (int j = 0; j < XL; ++j)
        load<0>(x_from[j], x_ring + buf * X_STEP, x_row(wave, j) / 4, lane, k, k_hi);
    };

#pragma unroll
    for (int c = 0; c < CT; ++c)
#pragma unroll
      for (int t = 0; t < MT; ++t) acc[c][t] = (float4v){0.f, 0.f, 0.f, 0.f};
    const int wc = wave % WC, wm = wave / WC;
    struct Operands {
      bf16x8 w[CT], x[MT];
    };
    const int w_at = (wc * 16 * CT + col) * ROW, x_at = (wm * 16 * MT + col) * ROW;
    auto read = [&](Operands& o, int buf, int q) {      // q: 32 of K
      const int at = ((q * 4 + grp) ^ col) * 16;
      const char* w = w_ring + buf * W_STEP + w_at + at;
      const char* x = x_ring + buf * X_STEP + x_at + at;
#pragma unroll
      for (int c = 0; c < CT; ++c)
        o.w[c] = *(const bf16x8*)(w + c * 16 * ROW);
#pragma unroll
      for (int t = 0; t < MT; ++t)
        o.x[t] = *(const bf16x8*)(x + t * 16 * ROW);
      __builtin_amdgcn_sched_barrier(0);
    };
    auto multiply = [&](const Operands& o) {
#pragma unroll
      for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int c = 0; c < CT; ++c)
          acc[c][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              o.w[c], o.x[t], acc[c][t], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    };
    // step s has landed, and so it has for the other waves, when only the next one is
    // under way
    auto landed = [&](int s) {
      if (s + 1 == steps)
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      else if (some)
        asm volatile("s_waitcnt vmcnt(%0)" ::"i"(WL + XL) : "memory");
      else
        asm volatile("s_waitcnt vmcnt(%0)" ::"i"(XL) : "memory");
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
    };

    // Operands are read 32 of K ahead of their products. At the barrier ahead of the
    // last of step s all of its operands are in registers: its places take step s +
    // RING.
    static_assert(RING == 3, "");
    issue(0, 0);
    if (1 < steps) issue(1, 1);
    Operands o0, o1;
    landed(0);
    if (2 < steps) issue(2, 2);
    read(o0, 0, 0);
    int buf = 0;
    for (int s = 0; s < steps; ++s) {
      read(o1, buf, 1);
      multiply(o0);
      read(o0, buf, 2);
      multiply(o1);
      read(o1, buf, 3);
      multiply(o0);
      if (s + 1 < steps) {
        landed(s + 1);
        if (s + RING < steps) issue(s + RING, buf);
        buf = buf + 1 == RING ? 0 : buf + 1;
        read(o0, buf, 0);
      }
      multiply(o1);
    }
  }
};

}  // namespace rows_core
