// experts.hip — feed-forward experts: the router, (token, expert) pairs sorted
// by expert, and the experts' products over them.
//
// A pair's inner row is act(weight * up[e] h): the weight scales the expert's
// input, and since the product is linear it is applied to the 32-bit sums.
// Pairs are sorted by expert (stable, so results do not depend on timing) and
// cut into tiles of one expert each; the product kernels take one tile and a
// block of output channels per workgroup:
//   expert_tiles   256, 192 or 128 pairs and 256 channels through LDS, for many pairs
//   expert_rows    up to 64 pairs, for few: there the weights' bytes are what counts
//   expert_plain   any size, bf16 or float
#include "elem.h"
#include "../rows_core.h"
#include "../tile_core.h"

#include <climits>

namespace {

// ---- router ----------------------------------------------------------------
// The `top` largest of z[0, E) by one wave: experts and sigmoids of their
// scores, largest first, the lower expert on ties. An expert's place is the
// number of experts ahead of it.
__device__ void take_top(const float* z, int E, int top, int32_t* ids,
                         float* wt) {
  for (int e = threadIdx.x % WAVE; e < E; e += WAVE) {
    const float mine = z[e];
    int place = 0;
#pragma unroll 8
    for (int i = 0; i < E; ++i)
      place += z[i] > mine || (z[i] == mine && i < e);
    if (place < top) {
      ids[place] = e;
      wt[place] = sigmoid_f(mine);
    }
  }
}

// any size; one workgroup per row
template <typename T>
__global__ __launch_bounds__(256) void route_plain_kernel(
    const T* __restrict__ h, const T* __restrict__ w, int32_t* __restrict__ ids,
    float* __restrict__ wt, int K, int E, int top) {
  extern __shared__ float z[];
  const int64_t row = blockIdx.x;
  const int wave = threadIdx.x / WAVE, lane = threadIdx.x % WAVE;
  for (int e = wave; e < E; e += 4) {
    float s = 0.f;
    for (int k = lane; k < K; k += WAVE)
      s += ld(h + row * K + k) * ld(w + (int64_t)e * K + k);
    s = wave_reduce_sum(s);
    if (lane == 0) z[e] = s;
  }
  __syncthreads();
  if (wave == 0) take_top(z, E, top, ids + row * top, wt + row * top);
}

// R rows per workgroup: 16 of a matrix instruction, or 4 where that is at most a round of
// workgroups. EG groups of KW waves have 16 ET experts each and share K.
// Bound by what a compute unit can load: the lanes of a load are to follow each other in
// a row of memory, as operands they lie in 16 rows and a load took four times as long.
// 32 experts of 4096, 60 rows 9.8 us (15.0), 7800 rows 20.4 (32.9); 64 experts 17.2
// (26.8), 31.0 (48.0); 128 of 2048 23.8 (38.4), 43.8 (61.8). By 4 rows a unit loads a
// quarter less and a wave chooses for one: 60 rows again, warm, by 16 / by 4: 8.3 / 6.6 us,
// 64 experts 13.6 / 10.6, 128 of 2048 19.5 / 15.7; 1000 rows 8.7 / 7.2, 14.2 / 11.1, 19.9 /
// 17.6. Two steps of K asked for together are no faster. 16 waves in place of 8 are
// no faster up to 64 experts (9.6 and 23.7 us for 32), above they are (27.3 and 40.6 by 8).
template <int ET, int EG, int KW, int R>
__global__ __launch_bounds__(EG * KW * WAVE) void route_kernel(
    const short* __restrict__ h, const short* __restrict__ w,
    int32_t* __restrict__ ids, float* __restrict__ wt, int64_t rows, int K,
    int E, int top) {
  extern __shared__ __align__(16) float lds[];   // 4 KB of a wave; [KW][16 rows][16 ES]
  constexpr int ES = ET * EG;
  const int wave = threadIdx.x / WAVE, lane = threadIdx.x % WAVE;
  const int col = lane % 16, grp = lane / 16;
  const int e0 = wave / KW * ET * 16, kw = wave % KW;
  const int64_t row0 = (int64_t)blockIdx.x * R;
  char* mine = (char*)lds + wave * 4096;
  const short8 zero = {0, 0, 0, 0, 0, 0, 0, 0};
  float4v acc[ET];
#pragma unroll
  for (int t = 0; t < ET; ++t) acc[t] = (float4v){0.f, 0.f, 0.f, 0.f};
  // past the end of K the row counts as zero; experts past E are not looked at
  const short* h0 = h + row0 * K;
  const int last = min(rows - 1 - row0, (int64_t)(R - 1));
  for (int k0 = kw * 128; k0 < K; k0 += KW * 128) {
    short8 a[4], b[ET][4];
    const int k = k0 + col * 8, kc = min(k, K - 8);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int r = j * 4 + grp;
      a[j] = j * 4 < R ? *(const short8*)(h0 + (uint32_t)(min(r, last) * K + kc)) : zero;
#pragma unroll
      for (int t = 0; t < ET; ++t)
        b[t][j] =
            *(const short8*)(w + (uint32_t)(min(e0 + t * 16 + r, E - 1) * K + kc));
    }
    __builtin_amdgcn_sched_barrier(0);       // all loads ahead of their first use
    if (k >= K)
#pragma unroll
      for (int j = 0; j < 4; ++j) a[j] = zero;
    to_operand(mine, lane, a);
#pragma unroll
    for (int t = 0; t < ET; ++t) {
      to_operand(mine, lane, b[t]);
#pragma unroll
      for (int f = 0; f < 4; ++f)
        acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
            __builtin_bit_cast(bf16x8, b[t][f]), __builtin_bit_cast(bf16x8, a[f]),
            acc[t], 0, 0, 0);
    }
  }
  __syncthreads();
#pragma unroll
  for (int t = 0; t < ET; ++t)
    *(float4v*)(lds + (kw * 16 + col) * 16 * ES + e0 + t * 16 + grp * 4) = acc[t];
  __syncthreads();
  for (int i = threadIdx.x; i < 16 * R * ES; i += EG * KW * WAVE) {
    float s = lds[i];
#pragma unroll
    for (int v = 1; v < KW; ++v) s += lds[v * 256 * ES + i];
    lds[i] = s;
  }
  __syncthreads();
  for (int r = wave; r < R && row0 + r < rows; r += EG * KW)
    take_top(lds + r * 16 * ES, E, top, ids + (row0 + r) * top,
             wt + (row0 + r) * top);
}

// ---- sorting ---------------------------------------------------------------
constexpr int ST = 1024, SV = 8;   // threads; pairs per thread and sweep
constexpr int TILE = 256;          // pairs of a tile of expert_tiles

// SV experts from place i on; -1 past the end (i is a multiple of SV)
__device__ __forceinline__ void load_ids(const int32_t* ids, int i, int P,
                                         int* x) {
  if (i + SV <= P) {
    const int4 a = *(const int4*)(ids + i), b = *(const int4*)(ids + i + 4);
    x[0] = a.x; x[1] = a.y; x[2] = a.z; x[3] = a.w;
    x[4] = b.x; x[5] = b.y; x[6] = b.z; x[7] = b.w;
  } else {
#pragma unroll
    for (int j = 0; j < SV; ++j) x[j] = i + j < P ? ids[i + j] : -1;
  }
}

// One workgroup per expert. order [P]: pairs by expert; tiles [1 + max_tiles]
// = (number of tiles, those ahead, ..), then (expert, first place in order,
// pairs, 0). Those more than half full go ahead, so that the shorter work comes
// last (2000 rows, 32 experts of 4096 x 3584, 4 each: 638 us, by expert 660;
// 2048 x 1536: 157 and 171). `share`: the weights are too many to stay in the
// last-level cache, and tiles of one expert want to run together. So they do,
// by expert, where workgroups read weights straight from memory (tiles of up to
// 64 pairs) and some expert has several (380 rows of uneven loads: 592 us for
// 617), and where every expert has several of the large ones (2500 rows: 812 us
// for 877).
__global__ __launch_bounds__(ST) void sort_pairs_kernel(
    const int32_t* __restrict__ ids, int32_t* __restrict__ order,
    int4* __restrict__ tiles, int P, int E, int tile, int share) {
  extern __shared__ int hist[];        // [E]
  __shared__ int sums[ST / WAVE], at[5];
  const int e = blockIdx.x, tid = threadIdx.x;
  const int wave = tid / WAVE, lane = tid % WAVE;
  for (int i = tid; i < E; i += ST) hist[i] = 0;
  __syncthreads();
  for (int i = tid * SV; i < P; i += ST * SV) {
    int x[SV];
    load_ids(ids, i, P, x);
#pragma unroll
    for (int j = 0; j < SV; ++j)
      if (x[j] >= 0 && x[j] < E) atomicAdd(&hist[x[j]], 1);
  }
  __syncthreads();
  if (wave == 0) {       // pairs and tiles of lower experts, those ahead of all
    int n = 0, full = 0, rest = 0, all = 0, ahead = tile / 2 + 1;
    if (share) {
      bool all_do = true, some_do = false;       // have several tiles
      for (int i = lane; i < E; i += WAVE) {
        all_do &= hist[i] > tile;
        some_do |= hist[i] > tile;
      }
      if (tile < TILE ? __any(some_do) : __all(all_do)) ahead = 1;
    }
    for (int i = lane; i < E; i += WAVE) {
      const int f = (hist[i] + tile - ahead) / tile;
      all += f;
      if (i < e) {
        n += hist[i];
        full += f;
        rest += (hist[i] + tile - 1) / tile - f;
      }
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      n += __shfl_xor(n, o, WAVE);
      full += __shfl_xor(full, o, WAVE);
      rest += __shfl_xor(rest, o, WAVE);
      all += __shfl_xor(all, o, WAVE);
    }
    if (lane == 0) {
      at[0] = n;
      at[1] = full;
      at[2] = rest;
      at[3] = all;
      at[4] = ahead;
    }
  }
  __syncthreads();
  const int first = at[0], count = hist[e];
  const int nt = (count + tile - 1) / tile;
  const int nf = (count + tile - at[4]) / tile;
  for (int j = tid; j < nt; j += ST)
    tiles[1 + (j < nf ? at[1] + j : at[3] + at[2])] =
        make_int4(e, first + j * tile, min(tile, count - j * tile), 0);
  if (e == E - 1 && tid == 0)
    tiles[0] = make_int4(at[3] + at[2] + nt - nf, at[3], 0, 0);
  int base = first;
  for (int i0 = 0; i0 < P; i0 += ST * SV) {   // workgroup-uniform
    const int i = i0 + tid * SV;
    int mine = 0, x[SV];
    load_ids(ids, i, P, x);
#pragma unroll
    for (int j = 0; j < SV; ++j) mine |= (x[j] == e) << j;
    const int n = __popc(mine);
    int before = n;                    // inclusive sum over the wave
#pragma unroll
    for (int o = 1; o < WAVE; o <<= 1) {
      const int v = __shfl_up(before, o, WAVE);
      if (lane >= o) before += v;
    }
    __syncthreads();
    if (lane == WAVE - 1) sums[wave] = before;
    __syncthreads();
    int total = 0, place = base + before - n;
#pragma unroll
    for (int w = 0; w < ST / WAVE; ++w) {
      if (w < wave) place += sums[w];
      total += sums[w];
    }
#pragma unroll
    for (int j = 0; j < SV; ++j)
      if (mine >> j & 1) order[place++] = i + j;
    base += total;
  }
}

// ---- products --------------------------------------------------------------
struct Pairs {
  const void* a;             // UP: h [T, K]; else inner rows [P, K], sorted
  const void* w;             // [E, N, K]
  void* out;                 // UP: inner rows [P, N], sorted; else [P, N]
  const int32_t* order;      // place -> pair
  const int4* tiles;
  const float* weights;      // [P]
  int N, K, top, act;
  int width;                 // expert_rows: channels of a workgroup
};

// input row of a place
template <bool UP>
__device__ __forceinline__ int64_t source(const Pairs& p, int place) {
  return UP ? p.order[place] / p.top : place;
}
template <bool UP>
__device__ __forceinline__ float finish(const Pairs& p, float sum, float wt) {
  return UP ? activate(p.act, sum * wt) : sum;
}

// grid (blocks of channels, tiles)
template <typename T, bool UP>
__global__ __launch_bounds__(256) void expert_plain_kernel(const Pairs p) {
  if ((int)blockIdx.y >= p.tiles[0].x) return;
  const int4 tile = p.tiles[1 + blockIdx.y];
  const int wave = threadIdx.x / WAVE, lane = threadIdx.x % WAVE;
  const int n1 = min(p.N, (int)(blockIdx.x + 1) * 64);
  for (int i = tile.y; i < tile.y + tile.z; ++i) {
    const int pair = p.order[i];
    const T* a = (const T*)p.a + source<UP>(p, i) * p.K;
    T* o = (T*)p.out + (int64_t)(UP ? i : pair) * p.N;
    for (int n = blockIdx.x * 64 + wave; n < n1; n += 4) {
      const T* w = (const T*)p.w + ((int64_t)tile.x * p.N + n) * p.K;
      float s = 0.f;
      for (int k = lane; k < p.K; k += WAVE) s += ld(a + k) * ld(w + k);
      s = wave_reduce_sum(s);
      if (lane == 0) st(o + n, finish<UP>(p, s, p.weights[pair]));
    }
  }
}

// grid (blocks of BN channels up to a multiple of 8, tiles of up to 16 RT pairs). The
// weights stream as in linear_rows.hip; by 64 channels there are two workgroups to a
// compute unit, whose ends overlap, by 128 the pairs' rows are read half as often. Both
// products, 32 experts of 4096 x 3584, 4 each, in us; before: weights straight to
// registers, by 32 bytes of a row (their bytes alone take 313 at 6.0 TB/s):
//   rows         8    60   150   300
//   before     238   344   414   518
//   64         225   325   338   360
//   128        225   328   334   350
// and 64 experts of 2048 x 1408, 6 each, 250 rows 191, 149, 151. So tiles of 64 pairs
// take 128.
//
// Weights that one tile reads go past the L2 caches (rows_core.h), not those that the
// next tile in the list reads too, which finds them there. Both products as above, by how
// uneven the loads are (standard deviation of the choice's logits), all weights by way of
// the caches / all past them / so:
//   rows         60                100               180               380
//   0     325 / 292 / 290   328 / 293 / 298   353 / 328 / 327   352 / 342 / 345
//   0.5   328 / 302 / 295   337 / 308 / 306   372 / 371 / 353   400 / 422 / 402
//   1.5   302 / 294 / 285   319 / 317 / 305   395 / 418 / 387   437 / 472 / 423
template <int RT, int BN, bool UP>
__global__ __launch_bounds__(BN / 16 * WAVE) void expert_rows_kernel(const Pairs p) {
  extern __shared__ __align__(16) char ring[];
  typedef rows_core::RowsCore<RT, BN> Core;
  constexpr int WL = Core::WL, XL = Core::XL, CT = Core::CT, MT = Core::MT;
  if ((int)blockIdx.y >= p.tiles[0].x) return;
  const int N = p.N, K = p.K, blocks = gridDim.x;
  const int i = rows_core::along_xcd(blockIdx.y * blocks + blockIdx.x,
                                     p.tiles[0].x * blocks, BN == 64 ? 512 : 256);
  const int at = i / blocks, tiles = p.tiles[0].x;
  const int4 tile = p.tiles[1 + at];
  const bool several = (at > 0 && p.tiles[at].x == tile.x) ||
                       (at + 1 < tiles && p.tiles[2 + at].x == tile.x);
  const int n0 = i % blocks * p.width, n1 = min(N, n0 + p.width);
  if (n0 >= N) return;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
  const int lane = threadIdx.x % WAVE, col = lane % 16, grp = lane / 16;
  const short *w_from[WL], *x_from[XL];
#pragma unroll
  for (int j = 0; j < XL; ++j) {
    const int r = Core::x_row(wave, j);    // uniform: places come by scalar loads
    int64_t from = 0;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int64_t f = source<UP>(p, tile.y + min(r + q, tile.z - 1));
      from = grp == q ? f : from;
    }
    x_from[j] = (const short*)p.a + from * K + Core::piece(r + grp, lane);
  }
#pragma unroll
  for (int j = 0; j < WL; ++j) {
    const int r = Core::w_row(wave, j) + grp;
    w_from[j] = (const short*)p.w +
                ((int64_t)tile.x * N + min(n0 + r, n1 - 1)) * K + Core::piece(r, lane);
  }
  float4v acc[CT][MT];
  const int steps = (K + rows_core::KS - 1) / rows_core::KS;
  // by the expert, not its tile's rank: a row's sums do not hang on what others chose
  const uint32_t first = uint32_t(tile.x * blocks + i % blocks) * BN / 128 * 3;
  auto run = [&](auto core) {
    decltype(core)::run(ring, wave, lane, w_from, x_from, 0, K, steps,
                        first % uint32_t(steps), wave * 16 < p.width, acc);
  };
  if (several)
    run(rows_core::RowsCore<RT, BN, 0>{});
  else
    run(Core{});
#pragma unroll
  for (int t = 0; t < MT; ++t) {
    const int m = (wave / Core::WC * MT + t) * 16 + col;
    if (m >= tile.z) continue;
    const int pair = p.order[tile.y + m];
    const float wt = UP ? p.weights[pair] : 1.f;
#pragma unroll
    for (int c = 0; c < CT; ++c) {
      const int n = n0 + (wave % Core::WC * CT + c) * 16 + grp * 4;
      if (n >= n1) continue;
      const float4v s = acc[c][t];
      *(short4v*)((short*)p.out + (int64_t)(UP ? tile.y + m : pair) * N + n) =
          (short4v){f32_to_bf16(finish<UP>(p, s[0], wt)),
                    f32_to_bf16(finish<UP>(p, s[1], wt)),
                    f32_to_bf16(finish<UP>(p, s[2], wt)),
                    f32_to_bf16(finish<UP>(p, s[3], wt))};
    }
  }
}

// Channels of a workgroup, of BN at most, with which about `tiles` tiles take the least of
// whole rounds of the chip (32 experts of 3584 channels: 3.5 rounds by 64, 4 by 56)
int even_width(int N, int BN, int tiles) {
  const int slots = BN == 64 ? 512 : 256;
  int best = BN, least = INT_MAX;
  for (int width = BN; width > BN / 2; width -= 8) {
    const int64_t blocks = (int64_t)((N + width - 1) / width) * tiles;
    const int64_t cost = (blocks + slots - 1) / slots * width;
    if (cost < least) least = (int)cost, best = width;
  }
  return best;
}

template <int RT, int BN, bool UP>
hipError_t launch_rows(Pairs p, int max_tiles, int tiles, hipStream_t stream) {
  typedef rows_core::RowsCore<RT, BN> Core;
  auto fn = expert_rows_kernel<RT, BN, UP>;
  const hipError_t e = hipFuncSetAttribute(
      (const void*)fn, hipFuncAttributeMaxDynamicSharedMemorySize, Core::RINGS);
  if (e != hipSuccess) return e;
  p.width = even_width(p.N, BN, tiles);
  hipLaunchKernelGGL(fn, dim3(((p.N + p.width - 1) / p.width + 7) / 8 * 8, max_tiles),
                     dim3(Core::NW * WAVE), Core::RINGS, stream, p);
  HIP_CHECK_LAST();
  return hipSuccess;
}

// 256 channels x 256 pairs, or 128 where a tile has no more (so nothing is lost by
// the larger tile): see tile_core.h for the loop and what bounds it. Both products,
// 7032 rows, 32 experts of 4096 x 3584, 4 each: 1290 us, 1280 TFLOP/s of useful
// work (1655 with 32x32 instructions, address arithmetic in the loop and places
// read while the results leave); 2000 rows 580 us (652); 16000 rows, 64 experts of
// 2048 x 1024, 2 each: 311 us (378). Four tiles of pairs side by side: a compute
// die's 32 workgroups share the loads of 4 + 8 tiles (8192 x 4096 -> 28672 in 1320
// us, 1366 with 3).
constexpr int TC = 256, BK = TILE_K, HALF = 128;
constexpr int TG = 4;                // tiles of pairs that run side by side
typedef TileCore<8, 8, 2> Whole;
typedef TileCore<8, 6, 2> Most;   // 192 pairs
typedef TileCore<4, 8, 4> Half;
static_assert(Whole::CHANNELS == TC && Most::CHANNELS == TC && Half::CHANNELS == TC &&
                  Whole::ROWS == TILE && Half::ROWS == HALF &&
                  Most::LDS_TURN <= Whole::LDS_TURN &&
                  Half::LDS_TURN <= Whole::LDS_TURN,
              "");

template <bool UP, typename Core>
__device__ __forceinline__ void tile_product(const Pairs& p, short* lds,
                                             const int4 tile, int n0) {
  Core core;
  constexpr int LW = Core::LW, LP = Core::LP, PT = Core::ROWS / 16 / Core::WP;
  constexpr int QP = Core::QP;
  const int N = p.N, K = p.K;
  // channels past the end and rows past the tile repeat the last one: they are
  // computed and dropped
  uint32_t wsrc[2][LW], asrc[2][LP];
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int j = 0; j < LP; ++j)
      asrc[h][j] = source<UP>(
          p, tile.y + min(h * Core::RH + core.template loaded<LP>(j),
                          tile.z - 1));
#pragma unroll
  for (int h = 0; h < 2; ++h) {
#pragma unroll
    for (int j = 0; j < LW; ++j)
      wsrc[h][j] =
          ((uint32_t)min(n0 + h * Core::CH + core.template loaded<LW>(j),
                         N - 1) * K + core.template piece<LW>(j)) * 2;
#pragma unroll
    for (int j = 0; j < LP; ++j)
      asrc[h][j] = (asrc[h][j] * K + core.template piece<LP>(j)) * 2;
  }
  // what the results need is on its way while the products run: weights by row,
  // or the places that the rows of a quarter go to
  float wt[PT];
  int32_t to[2];
  if constexpr (UP) {
#pragma unroll
    for (int t = 0; t < PT; ++t)
      wt[t] = p.weights[p.order[tile.y + min(core.row(t) + core.col,
                                             tile.z - 1)]];
  } else {
#pragma unroll
    for (int t = 0; t < 2; ++t)
      to[t] = p.order[tile.y + min(core.row(t * QP) + core.lane, tile.z - 1)];
  }
  // offsets stay under 4 GiB (lds_expert_tile)
  core.run(lds, (const char*)p.w + (int64_t)tile.x * N * K * 2,
           (uint32_t)N * K * 2, wsrc, p.a, 0xfffffff0u, asrc, K / BK,
           [](int s) { return s * BK * 2; });

  auto write = [&](auto act) {
#pragma unroll
    for (int b = 0; b < PT / 2; ++b)
      core.template turn<2 * Core::QC>(
          lds, b,
          [&](int c, int t, int x) {
            const float f = core.acc[c][t][x];
            return UP ? activate(act, f * wt[t]) : f;
          },
          [&](int row, int i, int c, short8 v) {
            int64_t at = tile.y + i;
            if constexpr (!UP) {
              at = __shfl(to[2 * b / QP], 2 * b % QP * 16 + row, WAVE);
              if (2 * b % QP + 1 == QP) {        // its 32 rows lie in two quarters
                const int next = __shfl(to[1], row - 16, WAVE);
                if (row >= 16) at = next;
              }
            }
            if (i < tile.z && n0 + c < N)       // N is a multiple of 8
              *(short8*)((short*)p.out + at * N + n0 + c) = v;
          });
  };
  using std::integral_constant;
  if (!UP || p.act == ACT_RELU_SQUARED)
    write(integral_constant<int, ACT_RELU_SQUARED>{});
  else if (p.act == ACT_SILU)
    write(integral_constant<int, ACT_SILU>{});
  else
    write(integral_constant<int, ACT_GELU_TANH>{});
}

template <bool UP>
__global__ __launch_bounds__(256, 1) void expert_tiles_kernel(const Pairs p) {
  extern __shared__ __align__(16) short tile_lds[];  
  // Workgroups go round the 8 XCDs in turn: each XCD gets a contiguous share
  // of the tiles more than half full, then one of the others (the shorter
  // work last), in which TG tiles of pairs walk the channels together.
  const int nx = (p.N + TC - 1) / TC;
  const int4 counts = p.tiles[0];
  int n = counts.y, base = 1, at = blockIdx.x / 8;
  int share = (n * nx + 7) / 8;
  if (at >= share) {
    at -= share;
    base += n;
    n = counts.x - n;
    share = (n * nx + 7) / 8;
  }
  const int id = blockIdx.x % 8 * share + at;
  if (at >= share || id >= n * nx) return;
  const int g = id / (TG * nx), in = id % (TG * nx);
  const int width = min(TG, n - g * TG);
  const int4 tile = p.tiles[base + g * TG + in % width];
  const int n0 = in / width * TC;
  // What a tile's rows do without is left out: 32 experts of 4096 x 3584, 4 each, 1300
  // rows 477 us with tiles of 256 and 128 alone, so 427; 1000 rows 416 and 397; 7821
  // rows, the same.
  if (tile.z > Most::ROWS)
    tile_product<UP, Whole>(p, tile_lds, tile, n0);
  else if (tile.z > HALF)
    tile_product<UP, Most>(p, tile_lds, tile, n0);
  else
    tile_product<UP, Half>(p, tile_lds, tile, n0);
}

template <bool UP>
hipError_t launch_tiles(const Pairs& p, int max_tiles, hipStream_t stream) {
  // every XCD's two shares are rounded up
  const int64_t n =
      (((int64_t)max_tiles * ((p.N + TC - 1) / TC) + 7) / 8 + 1) * 8;
  if (n > 0x7fffffff || p.N % 8 || p.K % BK || p.K < 2 * BK ||
      (int64_t)p.N * p.K >= 1ll << 31)
    return hipErrorInvalidValue;
  auto fn = expert_tiles_kernel<UP>;
  hipError_t e = hipFuncSetAttribute(
      (const void*)fn, hipFuncAttributeMaxDynamicSharedMemorySize, Whole::LDS_TURN);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(fn, dim3((uint32_t)n), dim3(256), Whole::LDS_TURN, stream, p);
  HIP_CHECK_LAST();
  return hipSuccess;
}

template <bool UP>
hipError_t product(int f32, int plain, int tile, int max_tiles, int tiles,
                   const Pairs& p, hipStream_t stream) {
  if (tile == TILE) return launch_tiles<UP>(p, max_tiles, stream);
  const dim3 grid((p.N + 63) / 64, max_tiles), block(256);
  if (max_tiles > 65535 || tile > 64) return hipErrorInvalidValue;
#define GO(KERNEL) hipLaunchKernelGGL((KERNEL), grid, block, 0, stream, p)
#define K2(NAME, ARG) NAME<ARG, UP>
  if (f32) GO(K2(expert_plain_kernel, float));
  else if (plain || p.N % 8 || p.K % 8) GO(K2(expert_plain_kernel, short));
  else if (tile <= 16) return launch_rows<1, 64, UP>(p, max_tiles, tiles, stream);
  else if (tile <= 32) return launch_rows<2, 64, UP>(p, max_tiles, tiles, stream);
  else return launch_rows<4, 128, UP>(p, max_tiles, tiles, stream);
#undef K2
#undef GO
  HIP_CHECK_LAST();
  return hipSuccess;
}

}  // namespace

extern "C" {

hipError_t lds_route(int f32, const void* h, const void* w, int32_t* ids,
                     float* wt, int64_t rows, int K, int E, int top,
                     hipStream_t stream) {
  if (rows == 0) return hipSuccess;
  if (top < 1 || top > E || E > 8192) return hipErrorInvalidValue;
  if (f32 || K % 8 || E > 256 || (int64_t)E * K >= 1ll << 31) {
    const size_t lds = E * sizeof(float);
    if (f32)
      hipLaunchKernelGGL(route_plain_kernel<float>, dim3((uint32_t)rows),
                         dim3(256), lds, stream, (const float*)h,
                         (const float*)w, ids, wt, K, E, top);
    else
      hipLaunchKernelGGL(route_plain_kernel<short>, dim3((uint32_t)rows),
                         dim3(256), lds, stream, (const short*)h,
                         (const short*)w, ids, wt, K, E, top);
    HIP_CHECK_LAST();
    return hipSuccess;
  }
#define GO(ET, EG, KW)                                                        \
  do {                                                                        \
    if (rows <= 4 * 256) GO_R(ET, EG, KW, 4);                                 \
    else GO_R(ET, EG, KW, 16);                                                \
  } while (0)
#define GO_R(ET, EG, KW, R)                                                   \
  hipLaunchKernelGGL((route_kernel<ET, EG, KW, R>),                           \
                     dim3((uint32_t)((rows + R - 1) / R)),                    \
                     dim3(EG * KW * WAVE), EG * KW * 4096, stream,            \
                     (const short*)h, (const short*)w, ids, wt, rows, K, E, top)
  if (E <= 16) GO(1, 1, 8); else if (E <= 32) GO(2, 1, 8);
  else if (E <= 64) GO(2, 2, 4); else if (E <= 128) GO(2, 4, 4);
  else GO(2, 8, 2);
#undef GO
#undef GO_R
  HIP_CHECK_LAST();
  return hipSuccess;
}

// pairs of one expert that a workgroup takes: about as many as an expert has
int lds_expert_tile(int f32, int plain, int P, int T, int E, int N, int K) {
  const int per = (P + E - 1) / E;
  const int64_t limit = 1ll << 31;      // elements: offsets stay under 4 GiB
  if (f32 || plain || per <= 12) return 16;
  if (per <= 24) return 32;
  if (per <= 48 || N % BK || K % BK || N < 2 * BK || K < 2 * BK ||
      (int64_t)N * K >= limit || (int64_t)T * K >= limit ||
      (int64_t)P * N >= limit)
    return 64;
  return TILE;
}

// tiles of P pairs at most
int lds_expert_max_tiles(int P, int E, int tile) {
  const int n = P / tile + E;
  return n < P ? n : P;
}

// order [P], tiles [1 + max_tiles, 4]; share: see sort_pairs_kernel
hipError_t lds_sort_pairs(const int32_t* ids, int32_t* order, void* tiles,
                          int P, int E, int tile, int share,
                          hipStream_t stream) {
  if (P == 0) return hipSuccess;
  if (E > 8192) return hipErrorInvalidValue;
  hipLaunchKernelGGL(sort_pairs_kernel, dim3(E), dim3(ST), E * sizeof(int),
                     stream, ids, order, (int4*)tiles, P, E, tile, share);
  HIP_CHECK_LAST();
  return hipSuccess;
}

// One layer of the experts (up: the first). a, out: see Pairs.
hipError_t lds_expert_product(int f32, int plain, int up, const void* a,
                              const void* w, void* out, const int32_t* order,
                              const void* tiles, int max_tiles, int tile,
                              const float* weights, int E, int N, int K, int top,
                              int act, hipStream_t stream) {
  if (max_tiles == 0) return hipSuccess;
  const Pairs p{a, w, out, order, (const int4*)tiles, weights, N, K, top, act, 0};
  const int some = E < max_tiles ? E : max_tiles;      // a tile per expert, or so
  return up ? product<true>(f32, plain, tile, max_tiles, some, p, stream)
            : product<false>(f32, plain, tile, max_tiles, some, p, stream);
}

}  // extern "C"
