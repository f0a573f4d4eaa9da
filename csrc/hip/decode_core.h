// decode_core.h — attention of single rows over paged keys and values (gfx950): heads of
// 128 in groups of up to 8 that share keys, bf16 or 8-bit caches. paged_attention.hip
// runs it over a pool of its own for keys and values, layered/paged_decode.hip over rows
// [key | value].
//
// Geometry: one workgroup per (sequence, kv_head, partition). Its waves take
// tiles of 32 tokens in turn, each with an online softmax of its own, and meet
// once at the end: no LDS and no barrier while the cache streams by. Both
// products run on the matrix cores, with the operands as they come from
// memory:
//   S' = K Q'  a lane holds 16 bytes of a token's key (bf16 matrix cores; the
//              order of the key's channels inside a step is free, Q follows).
//              It gets back the scores of 4 + 4 tokens for one head.
//   O  = P V   bf16 matrix cores, a step for 32 tokens and 16 channels: a
//              probability is the sum of three bf16, all 24 bits of it, as the
//              scores left them in the lane; values are bf16 as they are (fp8
//              ones exactly). A lane holds 8 channels of 8 tokens and turns them
//              round for itself.
// A tile's matrix work is 512 cycles (2176 with P V on the 32-bit cores, which
// for fp8 was as long as its bytes took, and the most power of a pass), its vector
// work 700 (bf16) to 930 (fp8): less than its bytes take at 5 TB/s with three waves
// a SIMD, so the 12 to 15 columns that a group of 1 to 4 heads leaves idle cost
// nothing.
//
// Values are read by whole rows and, where no other row reads them too, past the caches:
// as other loads they push keys out of them, a load of which takes 64 bytes of 16 rows,
// whose other halves have to be found again. Where sequences share blocks it is what one
// of them leaves in the caches that the others find. By way of them / past them / as the
// rows' tables say (shared), us, 8 key heads:
//   256 of 1500 tokens, none shared     271 / 251 / 252.5    8-bit 150 / 138 / 142
//   17 of 6800, none shared             95 / 87.5 / 87.8    56 / 52 / 52
//   30 of 1100, none shared             29.1 / 27.5 / 27.7    17.1 / 16.2 / 16.7
//   256 of 1500, 1000 of one prefix     166 / 182 / 169    95 / 104 / 97
//   256 of 1500, 1000 of 8 prefixes     170 / 196 / 173    96 / 112 / 99
//   256 of 1500, 500 of 8 prefixes      217 / 218 / 221    123 / 127 / 129
//   64 of 4100, 4000 of one prefix      82 / 101 / 82    54 / 59 / 56
// Chosen tile by tile the branch around the loads costs more than it gives (fp8, 64 of
// 4100, 4000 shared: 73).
//
// Measured alone, cold (8 key heads, ragged; before: P V on the 32-bit cores): 256
// sequences of 1500 tokens, groups of 4: 252 us, 6.2 TB/s (279), fp8 156 us (191), by 4
// waves 142, 5.5 TB/s; 30 of 1100, groups of 8: 27.5 us (31.5); 17 of 6800, fp8, in 4
// partitions by 8 waves: 51 us, 4.5 TB/s (66.5; with its sum 56.6, in 6 by 4 waves 50.6);
// 60 of 300: 15.7 us (19.9); one of 777: 9.3 us (10.3). Registers let a compute unit have
// 12 waves: one workgroup of 8 or three of 4. One of 12 is no faster.
//
// Flash-decoding sequence split (SPLIT): long sequences are cut into
// gridDim.z partitions so that small batches fill the chip. Each partition
// writes an UNNORMALIZED partial (o_acc, m, l) and a tiny combine kernel
// merges partitions: m* = max m_p; o = sum o_p*exp(m_p-m*); l likewise.
#pragma once
#include "hip_common.h"

#include <type_traits>

namespace decode {

constexpr int D = 128;        // head_dim (Llama-3 family)
constexpr int TILE = 32;      // tokens per wave and step
constexpr int MAX_QPG = 8;
constexpr float NEG = -1e30f;
constexpr float LOG2E = 1.4426950408889634f;
// The running maximum moves only when a score passes it by this much (log2):
// sums stay below 2^8 times a tile's, far inside 32-bit range, and the
// accumulators are rarely rescaled.
constexpr float SLACK = 8.f;

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) unsigned int uint4v;
typedef __attribute__((ext_vector_type(2))) unsigned int uint2v;

// How a cache type's loads map to operands.
//   KL loads of 16 bytes make up a lane's share of a key (its 4 steps)
//   dim(s, g): first of the 8 channels that lane group g holds in step s
template <typename CT> struct Cache;

template <> struct Cache<short> {
  static constexpr int KL = 4;
  typedef uint4v VReg;
  static __device__ __forceinline__ int dim(int s, int g) {
    return s * 32 + g * 8;
  }
  static __device__ __forceinline__ bf16x8 key(const uint4v* k, int s) {
    return __builtin_bit_cast(bf16x8, k[s]);
  }
  // channels CH d .. of a lane's 8 tokens as operands, two tokens per register
  static constexpr int CH = 2;
  static __device__ __forceinline__ void values(const VReg (&v)[2][4], int d,
                                                uint4v* o) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const unsigned int x = v[i / 2][i % 2 * 2][d];
      const unsigned int y = v[i / 2][i % 2 * 2 + 1][d];
      o[0][i] = __builtin_amdgcn_perm(y, x, 0x05040100);
      o[1][i] = __builtin_amdgcn_perm(y, x, 0x07060302);
    }
  }
};

template <> struct Cache<unsigned char> {
  static constexpr int KL = 2;
  typedef uint2v VReg;
  static __device__ __forceinline__ int dim(int s, int g) {
    return s / 2 * 64 + g * 16 + s % 2 * 8;
  }
  static __device__ __forceinline__ void widen(unsigned int v, float* f) {
    const float2v a = __builtin_amdgcn_cvt_pk_f32_fp8(v, false);
    const float2v b = __builtin_amdgcn_cvt_pk_f32_fp8(v, true);
    f[0] = a[0];
    f[1] = a[1];
    f[2] = b[0];
    f[3] = b[1];
  }
  // e4m3 values are bf16 values: the upper halves of the floats
  static __device__ __forceinline__ unsigned int pair(float a, float b) {
    return __builtin_amdgcn_perm(__builtin_bit_cast(uint32_t, b),
                                 __builtin_bit_cast(uint32_t, a), 0x07060302);
  }
  static constexpr int CH = 4;
  static __device__ __forceinline__ void values(const VReg (&v)[2][4], int d,
                                                uint4v* o) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      float x[4], y[4];
      widen(v[i / 2][i % 2 * 2][d], x);
      widen(v[i / 2][i % 2 * 2 + 1][d], y);
#pragma unroll
      for (int c = 0; c < 4; ++c) o[c][i] = pair(x[c], y[c]);
    }
  }
  static __device__ __forceinline__ bf16x8 key(const uint4v* k, int s) {
    float f[8];
    widen(k[s / 2][s % 2 * 2], f);
    widen(k[s / 2][s % 2 * 2 + 1], f + 4);
    uint4v r;
#pragma unroll
    for (int i = 0; i < 4; ++i) r[i] = pair(f[2 * i], f[2 * i + 1]);
    return __builtin_bit_cast(bf16x8, r);
  }
};

// 8 floats as sums of three bf16, exactly but for a last bit or two
__device__ __forceinline__ void split3(const float4v* x, bf16x8* parts) {
  float r[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) r[i] = x[i / 4][i % 4];
#pragma unroll
  for (int p = 0; p < 3; ++p) {
    uint4v w;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float2v two = {r[2 * i], r[2 * i + 1]};
      typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;
      w[i] = __builtin_bit_cast(unsigned int,
                                __builtin_convertvector(two, bf16x2));
      const unsigned int lo = w[i] << 16, up = w[i] & 0xffff0000u;
      r[2 * i] -= __builtin_bit_cast(float, lo);
      r[2 * i + 1] -= __builtin_bit_cast(float, up);
    }
    parts[p] = __builtin_bit_cast(bf16x8, w);
  }
}

// values as they are, but infinite ones 0
__device__ __forceinline__ uint4v finite(uint4v v) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if ((v[i] & 0x7fffu) == 0x7f80u) v[i] &= 0xffff0000u;
    if ((v[i] & 0x7fff0000u) == 0x7f800000u) v[i] &= 0xffffu;
  }
  return v;
}

// One launch's work. Strides in elements.
template <typename CT>
struct Work {
  const short* q;             // rows q_row apart, heads D apart
  int64_t q_row;
  const CT *k, *v;            // first key, first value; rows RS apart
  int64_t page, head;         // strides of a page, of a head inside it
  const int32_t* tables;      // [sequences, max_blocks]
  const int32_t* lens;        // tokens of row b: lens[b] + more
  const int32_t* seq;         // its table, or null: b
  int more, max_blocks, bs;
  short* out;                 // [B, KVH qpg, D]
  float* part_o;              // [B, KVH, NP, qpg, D] (SPLIT)
  float* part_ml;             // [B, KVH, NP, qpg, 2] (SPLIT), m in log2
  int kvh, qpg;
  int part_tokens;            // 0: each row's own share, in steps of 32
  int spread;
  int probe;                  // page by whose readers values are read: below max_blocks,
                              // or -1
  float scale, sink;          // sink: score (log2) of a key without a value
  int has_sink;
};

// RS: elements between a token's rows. PAGE16: pages of 16 tokens and partitions that
// begin on a page, so half a tile lies in one page; else every lane looks its tokens up
// one by one.
template <typename CT, int RS, bool SPLIT, bool PAGE16, int NW>
__global__ __launch_bounds__(NW * WAVE, 3) void decode_attention_kernel(
    const Work<CT> w_) {
  typedef Cache<CT> C;
  const int kvh = w_.kvh, qpg = w_.qpg, bs = w_.bs;
  // Workgroups go round the XCDs in turn: with an even number of sequences all
  // parts of one run on the same few. Where one is far longer than the others,
  // sequences take turns by part.
  const int b = SPLIT && w_.spread ? (blockIdx.x + blockIdx.z) % gridDim.x
                                   : blockIdx.x;
  const int kh = blockIdx.y;
  const int part = SPLIT ? blockIdx.z : 0;
  const int np = SPLIT ? gridDim.z : 1;
  const int64_t group = (int64_t)b * kvh + kh;
  const int tid = threadIdx.x;
  // Whether another row reads the page `probe` too: one of the 64 behind this one, a lane
  // each, is found wherever more than a few share a prefix. Asked for ahead of all else,
  // so that the answer comes little later than the first pages (a page that hangs on the
  // row's length 0.2 us later).
  const int32_t* bt =
      w_.tables + (int64_t)(w_.seq ? w_.seq[b] : b) * w_.max_blocks;
  bool shared = false;
  {
    const int rows = gridDim.x, others = w_.probe < 0 ? 0 : min(rows - 1, WAVE);
    int r = b + 1 + tid % WAVE;
    r -= r >= rows ? rows : 0;
    if (tid % WAVE < others) {
      const int64_t table = w_.seq ? w_.seq[r] : r;
      shared = w_.tables[table * w_.max_blocks + w_.probe] == bt[w_.probe];
    }
  }
  const int seq_len = w_.lens[b] + w_.more;
  const int share = w_.part_tokens ? w_.part_tokens
                                   : ((seq_len + np - 1) / np + 31) / 32 * 32;
  const int t_begin = SPLIT ? part * share : 0;
  // (the last part takes what is left, whatever the longest was said to be)
  const int t_end = SPLIT && part + 1 < np ? min(seq_len, t_begin + share) : seq_len;
  float* const part_o = w_.part_o;
  float* const part_ml = w_.part_ml;

  const int wave = __builtin_amdgcn_readfirstlane(tid / WAVE);
  const int lane = tid % WAVE;
  const int col = lane % 16, g = lane / 16;

  if (SPLIT && t_begin >= seq_len) {
    // empty partition: the combiner skips what has this maximum (others have NEG at
    // least)
    if (tid < qpg) {
      float* ml = part_ml + ((group * np + part) * qpg + tid) * 2;
      ml[0] = -INFINITY;
      ml[1] = 0.f;
    }
    return;
  }

  // column `col` of the scores is a head of the group; the others are zero
  const short* qb = w_.q + b * w_.q_row + kh * qpg * D;
  bf16x8 qf[4];
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    short8 z = {0, 0, 0, 0, 0, 0, 0, 0};
    if (col < qpg) z = *(const short8*)(qb + col * D + C::dim(s, g));
    qf[s] = __builtin_bit_cast(bf16x8, z);
  }
  const float scale_log2 = w_.scale * LOG2E;

  float m, l;                   // of head `col`; l: this lane's tokens only
  float4v acc[8];               // heads 4g + r, channels 8 col + i
#pragma unroll
  for (int i = 0; i < 8; ++i) acc[i] = (float4v){0.f, 0.f, 0.f, 0.f};
  auto begin = [&] {            // one wave's sums have the sink
    const bool sink = w_.has_sink && part == 0 && wave == 0;
    m = sink ? w_.sink : NEG;
    l = sink && g == 0 ? 1.f : 0.f;
  };
  begin();

  const CT* const k_head = w_.k + kh * w_.head;
  const CT* const v_head = w_.v + kh * w_.head;
  uint4v kr[2][C::KL];
  typename C::VReg vr[2][4];
  int page[2];
  // pages of the tile at t0, none past the sequence's last
  auto find = [&](int t0) {
    if constexpr (PAGE16) {
#pragma unroll
      for (int h = 0; h < 2; ++h)
        page[h] = bt[min(t0 / 16 + h, (t_end - 1) / 16)];
    }
  };
  // a token's row; past the end the last one's (only in the lookup form)
  auto row_of = [&](int t) {
    const int tc = min(t, t_end - 1);
    return bt[tc / bs] * w_.page + tc % bs * RS;
  };
  auto fetch_k = [&](int t0) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const CT* row;
      if constexpr (PAGE16)
        row = k_head + page[h] * w_.page + col * RS;
      else
        row = k_head + row_of(t0 + h * 16 + col);
#pragma unroll
      for (int i = 0; i < C::KL; ++i)
        kr[h][i] = *(const uint4v*)((const char*)row + i * 64 + g * 16);
    }
  };
  auto fetch_v = [&](auto past, int t0) {
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const CT* row;
        if constexpr (PAGE16)
          row = v_head + page[h] * w_.page + (g * 4 + j) * RS;
        else
          row = v_head + row_of(t0 + h * 16 + g * 4 + j);
        const auto* const v = (const typename C::VReg*)(row + col * 8);
        if constexpr (decltype(past)::value)
          vr[h][j] = __builtin_nontemporal_load(v);
        else
          vr[h][j] = *v;
      }
  };

  // ENDLESS: infinite values are no part of the lower products; no tile is read
  // ahead, which would take more registers than there are. past: values are read past the
  // caches.
  const int t_first = t_begin + wave * TILE;
  auto walk = [&](auto endless, auto past) {       // !ENDLESS: with the first tile's pages
    constexpr bool ENDLESS = decltype(endless)::value;
    int t0 = t_first;
    if (!ENDLESS && t0 < t_end) {
      fetch_k(t0);
      fetch_v(past, t0);
    }
    for (; t0 < t_end; t0 += NW * TILE) {
      const int next = t0 + NW * TILE;
      const bool more = !ENDLESS && next < t_end;
      if (ENDLESS) {
        find(t0);
        fetch_k(t0);
        fetch_v(past, t0);
      }
      if (more) find(next);
      float4v sc[2];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        sc[h] = (float4v){0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int s = 0; s < 4; ++s)
          sc[h] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(C::key(kr[h], s),
                                                          qf[s], sc[h], 0, 0, 0);
      }
      if (more) fetch_k(next);

      const bool tail = t0 + TILE > t_end;      // wave-uniform
      float mx = NEG;
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          sc[h][r] *= scale_log2;
          if (tail && t0 + h * 16 + g * 4 + r >= t_end) sc[h][r] = -INFINITY;
          mx = fmaxf(mx, sc[h][r]);
        }
      mx = fmaxf(mx, __shfl_xor(mx, 16, WAVE));
      mx = fmaxf(mx, __shfl_xor(mx, 32, WAVE));
      const bool moved = mx > m + SLACK;
      if (__any(moved)) {
        const float to = moved ? mx : m;
        const float alpha = __builtin_amdgcn_exp2f(m - to);
        m = to;
        l *= alpha;
        float4v a;
#pragma unroll
        for (int r = 0; r < 4; ++r) a[r] = __shfl(alpha, g * 4 + r, WAVE);
#pragma unroll
        for (int i = 0; i < 8; ++i) acc[i] *= a;
      }
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          sc[h][r] = __builtin_amdgcn_exp2f(sc[h][r] - m);
          l += sc[h][r];
        }
      if (tail) {      // a page's rows past the sequence may hold anything
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int j = 0; j < 4; ++j)
            if (t0 + h * 16 + g * 4 + j >= t_end)
              vr[h][j] = (typename C::VReg)(0u);
      }
      bf16x8 parts[3];
      split3(sc, parts);
#pragma unroll
      for (int d = 0; d < 8 / C::CH; ++d) {
        uint4v v[C::CH];
        C::values(vr, d, v);
#pragma unroll
        for (int p = 2; p >= 0; --p)
#pragma unroll
          for (int c = 0; c < C::CH; ++c)
            acc[d * C::CH + c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                parts[p],
                __builtin_bit_cast(bf16x8,
                                   ENDLESS && p > 0 ? finite(v[c]) : v[c]),
                acc[d * C::CH + c], 0, 0, 0);
      }
      if (more) fetch_v(past, next);
    }
  };
  if (t_first < t_end) find(t_first);
  if (w_.probe * bs < seq_len && __any(shared))
    walk(std::false_type{}, std::false_type{});
  else
    walk(std::false_type{}, std::true_type{});
  if constexpr (sizeof(CT) == 2) {
    // A probability's lower parts, 0 or negative as often as not, make no number
    // of an infinite value, where the whole one makes infinity: sums that are no
    // number are taken anew, with infinite values in the first product only.
    // (8-bit values have no infinities.)
    float4v all = acc[0];
#pragma unroll
    for (int i = 1; i < 8; ++i) all += acc[i];
    const float sum = all[0] + all[1] + all[2] + all[3];
    if (__any(sum != sum)) {
      begin();
#pragma unroll
      for (int i = 0; i < 8; ++i) acc[i] = (float4v){0.f, 0.f, 0.f, 0.f};
      walk(std::true_type{}, std::false_type{});
    }
  }
  l += __shfl_xor(l, 16, WAVE);
  l += __shfl_xor(l, 32, WAVE);

  // ---- the waves meet ----
  __shared__ float ml_sh[NW][MAX_QPG][2];
  __shared__ __align__(16) float o_sh[NW][MAX_QPG][D];
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int h = g * 4 + r;
    if (h >= qpg) continue;
    float4v lo, hi;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      lo[i] = acc[i][r];
      hi[i] = acc[4 + i][r];
    }
    *(float4v*)&o_sh[wave][h][col * 8] = lo;
    *(float4v*)&o_sh[wave][h][col * 8 + 4] = hi;
  }
  if (g == 0 && col < qpg) {
    ml_sh[wave][col][0] = m;
    ml_sh[wave][col][1] = l;
  }
  __syncthreads();
  for (int i = tid; i < qpg * D; i += NW * WAVE) {
    const int h = i / D, d = i % D;
    float top = NEG;
#pragma unroll
    for (int w = 0; w < NW; ++w) top = fmaxf(top, ml_sh[w][h][0]);
    float s = 0.f, sum = 0.f;
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      const float a = __builtin_amdgcn_exp2f(ml_sh[w][h][0] - top);
      s += a * o_sh[w][h][d];
      sum += a * ml_sh[w][h][1];
    }
    if (SPLIT) {
      part_o[((group * np + part) * qpg + h) * D + d] = s;   // unnormalized
      if (d == 0) {
        float* ml = part_ml + ((group * np + part) * qpg + h) * 2;
        ml[0] = top;
        ml[1] = sum;
      }
    } else {
      w_.out[(group * qpg + h) * D + d] = f32_to_bf16(seq_len > 0 ? s / sum : 0.f);
    }
  }
}

// Merge the NP partitions: one workgroup per (seq, q head), a thread per dim.
// The first wave weighs the partitions (a lane each), then every thread sums
// its column; the loads of a step do not wait for each other.
__global__ __launch_bounds__(D) void decode_combine_kernel(
    const float* __restrict__ part_o,   // [B, KVH, NP, QPG, D]
    const float* __restrict__ part_ml,  // [B, KVH, NP, QPG, 2]
    short* __restrict__ out,            // [B, QH, D]
    int qpg, int np) {
  __shared__ float weight[64];          // np <= 64
  const int64_t group = (int64_t)blockIdx.x * (gridDim.y / qpg) +
                        blockIdx.y / qpg;
  const int h = blockIdx.y % qpg, d = threadIdx.x;
  const int64_t first = group * np * qpg + h;
  if (d < WAVE) {
    const float* ml = part_ml + (first + (int64_t)min(d, np - 1) * qpg) * 2;
    const float m = d < np ? ml[0] : -INFINITY;
    const bool empty = m == -INFINITY;
    const float top = wave_reduce_max(m);
    const float w = empty ? 0.f : __builtin_amdgcn_exp2f(m - top);
    const float sum = wave_reduce_sum(empty ? 0.f : w * ml[1]);   // NaN stays NaN
    weight[d] = empty ? 0.f : w / sum;
  }
  __syncthreads();
  float o = 0.f;
#pragma unroll 8
  for (int p = 0; p < np; ++p) {
    const float x = part_o[(first + (int64_t)p * qpg) * D + d];
    const float w = weight[p];
    o += w == 0.f ? 0.f : w * x;        // an empty partition wrote no sums
  }
  out[((int64_t)blockIdx.x * gridDim.y + blockIdx.y) * D + d] = f32_to_bf16(o);
}

// One launch over n rows, and another where they are in parts.
template <bool SPLIT, int RS, typename CT>
hipError_t attend(const Work<CT>& w, int n, int parts, int waves,
                  hipStream_t stream) {
  const dim3 grid(n, w.kvh, parts);
#define GO(PAGE16, NW)                                                        \
  hipLaunchKernelGGL((decode_attention_kernel<CT, RS, SPLIT, PAGE16, NW>),    \
                     grid, dim3(NW * WAVE), 0, stream, w)
#define GO_NW(PAGE16)                                                         \
  do {                                                                        \
    if (waves == 8) GO(PAGE16, 8); else GO(PAGE16, 4);                        \
  } while (0)
  if (w.bs == 16 && w.part_tokens % 16 == 0) GO_NW(true);
  else GO_NW(false);
#undef GO_NW
#undef GO
  if (SPLIT)
    hipLaunchKernelGGL(decode_combine_kernel, dim3(n, w.kvh * w.qpg), dim3(D),
                       0, stream, w.part_o, w.part_ml, w.out, w.qpg, parts);
  HIP_CHECK_LAST();
  return hipSuccess;
}

}  // namespace decode
