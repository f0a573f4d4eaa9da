// flash_prefill.hip — fused causal varlen GQA prefill attention over the
// paged KV pool, MFMA-tiled for gfx950 (CDNA4).
//
// Replaces the composed einsum+softmax prefill path (materialized S matrix,
// ~6 HBM passes) with a flash-style kernel: per Q-tile, iterate KV tiles
// computing QK^T -> online softmax -> P.V entirely on matrix cores
// (v_mfma_f32_32x32x16_bf16), S never leaving registers.
//
// The attention of a tile is flash_core.h's: S^T = K.Q^T, so that a lane owns
// one query row and the online softmax is in-lane work. This kernel stages
// through registers, converting fp8 to bf16 on the way, and also takes bf16
// pools of contexts that flash_prefill_bf16.hip's table does not hold.
//
// Work decomposition:
//   grid = row tiles (128 "virtual rows" = (position, q-head-in-group)
//          pairs, v = p*QPG + g), last first, times kv heads (fastest)
//   workgroup = 4 waves; wave w owns v-rows [vrow0+32w, vrow0+32w+32)
//   KV loop: 64-token tiles in LDS (XOR-swizzled rows), two of them; a third is on
//            its way in registers, and its loads and LDS writes stand between the
//            matrix instructions. Where the rows of a wave's load lie in one page
//            (WHOLE) the page's address is scalar work.
//
// GQA: q-heads of one group share the kv_head's K/V tiles; causal masking
// is per-lane compares (kv <= prior + p), no divergence.
//
// Bound by vector work, of the softmax and of widening and moving tiles. 8-bit cache,
// groups of 4, 8 key heads; before: one tile in LDS, a division and 64-bit products per
// lane and row: one prompt of 7000 tokens 492 us (586), 8 of 1000 133 us (155), 4 of 1000
// behind 1000 164 us (200), 150 behind 1000 44 us (55).
#include "flash_core.h"

#include <type_traits>

namespace {

using namespace flash;

constexpr int D = 128;       // head_dim
constexpr int KVBLK = 64;    // tokens per KV tile (2 mfma sub-tiles)
constexpr int NW = 4;        // waves per workgroup
constexpr int QROWS = 32;    // q virtual-rows per wave

// 8 cache elements as they are, and as bf16
template <typename CT> struct Piece;
template <> struct Piece<short> {
  typedef short8 Raw;
  static __device__ __forceinline__ short8 wide(Raw r) { return r; }
};
template <> struct Piece<unsigned char> {
  typedef uint2 Raw;
  // e4m3 values are bf16 values: the upper halves of the floats
  static __device__ __forceinline__ short8 wide(Raw r) {
    float f[8];
    load_kv8((const unsigned char*)&r, f);
    uint4v w;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint32_t a = __builtin_bit_cast(uint32_t, f[2 * i]);
      const uint32_t b = __builtin_bit_cast(uint32_t, f[2 * i + 1]);
      w[i] = __builtin_amdgcn_perm(b, a, 0x07060302);
    }
    return __builtin_bit_cast(short8, w);
  }
};

template <int QPG, typename CT, bool WHOLE>
__global__ __launch_bounds__(NW * WAVE, 2) void flash_prefill_kernel(
    const short* __restrict__ q,        // [T, QH, D]
    const CT* __restrict__ k_cache,     // [NB, KVH, BS, D] bf16|fp8
    const CT* __restrict__ v_cache,     // [NB, KVH, BS, D] bf16|fp8
    const int32_t* __restrict__ block_tables,  // [S, max_blocks]
    const int32_t* __restrict__ seq_meta,      // [S, 3] start, chunk, prior
    const int32_t* __restrict__ tiles,         // [n_tiles, 2] seq, vrow0
    short* __restrict__ out,                   // [T, QH, D]
    int kvh, int bs, int shift, int max_blocks, float scale) {
  const int kh = blockIdx.x % kvh;
  const int tile = (gridDim.x - 1 - blockIdx.x) / kvh;
  const int seq = tiles[2 * tile];
  const int vrow0 = tiles[2 * tile + 1];
  const int seq_start = seq_meta[3 * seq];
  const int chunk = seq_meta[3 * seq + 1];
  const int prior = seq_meta[3 * seq + 2];
  const int rows = chunk * QPG;
  const int n_q_heads = kvh * QPG;
  const int32_t* bt = block_tables + (int64_t)seq * max_blocks;

  __shared__ __align__(16) short lds[2][2][KVBLK * D];   // keys, values: swizzled rows
  static_assert(KVBLK * 16 % (NW * WAVE) == 0, "staging divides evenly");

  const int tid = threadIdx.x;
  const int wave = tid / WAVE;
  const int lane = tid % WAVE;
  const int qcol = lane & 31;
  const int hi = lane >> 5;

  // this lane's query row; rows past the last repeat it and are not stored
  const int w0 = vrow0 + wave * QROWS, vrow = w0 + qcol;
  const bool active = vrow < rows;
  const int p = (active ? vrow : rows - 1) / QPG;
  const int qh = kh * QPG + (active ? vrow : rows - 1) % QPG;
  const int64_t q_row = (int64_t)(seq_start + p) * n_q_heads + qh;

  // Q^T B-fragments: qf[kk] covers head dims [16kk + 8hi, 16kk + 8hi+8)
  bf16x8 qf[D / 16];
  const unsigned int flip = scale < 0.f ? 0x80008000u : 0u;
#pragma unroll
  for (int kk = 0; kk < D / 16; ++kk) {
    const uint4v v = *(const uint4v*)(q + q_row * D + kk * 16 + hi * 8);
    qf[kk] = __builtin_bit_cast(bf16x8, v ^ flip);
  }
  const float scale_log2 = log2_scale(scale);

  Softmax st;
  f32x16 acc[D / 32];
#pragma unroll
  for (int t = 0; t < D / 32; ++t) acc[t] = (f32x16)(0.f);

  // causal KV extents
  const int last_wg = (min(vrow0 + NW * QROWS, rows) - 1) / QPG;
  const int first_w = min(w0, rows - 1) / QPG;
  const int last_w = (min(w0 + QROWS, rows) - 1) / QPG;
  const int kv_end_wg = prior + last_wg + 1;
  const int kv_end_w = w0 < rows ? prior + last_w + 1 : 0;

  // A tile goes through registers: rows past the last key that is seen repeat it (they
  // are masked).
  typedef typename Piece<CT>::Raw Raw;
  constexpr int REPS = KVBLK * 16 / (NW * WAVE), PER = WAVE / 16;
  const int last = kv_end_wg - 1;
  const int first_row = __builtin_amdgcn_readfirstlane(wave) * PER;
  Raw kn[REPS], vn[REPS];
  int pages[WHOLE ? 1 : REPS];   // of a tile; WHOLE: those from its first key's on, by lane
  auto row_of = [&](int tile0, int r) {
    return min(tile0 + r * NW * PER + first_row + lane / 16, last);
  };
  auto find = [&](int tile0) {
    if constexpr (WHOLE) {
      pages[0] = bt[min((tile0 >> shift) + lane, last >> shift)];
    } else {
#pragma unroll
      for (int r = 0; r < REPS; ++r) pages[r] = bt[row_of(tile0, r) / bs];
    }
  };
  // load i of the keys, then of the values
  auto fetch = [&](int tile0, int i) {
    const int r = i % REPS, t = row_of(tile0, r), c = lane % 16 * 8;
    const CT* from = i < REPS ? k_cache : v_cache;
    if constexpr (WHOLE) {
      const int first = min(tile0 + r * NW * PER + first_row, last);
      const uint32_t page = __builtin_amdgcn_readlane(
          pages[0], max((first >> shift) - (tile0 >> shift), 0));
      from += ((uint64_t)page * kvh + kh) * (bs * D) +
              (uint32_t)((t & (bs - 1)) * D + c);
    } else {
      from += (((int64_t)pages[WHOLE ? 0 : r] * kvh + kh) * bs + t % bs) * D + c;
    }
    (i < REPS ? kn : vn)[r] = *(const Raw*)from;
  };
  auto put = [&](int buf, int i) {
    const int r = i % REPS, row = r * NW * PER + wave * PER + lane / 16;
    const int at = row * 256 + (lane % 16 * 16 ^ swizzle(row));
    *(short8*)((char*)lds[buf][i / REPS] + at) =
        Piece<CT>::wide((i < REPS ? kn : vn)[r]);
  };
  const int i16 = lane % 16;
  const int v_col = (16 * ((lane & 31) >> 4) + (i16 % 4) * 4) * 2;
  find(0);
#pragma unroll
  for (int i = 0; i < 2 * REPS; ++i) fetch(0, i);
#pragma unroll
  for (int i = 0; i < 2 * REPS; ++i) put(0, i);
  if (KVBLK < kv_end_wg) {
    find(KVBLK);
#pragma unroll
    for (int i = 0; i < 2 * REPS; ++i) fetch(KVBLK, i);
    find(2 * KVBLK);
  }
  auto step = [&](int tile0, auto buf_) {
    constexpr int buf = decltype(buf_)::value;
    lds_barrier();
    // The last tile's values past the end count as 0: bf16 ones may be infinite, and a
    // probability of 0 makes no 0 of that. (As they are put: 225 -> 234 us, 4000 rows.)
    if (sizeof(CT) == 2 && tile0 + KVBLK > kv_end_wg) {
      const int n = kv_end_wg - tile0;
      for (int i = n * 16 + tid; i < KVBLK * 16; i += NW * WAVE)
        *(short8*)((char*)lds[buf][1] + i * 16) = (short8){0, 0, 0, 0, 0, 0, 0, 0};
      lds_barrier();
    }
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      const int sub0 = tile0 + 32 * half;
      auto next = [&](int i) {
        put(buf ^ 1, half * REPS + i);
        fetch(tile0 + 2 * KVBLK, half * REPS + i);
      };
      if (sub0 >= kv_end_w) {               // beyond this wave's horizon
#pragma unroll
        for (int i = 0; i < REPS; ++i) next(i);
        continue;
      }
      const char* kb = (const char*)lds[buf][0] + 32 * half * 256;
      const char* vb = (const char*)lds[buf][1] + 32 * half * 256;
      attend<D / 16, D / 32, 1, false>(
          [&](int, int kk) {
            return *(const bf16x8*)(kb + qcol * 256 +
                                    ((kk * 32 + hi * 16) ^ swizzle(qcol)));
          },
          [&](int, int row, int t) {
            return vb + row * 256 + ((t * 64 + v_col) ^ swizzle(row));
          },
          qf, scale_log2, sub0 + 31 <= prior + first_w, 0, prior + p - sub0,
          st, acc, [&](int m) {
            static_assert(D / 16 == 2 * REPS, "");
            if (m % 2 == 0) next(m / 2);
          });
    }
    find(tile0 + 3 * KVBLK);
  };
  for (int tile0 = 0; tile0 < kv_end_wg; tile0 += 2 * KVBLK) {
    step(tile0, std::integral_constant<int, 0>{});
    if (tile0 + KVBLK < kv_end_wg)
      step(tile0 + KVBLK, std::integral_constant<int, 1>{});
  }
  st.l = st.join();

  // ---- epilogue: out[seq_start+p][qh][dim] = acc / l ----
  if (active) {                             // it sees a key: l is above 0 or no number
    const float inv = 1.f / st.l;
#pragma unroll
    for (int t = 0; t < D / 32; ++t)
#pragma unroll
      for (int g = 0; g < 4; ++g)           // reg quads: 4 dims in order
        *(uint2*)(out + q_row * D + t * 32 + 8 * g + 4 * hi) = make_uint2(
            pack2(acc[t][4 * g] * inv, acc[t][4 * g + 1] * inv),
            pack2(acc[t][4 * g + 2] * inv, acc[t][4 * g + 3] * inv));
  }
}

}  // namespace

extern "C" {

hipError_t lds_flash_prefill(const void* q, const void* k_cache,
                             const void* v_cache,
                             const int32_t* block_tables,
                             const int32_t* seq_meta, const int32_t* tiles,
                             void* out, int n_tiles, int n_q_heads, int kvh,
                             int bs, int head_dim, int max_blocks, int kv_fp8,
                             float scale, hipStream_t stream) {
  if (n_tiles == 0) return hipSuccess;
  if (head_dim != D || (int64_t)n_tiles * kvh > 0x7fffffff)
    return hipErrorInvalidValue;
  const int qpg = n_q_heads / kvh;
  dim3 grid((uint32_t)n_tiles * kvh), block(NW * WAVE);
  const int shift = bs & bs - 1 ? -1 : __builtin_ctz(bs);
#define LAUNCH_ROWS(QPG, CT, WHOLE)                                           \
  hipLaunchKernelGGL((flash_prefill_kernel<QPG, CT, WHOLE>), grid, block, 0,  \
                     stream,                                                  \
                     (const short*)q, (const CT*)k_cache,                     \
                     (const CT*)v_cache, block_tables, seq_meta, tiles,       \
                     (short*)out, kvh, bs, shift, max_blocks, scale)
  // a wave's load has 4 rows
#define LAUNCH_CT(QPG, CT)                                                    \
  do {                                                                        \
    if (shift >= 2) LAUNCH_ROWS(QPG, CT, true);                               \
    else LAUNCH_ROWS(QPG, CT, false);                                         \
  } while (0)
#define LAUNCH(QPG)                                                           \
  do {                                                                        \
    if (kv_fp8) LAUNCH_CT(QPG, unsigned char);                                \
    else LAUNCH_CT(QPG, short);                                               \
  } while (0)
  switch (qpg) {
    case 1: LAUNCH(1); break;
    case 2: LAUNCH(2); break;
    case 4: LAUNCH(4); break;
    case 8: LAUNCH(8); break;
    default: return hipErrorInvalidValue;
  }
#undef LAUNCH
#undef LAUNCH_CT
#undef LAUNCH_ROWS
  HIP_CHECK_LAST();
  return hipSuccess;
}

}  // extern "C"
