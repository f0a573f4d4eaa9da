// flash_prefill_bf16.hip — prefill attention of bf16 caches: tiles of keys and
// values go through registers into LDS, two of them there, a third on its way. The
// attention of a tile is flash_core.h's; the tiles' loads and LDS writes stand
// between its matrix instructions (in a row they hold a wave up for 1200 cycles of
// 4900 per 64 keys). Loads straight to LDS are not used: the compiler waits for all
// of them ahead of each transposing read.
//
// A workgroup has 4 waves and one of two shapes:
//   rows   128 query rows, 32 per wave; all waves share tiles of 64 keys, with
//          one barrier per tile: it stands between the last read of a tile and
//          the writes of the one after the next.
//   keys   32 query rows; every wave takes each fourth tile of 32 keys through LDS
//          of its own, without barriers, and the waves' results meet in LDS at
//          the end. Four times the workgroups, half the serial chain, one
//          workgroup per compute unit (132 KB of LDS).
// Where the workgroups of the first shape leave compute units idle, one of the
// two takes the call by its work (see prefill_shape in ops/dispatch.py), and
// probabilities keep 17 bits in both: the matrix cores have the time, and a
// prompt's last tokens come out as decoding them would.
// Key heads run fastest over the grid: with 8 of them each XCD's L2 holds the
// keys and values of one. Tiles run from the last to the first: under the
// causal mask the last of a sequence has the most keys.
//
// What bounds it: per 64 keys the matrix cores work 1024 cycles for each of a
// SIMD's two waves, of 4450 that a pass takes; the rest is the vector work of both
// (650 to 850 cycles each), waits at the barrier, and the clock, which falls to 1.7
// GHz over long prompts.
// Measured (groups of 4, 8 key heads, alone; before: operands of K waited for one
// by one, tiles of 32 keys in a ring of loads to LDS): one prompt of 7900 tokens
// 547 us, 934 TFLOP/s (652); 8 of 1000 110 us (127). By keys / by rows with 17 bits
// (with 8): 150 tokens behind 1000 17 / 35 us (30; before 21 / 45); 500 behind 1000
// 40 / 47 (38; 49 / 59); 600 behind 4000 139 / 127 (102; 183 / 168); 12 prompts of
// 20 12 / 7 (7).
//
// 8-bit caches take the kernel in flash_prefill.hip, which widens them; the
// launcher in ops.hip picks per cache dtype.
#include "flash_core.h"

#include <type_traits>

namespace {

using namespace flash;

constexpr int D = 128;
constexpr int tile_of(bool keys) { return keys ? 32 : 64; }   // tokens
constexpr int NW = 4;
constexpr int QROWS = 32;
constexpr int BT_CAP = 1024;  // staged block-table entries (16K-token ctx)

__device__ __forceinline__ void raw_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

constexpr int lds_bytes(bool keys) {       // two tiles of keys and values
  return BT_CAP * 4 + 4 * tile_of(keys) * D * 2 * (keys ? NW : 1);
}

// FINE: see attend. SHIFT: block size 1 << shift; else any
template <int QPG, bool KEYS, bool FINE, bool SHIFT>
__global__ __launch_bounds__(NW * WAVE, 2)
void flash_prefill_bf16_kernel(
    const short* __restrict__ q, const short* __restrict__ k_cache,
    const short* __restrict__ v_cache,
    const int32_t* __restrict__ block_tables,
    const int32_t* __restrict__ seq_meta, const int32_t* __restrict__ tiles,
    short* __restrict__ out, int n_tiles, int kvh, int bs, int shift,
    int max_blocks, float scale) {
  constexpr int TILE = tile_of(KEYS), TILE_BYTES = TILE * D * 2;
  const int kh = blockIdx.x % kvh, at_tile = blockIdx.x / kvh;
  const int tile = n_tiles - 1 - at_tile / (KEYS ? NW : 1);
  const int sub = KEYS ? at_tile % NW : 0;
  const int seq = tiles[2 * tile];
  const int vrow0 = tiles[2 * tile + 1] + sub * QROWS;
  const int seq_start = seq_meta[3 * seq];
  const int chunk = seq_meta[3 * seq + 1];
  const int prior = seq_meta[3 * seq + 2];
  const int ctx = prior + chunk, rows = chunk * QPG;
  const int n_q_heads = kvh * QPG;
  if (KEYS && vrow0 >= rows) return;            // workgroup-uniform

  extern __shared__ __align__(16) char lds_raw[];
  int32_t* bt_lds = (int32_t*)lds_raw;

  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid / WAVE);
  const int lane = tid % WAVE;
  const int qcol = lane & 31;
  const int hi = lane >> 5;
  // a ring of this wave's, or of all waves'
  char* ring = lds_raw + BT_CAP * 4 +
               (KEYS ? wave * 4 * TILE_BYTES : 0);

  // rows past the last repeat it and are not stored
  const int w0 = vrow0 + (KEYS ? 0 : wave * QROWS);
  const int vrow = w0 + qcol;
  const bool active = vrow < rows;
  const int p = (active ? vrow : rows - 1) / QPG;
  const int qh = kh * QPG + (active ? vrow : rows - 1) % QPG;
  const int64_t q_row = (int64_t)(seq_start + p) * n_q_heads + qh;

  const int last_wg = (min(vrow0 + (KEYS ? QROWS : NW * QROWS), rows) - 1) / QPG;
  const int first_w = min(w0, rows - 1) / QPG;
  const int last_w = (min(w0 + QROWS, rows) - 1) / QPG;
  const int kv_end = prior + last_wg + 1;       // keys that a row here may see
  const int kv_end_w = w0 < rows ? prior + last_w + 1 : 0;
  const int n_kv_tiles = (kv_end + TILE - 1) / TILE;

  bf16x8 qf[D / 16];
  const unsigned int flip = scale < 0.f ? 0x80008000u : 0u;
#pragma unroll
  for (int kk = 0; kk < D / 16; ++kk) {
    const uint4v v = *(const uint4v*)(q + q_row * D + kk * 16 + hi * 8);
    qf[kk] = __builtin_bit_cast(bf16x8, v ^ flip);
  }
  const float scale_log2 = log2_scale(scale);
  const int n_bt =
      min(max_blocks, (SHIFT ? kv_end - 1 >> shift : (kv_end - 1) / bs) + 1);
  for (int i = tid; i < n_bt; i += NW * WAVE)
    bt_lds[i] = block_tables[(int64_t)seq * max_blocks + i];
  __syncthreads();

  // A tile goes through registers, one ahead of the two in LDS. A wave brings 4
  // rows per load: all of one page where pages are multiples of 4, whose place
  // lane g works out for load g. Rows past the last key that is seen repeat it: no
  // garbage bf16.
  constexpr int P = TILE / (KEYS ? 4 : 4 * NW);        // loads of a wave
  short8 kn[P], vn[P];
  uint64_t place = 0;
  const int lrow = lane / 16, last = kv_end - 1;
  const uint32_t page_bytes = (uint32_t)kvh * bs * D * 2;
  const char* const k_head = (const char*)(k_cache + (int64_t)kh * bs * D);
  const char* const v_head = (const char*)(v_cache + (int64_t)kh * bs * D);
  auto token = [&](int n, int g) {
    return n * TILE + (KEYS ? g * 4 : g * 4 * NW + wave * 4);
  };
  auto look = [&](int n) {
    if constexpr (SHIFT) {
      const int t = min(token(n, lane % P), last & ~3);
      place = (uint64_t)(uint32_t)bt_lds[t >> shift] * page_bytes +
              (uint32_t)(t & (bs - 1)) * (D * 2);
    }
  };
  auto fetch = [&](int n, int g) {
    const int t0 = token(n, g);
    uint64_t at;
    uint32_t off;
    if constexpr (SHIFT) {
      at = (uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(place >> 32), g)
               << 32 |
           (uint32_t)__builtin_amdgcn_readlane((int)place, g);
      off = (min(lrow, max(last - t0, last & 3)) * D + lane % 16 * 8) * 2;
    } else {
      const int t = min(t0 + lrow, last), pg = t / bs;
      at = ((uint64_t)(uint32_t)bt_lds[pg] * kvh * bs + (t - pg * bs)) * (D * 2);
      off = lane % 16 * 16;
    }
    // As one vector address where the matrix instructions take longer than the rest:
    // 150 rows behind 1000 19.0 us with a scalar one, so 17.5, 600 behind 4000 131 and
    // 126; else it costs more than it saves (one prompt of 7000 rows 445 and 461).
    if constexpr (FINE) {
      at += off;
      off = 0;
    }
    kn[g] = *(const short8*)(k_head + at + off);
    vn[g] = *(const short8*)(v_head + at + off);
  };
  constexpr int GAP = (KEYS ? 4 : 4 * NW) * 256;       // between its loads' rows
  const int row0 = (KEYS ? 0 : wave * 4) + lrow;
  auto put = [&](int buf, int g) {
    // (16 rows on, the swizzle is the same)
    const int row = row0 + (KEYS ? g % 4 * 4 : 0);
    char* to = ring + buf * 2 * TILE_BYTES + row0 * 256 + g * GAP +
               ((lane % 16 * 16) ^ swizzle(row));
    *(short8*)to = kn[g];
    *(short8*)(to + TILE_BYTES) = vn[g];
  };

  Softmax st;
  f32x16 acc[D / 32];
#pragma unroll
  for (int t = 0; t < D / 32; ++t) acc[t] = (f32x16)(0.f);

  // the lane's share of addresses in a tile
  const int i16 = lane % 16;
  const int k_row = qcol * 256, k_swz = swizzle(qcol);
  const int v_col = (16 * ((lane & 31) >> 4) + (i16 % 4) * 4) * 2;
  // Tile n from `buf`, while the next one of this wave leaves the registers and
  // the one after it comes in.
  auto step = [&](int n, int next2, int next3, auto buf_) {
    constexpr int buf = decltype(buf_)::value;
    if constexpr (!KEYS) raw_barrier();   // it is there; all are done with n - 1
    if (!KEYS && n * TILE >= kv_end_w) {  // beyond what this wave's rows see
#pragma unroll
      for (int g = 0; g < P; ++g) {
        put(buf ^ 1, g);
        fetch(next2, g);
      }
      look(next3);
      return;
    }
    const int tile0 = n * TILE;
    const char* kb = ring + buf * 2 * TILE_BYTES;
    const char* vb = kb + TILE_BYTES;
    attend<D / 16, D / 32, TILE / 32, FINE>(
        [&](int u, int kk) {
          return *(const bf16x8*)(kb + u * 32 * 256 + k_row +
                                  ((kk * 32 + hi * 16) ^ k_swz));
        },
        [&](int u, int row, int t) {
          return vb + (u * 32 + row) * 256 + ((t * 64 + v_col) ^ swizzle(row));
        },
        qf, scale_log2, tile0 + TILE - 1 <= prior + first_w, 0,
        prior + p - tile0, st, acc,
        [&](int i) {
          constexpr int N = D / 16 * TILE / 32;
          if (i * P % N == 0) {
            put(buf ^ 1, i * P / N);
            fetch(next2, i * P / N);
          }
          if (i == N - 1) look(next3);
        });
  };
  // this wave's tiles: every NWth by keys
  constexpr int EACH = KEYS ? NW : 1;
  const int n0 = KEYS ? wave : 0;
  if (n0 < n_kv_tiles) {
    look(n0);
#pragma unroll
    for (int g = 0; g < P; ++g) fetch(n0, g);
#pragma unroll
    for (int g = 0; g < P; ++g) put(0, g);
    if (n0 + EACH < n_kv_tiles) {
      look(n0 + EACH);
#pragma unroll
      for (int g = 0; g < P; ++g) fetch(n0 + EACH, g);
      look(n0 + 2 * EACH);
    }
    for (int n = n0; n < n_kv_tiles; n += 2 * EACH) {
      step(n, n + 2 * EACH, n + 3 * EACH, std::integral_constant<int, 0>{});
      if (n + EACH < n_kv_tiles)
        step(n + EACH, n + 3 * EACH, n + 4 * EACH,
             std::integral_constant<int, 1>{});
    }
  }
  st.l = st.join();

  if constexpr (KEYS) {
    // the waves meet: wave w sums channels 32 w .. of all four
    float* o_sh = (float*)(lds_raw + BT_CAP * 4);   // [wave][t][r][lane]
    float2* ml_sh = (float2*)lds_raw;               // [wave][lane]
    __syncthreads();                                // rings and table are done
#pragma unroll
    for (int t = 0; t < D / 32; ++t)
#pragma unroll
      for (int r = 0; r < 16; ++r)
        o_sh[((wave * (D / 32) + t) * 16 + r) * WAVE + lane] = acc[t][r];
    ml_sh[wave * WAVE + lane] = make_float2(st.m, st.l);
    __syncthreads();
    float m = NEG, l = 0.f;
#pragma unroll
    for (int w = 0; w < NW; ++w) m = fmaxf(m, ml_sh[w * WAVE + lane].x);
    f32x16 o = (f32x16)(0.f);
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      const float2 ml = ml_sh[w * WAVE + lane];
      const float a = __builtin_amdgcn_exp2f(ml.x - m);
      l += a * ml.y;
#pragma unroll
      for (int r = 0; r < 16; ++r)
        o[r] += a * o_sh[((w * (D / 32) + wave) * 16 + r) * WAVE + lane];
    }
    if (!active) return;                            // it sees a key: l > 0 or no number
    const float inv = 1.f / l;
    short* dst = out + q_row * D + wave * 32 + 4 * hi;
#pragma unroll
    for (int g = 0; g < 4; ++g)
      *(uint2*)(dst + 8 * g) = make_uint2(
          pack2(o[4 * g] * inv, o[4 * g + 1] * inv),
          pack2(o[4 * g + 2] * inv, o[4 * g + 3] * inv));
  } else if (active) {
    const float inv = 1.f / st.l;
#pragma unroll
    for (int t = 0; t < D / 32; ++t)
#pragma unroll
      for (int g = 0; g < 4; ++g)
        *(uint2*)(out + q_row * D + t * 32 + 8 * g + 4 * hi) = make_uint2(
            pack2(acc[t][4 * g] * inv, acc[t][4 * g + 1] * inv),
            pack2(acc[t][4 * g + 2] * inv, acc[t][4 * g + 3] * inv));
  }
}

template <int QPG, bool KEYS, bool FINE, bool SHIFT>
hipError_t go(const void* q, const void* k_cache, const void* v_cache,
              const int32_t* block_tables, const int32_t* seq_meta,
              const int32_t* tiles, void* out, int n_tiles, int kvh, int bs,
              int shift, int max_blocks, float scale, hipStream_t stream) {
  auto fn = flash_prefill_bf16_kernel<QPG, KEYS, FINE, SHIFT>;
  hipError_t e = hipFuncSetAttribute(
      (const void*)fn, hipFuncAttributeMaxDynamicSharedMemorySize,
      lds_bytes(KEYS));
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(fn, dim3((uint32_t)kvh * n_tiles * (KEYS ? NW : 1)),
                     dim3(NW * WAVE), lds_bytes(KEYS), stream, (const short*)q,
                     (const short*)k_cache, (const short*)v_cache,
                     block_tables, seq_meta, tiles, (short*)out, n_tiles, kvh,
                     bs, shift, max_blocks, scale);
  HIP_CHECK_LAST();
  return hipSuccess;
}

}  // namespace

extern "C" {

// shape: 0 by rows, 1 by keys, 2 by rows with probabilities of 17 bits; below
// 0, for callers that do not know the lengths: rows if these fill the chip,
// else keys in one round of workgroups, or in two where prompts are long enough
// to make up for the second (300 tokens behind 300 20 us by keys, 22 by rows; 4
// x 100 13 and 10).
hipError_t lds_flash_prefill_bf16(
    const void* q, const void* k_cache, const void* v_cache,
    const int32_t* block_tables, const int32_t* seq_meta,
    const int32_t* tiles, void* out, int n_tiles, int n_q_heads, int kvh,
    int bs, int head_dim, int max_blocks, float scale, int shape, int n_tokens,
    int n_seqs, hipStream_t stream) {
  if (n_tiles == 0) return hipSuccess;
  if (head_dim != D || max_blocks > BT_CAP || bs < 1 ||
      (int64_t)n_tiles * kvh * NW > 0x7fffffff)
    return hipErrorInvalidValue;
  const int qpg = n_q_heads / kvh;
  const int64_t groups = (int64_t)n_tiles * kvh;
  if (shape < 0)
    shape = groups >= 256  ? 0
            : groups <= 64 ? 1
            : groups <= 128 && n_tokens / 256 >= n_seqs ? 1
                                                        : 2;
  int shift = 0;
  while (1 << shift < bs && shift < 20) ++shift;
  const bool pow2 =
      1 << shift == bs && bs >= 4 && (int64_t)kvh * bs * D * 2 < 1ll << 32;
#define GO(QPG, KEYS, FINE, SHIFT)                                           \
  return go<QPG, KEYS, FINE, SHIFT>(q, k_cache, v_cache, block_tables, seq_meta,   \
                              tiles, out, n_tiles, kvh, bs, shift,           \
                              max_blocks, scale, stream)
#define GO_Q(QPG)                                                            \
  do {                                                                       \
    if (shape == 1) {                                                        \
      if (pow2) GO(QPG, true, true, true); else GO(QPG, true, true, false);  \
    } else if (shape == 2) {                                                 \
      if (pow2) GO(QPG, false, true, true);                                  \
      else GO(QPG, false, true, false);                                      \
    } else {                                                                 \
      if (pow2) GO(QPG, false, false, true);                                 \
      else GO(QPG, false, false, false);                                     \
    }                                                                        \
  } while (0)
  switch (qpg) {
    case 1: GO_Q(1);
    case 2: GO_Q(2);
    case 4: GO_Q(4);
    case 8: GO_Q(8);
    default: return hipErrorInvalidValue;
  }
#undef GO_Q
#undef GO
}

}  // extern "C"
