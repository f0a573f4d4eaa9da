// flash_prefill_glds.hip — the bf16-KV variant of the fused MFMA prefill
// attention with a glds staging pipeline: K/V tiles are DMA'd straight to LDS
// (`global_load_lds`) into a ring, ahead of their use, with COUNTED
// `s_waitcnt vmcnt(N)` (hipcc drains glds at any ordinary in-loop global load,
// so the block table is staged into LDS up front and the hot loop touches
// global memory ONLY through glds). The LDS image stays lane-linear (a glds
// constraint); the XOR bank swizzle is applied by permuting the per-lane
// SOURCE addresses. The attention of a tile is flash_core.h's.
//
// A workgroup has 4 waves and one of two shapes:
//   rows   128 query rows, 32 per wave; all waves share tiles of 32 keys in a
//          3-deep ring, two tiles ahead. Order: [counted vmcnt][raw barrier]
//          [compute tile n][issue tile n+2] — barrier n separates every wave's
//          last read of buffer (n-1)%3 from its rewrite for tile n+2.
//   keys   32 query rows; every wave takes each fourth tile of keys through a
//          2-deep ring of its own, without barriers, and the waves' results
//          meet in LDS at the end. Four times the workgroups, half the serial
//          chain, one workgroup per compute unit (132 KB of LDS).
// Where the workgroups of the first shape leave compute units idle, one of the
// two takes the call by its work (see prefill_shape in ops/dispatch.py), and
// probabilities keep 17 bits in both: the matrix cores have the time, and a
// prompt's last tokens come out as decoding them would.
// Key heads run fastest over the grid: with 8 of them each XCD's L2 holds the
// keys and values of one. Tiles run from the last to the first: under the
// causal mask the last of a sequence has the most keys.
//
// Measured (groups of 4, 8 key heads, alone; before: masks, packing and
// rescaling of every tile on the vector units): one prompt of 7900 tokens 650
// us, 785 TFLOP/s (before 1170); 8 of 1000 135 us (265); in a pass of layers one
// of 8190 takes 812, 676 TFLOP/s. By keys / by rows with 17 bits (with 8): 150
// tokens behind 1000 24 / 48 us (44; before 61); 500 behind 1000 52 / 66 (57;
// 79); 600 behind 4000 195 / 175 (159; 235); 12 prompts of 20 13 / 7 (6; 7).
//
// fp8 KV cannot ride glds (raw byte copy, no conversion point), so the fp8
// path keeps the convert-on-stage kernel in flash_prefill.hip; the launcher in
// ops.hip picks per cache dtype.
#include "flash_core.h"

namespace {

using namespace flash;

constexpr int D = 128;
constexpr int KVBLK = 32;    // tokens per KV tile (ring granularity)
constexpr int NW = 4;
constexpr int QROWS = 32;
constexpr int BT_CAP = 1024;  // staged block-table entries (16K-token ctx)

constexpr int TILE_BYTES = KVBLK * D * 2;        // of K, and of V
constexpr int RING_ROWS = 3, RING_KEYS = 2;      // tiles per ring

__device__ __forceinline__ void raw_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

constexpr int lds_bytes(bool keys) {
  return BT_CAP * 4 + 2 * TILE_BYTES * (keys ? RING_KEYS * NW : RING_ROWS);
}

// FINE: see attend32. SHIFT: block size 1 << shift; else any
template <int QPG, bool KEYS, bool FINE, bool SHIFT>
__global__ __launch_bounds__(NW * WAVE, KEYS ? 1 : 2)
void flash_prefill_glds_kernel(
    const short* __restrict__ q, const short* __restrict__ k_cache,
    const short* __restrict__ v_cache,
    const int32_t* __restrict__ block_tables,
    const int32_t* __restrict__ seq_meta, const int32_t* __restrict__ tiles,
    short* __restrict__ out, int n_tiles, int kvh, int bs, int shift,
    int max_blocks, float scale) {
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

  // ONE shared object (a second __shared__ symbol makes hipcc emit
  // vmcnt(0) before every ds_read)
  extern __shared__ __align__(16) char lds_raw[];
  int32_t* bt_lds = (int32_t*)lds_raw;

  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid / WAVE);
  const int lane = tid % WAVE;
  const int qcol = lane & 31;
  const int hi = lane >> 5;
  // a ring of this wave's, or of all waves'
  char* ring = lds_raw + BT_CAP * 4 +
               (KEYS ? wave * RING_KEYS * 2 * TILE_BYTES : 0);

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
  const int n_kv_tiles = (kv_end + KVBLK - 1) / KVBLK;

  // ---- prologue: Q fragments + block table; every ordinary global load
  //      completes before the first glds issues ----
  bf16x8 qf[D / 16];
  const unsigned int flip = scale < 0.f ? 0x80008000u : 0u;
#pragma unroll
  for (int kk = 0; kk < D / 16; ++kk) {
    const uint4v v = *(const uint4v*)(q + q_row * D + kk * 16 + hi * 8);
    qf[kk] = __builtin_bit_cast(bf16x8, v ^ flip);
  }
  const float scale_log2 = fabsf(scale) * LOG2E;
  auto page_of = [&](int t) { return SHIFT ? t >> shift : t / bs; };
  const int n_bt = min(max_blocks, page_of(kv_end - 1) + 1);
  for (int i = tid; i < n_bt; i += NW * WAVE)
    bt_lds[i] = block_tables[(int64_t)seq * max_blocks + i];
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();  // publish bt_lds (no glds in flight yet)

  // rows of a tile that a wave fetches, 4 per instruction
  constexpr int LOADS = KVBLK / 4 / (KEYS ? 1 : NW);
  auto stage = [&](int n, int buf) {
    char* kb = ring + buf * 2 * TILE_BYTES;
#pragma unroll
    for (int j = 0; j < LOADS; ++j) {
      const int part = (KEYS ? 0 : wave * LOADS) + j;
      const int row = part * 4 + lane / 16;
      const int src = lane % 16 ^ swizzle(row) >> 4;    // source-side swizzle
      // keys past the last that is seen repeat it: no garbage bf16
      const int t = min(n * KVBLK + row, kv_end - 1), pg = page_of(t);
      const int at = t - (SHIFT ? pg << shift : pg * bs);
      const int64_t base =
          (((int64_t)bt_lds[pg] * kvh + kh) * bs + at) * D + src * 8;
      typedef const __attribute__((address_space(1))) unsigned int gmem;
      typedef __attribute__((address_space(3))) unsigned int smem;
      __builtin_amdgcn_global_load_lds((gmem*)(k_cache + base),
                                       (smem*)(kb + part * 1024), 16, 0, 0);
      __builtin_amdgcn_global_load_lds(
          (gmem*)(v_cache + base), (smem*)(kb + TILE_BYTES + part * 1024), 16,
          0, 0);
    }
  };

  Softmax st;
  f32x16 acc[D / 32];
#pragma unroll
  for (int t = 0; t < D / 32; ++t) acc[t] = (f32x16)(0.f);

  // the lane's share of addresses in a tile
  const int i16 = lane % 16;
  const int k_row = qcol * 256, k_swz = swizzle(qcol);
  const int v_col = (16 * ((lane & 31) >> 4) + (i16 % 4) * 4) * 2;
  auto compute = [&](int n, int buf) {
    const int tile0 = n * KVBLK;
    const char* kb = ring + buf * 2 * TILE_BYTES;
    const char* vb = kb + TILE_BYTES;
    attend32<D / 16, D / 32, FINE>(
        [&](int kk) {
          return *(const bf16x8*)(kb + k_row +
                                  ((kk * 32 + hi * 16) ^ k_swz));
        },
        [&](int row, int t) {
          return vb + row * 256 + ((t * 64 + v_col) ^ swizzle(row));
        },
        qf, scale_log2, tile0 + KVBLK - 1 <= prior + first_w, 0,
        prior + p - tile0, st, acc);
  };

  if constexpr (KEYS) {
    // tiles wave, wave + NW, ..
    const int mine = n_kv_tiles > wave ? (n_kv_tiles - wave + NW - 1) / NW : 0;
    for (int i = 0; i < min(mine, RING_KEYS); ++i) stage(wave + i * NW, i);
    for (int i = 0; i < mine; ++i) {
      if (i + 1 < mine)
        asm volatile("s_waitcnt vmcnt(%0)" ::"i"(2 * LOADS) : "memory");
      else
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      compute(wave + i * NW, i % RING_KEYS);
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // reads are done
      if (i + RING_KEYS < mine)
        stage(wave + (i + RING_KEYS) * NW, i % RING_KEYS);
    }
  } else {
    stage(0, 0);
    if (n_kv_tiles > 1) stage(1, 1);
    int buf = 0, fill = 2;
    for (int n = 0; n < n_kv_tiles; ++n) {
      // tile n has landed when at most the NEXT tile's DMA remains in
      // flight (counted per-wave wait; vmcnt retires in order)
      if (n + 1 < n_kv_tiles)
        asm volatile("s_waitcnt vmcnt(%0)" ::"i"(2 * LOADS) : "memory");
      else
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      raw_barrier();
      if (n * KVBLK < kv_end_w) compute(n, buf);
      if (n + 2 < n_kv_tiles) stage(n + 2, fill);
      buf = buf + 1 == RING_ROWS ? 0 : buf + 1;
      fill = fill + 1 == RING_ROWS ? 0 : fill + 1;
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
    if (!active || !(l > 0.f)) return;
    const float inv = 1.f / l;
    short* dst = out + q_row * D + wave * 32 + 4 * hi;
#pragma unroll
    for (int g = 0; g < 4; ++g)
      *(uint2*)(dst + 8 * g) = make_uint2(
          pack2(o[4 * g] * inv, o[4 * g + 1] * inv),
          pack2(o[4 * g + 2] * inv, o[4 * g + 3] * inv));
  } else if (active && st.l > 0.f) {
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
  auto fn = flash_prefill_glds_kernel<QPG, KEYS, FINE, SHIFT>;
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
// to make up for the second (300 tokens behind 300 23 us by keys, 28 by rows; 4
// x 100 13 and 10).
hipError_t lds_flash_prefill_glds(
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
  const bool pow2 = 1 << shift == bs;
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
