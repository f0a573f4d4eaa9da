// context_prefill.hip — causal (windowed) prefill attention of long portions
// (bf16). A tile is 128 rows of (query, head): all heads of a key/value head
// share its tiles of keys. Keys and values come from
//   pages        grouped heads: cache rows [key | value], found through the
//                block table a tile ahead. Where the rows of a wave's load lie in
//                one page its address is a scalar's work; else each lane finds its
//                row (block sizes that are powers of two without divisions, which
//                took as long as the scores)
//   context rows latent attention: keys and values expanded from the latents
//                of everything a portion may see, the rotated key part shared
//                by all heads; a sequence's context row 0 sits at ctx.pos0
//
// The attention of 32 queries and 32 keys is flash_core.h's: S' = K Q' keeps a
// query per lane. Rows of the LDS tiles are padded instead of swizzled: 16
// bytes for K (16-byte row reads hit distinct banks), 64 bytes for V (the
// transposing reads of four rows do). Two tiles are in LDS, a third on its way in
// registers; its loads and LDS writes stand between the matrix instructions. Tiles
// run from the last to the first: under the causal mask the last of a sequence has
// the most keys.
//
// 7800 rows of 7 prompts behind 100 tokens, 32 heads of 128 on 8 key heads: 148 us (196
// with an address worked out per lane and row, 232 with one tile in LDS, divisions and
// operands of K waited for one by one; 231 in tiles of 32 keys); one prompt of 7100 rows
// 470 (620); 7750 rows of 8 prompts, 32 heads of 192 and 128: 157 us (178 with 64-bit
// products per load; 253 in tiles of 64 keys, whose scores do not fit the registers beside
// a tile).
#include "../flash_core.h"
#include "elem.h"

#include <type_traits>

namespace {

constexpr int NW = 4, NT = NW * WAVE;
constexpr int QW = 32;          // query rows per wave

using namespace flash;

struct Prefill {
  const short* q;
  int64_t q_row;             // rows of q, heads D + rot apart
  // context rows: key columns [0, D) at ka, the rest at kb, values at v
  const short *ka, *kb, *v;
  int64_t ka_tok, ka_head, kb_tok, v_tok, v_head;
  const int32_t* ctx;        // [n_seqs, 2] = first context row, its position
  // pages: rows of D + V elements from ka on
  const int32_t* block_tables;
  int max_blocks, bs, shift; // bs = 1 << shift; below 0: any
  int64_t page, head;        // strides of a page and of a head inside it
  const int32_t *seq_meta, *tiles;  // tiles [n, 2] = sequence, first query
  short* out;                // [rows, H V]
  int H, rep, D, rot, V, window;
  float scale, sink;         // sink: score (log2) of a key without a value
  int has_sink;
};

// keys per tile: as many as the registers hold scores of and a tile on its way
constexpr int keys_of(int DK, int DV) { return DK + DV <= 256 ? 64 : 32; }
constexpr int tile_of(int DK, int DV) {       // in LDS (shorts)
  return keys_of(DK, DV) * (DK + 8 + DV + 32);
}

// where rows lie: context rows, pages, pages that hold the rows of a wave's load whole
enum Rows { CONTEXT, PAGES, WHOLE };

// grid (key/value heads, tiles)
template <int DK, int DV, int ROWS>
__global__ __launch_bounds__(NT, DK + DV > 320 ? 1 : 2)
void context_prefill_kernel(const Prefill a_) {
  constexpr bool PAGED = ROWS != CONTEXT;
  constexpr int KS = DK + 8, VS = DV + 32;      // row strides in LDS (shorts)
  constexpr int KB = keys_of(DK, DV);
  constexpr int NK = DK * KB / 8 / NT, NV = DV * KB / 8 / NT;   // loads
  constexpr int TILE = tile_of(DK, DV);         // keys [KB][KS], values [KB][VS]
  extern __shared__ short lds[];
  const int kvh = blockIdx.x, rep = a_.rep;
  const int tile = gridDim.y - 1 - blockIdx.y;
  const int seq = a_.tiles[2 * tile], p0 = a_.tiles[2 * tile + 1];
  const Seq sq = load_seq(a_.seq_meta, seq);
  const int64_t ctx0 = PAGED ? 0 : a_.ctx[2 * seq];
  // query p sees keys <= off + p
  const int off = PAGED ? sq.prior : sq.prior - a_.ctx[2 * seq + 1];
  const int32_t* bt =
      PAGED ? a_.block_tables + (int64_t)seq * a_.max_blocks : nullptr;
  const int tid = threadIdx.x, wave = tid / WAVE, lane = tid % WAVE;
  const int qc = lane & 31, hi = lane >> 5;
  const int nq = NW * QW / rep;                 // queries per tile
  const int vr = wave * QW + qc;                // row of the tile
  const int p_last = min(p0 + nq, sq.n) - 1;
  const bool active = vr / rep < nq && p0 + vr / rep < sq.n;
  const int p = active ? p0 + vr / rep : p_last;
  const int h = kvh * rep + vr % rep;
  const int QD = a_.D + a_.rot, D = a_.D, V = a_.V, bs = a_.bs;
  const int window = a_.window;

  bf16x8 qf[DK / 16];
  const unsigned int flip = a_.scale < 0.f ? 0x80008000u : 0u;
  const float scale_log2 = log2_scale(a_.scale);
  {
    const short* qr = a_.q + (sq.row0 + p) * a_.q_row + h * QD;
#pragma unroll
    for (int kk = 0; kk < DK / 16; ++kk) {
      const int d = kk * 16 + hi * 8;
      uint4v z = {0, 0, 0, 0};
      if (d < QD) z = *(const uint4v*)(qr + d);
      qf[kk] = __builtin_bit_cast(bf16x8, z ^ flip);
    }
  }
  Softmax st;
  if (a_.has_sink) {             // one of the halves' sums has it
    st.m = a_.sink;
    st.l = hi ? 0.f : 1.f;
  }
  f32x16 acc[DV / 32];
#pragma unroll
  for (int t = 0; t < DV / 32; ++t) acc[t] = (f32x16)(0.f);

  auto first_key = [&](int pp) {
    return window > 0 ? max(0, off + pp - window + 1) : 0;
  };
  const int hi_wg = off + p_last + 1;           // one past the last key
  const int lo_wg = first_key(p0) / KB * KB;
  // queries of this wave: [pw0, pw1]
  const int pw0 = p0 + wave * QW / rep;
  const int pw1 = min(p0 + (wave * QW + QW - 1) / rep, p_last);
  const int hi_w = pw0 <= p_last ? off + pw1 + 1 : 0;
  const int lo_w = first_key(pw0);

  // A tile goes through registers: rows past the last key that is seen repeat it
  // (they are masked), channels past the end are 0.
  short8 kn[NK], vn[NV];
  // pages of a tile; WHOLE: those from its first key's on, one per lane
  int kp[ROWS == PAGES ? NK : 1], vp[ROWS == PAGES && DK != DV ? NV : 1];
  const int shift = a_.shift, page_mask = bs - 1;
  auto row_of = [&](int t0, int i, int per) {
    return min(t0 + (tid + i * NT) / per, hi_wg - 1);
  };
  auto find = [&](int t0) {
    if constexpr (ROWS == WHOLE)
      kp[0] = bt[min((t0 >> shift) + lane, (hi_wg - 1) >> shift)];
    if constexpr (ROWS == PAGES) {
#pragma unroll
      for (int i = 0; i < NK; ++i) {
        const int t = row_of(t0, i, DK / 8);
        kp[i] = bt[shift < 0 ? t / bs : t >> shift];
      }
      if constexpr (DK != DV)
#pragma unroll
        for (int i = 0; i < NV; ++i) {
          const int t = row_of(t0, i, DV / 8);
          vp[i] = bt[shift < 0 ? t / bs : t >> shift];
        }
    }
  };
  const short* const pages = a_.ka + kvh * a_.head;
  auto page_row = [&](int page, int t) {
    const uint32_t at = (shift < 0 ? t % bs : t & page_mask) * (D + V);
    return pages + ((uint64_t)(uint32_t)page * (uint64_t)a_.page + at);
  };
  // WHOLE: the row of load i, in the page of the wave's first one
  constexpr int PER = WAVE * 8 / DK;            // rows of a wave's load
  const int first_row = __builtin_amdgcn_readfirstlane(wave) * PER;
  auto whole_row = [&](int t0, int i) {
    const int t = t0 + first_row + i * NW * PER, last = hi_wg - 1;
    const int at = (min(t, last) >> shift) - (t0 >> shift);
    const uint32_t page = __builtin_amdgcn_readlane(kp[0], max(at, 0));
    const short* from = pages + (uint64_t)page * (uint32_t)a_.page;
    return from + (uint32_t)((min(t + lane / (DK / 8), last) & page_mask) * (DK + DV) +
                             lane % (DK / 8) * 8);
  };
  // CONTEXT: row 0 of each load's channels and the stride of its rows
  constexpr bool CTX = ROWS == CONTEXT;
  const short *k_from[CTX ? NK : 1], *v_from[CTX ? NV : 1];
  uint32_t k_tok[CTX ? NK : 1];
  if constexpr (CTX) {
#pragma unroll
    for (int i = 0; i < NK; ++i) {
      const int d = (tid + i * NT) % (DK / 8) * 8;
      k_from[i] = d < D ? a_.ka + ctx0 * a_.ka_tok + kvh * a_.ka_head + d
                        : a_.kb + ctx0 * a_.kb_tok + (d - D);
      k_tok[i] = d < D ? a_.ka_tok : a_.kb_tok;
    }
#pragma unroll
    for (int i = 0; i < NV; ++i)
      v_from[i] = a_.v + ctx0 * a_.v_tok + kvh * a_.v_head +
                  (tid + i * NT) % (DV / 8) * 8;
  }
  // load i of the keys, then of the values
  auto fetch = [&](int t0, int i) {
    if constexpr (ROWS == WHOLE) {
      static_assert(DK == DV, "");
      if (i < NK) kn[i] = *(const short8*)whole_row(t0, i);
      else vn[i - NK] = *(const short8*)(whole_row(t0, i - NK) + DK);
      return;
    }
    if (i < NK) {
      const int t = row_of(t0, i, DK / 8), d = (tid + i * NT) % (DK / 8) * 8;
      kn[i] = (short8){0, 0, 0, 0, 0, 0, 0, 0};
      if (d < QD) {
        if constexpr (PAGED)
          kn[i] = *(const short8*)(page_row(kp[ROWS == PAGES ? i : 0], t) + d);
        else
          kn[i] = *(const short8*)(k_from[CTX ? i : 0] +
                                   (uint64_t)(uint32_t)t * k_tok[CTX ? i : 0]);
      }
    } else {
      i -= NK;
      const int t = row_of(t0, i, DV / 8), d = (tid + i * NT) % (DV / 8) * 8;
      vn[i] = (short8){0, 0, 0, 0, 0, 0, 0, 0};
      if (d < V) {
        if constexpr (PAGED)
          vn[i] = *(const short8*)(
              page_row(DK == DV ? kp[ROWS == PAGES ? i : 0]
                                : vp[ROWS == PAGES && DK != DV ? i : 0], t) +
              D + d);
        else
          vn[i] = *(const short8*)(v_from[CTX ? i : 0] +
                                   (uint64_t)(uint32_t)t * (uint32_t)a_.v_tok);
      }
    }
  };
  auto put = [&](int buf, int i) {
    short* to = lds + buf * TILE;
    if (i < NK) {
      const int ch = tid + i * NT;
      *(short8*)(to + ch / (DK / 8) * KS + ch % (DK / 8) * 8) = kn[i];
    } else {
      i -= NK;
      const int ch = tid + i * NT;
      *(short8*)(to + KB * KS + ch / (DV / 8) * VS + ch % (DV / 8) * 8) = vn[i];
    }
  };
  const int i16 = lane % 16;
  // the tile at t0 from `buf`
  auto compute = [&](int t0, int buf, auto between) {
    const short* kb = lds + buf * TILE + qc * KS + hi * 8;
    const short* vb = lds + buf * TILE + KB * KS + 16 * ((lane & 31) >> 4) +
                      (i16 % 4) * 4;
    attend<DK / 16, DV / 32, KB / 32, false>(
        [&](int u, int kk) {
          return *(const bf16x8*)(kb + u * 32 * KS + kk * 16);
        },
        [&](int u, int row, int t) {
          return vb + (u * 32 + row) * VS + t * 32;
        },
        qf, scale_log2, t0 + KB - 1 <= off + pw0 && t0 >= first_key(pw1),
        first_key(p) - t0, off + p - t0, st, acc, between);
  };
  auto skips = [&](int t0) { return t0 >= hi_w || t0 + KB <= lo_w; };
  find(lo_wg);
#pragma unroll
  for (int i = 0; i < NK + NV; ++i) fetch(lo_wg, i);
  // Two tiles in LDS: while one is computed, the next one leaves the registers
  // and the one after it comes in, between the matrix instructions.
#pragma unroll
  for (int i = 0; i < NK + NV; ++i) put(0, i);
  if (lo_wg + KB < hi_wg) {
    find(lo_wg + KB);
#pragma unroll
    for (int i = 0; i < NK + NV; ++i) fetch(lo_wg + KB, i);
    find(lo_wg + 2 * KB);
  }
  auto step = [&](int t0, auto buf_) {
    constexpr int buf = decltype(buf_)::value;
    lds_barrier();
    if (skips(t0)) {                                 // wave-uniform
#pragma unroll
      for (int i = 0; i < NK + NV; ++i) {
        put(buf ^ 1, i);
        fetch(t0 + 2 * KB, i);
      }
      find(t0 + 3 * KB);
      return;
    }
    compute(t0, buf, [&](int m) {
      constexpr int N = DK / 16 * KB / 32;           // matrix instructions
#pragma unroll
      for (int i = 0; i < NK + NV; ++i)
        if (i * N / (NK + NV) == m) {
          put(buf ^ 1, i);
          fetch(t0 + 2 * KB, i);
        }
      if (m == N - 1) find(t0 + 3 * KB);
    });
  };
  for (int t0 = lo_wg; t0 < hi_wg; t0 += 2 * KB) {
    step(t0, std::integral_constant<int, 0>{});
    if (t0 + KB < hi_wg) step(t0 + KB, std::integral_constant<int, 1>{});
  }
  st.l = st.join();

  if (active) {
    const float inv = 1.f / st.l;
    short* o = a_.out + ((int64_t)(sq.row0 + p) * a_.H + h) * V;
#pragma unroll
    for (int t = 0; t < DV / 32; ++t)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int d = t * 32 + 8 * g + 4 * hi;
        if (d < V)
          *(uint2*)(o + d) =
              make_uint2(pack2(acc[t][4 * g] * inv, acc[t][4 * g + 1] * inv),
                         pack2(acc[t][4 * g + 2] * inv,
                               acc[t][4 * g + 3] * inv));
      }
  }
}

template <int DK, int DV, int ROWS>
hipError_t launch(const Prefill& a, int kv_heads, int n_tiles,
                  hipStream_t stream) {
  const int lds = 2 * tile_of(DK, DV) * (int)sizeof(short);
  auto fn = context_prefill_kernel<DK, DV, ROWS>;
  hipError_t e = hipFuncSetAttribute(
      (const void*)fn, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(fn, dim3(kv_heads, n_tiles), dim3(NT), lds, stream, a);
  HIP_CHECK_LAST();
  return hipSuccess;
}

}  // namespace

extern "C" {

// 0 if the sizes have no tiled form
int lds_latent_prefill_ok(int D, int rot, int V, int R) {
  return D % 8 == 0 && rot % 8 == 0 && V % 8 == 0 && R % 8 == 0 &&
         D + rot <= 192 && V <= 128;
}

hipError_t lds_latent_prefill(const void* q, const void* kv, const void* lat,
                              const int32_t* seq_meta, const int32_t* ctx,
                              const int32_t* tiles, int n_tiles, void* out,
                              int H, int D, int rot, int V, int lat_w,
                              int window, float scale, hipStream_t stream) {
  if (n_tiles == 0) return hipSuccess;
  if (n_tiles > 65535 || !lds_latent_prefill_ok(D, rot, V, lat_w - rot))
    return hipErrorInvalidValue;
  Prefill a{};
  a.q = (const short*)q;
  a.q_row = (int64_t)H * (D + rot);
  a.ka = (const short*)kv;
  a.kb = (const short*)lat + lat_w - rot;
  a.v = (const short*)kv + (int64_t)H * D;
  a.ka_tok = a.v_tok = (int64_t)H * (D + V);
  a.ka_head = D;
  a.kb_tok = lat_w;
  a.v_head = V;
  a.ctx = ctx;
  a.bs = 1;
  a.seq_meta = seq_meta;
  a.tiles = tiles;
  a.out = (short*)out;
  a.H = H;
  a.rep = 1;
  a.D = D;
  a.rot = rot;
  a.V = V;
  a.window = window;
  a.scale = scale;
  const int qd = D + rot;
#define GO(DK)                                                                \
  return V <= 64 ? launch<DK, 64, CONTEXT>(a, H, n_tiles, stream)               \
                 : launch<DK, 128, CONTEXT>(a, H, n_tiles, stream)
  if (qd <= 64) GO(64);
  if (qd <= 96) GO(96);
  if (qd <= 128) GO(128);
  GO(192);
#undef GO
}

int lds_grouped_prefill_ok(int D, int V, int rep, int64_t q_stride) {
  return D % 8 == 0 && V % 8 == 0 && q_stride % 8 == 0 && D <= 256 &&
         V <= 256 && rep <= NW * QW;
}

// q: first query of row 0, rows q_stride apart; cache [NB, G, bs, D + V];
// tiles hold 128 / (H / G) queries; out [rows, H V]
hipError_t lds_grouped_prefill(const void* q, int64_t q_stride,
                               const void* cache, const int32_t* block_tables,
                               int max_blocks, int bs,
                               const int32_t* seq_meta, const int32_t* tiles,
                               int n_tiles, void* out, int H, int G, int D,
                               int V, float scale, int has_sink, float sink,
                               hipStream_t stream) {
  if (n_tiles == 0) return hipSuccess;
  if (n_tiles > 65535 || !lds_grouped_prefill_ok(D, V, H / G, q_stride))
    return hipErrorInvalidValue;
  Prefill a{};
  a.q = (const short*)q;
  a.q_row = q_stride;
  a.ka = (const short*)cache;
  a.block_tables = block_tables;
  a.max_blocks = max_blocks;
  a.bs = bs;
  a.shift = bs & bs - 1 ? -1 : __builtin_ctz(bs);
  a.head = (int64_t)bs * (D + V);
  a.page = G * a.head;
  a.seq_meta = seq_meta;
  a.tiles = tiles;
  a.out = (short*)out;
  a.H = H;
  a.rep = H / G;
  a.D = D;
  a.V = V;
  a.scale = scale;
  a.has_sink = has_sink;
  a.sink = sink * LOG2E;
  // rows of a load of 1 KB in one page: 8 of 64, 4 of 128, 2 of 256
  if (D == V && a.shift >= 0 && bs * D >= 512 && a.page < 1ll << 32) {
    if (D == 64) return launch<64, 64, WHOLE>(a, G, n_tiles, stream);
    if (D == 128) return launch<128, 128, WHOLE>(a, G, n_tiles, stream);
    if (D == 256) return launch<256, 256, WHOLE>(a, G, n_tiles, stream);
  }
#define GO(DK)                                                                \
  return V <= 64    ? launch<DK, 64, PAGES>(a, G, n_tiles, stream)             \
         : V <= 128 ? launch<DK, 128, PAGES>(a, G, n_tiles, stream)            \
                    : launch<DK, 256, PAGES>(a, G, n_tiles, stream)
  if (D <= 64) GO(64);
  if (D <= 128) GO(128);
  if (D <= 192) GO(192);
  GO(256);
#undef GO
}

}  // extern "C"
