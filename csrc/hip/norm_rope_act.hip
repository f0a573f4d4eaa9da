// norm_rope_act.hip — fused memory-bound decoder-layer kernels for gfx950.
// All are HBM-bound: bf16 traffic is vectorized as short8 (16 B/lane,
// guide G13 — scalar bf16 is ~2x slower), fp32 math in registers.
//
// These replace what the reference delegates to vLLM inside its model-server
// pods (the router itself has no kernels); in the MI355X-native engine the
// per-GPU worker runs them directly.
#include "hip_common.h"

namespace {

// ---------------------------------------------------------------------------
// rmsnorm (+ optional fused residual add):
//   if residual: r = r + x  (written back);  src = r
//   else:        src = x
//   y = src * rsqrt(mean(src^2) + eps) * w
// x is bf16, or the partial sums of a product that split K: [parts, rows, H]
// 32-bit, summed here instead of by a launch of their own (8 parts, one row of
// 4096: sum and norm apart 8.7 us, so 4.1).
// One block per token row, of 256 threads, or 512 where the row is in parts and has
// more than 256 vectors of 8: most of its time is the loads' way, and so each thread has
// half of them. Row length H % 8 == 0. The first KEEP
// vectors of a thread stay in registers between the two passes, the rest are
// read again. Their number is known at compile time: an index that is not puts
// the array into scratch memory (8013 rows of 4096 with residual: 84 us, now
// 44, 5.9 TB/s).
// ---------------------------------------------------------------------------
constexpr int NT = 256;
constexpr int PT = 512;

// EARLY: with parts, all that a thread keeps is asked for at once, pair by pair. Up to
// 2048 channels always; above up to 512 rows where a thread has one vector, 256 where it
// has two, the second of which reads past the row's end. us, with residual, parts and
// residual in the caches, 512 threads early / not, 256 early / not:
//             rows      2 parts                   8 parts
//   1024         1   2.2  2.3  2.2  2.3      2.9  2.7  2.5  2.7
//              256   2.6  2.7  2.5  2.7      4.3  4.6  3.9  4.6
//              640   4.8  4.1  3.9  4.0      7.3  6.3  5.9  6.2
//   2048         1   2.3  2.4  2.2  2.3      3.0  2.8  2.6  2.8
//              256   3.5  3.7  3.4  3.7      5.5  5.6  5.1  5.6
//              640   5.6  5.2  4.9  5.2      9.4  9.5  9.0  9.5
//   4096         1   2.4  2.5  2.7  3.0      3.2  3.2  3.6  4.0
//              256   4.4  4.6  4.7  5.1      7.8  8.0  8.0  8.6
//              512   6.4  6.6  6.8  6.8     13.2 13.2 13.3 13.6
//   5120         1   3.0  3.1  3.2  3.7      4.4  4.1  4.9  5.1
//              256   5.3  5.5  5.6  6.2      9.3  9.9  9.8 10.7
//              400   7.8  7.1  7.0  7.5     14.3 13.5 13.7 13.8
// ROWS: ALL of them; PICKED: the rows that `rows` names, of n_rows, without a word to
// the residual; TABLE: rows of the table x that `rows` names (token ids), which become the
// residual. As in an index, rows below 0 count from the end. Rows that do not exist are
// NaN throughout: never another row's values.
enum Rows { ALL, PICKED, TABLE };

template <int BT, int KEEP, bool RESIDUAL, bool PARTS, bool EARLY, int ROWS>
__global__ __launch_bounds__(BT) void rmsnorm_kernel(
    const void* __restrict__ x, int parts, short* __restrict__ residual,
    const short* __restrict__ w, short* __restrict__ y, int H, float eps,
    const int64_t* __restrict__ rows, int64_t n_rows) {
  __shared__ float red[BT / WAVE];
  int64_t row = blockIdx.x;
  if constexpr (ROWS != ALL) {
    row = rows[row];
    row += row < 0 ? n_rows : 0;
  }
  const int nchunks = H / 8;
  short8* r8 = RESIDUAL ? (short8*)(residual + row * H)
               : ROWS == TABLE ? (short8*)(residual + (int64_t)blockIdx.x * H)
                               : nullptr;
  if (ROWS != ALL && (row < 0 || row >= n_rows)) {
    short8 nan;
#pragma unroll
    for (int j = 0; j < 8; ++j) nan[j] = 0x7fc0;
    for (int c = threadIdx.x; c < nchunks; c += BT) {
      ((short8*)(y + (int64_t)blockIdx.x * H))[c] = nan;
      if (ROWS == TABLE) r8[c] = nan;
    }
    return;
  }
  auto source = [&](int c, float* f) {
    if constexpr (EARLY) {
      const float4v* const p[1] = {(const float4v*)x + (row * H + c * 8) / 4};
      PartSums<1>(p, n_rows * H / 4, parts).get(0, f);
    } else if constexpr (PARTS) {
      const float4v* p = (const float4v*)x + (row * H + c * 8) / 4;
      const int64_t apart = n_rows * H / 4;
      float4v a = p[0], b = p[1];
#pragma unroll 4
      for (int i = 1; i < parts; ++i) {
        a += p[i * apart];
        b += p[i * apart + 1];
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        f[j] = a[j];
        f[4 + j] = b[j];
      }
    } else {
      const short8 v = ((const short8*)((const short*)x + row * H))[c];
#pragma unroll
      for (int j = 0; j < 8; ++j) f[j] = bf16_to_f32(v[j]);
    }
  };
  float vals[KEEP][8], ss = 0.f;
  static_assert(PARTS || !EARLY, "");
  constexpr bool AHEAD = EARLY;
  short8 rv[AHEAD ? KEEP : 1], wk[AHEAD ? KEEP : 1];
  if constexpr (AHEAD) {
    const int64_t apart = n_rows * H / 4;
#pragma unroll
    for (int i = 0; i < KEEP; ++i) {
      const int c = min((int)threadIdx.x + i * BT, nchunks - 1);
      if constexpr (RESIDUAL) rv[i] = r8[c];
      wk[i] = ((const short8*)w)[c];
    }
    constexpr int W = KEEP > 1 ? 2 : 1;
#pragma unroll
    for (int i = 0; i < KEEP; i += W) {
      const float4v* p[W];
#pragma unroll
      for (int j = 0; j < W; ++j)
        p[j] = (const float4v*)x + row * H / 4 +
               min((int)threadIdx.x + (i + j) * BT, nchunks - 1) * 2;
      const PartSums<W> sum(p, apart, parts);
#pragma unroll
      for (int j = 0; j < W; ++j) sum.get(j, vals[i + j]);
    }
  }
  auto first = [&](int c, float* f, int i) {
    if (!AHEAD || i < 0) source(c, f);
    if constexpr (RESIDUAL) {
      const short8 r = AHEAD && i >= 0 ? rv[AHEAD ? i : 0] : r8[c];
      short8 ro;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        f[j] += bf16_to_f32(r[j]);
        ro[j] = f32_to_bf16(f[j]);
      }
      if (ROWS == ALL) r8[c] = ro;  // residual stream updated in place
    } else if constexpr (ROWS == TABLE) {
      short8 ro;
#pragma unroll
      for (int j = 0; j < 8; ++j) ro[j] = f32_to_bf16(f[j]);
      r8[c] = ro;
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) ss += f[j] * f[j];
  };
#pragma unroll
  for (int i = 0; i < KEEP; ++i) {
    const int c = threadIdx.x + i * BT;
    if (c < nchunks) first(c, vals[i], i);
  }
  for (int c = threadIdx.x + KEEP * BT; c < nchunks; c += BT) {
    float f[8];
    first(c, f, -1);
  }
  const float inv =
      rsqrtf(block_reduce_sum<BT / WAVE>(ss, red) / (float)H + eps);
  auto second = [&](int c, const float* f, int i) {
    const short8 wv =
        AHEAD && i >= 0 ? wk[AHEAD ? i : 0] : ((const short8*)w)[c];
    short8 o;
#pragma unroll
    for (int j = 0; j < 8; ++j)
      o[j] = f32_to_bf16(f[j] * inv * bf16_to_f32(wv[j]));
    ((short8*)(y + (int64_t)blockIdx.x * H))[c] = o;
  };
#pragma unroll
  for (int i = 0; i < KEEP; ++i) {
    const int c = threadIdx.x + i * BT;
    if (c < nchunks) second(c, vals[i], i);
  }
  for (int c = threadIdx.x + KEEP * BT; c < nchunks; c += BT) {
    float f[8];
    if constexpr (RESIDUAL && ROWS == ALL) {   // this thread's own store above
      const short8 v = r8[c];
#pragma unroll
      for (int j = 0; j < 8; ++j) f[j] = bf16_to_f32(v[j]);
    } else if constexpr (RESIDUAL) {           // what it would have been
      const short8 v = r8[c];
      source(c, f);
#pragma unroll
      for (int j = 0; j < 8; ++j)
        f[j] = bf16_to_f32(f32_to_bf16(f[j] + bf16_to_f32(v[j])));
    } else {
      source(c, f);
    }
    second(c, f, -1);
  }
}

// ---------------------------------------------------------------------------
// What lies between a decoder layer's qkv product and its attention, in one
// pass: heads of q and k are normed (Qwen3; where qw is set), rotated
// (rotate-half, angles from the host's table) and rounded; q goes to a packed
// [T, QH, D], k and v to their slots in the paged cache.
//   qkv: [T, QH + 2 KVH heads, D] bf16, rows apart by `stride` elements, or
//   the 32-bit partial sums [parts, T, ..] of the product
// A thread owns 8 channels of a head's first half and the 8 they rotate with;
// D / 16 threads share a head. Bound by its bytes: it reads and writes each
// value once, where separate copies, rotation and scatter took five passes
// (8013 rows of 48 heads: 37 us, was 142).
// ---------------------------------------------------------------------------
struct Heads {
  const void* qkv;
  int parts;
  int64_t stride;
  const short *qw, *kw;          // [D] or null
  const float* cos_sin;          // [max_pos, D / 2, 2]
  const int32_t* positions;      // [T]
  const int64_t* slots;          // [T], below 0: not cached
  short* q;                      // [T, QH, D]
  void *k_cache, *v_cache;       // [NB, KVH, BS, D]
  int T, qh, kvh, bs, d;
  float eps;
};

template <typename CT, bool PARTS, bool NORM>
__global__ __launch_bounds__(NT) void heads_kernel(const Heads p) {
  const int per = p.d / 16, heads = p.qh + 2 * p.kvh, half = p.d / 2;
  const uint32_t i = blockIdx.x * NT + threadIdx.x, hd = i / per;
  const int t = hd / heads, h = hd % heads, c = i % per * 8;
  if (t >= p.T) return;          // whole heads: lanes of one stay together
  float f[2][8];
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    const int64_t at = t * p.stride + h * p.d + s * half + c;
    if constexpr (PARTS) {
      const float4v* src = (const float4v*)((const float*)p.qkv + at);
      const int64_t apart = p.T * p.stride / 4;
      float4v a = src[0], b = src[1];
#pragma unroll 4
      for (int k = 1; k < p.parts; ++k) {
        a += src[k * apart];
        b += src[k * apart + 1];
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        f[s][j] = a[j];
        f[s][4 + j] = b[j];
      }
    } else {
      const short8 v = *(const short8*)((const short*)p.qkv + at);
#pragma unroll
      for (int j = 0; j < 8; ++j) f[s][j] = bf16_to_f32(v[j]);
    }
  }
  const bool value = h >= p.qh + p.kvh, key = !value && h >= p.qh;
  if (NORM) {
    float ss = 0.f;
#pragma unroll
    for (int j = 0; j < 8; ++j)
      ss += f[0][j] * f[0][j] + f[1][j] * f[1][j];
    for (int o = 1; o < per; o <<= 1) ss += __shfl_xor(ss, o, WAVE);
    if (!value) {
      const float inv = rsqrtf(ss / (float)p.d + p.eps);
      const short* w = key ? p.kw : p.qw;
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        const short8 wv = *(const short8*)(w + s * half + c);
#pragma unroll
        for (int j = 0; j < 8; ++j) f[s][j] *= inv * bf16_to_f32(wv[j]);
      }
    }
  }
  short8 lo, hi;
  if (value) {
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      lo[j] = f32_to_bf16(f[0][j]);
      hi[j] = f32_to_bf16(f[1][j]);
    }
  } else {
    const float4v* cs = (const float4v*)(
        p.cos_sin + ((int64_t)p.positions[t] * half + c) * 2);
#pragma unroll
    for (int j = 0; j < 8; j += 2) {
      const float4v a = cs[j / 2];
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        const float co = a[2 * k], si = a[2 * k + 1];
        const float u = f[0][j + k], v = f[1][j + k];
        lo[j + k] = f32_to_bf16(u * co - v * si);
        hi[j + k] = f32_to_bf16(v * co + u * si);
      }
    }
  }
  if (h < p.qh) {
    short* o = p.q + ((int64_t)t * p.qh + h) * p.d + c;
    *(short8*)o = lo;
    *(short8*)(o + half) = hi;
    return;
  }
  const int64_t slot = p.slots[t];
  if (slot < 0) return;          // padding token
  const int kh = h - p.qh - (value ? p.kvh : 0);
  CT* o = (CT*)(value ? p.v_cache : p.k_cache) +
          ((slot / p.bs * p.kvh + kh) * p.bs + slot % p.bs) * p.d + c;
  store_kv8(o, lo);
  store_kv8(o + half, hi);
}

// ---------------------------------------------------------------------------
// RoPE (Llama/NeoX rotate-half), in place on q and k.
//   q: [T, n_q_heads, D], k: [T, n_kv_heads, D], D = 2*half
//   cos_sin: [max_pos, half, 2] f32 precomputed on host (guide App. B: no
//   on-device trig), positions: [T] int32
// grid = (T, n_q_heads + n_kv_heads); one wave per (token, head);
// lane i < half handles the (i, i+half) pair.
// ---------------------------------------------------------------------------
__global__ void rope_kernel(short* __restrict__ q, short* __restrict__ k,
                            const float* __restrict__ cos_sin,
                            const int32_t* __restrict__ positions, int n_tokens,
                            int n_q_heads, int n_kv_heads, int D) {
  const int t = blockIdx.x;
  const int head = blockIdx.y;
  const int half = D / 2;
  const int lane = threadIdx.x;
  if (t >= n_tokens || lane >= half) return;
  short* base = (head < n_q_heads)
                    ? q + ((int64_t)t * n_q_heads + head) * D
                    : k + ((int64_t)t * n_kv_heads + (head - n_q_heads)) * D;
  const float* cs = cos_sin + ((int64_t)positions[t] * half + lane) * 2;
  const float c = cs[0], s = cs[1];
  float x1 = bf16_to_f32(base[lane]);
  float x2 = bf16_to_f32(base[lane + half]);
  base[lane] = f32_to_bf16(x1 * c - x2 * s);
  base[lane + half] = f32_to_bf16(x2 * c + x1 * s);
}

// ---------------------------------------------------------------------------
// silu_mul: y = silu(gate) * up. gate/up are the two halves of one fused
// [T, 2*I] gate_up projection output (so the producing GEMM stays a single
// hipBLASLt call). Vectorized grid-stride over T rows.
// ---------------------------------------------------------------------------
__global__ void silu_mul_kernel(const short* __restrict__ gate_up,
                                short* __restrict__ y, int64_t T, int I) {
  const int nchunks = I / 8;
  const int64_t total = T * nchunks;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total;
       i += (int64_t)gridDim.x * blockDim.x) {
    int64_t row = i / nchunks;
    int c = (int)(i % nchunks);
    const short8* g8 = (const short8*)(gate_up + row * 2 * I);
    const short8* u8 = (const short8*)(gate_up + row * 2 * I + I);
    short8 g = g8[c], u = u8[c];
    short8 o;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      float gf = bf16_to_f32(g[j]);
      float uf = bf16_to_f32(u[j]);
      float sig = 1.f / (1.f + __expf(-gf));
      o[j] = f32_to_bf16(gf * sig * uf);
    }
    ((short8*)(y + row * I))[c] = o;
  }
}

}  // namespace

extern "C" {

// parts > 0: x are that many partial sums in 32-bit. rows: null, or n of the n_rows rows
// of x and of the residual, or (table) of the table x, whose copies fill the residual.
hipError_t lds_rmsnorm(const void* x, int parts, void* residual, const void* w,
                       void* y, int64_t n_rows, int H, float eps,
                       const int64_t* rows, int64_t n, int table,
                       hipStream_t stream) {
  if (!rows) n = n_rows;
  if (n == 0) return hipSuccess;
  if (n > 0x7fffffff || n_rows < 1 || H < 1 || (table && (!rows || !residual || parts)))
    return hipErrorInvalidValue;
#define GO(BT, KEEP, RES, PARTS, EARLY, ROWS)                                \
  hipLaunchKernelGGL((rmsnorm_kernel<BT, KEEP, RES, PARTS, EARLY, ROWS>),    \
                     dim3((uint32_t)n), dim3(BT), 0, stream, x, parts,       \
                     (short*)residual, (const short*)w, (short*)y, H, eps,   \
                     rows, n_rows)
#define GO_K(BT, RES, PARTS, EARLY, ROWS)                                    \
  do {                                                                       \
    if (H <= BT * 8) GO(BT, 1, RES, PARTS, EARLY, ROWS);                     \
    else if (H <= 2 * BT * 8) GO(BT, 2, RES, PARTS, EARLY, ROWS);            \
    else GO(BT, 4, RES, PARTS, EARLY, ROWS);                                 \
  } while (0)
#define GO_P(RES, ROWS)                                                      \
  do {                                                                       \
    if (H <= NT * 8) GO(NT, 1, RES, true, true, ROWS);                       \
    else if (n <= (H <= PT * 8 ? 512 : 256)) GO_K(PT, RES, true, true, ROWS); \
    else GO_K(PT, RES, true, false, ROWS);                                   \
  } while (0)
  if (table) {
    GO_K(NT, false, false, false, TABLE);
  } else if (rows && parts > 0) {
    if (residual) GO_P(true, PICKED); else GO_P(false, PICKED);
  } else if (rows) {
    if (residual) GO_K(NT, true, false, false, PICKED);
    else GO_K(NT, false, false, false, PICKED);
  } else if (parts > 0) {
    if (residual) GO_P(true, ALL); else GO_P(false, ALL);
  } else {
    if (residual) GO_K(NT, true, false, false, ALL);
    else GO_K(NT, false, false, false, ALL);
  }
#undef GO_P
#undef GO_K
#undef GO
  HIP_CHECK_LAST();
  return hipSuccess;
}

// 1 if heads of D channels have the one-pass form
int lds_heads_ok(int d, int norm) {
  const int per = d / 16;
  return d >= 16 && d % 16 == 0 &&
         (!norm || (per <= WAVE && (per & (per - 1)) == 0));
}

// see Heads; parts > 0: qkv are that many partial sums in 32-bit
hipError_t lds_heads(const void* qkv, int parts, int64_t stride,
                     const void* qw, const void* kw, const float* cos_sin,
                     const int32_t* positions, const int64_t* slots, void* q,
                     void* k_cache, void* v_cache, int T, int qh, int kvh,
                     int bs, int d, int kv_fp8, float eps,
                     hipStream_t stream) {
  if (T == 0) return hipSuccess;
  const int64_t n = (int64_t)T * (qh + 2 * kvh) * (d / 16);
  if (!lds_heads_ok(d, qw != nullptr) || stride % 8 || n >= 1ll << 31)
    return hipErrorInvalidValue;
  const Heads p{qkv, parts, stride, (const short*)qw, (const short*)kw,
                cos_sin, positions, slots, (short*)q, k_cache, v_cache, T, qh,
                kvh, bs, d, eps};
  const dim3 grid((uint32_t)((n + NT - 1) / NT));
#define GO(CT, PARTS, NORM)                                                  \
  hipLaunchKernelGGL((heads_kernel<CT, PARTS, NORM>), grid, dim3(NT), 0,     \
                     stream, p)
#define GO_CT(PARTS, NORM)                                                   \
  do {                                                                       \
    if (kv_fp8) GO(unsigned char, PARTS, NORM); else GO(short, PARTS, NORM); \
  } while (0)
  if (parts > 0) {
    if (qw) GO_CT(true, true); else GO_CT(true, false);
  } else {
    if (qw) GO_CT(false, true); else GO_CT(false, false);
  }
#undef GO_CT
#undef GO
  HIP_CHECK_LAST();
  return hipSuccess;
}

hipError_t lds_rope(void* q, void* k, const float* cos_sin,
                    const int32_t* positions, int n_tokens, int n_q_heads,
                    int n_kv_heads, int head_dim, hipStream_t stream) {
  if (n_tokens == 0) return hipSuccess;
  dim3 grid((uint32_t)n_tokens, (uint32_t)(n_q_heads + n_kv_heads));
  dim3 block(head_dim / 2 > 64 ? head_dim / 2 : 64);
  hipLaunchKernelGGL(rope_kernel, grid, block, 0, stream, (short*)q, (short*)k,
                     cos_sin, positions, n_tokens, n_q_heads, n_kv_heads,
                     head_dim);
  HIP_CHECK_LAST();
  return hipSuccess;
}

hipError_t lds_silu_mul(const void* gate_up, void* y, int64_t T, int I,
                        hipStream_t stream) {
  if (T == 0) return hipSuccess;
  int64_t total = T * (I / 8);
  int threads = 256;
  int blocks = (int)((total + threads - 1) / threads);
  if (blocks > 2048) blocks = 2048;  // grid-stride (guide G11)
  hipLaunchKernelGGL(silu_mul_kernel, dim3(blocks), dim3(threads), 0, stream,
                     (const short*)gate_up, (short*)y, T, I);
  HIP_CHECK_LAST();
  return hipSuccess;
}

}  // extern "C"
