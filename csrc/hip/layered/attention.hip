// attention.hip — cache rows of latent attention and of grouped heads, and
// plain attention over either.
//
// Latent attention caches per token: [latent (kv_rank, normed) | rotated key part (rot_dim)],
// pages [n_blocks, block_size, kv_rank + rot_dim]. Rows that come alone (or
// in short portions) attend to the pages directly, with the key projection
// absorbed into the query; long portions expand keys and values first
// (context_prefill.hip). attn_rows is the plain kernel for either form and for
// grouped heads: any size, bf16 or float.
#include "elem.h"

namespace {

constexpr int NT = 256;
constexpr int NWV = NT / WAVE;

// cos_sin: [max_pos, dims / 2, 2]. Rotates pairs (2i, 2i + 1).
template <typename T>
__device__ __forceinline__ void rotate_pair(const T* src, T* dst,
                                            const float* cs) {
  const float u = ld(src), v = ld(src + 1);
  st(dst, u * cs[0] - v * cs[1]);
  st(dst + 1, v * cs[0] + u * cs[1]);
}

// One workgroup per row of [.., q_rank | kv_rank | rot]: norms the query
// latent into cq, norms the latent and rotates the key part into the cache.
template <typename T>
__global__ __launch_bounds__(NT) void latent_prep_kernel(
    const T* __restrict__ proj, int64_t pstride, const float* __restrict__ wq,
    const float* __restrict__ wkv, const float* __restrict__ cos_sin,
    const int32_t* __restrict__ positions, const int64_t* __restrict__ slots,
    T* __restrict__ cq, T* __restrict__ cache, int q_rank, int kv_rank,
    int rot, float eps) {
  __shared__ float red[2][NWV];
  const int64_t row = blockIdx.x;
  const T* p = proj + row * pstride;
  float ss = 0.f;
  for (int d = threadIdx.x; d < q_rank; d += NT) {
    const float x = ld(p + d);
    ss += x * x;
  }
  float inv = 1.f / sqrtf(block_sum<NWV>(ss, red[0]) / (float)q_rank + eps);
  for (int d = threadIdx.x; d < q_rank; d += NT)
    st(cq + row * q_rank + d, ld(p + d) * inv * wq[d]);
  if (!cache) return;
  p += q_rank;
  ss = 0.f;
  for (int d = threadIdx.x; d < kv_rank; d += NT) {
    const float x = ld(p + d);
    ss += x * x;
  }
  inv = 1.f / sqrtf(block_sum<NWV>(ss, red[1]) / (float)kv_rank + eps);
  T* dst = cache + slots[row] * (kv_rank + rot);
  for (int d = threadIdx.x; d < kv_rank; d += NT)
    st(dst + d, ld(p + d) * inv * wkv[d]);
  const float* cs = cos_sin + (int64_t)positions[row] * rot;
  for (int i = threadIdx.x; i < rot / 2; i += NT)
    rotate_pair(p + kv_rank + 2 * i, dst + kv_rank + 2 * i, cs + 2 * i);
}

// The same by pieces of 8 channels, PIECES per thread at most: both sums are of what is
// then in registers (50 rows of 1536 + 512 + 64: 6.5 us a channel at a time).
constexpr int PIECES = 4;
__global__ __launch_bounds__(NT) void latent_prep_vec_kernel(
    const short* __restrict__ proj, int64_t pstride,
    const float* __restrict__ wq, const float* __restrict__ wkv,
    const float* __restrict__ cos_sin, const int32_t* __restrict__ positions,
    const int64_t* __restrict__ slots, short* __restrict__ cq,
    short* __restrict__ cache, int q_rank, int kv_rank, int rot, float eps) {
  __shared__ float red[2][NWV];
  const int64_t row = blockIdx.x;
  const short* p = proj + row * pstride;
  const int all = (cache ? q_rank + kv_rank + rot : q_rank) / 8;
  float x[PIECES][8], sq = 0.f, skv = 0.f;
  const int64_t slot = cache ? slots[row] : 0;
  const float* cs = cos_sin + (cache ? (int64_t)positions[row] * rot : 0);
#pragma unroll
  for (int i = 0; i < PIECES; ++i) {
    const int c = threadIdx.x + i * NT;
    if (c < all) ldn<8>(p + c * 8, x[i]);
  }
#pragma unroll
  for (int i = 0; i < PIECES; ++i) {
    const int c = (threadIdx.x + i * NT) * 8;
    float ss = 0.f;
#pragma unroll
    for (int j = 0; j < 8; ++j) ss += x[i][j] * x[i][j];
    if (c < q_rank) sq += ss;
    else if (c < q_rank + kv_rank && c < all * 8) skv += ss;
  }
  const float iq =
      1.f / sqrtf(block_sum<NWV>(sq, red[0]) / (float)q_rank + eps);
  const float ikv =
      cache ? 1.f / sqrtf(block_sum<NWV>(skv, red[1]) / (float)kv_rank + eps) : 0.f;
  short* dst = cache + slot * (kv_rank + rot);
#pragma unroll
  for (int i = 0; i < PIECES; ++i) {
    int c = (threadIdx.x + i * NT) * 8;
    if (c >= all * 8) break;
    float w[8], f[8];
    if (c < q_rank) {
      ldn<8>(wq + c, w);
#pragma unroll
      for (int j = 0; j < 8; ++j) f[j] = x[i][j] * iq * w[j];
      stn<8>(cq + row * q_rank + c, f);
      continue;
    }
    c -= q_rank;
    if (c < kv_rank) {
      ldn<8>(wkv + c, w);
#pragma unroll
      for (int j = 0; j < 8; ++j) f[j] = x[i][j] * ikv * w[j];
    } else {
      ldn<8>(cs + c - kv_rank, w);
#pragma unroll
      for (int j = 0; j < 8; j += 2) {
        f[j] = x[i][j] * w[j] - x[i][j + 1] * w[j + 1];
        f[j + 1] = x[i][j + 1] * w[j] + x[i][j] * w[j + 1];
      }
    }
    stn<8>(dst + c, f);
  }
}

// In place on the rotated part of q [rows, H, D + rot]; the unrotated part
// of the first n_abs rows is laid out by head for the absorbing product.
template <typename T>
__global__ __launch_bounds__(NT) void rope_part_kernel(
    T* __restrict__ q, T* __restrict__ by_head,  // [H, n_abs, D]
    const float* __restrict__ cos_sin, const int32_t* __restrict__ positions,
    int n_abs, int H, int D, int rot) {
  const int64_t row = blockIdx.x;
  T* qr = q + row * H * (D + rot);
  const float* cs = cos_sin + (int64_t)positions[row] * rot;
  const int half = rot / 2;
  for (int i = threadIdx.x; i < H * half; i += NT) {
    const int h = i / half, d = i % half;
    T* p = qr + (int64_t)h * (D + rot) + D + 2 * d;
    rotate_pair(p, p, cs + 2 * d);
  }
  if (row < n_abs) {
    for (int i = threadIdx.x; i < H * D; i += NT) {
      const int h = i / D, d = i % D;
      by_head[((int64_t)h * n_abs + row) * D + d] =
          qr[(int64_t)h * (D + rot) + d];
    }
  }
}

// The same by pieces of 8 channels: those to be rotated, then those to be laid out (50
// rows of 32 heads of 128 + 64: 6.5 us a row per workgroup, a channel at a time).
__global__ __launch_bounds__(NT) void rope_part_vec_kernel(
    short* __restrict__ q, short* __restrict__ by_head,
    const float* __restrict__ cos_sin, const int32_t* __restrict__ positions,
    int64_t rows, int64_t n_abs, int H, int D, int rot) {
  const int turn = rot / 8, lay = D / 8;
  const int64_t turned = rows * H * turn;
  int64_t i = (int64_t)blockIdx.x * NT + threadIdx.x;
  if (i < turned) {
    const int64_t rh = i / turn, row = rh / H;
    const int d = (int)(i % turn) * 8;
    short* p = q + rh * (D + rot) + D + d;
    float x[8], w[8], f[8];
    ldn<8>(p, x);
    ldn<8>(cos_sin + (int64_t)positions[row] * rot + d, w);
#pragma unroll
    for (int j = 0; j < 8; j += 2) {
      f[j] = x[j] * w[j] - x[j + 1] * w[j + 1];
      f[j + 1] = x[j + 1] * w[j] + x[j] * w[j + 1];
    }
    stn<8>(p, f);
    return;
  }
  i -= turned;
  if (i >= n_abs * H * lay) return;
  const int64_t rh = i / lay, row = rh / H, h = rh % H;
  const int d = (int)(i % lay) * 8;
  *(short8*)(by_head + (h * n_abs + row) * D + d) =
      *(const short8*)(q + rh * (D + rot) + d);
}

// [H, n_abs, V] -> rows of [.., H V]
template <typename T>
__global__ __launch_bounds__(NT) void heads_to_rows_kernel(
    const T* __restrict__ src, T* __restrict__ dst, int n_abs, int H, int V) {
  const int64_t row = blockIdx.x;
  for (int i = threadIdx.x; i < H * V; i += NT)
    dst[row * H * V + i] = src[((int64_t)(i / V) * n_abs + row) * V + i % V];
}

// y[t][h] = x[t][h] w[h]' for few rows t of every head (bf16, 32-bit sums): the products
// around latent decode attention. A head's weights are small, so what a launch takes is
// one way of loads: workgroups of 16 rows by 64 channels, whose four waves share K in
// steps of 128, or the channels where K is short, load everything of a step by 256 bytes
// of a row at once. 32 heads, 128 -> 512 and 512 -> 128: 1 row 3.3 and 3.6 us, 50 rows 3.7
// and 3.9 (the library's batched products 11.4 and 6.4), 256 rows 8.9 and 6.9, 512 rows
// 16.8 and 11.7.
struct HeadProducts {
  const short *x, *w;        // w [H, N, K]
  short* y;
  int64_t x_row, x_head, y_row, y_head;   // strides in elements
  int T, N, K;
};
template <int KW>            // waves that share K: 1, 2 or 4
__global__ __launch_bounds__(256) void head_products_kernel(const HeadProducts p) {
  typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
  typedef __attribute__((ext_vector_type(4))) __bf16 bf16x4;
  __shared__ __align__(16) char lds[4 * 4096];   // 4 KB of a wave; then the waves' sums
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
  const int lane = threadIdx.x % WAVE, col = lane % 16, grp = lane / 16;
  const int kw = wave % KW, c0 = wave / KW * KW;         // of the 64 channels, by 16
  const int n0 = blockIdx.x * 64, h = blockIdx.y, t0 = blockIdx.z * 16;
  const int N = p.N, K = p.K;
  const short* const x = p.x + (int64_t)t0 * p.x_row + h * p.x_head;
  const short* const w = p.w + (int64_t)h * N * K;
  char* const mine = lds + wave * 4096;
  const short8 zero = {0, 0, 0, 0, 0, 0, 0, 0};
  const int last = min(p.T - 1 - t0, 15);
  float4v acc[KW];
#pragma unroll
  for (int c = 0; c < KW; ++c) acc[c] = (float4v){0.f, 0.f, 0.f, 0.f};
  // past the end of K both count as zero (a weight may be infinite); rows and channels
  // past the end repeat the last one
  for (int k0 = kw * 128; k0 < K; k0 += KW * 128) {
    short8 a[4], b[KW][4];
    const int k = k0 + col * 8, kc = min(k, K - 8);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int r = j * 4 + grp;
      a[j] = *(const short8*)(x + min(r, last) * p.x_row + kc);
#pragma unroll
      for (int c = 0; c < KW; ++c)
        b[c][j] = *(const short8*)(
            w + (int64_t)min(n0 + (c0 + c) * 16 + r, N - 1) * K + kc);
    }
    __builtin_amdgcn_sched_barrier(0);       // all loads ahead of their first use
    if (k >= K)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        a[j] = zero;
#pragma unroll
        for (int c = 0; c < KW; ++c) b[c][j] = zero;
      }
    to_operand(mine, lane, a);
#pragma unroll
    for (int c = 0; c < KW; ++c) {
      to_operand(mine, lane, b[c]);
#pragma unroll
      for (int f = 0; f < 4; ++f)
        acc[c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
            __builtin_bit_cast(bf16x8, b[c][f]), __builtin_bit_cast(bf16x8, a[f]),
            acc[c], 0, 0, 0);
    }
  }
  // wave: 16 channels of the sums
  float4v sum = acc[0];
  if constexpr (KW > 1) {
    float4v* const sums = (float4v*)lds;
    __syncthreads();
#pragma unroll
    for (int c = 0; c < KW; ++c) sums[(kw * 4 + c0 + c) * WAVE + lane] = acc[c];
    __syncthreads();
    sum = sums[wave * WAVE + lane];
#pragma unroll
    for (int v = 1; v < KW; ++v) sum += sums[(v * 4 + wave) * WAVE + lane];
  }
  const int n = n0 + wave * 16 + grp * 4;
  if (col <= last && n < N)
    *(bf16x4*)(p.y + (int64_t)(t0 + col) * p.y_row + h * p.y_head + n) =
        __builtin_convertvector(sum, bf16x4);
}

// rows of the cache at `slots`, contiguous; unit: bytes moved per lane
template <typename U>
__global__ __launch_bounds__(NT) void gather_rows_kernel(
    const U* __restrict__ cache, const int64_t* __restrict__ slots,
    U* __restrict__ out, int64_t rows, int width) {
  const int64_t total = rows * width;
  for (int64_t i = (int64_t)blockIdx.x * NT + threadIdx.x; i < total;
       i += (int64_t)gridDim.x * NT)
    out[i] = cache[slots[i / width] * width + i % width];
}

// Keys and values as the plain kernel sees them: score = qa.ka + qb.kb.
// Strides in elements; a token is a row of a page (block table given) or a
// context row. `rep` query heads share a key/value head.
template <typename T>
struct View {
  const T *qa, *qb, *ka, *kb, *v;
  int64_t qa_row, qa_head, qb_row, qb_head;
  int64_t ka_tok, ka_head, kb_tok, v_tok, v_head, page;
  int da, db, dv, rep;
  int has_sink;
  float sink;                    // score of a key without a value
};

// One workgroup per (head, row).
//   paged: keys of positions (pos - window, pos] through the block table
//   else:  ctx [n_seqs, 2] = first context row, its position
template <typename T, int MAXV>
__global__ __launch_bounds__(NT) void attn_rows_kernel(
    View<T> a, const int32_t* __restrict__ positions,
    const int32_t* __restrict__ row_seq, int row_base,
    const int32_t* __restrict__ block_tables, int max_blocks, int block_size,
    const int32_t* __restrict__ ctx, int window, float scale,
    T* __restrict__ out, int64_t o_row, int64_t o_head) {
  extern __shared__ float qv[];  // da + db
  __shared__ float p[NT], redm[NWV], reds[NWV];
  const int h = blockIdx.x, kvh = h / a.rep;
  const int64_t i = blockIdx.y;       // row of q and out
  const int64_t row = row_base + i;   // row of the batch
  const int seq = row_seq[row];
  const int pos = positions[row];
  const int lo = window > 0 && pos + 1 > window ? pos + 1 - window : 0;
  const int32_t* bt =
      block_tables ? block_tables + (int64_t)seq * max_blocks : nullptr;
  const int64_t shift =
      bt ? 0 : (int64_t)ctx[2 * seq] - ctx[2 * seq + 1];
  // element offset of a token whose rows are `stride` apart
  auto at = [&](int t, int64_t stride) -> int64_t {
    return bt ? bt[t / block_size] * a.page + t % block_size * stride
              : (t + shift) * stride;
  };
  for (int d = threadIdx.x; d < a.da; d += NT)
    qv[d] = ld(a.qa + i * a.qa_row + h * a.qa_head + d);
  for (int d = threadIdx.x; d < a.db; d += NT)
    qv[a.da + d] = ld(a.qb + i * a.qb_row + h * a.qb_head + d);
  float acc[MAXV];
#pragma unroll
  for (int j = 0; j < MAXV; ++j) acc[j] = 0.f;
  float m = a.has_sink ? a.sink : -INFINITY, l = a.has_sink ? 1.f : 0.f;
  for (int t0 = lo; t0 <= pos; t0 += NT) {
    __syncthreads();
    const int t = t0 + threadIdx.x;
    float s = -INFINITY;
    if (t <= pos) {
      const T* ka = a.ka + at(t, a.ka_tok) + kvh * a.ka_head;
      const T* kb = a.kb + at(t, a.kb_tok);
      float dot = 0.f;
      for (int d = 0; d < a.da; ++d) dot += qv[d] * ld(ka + d);
      for (int d = 0; d < a.db; ++d) dot += qv[a.da + d] * ld(kb + d);
      s = dot * scale;
    }
    float mx = wave_reduce_max(s);
    if (threadIdx.x % WAVE == 0) redm[threadIdx.x / WAVE] = mx;
    __syncthreads();
#pragma unroll
    for (int w = 0; w < NWV; ++w) mx = fmaxf(mx, redm[w]);
    const float mn = fmaxf(m, mx);      // finite: key lo..pos is not empty
    const float alpha = expf(m - mn);   // 0 at the first tile without a sink
    const float e = t <= pos ? expf(s - mn) : 0.f;
    p[threadIdx.x] = e;
    l = l * alpha + block_sum<NWV>(e, reds);
    m = mn;
    const int n = min(NT, pos + 1 - t0);
#pragma unroll
    for (int j = 0; j < MAXV; ++j) {
      const int d = threadIdx.x + j * NT;
      if (d < a.dv) {
        float o = acc[j] * alpha;
        for (int x = 0; x < n; ++x)
          o += p[x] * ld(a.v + at(t0 + x, a.v_tok) + kvh * a.v_head + d);
        acc[j] = o;
      }
    }
  }
#pragma unroll
  for (int j = 0; j < MAXV; ++j) {
    const int d = threadIdx.x + j * NT;
    if (d < a.dv) st(out + i * o_row + h * o_head + d, acc[j] / l);
  }
}

// rows [.., keys of all heads | values of all heads] from column 0 of kv on
// -> pages [NB, G, bs, D + V]; U: the unit moved per lane
template <typename U>
__global__ __launch_bounds__(NT) void store_heads_kernel(
    const U* __restrict__ kv, int64_t stride,
    const int64_t* __restrict__ slots, U* __restrict__ cache, int64_t rows,
    int G, int bs, int D, int V) {
  const int W = D + V, width = G * W;
  const int64_t total = rows * width;
  for (int64_t i = (int64_t)blockIdx.x * NT + threadIdx.x; i < total;
       i += (int64_t)gridDim.x * NT) {
    const int64_t row = i / width, slot = slots[row];
    const int c = (int)(i % width), g = c / W, d = c % W;
    cache[((slot / bs * G + g) * bs + slot % bs) * W + d] =
        kv[row * stride + (d < D ? g * D + d : G * D + g * V + (d - D))];
  }
}

// The same of rows [queries | keys | values] that are in parts of 32 bits (rows apart by P
// channels, the parts by all of them): their sums, rounded to bf16; the queries, col
// channels, go to q. A launch of its own for the sums took as long again (60 rows of 6144
// in 5 parts: 4.7 + 4.2 us, so 5.2).
__global__ __launch_bounds__(NT) void store_heads_parts_kernel(
    const float* __restrict__ part, int parts, int P, int col,
    const int64_t* __restrict__ slots, short* __restrict__ q,
    short* __restrict__ cache, int64_t rows, int G, int bs, int D, int V) {
  const int W = D + V, pieces = (col + G * W) / 8;
  const int64_t i = (int64_t)blockIdx.x * NT + threadIdx.x;
  if (i >= rows * pieces) return;
  const int64_t row = i / pieces;
  const int c = (int)(i % pieces) * 8;
  const float4v* const src[1] = {(const float4v*)(part + row * P + c)};
  float f[8];
  PartSums<1>(src, rows * P / 4, parts).get(0, f);
  short* to = q + row * col + c;
  if (c >= col) {
    const int64_t slot = slots[row];
    const int x = c - col, v = x - G * D;       // of all heads' keys, of their values
    const int g = v < 0 ? x / D : v / V, d = v < 0 ? x % D : D + v % V;
    to = cache + ((slot / bs * G + g) * bs + slot % bs) * W + d;
  }
  stn<8>(to, f);
}

template <typename T>
hipError_t attn_rows_t(const void* const* ptr, const int64_t* stride, int da,
                       int db, int dv, int rep, int has_sink, float sink,
                       const int32_t* positions, const int32_t* row_seq,
                       int row_base, const int32_t* block_tables,
                       int max_blocks, int block_size, const int32_t* ctx,
                       int window, float scale, void* out, int64_t o_row,
                       int64_t o_head, int rows, int H, hipStream_t stream) {
  View<T> a{(const T*)ptr[0], (const T*)ptr[1], (const T*)ptr[2],
            (const T*)ptr[3], (const T*)ptr[4],
            stride[0], stride[1], stride[2], stride[3], stride[4], stride[5],
            stride[6], stride[7], stride[8], stride[9], da, db, dv, rep,
            has_sink, sink};
  if (dv > 8 * NT || da + db > 8192) return hipErrorInvalidValue;
  const size_t lds = (size_t)(da + db) * sizeof(float);
  const dim3 block(NT);
  for (int r = 0; r < rows; r += 32768) {  // grid.y limit
    const int n = rows - r < 32768 ? rows - r : 32768;
    const dim3 grid(H, n);
    View<T> b = a;
    b.qa += r * a.qa_row;
    b.qb += r * a.qb_row;
    T* o = (T*)out + r * o_row;
#define GO(M)                                                                 \
  hipLaunchKernelGGL((attn_rows_kernel<T, M>), grid, block, lds, stream, b,   \
                     positions, row_seq, row_base + r, block_tables,          \
                     max_blocks, block_size, ctx, window, scale, o, o_row,    \
                     o_head)
    if (dv <= NT) GO(1); else if (dv <= 2 * NT) GO(2); else GO(8);
#undef GO
  }
  HIP_CHECK_LAST();
  return hipSuccess;
}

}  // namespace

extern "C" {

hipError_t lds_latent_prep(int f32, const void* proj, int64_t pstride,
                           const float* wq, const float* wkv,
                           const float* cos_sin, const int32_t* positions,
                           const int64_t* slots, void* cq, void* cache,
                           int rows, int q_rank, int kv_rank, int rot,
                           float eps, hipStream_t stream) {
  if (rows == 0) return hipSuccess;
  const auto at16 = [](const void* p) { return (uintptr_t)p % 16 == 0; };
  if (!f32 && pstride % 8 == 0 && q_rank % 8 == 0 && kv_rank % 8 == 0 &&
      rot % 8 == 0 && q_rank + kv_rank + rot <= PIECES * NT * 8 && at16(proj) &&
      at16(wq) && at16(wkv) && at16(cos_sin) && at16(cq) && at16(cache)) {
    hipLaunchKernelGGL(latent_prep_vec_kernel, dim3(rows), dim3(NT), 0, stream,
                       (const short*)proj, pstride, wq, wkv, cos_sin, positions,
                       slots, (short*)cq, (short*)cache, q_rank, kv_rank, rot,
                       eps);
    HIP_CHECK_LAST();
    return hipSuccess;
  }
#define GO(T)                                                                 \
  hipLaunchKernelGGL(latent_prep_kernel<T>, dim3(rows), dim3(NT), 0, stream,  \
                     (const T*)proj, pstride, wq, wkv, cos_sin, positions,    \
                     slots, (T*)cq, (T*)cache, q_rank, kv_rank, rot, eps)
  if (f32) GO(float); else GO(short);
#undef GO
  HIP_CHECK_LAST();
  return hipSuccess;
}

hipError_t lds_rope_part(int f32, void* q, void* by_head, const float* cos_sin,
                         const int32_t* positions, int rows, int n_abs, int H,
                         int D, int rot, hipStream_t stream) {
  if (rows == 0) return hipSuccess;
  const int64_t pieces =
      ((int64_t)rows * H * rot + (int64_t)n_abs * H * D) / 8, blocks = (pieces + NT - 1) / NT;
  const auto at16 = [](const void* p) { return (uintptr_t)p % 16 == 0; };
  if (!f32 && D % 8 == 0 && rot % 8 == 0 && blocks <= 0x7fffffff && at16(q) &&
      at16(by_head) && at16(cos_sin)) {
    if (blocks)
      hipLaunchKernelGGL(rope_part_vec_kernel, dim3((uint32_t)blocks), dim3(NT), 0,
                         stream, (short*)q, (short*)by_head, cos_sin, positions,
                         rows, n_abs, H, D, rot);
    HIP_CHECK_LAST();
    return hipSuccess;
  }
#define GO(T)                                                                 \
  hipLaunchKernelGGL(rope_part_kernel<T>, dim3(rows), dim3(NT), 0, stream,    \
                     (T*)q, (T*)by_head, cos_sin, positions, n_abs, H, D, rot)
  if (f32) GO(float); else GO(short);
#undef GO
  HIP_CHECK_LAST();
  return hipSuccess;
}

hipError_t lds_heads_to_rows(int f32, const void* src, void* dst, int n_abs,
                             int H, int V, hipStream_t stream) {
  if (n_abs == 0) return hipSuccess;
#define GO(T)                                                                 \
  hipLaunchKernelGGL(heads_to_rows_kernel<T>, dim3(n_abs), dim3(NT), 0,       \
                     stream, (const T*)src, (T*)dst, n_abs, H, V)
  if (f32) GO(float); else GO(short);
#undef GO
  HIP_CHECK_LAST();
  return hipSuccess;
}

// x, y: rows and heads apart by strides of 4 elements and more, 16 and 8 bytes aligned; N
// and K multiples of 8
hipError_t lds_head_products(const void* x, int64_t x_row, int64_t x_head, const void* w,
                             void* y, int64_t y_row, int64_t y_head, int T, int H, int N,
                             int K, hipStream_t stream) {
  if (T == 0) return hipSuccess;
  if (N < 8 || N % 8 || K < 8 || K % 8 || x_row % 8 || x_head % 8 || y_row % 4 ||
      y_head % 4 || T > 16 * 65535 || H > 65535)
    return hipErrorInvalidValue;
  const HeadProducts p{(const short*)x, (const short*)w, (short*)y, x_row, x_head,
                       y_row, y_head, T, N, K};
  const dim3 grid((N + 63) / 64, H, (T + 15) / 16);
  if (K <= 128)
    hipLaunchKernelGGL(head_products_kernel<1>, grid, dim3(256), 0, stream, p);
  else if (K <= 256)
    hipLaunchKernelGGL(head_products_kernel<2>, grid, dim3(256), 0, stream, p);
  else
    hipLaunchKernelGGL(head_products_kernel<4>, grid, dim3(256), 0, stream, p);
  HIP_CHECK_LAST();
  return hipSuccess;
}

hipError_t lds_gather_rows(const void* cache, const int64_t* slots, void* out,
                           int64_t rows, int64_t row_bytes,
                           hipStream_t stream) {
  if (rows == 0) return hipSuccess;
  const int unit = row_bytes % 16 == 0 ? 16 : row_bytes % 4 == 0 ? 4 : 2;
  if (row_bytes % unit) return hipErrorInvalidValue;
  const int width = (int)(row_bytes / unit);
  int64_t blocks = (rows * width + NT - 1) / NT;
  if (blocks > 4096) blocks = 4096;
#define GO(U)                                                                 \
  hipLaunchKernelGGL(gather_rows_kernel<U>, dim3((uint32_t)blocks), dim3(NT), \
                     0, stream, (const U*)cache, slots, (U*)out, rows, width)
  if (unit == 16) GO(short8); else if (unit == 4) GO(float); else GO(short);
#undef GO
  HIP_CHECK_LAST();
  return hipSuccess;
}

// ptr: qa, qb, ka, kb, v; stride: qa row/head, qb row/head, ka token/head,
// kb token, v token/head, page (elements)
hipError_t lds_attn_rows(int f32, const void* const* ptr,
                         const int64_t* stride, int da, int db, int dv,
                         int rep, int has_sink, float sink,
                         const int32_t* positions, const int32_t* row_seq,
                         int row_base, const int32_t* block_tables,
                         int max_blocks, int block_size, const int32_t* ctx,
                         int window, float scale, void* out, int64_t o_row,
                         int64_t o_head, int rows, int H,
                         hipStream_t stream) {
  if (rows == 0) return hipSuccess;
  auto fn = f32 ? attn_rows_t<float> : attn_rows_t<short>;
  return fn(ptr, stride, da, db, dv, rep, has_sink, sink, positions, row_seq,
            row_base, block_tables, max_blocks, block_size, ctx, window, scale,
            out, o_row, o_head, rows, H, stream);
}

// es: bytes per element
hipError_t lds_store_heads(const void* kv, int64_t stride,
                           const int64_t* slots, void* cache, int64_t rows,
                           int G, int bs, int D, int V, int es,
                           hipStream_t stream) {
  if (rows == 0) return hipSuccess;
  const int n = 16 / es;      // elements of a 16-byte unit
  const int u = D % n == 0 && V % n == 0 && stride % n == 0 &&
                        (uintptr_t)kv % 16 == 0
                    ? n
                    : 1;
  int64_t blocks = (rows * G * (D + V) / u + NT - 1) / NT;
  if (blocks > 4096) blocks = 4096;
#define GO(U)                                                                 \
  hipLaunchKernelGGL(store_heads_kernel<U>, dim3((uint32_t)blocks), dim3(NT), \
                     0, stream, (const U*)kv, stride / u, slots, (U*)cache,   \
                     rows, G, bs, D / u, V / u)
  if (u > 1) GO(short8); else if (es == 4) GO(float); else GO(short);
#undef GO
  HIP_CHECK_LAST();
  return hipSuccess;
}

// part [parts, rows, P]; q [rows, col]; bf16 cache. col, D and V in steps of 8.
hipError_t lds_store_heads_parts(const float* part, int parts, int P, int col,
                                 const int64_t* slots, void* q, void* cache,
                                 int64_t rows, int G, int bs, int D, int V,
                                 hipStream_t stream) {
  if (rows == 0) return hipSuccess;
  const int64_t blocks = (rows * ((col + G * (D + V)) / 8) + NT - 1) / NT;
  if (col % 8 || D % 8 || V % 8 || P % 8 || blocks > 0x7fffffff)
    return hipErrorInvalidValue;
  hipLaunchKernelGGL(store_heads_parts_kernel, dim3((uint32_t)blocks), dim3(NT),
                     0, stream, part, parts, P, col, slots, (short*)q,
                     (short*)cache, rows, G, bs, D, V);
  HIP_CHECK_LAST();
  return hipSuccess;
}

}  // extern "C"
