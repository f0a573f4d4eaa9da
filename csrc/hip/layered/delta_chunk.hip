// delta_chunk.hip — the gated delta rule of delta_rule.hip over chunks of 64
// tokens on the matrix cores, in 32-bit (v_mfma_f32_16x16x4f32) or, in the scan of
// many sequences, in bf16 with each value in three parts, 24 bits.
//
// With G the running sum of log decays inside a chunk (token's own included)
// and S0 the state before it, per head:
//   A[i][j] = sum_d k_i k_j e^(G_i - G_j)   (j < i)
//   P[i][j] = sum_d q_i k_j e^(G_i - G_j)   (j <= i)
//   (I + diag(beta) A) U = diag(beta) (V - (k e^G) S0)
//   O = (q e^G) S0 + P U,   S = e^(G_last) S0 + (k e^(G_last - G))' U
// A and P are products of scaled rows, in blocks of 16 tokens. The sum before
// the later block is the reference, so off the diagonal no exponent is positive.
// On the diagonal they are up to e^24, as long as no channel decays by more than
// that inside a block (every term has its own relative error, whatever the
// reference); else every pair is taken by itself. So any decay down to 0 is right.
//
// delta_chunk_local  everything that does not need S0, one workgroup per
//                    (head, chunk): U0 and W with U = U0 - W S0, P, the
//                    scaled q and k -> workspace
// delta_chunk_scan   one workgroup per (head, 16 or 32 columns of S, sequence)
//                    walks the chunks with S in LDS
// delta_gate         gated output norm
//
// MFMA operands: lane l gives A[l % 16][k] and B[k][l % 16] with k = l / 16,
// and holds D[4 (l / 16) + r][l % 16] in register r. Taking k = 4 (l / 16) + r
// in step r instead makes a D tile usable as B as it is, and an A operand one
// 16-byte read per four steps.
#include "elem.h"

namespace {

constexpr int BUFFER_BYTES = 0x00027000;       // fourth word of a buffer: raw bytes
constexpr int C = 64;       // tokens per chunk
constexpr int B = 16;       // tokens per block
constexpr int LT = 512;     // threads of delta_chunk_local
constexpr int ST = 256;     // threads of delta_chunk_scan

__device__ __forceinline__ float4v mfma4(float4v a, float4v b, float4v c) {
#pragma unroll
  for (int r = 0; r < 4; ++r)
    c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[r], b[r], c, 0, 0, 0);
  return c;
}

// Workspace of one (chunk, head), floats; KP, VP: sizes rounded up. All but
// gl are 16 x 16 tiles in operand order (256 floats, 4 per lane: the scan
// reads a kilobyte per instruction):
//   u0 [VP / 16][4]       D: lane (c, g) holds tokens 4 g .. of channel c
//   w, qe [4][KP / 16]    A: lane (t, g) holds channels 4 g .. of token t
//   kt [KP / 16][4]       A: lane (c, g) holds tokens 4 g .. of channel c
//   p [4][4]              A: lane (t, g) holds columns 4 g .. of token t
struct Work {
  float *u0, *w, *qe, *kt, *p, *gl;
};
__host__ __device__ __forceinline__ int64_t work_size(int KP, int VP) {
  return (int64_t)C * VP + 3 * C * KP + C * C + KP;
}
__device__ __forceinline__ Work work_at(float* ws, int64_t i, int KP, int VP) {
  float* p = ws + i * work_size(KP, VP);
  return {p, p + C * VP, p + C * VP + C * KP, p + C * VP + 2 * C * KP,
          p + C * VP + 3 * C * KP, p + C * VP + 3 * C * KP + C * C};
}

// 4 channels from p, of which the first `left` exist; `whole` rows only hold
// multiples of 4 (and are aligned)
__device__ __forceinline__ float4v load4(const float* p, int left,
                                         bool whole) {
  float4v f = {0.f, 0.f, 0.f, 0.f};
  if (whole) {
    if (left > 0) f = *(const float4v*)p;
  } else {
#pragma unroll
    for (int x = 0; x < 4; ++x)
      if (x < left) f[x] = p[x];
  }
  return f;
}
__device__ __forceinline__ float4v load4(const short* p, int left,
                                         bool whole) {
  float4v f = {0.f, 0.f, 0.f, 0.f};
  if (whole) {
    if (left > 0) {
      const short4v v = *(const short4v*)p;
#pragma unroll
      for (int x = 0; x < 4; ++x) f[x] = bf16_to_f32(v[x]);
    }
  } else {
#pragma unroll
    for (int x = 0; x < 4; ++x)
      if (x < left) f[x] = bf16_to_f32(p[x]);
  }
  return f;
}

constexpr float LOG2E = 1.4426950408889634f;
constexpr float DECAY_LIMIT = 24.f * LOG2E;    // of a block, in powers of two
// beta A in LDS, 16 x 16 blocks of the lower triangle: groups of 4 columns change
// places by XOR with the row, so that 16 rows' groups meet all banks
constexpr int AB = B * B;
__device__ __forceinline__ int block_at(int bi, int bj) {
  return (bi * (bi + 1) / 2 + bj) * AB;
}
__device__ __forceinline__ int group_at(int r, int g) {
  return r * B + (g ^ (r / 4)) * 4;
}
__device__ __forceinline__ float exp2_f(float x) {
  return __builtin_amdgcn_exp2f(x);
}

// channels d .. d + 3 of a row of K: past the end the last ones, which come() drops.
// No load is under a condition, so that the compiler can count those under way.
template <typename T> struct Raw;
template <> struct Raw<float> { typedef float4v type; };
template <> struct Raw<short> { typedef short4v type; };
template <typename T>
__device__ __forceinline__ typename Raw<T>::type ask4(const T* row, int d, int K,
                                                      bool whole) {
  typedef typename Raw<T>::type Four;
  if (whole) return *(const Four*)(row + min(d, K - 4));
  Four f;
#pragma unroll
  for (int x = 0; x < 4; ++x) f[x] = row[min(d + x, K - 1)];
  return f;
}
template <typename F>
__device__ __forceinline__ float4v come(F f, bool in, int d, int K) {
  float4v o;
#pragma unroll
  for (int x = 0; x < 4; ++x) {
    float v;
    if constexpr (sizeof(F) == 16) v = f[x]; else v = bf16_to_f32(f[x]);
    o[x] = in && d + x < K ? v : 0.f;
  }
  return o;
}

// grid (H, chunks); chunks [n, 2] = first row, tokens. Everything the waves
// share goes through LDS (80 KB: two workgroups per CU), so its barriers let
// global loads and stores run on.
//
// Decays are powers of two and taken once per token and channel: with g the sum
// inside a block up to the token, t the block's whole sum, LDS keeps k 2^g, k
// 2^(t - g) and 2^t, and all else is products of these. Four waves do the blocks
// of A, each 16 tokens' row of them and its diagonal block's inverse, four those
// of P, the longest of these beside the shortest of those on a SIMD; operands of
// the row stay in registers, and results come out turned, whole groups of 4.
// Loads of q and v are under way a phase ahead. What bounds it is no one thing:
// loads and stores take half of a workgroup's 67000 cycles (260 KB each, 3.4 TB/s
// over the chip), matrix instructions a third; with decays taken per pair of
// blocks, references in the middle of diagonal ones and results stored one value
// at a time it was 105000. 1024 chunks of 32 heads of 128 x 128, with the scan:
// 197 -> 166 us; here alone, in a pass, 128 -> 101. Steep blocks take half as long again.
template <typename T, int KP>
__global__ __launch_bounds__(LT, 4) void delta_chunk_local_kernel(
    const float* __restrict__ q, const float* __restrict__ k,
    const float* __restrict__ v, const T* __restrict__ beta, int64_t bstride,
    const T* __restrict__ decay, const float* __restrict__ dt_bias,
    const float* __restrict__ neg_a, const int32_t* __restrict__ chunks,
    float* __restrict__ ws, int KH, int H, int K, int V, int VP) {
  constexpr int LD = KP + 4;          // row stride in LDS
  constexpr int NT = KP / 16;
  extern __shared__ float lds[];
  float* kl = lds;                    // [C][LD]: k, then k 2^g
  float* gl = kl + C * LD;            // [C][LD]: g, then k 2^(t - g)
  float* tl = gl + C * LD;            // [4][KP]: 2^t
  float* al = tl + 4 * KP;            // beta A, lower blocks; the diagonal
                                      // ones become their inverses
  float* bl = al + 10 * AB;           // beta [C]
  int* steep = (int*)(bl + C);        // per wave: a block decays too much
  const int h = blockIdx.x;
  const int kh = h / (H / KH);
  const int64_t row0 = chunks[2 * blockIdx.y];
  const int n = chunks[2 * blockIdx.y + 1];
  const Work wk = work_at(ws, (int64_t)blockIdx.y * H + h, KP, VP);
  const int tid = threadIdx.x, lane = tid % WAVE;
  const int wave = __builtin_amdgcn_readfirstlane(tid / WAVE);
  const int col = lane % 16, g4 = 4 * (lane / 16);
  // bases of this chunk and head; offsets from them fit 32 bits
  const float* kc = k + (row0 * KH + kh) * K;
  const float* qc = q + (row0 * KH + kh) * K;
  const float* vc = v + (row0 * H + h) * V;
  const T* dc = decay + (row0 * H + h) * K;
  const unsigned krow = KH * K, drow = H * K, vrow = H * V;
  const bool whole = K % 4 == 0;
  // the wave's 16 tokens: waves 0 to 3 have their rows of A, 7 to 4 of P
  const bool of_p = wave >= 4;
  const int bi = of_p ? 7 - wave : wave, mine = bi * B + col;

  // ---- load; rows and channels past the end are zero. All loads of a
  // thread are under way before the first is used ----
  constexpr int Q4 = C * KP / 4 / LT;            // groups of 4 channels
  const int d4 = tid % (KP / 4) * 4, t4 = tid / (KP / 4);
  float4v row[NT];                               // of q or k; later times 2^g
  {
    float4v kr[Q4], bias;
    typename Raw<T>::type dr[Q4];
    if (of_p) {
      const float* qrow = qc + (unsigned)min(mine, n - 1) * krow;
#pragma unroll
      for (int t = 0; t < NT; ++t) row[t] = ask4(qrow, 16 * t + g4, K, whole);
    }
    const float na = neg_a[h] * LOG2E;
    const float b0 = ld(beta + (row0 + min(tid % C, n - 1)) * bstride + h);
    bias = ask4(dt_bias + (int64_t)h * K, d4, K, whole);
#pragma unroll
    for (int i = 0; i < Q4; ++i) {
      const unsigned t = min(t4 + i * (LT * 4 / KP), n - 1);
      dr[i] = ask4(dc + t * drow, d4, K, whole);
      kr[i] = ask4(kc + t * krow, d4, K, whole);
    }
    __builtin_amdgcn_sched_barrier(0);
    if (tid < C) bl[tid] = tid < n ? sigmoid_f(b0) : 0.f;
#pragma unroll
    for (int i = 0; i < Q4; ++i) {
      const int t = t4 + i * (LT * 4 / KP);
      const float4v d = come(dr[i], t < n, d4, K);
      float4v gv;
#pragma unroll
      for (int x = 0; x < 4; ++x)
        gv[x] = t < n && d4 + x < K ? na * softplus_f(d[x] + bias[x]) : 0.f;
      *(float4v*)(kl + t * LD + d4) = come(kr[i], t < n, d4, K);
      *(float4v*)(gl + t * LD + d4) = gv;
    }
  }
  lds_barrier();
  // ---- running sums inside blocks of 16: differences of small sums stay
  // exact where a chunk's whole sum would have swallowed them ----
  static_assert(4 * KP <= LT, "one pass");
  const bool has = tid < 4 * KP;                 // wave-uniform
  const int column = tid / KP % 4 * B * LD + tid % KP;
  bool over = false;
  if (has) {
    float sum[B];
#pragma unroll
    for (int t = 0; t < B; ++t) sum[t] = gl[column + t * LD];
#pragma unroll
    for (int t = 1; t < B; ++t) {
      sum[t] += sum[t - 1];
      gl[column + t * LD] = sum[t];
    }
    tl[tid] = exp2_f(sum[B - 1]);
    over = sum[B - 1] < -DECAY_LIMIT;
  }
  {
    const bool any = __any(over);
    if (lane == 0) steep[wave] = any;
  }
  lds_barrier();
  bool slow = false;
#pragma unroll
  for (int w = 0; w < LT / WAVE; ++w) slow |= steep[w] != 0;
  slow = __builtin_amdgcn_readfirstlane(slow);

  // ---- diagonal blocks pair by pair: 8 threads share token i ----
  const int di = tid / 8, ds = tid % 8;          // token, slice
  constexpr int DS = KP / 32;                    // its groups of 4 channels
  float pk[2] = {0.f, 0.f};          // this thread's share of P's row
  if (slow) {
    const int i = di, s = ds, b0 = i / B * B;
    const int top = (wave * 8 + 7) % B + b0;   // largest token of the wave
    float4v gi[DS], ki[DS], qi[DS];
#pragma unroll
    for (int d = 0; d < DS; ++d) {
      gi[d] = *(const float4v*)(gl + i * LD + s * 4 + d * 32);
      ki[d] = *(const float4v*)(kl + i * LD + s * 4 + d * 32);
      qi[d] = load4(qc + i * krow + s * 4 + d * 32,
                    i < n ? K - s * 4 - d * 32 : 0, whole);
    }
    const float beta_i = bl[i];
    float* ab = al + block_at(i / B, i / B);
#pragma unroll 1
    for (int j = b0; j < b0 + B; ++j) {
      float a = 0.f, p = 0.f;
      if (j <= top) {                // wave-uniform
#pragma unroll
        for (int d = 0; d < DS; ++d) {
          const float4v gj = *(const float4v*)(gl + j * LD + s * 4 + d * 32);
          const float4v kj = *(const float4v*)(kl + j * LD + s * 4 + d * 32);
#pragma unroll
          for (int x = 0; x < 4; ++x) {
            // pairs with j > i are thrown away below; their exponent is cut
            const float e = exp2_f(fminf(gi[d][x] - gj[x], 0.f)) * kj[x];
            a += ki[d][x] * e;
            p += qi[d][x] * e;
          }
          __builtin_amdgcn_sched_barrier(0);   // keep the reads from taking
        }                                      // all registers
#pragma unroll
        for (int o = 1; o < 8; o *= 2) {
          a += __shfl_xor(a, o, WAVE);
          p += __shfl_xor(p, o, WAVE);
        }
      }
      if (s == 0)
        ab[group_at(i % B, (j - b0) / 4) + j % 4] = j < i ? beta_i * a : 0.f;
      p = j <= i ? p : 0.f;
      if (j - b0 == 2 * s) pk[0] = p;
      if (j - b0 == 2 * s + 1) pk[1] = p;
    }
  }
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    const int o = 16 * t + g4;
    const float4v g = *(const float4v*)(gl + mine * LD + o);
    row[t] = of_p ? come(row[t], mine < n, o, K)
                  : *(const float4v*)(kl + mine * LD + o);
#pragma unroll
    for (int x = 0; x < 4; ++x) row[t][x] *= exp2_f(g[x]);
  }
  float sum[B], kcol[B];
  if (has) {
#pragma unroll
    for (int t = 0; t < B; ++t) {
      sum[t] = gl[column + t * LD];
      kcol[t] = kl[column + t * LD];
    }
  }
  lds_barrier();
  if (has) {
#pragma unroll
    for (int t = 0; t < B; ++t) {
      kl[column + t * LD] = kcol[t] * exp2_f(sum[t]);
      gl[column + t * LD] = kcol[t] * exp2_f(sum[B - 1] - sum[t]);
    }
  }
  // Loads wait for the stores issued before them, so this wave's first tile
  // of v comes now and every store after it.
  float vpre[4][4];
#pragma unroll
  for (int b = 0; b < 4; ++b)
#pragma unroll
    for (int r = 0; r < 4; ++r)
      vpre[b][r] = vc[(unsigned)min(b * B + g4 + r, n - 1) * vrow +
                      min(wave * 16 + col, V - 1)];
  lds_barrier();

  // products of 2^t over the blocks b0 <= b < b1, of 4 channels or of one
  auto span4 = [&](int b0, int b1, int d) {
    float4v f = {1.f, 1.f, 1.f, 1.f};
    for (int b = b0; b < b1; ++b) f *= *(const float4v*)(tl + b * KP + d);
    return f;
  };
  auto span = [&](int b0, int b1, int d) {
    float f = 1.f;
    for (int b = b0; b < b1; ++b) f *= tl[b * KP + d];
    return f;
  };
  // ---- one block of the wave's row, turned: lane (i, g) has columns 4 g .. ----
  auto block = [&](int bj) -> float4v {
    float4v a = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const int o = 16 * t + g4;
      float4v kb = *(const float4v*)(gl + (bj * B + col) * LD + o);
      if (bi == bj) {                            // 2^-g_j, at most e^24
        const float4v f = *(const float4v*)(tl + bi * KP + o);
#pragma unroll
        for (int x = 0; x < 4; ++x) kb[x] *= rcp_f(f[x]);
      } else if (bi > bj + 1) {
        kb *= span4(bj + 1, bi, o);
      }
      a = mfma4(kb, row[t], a);
    }
    return a;
  };
  if (!of_p) {
    if (!slow) {
      float4v a = block(bi);
#pragma unroll
      for (int x = 0; x < 4; ++x)
        a[x] = g4 + x < col ? bl[mine] * a[x] : 0.f;
      *(float4v*)(al + block_at(bi, bi) + group_at(col, g4 / 4)) = a;
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    }
    // inverse of the unit lower triangular diagonal block, in place
    if (lane < B) {
      float* a = al + block_at(bi, bi);
      float x[B];
#pragma unroll
      for (int i = 0; i < B; ++i) {
        float s = i == lane ? 1.f : 0.f;
#pragma unroll
        for (int j = 0; j < i; ++j)
          s -= a[group_at(i, j / 4) + j % 4] * x[j];
        x[i] = s;
      }
#pragma unroll
      for (int i = 0; i < B; ++i) a[group_at(i, lane / 4) + lane % 4] = x[i];
    }
    for (int bj = 0; bj < bi; ++bj)
      *(float4v*)(al + block_at(bi, bj) + group_at(col, g4 / 4)) =
          bl[mine] * block(bj);
  } else {
    for (int bj = 0; bj < bi + !slow; ++bj) {
      float4v p = block(bj);
      if (bi == bj) {
#pragma unroll
        for (int x = 0; x < 4; ++x)
          if (g4 + x > col) p[x] = 0.f;
      }
      *(float4v*)(wk.p + (bi * 4 + bj) * 256 + lane * 4) = p;
    }
    // scaled q and k
#pragma unroll
    for (int t = 0; t < NT; ++t)
      *(float4v*)(wk.qe + (bi * NT + t) * 256 + lane * 4) =
          row[t] * span4(0, bi, 16 * t + g4);
    for (int tile = wave - 4; tile < 4 * NT; tile += 4) {
      const int d = tile / 4 * 16 + col, t = tile % 4 * 16 + g4;
      const float after = span(tile % 4 + 1, 4, d);
      float4v o;
#pragma unroll
      for (int x = 0; x < 4; ++x) o[x] = gl[(t + x) * LD + d] * after;
      *(float4v*)(wk.kt + tile * 256 + lane * 4) = o;
    }
  }
  if (slow) {
    float* o = wk.p + di / B * (4 + 1) * 256;     // tile (b, b)
    typedef __attribute__((ext_vector_type(2))) float f2;
    *(f2*)(o + (di % B + 16 * (ds / 2)) * 4 + ds % 2 * 2) =
        (f2){pk[0], pk[1]};
  }
  if (tid < KP) wk.gl[tid] = span(0, 4, tid);
  lds_barrier();

  // ---- forward substitution by blocks, 16 columns of [V | K] at a time ----
  for (int tile = wave; tile < (VP + KP) / 16; tile += LT / WAVE) {
    const bool is_v = tile < VP / 16;            // wave-uniform
    const int c = (is_v ? tile : tile - VP / 16) * 16 + col;
    float4v f[4], x[4];
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      const float before = is_v ? 1.f : span(0, b, c);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int t = b * B + g4 + r;
        if (!is_v)
          f[b][r] = -kl[t * LD + c] * before;
        else if (tile == wave)
          f[b][r] = t < n && c < V ? vpre[b][r] : 0.f;
        else
          f[b][r] = t < n && c < V ? vc[t * vrow + c] : 0.f;
      }
    }
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      float4v acc = *(const float4v*)(bl + b * B + g4) * f[b];
#pragma unroll
      for (int p = 0; p < b; ++p) {
        const float4v a =
            *(const float4v*)(al + block_at(b, p) + group_at(col, g4 / 4));
        acc = mfma4(-a, x[p], acc);
      }
      const float4v inv =
          *(const float4v*)(al + block_at(b, b) + group_at(col, g4 / 4));
      x[b] = mfma4(inv, acc, (float4v){0.f, 0.f, 0.f, 0.f});
      if (is_v) {
        *(float4v*)(wk.u0 + (tile * 4 + b) * 256 + lane * 4) = x[b];
      } else {
        // -W, turned by taking the last product the other way round
        *(float4v*)(wk.w + (b * NT + tile - VP / 16) * 256 + lane * 4) =
            mfma4(acc, inv, (float4v){0.f, 0.f, 0.f, 0.f});
      }
    }
  }
}

// grid (H, VP / (16 NC), sequences); walk [n, 4] = first row, tokens, slot,
// first chunk | (1 << 30 if the state starts at zero). A workgroup has NC tiles
// of 16 columns. S lies in LDS between the chunks, as operands; a wave keeps
// the tiles of it that it brings up to date, takes 16 tokens of the products
// with it, and asks for a chunk's operands of these during the chunk before.
//
// In 32-bit the matrix instructions bound it: 223 us of 297 for 16 chunks of 8
// sequences, 32 heads of 128 x 128. With two tiles values are sums of three bf16
// instead, six products of which take 3/8 of the time: 254 us, 172 of them with
// operands that are in cache, the error of outputs 3.52e-7 instead of 4.18e-7. Vector
// instructions bound it then, the splitting of operands first of them: with a rounded
// pair taken out of one word, operands by way of a buffer and no masks around whole
// chunks' stores it is 1500 instructions per chunk and wave (1970), 126 chunks of 8
// prompts in a pass 287 -> 253 us, the same bits.
// With one tile the splitting costs more than it saves (31 chunks of one sequence
// 112 us, in 32-bit 91); four tiles do not fit the registers (+ 7 %).
typedef __attribute__((ext_vector_type(8))) float float8v;
typedef __attribute__((ext_vector_type(4))) __bf16 bf16x4;
typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
template <int N> struct Vec;
template <> struct Vec<4> { typedef float4v F; typedef bf16x4 H; };
template <> struct Vec<8> { typedef float8v F; typedef bf16x8 H; };
// 32-bit values as sums of three bf16 (high, middle, low): 24 bits of them. Two at a
// time, the rounded values taken out of the word that holds both (converted back as
// vectors each is rounded once more by itself, 4 instructions of 15 per pair and part).
template <int N>
__device__ __forceinline__ void split(typename Vec<N>::F f,
                                      typename Vec<N>::H (&o)[3]) {
  typedef __attribute__((ext_vector_type(N / 2))) unsigned int Words;
  typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    Words w;
#pragma unroll
    for (int x = 0; x < N; x += 2) {
      const unsigned int two = __builtin_bit_cast(
          unsigned int, __builtin_convertvector((float2v){f[x], f[x + 1]}, bf16x2));
      w[x / 2] = two;
      f[x] -= __builtin_bit_cast(float, two << 16);
      f[x + 1] -= __builtin_bit_cast(float, two & 0xffff0000u);
    }
    o[i] = __builtin_bit_cast(typename Vec<N>::H, w);
  }
}
__device__ __forceinline__ void split2(float4v a, float4v b, bf16x8 (&o)[3]) {
  split<8>(__builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7), o);
}
// products of 32 k, without those below 2^-24 of the largest: a[i] b[term - i]
__device__ __forceinline__ float4v mfma_split(const bf16x8 (&a)[3],
                                              const bf16x8 (&b)[3],
                                              float4v c) {
#pragma unroll
  for (int term = 2; term >= 0; --term)
#pragma unroll
    for (int i = term; i >= 0; --i)
      c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i], b[term - i], c, 0, 0,
                                                  0);
  return c;
}

template <int KT, int NC>
__global__ __launch_bounds__(ST, 2) void delta_chunk_scan_kernel(
    float* __restrict__ ws, float* __restrict__ state,  // [slots, H, K, V]
    const int32_t* __restrict__ walk, float* __restrict__ out,  // [rows, H V]
    int H, int K, int V, int VP) {
  constexpr int KP = KT * 16;
  constexpr int MY = (KT + 3) / 4;    // tiles of 16 rows of S per wave
  constexpr bool SPLIT = NC > 1;
  // tiles of 16 rows, 32-bit or split: a lane's values of two tiles together
  constexpr int TILE = SPLIT ? WAVE * 3 / 2 : WAVE;
  __shared__ float4v s_lds[NC][KT * TILE], u_lds[NC][4 * TILE];
  const int h = blockIdx.x, lane = threadIdx.x % WAVE;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
  const int col = lane % 16, g4 = 4 * (lane / 16);
  auto put = [&](float4v* to, int tile, float4v f) {
    if constexpr (SPLIT) {
      bf16x4 o[3];
      split<4>(f, o);
#pragma unroll
      for (int i = 0; i < 3; ++i)
        ((bf16x4*)(to + (tile / 2 * 3 + i) * WAVE + lane))[tile % 2] = o[i];
    } else {
      to[tile * WAVE + lane] = f;
    }
  };
  auto get = [&](const float4v* from, int tile, bf16x8 (&o)[3]) {
#pragma unroll
    for (int i = 0; i < 3; ++i)
      o[i] = __builtin_bit_cast(bf16x8,
                                from[(tile / 2 * 3 + i) * WAVE + lane]);
  };
  const int c0 = blockIdx.y * 16 * NC + col;
  const int4 m = ((const int4*)walk)[blockIdx.z];
  const int64_t row0 = m.x;
  const int n = m.y;
  const bool fresh = m.w >> 30;
  const int64_t chunk0 = m.w & ((1 << 30) - 1);
  float* Sp = state + ((int64_t)m.z * H + h) * K * V;

  float4v S[NC][MY];
#pragma unroll
  for (int x = 0; x < NC; ++x)
#pragma unroll
    for (int i = 0; i < MY; ++i) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int d = 16 * (wave + 4 * i) + g4 + r, c = c0 + 16 * x;
        S[x][i][r] = !fresh && d < K && c < V ? Sp[(int64_t)d * V + c] : 0.f;
      }
      if (wave + 4 * i < KT) put(s_lds[x], wave + 4 * i, S[x][i]);
    }
  lds_barrier();

  // uniform bases, per-lane offsets that stay the same for every chunk
  const int tw = wave * B;            // this wave's 16 tokens
  const int64_t stride = (int64_t)H * work_size(KP, VP);
  const float* base = ws + (chunk0 * H + h) * work_size(KP, VP);
  const unsigned at_w = wave * KT * 1024 + lane * 16;    // bytes
  unsigned at_u[NC];                  // past the last tile: that one's
#pragma unroll
  for (int x = 0; x < NC; ++x)
    at_u[x] = (min((int)blockIdx.y * NC + x, VP / 16 - 1) * 4 + wave) * 1024 +
              lane * 16;
  const unsigned at_p = wave * 4 * 1024 + lane * 16;
  // of 32 channels, the third and fourth wave have no tile of their own
  const unsigned at_k = wave % KT * 4 * 1024 + lane * 16;
  const unsigned at_g = (wave % KT * B + g4) * 4;
  // by way of a buffer, whose offsets take no vector instructions
  const int work_bytes = (int)work_size(KP, VP) * 4;
  auto buffer = [&](const float* p) {
    return __builtin_amdgcn_make_buffer_rsrc((void*)p, 0, work_bytes, BUFFER_BYTES);
  };
  auto load = [&](__amdgpu_buffer_rsrc_t b, unsigned lane_at, int at) {
    return __builtin_bit_cast(float4v,
                              __builtin_amdgcn_raw_buffer_load_b128(b, lane_at, at, 0));
  };
  const int off_w = C * VP * 4, off_q = off_w + C * KP * 4, off_k = off_q + C * KP * 4;
  const int off_p = off_k + C * KP * 4, off_g = off_p + C * C * 4;
  float4v w[KT], qe[KT], u[NC];
  auto fetch = [&](const float* p) {  // in the order of their use
    const auto b = buffer(p);
#pragma unroll
    for (int x = 0; x < NC; ++x) u[x] = load(b, at_u[x], 0);
#pragma unroll
    for (int t = 0; t < KT; ++t) {
      w[t] = load(b, at_w, off_w + 1024 * t);
      qe[t] = load(b, at_w, off_q + 1024 * t);
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  fetch(base);
  float* oc = out + (row0 * H + h) * V;
  const unsigned at_o = (tw + g4) * (H * V) + c0, orow = H * V;
  const bool all_columns = (int)(blockIdx.y + 1) * 16 * NC <= V;
  // No load of the loop is under a condition: the compiler could not count
  // what is under way, and would wait for all of it.
  for (int t0 = 0; t0 < n; t0 += C, oc += C * orow) {
    // operands of the state update and of P U, used after the first products
    float4v kt[MY][4], decay[MY], p[4];
    const auto b = buffer(base);
#pragma unroll
    for (int i = 0; i < MY; ++i) {
#pragma unroll
      for (int x = 0; x < 4; ++x) kt[i][x] = load(b, at_k, off_k + i * 16384 + 1024 * x);
      decay[i] = load(b, at_g, off_g + i * 4 * B * 4);
    }
#pragma unroll
    for (int x = 0; x < 4; ++x)       // those past the wave's own are not used
      p[x] = load(b, at_p, off_p + 1024 * x);
    __builtin_amdgcn_sched_barrier(0);    // now, not where they are used
    float4v o[NC];
#pragma unroll
    for (int x = 0; x < NC; ++x) o[x] = (float4v){0.f, 0.f, 0.f, 0.f};
    if constexpr (SPLIT) {
#pragma unroll
      for (int t = 0; t < KT; t += 2) {
        bf16x8 ws[3], qs[3], ss[3];
        split2(w[t], w[t + 1], ws);
        split2(qe[t], qe[t + 1], qs);
#pragma unroll
        for (int x = 0; x < NC; ++x) {
          get(s_lds[x], t, ss);
          u[x] = mfma_split(ws, ss, u[x]);
          o[x] = mfma_split(qs, ss, o[x]);
        }
      }
    } else {
      // the sums take turns: a product waits for the one before it on its sum
#pragma unroll
      for (int t = 0; t < KT; ++t) {
        const float4v s = s_lds[0][t * WAVE + lane];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          u[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(w[t][r], s[r], u[0], 0, 0,
                                                      0);
          o[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(qe[t][r], s[r], o[0], 0,
                                                      0, 0);
        }
      }
    }
#pragma unroll
    for (int x = 0; x < NC; ++x) put(u_lds[x], wave, u[x]);
    // w, qe and u are free now: the next chunk's arrive during the rest (the
    // last one's once more)
    if (t0 + C < n) base += stride;
    fetch(base);
    lds_barrier();
#pragma unroll
    for (int x = 0; x < NC; ++x)
#pragma unroll
      for (int i = 0; i < MY; ++i) S[x][i] = S[x][i] * decay[i];
    if constexpr (SPLIT) {
#pragma unroll
      for (int y = 0; y < 4; y += 2) {
        bf16x8 us[NC][3], ks[MY][3];
#pragma unroll
        for (int i = 0; i < MY; ++i) split2(kt[i][y], kt[i][y + 1], ks[i]);
#pragma unroll
        for (int x = 0; x < NC; ++x) {
          get(u_lds[x], y, us[x]);
#pragma unroll
          for (int i = 0; i < MY; ++i)
            S[x][i] = mfma_split(ks[i], us[x], S[x][i]);
        }
        if (y <= wave) {
          // of columns that P does not have nothing was written
          bf16x8 ps[3];
          split2(p[y], y < wave ? p[y + 1] : (float4v){0.f, 0.f, 0.f, 0.f},
                 ps);
#pragma unroll
          for (int x = 0; x < NC; ++x) o[x] = mfma_split(ps, us[x], o[x]);
        }
      }
    } else {
#pragma unroll
      for (int y = 0; y < 4; ++y) {
        const float4v us = u_lds[0][y * WAVE + lane];
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
          for (int i = 0; i < MY; ++i)
            S[0][i] = __builtin_amdgcn_mfma_f32_16x16x4f32(kt[i][y][r], us[r],
                                                           S[0][i], 0, 0, 0);
        if (y <= wave) o[0] = mfma4(p[y], us, o[0]);
      }
    }
#pragma unroll
    for (int x = 0; x < NC; ++x)
#pragma unroll
      for (int i = 0; i < MY; ++i)
        if (KT % 4 == 0 || wave + 4 * i < KT) put(s_lds[x], wave + 4 * i, S[x][i]);
    if (t0 + C <= n && all_columns) {
#pragma unroll
      for (int x = 0; x < NC; ++x)
#pragma unroll
        for (int r = 0; r < 4; ++r) oc[at_o + r * orow + 16 * x] = o[x][r];
    } else {
#pragma unroll
      for (int x = 0; x < NC; ++x)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (t0 + tw + g4 + r < n && c0 + 16 * x < V)
            oc[at_o + r * orow + 16 * x] = o[x][r];
    }
    lds_barrier();
  }

#pragma unroll
  for (int x = 0; x < NC; ++x)
#pragma unroll
    for (int i = 0; i < MY; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int d = 16 * (wave + 4 * i) + g4 + r, c = c0 + 16 * x;
        if (wave + 4 * i < KT && d < K && c < V)
          Sp[(int64_t)d * V + c] = S[x][i][r];
      }
}

// out = o / rms(o) * w * sigmoid(gate) per head; LANES threads per (row,
// head), N channels each at a time
template <typename T, int LANES, int N>
__global__ __launch_bounds__(256) void delta_gate_kernel(
    const float* __restrict__ o, const T* __restrict__ gate,
    const float* __restrict__ norm_w, T* __restrict__ out, int64_t n, int V,
    float eps) {
  const int64_t i =
      (int64_t)blockIdx.x * (256 / LANES) + threadIdx.x / LANES;
  const int lane = threadIdx.x % LANES;
  const bool in = i < n;
  float ss = 0.f;
  if (in)
    for (int d = lane * N; d < V; d += LANES * N) {
      float f[N];
      ldn<N>(o + i * V + d, f);
#pragma unroll
      for (int x = 0; x < N; ++x) ss += f[x] * f[x];
    }
#pragma unroll
  for (int x = LANES / 2; x > 0; x /= 2) ss += __shfl_xor(ss, x, WAVE);
  if (!in) return;
  const float inv = 1.f / sqrtf(ss / (float)V + eps);
  for (int d = lane * N; d < V; d += LANES * N) {
    float f[N], g[N], w[N];
    ldn<N>(o + i * V + d, f);
    ldn<N>(gate + i * V + d, g);
    ldn<N>(norm_w + d, w);
#pragma unroll
    for (int x = 0; x < N; ++x) f[x] = f[x] * inv * w[x] * sigmoid_f(g[x]);
    stn<N>(out + i * V + d, f);
  }
}

int padded_k(int K) { return K <= 32 ? 32 : K <= 64 ? 64 : 128; }

}  // namespace

extern "C" {

// floats of workspace per (chunk, head); 0: sizes without a chunked form
int64_t lds_delta_chunk_work(int K, int V) {
  return K > 128 ? 0 : work_size(padded_k(K), (V + 15) / 16 * 16);
}

hipError_t lds_delta_chunk(int f32, const float* q, const float* k,
                           const float* v, const void* beta, int64_t bstride,
                           const void* decay, const float* dt_bias,
                           const float* neg_a, float* state,
                           const int32_t* chunks, int n_chunks,
                           const int32_t* walk, int n_seqs, float* ws,
                           float* out, int KH, int H, int K, int V,
                           hipStream_t stream) {
  if (n_chunks == 0) return hipSuccess;
  if (K > 128) return hipErrorInvalidValue;
  const int KP = padded_k(K), VP = (V + 15) / 16 * 16;
  const size_t lds =
      (2 * C * (KP + 4) + 4 * KP + 10 * AB + C + LT / WAVE) * sizeof(float);
  const dim3 g1(H, n_chunks);
  const int tiles = VP / 16, pairs = (tiles + 1) / 2;
  // two workgroups per compute unit at least, else one tile each
  const bool two = (int64_t)H * pairs * n_seqs >= 512;
#define LOCAL(T, KPV)                                                         \
  do {                                                                        \
    auto fn = delta_chunk_local_kernel<T, KPV>;                               \
    hipError_t e = hipFuncSetAttribute(                                       \
        (const void*)fn, hipFuncAttributeMaxDynamicSharedMemorySize,          \
        (int)lds);                                                            \
    if (e != hipSuccess) return e;                                            \
    hipLaunchKernelGGL(fn, g1, dim3(LT), lds, stream, q, k, v,                \
                       (const T*)beta, bstride, (const T*)decay, dt_bias,     \
                       neg_a, chunks, ws, KH, H, K, V, VP);                   \
  } while (0)
#define GO(KPV)                                                               \
  do {                                                                        \
    if (f32) LOCAL(float, KPV); else LOCAL(short, KPV);                       \
    if (two)                                                                  \
      hipLaunchKernelGGL((delta_chunk_scan_kernel<KPV / 16, 2>),              \
                         dim3(H, pairs, n_seqs), dim3(ST), 0, stream, ws,     \
                         state, walk, out, H, K, V, VP);                      \
    else                                                                      \
      hipLaunchKernelGGL((delta_chunk_scan_kernel<KPV / 16, 1>),              \
                         dim3(H, tiles, n_seqs), dim3(ST), 0, stream, ws,     \
                         state, walk, out, H, K, V, VP);                      \
  } while (0)
  if (KP == 32) GO(32); else if (KP == 64) GO(64); else GO(128);
#undef GO
#undef LOCAL
  HIP_CHECK_LAST();
  return hipSuccess;
}

hipError_t lds_delta_gate(int f32, const float* o, const void* gate,
                          const float* norm_w, void* out, int64_t n, int V,
                          float eps, hipStream_t stream) {
  if (n == 0) return hipSuccess;
#define GO2(T, L, N)                                                          \
  hipLaunchKernelGGL((delta_gate_kernel<T, L, N>),                            \
                     dim3((uint32_t)((n + 256 / L - 1) / (256 / L))),         \
                     dim3(256), 0, stream, o, (const T*)gate, norm_w,         \
                     (T*)out, n, V, eps)
#define GO(L, N)                                                              \
  do {                                                                        \
    if (f32) GO2(float, L, N); else GO2(short, L, N);                         \
  } while (0)
  if (V % 8 == 0) GO(16, 8); else GO(64, 1);
#undef GO
#undef GO2
  HIP_CHECK_LAST();
  return hipSuccess;
}

}  // extern "C"
