// delta_rule.hip — gated delta rule with one decay per head and key channel.
//
// Per head, with S [K, V] in 32-bit floats, token by token:
//   S <- diag(g) S;  u = beta (v - S'k);  S <- S + k u';  o = S'q
//
// delta_prep     short causal convolutions + silu of q, k, v; unit norms
// delta_conv     convolution inputs kept for the next step
// delta_step     the recurrence itself, one workgroup per (head, sequence),
//                with gates and the gated output norm (decode, short rows);
//                of single rows with what the other two do (delta_single)
// The chunked form for long rows is in delta_chunk.hip.
#include "elem.h"

#include <type_traits>

namespace {

constexpr int NT = 256;
constexpr int NWV = NT / WAVE;
constexpr int AHEAD = 4;  // rows that delta_prep's threads ask for at once
constexpr int MAXU = 8;  // unit norm over up to MAXU * 64 channels

// grid (rows, y): waves share the units of one row. Units: KH of q, KH of k
// (K channels each, unit-normed), H of v (V channels).
template <typename T>
__global__ __launch_bounds__(NT) void delta_prep_kernel(
    const T* __restrict__ proj, int64_t pstride,  // [rows, >= C]
    const float* __restrict__ taps,               // [n_taps, C]
    T* __restrict__ conv_state,                   // [slots, n_taps - 1, C]
    const int32_t* __restrict__ row_seq, const int32_t* __restrict__ seq_meta,
    float* __restrict__ q, float* __restrict__ k, float* __restrict__ v,
    int KH, int H, int K, int V, int n_taps, float q_scale, float unit_eps) {
  const int row = blockIdx.x;
  const int lane = threadIdx.x % WAVE;
  const int wave = threadIdx.x / WAVE + blockIdx.y * NWV;
  const int C = 2 * KH * K + H * V;
  const Seq sq = load_seq(seq_meta, row_seq[row]);
  const int pos = row - sq.row0;
  T* state = conv_state + (int64_t)sq.slot * (n_taps - 1) * C;
  const bool roll = sq.n == 1;  // this thread is the only user of its channel

  for (int unit = wave; unit < 2 * KH + H; unit += NWV * gridDim.y) {
    const bool qk = unit < 2 * KH;
    const int len = qk ? K : V;
    const int c0 = qk ? unit * K : 2 * KH * K + (unit - 2 * KH) * V;
    float* dst = unit < KH ? q + ((int64_t)row * KH + unit) * K
                 : qk      ? k + ((int64_t)row * KH + unit - KH) * K
                           : v + ((int64_t)row * H + unit - 2 * KH) * V;
    float keep[MAXU];
    float ss = 0.f;
    auto channel = [&](int d) {
      const int c = c0 + d;
      float acc = 0.f;
      for (int j = 0; j < n_taps; ++j) {
        const int p = pos - (n_taps - 1) + j;
        float in = 0.f;
        if (p >= 0)
          in = ld(proj + (int64_t)(sq.row0 + p) * pstride + c);
        else if (sq.prior > 0)
          in = ld(state + (int64_t)(n_taps - 1 + p) * C + c);
        if (roll && j > 0) st(state + (int64_t)(j - 1) * C + c, in);
        acc += taps[(int64_t)j * C + c] * in;
      }
      return acc * sigmoid_f(acc);
    };
    if (!qk) {
      for (int d = lane; d < len; d += WAVE) dst[d] = channel(d);
      continue;
    }
#pragma unroll
    for (int i = 0; i < MAXU; ++i) {
      const int d = lane + i * WAVE;
      keep[i] = d < len ? channel(d) : 0.f;
      ss += keep[i] * keep[i];
    }
    const float norm = sqrtf(wave_reduce_sum(ss) + unit_eps);
    const float mul = (unit < KH ? q_scale : 1.f) / norm;
#pragma unroll
    for (int i = 0; i < MAXU; ++i) {
      const int d = lane + i * WAVE;
      if (d < len) dst[d] = keep[i] * mul;
    }
  }
}

// The same for sizes in vectors: a thread owns 8 channels and walks RB rows
// with the last TAPS - 1 inputs in registers; K / 8 threads (a power of two)
// share a unit norm. grid (channel blocks, row blocks)
// Bound by memory, 4.5 TB/s, once the loads of AHEAD rows are under way: 7749 rows of
// 12288 channels 126 us in a pass; 141 with a row's load, behind those of its sequence's
// number and place, at a time.
template <typename T, int TAPS>
__global__ __launch_bounds__(NT) void delta_prep_vec_kernel(
    const T* __restrict__ proj, int64_t pstride, const float* __restrict__ taps,
    T* __restrict__ conv_state, const int32_t* __restrict__ row_seq,
    const int32_t* __restrict__ seq_meta, float* __restrict__ q,
    float* __restrict__ k, float* __restrict__ v, int rows, int RB, int KH,
    int H, int K, int V, float q_scale, float unit_eps) {
  const int C = 2 * KH * K + H * V, QK = KH * K;
  const int c = (blockIdx.x * NT + threadIdx.x) * 8;
  const bool in = c < C;
  const int cc = in ? c : 0;
  const bool qk = cc < 2 * QK;
  float w[TAPS][8], x[TAPS][8];
#pragma unroll
  for (int j = 0; j < TAPS; ++j) ldn<8>(taps + (int64_t)j * C + cc, w[j]);
  const int r0 = blockIdx.y * RB, r1 = min(rows, r0 + RB);
  typedef typename std::conditional<
      sizeof(T) == 2, short8, __attribute__((ext_vector_type(8))) float>::type Eight;
  // a block's rows are of one sequence, as a rule: it is looked up once then
  const int s0 = row_seq[r0];
  const bool one = row_seq[r1 - 1] == s0;
  Seq sq = load_seq(seq_meta, s0);
  Eight raw[AHEAD];
  auto ask = [&](int row) {
#pragma unroll
    for (int i = 0; i < AHEAD; ++i)
      raw[i] = *(const Eight*)(proj + (int64_t)min(row + i, r1 - 1) * pstride + cc);
  };
  ask(r0);
  for (int first = r0; first < r1; first += AHEAD) {
    Eight now[AHEAD];
#pragma unroll
    for (int i = 0; i < AHEAD; ++i) now[i] = raw[i];
    if (first + AHEAD < r1) ask(first + AHEAD);
#pragma unroll
    for (int i = 0; i < AHEAD; ++i) {
      const int row = first + i;
      if (row >= r1) break;
      if (!one) sq = load_seq(seq_meta, row_seq[row]);
      const int pos = row - sq.row0;
      T* state = conv_state + (int64_t)sq.slot * (TAPS - 1) * C + cc;
      if (row == r0 || pos == 0) {
#pragma unroll
        for (int j = 0; j < TAPS - 1; ++j) {
          const int p = pos - (TAPS - 1) + j;
          if (p >= 0) {
            ldn<8>(proj + (int64_t)(sq.row0 + p) * pstride + cc, x[j]);
          } else if (sq.prior > 0) {
            ldn<8>(state + (int64_t)(TAPS - 1 + p) * C, x[j]);
          } else {
#pragma unroll
            for (int e = 0; e < 8; ++e) x[j][e] = 0.f;
          }
        }
      }
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        if constexpr (sizeof(T) == 2)
          x[TAPS - 1][e] = bf16_to_f32(now[i][e]);
        else
          x[TAPS - 1][e] = now[i][e];
      }
      if (sq.n == 1 && in) {
#pragma unroll
        for (int j = 0; j < TAPS - 1; ++j) stn<8>(state + (int64_t)j * C, x[j + 1]);
      }
      float f[8], ss = 0.f;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        float a = 0.f;
#pragma unroll
        for (int j = 0; j < TAPS; ++j) a += w[j][e] * x[j][e];
        f[e] = a * sigmoid_f(a);
        ss += f[e] * f[e];
      }
      for (int o = K / 16; o > 0; o /= 2) ss += __shfl_xor(ss, o, WAVE);
      if (qk) {
        const float m = (cc < QK ? q_scale : 1.f) / sqrtf(ss + unit_eps);
#pragma unroll
        for (int e = 0; e < 8; ++e) f[e] *= m;
      }
      if (in)
        stn<8>(cc < QK       ? q + (int64_t)row * QK + cc
               : cc < 2 * QK ? k + (int64_t)row * QK + cc - QK
                             : v + (int64_t)row * H * V + cc - 2 * QK,
               f);
#pragma unroll
      for (int j = 0; j < TAPS - 1; ++j)
#pragma unroll
        for (int e = 0; e < 8; ++e) x[j][e] = x[j + 1][e];
    }
  }
}

// grid (channel blocks, sequences): keep the last n_taps - 1 inputs of every
// sequence with more than one row (single rows roll in delta_prep)
template <typename T>
__global__ __launch_bounds__(NT) void delta_conv_kernel(
    const T* __restrict__ proj, int64_t pstride, T* __restrict__ conv_state,
    const int32_t* __restrict__ seq_meta, int C, int n_taps) {
  const Seq sq = load_seq(seq_meta, blockIdx.y);
  const int c = blockIdx.x * NT + threadIdx.x;
  if (c >= C || sq.n == 1) return;
  T* state = conv_state + (int64_t)sq.slot * (n_taps - 1) * C;
  // entry i takes an input that is newer than entry i: ascending is in place
  for (int i = 0; i < n_taps - 1; ++i) {
    const int p = sq.n - (n_taps - 1) + i;
    float in = 0.f;
    if (p >= 0)
      in = ld(proj + (int64_t)(sq.row0 + p) * pstride + c);
    else if (sq.prior > 0)
      in = ld(state + (int64_t)(n_taps - 1 + p) * C + c);
    st(state + (int64_t)i * C + c, in);
  }
}

// One workgroup per (head, sequence). S is spread over the threads: a thread
// owns 4 columns (lanes_v threads cover V) and every groups-th row.
// RPT: rows per thread. VEC: V % 4 == 0.
//
// The bytes of S, read and written once, are what counts; what kept it from
// their rate were two workgroups per compute unit, each with a chain of loads.
// So all of a token's inputs are asked for ahead of S, barriers wait for LDS
// alone, and 16 rows per thread stay within 168 registers, for three (for four
// they spill). S is not seen again before the next step of the model: marked
// non-temporal, both ways, it leaves the last-level cache to the weights. us of
// 50 sequences of 32 heads of 128 x 128, and with a gated product of 4096 -> 2 x
// 14336 behind it: 56; 50 and 102 by the shorter chain; 47 and 103 with the
// stores non-temporal; 42 (4.9 TB/s) and 88 with both. 200 sequences 186 -> 157,
// 24 30 -> 17.5, 1 9.2 -> 8.7.
//
// CONV: sequences of one row each, every head with q and k of its own; q, k and v are
// what delta_prep makes of the row, made here while S is on its way (50 sequences of 32
// heads of 128 x 128: 46.8 us, apart 6.4 and 44.0).
template <typename T>
struct Conv {
  const T* proj;             // [rows, >= C]
  int64_t pstride;
  const float* taps;         // [n_taps, C], 2 to 4
  T* state;                  // [slots, n_taps - 1, C]
  int n_taps;
  float q_scale, unit_eps;
};

template <typename T, int RPT, bool VEC, bool CONV>
__global__ __launch_bounds__(NT, RPT <= 8    ? 4
                                 : RPT == 16 ? 3
                                             : 1) void delta_step_kernel(
    const float* __restrict__ q, const float* __restrict__ k,
    const float* __restrict__ v,                 // [rows, KH|KH|H, K|K|V]
    const T* __restrict__ beta, int64_t bstride,  // [rows, H] before sigmoid
    const T* __restrict__ decay,                 // [rows, H K] before bias
    const float* __restrict__ dt_bias,           // [H K]
    const float* __restrict__ neg_a,             // [H]: -exp(A_log)
    const T* __restrict__ gate,                  // [rows, H V] before sigmoid
    const float* __restrict__ norm_w,            // [V]
    float* __restrict__ state,                   // [slots, H, K, V]
    const int32_t* __restrict__ seq_meta, T* __restrict__ out, int KH, int H,
    int K, int V, int lanes_v, float eps, const Conv<T> in_) {
  const int h = blockIdx.x;
  const Seq sq = load_seq(seq_meta, blockIdx.y);
  const int kh = h / (H / KH);
  const int groups = NT / lanes_v;
  const unsigned tv = threadIdx.x % lanes_v, grp = threadIdx.x / lanes_v;
  const unsigned c0 = tv * 4;

  constexpr int KT = 512 / NT;        // channels of K per thread, at most
  __shared__ float4v gkq[512];        // decay, k, q of a channel
  __shared__ float4v sk[NT], so[NT];
  __shared__ float kq[NT];
  __shared__ float red[NWV];

  // a token's inputs, as they are in memory; past the end they repeat the last
  const unsigned tid = threadIdx.x, last = V - 1, cv = VEC ? min(c0, V - 4u) : c0;
  auto channel = [&](int j) { return VEC ? cv + j : min(cv + j, last); };
  float qr[KT], kr[KT], vr[4], bias[KT], nw[4];
  T dr[KT], gr[4], br;
  auto fetch = [&](int t) {
    const int64_t row = sq.row0 + t;
    const float* qt = q + (row * KH + kh) * K;
    const float* kt = k + (row * KH + kh) * K;
    const T* dt = decay + (row * H + h) * K;
    const float* vt = v + (row * H + h) * V;
    const T* gt = gate + (row * H + h) * V;
#pragma unroll
    for (int i = 0; i < KT; ++i) {
      const unsigned d = min(tid + i * NT, K - 1u);
      if constexpr (!CONV) {
        qr[i] = qt[d];
        kr[i] = kt[d];
      }
      dr[i] = dt[d];
    }
    br = beta[row * bstride + h];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      if constexpr (!CONV) vr[j] = vt[channel(j)];
      gr[j] = gt[channel(j)];
    }
  };
  const float na = neg_a[h];
  const float* bt = dt_bias + (int64_t)h * K;
#pragma unroll
  for (int i = 0; i < KT; ++i) bias[i] = bt[min(tid + i * NT, K - 1u)];
#pragma unroll
  for (int j = 0; j < 4; ++j) nw[j] = norm_w[channel(j)];
  if (sq.n > 0) fetch(0);
  // the head's channels of q, k and v: a thread's inputs, oldest first, and taps
  constexpr int CT = CONV ? 2 : 1, TAPS = 4;
  __shared__ float conv[CONV ? 2 * NT : 1], unit[2];
  T cx[CT][TAPS];
  float cw[CT][TAPS];
  const int QK = KH * K, all = 2 * K + V, C = 2 * QK + H * V;
  auto column = [&](int i) {
    const int d = min((int)tid + i * NT, all - 1);
    return d < K ? kh * K + d : d < 2 * K ? QK + kh * K + d - K
                                          : 2 * QK + h * V + d - 2 * K;
  };
  T* const kept = CONV ? in_.state + (int64_t)sq.slot * (in_.n_taps - 1) * C : nullptr;
  if constexpr (CONV) {
    // a sequence without rows has no proj[row0]; a branch here cost 0.5 us of 8.4
    const T* x = in_.proj + (sq.n > 0 ? sq.row0 : 0) * in_.pstride;
#pragma unroll
    for (int i = 0; i < CT; ++i) {
      const int c = column(i);
#pragma unroll
      for (int j = 0; j < TAPS; ++j) {
        cw[i][j] = in_.taps[(int64_t)min(j, in_.n_taps - 1) * C + c];
        cx[i][j] = j < in_.n_taps - 1 ? kept[(int64_t)j * C + c] : x[c];
      }
    }
  }

  float S[RPT][4];
  float* Sp = state + ((int64_t)sq.slot * H + h) * K * V;
  const unsigned at = grp * V + c0, step = groups * V;
#pragma unroll
  for (int i = 0; i < RPT; ++i) {
    const int r = grp + i * groups;
#pragma unroll
    for (int j = 0; j < 4; ++j) S[i][j] = 0.f;
    if (r < K && sq.prior > 0) {
      if constexpr (VEC) {
        if (c0 < (unsigned)V) {
          const float4v t =
              __builtin_nontemporal_load((const float4v*)(Sp + i * step + at));
#pragma unroll
          for (int j = 0; j < 4; ++j) S[i][j] = t[j];
        }
      } else {
#pragma unroll
        for (int j = 0; j < 4; ++j)
          if (c0 + j < (unsigned)V) S[i][j] = Sp[i * step + at + j];
      }
    }
  }

  if constexpr (CONV) {
    if (sq.n > 0) {                                  // workgroup-uniform
#pragma unroll
      for (int i = 0; i < CT; ++i) {
        const int d = tid + i * NT, c = column(i);
        float x[TAPS], a = 0.f;
#pragma unroll
        for (int j = 0; j < TAPS; ++j) {
          x[j] = j < in_.n_taps - 1 && sq.prior <= 0 ? 0.f : ld(&cx[i][j]);
          if (j < in_.n_taps) a += cw[i][j] * x[j];
        }
        if (d < all) {
          conv[d] = a * sigmoid_f(a);
#pragma unroll
          for (int j = 0; j < TAPS - 1; ++j)
            if (j < in_.n_taps - 1) st(kept + (int64_t)j * C + c, x[j + 1]);
        }
      }
      lds_barrier();
      if (tid < 2 * WAVE) {
        float ss = 0.f;
        for (int d = tid % WAVE; d < K; d += WAVE) {
          const float x = conv[tid / WAVE * K + d];
          ss += x * x;
        }
        ss = wave_reduce_sum(ss);
        if (tid % WAVE == 0)
          unit[tid / WAVE] = (tid < WAVE ? in_.q_scale : 1.f) / sqrtf(ss + in_.unit_eps);
      }
      lds_barrier();
#pragma unroll
      for (int i = 0; i < KT; ++i) {
        const unsigned d = min(tid + i * NT, K - 1u);
        qr[i] = conv[d] * unit[0];
        kr[i] = conv[K + d] * unit[1];
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) vr[j] = conv[2 * K + channel(j)];
    }
  }
  for (int t = 0; t < (CONV ? min(sq.n, 1) : sq.n); ++t) {
    const int64_t row = sq.row0 + t;
    // readers of gkq and kq of the token before are past a barrier (block_sum)
#pragma unroll
    for (int i = 0; i < KT; ++i) {
      const int d = tid + i * NT;
      if (d < K)
        gkq[d] = (float4v){expf(na * softplus_f(ld(&dr[i]) + bias[i])), kr[i],
                           qr[i], 0.f};
    }
    lds_barrier();
    float4v a = {0.f, 0.f, 0.f, 0.f}, b = a;
    float c = 0.f;
#pragma unroll
    for (int i = 0; i < RPT; ++i) {
      const int r = grp + i * groups;
      if (r < K) {
        const float4v x = gkq[r];
        c += x[1] * x[2];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          S[i][j] *= x[0];
          a[j] += S[i][j] * x[1];
          b[j] += S[i][j] * x[2];
        }
      }
      if (i % 4 == 3) __builtin_amdgcn_sched_barrier(0);   // registers
    }
    sk[threadIdx.x] = a;
    so[threadIdx.x] = b;
    if (tv == 0) kq[grp] = c;
    lds_barrier();
    // S'k and S'q of the decayed state; the new write adds (k.q) u to o
    float4v u = {0.f, 0.f, 0.f, 0.f}, o = u;
    float dot = 0.f;
#pragma unroll 2
    for (int p = 0; p < groups; ++p) {
      dot += kq[p];
      u += sk[p * lanes_v + tv];
      o += so[p * lanes_v + tv];
    }
    const float write = sigmoid_f(ld(&br));
    float ss = 0.f;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const bool in = c0 + j < (unsigned)V;
      u[j] = in ? write * (vr[j] - u[j]) : 0.f;
      o[j] += dot * u[j];
      if (in && grp == 0) ss += o[j] * o[j];
    }
#pragma unroll
    for (int i = 0; i < RPT; ++i) {
      const int r = grp + i * groups;
      if (r < K) {
        const float kd = gkq[r][1];
#pragma unroll
        for (int j = 0; j < 4; ++j) S[i][j] += kd * u[j];
      }
      if (i % 4 == 3) __builtin_amdgcn_sched_barrier(0);
    }
    T gt[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) gt[j] = gr[j];
    if (!CONV && t + 1 < sq.n) fetch(t + 1);
    const float inv =
        1.f / sqrtf(block_sum<NWV>(ss, red) / (float)V + eps);
    T* ot = out + (row * H + h) * V;
    if (grp == 0) {
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (c0 + j < (unsigned)V)
          st(ot + c0 + j,
             o[j] * inv * nw[j] * sigmoid_f(ld(&gt[j])));
    }
  }

#pragma unroll
  for (int i = 0; i < RPT; ++i) {
    const int r = grp + i * groups;
    if (r < K) {
      if constexpr (VEC) {
        if (c0 < (unsigned)V)
          __builtin_nontemporal_store(
              (float4v){S[i][0], S[i][1], S[i][2], S[i][3]},
              (float4v*)(Sp + i * step + at));
      } else {
#pragma unroll
        for (int j = 0; j < 4; ++j)
          if (c0 + j < (unsigned)V) Sp[i * step + at + j] = S[i][j];
      }
    }
  }
}

// Threads along a row of the state, 4 channels each, and its rows per thread
int state_lanes(int V) {
  int lanes = 1;
  while (lanes * 4 < V) lanes *= 2;
  return lanes;
}

int state_rows(int K, int V) {
  const int groups = NT / state_lanes(V);
  return (K + groups - 1) / groups;
}

constexpr int SINGLE_ROWS = 32;      // of delta_single; delta_step has a form of 64

}  // namespace

extern "C" {

hipError_t lds_delta_prep(int f32, const void* proj, int64_t pstride,
                          const float* taps, void* conv_state,
                          const int32_t* row_seq, const int32_t* seq_meta,
                          float* q, float* k, float* v, int rows, int n_seqs,
                          int multi_row, int KH, int H, int K, int V,
                          int n_taps, float q_scale, float unit_eps,
                          hipStream_t stream) {
  if (rows == 0) return hipSuccess;
  if (K > MAXU * WAVE || n_taps < 1) return hipErrorInvalidValue;
  const int units = 2 * KH + H, C = 2 * KH * K + H * V;
  int gy = (units + NWV - 1) / NWV;
  if (rows >= 1024 && gy > 4) gy = 4;
  const dim3 grid(rows, gy), cgrid((C + NT - 1) / NT, n_seqs);
  const bool vec = K % 8 == 0 && V % 8 == 0 && pstride % 8 == 0 &&
                   K / 8 <= WAVE && (K / 8 & (K / 8 - 1)) == 0 &&
                   n_taps >= 2 && n_taps <= 4;
  int rb = 1;       // rows per thread: long walks only with enough of them
  while (rb < 32 && (int64_t)rows * C / 8 / NT / (2 * rb) >= 2048) rb *= 2;
  const dim3 vgrid((C / 8 + NT - 1) / NT, (rows + rb - 1) / rb);
#define VEC(T, TAPS)                                                          \
  hipLaunchKernelGGL((delta_prep_vec_kernel<T, TAPS>), vgrid, dim3(NT), 0,    \
                     stream, (const T*)proj, pstride, taps, (T*)conv_state,   \
                     row_seq, seq_meta, q, k, v, rows, rb, KH, H, K, V,       \
                     q_scale, unit_eps)
#define GO(T)                                                                 \
  do {                                                                        \
    if (vec && n_taps == 2) VEC(T, 2);                                        \
    else if (vec && n_taps == 3) VEC(T, 3);                                   \
    else if (vec) VEC(T, 4);                                                  \
    else                                                                      \
      hipLaunchKernelGGL(delta_prep_kernel<T>, grid, dim3(NT), 0, stream,     \
                         (const T*)proj, pstride, taps, (T*)conv_state,       \
                         row_seq, seq_meta, q, k, v, KH, H, K, V, n_taps,     \
                         q_scale, unit_eps);                                  \
    if (multi_row && n_taps > 1)                                              \
      hipLaunchKernelGGL(delta_conv_kernel<T>, cgrid, dim3(NT), 0, stream,    \
                         (const T*)proj, pstride, (T*)conv_state, seq_meta,   \
                         C, n_taps);                                          \
  } while (0)
  if (f32) GO(float); else GO(short);
#undef VEC
#undef GO
  HIP_CHECK_LAST();
  return hipSuccess;
}

hipError_t lds_delta_step(int f32, const float* q, const float* k,
                          const float* v, const void* beta, int64_t bstride,
                          const void* decay, const float* dt_bias,
                          const float* neg_a, const void* gate,
                          const float* norm_w, float* state,
                          const int32_t* seq_meta, void* out, int n_seqs,
                          int KH, int H, int K, int V, float eps,
                          hipStream_t stream) {
  if (n_seqs == 0) return hipSuccess;
  if (V > 4 * NT || K > 512) return hipErrorInvalidValue;
  const int lanes_v = state_lanes(V), need = state_rows(K, V);
  int rpt = 1;
  while (rpt < need) rpt *= 2;
  const dim3 grid(H, n_seqs);
#define GO2(T, R, VEC)                                                        \
  hipLaunchKernelGGL((delta_step_kernel<T, R, VEC, false>), grid, dim3(NT),   \
                     0, stream, q, k, v, (const T*)beta, bstride,             \
                     (const T*)decay, dt_bias, neg_a, (const T*)gate, norm_w, \
                     state, seq_meta, (T*)out, KH, H, K, V, lanes_v, eps,     \
                     Conv<T>{})
#define GO1(T, R)                                                             \
  do {                                                                        \
    if (V % 4 == 0) GO2(T, R, true); else GO2(T, R, false);                   \
  } while (0)
#define GO(R)                                                                 \
  do {                                                                        \
    if (f32) GO1(float, R); else GO1(short, R);                               \
  } while (0)
  switch (rpt) {
    case 1: GO(1); break;
    case 2: GO(2); break;
    case 4: GO(4); break;
    case 8: GO(8); break;
    case 16: GO(16); break;
    case 32: GO(32); break;
    case 64: GO(64); break;
    default: return hipErrorInvalidValue;
  }
#undef GO
#undef GO1
#undef GO2
  HIP_CHECK_LAST();
  return hipSuccess;
}

// Whether lds_delta_single takes the sizes
int lds_delta_single_ok(int f32, int KH, int H, int K, int V, int n_taps) {
  return !f32 && KH == H && V % 4 == 0 && V >= 4 && 2 * K + V <= 2 * NT &&
         state_rows(K, V) <= SINGLE_ROWS && n_taps >= 2 && n_taps <= 4;
}

// delta_prep and delta_step of sequences of one row each (bf16), in one kernel
hipError_t lds_delta_single(const void* proj, int64_t pstride, const float* taps,
                            void* conv_state, int n_taps, float q_scale,
                            float unit_eps, const void* beta, const void* decay,
                            const float* dt_bias, const float* neg_a,
                            const void* gate, const float* norm_w, float* state,
                            const int32_t* seq_meta, void* out, int n_seqs, int H,
                            int K, int V, float eps, hipStream_t stream) {
  if (n_seqs == 0) return hipSuccess;
  if (!lds_delta_single_ok(0, H, H, K, V, n_taps)) return hipErrorInvalidValue;
  const int lanes_v = state_lanes(V), need = state_rows(K, V);
  const Conv<short> cv{(const short*)proj, pstride, taps, (short*)conv_state,
                       n_taps, q_scale, unit_eps};
#define GO(R)                                                                 \
  hipLaunchKernelGGL((delta_step_kernel<short, R, true, true>),               \
                     dim3(H, n_seqs), dim3(NT), 0, stream, nullptr, nullptr,  \
                     nullptr, (const short*)beta, pstride,                    \
                     (const short*)decay, dt_bias, neg_a, (const short*)gate, \
                     norm_w, state, seq_meta, (short*)out, H, H, K, V,        \
                     lanes_v, eps, cv)
  if (need <= 4) GO(4);
  else if (need <= 8) GO(8);
  else if (need <= 16) GO(16);
  else GO(SINGLE_ROWS);
#undef GO
  HIP_CHECK_LAST();
  return hipSuccess;
}

}  // extern "C"
