// residual_norm.hip — the 32-bit residual stream: embedding, what sublayers
// and loop passes add to it, RMS norms, activations. HBM-bound; one pass over
// the stream per sublayer.
#include "elem.h"

namespace {

constexpr int NT = 256;
constexpr int PT = 512;  // of rows in parts of more than 256 vectors

template <typename T> struct Eight;
template <> struct Eight<short> {
  typedef short8 type;
  static __device__ __forceinline__ float get(type v, int j) { return bf16_to_f32(v[j]); }
};
template <> struct Eight<float> {
  typedef __attribute__((ext_vector_type(8))) float type;
  static __device__ __forceinline__ float get(type v, int j) { return v[j]; }
};

enum Mode { EMBED, POST, ADD, LOOP };

template <typename T>
struct Stream {
  float* x;                  // [T, H]
  const T* y;                // [T, H], or the embedding table
  const float* yp;           // or 32-bit partial sums [parts, T, H] of a
  int parts;                 // product that split K
  const int64_t* ids;        // EMBED
  const float* pos;          // EMBED: [positions, H] or null
  const int32_t* positions;
  const float* wb;           // POST
  const T* rows;             // POST, ADD: [T n_rows, H], n_rows of each token
  int n_rows;
  const float *a, *b, *v;    // LOOP: [T, H], [T, H], [H]
  const float* wn;           // null: h = x
  T* h;
  int H;
  float scale, offset, eps;
};

// One workgroup per row of the stream.
//   EMBED: x = table[id] * scale + pos[position]
//   POST:  x += y / rms(y) * (wb + offset) + the token's rows
//   ADD:   x += y + the token's rows (either may be missing)
//   LOOP:  x = a + b + v
//   h = x / rms(x) * (wn + offset)
//   PARTS: y is in parts, 8 channels per vector; so many of them stay in a thread's
//   registers, the others' threads keep four. What a row takes is the time of its loads,
//   one after the other: everything that is known ahead is asked for at once, by as many
//   threads as there are vectors, up to 512 (50 rows of 4096 in 8 parts in a pass: 5.3 us;
//   256 threads, and weights and rows of experts when they are needed: 7.3).
template <typename T, int N, int MODE, int PARTS, int BT>
__global__ __launch_bounds__(BT) void stream_norm_kernel(const Stream<T> s) {
  static_assert(!PARTS || N == 8, "");
  constexpr int KEEP = PARTS ? PARTS : 4;  // vectors kept in registers per thread
  __shared__ float red[2][BT / WAVE];
  const int64_t row = blockIdx.x;
  const int H = s.H;
  float* xr = s.x + row * H;
  const T* yr = MODE == EMBED ? s.y + s.ids[row] * H : s.y + row * H;
  // the sublayer's output; its parts are summed here rather than by a launch
  // of their own, one of 3 us
  auto load_y = [&](int64_t c, float* f) {
    if (!s.yp) {
      ldn<N>(yr + c, f);
      return;
    }
    const float* p = s.yp + row * H + c;
    ldn<N>(p, f);
#pragma unroll 4
    for (int k = 1; k < s.parts; ++k) {
      float g[N];
      ldn<N>(p + (int64_t)k * gridDim.x * H, g);
#pragma unroll
      for (int j = 0; j < N; ++j) f[j] += g[j];
    }
  };
  // vector i of this thread starts at element at(i); the first KEEP stay in
  // registers between the passes, the rest are read again
  float keep[KEEP][N];
  auto at = [&](int i) { return (int64_t)(threadIdx.x + i * BT) * N; };
  // All parts of what a thread keeps are asked for together, the stream's values, the
  // weights and the first ROWS of the token's rows (with two vectors they have no room)
  // ahead of them.
  constexpr int ROWS = PARTS == 1 ? 4 : 0;
  float xk[PARTS ? KEEP : 1][N], wbk[PARTS ? KEEP : 1][N], wnk[PARTS ? KEEP : 1][N];
  typename Eight<T>::type rk[PARTS ? KEEP : 1][ROWS ? ROWS : 1];   // as in memory
  if constexpr (PARTS) {
#pragma unroll
    for (int i = 0; i < KEEP; ++i)
      if (i * BT * N < H) {
        const int64_t c = min(at(i), (int64_t)H - N);
        ldn<N>(xr + c, xk[i]);
        if (MODE == POST) ldn<N>(s.wb + c, wbk[i]);
        if (s.wn) ldn<N>(s.wn + c, wnk[i]);
        if (s.n_rows)
#pragma unroll
          for (int r = 0; r < ROWS; ++r)
            rk[i][r] = *(const typename Eight<T>::type*)(
                s.rows + (row * s.n_rows + min(r, s.n_rows - 1)) * H + c);
      }
#pragma unroll
    for (int i = 0; i < KEEP; i += 2)
      if (KEEP == 1 || (i * BT * N < H && (i + 1) * BT * N >= H)) {  // the last one alone
        const float4v* const src[1] = {
            (const float4v*)(s.yp + row * H + min(at(i), (int64_t)H - N))};
        PartSums<1>(src, (int64_t)gridDim.x * H / 4, s.parts).get(0, keep[i]);
      } else if (i * BT * N < H) {
        const float4v* src[2];
#pragma unroll
        for (int j = 0; j < 2; ++j)
          src[j] = (const float4v*)(s.yp + row * H +
                                    min(at(i + j), (int64_t)H - N));
        const PartSums<2> sum(src, (int64_t)gridDim.x * H / 4, s.parts);
        sum.get(0, keep[i]);
        sum.get(1, keep[i + 1]);
      }
  }
  float inv_y = 0.f;
  if constexpr (MODE == POST) {
    float ss = 0.f;
    auto square = [&](int i, float* f) {
      if (!PARTS || i >= KEEP) load_y(at(i), f);
#pragma unroll
      for (int j = 0; j < N; ++j) ss += f[j] * f[j];
    };
#pragma unroll
    for (int i = 0; i < KEEP; ++i)
      if (at(i) < H) square(i, keep[i]);
    for (int i = KEEP; at(i) < H; ++i) {
      float f[N];
      square(i, f);
    }
    inv_y = 1.f / sqrtf(block_sum<BT / WAVE>(ss, red[0]) / (float)H + s.eps);
  }
  float ss = 0.f;
  auto update = [&](int i, float* f) {  // POST: y's vector in; stream's out
    const int64_t c = at(i);
    float g[N];
    if constexpr (MODE == EMBED) {
      ldn<N>(yr + c, f);
#pragma unroll
      for (int j = 0; j < N; ++j) f[j] *= s.scale;
      if (s.pos) {
        ldn<N>(s.pos + (int64_t)s.positions[row] * H + c, g);
#pragma unroll
        for (int j = 0; j < N; ++j) f[j] += g[j];
      }
      stn<N>(xr + c, f);
    } else if constexpr (MODE == LOOP) {
      ldn<N>(s.a + row * H + c, f);
      ldn<N>(s.b + row * H + c, g);
#pragma unroll
      for (int j = 0; j < N; ++j) f[j] += g[j];
      ldn<N>(s.v + c, g);
#pragma unroll
      for (int j = 0; j < N; ++j) f[j] += g[j];
      stn<N>(xr + c, f);
    } else {
      float d[N];                       // what the row gets
#pragma unroll
      for (int j = 0; j < N; ++j) d[j] = 0.f;
      if constexpr (MODE == POST) {
        float w[N];
        if (PARTS && i < KEEP)
#pragma unroll
          for (int j = 0; j < N; ++j) w[j] = wbk[PARTS ? i : 0][j];
        else
          ldn<N>(s.wb + c, w);
#pragma unroll
        for (int j = 0; j < N; ++j) d[j] = f[j] * inv_y * (w[j] + s.offset);
      } else if (PARTS && i < KEEP) {
#pragma unroll
        for (int j = 0; j < N; ++j) d[j] = f[j];
      } else if (s.y || s.yp) {
        load_y(c, d);
      }
      int r = 0;
      if (PARTS && i < KEEP)
#pragma unroll
        for (; r < ROWS; ++r)
          if (r < s.n_rows)
#pragma unroll
            for (int j = 0; j < N; ++j) d[j] += Eight<T>::get(rk[PARTS ? i : 0][r], j);
      for (; r < s.n_rows; ++r) {
        ldn<N>(s.rows + (row * s.n_rows + r) * H + c, g);
#pragma unroll
        for (int j = 0; j < N; ++j) d[j] += g[j];
      }
      if (PARTS && i < KEEP) {
#pragma unroll
        for (int j = 0; j < N; ++j) f[j] = xk[PARTS ? i : 0][j];
      } else {
        ldn<N>(xr + c, f);
      }
#pragma unroll
      for (int j = 0; j < N; ++j) f[j] += d[j];
      if (MODE == POST || s.y || s.yp || s.n_rows) stn<N>(xr + c, f);
    }
#pragma unroll
    for (int j = 0; j < N; ++j) ss += f[j] * f[j];
  };
#pragma unroll
  for (int i = 0; i < KEEP; ++i)
    if (at(i) < H) update(i, keep[i]);
  for (int i = KEEP; at(i) < H; ++i) {
    float f[N];
    if (MODE == POST) load_y(at(i), f);
    update(i, f);
  }
  const float inv = s.wn ? 1.f / sqrtf(block_sum<BT / WAVE>(ss, red[1]) /
                                       (float)H + s.eps)
                         : 1.f;
  auto finish = [&](int i, float* f) {
    if (s.wn) {
      float w[N];
      if (PARTS && i < KEEP)
#pragma unroll
        for (int j = 0; j < N; ++j) w[j] = wnk[PARTS ? i : 0][j];
      else
        ldn<N>(s.wn + at(i), w);
#pragma unroll
      for (int j = 0; j < N; ++j) f[j] *= inv * (w[j] + s.offset);
    }
    stn<N>(s.h + row * H + at(i), f);
  };
#pragma unroll
  for (int i = 0; i < KEEP; ++i)
    if (at(i) < H) finish(i, keep[i]);
  for (int i = KEEP; at(i) < H; ++i) {
    float f[N];
    ldn<N>(xr + at(i), f);  // this thread's own store above
    finish(i, f);
  }
}

// y = act(gate) * up on packed [T, 2 I] rows, or act(x) on [T, I] rows
template <typename T, int N, bool GATED>
__global__ __launch_bounds__(NT) void act_kernel(
    const T* __restrict__ x, T* __restrict__ y, int64_t T_, int I, int act) {
  const int nv = I / N;
  const int64_t total = T_ * nv;
  for (int64_t i = (int64_t)blockIdx.x * NT + threadIdx.x; i < total;
       i += (int64_t)gridDim.x * NT) {
    const int64_t row = i / nv;
    const int c = (int)(i % nv) * N;
    const T* p = x + row * I * (GATED ? 2 : 1) + c;
    float g[N], u[N];
    ldn<N>(p, g);
    if constexpr (GATED) ldn<N>(p + I, u);
#pragma unroll
    for (int j = 0; j < N; ++j) {
      g[j] = activate(act, g[j]);
      if constexpr (GATED) g[j] *= u[j];
    }
    stn<N>(y + row * I + c, g);
  }
}

template <typename T>
hipError_t stream_norm_t(int mode, const void* const* p, int64_t rows,
                         int parts, int n_rows, int H, float scale,
                         float offset, float eps, hipStream_t stream) {
  const Stream<T> s{(float*)p[0], parts ? nullptr : (const T*)p[1],
                    parts ? (const float*)p[1] : nullptr, parts,
                    (const int64_t*)p[2],
                    (const float*)p[3], (const int32_t*)p[4],
                    (const float*)p[5], (const T*)p[6], n_rows,
                    (const float*)p[7], (const float*)p[8],
                    (const float*)p[9], (const float*)p[10], (T*)p[11], H,
                    scale, offset, eps};
  const dim3 grid((uint32_t)rows);
#define GO(N, M, PARTS, BT)                                                   \
  hipLaunchKernelGGL((stream_norm_kernel<T, N, M, PARTS, BT>), grid, dim3(BT), \
                     0, stream, s)
#define GOM(N)                                                                \
  do {                                                                        \
    if (mode == EMBED) GO(N, EMBED, 0, NT);                                   \
    else if (mode == POST) GO(N, POST, 0, NT);                                \
    else if (mode == ADD) GO(N, ADD, 0, NT);                                  \
    else GO(N, LOOP, 0, NT);                                                  \
  } while (0)
#define GOP(PARTS, BT)                                                        \
  do {                                                                        \
    if (mode == POST) GO(8, POST, PARTS, BT); else GO(8, ADD, PARTS, BT);     \
  } while (0)
  // Ahead, up to 256 rows: past them enough is under way, and of two vectors what is
  // asked for takes the registers of other rows. us, not ahead / by 512 threads / by 256
  // threads, 8 parts, with a norm of the sum and four rows of experts:
  //              1 row              50 rows             256 rows            300 rows
  //   1024   4.2 / 4.2 / 3.6     4.7 / 4.5 / 3.9     6.8 / 5.8 / 5.1     7.2 / 7.2 / 5.8
  //   2048   4.5 / 4.2 / 3.6     6.1 / 5.0 / 4.3     7.9 / 7.3 / 6.7     8.6 / 9.0 / 7.7
  //   4096   6.6 / 4.4 / 5.8     9.9 / 5.8 / 8.3    12.6 /10.4 /12.0    14.1 /12.7 /13.9
  //   5120   8.4 / 6.7          13.5 / 9.0          16.1 /13.5          18.1 /20.4
  if (parts && H > 0 && H % 8 == 0 && (mode == POST || mode == ADD) && rows <= 256) {
    if (H <= NT * 8) GOP(1, NT);
    else if (H <= PT * 8) GOP(1, PT);
    else GOP(2, PT);
  } else if (H % 8 == 0) {
    GOM(8);
  } else {
    GOM(1);
  }
#undef GOP
#undef GOM
#undef GO
  HIP_CHECK_LAST();
  return hipSuccess;
}

template <typename T, bool GATED>
hipError_t act_t(const void* x, void* y, int64_t rows, int I, int act,
                 hipStream_t stream) {
  const int n = I % 8 == 0 ? 8 : 1;
  int64_t blocks = (rows * (I / n) + NT - 1) / NT;
  if (blocks > 4096) blocks = 4096;
  const dim3 grid((uint32_t)blocks), block(NT);
  if (n == 8)
    hipLaunchKernelGGL((act_kernel<T, 8, GATED>), grid, block, 0, stream,
                       (const T*)x, (T*)y, rows, I, act);
  else
    hipLaunchKernelGGL((act_kernel<T, 1, GATED>), grid, block, 0, stream,
                       (const T*)x, (T*)y, rows, I, act);
  HIP_CHECK_LAST();
  return hipSuccess;
}

}  // namespace

extern "C" {

// parts > 0: y are that many partial sums in 32-bit
// ptr: x, y or table, ids, pos, positions, wb, rows, a, b, v, wn, h (null
// where the mode has none): see Stream
hipError_t lds_stream_norm(int f32, int mode, const void* const* ptr,
                           int64_t rows, int parts, int n_rows, int H,
                           float scale, float offset, float eps,
                           hipStream_t stream) {
  if (rows == 0) return hipSuccess;
  return f32 ? stream_norm_t<float>(mode, ptr, rows, parts, n_rows, H, scale,
                                    offset, eps, stream)
             : stream_norm_t<short>(mode, ptr, rows, parts, n_rows, H, scale,
                                    offset, eps, stream);
}

hipError_t lds_act(int f32, int gated, const void* x, void* y, int64_t rows,
                   int I, int act, hipStream_t stream) {
  if (rows == 0 || I == 0) return hipSuccess;
  if (gated)
    return f32 ? act_t<float, true>(x, y, rows, I, act, stream)
               : act_t<short, true>(x, y, rows, I, act, stream);
  return f32 ? act_t<float, false>(x, y, rows, I, act, stream)
             : act_t<short, false>(x, y, rows, I, act, stream);
}

}  // extern "C"
