// linear_bind.h — torch binding of linear_rows.hip, linear_tiles.hip,
// linear_split.hip and linear_act.hip, shared by the extensions. Products go to
// these kernels where their rule holds, else to the library, of many rows in two
// calls where that is faster.
#pragma once
#include <torch/extension.h>
#include <ATen/autocast_mode.h>
#include <ATen/hip/HIPContext.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <torch/csrc/jit/frontend/tracer.h>

#include <hip/hip_runtime.h>

extern "C" {
int lds_linear_rows_parts(int M, int N, int K);
int lds_linear_plain_parts(int M, int N, int K);
hipError_t lds_linear_pair(const void*, const void*, int64_t, const void*,
                           const void*, int64_t, void*, void*, int, int, int,
                           hipStream_t);
int lds_linear_rows_takes(int M, int N, int K, int gated, int parts);
hipError_t lds_linear_rows(const void*, int64_t, const void*, int64_t, void*,
                           float*, int, int, int, int, int, hipStream_t);
hipError_t lds_activated_rows(const void*, int64_t, const void*, int64_t,
                              void*, int, int, int, int, hipStream_t);
hipError_t lds_gated_rows(const void*, int64_t, const void*, int64_t, void*,
                          int, int, int, int, hipStream_t);
int lds_linear_act_rows(int64_t, int64_t, int64_t, int);
hipError_t lds_linear_act(const void*, int64_t, const void*, int64_t, void*,
                          int, int, int, int, int, int, hipStream_t);
hipError_t lds_sum_parts(const float*, void*, int64_t, int, int, int,
                         hipStream_t);
int lds_linear_split_plan(int64_t, int64_t, int64_t);
hipError_t lds_linear_split(const void*, int64_t, const void*, int64_t, void*,
                            float*, int, int, int, int, hipStream_t);
hipError_t lds_lay_weights(const float*, void*, int, int, hipStream_t);
}

namespace linear_bind {

using torch::Tensor;

inline bool rows_of_16_bytes(const Tensor& t) {
  return t.stride(1) == 1 && t.stride(0) % 8 == 0 &&
         t.stride(0) >= t.size(1) && (uintptr_t)t.data_ptr() % 16 == 0;
}

// bf16 matrices on one GPU, of matching sizes, whose product is what this
// header computes and nothing else: autograd, a trace, a dispatch mode or a
// functional transform does not follow it, autocast gives it no other type, and
// both have memory (a tensor known to be zero has none)
inline bool plain_matrices(const Tensor& x, const Tensor& w) {
  if (x.dim() != 2 || w.dim() != 2 || !x.is_cuda() ||
      x.device() != w.device() || x.scalar_type() != at::kBFloat16 ||
      w.scalar_type() != at::kBFloat16 || w.size(1) != x.size(1))
    return false;
  if (at::GradMode::is_enabled() && (x.requires_grad() || w.requires_grad()))
    return false;
  if (c10::impl::TorchDispatchModeTLS::any_modes_set() ||
      (at::autocast::is_autocast_enabled(at::kCUDA) &&
       at::autocast::get_autocast_dtype(at::kCUDA) != at::kBFloat16))
    return false;
  for (const Tensor* t : {&x, &w})
    if (!t->has_storage() || t->layout() != at::kStrided || t->is_neg() ||
        t->_is_zerotensor() || t->_fw_grad(0).defined() ||
        t->key_set().has(c10::DispatchKey::Python))
      return false;
  return !torch::jit::tracer::isTracing();
}

enum Use { PLAIN, GATED, PARTS };

// Whether x w' goes to the framework's kernels (where they are faster:
// lds_linear_rows_takes). What autograd and the like follow stays with the
// library, as do odd layouts.
inline bool few_rows(const Tensor& x, const Tensor& w, Use use) {
  if (!plain_matrices(x, w)) return false;
  const int64_t M = x.size(0), K = x.size(1), N = w.size(0), limit = 1ll << 31;
  // gated ones of more rows have one kernel, which goes by lines: its offsets stay
  // under 4 GiB
  const bool near = use != GATED || M <= 192;
  return M >= 1 && M <= 256 && K >= 8 && K % 8 == 0 && N >= 8 && N % 8 == 0 &&
         N <= (1 << 24) && K <= (1 << 24) && (use != GATED || N % 16 == 0) &&
         lds_linear_rows_takes((int)M, (int)(use == GATED ? N / 2 : N), (int)K,
                               use == GATED, use == PARTS) &&
         rows_of_16_bytes(x) && rows_of_16_bytes(w) &&
         (near || (M < limit / x.stride(0) && N < limit / w.stride(0)));
}

// Rows of a tile where a product of many rows and its activation are one kernel
// (linear_act.hip), else 0
inline int many_rows(const Tensor& x, const Tensor& w, bool gated) {
  if (!plain_matrices(x, w) || (gated && w.size(0) % 2)) return 0;
  const int64_t M = x.size(0), K = x.size(1), limit = 1ll << 31;
  if (K < 1 || M >= limit / K || w.size(0) >= limit / K ||
      !rows_of_16_bytes(x) || !rows_of_16_bytes(w) ||
      M * x.stride(0) >= limit || w.size(0) * w.stride(0) >= limit)
    return 0;               // offsets stay under 4 GiB
  return lds_linear_act_rows(M, w.size(0) / (gated ? 2 : 1), K, gated);
}

// The plan of a product of many rows in parts of K (linear_split.hip), 0 where it
// is not taken
inline int split_plan(const Tensor& x, const Tensor& w) {
  if (!plain_matrices(x, w)) return 0;
  const int plan = lds_linear_split_plan(x.size(0), w.size(0), x.size(1));
  const int64_t limit = 1ll << 31;       // elements: offsets stay under 4 GiB
  return plan && rows_of_16_bytes(x) && rows_of_16_bytes(w) &&
                 x.size(0) < limit / x.stride(0) &&
                 w.size(0) < limit / w.stride(0)
             ? plan
             : 0;
}

// Rows of a product of many that go in a call of their own: those that make up
// whole rounds of tiles of 256 x 256 over the 256 compute units. The library
// often takes a kernel of half the rate where the rest is little (14336 ->
// 4096: 8533 rows 1074 us in one call, 658 in two; 6540 rows 841 and 510; 4096
// -> 28672: 8533 rows 1444 and 1312). 0, one call, where
//   - the rest is two rounds of tiles or more: the second call is as likely as
//     the one to get the poor kernel (5120 -> 10240, 12852 rows: 869 us in one
//     call, 1065 in two; 4096 -> 14336, 11518 rows: 878 and 1039);
//   - it ends in a round that is full but for 1/16: nothing to gain (a pass of
//     8 delta layers, 7749 rows: 31.7 ms, 31.95 with its products to 4096
//     channels in two calls);
//   - it is more than half a round beside a single whole one and K is short:
//     the second call costs what the round would (2048 -> 4096, 6266 rows: 88
//     us and 95).
// Over 1519 draws of 32 sizes and 2048 to 24000 rows: 1.12 times as fast as in
// one call, 0.94 at the least (2048 -> 6144, 9515 rows), where calls of one
// kind differ by 0.03.
inline int64_t whole_rounds(int64_t M, int64_t N, int64_t K) {
  const int64_t across = (N + 255) / 256;
  int64_t down = 256;                     // tiles of rows in whole rounds
  while (down > 1 && across * (down / 2) % 256 == 0) down /= 2;
  const int64_t rows = M / (down * 256) * (down * 256);
  const int64_t rest = (M - rows + 255) / 256 * across, last = rest % 256;
  if (rows < 2048 || rest == 0 || rest >= 512) return 0;
  if (rest <= 128) return rows;
  const bool worth = K >= 4096 || rows / 256 * across >= 512;
  return worth && last > 0 && last <= 240 ? rows : 0;
}

inline void check(hipError_t e) {
  TORCH_CHECK(e == hipSuccess, "linear_rows: ", hipGetErrorString(e));
}

// y: contiguous [M, N], bf16 or (f32) 32-bit
inline void linear_rows(const Tensor& x, const Tensor& w, const Tensor& y,
                        bool f32) {
  const c10::DeviceGuard guard(x.device());
  const int M = (int)x.size(0), K = (int)x.size(1), N = (int)w.size(0);
  const auto wide = x.options().dtype(at::kFloat);
  Tensor part;
  const int parts = lds_linear_plain_parts(M, N, K);
  if (parts > 1) part = torch::empty({parts, M, N}, wide);
  check(lds_linear_rows(
      x.data_ptr(), x.stride(0), w.data_ptr(), w.stride(0), y.data_ptr(),
      parts > 1 ? part.data_ptr<float>() : nullptr, parts, M, N, K, f32,
      at::hip::getCurrentHIPStreamMasqueradingAsCUDA().stream()));
}

inline Tensor linear_rows(const Tensor& x, const Tensor& w, bool f32) {
  Tensor y = torch::empty({x.size(0), w.size(0)},
                          x.options().dtype(f32 ? at::kFloat : at::kBFloat16));
  linear_rows(x, w, y, f32);
  return y;
}

// the parts [parts, M, N] of a product with a plan, and their sum in y if there is
// one
inline Tensor linear_split(const Tensor& x, const Tensor& w, int plan,
                           const Tensor* y) {
  const c10::DeviceGuard guard(x.device());
  const int M = (int)x.size(0), K = (int)x.size(1), N = (int)w.size(0);
  Tensor part = torch::empty({plan >> 16, M, N}, x.options().dtype(at::kFloat));
  check(lds_linear_split(
      x.data_ptr(), x.stride(0), w.data_ptr(), w.stride(0),
      y ? y->data_ptr() : nullptr, part.data_ptr<float>(), plan, M, N, K,
      at::hip::getCurrentHIPStreamMasqueradingAsCUDA().stream()));
  return part;
}

// x [M, K] @ w' of w [N, K]
inline Tensor linear(const Tensor& x, const Tensor& w) {
  if (few_rows(x, w, PLAIN)) return linear_rows(x, w, false);
  if (const int plan = split_plan(x, w)) {
    Tensor y = torch::empty({x.size(0), w.size(0)}, x.options());
    linear_split(x, w, plan, &y);
    return y;
  }
  int64_t whole = 0;
  if (plain_matrices(x, w)) whole = whole_rounds(x.size(0), w.size(0), x.size(1));
  if (whole == 0) return at::matmul(x, w.t());
  Tensor y = torch::empty({x.size(0), w.size(0)}, x.options());
  const int64_t left = x.size(0) - whole;
  const Tensor first = x.narrow(0, 0, whole), rest = x.narrow(0, whole, left);
  Tensor y0 = y.narrow(0, 0, whole), y1 = y.narrow(0, whole, left);
  at::mm_out(y0, first, w.t());
  if (few_rows(rest, w, PLAIN))
    linear_rows(rest, w, y1, false);
  else if (const int plan = split_plan(rest, w))
    linear_split(rest, w, plan, &y1);
  else
    at::mm_out(y1, rest, w.t());
  return y;
}

// the same for a caller that sums the parts of K itself: [M, N], or 32-bit
// [parts, M, N]
inline Tensor linear_parts(const Tensor& x, const Tensor& w) {
  if (!few_rows(x, w, PARTS)) {
    const int plan = split_plan(x, w);
    return plan ? linear_split(x, w, plan, nullptr) : linear_bind::linear(x, w);
  }
  const int M = (int)x.size(0), K = (int)x.size(1), N = (int)w.size(0);
  const int parts = lds_linear_rows_parts(M, N, K);
  if (parts == 1) return linear_rows(x, w, false);
  const c10::DeviceGuard guard(x.device());
  Tensor part = torch::empty({parts, M, N}, x.options().dtype(at::kFloat));
  check(lds_linear_rows(
      x.data_ptr(), x.stride(0), w.data_ptr(), w.stride(0), nullptr,
      part.data_ptr<float>(), parts, M, N, K, 0,
      at::hip::getCurrentHIPStreamMasqueradingAsCUDA().stream()));
  return part;
}

// the same with a 32-bit result; None where the library has to do it
inline c10::optional<Tensor> linear32(const Tensor& x, const Tensor& w) {
  if (!few_rows(x, w, PLAIN)) return c10::nullopt;
  return linear_rows(x, w, true);
}

// x w' and x2 w2' of one shape in a launch, or None: for few rows of short K, whose
// products are one part each
inline c10::optional<std::tuple<Tensor, Tensor>> linear_pair(
    const Tensor& x, const Tensor& w, const Tensor& x2, const Tensor& w2) {
  if (!few_rows(x, w, PLAIN) || !few_rows(x2, w2, PLAIN) ||
      x.sizes() != x2.sizes() || w.sizes() != w2.sizes() ||
      x.stride(0) != x2.stride(0) || w.stride(0) != w2.stride(0) ||
      x.device() != x2.device())
    return c10::nullopt;
  const int M = (int)x.size(0), K = (int)x.size(1), N = (int)w.size(0);
  if (M > 64 || K > 1024 || lds_linear_plain_parts(M, N, K) != 1)
    return c10::nullopt;
  const c10::DeviceGuard guard(x.device());
  Tensor y = torch::empty({M, N}, x.options());
  Tensor y2 = torch::empty({M, N}, x.options());
  check(lds_linear_pair(
      x.data_ptr(), x2.data_ptr(), x.stride(0), w.data_ptr(), w2.data_ptr(),
      w.stride(0), y.data_ptr(), y2.data_ptr(), M, N, K,
      at::hip::getCurrentHIPStreamMasqueradingAsCUDA().stream()));
  return std::make_tuple(y, y2);
}

inline Tensor linear_act(const Tensor& x, const Tensor& w, int64_t act,
                         bool gated, int rows) {
  const c10::DeviceGuard guard(x.device());
  const int M = (int)x.size(0), K = (int)x.size(1);
  const int N = (int)w.size(0) / (gated ? 2 : 1);
  Tensor y = torch::empty({M, N}, x.options());
  check(lds_linear_act(
      x.data_ptr(), x.stride(0), w.data_ptr(), w.stride(0), y.data_ptr(), rows,
      M, N, K, (int)act, gated,
      at::hip::getCurrentHIPStreamMasqueradingAsCUDA().stream()));
  return y;
}

// act(x gate') * (x up') of w [2 N, K] = [gate; up]; None where the product
// and the activation have to be two calls
inline c10::optional<Tensor> gated_linear(const Tensor& x, const Tensor& w,
                                          int64_t act) {
  if (const int rows = many_rows(x, w, true))
    return linear_act(x, w, act, true, rows);
  if (!few_rows(x, w, GATED)) return c10::nullopt;
  const c10::DeviceGuard guard(x.device());
  const int M = (int)x.size(0), K = (int)x.size(1), N = (int)w.size(0) / 2;
  Tensor y = torch::empty({M, N}, x.options());
  check(lds_gated_rows(
      x.data_ptr(), x.stride(0), w.data_ptr(), w.stride(0), y.data_ptr(), M, N,
      K, (int)act, at::hip::getCurrentHIPStreamMasqueradingAsCUDA().stream()));
  return y;
}

// act(x w'), or None as above. Of few rows the kernel that sums the parts of K takes
// the activation too (60 rows, 4096 -> 7168: a launch of 5 us of 24 less), or that of
// the product; one part of more than 64 rows or 128 x 128 channels is left to the
// caller.
inline c10::optional<Tensor> activated_linear(const Tensor& x, const Tensor& w,
                                              int64_t act) {
  // (the sum of parts takes what is below 0 for no activation)
  TORCH_CHECK(act >= 0 && act < 3, "activation ", act);
  if (const int rows = many_rows(x, w, false))
    return linear_act(x, w, act, false, rows);
  if (!few_rows(x, w, PLAIN)) return c10::nullopt;
  const int M = (int)x.size(0), K = (int)x.size(1), N = (int)w.size(0);
  const int parts = lds_linear_plain_parts(M, N, K);
  const bool one = parts == 1 && M <= 64 && N <= 128 * 128;
  if (parts == 1 && !one) return c10::nullopt;
  const c10::DeviceGuard guard(x.device());
  const auto stream =
      at::hip::getCurrentHIPStreamMasqueradingAsCUDA().stream();
  Tensor y = torch::empty({M, N}, x.options());
  if (one) {
    check(lds_activated_rows(x.data_ptr(), x.stride(0), w.data_ptr(),
                             w.stride(0), y.data_ptr(), M, N, K, (int)act,
                             stream));
    return y;
  }
  Tensor part = torch::empty({parts, M, N}, x.options().dtype(at::kFloat));
  check(lds_linear_rows(x.data_ptr(), x.stride(0), w.data_ptr(), w.stride(0),
                        nullptr, part.data_ptr<float>(), parts, M, N, K, 0,
                        stream));
  check(lds_sum_parts(part.data_ptr<float>(), y.data_ptr(), (int64_t)M * N,
                      parts, 0, (int)act, stream));
  return y;
}

// drawn weights [in, out] in 32-bit -> [out, in] in bf16
inline Tensor lay_weights(const Tensor& w) {
  TORCH_CHECK(w.dim() == 2 && w.is_cuda() && w.is_contiguous() &&
                  w.scalar_type() == at::kFloat,
              "lay_weights takes contiguous 32-bit weights on the GPU");
  if (w.size(0) % 8 || w.size(1) % 4 || w.numel() == 0 ||
      w.size(0) > (1 << 21) || (uintptr_t)w.data_ptr() % 16)
    return w.to(at::kBFloat16).t().contiguous();
  const c10::DeviceGuard guard(w.device());
  Tensor out = torch::empty({w.size(1), w.size(0)},
                            w.options().dtype(at::kBFloat16));
  check(lds_lay_weights(
      w.data_ptr<float>(), out.data_ptr(), (int)w.size(0), (int)w.size(1),
      at::hip::getCurrentHIPStreamMasqueradingAsCUDA().stream()));
  return out;
}

inline void bind(pybind11::module& m) {
  m.def("lay_weights", &lay_weights, "[in, out] 32-bit -> [out, in] bf16");
  m.def("linear", &linear, "x @ w' of w [N, K]");
  m.def("linear_parts", &linear_parts, "the same, or its parts of K");
  m.def("linear32", &linear32, "the same with a 32-bit result, or None");
  m.def("linear_pair", &linear_pair, "x @ w' and x2 @ w2' in a launch, or None");
  m.def("gated_linear", &gated_linear,
        "act(x gate') * (x up') of w = [gate; up], or None");
  m.def("activated_linear", &activated_linear, "act(x w'), or None");
  m.def("few_rows",
        [](const Tensor& x, const Tensor& w) { return few_rows(x, w, PLAIN); },
        "whether x @ w' takes the streaming kernel");
  m.def("act_rows", &lds_linear_act_rows,
        "rows of a tile of a product and its activation in one kernel, or 0");
  m.def("split_plan", &lds_linear_split_plan,
        "rows of a tile | parts of K << 16 of such a product of many rows, or 0");
  m.def("whole_rounds", &whole_rounds,
        "rows of [M, K] @ [K, N] that go in a call of their own");
}

}  // namespace linear_bind
