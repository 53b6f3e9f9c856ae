// Host side of the ops in native code: output allocation, argument checks that need tensors, and the sequences of
// launches an expert MLP is made of, one call from Python each.  The kernels are reached through the C ABI of
// libatorch_amd_fp8.so; nothing here computes, synchronises or keeps state between calls.
//
// Why: a launch costs the host about 2.5 us, but a wrapper written in Python (two torch.empty, the current stream,
// a ctypes call with a dozen arguments) costs 11 us, so that small and medium calls were bound by the host: a
// decoding step of an MoE layer took 130 us of host time for 60 us of kernels.
#include <ATen/core/Tensor.h>
#include <ATen/ops/empty.h>
#include <ATen/ops/empty_strided.h>
#include <ATen/ops/stack.h>
#include <ATen/ops/zeros.h>
#include <c10/hip/HIPCachingAllocator.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/utils/pybind.h>

#include <tuple>

#include "../../include/atorch_amd_fp8.h"
#include "routing.hpp"

namespace {

using at::Tensor;
using OptTensor = std::optional<Tensor>;
constexpr int64_t kTile = 128;

void check(int rc) {
  if (__builtin_expect(rc == AAMD_OK, 1)) return;
  if (rc == AAMD_ERR_ARG) throw py::value_error(aamd_last_error());
  throw std::runtime_error(aamd_last_error());
}
// Refuses what the kernels would answer with reads or writes out of range: they see pointers and sizes, not tensors.
void require(bool ok, const char* what) {
  if (__builtin_expect(ok, 1)) return;
  PyErr_SetString(PyExc_AssertionError, what);
  throw py::error_already_set();
}
void check_offsets(const Tensor& goff, int64_t E) {
  require(goff.scalar_type() == at::kLong && goff.numel() == E + 1 && goff.is_contiguous(),
          "group offsets must be int64 [groups + 1] and contiguous");
}
void check_bias(const Tensor& bias, int64_t E, int64_t N) {
  require(bias.dim() == 2 && bias.size(0) == E && bias.size(1) == N && bias.is_contiguous(),
          "bias must be [groups, outputs] and contiguous");
}
void* stream() { return c10::hip::getCurrentHIPStream().stream(); }

void on_gpu(const Tensor& t) {
  if (__builtin_expect(!t.is_cuda(), 0))
    throw py::value_error("atorch_amd ops need tensors on the GPU (there is no CPU path)");
}
template <typename T = void>
T* ptr(const Tensor& t) {
  on_gpu(t);
  return reinterpret_cast<T*>(t.data_ptr());
}
template <typename T = void>
T* ptr(const OptTensor& t) {
  return t.has_value() ? ptr<T>(*t) : nullptr;
}
int dtype_code(at::ScalarType dt, bool quantiser_input = false) {
  if (dt == at::kBFloat16) return AAMD_BF16;
  if (dt == at::kFloat) return AAMD_F32;
  if (dt == at::kHalf && quantiser_input) return AAMD_F16;
  throw py::value_error(std::string("atorch_amd: unsupported dtype ") + c10::toString(dt) +
                        " (bf16 and fp32 are supported; fp16 as quantiser input)");
}
Tensor empty(at::IntArrayRef shape, at::ScalarType dt, const Tensor& like) {
  on_gpu(like);
  return at::empty(shape, at::TensorOptions().dtype(dt).device(like.device()));
}
constexpr auto kFp8 = at::kFloat8_e4m3fn;

// the transposed codes of `rows` columns and ld_t padded tokens
c10::SmallVector<int64_t, 3> qt_shape(int64_t rows, int64_t ld_t, bool blocked) {
  return blocked ? c10::SmallVector<int64_t, 3>{ld_t / kTile, rows, kTile} : c10::SmallVector<int64_t, 3>{rows, ld_t};
}
Tensor alloc_qt(int64_t rows, int64_t ld_t, bool blocked, const Tensor& like) { return empty(qt_shape(rows, ld_t, blocked), kFp8, like); }
int64_t qt_ld(const Tensor& q_t) { return q_t.dim() == 3 ? q_t.size(0) * kTile : q_t.size(1); }
int64_t padded_bound(int64_t rows, int64_t groups) { return (rows / kTile + groups) * kTile; }

// row-wise codes and scales, transposed codes and scales (undefined where not asked for)
struct Quantised {
  Tensor q, s, q_t, s_t;
};
using QuantTuple = std::tuple<OptTensor, OptTensor, Tensor, Tensor>;
OptTensor opt(const Tensor& t) { return t.defined() ? OptTensor(t) : OptTensor(); }

Quantised alloc_dual(int64_t M, int64_t cols, int64_t ld_t, bool rowwise, bool blocked, const Tensor& like) {
  Quantised r;
  if (rowwise) {
    r.q = empty({M, cols}, kFp8, like);
    r.s = empty({M, cols / kTile}, at::kFloat, like);
  }
  r.q_t = alloc_qt(cols, ld_t, blocked, like);
  r.s_t = empty({ld_t / kTile, cols}, at::kFloat, like);
  return r;
}
template <typename T = void>
T* raw(const Tensor& t) {
  return t.defined() ? ptr<T>(t) : nullptr;
}

// ---- quantisers ------------------------------------------------------------------------------
std::tuple<Tensor, Tensor> tile_quant(const Tensor& x, double eps) {
  const int64_t cols = x.size(-1), rows = cols ? x.numel() / cols : 0;
  Tensor q = empty(x.sizes(), kFp8, x);
  std::vector<int64_t> ss(x.sizes().begin(), x.sizes().end());
  ss.back() = cols / kTile;
  Tensor s = empty(ss, at::kFloat, x);
  check(aamd_quant_1x128(ptr(x), dtype_code(x.scalar_type(), true), rows, cols, cols, ptr<uint8_t>(q), ptr<float>(s),
                         (float)eps, stream()));
  return {q, s};
}

std::tuple<Tensor, Tensor> permute_tile_quant(const Tensor& x, const Tensor& row_map, int64_t topk, int64_t n_out, double eps) {
  const int64_t T = x.size(0), cols = x.size(1);
  Tensor q = empty({n_out, cols}, kFp8, x), s = empty({n_out, cols / kTile}, at::kFloat, x);
  check(aamd_permute_quant_1x128(ptr(x), dtype_code(x.scalar_type(), true), T, cols, cols, ptr<int32_t>(row_map), (int)topk,
                                 n_out, ptr<uint8_t>(q), ptr<float>(s), (float)eps, stream()));
  return {q, s};
}

// (without offsets: one group of all rows)
Quantised dual(const Tensor& x, const OptTensor& goff, int64_t E, double eps, int64_t ld_t, bool rowwise, bool blocked) {
  const int64_t M = x.size(0), cols = x.size(1);
  if (goff.has_value()) check_offsets(*goff, E);
  Quantised r = alloc_dual(M, cols, ld_t, rowwise, blocked, x);
  check(aamd_quant_1x128_dual_grouped(ptr(x), dtype_code(x.scalar_type(), true), M, cols, cols, ptr<int64_t>(goff), (int)E,
                                      nullptr, raw<uint8_t>(r.q), raw<float>(r.s), ptr<uint8_t>(r.q_t), ptr<float>(r.s_t),
                                      ld_t, blocked, (float)eps, stream()));
  return r;
}

// Rows [M, cols] of one group with both transposed results row-major, q_t [cols, ld_t] and s_t [cols, ld_t / 128].
QuantTuple dual_rows(const Tensor& x, double eps) {
  const int64_t M = x.size(0), cols = x.size(1), ld_t = (M + kTile - 1) / kTile * kTile;
  Quantised r = alloc_dual(M, cols, ld_t, true, false, x);
  r.s_t = r.s_t.view({cols, ld_t / kTile});
  check(aamd_quant_1x128_dual_grouped(ptr(x), dtype_code(x.scalar_type(), true), M, cols, cols, nullptr, 1, nullptr, ptr<uint8_t>(r.q),
                                      ptr<float>(r.s), ptr<uint8_t>(r.q_t), ptr<float>(r.s_t), ld_t, AAMD_QT_ROWS_SCALES, (float)eps,
                                      stream()));
  return {r.q, r.s, r.q_t, r.s_t};
}

Quantised permute_dual(const Tensor& x, const Tensor& sorted_idx, int64_t topk, const Tensor& goff, int64_t E, double eps,
                       int64_t ld_t, bool rowwise, bool blocked) {
  const int64_t T = x.size(0), cols = x.size(1), M = sorted_idx.numel();
  check_offsets(goff, E);
  Quantised r = alloc_dual(M, cols, ld_t, rowwise, blocked, x);
  check(aamd_permute_quant_1x128_dual_grouped(ptr(x), dtype_code(x.scalar_type(), true), T, cols, cols,
                                              ptr<int64_t>(sorted_idx), (int)topk, M, ptr<int64_t>(goff), (int)E, nullptr,
                                              raw<uint8_t>(r.q), raw<float>(r.s), ptr<uint8_t>(r.q_t), ptr<float>(r.s_t),
                                              ld_t, blocked, (float)eps, stream()));
  return r;
}

// the activation between the two linears, quantised: codes, scales and (keep) the activation itself
std::tuple<Tensor, Tensor, OptTensor> act_quant(const Tensor& fc1, bool glu, bool keep) {
  const int64_t width = fc1.size(-1), F = glu ? width / 2 : width, rows = width ? fc1.numel() / width : 0;
  std::vector<int64_t> sh(fc1.sizes().begin(), fc1.sizes().end());
  sh.back() = F;
  Tensor q = empty(sh, kFp8, fc1);
  Tensor h = keep ? empty(sh, at::kBFloat16, fc1) : Tensor();
  sh.back() = F / kTile;
  Tensor s = empty(sh, at::kFloat, fc1);
  check((glu ? aamd_swiglu_quant_1x128 : aamd_gelu_quant_1x128)(ptr(fc1), rows, F, width, raw(h), ptr<uint8_t>(q), ptr<float>(s),
                                                                stream()));
  return {q, s, opt(h)};
}

// row-wise and transposed codes of the activation (grad undefined) or of the gradient through it
std::tuple<Quantised, Tensor> act_dual(const Tensor& fc1, const Tensor& dh, bool glu, const Tensor& goff, int64_t E, int64_t ld_t,
                                       bool rowwise, bool blocked, bool keep) {
  const int64_t M = fc1.size(0), width = fc1.size(1), F = glu ? width / 2 : width;
  const int64_t cols = glu && dh.defined() ? width : F;
  check_offsets(goff, E);
  Quantised r = alloc_dual(M, cols, ld_t, rowwise, blocked, fc1);
  Tensor kept = keep ? empty({M, cols}, at::kBFloat16, fc1) : Tensor();
  int rc;
  if (!glu)
    rc = aamd_gelu_quant_1x128_dual_grouped(ptr(fc1), raw(dh), M, F, F, ptr<int64_t>(goff), (int)E, nullptr, raw(kept),
                                            raw<uint8_t>(r.q), raw<float>(r.s), ptr<uint8_t>(r.q_t), ptr<float>(r.s_t), ld_t,
                                            blocked, stream());
  else if (!dh.defined())
    rc = aamd_swiglu_quant_1x128_dual_grouped(ptr(fc1), M, F, width, ptr<int64_t>(goff), (int)E, nullptr, raw(kept),
                                              raw<uint8_t>(r.q), raw<float>(r.s), ptr<uint8_t>(r.q_t), ptr<float>(r.s_t), ld_t,
                                              blocked, stream());
  else
    rc = aamd_swiglu_bwd_quant_1x128_dual_grouped(ptr(dh), F, ptr(fc1), width, M, F, ptr<int64_t>(goff), (int)E, nullptr,
                                                  raw(kept), raw<uint8_t>(r.q), raw<float>(r.s), ptr<uint8_t>(r.q_t),
                                                  ptr<float>(r.s_t), ld_t, blocked, stream());
  check(rc);
  return {r, kept};
}

// ---- grouped GEMMs ---------------------------------------------------------------------------
// Is the stack b [E, N, K] the transposed view of a dense [E, K, N]?  (Sizes are multiples of 128.)
bool is_transposed_view(const Tensor& b) {
  return b.dim() == 3 && b.size(2) > 1 && b.stride(1) == 1 && b.stride(2) == b.size(1) && b.stride(0) == b.size(1) * b.size(2);
}
// Is there memory for `bytes` more without the allocator returning what it holds in reserve, which is what it tries before it
// reports that there is none?  (A block at hand may be another stream's; an allocator that cannot say is asked.)
bool memory_at_hand(int64_t bytes, const Tensor& like) {
  namespace allocator = c10::hip::HIPCachingAllocator;
  const c10::DeviceIndex device = like.device().index();
  try {
    size_t largest = 1;  // (0 would ask the driver too, which takes longer)
    allocator::cacheInfo(device, &largest);
    if ((int64_t)largest >= bytes) return true;
    const auto [free, total] = allocator::get()->getMemoryInfo(device);
    const int64_t held = allocator::getDeviceStats(device).reserved_bytes[0].current;
    return (int64_t)free >= bytes && (double)(held + bytes) <= allocator::getMemoryFraction(device) * (double)total;
  } catch (const c10::Error&) {
    return true;
  }
}
// Workspace of a GEMM with block-scaled weights; undefined where it has no use for one, or where there is no memory for it.
Tensor gemm_workspace(int64_t M, int64_t N, int64_t K, int64_t E, bool grouped, bool b_rows, const Tensor& like) {
  const int64_t bytes = aamd_grouped_gemm_fp8_ws_bytes(M, N, K, (int)E, grouped, b_rows);
  if (bytes == 0) return Tensor();
  on_gpu(like);
  if (!memory_at_hand(bytes, like)) return Tensor();
  try {
    return empty({bytes / 4}, at::kFloat, like);
  } catch (const c10::OutOfMemoryError&) {
    return Tensor();
  }
}
Tensor gemm_nt(const Tensor& a, const Tensor& a_s, const Tensor& b, const Tensor& b_s, const OptTensor& goff, const OptTensor& out,
               at::ScalarType out_dtype, const OptTensor& bias) {
  const int64_t M = a.size(0), K = a.size(1), E = b.size(0), N = b.size(1);
  const bool b_rows = is_transposed_view(b), b_tile_scaled = !b_rows && b_s.size(1) == N;
  require(b.size(2) == K && a.stride(1) == 1 && (b_rows || b.is_contiguous()), "rows and weights must share their contraction length");
  require(a_s.numel() >= M * (K / kTile) && b_s.numel() >= E * (b_tile_scaled ? N : N / kTile) * (K / kTile) && a_s.is_contiguous() &&
              (!b_rows || (b_s.dim() == 3 && b_s.size(1) == N / kTile)),
          "scales do not cover the codes");
  // (codes and scales come as views of one layout; who keeps tensors for a backward may have made one of them dense)
  require(b_s.is_contiguous() || (!b_tile_scaled && b_s.dim() == 3 && b_s.transpose(1, 2).is_contiguous()),
          "scales must be dense, in the order of either orientation");
  const Tensor bs = b_rows ? b_s.transpose(1, 2).contiguous() : b_s.contiguous();
  if (goff.has_value()) check_offsets(*goff, E);
  if (bias.has_value()) check_bias(*bias, E, N);
  Tensor c = out.has_value() ? *out : empty({M, N}, out_dtype, a);
  const Tensor ws = b_tile_scaled ? Tensor() : gemm_workspace(M, N, K, E, goff.has_value(), b_rows, a);
  if (ws.defined())
    check(aamd_grouped_gemm_fp8_ws(ptr<uint8_t>(a), a.stride(0), ptr<float>(a_s), ptr<uint8_t>(b), ptr<float>(bs), b_rows,
                                   ptr<int64_t>(goff), (int)E, M, N, K, ptr(c), dtype_code(c.scalar_type()), c.stride(0), ptr(bias),
                                   bias.has_value() ? dtype_code(bias->scalar_type()) : AAMD_NONE, ptr<float>(ws), ws.numel() * 4,
                                   stream()));
  else if (b_rows)
    check(aamd_grouped_gemm_fp8_nn(ptr<uint8_t>(a), a.stride(0), ptr<float>(a_s), ptr<uint8_t>(b), ptr<float>(bs), ptr<int64_t>(goff),
                                   (int)E, M, N, K, ptr(c), dtype_code(c.scalar_type()), c.stride(0), ptr(bias),
                                   bias.has_value() ? dtype_code(bias->scalar_type()) : AAMD_NONE, stream()));
  else
    check(aamd_grouped_gemm_fp8_nt(ptr<uint8_t>(a), a.stride(0), ptr<float>(a_s), ptr<uint8_t>(b), ptr<float>(bs), b_tile_scaled,
                                 ptr<int64_t>(goff), (int)E, nullptr, M, N, K, ptr(c), dtype_code(c.scalar_type()), c.stride(0),
                                 ptr(bias), bias.has_value() ? dtype_code(bias->scalar_type()) : AAMD_NONE, stream()));
  return c;
}

void check_wgrad(const Tensor& dy_t, const Tensor& sdy_t, const Tensor& x_t, const Tensor& sx_t, const Tensor& goff, int64_t N, int64_t K) {
  const int64_t ld_t = qt_ld(dy_t);
  check_offsets(goff, goff.numel() - 1);
  require(x_t.dim() == dy_t.dim() && qt_ld(x_t) == ld_t && dy_t.numel() == N * ld_t && x_t.numel() == K * ld_t &&
              sdy_t.numel() >= ld_t / kTile * N && sx_t.numel() >= ld_t / kTile * K,
          "transposed operands must share their layout and length, with a scale per row and block");
}
// dw[g] (+)= dY_g^T X_g into matrices [N, K] that lie `stride` elements apart
void wgrad_into(const Tensor& dy_t, const Tensor& sdy_t, const Tensor& x_t, const Tensor& sx_t, const Tensor& goff, int64_t N, int64_t K,
                void* dw, at::ScalarType dtype, int64_t stride, bool accumulate) {
  check(aamd_grouped_gemm_fp8_wgrad(ptr<uint8_t>(dy_t), ptr<float>(sdy_t), ptr<uint8_t>(x_t), ptr<float>(sx_t), qt_ld(dy_t),
                                    dy_t.dim() == 3, ptr<int64_t>(goff), (int)(goff.numel() - 1), nullptr, N, K, dw,
                                    dtype_code(dtype), stride, accumulate, stream()));
}
Tensor gemm_wgrad(const Tensor& dy_t, const Tensor& sdy_t, const Tensor& x_t, const Tensor& sx_t, const Tensor& goff,
                  const OptTensor& out, at::ScalarType out_dtype, bool accumulate) {
  const bool blocked = dy_t.dim() == 3;
  const int64_t N = dy_t.size(blocked), K = x_t.size(blocked), E = goff.numel() - 1;
  check_wgrad(dy_t, sdy_t, x_t, sx_t, goff, N, K);
  require(!out.has_value() || (out->dim() == 3 && out->size(0) == E && out->size(1) == N && out->size(2) == K &&
                               out->stride(2) == 1 && out->stride(1) == K),
          "the output must be [groups, N, K] with dense matrices");
  Tensor c = out.has_value() ? *out : empty({E, N, K}, out_dtype, dy_t);
  wgrad_into(dy_t, sdy_t, x_t, sx_t, goff, N, K, ptr(c), c.scalar_type(), E > 1 ? c.stride(0) : N * K, accumulate);
  return c;
}

Tensor transpose_scales(const Tensor& s) {
  Tensor t = empty({s.size(1), s.size(0)}, at::kFloat, s);
  check(aamd_transpose_scales(ptr<float>(s), s.size(0), s.size(1), ptr<float>(t), stream()));
  return t;
}
// C = A @ B^T of one group, 1x128 scales on A, 128x128 or 1x128 scales on B.
Tensor fp8_gemm(const Tensor& a, const Tensor& a_s, const Tensor& b, const Tensor& b_s, at::ScalarType dtype) {
  const int64_t K = a.size(-1), M = K ? a.numel() / K : 0, N = b.size(0), blocks = K / kTile;
  std::vector<int64_t> shape(a.sizes().begin(), a.sizes().end());
  shape.back() = N;
  Tensor c = empty(shape, dtype, a);
  const bool b_tile_scaled = b_s.size(0) == N;
  // Both sides scaled per row, as in the dense weight gradient: the weight-gradient kernel is built for it, but reads
  // the scales block by block.  Two small launches turn them round, which pays for large outputs (us, without and with:
  // 14336 x 4096 x 4096 327 -> 280, x 1024 117 -> 104, x 256 64 -> 58; 4096 x 4096 x 4096 95 -> 100; the results are equal).
  constexpr int64_t kDenseWgradTiles = 2048;  // 128 x 128 outputs
  if (b_tile_scaled && M % kTile == 0 && N % kTile == 0 && (M / kTile) * (N / kTile) >= kDenseWgradTiles) {
    Tensor at = empty({blocks, M}, at::kFloat, a), bt = empty({blocks, N}, at::kFloat, a);
    check(aamd_transpose_scales_pair(ptr<float>(a_s), M, ptr<float>(at), ptr<float>(b_s), N, ptr<float>(bt), blocks, stream()));
    check(aamd_grouped_gemm_fp8_wgrad(ptr<uint8_t>(a), ptr<float>(at), ptr<uint8_t>(b), ptr<float>(bt), K, AAMD_QT_ROWS, nullptr,
                                      1, nullptr, M, N, ptr(c), dtype_code(dtype), M * N, 0, stream()));
    return c;
  }
  const Tensor ws = b_tile_scaled ? Tensor() : gemm_workspace(M, N, K, 1, false, false, a);
  if (ws.defined()) {
    check(aamd_grouped_gemm_fp8_ws(ptr<uint8_t>(a), K, ptr<float>(a_s), ptr<uint8_t>(b), ptr<float>(b_s), 0, nullptr, 1, M, N, K, ptr(c),
                                   dtype_code(dtype), N, nullptr, AAMD_NONE, ptr<float>(ws), ws.numel() * 4, stream()));
    return c;
  }
  check(aamd_grouped_gemm_fp8_nt(ptr<uint8_t>(a), K, ptr<float>(a_s), ptr<uint8_t>(b), ptr<float>(b_s), b_tile_scaled, nullptr, 1,
                                 nullptr, M, N, K, ptr(c), dtype_code(dtype), N, nullptr, AAMD_NONE, stream()));
  return c;
}

// ---- routing ---------------------------------------------------------------------------------
struct Routing {
  Tensor sorted_idx, row_map, goff;
};
Routing alloc_routing(const Tensor& ids, int64_t E, bool want_sorted) {
  // (the kernels read whole words of the ids)
  require((ids.scalar_type() == at::kLong || ids.scalar_type() == at::kInt) && ids.is_contiguous(),
          "expert ids must be int64 or int32 and contiguous");
  const int64_t n = ids.numel();
  Routing r;
  if (want_sorted) r.sorted_idx = empty({n}, at::kLong, ids);
  r.row_map = empty({n}, at::kInt, ids);
  r.goff = empty({E + 1}, at::kLong, ids);
  return r;
}
void run_routing(const Routing& r, const Tensor& ids, int64_t E) {
  const int64_t n = ids.numel();
  // (one workgroup needs no scratch)
  Tensor ws = !aamd_route_takes_scratch(n, E) ? Tensor() : empty({std::max<int64_t>(1, aamd_moe_preprocess_ws_ints(n, (int)E))}, at::kInt, ids);
  check(aamd_moe_preprocess(ptr(ids), ids.scalar_type() == at::kLong, n, (int)E, raw<int64_t>(r.sorted_idx), ptr<int32_t>(r.row_map),
                            ptr<int64_t>(r.goff), raw<int32_t>(ws), stream()));
}
std::tuple<OptTensor, Tensor, Tensor> moe_preprocess(const Tensor& ids, int64_t E, bool want_sorted) {
  const Routing r = alloc_routing(ids, E, want_sorted);
  run_routing(r, ids, E);
  return {opt(r.sorted_idx), r.row_map, r.goff};
}

Tensor invert_permutation(const Tensor& sorted_idx, int64_t n_flat) {
  Tensor m = empty({n_flat}, at::kInt, sorted_idx);
  check(aamd_invert_permutation(ptr<int64_t>(sorted_idx), sorted_idx.numel(), n_flat, ptr<int32_t>(m), stream()));
  return m;
}

Tensor permute_rows(const Tensor& x, const Tensor& row_map, int64_t topk, int64_t n_out) {
  Tensor out = empty({n_out, x.size(1)}, x.scalar_type(), x);
  check(aamd_permute_rows(ptr(x), dtype_code(x.scalar_type()), x.size(0), x.size(1), ptr<int32_t>(row_map), (int)topk, n_out,
                          ptr(out), stream()));
  return out;
}

// rows and weights multiply in their common type: fp32 if either is
at::ScalarType promote(const Tensor& y, const OptTensor& probs) {
  return y.scalar_type() == at::kFloat || (probs.has_value() && probs->scalar_type() == at::kFloat) ? at::kFloat : y.scalar_type();
}
Tensor unpermute_combine(const Tensor& y, const Tensor& row_map, const OptTensor& probs, int64_t T, int64_t topk) {
  const int64_t M = y.size(0), H = y.size(1);
  const int pd = probs.has_value() ? dtype_code(probs->scalar_type()) : AAMD_NONE;
  Tensor out = empty({T, H}, promote(y, probs), y);
  check(aamd_unpermute_combine(ptr(y), dtype_code(y.scalar_type()), M, H, ptr<int32_t>(row_map), ptr(probs), pd, T, (int)topk,
                               ptr(out), stream()));
  return out;
}

Tensor permute_rows_scaled(const Tensor& x, const Tensor& row_map, int64_t topk, int64_t n_out, const OptTensor& probs,
                           at::ScalarType out_dtype) {
  const int64_t T = x.size(0), cols = x.size(1);
  // dropped copies leave rows unwritten
  Tensor out = n_out == T * topk ? empty({n_out, cols}, out_dtype, x)
                                 : at::zeros({n_out, cols}, at::TensorOptions().dtype(out_dtype).device(x.device()));
  const int pd = probs.has_value() ? dtype_code(probs->scalar_type()) : AAMD_NONE;
  check(aamd_permute_rows_scaled(ptr(x), dtype_code(x.scalar_type()), T, cols, ptr<int32_t>(row_map), (int)topk, ptr(probs), pd,
                                 n_out, ptr(out), dtype_code(out_dtype), stream()));
  return out;
}

Tensor unpermute_probs_grad(const Tensor& dout, const Tensor& y, const Tensor& row_map, int64_t topk) {
  const int64_t T = dout.size(0), H = dout.size(1);
  Tensor dp = empty({T, topk}, at::kFloat, dout);
  check(aamd_unpermute_probs_grad(ptr(dout), dtype_code(dout.scalar_type()), ptr(y), dtype_code(y.scalar_type()), y.size(0), H,
                                  ptr<int32_t>(row_map), T, (int)topk, ptr<float>(dp), stream()));
  return dp;
}

// Gradients of the combine: of the permuted rows and (in the weights' type) of the weights, in one pass.
std::tuple<Tensor, Tensor> unpermute_backward(const Tensor& dout, const Tensor& y, const Tensor& row_map, const Tensor& probs,
                                              int64_t topk) {
  const int64_t T = dout.size(0), H = dout.size(1), M = y.size(0);
  // dropped copies leave rows unwritten
  Tensor drows = M == T * topk ? empty({M, H}, y.scalar_type(), y) : at::zeros({M, H}, y.options());
  Tensor dprobs = empty(probs.sizes(), probs.scalar_type(), probs);
  check(aamd_unpermute_backward(ptr(dout), dtype_code(dout.scalar_type()), ptr(y), dtype_code(y.scalar_type()), M, H,
                                ptr<int32_t>(row_map), ptr(probs), dtype_code(probs.scalar_type()), T, (int)topk, ptr(drows),
                                ptr(dprobs), stream()));
  return {drows, dprobs};
}

// Exclusive prefix of rows per group, int64 [E + 1] on `device`, from a host list or an int64 tensor on either side.
Tensor offsets_from_list(const std::vector<int64_t>& counts, at::Device device) {
  Tensor goff = at::empty({(int64_t)counts.size() + 1}, at::TensorOptions().dtype(at::kLong).device(device));
  check(aamd_group_offsets(counts.data(), 1, (int)counts.size(), ptr<int64_t>(goff), stream()));
  return goff;
}
Tensor offsets_from_tensor(const Tensor& counts, at::Device device) {
  require(counts.scalar_type() == at::kLong && counts.is_contiguous(), "rows per group must be int64 and contiguous");
  Tensor goff = at::empty({counts.numel() + 1}, at::TensorOptions().dtype(at::kLong).device(device));
  check(aamd_group_offsets(reinterpret_cast<const int64_t*>(counts.data_ptr()), !counts.is_cuda(), (int)counts.numel(),
                           ptr<int64_t>(goff), stream()));
  return goff;
}

// Equally shaped tensors as one [n, ...] tensor without a copy, when they are dense, lie one behind the other in one
// storage; else nothing.  (Adjacent addresses are not enough: after module.to() or load_state_dict tensors may sit side
// by side in memory and still own separate storages.)
OptTensor stack_of(const std::vector<Tensor>& ts) {
  if (ts.empty()) return {};
  const Tensor& t0 = ts[0];
  const int64_t n = t0.numel();
  if (n == 0) return {};
  const auto* base = static_cast<const char*>(t0.data_ptr());
  const int64_t bytes = n * t0.element_size();
  const auto& storage = t0.storage();
  for (size_t i = 0; i < ts.size(); i++) {
    const Tensor& t = ts[i];
    if (!t.is_contiguous() || t.dtype() != t0.dtype() || t.sizes() != t0.sizes() ||
        static_cast<const char*>(t.data_ptr()) != base + (int64_t)i * bytes || t.storage().data() != storage.data())
      return {};
  }
  if ((t0.storage_offset() + (int64_t)ts.size() * n) * t0.element_size() > (int64_t)storage.nbytes()) return {};
  std::vector<int64_t> sizes{(int64_t)ts.size()}, strides{n};
  sizes.insert(sizes.end(), t0.sizes().begin(), t0.sizes().end());
  strides.insert(strides.end(), t0.strides().begin(), t0.strides().end());
  return t0.detach().as_strided(sizes, strides);
}

// Where tensors of n elements lie that are dense and equally far apart in memory, in one storage or in several (gradient
// buffers that also hold the biases' gradients, tensors taken one by one from the allocator); nothing else fits a
// kernel's base address and stride.  Aligned for the kernels' 16-byte accesses.
struct Spaced {
  void* base;
  int64_t stride;  // elements
};
std::optional<Spaced> spaced(const std::vector<Tensor>& ts, int64_t n) {
  if (ts.empty() || n == 0) return {};
  const Tensor& t0 = ts[0];
  auto* const base = static_cast<char*>(t0.data_ptr());
  const int64_t size = t0.element_size();
  const int64_t step = ts.size() > 1 ? static_cast<char*>(ts[1].data_ptr()) - base : n * size;
  if (step < n * size || step % (8 * size) != 0 || reinterpret_cast<uintptr_t>(base) % 16 != 0) return {};
  for (size_t i = 0; i < ts.size(); i++) {
    const Tensor& t = ts[i];
    if (!t.is_contiguous() || t.numel() != n || t.scalar_type() != t0.scalar_type() || t.device() != t0.device() ||
        static_cast<char*>(t.data_ptr()) != base + (int64_t)i * step)
      return {};
  }
  return Spaced{base, step / size};
}

// 128x128 codes of weights [N, K] into stacked outputs: as stored, and with `transpose` in the other orientation too.  The
// scale is that of a whole block, so the codes are the same bytes either way, and with `one` only one orientation is
// written and the other pair is its transposed view, which gemm_nt reads as well: kStored writes the codes as stored,
// kTurned the transposed ones.  (A weight is read by two products, one along each side.)
enum Written { kBoth = 0, kStored = 1, kTurned = 2 };
struct BlockQuantised {
  Tensor q, s, q_t, s_t;
  int64_t N, K;
  BlockQuantised(int64_t E, int64_t N, int64_t K, bool transpose, int one, const Tensor& like) : N(N), K(K) {
    require(one >= kBoth && one <= kTurned && (transpose || one == kBoth), "one written orientation stands for two");
    if (one != kTurned) {
      q = empty({E, N, K}, kFp8, like);
      s = empty({E, N / kTile, K / kTile}, at::kFloat, like);
    }
    if (transpose && one != kStored) {
      q_t = empty({E, K, N}, kFp8, like);
      s_t = empty({E, K / kTile, N / kTile}, at::kFloat, like);
    }
  }
  // goff: only the codes of experts with rows are made
  void run(const void* w, at::ScalarType dtype, int64_t first, int64_t E, int64_t stride, double eps, const int64_t* goff = nullptr) {
    const int64_t at = first * N * K, at_s = first * (N / kTile) * (K / kTile);
    if (goff != nullptr)
      check(aamd_quant_128x128_grouped(w, dtype_code(dtype, true), E, N, K, stride, goff, raw<uint8_t>(q), raw<float>(s), raw<uint8_t>(q_t),
                                       raw<float>(s_t), (float)eps, stream()));
    else if (!q.defined())
      check(aamd_quant_128x128_t(w, dtype_code(dtype, true), E, N, K, stride, ptr<uint8_t>(q_t) + at, ptr<float>(s_t) + at_s,
                                 (float)eps, stream()));
    else
      check(aamd_quant_128x128(w, dtype_code(dtype, true), E, N, K, stride, ptr<uint8_t>(q) + at, ptr<float>(s) + at_s,
                             q_t.defined() ? ptr<uint8_t>(q_t) + at : nullptr, s_t.defined() ? ptr<float>(s_t) + at_s : nullptr,
                             (float)eps, stream()));
  }
  std::tuple<Tensor, Tensor, OptTensor, OptTensor> get(bool transpose) const {
    if (!transpose) return {q, s, {}, {}};
    if (!q.defined()) return {q_t.transpose(1, 2), s_t.transpose(1, 2), q_t, s_t};
    if (!q_t.defined()) return {q, s, q.transpose(1, 2), s.transpose(1, 2)};
    return {q, s, q_t, s_t};
  }
};
std::tuple<Tensor, Tensor, OptTensor, OptTensor> block_quant(const Tensor& w, double eps, bool transpose, int one, const OptTensor& goff) {
  const int64_t E = w.size(0), N = w.size(1), K = w.size(2);
  if (goff.has_value()) check_offsets(*goff, E);
  BlockQuantised r(E, N, K, transpose, one, w);
  r.run(ptr(w), w.scalar_type(), 0, E, E > 1 ? w.stride(0) : N * K, eps, ptr<int64_t>(goff));
  return r.get(transpose);
}
// The same from separate tensors of one shape: in one launch where they are equally far apart; else in one launch each or,
// small ones, from a copy (us, the one launch / copied / one launch each: 60 x 512 x 512 13 / 28 / 232, 60 x 1024 x 1024
// 44 / 94 / 246, 8 x 1024 x 4096 24 / 51 / 39, 64 x 1408 x 2048 126 / 363 / 290, 8 x 28672 x 4096 661 / 1949 / 702).
constexpr int64_t kWeightOfItsOwn = (int64_t)1 << 21;  // elements
std::tuple<Tensor, Tensor, OptTensor, OptTensor> block_quant_list(const std::vector<Tensor>& ws, double eps, bool transpose, int one) {
  require(!ws.empty() && ws[0].dim() == 2, "weights must be matrices");
  const int64_t E = (int64_t)ws.size(), N = ws[0].size(0), K = ws[0].size(1);
  bool direct = N * K >= kWeightOfItsOwn;
  for (const Tensor& w : ws) {
    require(w.sizes() == ws[0].sizes() && w.scalar_type() == ws[0].scalar_type(), "weights must share shape and type");
    direct = direct && w.is_contiguous() && reinterpret_cast<uintptr_t>(w.data_ptr()) % 16 == 0;
  }
  const auto at = spaced(ws, N * K);
  if (!at.has_value() && !direct) return block_quant(at::stack(ws), eps, transpose, one, {});
  BlockQuantised r(E, N, K, transpose, one, ws[0]);
  if (at.has_value()) r.run(at->base, ws[0].scalar_type(), 0, E, at->stride, eps);
  else
    for (int64_t e = 0; e < E; e++) r.run(ptr(ws[e]), ws[e].scalar_type(), e, 1, N * K, eps);
  return r.get(transpose);
}

// ---- the expert MLP --------------------------------------------------------------------------
// linear -> activation -> linear on rows grouped by expert.  With `row_map` the rows are the tokens of x in the order
// of the routing (row_map, and sorted_idx where a backward follows), and the permute happens inside the quantiser.
// Returns the output and what the backward reads: (out, fc1, qx_t, sx_t, qh_t, sh_t), the last five only with `train`.
// (x, the codes of the weights [E, N1, H] and [E, H2, F] and the biases fit each other, before anything is launched)
void check_mlp(const Tensor& x, const Tensor& q1, const Tensor& q2, const OptTensor& b1, const OptTensor& b2, bool glu) {
  const int64_t E = q1.size(0), n1 = q1.size(1), F = q2.size(2);
  require(x.dim() == 2 && x.is_contiguous() && q1.dim() == 3 && q2.dim() == 3 && x.size(1) == q1.size(2),
          "hidden states and first weights must share the hidden size");
  require(q2.size(0) == E && n1 == (glu ? 2 * F : F), "first and second weights must share the experts and the feed-forward size");
  if (b1.has_value()) check_bias(*b1, E, n1);
  if (b2.has_value()) check_bias(*b2, E, q2.size(1));
}
// Quantiser and GEMM in one launch: the output, or nothing where the sizes or operands are not for it (most: rows a group can have).
bool quant_gemm_fits(const Tensor& rows, int64_t M, int64_t most, const Tensor& q, const Tensor& s) {
  const int64_t E = q.size(0), N = q.size(1), K = q.size(2);
  return rows.scalar_type() == at::kBFloat16 && rows.is_contiguous() && q.is_contiguous() && s.is_contiguous() && s.dim() == 3 &&
         s.size(1) == N / kTile && aamd_quant_grouped_gemm_fits(M, N, K, (int)E, most);
}
OptTensor quant_gemm(int what, const Tensor& rows, const OptTensor& sorted_idx, int64_t topk, int64_t M, int64_t most, const Tensor& q,
                     const Tensor& s, const Tensor& goff, const OptTensor& bias) {
  const int64_t E = q.size(0), N = q.size(1), K = q.size(2);
  if (!quant_gemm_fits(rows, M, most, q, s)) return {};
  Tensor c = empty({M, N}, at::kBFloat16, rows);
  check(aamd_quant_grouped_gemm_fp8_nt(what, ptr(rows), rows.size(1), ptr<int64_t>(sorted_idx), (int)topk, rows.size(0), ptr<uint8_t>(q),
                                       ptr<float>(s), ptr<int64_t>(goff), (int)E, M, N, K, ptr(c), N, ptr(bias),
                                       bias.has_value() ? dtype_code(bias->scalar_type()) : AAMD_NONE, stream()));
  return c;
}
// The same of tokens through the router's choices, which makes the routing too.
OptTensor route_quant_gemm(const Tensor& x, const Tensor& ids, int64_t topk, const Routing& r, const Tensor& q, const Tensor& s,
                           const OptTensor& bias) {
  const int64_t E = q.size(0), N = q.size(1), K = q.size(2), T = x.size(0), M = ids.numel();
  if (!aamd_route_quant_grouped_gemm_fits(T, (int)topk, N, K, (int)E) || !quant_gemm_fits(x, M, std::min(M, T), q, s)) return {};
  Tensor c = empty({M, N}, at::kBFloat16, x);
  check(aamd_route_quant_grouped_gemm_fp8_nt(ptr(ids), ids.scalar_type() == at::kLong, (int)topk, T, ptr(x), K, ptr<uint8_t>(q), ptr<float>(s),
                                             (int)E, N, K, ptr(c), N, ptr(bias), bias.has_value() ? dtype_code(bias->scalar_type()) : AAMD_NONE,
                                             ptr<int64_t>(r.sorted_idx), ptr<int32_t>(r.row_map), ptr<int64_t>(r.goff), stream()));
  return c;
}
// Activation, second GEMM and weighted combine of such rows: the tokens, or nothing where it is not for them.
OptTensor act_gemm_combine(const Tensor& fc1, const Tensor& ids, int64_t topk, const Routing& r, const Tensor& probs, const Tensor& q,
                           const Tensor& s, const OptTensor& bias, bool glu) {
  const int64_t E = q.size(0), N = q.size(1), K = q.size(2), M = ids.numel(), T = M / topk;
  if ((probs.scalar_type() != at::kBFloat16 && probs.scalar_type() != at::kFloat) || !quant_gemm_fits(fc1, M, std::min(M, T), q, s) ||
      !aamd_quant_grouped_gemm_combine_fits(T, (int)topk, N, K, (int)E))
    return {};
  Tensor out = empty({T, N}, probs.scalar_type(), fc1);
  check(aamd_quant_grouped_gemm_combine_fp8_nt(glu ? AAMD_ROWS_SWIGLU : AAMD_ROWS_GELU, ptr(fc1), fc1.size(1), ptr(ids),
                                               ids.scalar_type() == at::kLong, ptr<int32_t>(r.row_map), ptr(probs),
                                               dtype_code(probs.scalar_type()), (int)topk, T, ptr<uint8_t>(q), ptr<float>(s), (int)E, N, K,
                                               ptr(out), ptr(bias), bias.has_value() ? dtype_code(bias->scalar_type()) : AAMD_NONE, stream()));
  return out;
}
using MlpResult = std::tuple<Tensor, OptTensor, OptTensor, OptTensor, OptTensor, OptTensor>;
MlpResult mlp_rows(const Tensor& x, const Tensor& goff, const OptTensor& sorted_idx, const OptTensor& row_map, int64_t topk,
                   const Tensor& q1, const Tensor& s1, const Tensor& q2, const Tensor& s2, const OptTensor& b1,
                   const OptTensor& b2, bool glu, bool train, bool own_routing, OptTensor fused) {
  const int64_t E = q1.size(0);
  check_mlp(x, q1, q2, b1, b2, glu);
  check_offsets(goff, E);
  require(!row_map.has_value() || (row_map->scalar_type() == at::kInt && row_map->is_contiguous() && row_map->numel() == x.size(0) * topk),
          "the row map must be int32 [tokens * topk] and contiguous");
  require(row_map.has_value() == sorted_idx.has_value() && (!row_map.has_value() || sorted_idx->numel() <= row_map->numel()),
          "a routing has a row map and the sorted indices of the rows that are kept");
  require(!row_map.has_value() || !train || (sorted_idx->scalar_type() == at::kLong && sorted_idx->dim() == 1 && sorted_idx->is_contiguous()),
          "the sorted indices must be int64, of one dimension and contiguous");
  const int64_t M = row_map.has_value() ? sorted_idx->numel() : x.size(0);  // (fewer than the map's entries where copies were dropped)
  Quantised qx;
  const int64_t ld_t = padded_bound(M, E);
  const int64_t most = own_routing ? std::min(M, x.size(0)) : M;  // (a token goes to an expert once)
  // (the indices of a routing made here name a row for every row of a group)
  if (!train && own_routing && !fused.has_value()) fused = quant_gemm(AAMD_ROWS_PERMUTED, x, sorted_idx, topk, M, most, q1, s1, goff, b1);
  if (fused.has_value())
    ;
  else if (train)
    qx = row_map.has_value() ? permute_dual(x, *sorted_idx, topk, goff, E, 0.0, ld_t, true, true)
                             : dual(x, goff, E, 0.0, ld_t, true, true);
  else
    std::tie(qx.q, qx.s) = row_map.has_value() ? permute_tile_quant(x, *row_map, topk, M, 0.0) : tile_quant(x, 0.0);
  Tensor fc1 = fused.has_value() ? *fused : gemm_nt(qx.q, qx.s, q1, s1, goff, {}, at::kBFloat16, b1);
  Quantised qh;
  if (train) {
    qh = std::get<0>(act_dual(fc1, Tensor(), glu, goff, E, ld_t, true, true, false));
  } else {
    if (x.scalar_type() == at::kBFloat16)
      if (OptTensor out = quant_gemm(glu ? AAMD_ROWS_SWIGLU : AAMD_ROWS_GELU, fc1, {}, 0, M, most, q2, s2, goff, b2); out.has_value())
        return {*out, {}, {}, {}, {}, {}};
    OptTensor none;
    std::tie(qh.q, qh.s, none) = act_quant(fc1, glu, false);
  }
  Tensor out = gemm_nt(qh.q, qh.s, q2, s2, goff, {}, x.scalar_type(), b2);
  if (!train) return {out, {}, {}, {}, {}, {}};
  return {out, fc1, qx.q_t, qx.s_t, qh.q_t, qh.s_t};
}

MlpResult mlp_forward(const Tensor& x, const Tensor& goff, const OptTensor& sorted_idx, const OptTensor& row_map, int64_t topk,
                      const Tensor& q1, const Tensor& s1, const Tensor& q2, const Tensor& s2, const OptTensor& b1,
                      const OptTensor& b2, bool glu, bool train) {
  return mlp_rows(x, goff, sorted_idx, row_map, topk, q1, s1, q2, s2, b1, b2, glu, train, false, {});
}

// The same from the router's choices, routing and weighted combine included: (out, sorted_idx, row_map, goff) and, with
// `train`, the experts' output and what mlp_forward returns for the backward.
py::tuple layer_forward(const Tensor& x, const Tensor& probs, const Tensor& ids, int64_t topk, const Tensor& q1, const Tensor& s1,
                          const Tensor& q2, const Tensor& s2, const OptTensor& b1, const OptTensor& b2, bool glu, bool train) {
  check_mlp(x, q1, q2, b1, b2, glu);
  require(ids.numel() == x.size(0) * topk && probs.dim() == 2 && probs.size(0) == x.size(0) && probs.size(1) == topk &&
              probs.is_contiguous() && q2.size(1) == x.size(1),
          "router weights and choices are [tokens, topk], and the experts return the hidden size");
  const Routing r = alloc_routing(ids, q1.size(0), true);
  OptTensor fc1;
  if (!train) fc1 = route_quant_gemm(x, ids, topk, r, q1, s1, b1);
  if (!fc1.has_value()) run_routing(r, ids, q1.size(0));
  else if (OptTensor out = act_gemm_combine(*fc1, ids, topk, r, probs, q2, s2, b2, glu); out.has_value())
    return py::make_tuple(*out, r.sorted_idx, r.row_map, r.goff);
  MlpResult m = mlp_rows(x, r.goff, r.sorted_idx, r.row_map, topk, q1, s1, q2, s2, b1, b2, glu, train, true, fc1);
  Tensor& y = std::get<0>(m);
  Tensor out = unpermute_combine(y, r.row_map, probs, x.size(0), topk);
  if (!train) return py::make_tuple(out, r.sorted_idx, r.row_map, r.goff);
  return py::make_tuple(out, r.sorted_idx, r.row_map, r.goff, y, *std::get<1>(m), *std::get<2>(m), *std::get<3>(m),
                        *std::get<4>(m), *std::get<5>(m));
}

// Dual quantiser of a gradient with the sums of its columns per group, in `dtype`: a bias gradient on the side.
std::tuple<Quantised, Tensor> dual_with_sums(int what, const Tensor& x, const Tensor& dh, const Tensor& goff, int64_t E,
                                             int64_t ld_t, double eps, at::ScalarType dtype) {
  const int64_t M = x.size(0), width = x.size(1);
  check_offsets(goff, E);
  Quantised r = alloc_dual(M, width, ld_t, true, true, x);
  Tensor tiles = empty({ld_t / kTile, width}, at::kFloat, x), sums = empty({E, width}, dtype, x);
  check(aamd_dual_grouped_with_sums(what, ptr(x), raw(dh), M, width, ptr<int64_t>(goff), (int)E, ptr<uint8_t>(r.q), ptr<float>(r.s),
                                    ptr<uint8_t>(r.q_t), ptr<float>(r.s_t), ld_t, AAMD_QT_BLOCKED, (float)eps, ptr<float>(tiles), stream()));
  check(aamd_group_sums(ptr<float>(tiles), width, ptr<int64_t>(goff), (int)E, ptr(sums), dtype_code(dtype), stream()));
  return {r, sums};
}

// Gradients of the MLP: (dx, dw1, dw2, db1, db2), the last two where asked for, from the codes of the gradient of its output rows (and
// the sums of these, db2).  With topk > 0 the rows were tokens permuted through row_map, and dx goes back to token order as the sum over
// a token's copies.
using MlpGradients = std::tuple<Tensor, Tensor, Tensor, OptTensor, OptTensor>;
MlpGradients mlp_gradients(const Quantised& qdy, const Tensor& db2, const Tensor& goff, const OptTensor& row_map, int64_t topk, const Tensor& fc1,
                           const Tensor& qx_t, const Tensor& sx_t, const Tensor& qh_t, const Tensor& sh_t, const Tensor& q1_t,
                           const Tensor& s1_t, const Tensor& q2, const Tensor& s2, bool glu, bool transpose_w1, bool want_b1,
                           at::ScalarType x_dtype, at::ScalarType w1_dtype, at::ScalarType w2_dtype) {
  const int64_t E = goff.numel() - 1, ld_t = qt_ld(qx_t);
  Quantised qg;
  Tensor db1;
  // through the second linear: dh = dy @ w2^T ([M, F]); dw2[f, h] = sum_m h[m, f] dy[m, h]
  Tensor dh = gemm_nt(qdy.q, qdy.s, q2, s2, goff, {}, at::kBFloat16, {});
  Tensor dw2 = gemm_wgrad(qh_t, sh_t, qdy.q_t, qdy.s_t, goff, {}, w2_dtype, false);
  // through the activation: the gradient of fc1 is quantised, and summed where there is a bias, by the kernel that
  // computes it, and never written
  if (want_b1)
    std::tie(qg, db1) = dual_with_sums(glu ? AAMD_SUMS_SWIGLU_BWD : AAMD_SUMS_GELU_BWD, fc1, dh, goff, E, ld_t, 0.0, at::kBFloat16);
  else
    qg = std::get<0>(act_dual(fc1, dh, glu, goff, E, ld_t, true, true, false));
  // through the first linear: dx = dfc1 @ w1 ([M, H]); dw1[n, h] = sum_m dfc1[m, n] x[m, h]
  Tensor dx = gemm_nt(qg.q, qg.s, q1_t, s1_t, goff, {}, x_dtype, {});
  if (topk > 0) dx = unpermute_combine(dx, *row_map, {}, row_map->numel() / topk, topk);
  Tensor dw1 = transpose_w1 ? gemm_wgrad(qg.q_t, qg.s_t, qx_t, sx_t, goff, {}, w1_dtype, false)
                            : gemm_wgrad(qx_t, sx_t, qg.q_t, qg.s_t, goff, {}, w1_dtype, false);
  return {dx, dw1, dw2, opt(db1), opt(db2)};
}
void check_gradients(int64_t M, const Tensor& goff, const Tensor& fc1, const Tensor& q1_t, const Tensor& q2, bool glu) {
  check_offsets(goff, goff.numel() - 1);
  require(M == fc1.size(0) && fc1.size(1) == q1_t.size(2) && q2.size(1) * (glu ? 2 : 1) == fc1.size(1),
          "the gradient, the saved activations and the weights do not fit each other");
}
MlpGradients mlp_backward(const Tensor& dy, const Tensor& goff, const OptTensor& row_map, int64_t topk, const Tensor& fc1, const Tensor& qx_t,
                          const Tensor& sx_t, const Tensor& qh_t, const Tensor& sh_t, const Tensor& q1_t, const Tensor& s1_t,
                          const Tensor& q2, const Tensor& s2, bool glu, bool transpose_w1, bool want_b1, bool want_b2,
                          at::ScalarType x_dtype, at::ScalarType w1_dtype, at::ScalarType w2_dtype) {
  const int64_t E = goff.numel() - 1, ld_t = qt_ld(qx_t);
  check_gradients(dy.size(0), goff, fc1, q1_t, q2, glu);
  require(dy.is_contiguous(), "the gradient must be contiguous");
  Quantised qdy;
  Tensor db2;
  if (want_b2) std::tie(qdy, db2) = dual_with_sums(AAMD_SUMS_PLAIN, dy, Tensor(), goff, E, ld_t, 0.0, at::kBFloat16);
  else qdy = dual(dy, goff, E, 0.0, ld_t, true, true);
  return mlp_gradients(qdy, db2, goff, row_map, topk, fc1, qx_t, sx_t, qh_t, sh_t, q1_t, s1_t, q2, s2, glu, transpose_w1, want_b1, x_dtype,
                       w1_dtype, w2_dtype);
}
// Is the gradient of the permuted rows quantised as it is gathered, M rows of H, and not written first by the kernel that makes the
// gradient of the router weights on the side?  In bf16 that saves a write and a read of the rows and costs nothing that they did not; in
// fp32 (the type of fp32 router weights) a row is gathered once per copy at twice the bytes.  Both kernels, replayed in a graph, us,
// written -> gathered, with the weights' gradient and without (T, topk, H): bf16 64, 2, 512 9.9 -> 10.3, 9.2 -> 7.6; 128, 4, 2048 15.2 ->
// 15.6, 13.8 -> 11.8; 1200, 1, 1024 11.1 -> 10.9; 200, 2, 4096 12.3 -> 11.9; 500, 4, 4096 20.1 -> 17.4; 8191, 4, 2048 107 -> 86, 85 -> 57;
// 4096, 8, 7168 363 -> 267, 285 -> 181; fp32 500, 4, 4096 20.4 -> 24.5, 19.8 -> 18.7; 8191, 4, 2048 109 -> 120, 92 -> 88; 16384, 8, 2048
// 396 -> 421, 323 -> 324; 300, 8, 2048 18.6 -> 17.4, 16.0 -> 12.1; 1000, 8, 2048 35.5 -> 40.2, 29.4 -> 31.5.
bool gathers_gradient(int64_t M, int64_t H, int64_t topk, bool bf16, bool want_probs) {
  if (want_probs) return bf16 && M * H >= 5 << 18;
  return bf16 || topk <= 7 || M * H < 1 << 23;
}
// From the gradient of the layer's output: (gradients of the MLP, d_probs in the weights' type where asked for).  y: the experts' rows.
std::tuple<MlpGradients, OptTensor> layer_backward(const Tensor& dout, const Tensor& y, const Tensor& probs, const Tensor& sorted_idx,
                                                   const Tensor& goff, const Tensor& row_map, int64_t topk, const Tensor& fc1,
                                                   const Tensor& qx_t, const Tensor& sx_t, const Tensor& qh_t, const Tensor& sh_t,
                                                   const Tensor& q1_t, const Tensor& s1_t, const Tensor& q2, const Tensor& s2, bool glu,
                                                   bool transpose_w1, bool want_probs, bool want_b1, bool want_b2,
                                                   at::ScalarType x_dtype, at::ScalarType w1_dtype, at::ScalarType w2_dtype) {
  const int64_t E = goff.numel() - 1, ld_t = qt_ld(qx_t), T = dout.size(0), H = dout.size(1), M = T * topk;
  check_gradients(M, goff, fc1, q1_t, q2, glu);
  require(dout.is_contiguous() && y.is_contiguous() && y.size(0) == M && y.size(1) == H && probs.is_contiguous() && probs.numel() == M &&
              row_map.scalar_type() == at::kInt && row_map.is_contiguous() && row_map.numel() == M && sorted_idx.scalar_type() == at::kLong &&
              sorted_idx.is_contiguous() && sorted_idx.numel() == M,
          "the gradient and the routing do not fit each other");
  OptTensor d_probs;
  if (!gathers_gradient(M, H, topk, dout.scalar_type() == at::kBFloat16, want_probs)) {
    Tensor dy;
    if (want_probs) {
      auto [rows, weights] = unpermute_backward(dout, y, row_map, probs, topk);
      dy = rows;
      d_probs = weights;
    } else {
      dy = permute_rows_scaled(dout, row_map, topk, M, probs, at::kBFloat16);
    }
    return {mlp_backward(dy, goff, row_map, topk, fc1, qx_t, sx_t, qh_t, sh_t, q1_t, s1_t, q2, s2, glu, transpose_w1, want_b1, want_b2, x_dtype,
                         w1_dtype, w2_dtype), d_probs};
  }
  if (want_probs) {
    d_probs = empty(probs.sizes(), probs.scalar_type(), probs);
    check(aamd_unpermute_probs_grad_as(ptr(dout), dtype_code(dout.scalar_type()), ptr(y), dtype_code(y.scalar_type()), M, H,
                                       ptr<int32_t>(row_map), T, (int)topk, ptr(*d_probs), dtype_code(probs.scalar_type()), stream()));
  }
  Quantised qdy = alloc_dual(M, H, ld_t, true, true, dout);
  Tensor tiles, db2;
  if (want_b2) tiles = empty({ld_t / kTile, H}, at::kFloat, dout);
  check(aamd_combine_grad_quant_1x128_dual_grouped(ptr(dout), dtype_code(dout.scalar_type()), T, H, ptr<int64_t>(sorted_idx), (int)topk, M,
                                                   ptr(probs), dtype_code(probs.scalar_type()), ptr<int64_t>(goff), (int)E,
                                                   ptr<uint8_t>(qdy.q), ptr<float>(qdy.s), ptr<uint8_t>(qdy.q_t), ptr<float>(qdy.s_t), ld_t,
                                                   AAMD_QT_BLOCKED, raw<float>(tiles), stream()));
  if (want_b2) {
    db2 = empty({E, H}, at::kBFloat16, dout);
    check(aamd_group_sums(ptr<float>(tiles), H, ptr<int64_t>(goff), (int)E, ptr(db2), AAMD_BF16, stream()));
  }
  return {mlp_gradients(qdy, db2, goff, row_map, topk, fc1, qx_t, sx_t, qh_t, sh_t, q1_t, s1_t, q2, s2, glu, transpose_w1, want_b1, x_dtype,
                        w1_dtype, w2_dtype), d_probs};
}

// ---- the grouped linear ----------------------------------------------------------------------
// Forward on rows grouped by expert, from the groups' offsets or (goff empty) their sizes in a host list:
// (out, goff, qx_t, sx_t), the last two only with `train`.
std::tuple<Tensor, Tensor, OptTensor, OptTensor> linear_forward(const Tensor& x, const OptTensor& goff_in,
                                                                const std::vector<int64_t>& splits, const Tensor& qw, const Tensor& sw,
                                                                const OptTensor& bias, at::ScalarType out_dtype, double eps,
                                                                bool train) {
  const int64_t E = qw.size(0);
  require(x.dim() == 2 && x.is_contiguous() && qw.dim() == 3 && x.size(1) == qw.size(2), "GEMM not possible");
  require(goff_in.has_value() || (int64_t)splits.size() == E, "Number of splits should match number of GEMMs.");
  if (goff_in.has_value()) check_offsets(*goff_in, E);
  if (bias.has_value()) check_bias(*bias, E, qw.size(1));
  Quantised q;
  if (!goff_in.has_value() && !train) {  // offsets and codes in one launch
    Tensor goff = at::empty({E + 1}, at::TensorOptions().dtype(at::kLong).device(x.device()));
    q.q = empty(x.sizes(), kFp8, x);
    q.s = empty({x.size(0), x.size(1) / kTile}, at::kFloat, x);
    check(aamd_quant_1x128_with_offsets(ptr(x), dtype_code(x.scalar_type(), true), x.size(0), x.size(1), x.size(1), splits.data(), (int)E,
                                        ptr<int64_t>(goff), ptr<uint8_t>(q.q), ptr<float>(q.s), (float)eps, stream()));
    return {gemm_nt(q.q, q.s, qw, sw, goff, {}, out_dtype, bias), goff, {}, {}};
  }
  Tensor goff = goff_in.has_value() ? *goff_in : offsets_from_list(splits, x.device());
  if (train) q = dual(x, goff, E, eps, padded_bound(x.size(0), E), true, true);
  else std::tie(q.q, q.s) = tile_quant(x, eps);
  return {gemm_nt(q.q, q.s, qw, sw, goff, {}, out_dtype, bias), goff, opt(q.q_t), opt(q.s_t)};
}
// The gradients: (dx, dw, db), db [E, N] in fp32 where asked for (bf16 gradients only).  `mains`: the weights' gradient
// buffers; where they are equally far apart the gradient is added to them (`accumulate`) or written over them and dw is
// empty, else it comes in a buffer of its own.
std::tuple<Tensor, OptTensor, OptTensor> linear_backward(const Tensor& dy, const Tensor& goff, const Tensor& qx_t, const Tensor& sx_t,
                                                         const Tensor& qw_t, const Tensor& sw_t, at::ScalarType dx_dtype,
                                                         const std::optional<std::vector<Tensor>>& mains, at::ScalarType dw_dtype,
                                                         bool accumulate, double eps, bool want_bias) {
  const int64_t E = qw_t.size(0), K = qw_t.size(1), N = qw_t.size(2);
  check_offsets(goff, E);
  std::optional<Spaced> main;
  at::ScalarType main_dtype = at::kFloat;
  if (mains.has_value()) {
    require((int64_t)mains->size() == E, "one gradient buffer per weight");
    for (const Tensor& m : *mains) require(m.numel() == N * K, "a gradient buffer has another size than its weight");
    main_dtype = mains->front().scalar_type();
    if (main_dtype == at::kFloat || main_dtype == at::kBFloat16) main = spaced(*mains, N * K);
  }
  Quantised q;
  Tensor db;
  if (want_bias) std::tie(q, db) = dual_with_sums(AAMD_SUMS_PLAIN, dy, Tensor(), goff, E, qt_ld(qx_t), eps, at::kFloat);
  else q = dual(dy, goff, E, eps, qt_ld(qx_t), true, true);
  Tensor dx = gemm_nt(q.q, q.s, qw_t, sw_t, goff, {}, dx_dtype, {});
  if (!main.has_value()) return {dx, gemm_wgrad(q.q_t, q.s_t, qx_t, sx_t, goff, {}, dw_dtype, false), opt(db)};
  on_gpu(mains->front());
  check_wgrad(q.q_t, q.s_t, qx_t, sx_t, goff, N, K);
  wgrad_into(q.q_t, q.s_t, qx_t, sx_t, goff, N, K, main->base, main_dtype, main->stride, accumulate);
  return {dx, {}, opt(db)};
}

QuantTuple pack(const Quantised& r) { return {opt(r.q), opt(r.s), r.q_t, r.s_t}; }

}  // namespace

PYBIND11_MODULE(_host, m) {
  m.def("tile_quant", &tile_quant);
  m.def("permute_tile_quant", &permute_tile_quant);
  m.def("dual_rows", &dual_rows);
  m.def("dual", [](const Tensor& x, const OptTensor& goff, int64_t E, double eps, int64_t ld_t, bool rowwise, bool blocked) {
    return pack(dual(x, goff, E, eps, ld_t, rowwise, blocked));
  });
  m.def("permute_dual", [](const Tensor& x, const Tensor& sorted_idx, int64_t topk, const Tensor& goff, int64_t E, double eps,
                           int64_t ld_t, bool rowwise, bool blocked) {
    return pack(permute_dual(x, sorted_idx, topk, goff, E, eps, ld_t, rowwise, blocked));
  });
  m.def("act_quant", &act_quant);
  m.def("act_dual", [](const Tensor& fc1, const OptTensor& dh, bool glu, const Tensor& goff, int64_t E, int64_t ld_t, bool rowwise,
                       bool blocked, bool keep) {
    auto [r, kept] = act_dual(fc1, dh.has_value() ? *dh : Tensor(), glu, goff, E, ld_t, rowwise, blocked, keep);
    return std::make_tuple(opt(r.q), opt(r.s), r.q_t, r.s_t, opt(kept));
  });
  m.def("dual_with_sums", [](int what, const Tensor& x, const OptTensor& dh, const Tensor& goff, int64_t E, int64_t ld_t, double eps,
                             at::ScalarType dtype) {
    auto [r, sums] = dual_with_sums(what, x, dh.has_value() ? *dh : Tensor(), goff, E, ld_t, eps, dtype);
    return std::make_tuple(r.q, r.s, r.q_t, r.s_t, sums);
  });
  m.def("qt_shape", [](int64_t rows, int64_t ld_t, bool blocked) {
    const auto shape = qt_shape(rows, ld_t, blocked);
    return std::vector<int64_t>(shape.begin(), shape.end());
  });
  m.def("block_quant", &block_quant, py::arg("w"), py::arg("eps"), py::arg("transpose"), py::arg("one") = (int)kBoth,
        py::arg("group_offsets") = OptTensor());
  m.def("block_quant_list", &block_quant_list, py::arg("ws"), py::arg("eps"), py::arg("transpose"), py::arg("one") = (int)kBoth);
  m.def("gemm_nt", &gemm_nt);
  m.def("gemm_wgrad", &gemm_wgrad);
  m.def("transpose_scales", &transpose_scales);
  m.def("fp8_gemm", &fp8_gemm);
  m.def("moe_preprocess", &moe_preprocess);
  m.def("invert_permutation", &invert_permutation);
  m.def("permute_rows", &permute_rows);
  m.def("unpermute_combine", &unpermute_combine);
  m.def("permute_rows_scaled", &permute_rows_scaled);
  m.def("unpermute_probs_grad", &unpermute_probs_grad);
  m.def("unpermute_backward", &unpermute_backward);
  m.def("offsets_from_list", &offsets_from_list);
  m.def("offsets_from_tensor", &offsets_from_tensor);
  m.def("stack_of", &stack_of);
  m.def("spaced", [](const std::vector<Tensor>& ts, int64_t n) {
    const auto s = spaced(ts, n);
    return s.has_value() ? std::optional(std::make_tuple(reinterpret_cast<uintptr_t>(s->base), s->stride)) : std::nullopt;
  });
  m.def("linear_forward", &linear_forward);
  m.def("linear_backward", &linear_backward);
  m.def("mlp_forward", &mlp_forward);
  m.def("mlp_backward", &mlp_backward);
  m.def("layer_forward", &layer_forward);
  m.def("layer_backward", &layer_backward);
  m.def("gathers_gradient", &gathers_gradient);
}
