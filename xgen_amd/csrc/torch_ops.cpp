// CUDA-key implementations of the xgen_amd operators (xgen_amd/ops.py defines their schemas and
// Meta implementations): argument checks, outputs from the caching allocator, one C ABI call on
// the tensors' current stream.  Native because a small call is bound by this work: in Python
// an operator took 13 to 15 us of host time with its launch (a 256 x 1,024 x 1,024 projection, two
// operators and 8 us of kernels under a module, 35 us a call); from here 5 to 6 (17 us a call).
//
// This library links torch only.  The kernels' library is opened on the first operator call, from
// XGEN_AMD_LIBRARY or this library's own folder, as xgen_amd/_native.py opens it.
#include <ATen/ATen.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>
#include <dlfcn.h>
#include <torch/library.h>

#include <cstdlib>
#include <filesystem>
#include <string>
#include <tuple>

#include "xgen_amd.h"

namespace {

using at::Tensor;
using OptTensor = std::optional<Tensor>;

// The C ABI's entry points, resolved from the opened library.
struct Api {
#define XGEN_API(X)                                                                                         \
  X(xgen_status_string) X(xgen_last_error) X(xgen_quantize_rows) X(xgen_quantize_rows_gelu)                 \
  X(xgen_abs_peak_workspace_bytes) X(xgen_abs_peak) X(xgen_fp8_tensor_scale) X(xgen_fp8_pack)               \
  X(xgen_norm_affine_quant) X(xgen_scaled_mm_fp8) X(xgen_scaled_mm_fp8_exact) X(xgen_quant_matmul_int8)     \
  X(xgen_gate_residual) X(xgen_indexed_modulate) X(xgen_merge_quant) X(xgen_w8a8_gate_residual)
#define XGEN_FIELD(f) decltype(&::f) f;
  XGEN_API(XGEN_FIELD)
  // added within ABI version 1: null where XGEN_AMD_LIBRARY names a library from before it
  decltype(&::xgen_fp8_quantize_tensor) xgen_fp8_quantize_tensor;
};

Api open_api() {
  namespace fs = std::filesystem;
  std::string path;
  if (const char *env = std::getenv("XGEN_AMD_LIBRARY")) {
    path = env;
  } else {
    Dl_info info{};
    TORCH_CHECK(dladdr(reinterpret_cast<void *>(&open_api), &info) && info.dli_fname, "xgen_amd: own path unknown");
    path = (fs::path(info.dli_fname).parent_path() / "libxgen_amd.so").string();
  }
  std::error_code ec;
  path = fs::weakly_canonical(path, ec).string();
  TORCH_CHECK(fs::is_regular_file(path, ec), "xgen_amd native library not found at ", path,
              "; build it with `python -c 'import __graft_entry__ as g; g.build()'`");
  void *handle = dlopen(path.c_str(), RTLD_NOW | RTLD_LOCAL);
  TORCH_CHECK(handle, dlerror());
  Api a{};
#define XGEN_RESOLVE(f)                                                   \
  a.f = reinterpret_cast<decltype(&::f)>(dlsym(handle, #f));              \
  TORCH_CHECK(a.f, path, ": undefined symbol ", #f);
  XGEN_API(XGEN_RESOLVE)
  a.xgen_fp8_quantize_tensor =
      reinterpret_cast<decltype(&::xgen_fp8_quantize_tensor)>(dlsym(handle, "xgen_fp8_quantize_tensor"));
  const auto version = reinterpret_cast<decltype(&::xgen_abi_version)>(dlsym(handle, "xgen_abi_version"));
  TORCH_CHECK(version && version() == XGEN_ABI_VERSION, path, ": unexpected ABI version");
  return a;
}

const Api &api() {
  static const Api a = open_api();  // (a failed opening throws, and is tried again on the next call)
  return a;
}

void check(int status, const char *fn) {
  TORCH_CHECK(status == XGEN_OK, fn, ": ", api().xgen_status_string(status), ": ", api().xgen_last_error());
}

int dtype_code(at::ScalarType t) {
  switch (t) {
    case at::kBFloat16: return XGEN_DTYPE_BF16;
    case at::kHalf: return XGEN_DTYPE_F16;
    case at::kFloat: return XGEN_DTYPE_F32;
    case at::kFloat8_e4m3fn: return XGEN_DTYPE_E4M3;
    case at::kChar: return XGEN_DTYPE_I8;
    default: return XGEN_DTYPE_NONE;
  }
}

bool is_half(const Tensor &t) { return t.scalar_type() == at::kBFloat16 || t.scalar_type() == at::kHalf; }
bool is_quant(at::ScalarType t) { return t == at::kFloat8_e4m3fn || t == at::kChar; }
bool aligned16(const Tensor &t) { return (reinterpret_cast<uintptr_t>(t.data_ptr()) & 15) == 0; }

void on_gpu(const Tensor &first) {
  TORCH_CHECK(first.is_cuda(), "xgen_amd operators require tensors on a HIP (cuda) device");
}
template <class... T>
void on_gpu(const Tensor &first, const T &...rest) {
  on_gpu(first);
  auto same = [&](const auto &t) {
    if constexpr (std::is_same_v<std::decay_t<decltype(t)>, OptTensor>)
      return !t.has_value() || t->device() == first.device();
    else
      return t.device() == first.device();
  };
  TORCH_CHECK((same(rest) && ...), "xgen_amd operators require all tensors on the same device");
}

hipStream_t stream_of(const Tensor &t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

Tensor empty(at::IntArrayRef sizes, at::ScalarType dtype, const Tensor &like) {
  return at::empty(sizes, like.options().dtype(dtype).memory_format(std::nullopt));
}

// t [..., rows, cols] as the kernels read it: unit column stride, every outer stride a multiple of
// row_align elements, a row stride that covers the row, a 16-byte aligned base; other views are
// copied (the kernels move rows in 16-byte pieces).
Tensor kernel_rows(const Tensor &t, int64_t row_align) {
  bool ok = t.stride(-1) == 1 && t.stride(-2) >= t.size(-1) && aligned16(t);
  for (int64_t d = 0; ok && d < t.dim() - 1; ++d) ok = t.stride(d) % row_align == 0;
  return ok ? t : t.clone(at::MemoryFormat::Contiguous);
}

// t contiguous with a 16-byte aligned base (copied if not).
Tensor aligned_flat(const Tensor &t) {
  Tensor c = t.contiguous();
  return aligned16(c) ? c : c.clone();
}

// [..., K] -> [M, K] with unit last stride (copies only if needed).
Tensor rows_view(const Tensor &x) {
  Tensor m = x.dim() == 2 ? x : x.reshape({-1, x.size(-1)});
  if (m.stride(-1) != 1 || (m.size(0) > 1 && m.stride(0) < m.size(1))) m = m.contiguous();
  return m;
}

// --- quantizers --------------------------------------------------------------------
std::tuple<Tensor, Tensor> quantize_rows(const Tensor &x, at::ScalarType out_dtype, int64_t activation) {
  on_gpu(x);
  TORCH_CHECK(is_half(x), "quantize_rows: BF16/F16 input required");
  TORCH_CHECK(activation == XGEN_ACT_NONE || activation == XGEN_ACT_GELU_TANH,
              "quantize_rows: activation must be none or gelu_tanh");
  TORCH_CHECK(is_quant(out_dtype), "quantize_rows: out_dtype must be float8_e4m3fn or int8");
  TORCH_CHECK(x.dim() >= 1 && x.size(-1) > 0, "quantize_rows: input needs a non-empty last dimension");
  const c10::DeviceGuard guard(x.device());
  Tensor q = empty(x.sizes(), out_dtype, x), scale = empty({x.numel() / x.size(-1)}, at::kFloat, x);
  if (x.numel() == 0) return {q, scale};
  const Tensor m = rows_view(x);
  const bool gelu = activation == XGEN_ACT_GELU_TANH;
  check((gelu ? api().xgen_quantize_rows_gelu : api().xgen_quantize_rows)(
            dtype_code(x.scalar_type()), m.data_ptr(), m.size(0), m.size(1), m.stride(0), dtype_code(out_dtype),
            q.data_ptr(), m.size(1), scale.data_ptr<float>(), stream_of(x)),
        gelu ? "xgen_quantize_rows_gelu" : "xgen_quantize_rows");
  return {q, scale};
}

template <class Fn>
Tensor peak_common(const Tensor &x, Fn Api::*entry, const char *fn) {
  on_gpu(x);
  TORCH_CHECK(is_half(x), "abs_peak: BF16/F16 input required");
  TORCH_CHECK(x.numel() > 0, fn, ": empty input");
  const c10::DeviceGuard guard(x.device());
  Tensor out = empty({}, at::kFloat, x);
  const Tensor xc = aligned_flat(x);
  const size_t bytes = api().xgen_abs_peak_workspace_bytes(xc.numel());
  Tensor ws = empty({(int64_t)bytes}, at::kByte, x);
  check((api().*entry)(dtype_code(x.scalar_type()), xc.data_ptr(), xc.numel(), out.data_ptr<float>(), ws.data_ptr(),
                       bytes, stream_of(x)),
        fn);
  return out;
}
Tensor abs_peak(const Tensor &x) { return peak_common(x, &Api::xgen_abs_peak, "xgen_abs_peak"); }
Tensor fp8_tensor_scale(const Tensor &x) {
  return peak_common(x, &Api::xgen_fp8_tensor_scale, "xgen_fp8_tensor_scale");
}

Tensor fp8_pack(const Tensor &x, const Tensor &scale) {
  on_gpu(x, scale);
  TORCH_CHECK(is_half(x), "fp8_pack: BF16/F16 input required");
  TORCH_CHECK(scale.scalar_type() == at::kFloat && scale.numel() == 1, "fp8_pack: one float32 scale required");
  const c10::DeviceGuard guard(x.device());
  Tensor q = empty(x.sizes(), at::kFloat8_e4m3fn, x);
  if (x.numel() == 0) return q;
  const Tensor xc = aligned_flat(x);
  check(api().xgen_fp8_pack(dtype_code(x.scalar_type()), xc.data_ptr(), xc.numel(), scale.data_ptr<float>(),
                            q.data_ptr(), stream_of(x)),
        "xgen_fp8_pack");
  return q;
}

std::tuple<Tensor, Tensor> fp8_quantize_tensor(const Tensor &x) {
  const char *fn = "xgen_fp8_quantize_tensor";
  on_gpu(x);
  TORCH_CHECK(is_half(x), "abs_peak: BF16/F16 input required");
  TORCH_CHECK(x.numel() > 0, "xgen_fp8_tensor_scale: empty input");
  if (!api().xgen_fp8_quantize_tensor) {  // the same scale and bytes in two calls
    const Tensor scale = fp8_tensor_scale(x);
    return {fp8_pack(x, scale), scale};
  }
  const c10::DeviceGuard guard(x.device());
  Tensor q = empty(x.sizes(), at::kFloat8_e4m3fn, x), scale = empty({}, at::kFloat, x);
  const Tensor xc = aligned_flat(x);
  const size_t bytes = api().xgen_abs_peak_workspace_bytes(xc.numel());
  Tensor ws = empty({(int64_t)bytes}, at::kByte, x);
  check(api().xgen_fp8_quantize_tensor(dtype_code(x.scalar_type()), xc.data_ptr(), xc.numel(), q.data_ptr(),
                                       scale.data_ptr<float>(), ws.data_ptr(), bytes, stream_of(x)),
        fn);
  return {q, scale};
}

std::tuple<Tensor, Tensor, Tensor> norm_affine_quant(const Tensor &x_in, const OptTensor &weight, const Tensor &scale_in,
                                                     const Tensor &shift_in, const Tensor &indices, double eps,
                                                     int64_t norm_kind, at::ScalarType out_dtype, bool return_normed) {
  on_gpu(x_in, weight, scale_in, shift_in, indices);
  TORCH_CHECK(x_in.dim() == 3 && x_in.scalar_type() == at::kBFloat16 && x_in.stride(2) == 1 && x_in.size(2) > 0,
              "norm_affine_quant: BF16 [B,S,H] with last stride 1 required");
  const int64_t B = x_in.size(0), S = x_in.size(1), H = x_in.size(2);
  TORCH_CHECK(H <= XGEN_NORM_MAX_WIDTH, "norm_affine_quant: H <= 8192 required");
  TORCH_CHECK(!weight || (weight->dim() == 1 && weight->size(0) == H && weight->is_contiguous() &&
                          (weight->scalar_type() == at::kBFloat16 || weight->scalar_type() == at::kFloat)),
              "norm_affine_quant: BF16/F32 norm weight [H] or None required");
  TORCH_CHECK(scale_in.dim() == 2 && scale_in.size(0) > 0 && scale_in.size(1) == H &&
                  shift_in.sizes() == scale_in.sizes() && scale_in.scalar_type() == at::kBFloat16 &&
                  shift_in.scalar_type() == at::kBFloat16 && scale_in.stride(1) == 1 && shift_in.stride(1) == 1,
              "norm_affine_quant: BF16 tables [T,H] with last stride 1 required");
  TORCH_CHECK(indices.dim() == 1 && indices.size(0) == S && indices.scalar_type() == at::kLong && indices.is_contiguous(),
              "norm_affine_quant: contiguous INT64 indices [S] required");
  TORCH_CHECK(0 < eps && eps < 1, "norm_affine_quant: eps must be in (0, 1)");
  const int64_t base = norm_kind & ~(int64_t)XGEN_NORM_SCALE_ONE_PLUS;
  TORCH_CHECK(base == XGEN_NORM_LAYER || base == XGEN_NORM_RMS,
              "norm_affine_quant: norm_kind must be 0 (layer) or 1 (rms), optionally | 0x100 (scale is 1 + scale)");
  TORCH_CHECK(is_quant(out_dtype), "norm_affine_quant: out_dtype must be float8_e4m3fn or int8");
  const c10::DeviceGuard guard(x_in.device());
  const int64_t rows = B * S;
  Tensor q = empty({rows, H}, out_dtype, x_in), s = empty({rows}, at::kFloat, x_in);
  Tensor normed = return_normed ? empty({rows, H}, at::kBFloat16, x_in) : empty({0}, at::kBFloat16, x_in);
  if (rows == 0) return {q, s, normed};
  const Tensor x = kernel_rows(x_in, 8), scale = kernel_rows(scale_in, 8), shift = kernel_rows(shift_in, 8);
  const Tensor w = weight ? aligned_flat(*weight) : Tensor();
  check(api().xgen_norm_affine_quant(
            x.data_ptr(), B, S, H, x.stride(0), x.stride(1), (int)norm_kind, weight ? w.data_ptr() : nullptr,
            weight ? dtype_code(w.scalar_type()) : XGEN_DTYPE_NONE, (float)eps, scale.data_ptr(), scale.stride(0),
            shift.data_ptr(), shift.stride(0), scale.size(0), indices.data_ptr<int64_t>(), dtype_code(out_dtype),
            q.data_ptr(), s.data_ptr<float>(), return_normed ? normed.data_ptr() : nullptr, stream_of(x)),
        "xgen_norm_affine_quant");
  return {q, s, normed};
}

// --- GEMMs ---------------------------------------------------------------------------
void mm_check(const Tensor &a, const Tensor &w, const Tensor &a_scale, const Tensor &w_scale, const OptTensor &bias,
              at::ScalarType out_dtype, int64_t activation) {
  TORCH_CHECK(is_quant(a.scalar_type()) && w.scalar_type() == a.scalar_type(),
              "scaled_mm: operands must both be float8_e4m3fn or both int8");
  TORCH_CHECK(a.dim() == 2 && w.dim() == 2 && a.size(1) == w.size(1), "scaled_mm: a [M,K] and w [N,K] required");
  const int64_t M = a.size(0), K = a.size(1), Nf = w.size(0);
  TORCH_CHECK(a_scale.scalar_type() == at::kFloat && (a_scale.numel() == 1 || a_scale.numel() == M),
              "scaled_mm: float32 activation scale with 1 or M elements required");
  TORCH_CHECK(w_scale.scalar_type() == at::kFloat && (w_scale.numel() == 1 || w_scale.numel() == Nf),
              "scaled_mm: float32 weight scale with 1 or N elements required");
  TORCH_CHECK(!bias || (bias->dim() == 1 && bias->size(0) == Nf && (is_half(*bias) || bias->scalar_type() == at::kFloat)),
              "scaled_mm: bias [N] of BF16/F16/F32 required");
  TORCH_CHECK(out_dtype == at::kBFloat16 || out_dtype == at::kHalf, "scaled_mm: out_dtype must be bfloat16 or float16");
  TORCH_CHECK(activation == XGEN_ACT_NONE || activation == XGEN_ACT_GELU_TANH,
              "scaled_mm: activation must be 0 (none) or 1 (gelu_tanh)");
  TORCH_CHECK(K % 16 == 0 && Nf % 16 == 0, "scaled_mm: K and N must be multiples of 16");
}

// The operands of one product as the C ABI takes them (views it cannot read are copied).
struct MmOperands {
  Tensor a, w, a_scale, w_scale, bias;
  int64_t sa_stride, sw_stride;
  int bias_dtype;
  const void *bias_ptr;
  MmOperands(const Tensor &a_in, const Tensor &w_in, const Tensor &sa, const Tensor &sw, const OptTensor &b)
      : a(kernel_rows(a_in, 16)), w(kernel_rows(w_in, 16)), a_scale(sa.contiguous()), w_scale(sw.contiguous()) {
    if (b) bias = b->contiguous();
    sa_stride = a_scale.numel() == a.size(0) && a.size(0) > 1 ? 1 : 0;
    sw_stride = w_scale.numel() == w.size(0) && w.size(0) > 1 ? 1 : 0;
    bias_dtype = b ? dtype_code(bias.scalar_type()) : XGEN_DTYPE_NONE;
    bias_ptr = b ? bias.data_ptr() : nullptr;
  }
};

std::tuple<Tensor, Tensor> scaled_mm(const Tensor &a, const Tensor &w, const Tensor &a_scale, const Tensor &w_scale,
                                     const OptTensor &bias, at::ScalarType out_dtype, int64_t activation,
                                     bool return_acc, bool exact) {
  on_gpu(a, w, a_scale, w_scale, bias);
  mm_check(a, w, a_scale, w_scale, bias, out_dtype, activation);
  const bool fp8 = a.scalar_type() == at::kFloat8_e4m3fn;
  TORCH_CHECK(!exact || fp8, "scaled_mm: exact accumulation applies to FP8 operands");
  const c10::DeviceGuard guard(a.device());
  const int64_t M = a.size(0), K = a.size(1), Nf = w.size(0);
  Tensor out = empty({M, Nf}, out_dtype, a);
  Tensor acc = return_acc ? empty({M, Nf}, fp8 ? at::kFloat : at::kInt, a) : empty({0}, fp8 ? at::kFloat : at::kInt, a);
  if (M == 0) return {out, acc};
  const MmOperands o(a, w, a_scale, w_scale, bias);
  void *acc_ptr = return_acc ? acc.data_ptr() : nullptr;
  const hipStream_t stream = stream_of(a);
  if (fp8) {
    check((exact ? api().xgen_scaled_mm_fp8_exact : api().xgen_scaled_mm_fp8)(
              o.a.data_ptr(), o.a.stride(0), o.w.data_ptr(), o.w.stride(0), M, Nf, K, o.a_scale.data_ptr<float>(),
              o.sa_stride, o.w_scale.data_ptr<float>(), o.sw_stride, o.bias_ptr, o.bias_dtype, (int)activation,
              out.data_ptr(), dtype_code(out_dtype), out.stride(0), static_cast<float *>(acc_ptr), stream),
          exact ? "xgen_scaled_mm_fp8_exact" : "xgen_scaled_mm_fp8");
  } else {
    check(api().xgen_quant_matmul_int8(
              o.a.data_ptr(), o.a.stride(0), o.w.data_ptr(), o.w.stride(0), M, Nf, K, o.a_scale.data_ptr<float>(),
              o.sa_stride, o.w_scale.data_ptr<float>(), o.sw_stride, o.bias_ptr, o.bias_dtype, (int)activation,
              out.data_ptr(), dtype_code(out_dtype), out.stride(0), static_cast<int32_t *>(acc_ptr), stream),
          "xgen_quant_matmul_int8");
  }
  return {out, acc};
}

Tensor scaled_mm_gate_residual(const Tensor &a, const Tensor &w, const Tensor &a_scale, const Tensor &w_scale,
                               const OptTensor &bias, const Tensor &residual_in, const Tensor &gate_in,
                               const Tensor &indices_in) {
  on_gpu(a, w, a_scale, w_scale, bias, residual_in, gate_in, indices_in);
  mm_check(a, w, a_scale, w_scale, bias, at::kBFloat16, XGEN_ACT_NONE);
  const int64_t M = a.size(0), K = a.size(1), Nf = w.size(0);
  TORCH_CHECK(residual_in.dim() == 2 && residual_in.size(0) == M && residual_in.size(1) == Nf &&
                  residual_in.scalar_type() == at::kBFloat16,
              "scaled_mm_gate_residual: residual BF16 [M, N] required");
  TORCH_CHECK(gate_in.dim() == 2 && gate_in.size(1) == Nf && gate_in.size(0) > 0 && gate_in.scalar_type() == at::kBFloat16,
              "scaled_mm_gate_residual: gate_table BF16 [T, N] required");
  TORCH_CHECK(indices_in.dim() == 1 && indices_in.scalar_type() == at::kLong && indices_in.size(0) > 0 &&
                  M % indices_in.size(0) == 0,
              "scaled_mm_gate_residual: int64 indices [S] with M % S == 0 required");
  const c10::DeviceGuard guard(a.device());
  Tensor out = empty({M, Nf}, at::kBFloat16, a);
  if (M == 0) return out;
  const MmOperands o(a, w, a_scale, w_scale, bias);
  const Tensor residual = kernel_rows(residual_in, 8), gate = kernel_rows(gate_in, 8), indices = indices_in.contiguous();
  check(api().xgen_w8a8_gate_residual(
            dtype_code(a.scalar_type()), o.a.data_ptr(), o.a.stride(0), o.w.data_ptr(), o.w.stride(0), M, Nf, K,
            o.a_scale.data_ptr<float>(), o.sa_stride, o.w_scale.data_ptr<float>(), o.sw_stride, o.bias_ptr,
            o.bias_dtype, residual.data_ptr(), residual.stride(0), gate.data_ptr(), gate.stride(0), gate.size(0),
            indices.data_ptr<int64_t>(), indices.size(0), out.data_ptr(), out.stride(0), stream_of(a)),
        "xgen_w8a8_gate_residual");
  return out;
}

// --- indexed rows -----------------------------------------------------------------------
Tensor gate_residual(const Tensor &residual_in, const Tensor &branch_in, const Tensor &gate_in, const Tensor &indices_in) {
  on_gpu(residual_in, branch_in, gate_in, indices_in);
  TORCH_CHECK(residual_in.dim() == 3 && branch_in.sizes() == residual_in.sizes() && residual_in.size(2) > 0,
              "gate_residual: residual/branch [B,S,H] shapes must match");
  const int64_t B = residual_in.size(0), S = residual_in.size(1), H = residual_in.size(2);
  TORCH_CHECK(gate_in.dim() == 2 && gate_in.size(0) > 0 && gate_in.size(1) == H, "gate_residual: gate_table [T,H] required");
  TORCH_CHECK(indices_in.dim() == 1 && indices_in.size(0) == S && indices_in.scalar_type() == at::kLong,
              "gate_residual: int64 indices [S] required");
  TORCH_CHECK(residual_in.scalar_type() == at::kBFloat16 && branch_in.scalar_type() == at::kBFloat16 &&
                  gate_in.scalar_type() == at::kBFloat16,
              "gate_residual: BF16 inputs required");
  const c10::DeviceGuard guard(residual_in.device());
  Tensor out = empty(residual_in.sizes(), at::kBFloat16, residual_in);
  if (out.numel() == 0) return out;
  const Tensor residual = kernel_rows(residual_in, 8), branch = kernel_rows(branch_in, 8), gate = kernel_rows(gate_in, 8);
  const Tensor indices = indices_in.contiguous();
  check(api().xgen_gate_residual(residual.data_ptr(), residual.stride(0), residual.stride(1), branch.data_ptr(),
                                 branch.stride(0), branch.stride(1), gate.data_ptr(), gate.stride(0), gate.size(0),
                                 indices.data_ptr<int64_t>(), B, S, H, out.data_ptr(), stream_of(residual)),
        "xgen_gate_residual");
  return out;
}

Tensor indexed_modulate(const Tensor &x_in, const Tensor &scale_in, const Tensor &shift_in, const Tensor &indices_in,
                        bool scale_is_one_plus) {
  on_gpu(x_in, scale_in, shift_in, indices_in);
  TORCH_CHECK(x_in.dim() == 3 && x_in.size(2) > 0, "indexed_modulate: x [B,S,H] required");
  const int64_t B = x_in.size(0), S = x_in.size(1), H = x_in.size(2);
  TORCH_CHECK(scale_in.dim() == 2 && scale_in.size(0) > 0 && scale_in.size(1) == H && shift_in.sizes() == scale_in.sizes(),
              "indexed_modulate: scale/shift tables [T,H] required");
  TORCH_CHECK(indices_in.dim() == 1 && indices_in.size(0) == S && indices_in.scalar_type() == at::kLong,
              "indexed_modulate: int64 indices [S] required");
  TORCH_CHECK(x_in.scalar_type() == at::kBFloat16 && scale_in.scalar_type() == at::kBFloat16 &&
                  shift_in.scalar_type() == at::kBFloat16,
              "indexed_modulate: BF16 inputs required");
  const c10::DeviceGuard guard(x_in.device());
  Tensor out = empty(x_in.sizes(), at::kBFloat16, x_in);
  if (out.numel() == 0) return out;
  const Tensor x = kernel_rows(x_in, 8), scale = kernel_rows(scale_in, 8), shift = kernel_rows(shift_in, 8);
  const Tensor indices = indices_in.contiguous();
  check(api().xgen_indexed_modulate(x.data_ptr(), x.stride(0), x.stride(1), scale.data_ptr(), scale.stride(0),
                                    shift.data_ptr(), shift.stride(0), scale.size(0), indices.data_ptr<int64_t>(), B, S,
                                    H, scale_is_one_plus ? 1 : 0, out.data_ptr(), stream_of(x)),
        "xgen_indexed_modulate");
  return out;
}

std::tuple<Tensor, Tensor> merge_quant(const Tensor &x, at::ScalarType out_dtype) {
  constexpr int64_t kMaxWidth = 16384;
  on_gpu(x);
  TORCH_CHECK(x.dim() == 5 && x.scalar_type() == at::kBFloat16,
              "merge_quant: BF16 back_recv [splits, owners, seq, batch, chunk] required");
  const int64_t splits = x.size(0), owners = x.size(1), seq = x.size(2), batch = x.size(3), chunk = x.size(4);
  TORCH_CHECK(splits > 0 && owners > 0 && chunk > 0 && chunk % 8 == 0,
              "merge_quant: chunk must be a positive multiple of 8");
  const int64_t width = splits * owners * chunk;
  TORCH_CHECK(width <= kMaxWidth, "merge_quant: splits*owners*chunk must be <= ", kMaxWidth);
  TORCH_CHECK(seq * batch < (int64_t(1) << 31), "merge_quant: seq*batch must be below 2^31");
  TORCH_CHECK(is_quant(out_dtype), "merge_quant: out_dtype must be float8_e4m3fn or int8");
  const c10::DeviceGuard guard(x.device());
  Tensor q = empty({batch * seq, width}, out_dtype, x), scale = empty({batch * seq}, at::kFloat, x);
  if (q.numel() == 0) return {q, scale};
  const Tensor xc = aligned_flat(x);
  check(api().xgen_merge_quant(dtype_code(out_dtype), xc.data_ptr(), splits, owners, seq, batch, chunk, q.data_ptr(),
                               scale.data_ptr<float>(), stream_of(x)),
        "xgen_merge_quant");
  return {q, scale};
}

}  // namespace

TORCH_LIBRARY_IMPL(xgen_amd, CUDA, m) {
  m.impl("quantize_rows", quantize_rows);
  m.impl("abs_peak", abs_peak);
  m.impl("fp8_tensor_scale", fp8_tensor_scale);
  m.impl("fp8_pack", fp8_pack);
  m.impl("fp8_quantize_tensor", fp8_quantize_tensor);
  m.impl("norm_affine_quant", norm_affine_quant);
  m.impl("scaled_mm", scaled_mm);
  m.impl("scaled_mm_gate_residual", scaled_mm_gate_residual);
  m.impl("gate_residual", gate_residual);
  m.impl("indexed_modulate", indexed_modulate);
  m.impl("merge_quant", merge_quant);
}
