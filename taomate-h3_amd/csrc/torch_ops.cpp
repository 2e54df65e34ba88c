// The tensor wrappers of ops.py in native code: the same checks, the same
// output allocations and the same C entry points, without the interpreter
// between them.  Each function takes torch tensors and the raw stream of the
// first one's device, and returns None for anything out of the ordinary (a
// wrong type, shape, stride or device, an empty tensor, a call that the library
// refuses): ops.py then runs its own checks on the same arguments and raises
// what it always raised.  Nothing is kept between calls.  The interpreter lock is
// released from the checks to the last launch, as ctypes releases it: a launch
// queue that is full, or the first SwiGLU call's wait for its table, holds up no
// other thread of the program.
//
// What it saves is the host's time per call, which bounds every call of a few
// dozen rows (measured on an MI355X host, Python wrapper -> this: quantizer 11.1
// -> 5.7 us, scaled GEMM 13.7 -> 5.5 us, of which the launch itself is about 3).
#include <torch/extension.h>

#include <optional>
#include <tuple>

#include "../../include/taomate_h3_amd.h"

using at::Tensor;
using Opt = std::optional<Tensor>;
using OptInt = std::optional<int64_t>;
using Pair = std::tuple<Tensor, Tensor>;
using Three = std::tuple<Tensor, Tensor, Tensor>;
using Triple = std::tuple<Opt, Opt, Opt>;

namespace {

bool on(const Tensor& t, const Tensor& first) { return t.is_cuda() && t.device() == first.device(); }

// A 2-D tensor of the given type with unit stride along its rows.
bool rows_2d(const Tensor& t, at::ScalarType type) {
    return t.scalar_type() == type && t.dim() == 2 && (t.size(1) <= 1 || t.stride(1) == 1);
}

at::ScalarType code_type(int64_t fmt) { return fmt == H3Q_FMT_INT8 ? at::kChar : at::kFloat8_e4m3fn; }

bool valid_fmt(int64_t fmt) { return fmt == H3Q_FMT_INT8 || fmt == H3Q_FMT_E4M3FN; }

Tensor empty(const Tensor& like, at::IntArrayRef shape, at::ScalarType type) {
    return at::empty(shape, like.options().dtype(type));
}

bool scales_ok(const Tensor& s, const Tensor& first, int64_t count) {
    return on(s, first) && s.scalar_type() == at::kFloat && s.numel() == count && s.is_contiguous();
}

void* stream_of(int64_t raw) { return reinterpret_cast<void*>(raw); }

float* floats(const Tensor& t) { return static_cast<float*>(t.data_ptr()); }

const void* ptr(const Opt& t) { return t ? t->data_ptr() : nullptr; }

std::optional<Pair> quant_rows(const Tensor& x, int64_t fmt, int64_t rounding, Opt codes, Opt scales, int64_t stream) {
    if (!x.is_cuda() || !rows_2d(x, at::kBFloat16) || !valid_fmt(fmt) || x.size(0) == 0) return std::nullopt;
    const int64_t rows = x.size(0), cols = x.size(1);
    if (codes && !(on(*codes, x) && rows_2d(*codes, code_type(fmt)) && codes->size(0) == rows && codes->size(1) == cols))
        return std::nullopt;
    if (scales && !scales_ok(*scales, x, rows)) return std::nullopt;
    if (!codes) codes = empty(x, {rows, cols}, code_type(fmt));
    if (!scales) scales = empty(x, {rows, 1}, at::kFloat);
    if (h3q_quant_rows(x.data_ptr(), rows, cols, x.stride(0), (int)fmt, (int)rounding, codes->data_ptr(),
                       codes->stride(0), floats(*scales), stream_of(stream)))
        return std::nullopt;
    return Pair(*codes, *scales);
}

std::optional<Pair> quant_rows_tiled(const Tensor& x, int64_t fmt, int64_t rounding, Opt codes, int64_t row0,
                                     Opt scales, int64_t stream) {
    if (!x.is_cuda() || !rows_2d(x, at::kBFloat16) || !valid_fmt(fmt) || x.size(0) == 0) return std::nullopt;
    const int64_t rows = x.size(0), cols = x.size(1);
    if (cols % 128 || row0 < 0 || (!codes && row0)) return std::nullopt;
    if (codes && !(on(*codes, x) && codes->scalar_type() == code_type(fmt) && codes->dim() == 2 &&
                   codes->size(1) == cols && codes->is_contiguous() && codes->size(0) % 16 == 0 &&
                   row0 + rows <= codes->size(0)))
        return std::nullopt;
    if (scales && !scales_ok(*scales, x, rows)) return std::nullopt;
    if (!codes) codes = empty(x, {(rows + 15) / 16 * 16, cols}, code_type(fmt));
    if (!scales) scales = empty(x, {rows, 1}, at::kFloat);
    if (h3q_quant_rows_tiled(x.data_ptr(), rows, cols, x.stride(0), (int)fmt, (int)rounding, row0, codes->data_ptr(),
                             floats(*scales), stream_of(stream)))
        return std::nullopt;
    return Pair(*codes, *scales);
}

// Per row, per tensor, or -1 for neither.
int scale_kind(const Tensor& s, const Tensor& first, int64_t count) {
    if (!on(s, first) || s.scalar_type() != at::kFloat || !s.is_contiguous()) return -1;
    if (s.numel() == 1 && count != 1) return H3Q_SCALE_PER_TENSOR;
    return s.numel() == count ? H3Q_SCALE_PER_ROW : -1;
}

// rows_a, rows_b: the logical row counts where they are not those of a and b.
Opt scaled_mm(const Tensor& a, const Tensor& b, const Tensor& a_scale, const Tensor& b_scale, const Opt& bias,
              const Opt& lora_t, const Opt& lora_b, double lora_scale, Opt out, bool a_tiled, bool b_tiled, OptInt rows_a,
              OptInt rows_b, bool f16, int64_t stream) {
    const at::ScalarType type = a.scalar_type();
    if (!a.is_cuda() || (type != at::kChar && type != at::kFloat8_e4m3fn) || !on(b, a)) return std::nullopt;
    if (!rows_2d(a, type) || !rows_2d(b, type) || b.size(1) != a.size(1)) return std::nullopt;
    const int64_t k = a.size(1), m = rows_a.value_or(a.size(0)), n = rows_b.value_or(b.size(0));
    if (m <= 0 || n <= 0) return std::nullopt;
    const auto held = [](const Tensor& t, int64_t rows, bool tiled) {
        return t.size(0) >= (tiled ? (rows + 15) / 16 * 16 : rows) && (!tiled || t.is_contiguous());
    };
    if (!held(a, m, a_tiled) || !held(b, n, b_tiled)) return std::nullopt;
    const int ak = scale_kind(a_scale, a, m), bk = scale_kind(b_scale, a, n);
    if (ak < 0 || bk < 0) return std::nullopt;
    const at::ScalarType out_type = f16 ? at::kHalf : at::kBFloat16;
    if (bias && !(on(*bias, a) && bias->scalar_type() == out_type && bias->numel() == n && bias->is_contiguous()))
        return std::nullopt;
    if (lora_t.has_value() != lora_b.has_value()) return std::nullopt;
    int64_t rank = 0;
    if (lora_t) {
        if (!on(*lora_t, a) || !on(*lora_b, a) || !rows_2d(*lora_t, at::kBFloat16) || !rows_2d(*lora_b, at::kBFloat16))
            return std::nullopt;
        rank = lora_t->size(1);
        if (lora_t->size(0) != m || lora_b->size(0) != n || lora_b->size(1) != rank) return std::nullopt;
    }
    if (out && !(on(*out, a) && rows_2d(*out, out_type) && out->size(0) == m && out->size(1) == n)) return std::nullopt;
    if (!out) out = empty(a, {m, n}, out_type);
    const int fmt = (type == at::kChar ? H3Q_FMT_INT8 : H3Q_FMT_E4M3FN) | (f16 ? H3Q_OUT_F16 : 0);
    if (h3q_scaled_mm(fmt, a.data_ptr(), a.stride(0), a_tiled ? H3Q_LAYOUT_TILED : H3Q_LAYOUT_ROWS, floats(a_scale), ak,
                      b.data_ptr(), b.stride(0), b_tiled ? H3Q_LAYOUT_TILED : H3Q_LAYOUT_ROWS, floats(b_scale), bk,
                      ptr(bias), ptr(lora_t), lora_t ? lora_t->stride(0) : 0, ptr(lora_b),
                      lora_b ? lora_b->stride(0) : 0, rank, (float)lora_scale, out->data_ptr(), out->stride(0), m, n, k,
                      stream_of(stream)))
        return std::nullopt;
    return out;
}

Opt lora_down(const Tensor& x, const Tensor& lora_a, Opt out, int64_t stream) {
    if (!x.is_cuda() || !on(lora_a, x) || !rows_2d(x, at::kBFloat16) || !rows_2d(lora_a, at::kBFloat16)) return std::nullopt;
    const int64_t m = x.size(0), k = x.size(1), rank = lora_a.size(0);
    if (m == 0 || lora_a.size(1) != k) return std::nullopt;
    if (out && !(on(*out, x) && rows_2d(*out, at::kBFloat16) && out->size(0) >= m && out->size(1) >= rank))
        return std::nullopt;
    if (!out) out = empty(x, {m, rank}, at::kBFloat16);
    const int64_t bytes = h3q_lora_down_workspace_bytes(m, k, rank);
    int rc;
    if (bytes == 0) {
        rc = h3q_lora_down(x.data_ptr(), x.stride(0), lora_a.data_ptr(), lora_a.stride(0), out->data_ptr(),
                           out->stride(0), m, k, rank, stream_of(stream));
    } else {  // from torch's allocator: reused in stream order, kept by a graph capture
        const Tensor ws = empty(x, {bytes}, at::kByte);
        rc = h3q_lora_down_ws(x.data_ptr(), x.stride(0), lora_a.data_ptr(), lora_a.stride(0), out->data_ptr(),
                              out->stride(0), m, k, rank, ws.data_ptr(), bytes, stream_of(stream));
    }
    if (rc) return std::nullopt;
    return out;
}

// A [T, cols] bf16 modulation table; its row stride, or -1.
int64_t table_stride(const Tensor& t, const Tensor& first, int64_t cols) {
    if (!on(t, first) || !rows_2d(t, at::kBFloat16) || t.size(1) != cols) return -1;
    const int64_t stride = t.size(0) > 1 ? t.stride(0) : cols;
    return stride % 8 ? -1 : stride;
}

// No fmt: no codes.  Returns (out, codes, scales), None for those not wanted.  gated:
// (branch, gate, hidden).
std::optional<Triple> norm_modulate_quant(const Tensor& value, const Tensor& weight, const Tensor& scale,
                                          const Tensor& shift, const Tensor& indices, double eps, OptInt fmt,
                                          int64_t rounding, bool want_out, const std::optional<Three>& gated,
                                          int64_t stream) {
    if (!value.is_cuda() || !rows_2d(value, at::kBFloat16) || value.size(0) == 0) return std::nullopt;
    const int64_t rows = value.size(0), cols = value.size(1);
    if (!on(weight, value) || weight.scalar_type() != at::kBFloat16 || weight.numel() != cols || !weight.is_contiguous())
        return std::nullopt;
    const int64_t stride = table_stride(scale, value, cols);
    if (stride < 0 || table_stride(shift, value, cols) != stride) return std::nullopt;
    if (!on(indices, value) || indices.scalar_type() != at::kLong || indices.numel() != rows || !indices.is_contiguous())
        return std::nullopt;
    if (fmt ? !valid_fmt(*fmt) : !want_out) return std::nullopt;
    const auto matrix = [&](const Tensor& t) {
        return on(t, value) && rows_2d(t, at::kBFloat16) && t.size(0) == rows && t.size(1) == cols;
    };
    const Tensor none;
    const auto& [branch, gate, hidden] = gated ? *gated : Three(none, none, none);
    if (gated && !(matrix(branch) && matrix(hidden) && table_stride(gate, value, cols) == stride)) return std::nullopt;
    Opt out, codes, scales;
    if (want_out) out = empty(value, {rows, cols}, at::kBFloat16);
    if (fmt) {
        codes = empty(value, {rows, cols}, code_type(*fmt));
        scales = empty(value, {rows, 1}, at::kFloat);
    }
    const auto ld = [&](const Tensor& t) { return rows > 1 ? t.stride(0) : cols; };
    const int f = (int)fmt.value_or(H3Q_FMT_INT8);
    void* const out_p = out ? out->data_ptr() : nullptr;
    void* const codes_p = codes ? codes->data_ptr() : nullptr;
    float* const scales_p = scales ? floats(*scales) : nullptr;
    const int64_t* const idx = static_cast<const int64_t*>(indices.data_ptr());
    const int rc =
        gated ? h3q_residual_gate_rms_norm_modulate_quant(
                    value.data_ptr(), ld(value), branch.data_ptr(), ld(branch), gate.data_ptr(), weight.data_ptr(),
                    scale.data_ptr(), shift.data_ptr(), stride, idx, rows, cols, (float)eps, hidden.data_ptr(),
                    ld(hidden), out_p, cols, f, (int)rounding, codes_p, cols, scales_p, stream_of(stream))
              : h3q_rms_norm_modulate_quant(value.data_ptr(), ld(value), weight.data_ptr(), scale.data_ptr(),
                                            shift.data_ptr(), stride, idx, rows, cols, (float)eps, out_p, cols, f,
                                            (int)rounding, codes_p, cols, scales_p, stream_of(stream));
    if (rc) return std::nullopt;
    return Triple(out, codes, scales);
}

std::optional<Triple> swiglu_quant(const Tensor& x, OptInt fmt, int64_t rounding, bool want_out, int64_t stream) {
    if (!x.is_cuda() || !rows_2d(x, at::kBFloat16) || x.size(0) == 0 || x.size(1) % 2) return std::nullopt;
    if (fmt ? !valid_fmt(*fmt) : !want_out) return std::nullopt;
    const int64_t rows = x.size(0), half = x.size(1) / 2;
    Opt out, codes, scales;
    if (want_out) out = empty(x, {rows, half}, at::kBFloat16);
    if (fmt) {
        codes = empty(x, {rows, half}, code_type(*fmt));
        scales = empty(x, {rows, 1}, at::kFloat);
    }
    if (h3q_swiglu_quant(x.data_ptr(), rows > 1 ? x.stride(0) : 2 * half, rows, half, out ? out->data_ptr() : nullptr,
                         half, (int)fmt.value_or(H3Q_FMT_INT8), (int)rounding, codes ? codes->data_ptr() : nullptr,
                         half, scales ? floats(*scales) : nullptr, stream_of(stream)))
        return std::nullopt;
    return Triple(out, codes, scales);
}

std::optional<Pair> quant_per_head(const Tensor& x, int64_t stream) {
    if (!x.is_cuda() || x.scalar_type() != at::kBFloat16 || x.dim() != 4 || !x.is_contiguous() || x.numel() == 0)
        return std::nullopt;
    const int64_t b = x.size(0), s = x.size(1), h = x.size(2), d = x.size(3);
    const Tensor codes = empty(x, x.sizes(), at::kFloat8_e4m3fn), scales = empty(x, {b, h}, at::kFloat);
    const Tensor ws = empty(x, {h3q_quant_per_head_workspace_floats(b, s, h, d)}, at::kFloat);
    if (h3q_quant_per_head_e4m3(x.data_ptr(), b, s, h, d, floats(ws), codes.data_ptr(), floats(scales),
                                stream_of(stream)))
        return std::nullopt;
    return Pair(codes, scales);
}

std::optional<Pair> quant_tensor(const Tensor& x, const Opt& static_scale, bool eager, int64_t stream) {
    const at::ScalarType type = x.scalar_type();
    if (!x.is_cuda() || x.numel() == 0 || x.dim() < 1 || !x.is_contiguous()) return std::nullopt;
    const int dtype = type == at::kBFloat16 ? H3Q_DTYPE_BF16 : type == at::kHalf ? H3Q_DTYPE_F16
                      : type == at::kFloat ? H3Q_DTYPE_F32 : -1;
    if (dtype < 0) return std::nullopt;
    if (static_scale && !scales_ok(*static_scale, x, 1)) return std::nullopt;
    const int64_t cols = x.size(-1), rows = x.numel() / cols;
    const Tensor codes = empty(x, x.sizes(), at::kFloat8_e4m3fn), scale = empty(x, {}, at::kFloat);
    Opt ws;
    if (!static_scale) ws = empty(x, {h3q_quant_tensor_workspace_floats(rows, cols)}, at::kFloat);
    if (h3q_quant_tensor_e4m3_typed(x.data_ptr(), dtype, eager ? H3Q_QUOTIENT_EAGER : H3Q_QUOTIENT_TRITON, rows, cols,
                                    cols, static_scale ? floats(*static_scale) : nullptr, ws ? floats(*ws) : nullptr,
                                    codes.data_ptr(), cols, floats(scale), stream_of(stream)))
        return std::nullopt;
    return Pair(codes, scale);
}

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
    m.def("quant_rows", torch::wrap_pybind_function_no_gil(&quant_rows));
    m.def("quant_rows_tiled", torch::wrap_pybind_function_no_gil(&quant_rows_tiled));
    m.def("scaled_mm", torch::wrap_pybind_function_no_gil(&scaled_mm));
    m.def("lora_down", torch::wrap_pybind_function_no_gil(&lora_down));
    m.def("norm_modulate_quant", torch::wrap_pybind_function_no_gil(&norm_modulate_quant));
    m.def("swiglu_quant", torch::wrap_pybind_function_no_gil(&swiglu_quant));
    m.def("quant_per_head", torch::wrap_pybind_function_no_gil(&quant_per_head));
    m.def("quant_tensor", torch::wrap_pybind_function_no_gil(&quant_tensor));
}
