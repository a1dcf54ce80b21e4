// The host side of the calls that a decode step or a short prompt makes again and again, in native code.
//
// What bounds them is the host: allocating results, reading shapes and strides and marshalling fifteen arguments in Python took
// 23 us for a 16-row linear layer (a quantization and a product) whose kernels take 7.  Here a call checks the usual case,
// allocates and launches; it returns None for anything unusual -- another device current, a layout that needs a copy, a shape
// or type that is an error -- and the caller goes on with its own code, which copies or says what is wrong.
// (Operand checks here instead of in Python and one layer of calls less: a 160-token prompt 11.1 -> 10.8 us, a 16-row linear layer
// 13.9 -> 13.4, of which 7 are the two launches; two processes of one build differ by as much and more.)
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/utils/pybind.h>
#include <ATen/ATen.h>
#include <hip/hip_runtime_api.h>
#include <optional>
#include "../../include/mpsa.h"

namespace py = pybind11;
using at::Tensor;

namespace {

// Operands come as they are: one that is no tensor is the caller's to refuse.  (No second reference to a tensor is taken either.)
const Tensor* tensor(py::handle x) { return THPVariable_Check(x.ptr()) ? &THPVariable_Unpack(x.ptr()) : nullptr; }

// on the device that is current
bool here(const Tensor& t) {
    int device = -1;
    return t.is_cuda() && hipGetDevice(&device) == hipSuccess && device == t.get_device();
}

bool aligned16(const Tensor& t) { return (reinterpret_cast<uintptr_t>(t.const_data_ptr()) & 15) == 0; }

int dtype_id(at::ScalarType t) {
    switch (t) {
        case at::kBFloat16: return MPSA_BF16;
        case at::kHalf: return MPSA_F16;
        case at::kFloat: return MPSA_F32;
        case at::kFloat8_e5m2: return MPSA_F8E5M2;
        default: return -1;
    }
}

// Allocating can wait for the device (cached memory given back under pressure) and so can launching (a full queue): other
// Python threads run meanwhile, as under torch's own allocations and a ctypes call.  (py::gil_scoped_release looks up pybind11's
// own thread state as well, which nothing here needs.)
struct Unlocked {
    PyThreadState* const state = PyEval_SaveThread();
    ~Unlocked() { PyEval_RestoreThread(state); }
};

mpsa_stream_t stream_of(int64_t s) { return reinterpret_cast<mpsa_stream_t>(s); }

py::object quantize(py::handle arg, double pre, int fmt, int emax, std::optional<int64_t> rows, bool code_per_byte, bool scales_5d, int64_t stream) {
    const Tensor* const given = tensor(arg);
    if (!given) return py::none();
    const Tensor& x = *given;
    if (x.dim() != 4 || !here(x) || (x.scalar_type() != at::kBFloat16 && x.scalar_type() != at::kHalf)) return py::none();
    const auto s = x.strides();
    if (s[3] != 1 || ((s[0] | s[1] | s[2]) & 7) || !aligned16(x)) return py::none();
    const int64_t B = x.size(0), H = x.size(1), L = x.size(2), D = x.size(3), n = rows.value_or(L);
    if (D % 32 || D == 0 || n < L || (scales_5d && (D % 128 || n % 128))) return py::none();
    const bool four = fmt == MPSA_FMT_E2M1;
    Tensor codes, scales;
    int rc;
    {
        Unlocked unlocked;
        const auto bytes = x.options().dtype(at::kByte);
        codes = at::empty({B, H, n, four && !code_per_byte ? D / 2 : D}, bytes);
        scales = scales_5d ? at::empty({B, H, n / 128, D / 128, 32, 4, 4}, bytes) : at::empty({B, H, n, D / 32}, bytes);
        rc = mpsa_quantize_mx_as(x.const_data_ptr(), dtype_id(x.scalar_type()), B, H, L, D, s.data(), nullptr, (float)pre, fmt, emax,
                                 codes.data_ptr<uint8_t>(), scales.data_ptr<uint8_t>(), n, code_per_byte, scales_5d, stream_of(stream));
    }
    if (rc != MPSA_OK) return py::none();
    return py::make_tuple(std::move(codes), std::move(scales));
}

// Two tensors of one type in one launch; two matrices count as [1, 1, rows, K] and their results come back as matrices.
py::object quantize_pair(const Tensor& a, const Tensor& b, double pre_a, double pre_b, int fmt_a, int fmt_b, int emax_a, int emax_b, bool code_per_byte, bool scales_5d, int64_t stream) {
    if (!here(a) || !b.is_cuda() || b.get_device() != a.get_device() || a.scalar_type() != b.scalar_type() || (a.scalar_type() != at::kBFloat16 && a.scalar_type() != at::kHalf)) return py::none();
    mpsa_quantize_job jobs[2];
    const Tensor* const x[2] = {&a, &b};
    for (int i = 0; i < 2; ++i) {
        const Tensor& t = *x[i];
        mpsa_quantize_job& j = jobs[i];
        if (t.dim() != a.dim() || (t.dim() != 4 && t.dim() != 2) || !aligned16(t) || t.numel() == 0) return py::none();
        const bool matrix = t.dim() == 2;
        j.B = matrix ? 1 : t.size(0); j.H = matrix ? 1 : t.size(1); j.N = t.size(-2); j.D = t.size(-1);
        j.x_strides[0] = matrix ? 0 : t.stride(0); j.x_strides[1] = matrix ? 0 : t.stride(1); j.x_strides[2] = t.stride(-2); j.x_strides[3] = t.stride(-1);
        if (j.x_strides[3] != 1 || ((j.x_strides[0] | j.x_strides[1] | j.x_strides[2]) & 7) || j.D % 32 || (scales_5d && (j.D % 128 || j.N % 128))) return py::none();
        j.x = t.const_data_ptr();
        j.out_rows = j.N;
        j.pre_scale = (float)(i ? pre_b : pre_a); j.fmt = i ? fmt_b : fmt_a; j.emax_elem = i ? emax_b : emax_a;
    }
    Tensor codes[2], scales[2];
    int rc;
    {
        Unlocked unlocked;
        const auto bytes = a.options().dtype(at::kByte);
        for (int i = 0; i < 2; ++i) {
            mpsa_quantize_job& j = jobs[i];
            const bool matrix = x[i]->dim() == 2;
            const int64_t width = j.fmt == MPSA_FMT_E2M1 && !code_per_byte ? j.D / 2 : j.D;
            codes[i] = matrix ? at::empty({j.N, width}, bytes) : at::empty({j.B, j.H, j.N, width}, bytes);
            if (scales_5d) scales[i] = matrix ? at::empty({j.N / 128, j.D / 128, 32, 4, 4}, bytes) : at::empty({j.B, j.H, j.N / 128, j.D / 128, 32, 4, 4}, bytes);
            else           scales[i] = matrix ? at::empty({j.N, j.D / 32}, bytes) : at::empty({j.B, j.H, j.N, j.D / 32}, bytes);
            j.codes = codes[i].data_ptr<uint8_t>(); j.scales = scales[i].data_ptr<uint8_t>();
        }
        rc = mpsa_quantize_mx_pair(&jobs[0], &jobs[1], dtype_id(a.scalar_type()), code_per_byte, scales_5d, stream_of(stream));
    }
    if (rc != MPSA_OK) return py::none();
    return py::make_tuple(std::move(codes[0]), std::move(scales[0]), std::move(codes[1]), std::move(scales[1]));
}

// E2M1 codes of two tensors, one per byte, packed along their last dim
py::object pack_pair(const Tensor& a, const Tensor& b, int64_t stream) {
    if (!here(a) || !b.is_cuda() || b.get_device() != a.get_device() || a.scalar_type() != at::kByte || b.scalar_type() != at::kByte || a.dim() == 0 || b.dim() == 0 ||
        !a.is_contiguous() || !b.is_contiguous() || a.numel() == 0 || b.numel() == 0)
        return py::none();
    Tensor packed[2];
    int rc;
    {
        Unlocked unlocked;
        for (int i = 0; i < 2; ++i) {
            auto shape = (i ? b : a).sizes().vec();
            shape.back() = (shape.back() + 1) / 2;
            packed[i] = at::empty(shape, a.options());
        }
        rc = mpsa_e2m1_pack_pair(a.const_data_ptr<uint8_t>(), a.numel() / a.size(-1), a.size(-1), packed[0].data_ptr<uint8_t>(),
                                 b.const_data_ptr<uint8_t>(), b.numel() / b.size(-1), b.size(-1), packed[1].data_ptr<uint8_t>(), stream_of(stream));
    }
    if (rc != MPSA_OK) return py::none();
    return py::make_tuple(std::move(packed[0]), std::move(packed[1]));
}

// codes of `rows` rows of K elements behind the leading dims, bytes, contiguous
bool operand(const Tensor& t, const Tensor& scale, at::IntArrayRef lead, int64_t rows, int64_t K, int fmt, bool packed, int device) {
    const size_t n = lead.size();
    if (!t.is_cuda() || !scale.is_cuda() || t.get_device() != device || scale.get_device() != device) return false;
    if (t.element_size() != 1 || scale.scalar_type() != at::kByte || !t.is_contiguous() || !scale.is_contiguous()) return false;
    if (t.dim() != (int64_t)n + 2 || scale.dim() != (int64_t)n + (packed ? 5 : 2)) return false;
    for (size_t i = 0; i < n; ++i)
        if (t.size(i) != lead[i] || scale.size(i) != lead[i]) return false;
    if (t.size(n) != rows || t.size(n + 1) != (fmt == MPSA_FMT_E2M1 ? K / 2 : K)) return false;
    if (packed) return scale.size(n) == rows / 128 && scale.size(n + 1) == K / 128 && scale.size(n + 2) == 32 && scale.size(n + 3) == 4 && scale.size(n + 4) == 4;
    return scale.size(n) == rows && scale.size(n + 1) == K / 32;
}

py::object matmul(py::handle arg_a, py::handle arg_sa, int fmt_a, py::handle arg_b, py::handle arg_sb, int fmt_b, at::ScalarType dtype,
                  int64_t M, int64_t N, int64_t K, int64_t stream) {
    const Tensor* const given[4] = {tensor(arg_a), tensor(arg_sa), tensor(arg_b), tensor(arg_sb)};
    if (!given[0] || !given[1] || !given[2] || !given[3]) return py::none();
    const Tensor &a = *given[0], &sa = *given[1], &b = *given[2], &sb = *given[3];
    const bool packed = sa.dim() == 5 && sb.dim() == 5;
    if (!here(a) || dtype_id(dtype) < 0 || M <= 0 || N <= 0 || K <= 0 || !operand(a, sa, {}, M, K, fmt_a, packed, a.get_device()) ||
        !operand(b, sb, {}, N, K, fmt_b, packed, a.get_device()))
        return py::none();
    Tensor c;
    int rc;
    {
        Unlocked unlocked;
        c = at::empty({M, N}, a.options().dtype(dtype));
        const auto entry = packed ? mpsa_gemm_mx_packed : mpsa_gemm_mx;
        rc = entry(static_cast<const uint8_t*>(a.const_data_ptr()), sa.const_data_ptr<uint8_t>(), fmt_a, static_cast<const uint8_t*>(b.const_data_ptr()),
                   sb.const_data_ptr<uint8_t>(), fmt_b, M, N, K, c.data_ptr(), dtype_id(dtype), N, stream_of(stream));
    }
    if (rc != MPSA_OK) return py::none();
    return py::cast(std::move(c));
}

py::object matmul_batched(const Tensor& a, const Tensor& sa, int fmt_a, const Tensor& b, const Tensor& sb, int fmt_b, at::ScalarType dtype,
                          int64_t B, int64_t H, int64_t M, int64_t N, int64_t K, int64_t stream) {
    const bool packed = sa.dim() == 7 && sb.dim() == 7;
    if (!here(a) || dtype_id(dtype) < 0 || b.dim() != 4 || B <= 0 || H <= 0 || M <= 0 || N <= 0 || K <= 0) return py::none();
    const int64_t Hb = b.size(1);
    if (Hb <= 0 || H % Hb || !operand(a, sa, {B, H}, M, K, fmt_a, packed, a.get_device()) || !operand(b, sb, {B, Hb}, N, K, fmt_b, packed, a.get_device()))
        return py::none();
    Tensor c;
    int rc;
    {
        Unlocked unlocked;
        c = at::empty({B, H, M, N}, a.options().dtype(dtype));
        const auto entry = packed ? mpsa_gemm_mx_batched_packed : mpsa_gemm_mx_batched;
        rc = entry(static_cast<const uint8_t*>(a.const_data_ptr()), sa.const_data_ptr<uint8_t>(), fmt_a, static_cast<const uint8_t*>(b.const_data_ptr()),
                   sb.const_data_ptr<uint8_t>(), fmt_b, B, H, Hb, M, N, K, c.data_ptr(), dtype_id(dtype), N, stream_of(stream));
    }
    if (rc != MPSA_OK) return py::none();
    return py::cast(std::move(c));
}

// mpsa_attn_call_on with the output and the workspace allocated here; desc is the address of an mpsa_attn_desc
py::object attention(int kernel, int64_t desc, int64_t workspace, const std::vector<int64_t>& shape, at::ScalarType dtype, const Tensor& q, const Tensor& k,
                     const Tensor& v, int64_t stream) {
    if (!here(q)) return py::none();
    Tensor out;
    int rc;
    {
        Unlocked unlocked;
        out = at::empty(shape, q.options().dtype(dtype));
        Tensor work = at::empty({workspace}, q.options().dtype(at::kByte));
        rc = mpsa_attn_call_on(kernel, reinterpret_cast<const mpsa_attn_desc*>(desc), q.const_data_ptr(), k.const_data_ptr(), v.const_data_ptr(),
                               out.data_ptr(), work.data_ptr(), nullptr, stream_of(stream));
    }
    if (rc != MPSA_OK) return py::none();
    return py::cast(std::move(out));
}

}  // namespace

PYBIND11_MODULE(mpsa_host, m) {
    m.def("quantize", &quantize);
    m.def("quantize_pair", &quantize_pair);
    m.def("pack_pair", &pack_pair);
    m.def("matmul", &matmul);
    m.def("matmul_batched", &matmul_batched);
    m.def("attention", &attention);
}
