// The torch operators of the package (torch.ops.vq_gemm_amd.*) and the direct calls behind its layers.  Host-only C++:
// tensors are checked, the result is allocated with torch's allocator, raw pointers and the current stream go to the
// C ABI of libvqgemm.so.
//
// A decode-size product is a kernel of three to twelve microseconds, so what surrounds the launch is what a layer call
// costs: as a Python custom operator over ctypes it took 26 us per call on 4096 x 4096 with one row of X (the kernel:
// 3.7).  The operators are therefore registered here, and the layers (vq_gemm_amd/nn.py) call `linear` and `gated` below
// without going through the dispatcher at all; those two step aside (return None) whenever something else is to see
// the call - a fake or wrapped tensor, a tensor subclass, a dispatch or function mode, a tracer - and the layer then calls
// the registered operator.  The direct calls work without the GIL, as the operators do: a launch that waits on a full
// queue must not hold up the other threads.
#include <torch/extension.h>
#include <torch/csrc/PyInterpreter.h>
#include <torch/csrc/autograd/python_variable.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/hip/EmptyTensor.h>
#include <ATen/record_function.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/hip/HIPStream.h>

#include "../../include/vq_gemm.h"
#include "seeded_pick.h"

namespace {

using at::Tensor;
using OptTensor = c10::optional<Tensor>;

void check_rc(int rc, const char *what)
{
    TORCH_CHECK(rc == 0, what, " failed with code ", rc, ": ", vqgemm_error_string(rc));
}

bool aligned16(const Tensor &t) { return (reinterpret_cast<uintptr_t>(t.data_ptr()) & 15) == 0; }

// An activation as the kernels want it: contiguous and 16-byte aligned (a view into a larger buffer may start anywhere,
// and a copy costs far less than the scalar kernel that takes unaligned operands).
void *dense_of(const Tensor &t, Tensor &hold)
{
    if (t.is_contiguous() && aligned16(t)) return t.data_ptr();
    hold = t.is_contiguous() ? t.clone() : t.contiguous();
    if (!aligned16(hold)) hold = hold.clone();
    return hold.data_ptr();
}

// Sizes of a product, after every check that raw pointers need: types, devices, element counts.
struct Dims {
    int64_t M, K, N;
    int vec, entries, books, bits;
};

Dims check_linear(const char *name, const Tensor &x, const Tensor &codes, const Tensor &codebook, const OptTensor &bias,
                  int64_t k_repeat)
{
    TORCH_CHECK_VALUE(codes.dim() == 2 && (codebook.dim() == 2 || codebook.dim() == 3) && x.dim() >= 1, name,
                      ": x [..., K], codes [N, K/vec], codebook [E, vec] or [G, E, vec]");
    const bool u8 = codes.scalar_type() == at::kByte;
    TORCH_CHECK_VALUE(u8 || codes.scalar_type() == at::kUInt16, name, ": codes must be uint8 or uint16, got ", codes.scalar_type());
    TORCH_CHECK_VALUE(x.scalar_type() == at::kHalf && codebook.scalar_type() == at::kHalf, name, ": x and codebook must be float16");
    Dims d;
    d.vec = (int)codebook.size(-1);
    d.entries = (int)codebook.size(-2);
    d.books = codebook.dim() == 3 ? (int)codebook.size(0) : 1;
    d.bits = u8 ? 8 : 16;
    d.N = codes.size(0);
    d.K = codes.size(1) * d.vec;
    TORCH_CHECK_VALUE(x.size(-1) * k_repeat == d.K, name, ": x has ", x.size(-1), " features, codes x vec give ", d.K, " / ", k_repeat);
    TORCH_CHECK_VALUE(d.books > 0 && d.N % d.books == 0, name, ": rows of codes must be a multiple of the number of codebooks");
    d.M = 1;
    for (int64_t i = 0; i + 1 < x.dim(); i++) d.M *= x.size(i);
    const c10::Device dev = x.device();
    TORCH_CHECK_VALUE(dev.is_cuda() && codes.device() == dev && codebook.device() == dev, name,
                      ": all tensors must be on one device, in GPU memory");
    if (bias.has_value() && bias->defined())
        TORCH_CHECK_VALUE(bias->scalar_type() == at::kHalf && bias->dim() == 1 && bias->size(0) == d.N && bias->device() == dev, name,
                          ": bias must be a float16 tensor on x's device with one entry per output column");
    return d;
}

Tensor new_result(const Tensor &x, int64_t columns)
{
    c10::SmallVector<int64_t, 6> shape(x.sizes().begin(), x.sizes().end());
    shape.back() = columns;
    return at::detail::empty_cuda(shape, at::kHalf, x.device(), c10::nullopt);
}

void *stream_of(const Tensor &t) { return c10::hip::getCurrentHIPStream(t.get_device()).stream(); }

// A tensor's own data where the kernels can read it as it lies, else the data of a copy kept in `hold`.
void *data_of(const Tensor &t, Tensor &hold)
{
    if (t.is_contiguous()) return t.data_ptr();
    hold = t.contiguous();
    return hold.data_ptr();
}

// x @ W.T (+ bias), W in k_repeat stages side by side along K that all multiply the same x
Tensor linear_impl(const Tensor &x, const Tensor &codes, const Tensor &codebook, const OptTensor &bias, int64_t k_repeat,
                   int variant = VQGEMM_VARIANT_AUTO)
{
    const Dims d = check_linear("vq_linear", x, codes, codebook, bias, k_repeat);
    const c10::OptionalDeviceGuard guard(x.device());
    Tensor hold_x, hold_codes, hold_cb, hold_bias;
    const void *xp = dense_of(x, hold_x), *codes_p = data_of(codes, hold_codes), *cb_p = data_of(codebook, hold_cb);
    const void *bias_p = bias.has_value() && bias->defined() ? data_of(*bias, hold_bias) : nullptr;
    Tensor y = new_result(x, d.N);
    void *s = stream_of(x);
    // scratch for the shapes where the automatic choice may split K (never with a slab of 16 rows or fewer) or wants x
    // repeated; the caching allocator hands out stream-ordered blocks
    int64_t need = 0;
    if (k_repeat > 1) need = vqgemm_stages_workspace_bytes_b(d.M, d.K, d.N, d.vec, d.entries, d.books, d.bits, (int)k_repeat);
    else if (variant == VQGEMM_VARIANT_AUTO && d.M > 16)
        need = vqgemm_workspace_bytes_b(d.M, d.K, d.N, d.vec, d.entries, d.books, d.bits, variant);
    Tensor ws;
    if (need > 0) ws = at::detail::empty_cuda({need}, at::kByte, x.device(), c10::nullopt);
    void *ws_p = need > 0 ? ws.data_ptr() : nullptr;
    const int64_t ws_bytes = need > 0 ? need : 0;
    int rc;
    if (k_repeat > 1)
        rc = vqgemm_e2e_gemm_b_stages(xp, codes_p, cb_p, bias_p, y.data_ptr(), d.M, d.K, d.N, d.vec, d.entries, d.books, d.bits,
                                      (int)k_repeat, ws_p, ws_bytes, s);
    else if (need > 0)
        rc = vqgemm_e2e_gemm_b_ws(xp, codes_p, cb_p, bias_p, y.data_ptr(), d.M, d.K, d.N, d.vec, d.entries, d.books, d.bits, variant,
                                  ws_p, ws_bytes, s);
    else
        rc = vqgemm_e2e_gemm_b_bias(xp, codes_p, cb_p, bias_p, y.data_ptr(), d.M, d.K, d.N, d.vec, d.entries, d.books, d.bits, variant,
                                    nullptr, s);
    check_rc(rc, "vq_linear");
    return y;
}

Tensor gated_impl(const Tensor &x, const Tensor &codes, const Tensor &codebook, const OptTensor &bias)
{
    const Dims d = check_linear("vq_gated_linear", x, codes, codebook, bias, 1);
    TORCH_CHECK_VALUE(d.N % 32 == 0, "vq_gated_linear: the interleaved gate/up rows come in whole groups of 32");
    const c10::OptionalDeviceGuard guard(x.device());
    Tensor hold_x, hold_codes, hold_cb, hold_bias;
    const void *xp = dense_of(x, hold_x), *codes_p = data_of(codes, hold_codes), *cb_p = data_of(codebook, hold_cb);
    const void *bias_p = bias.has_value() && bias->defined() ? data_of(*bias, hold_bias) : nullptr;
    Tensor y = new_result(x, d.N / 2);
    check_rc(vqgemm_e2e_gemm_b_gated(xp, codes_p, cb_p, bias_p, y.data_ptr(), d.M, d.K, d.N, d.vec, d.entries, d.books, d.bits,
                                     VQGEMM_VARIANT_AUTO, nullptr, stream_of(x)),
             "vq_gated_linear");
    return y;
}

Tensor silu_mul_impl(const Tensor &gate_up)
{
    TORCH_CHECK_VALUE(gate_up.scalar_type() == at::kHalf && gate_up.dim() >= 1 && gate_up.size(-1) % 2 == 0,
                      "silu_mul: expected a float16 tensor with an even last dimension");
    const c10::OptionalDeviceGuard guard(gate_up.device());
    const Tensor a = gate_up.contiguous();
    const int64_t n2 = a.size(-1), m = n2 > 0 ? a.numel() / n2 : 0;
    Tensor y = new_result(a, n2 / 2);
    check_rc(vqgemm_silu_mul(a.data_ptr(), y.data_ptr(), m, n2 / 2, stream_of(a)), "silu_mul");
    return y;
}

// ---- the registered operators ---------------------------------------------------------------------------------

Tensor vq_linear(const Tensor &x, const Tensor &codes, const Tensor &codebook, const OptTensor &bias)
{
    return linear_impl(x, codes, codebook, bias, 1);
}

Tensor vq_linear_packed(const Tensor &x, const Tensor &codes, const Tensor &codebook, const OptTensor &bias)
{
    return linear_impl(x, codes, codebook, bias, 1, VQGEMM_VARIANT_DECODE_PACKED);
}

// No gradient flows: an input that wants one gets a result whose backward raises.
struct NoGradient : torch::autograd::Function<NoGradient> {
    static Tensor forward(torch::autograd::AutogradContext *, const Tensor &y_of, const Tensor &y)
    {
        (void)y_of;
        return y.view_as(y);
    }
    static torch::autograd::variable_list backward(torch::autograd::AutogradContext *, torch::autograd::variable_list)
    {
        TORCH_CHECK(false, "the vector-quantised products are for inference: no backward formula is registered");
    }
};

Tensor no_gradient(Tensor y, std::initializer_list<const Tensor *> inputs)
{
    if (at::GradMode::is_enabled())
        for (const Tensor *t : inputs)
            if (t->defined() && t->requires_grad()) return NoGradient::apply(*t, y);
    return y;
}

// Whether nothing but this library is to see a call on `x`: an ordinary tensor in GPU memory, no dispatch mode, no
// functional transform, no tracer.
bool plain_tensor(const Tensor &x)
{
    if (!x.defined() || !x.is_cuda()) return false;
    constexpr c10::DispatchKeySet wrappers({c10::DispatchKey::Python, c10::DispatchKey::PythonTLSSnapshot, c10::DispatchKey::Functionalize,
                                            c10::DispatchKey::FuncTorchBatched, c10::DispatchKey::FuncTorchGradWrapper,
                                            c10::DispatchKey::BatchedNestedTensor, c10::DispatchKey::NestedTensor});
    return !x.key_set().has_any(wrappers);
}

bool plain_thread() { return (c10::impl::tls_local_dispatch_key_set().included_ - c10::default_included_set).empty(); }

bool plain_call(const Tensor &x) { return plain_tensor(x) && plain_thread(); }

// The autograd kernels call the device implementation directly (one dispatch per call instead of two), unless the tensors
// only stand for data: then the call goes on to whoever wrapped them.
typedef Tensor (*LinearFn)(const Tensor &, const Tensor &, const Tensor &, const OptTensor &);

template <LinearFn Impl, const char *Name>
Tensor with_autograd(const Tensor &x, const Tensor &codes, const Tensor &codebook, const OptTensor &bias)
{
    const bool plain = plain_call(x);
    Tensor y;
    {
        at::AutoDispatchBelowADInplaceOrView below;
        if (plain) {
            y = Impl(x, codes, codebook, bias);
        } else {
            static const auto op = c10::Dispatcher::singleton().findSchemaOrThrow(Name, "").typed<Tensor(const Tensor &, const Tensor &, const Tensor &, const OptTensor &)>();
            y = op.call(x, codes, codebook, bias);
        }
    }
    const Tensor b = bias.has_value() ? *bias : Tensor();
    return no_gradient(y, {&x, &codebook, &b});
}

Tensor silu_mul_autograd(const Tensor &gate_up)
{
    const bool plain = plain_call(gate_up);
    Tensor y;
    {
        at::AutoDispatchBelowADInplaceOrView below;
        if (plain) {
            y = silu_mul_impl(gate_up);
        } else {
            static const auto op = c10::Dispatcher::singleton().findSchemaOrThrow("vq_gemm_amd::silu_mul", "").typed<Tensor(const Tensor &)>();
            y = op.call(gate_up);
        }
    }
    return no_gradient(y, {&gate_up});
}

constexpr char kLinear[] = "vq_gemm_amd::vq_linear", kLinearPacked[] = "vq_gemm_amd::vq_linear_packed", kGated[] = "vq_gemm_amd::vq_gated_linear";

// ---- the layers' direct calls ---------------------------------------------------------------------------------

// Whether a function mode is to see the call.  A default device (torch.set_default_device, `with torch.device(...)`) is such
// a mode too, but looks at factory functions only.
PyObject *default_device_mode = nullptr, *no_torch_function = nullptr;  // its class, and what a class without an override has; set on loading
bool function_mode_watches()
{
    if (!at::impl::torch_function_mode_enabled()) return false;
    for (int64_t i = 0; i < at::impl::PythonTorchFunctionTLS::stack_len(); i++)
        if ((PyObject *)Py_TYPE(at::impl::PythonTorchFunctionTLS::get_stack_at(i)->ptr(getPyInterpreter())) != default_device_mode) return true;
    return false;
}

// Whether the tensor's class overrides __torch_function__.
bool subclass_watches(PyObject *tensor)
{
    if (THPVariable_CheckTypeExact(Py_TYPE(tensor))) return false;
    if (at::impl::PythonTorchFunctionTLS::get_disabled_state() != at::impl::TorchFunctionDisabledState::ENABLED) return false;
    return py::object(py::handle(tensor).attr("__torch_function__")).ptr() != no_torch_function;
}

// The tensor behind an argument, without a reference of its own: the caller's arguments live as long as the call.
const Tensor &tensor_of(py::handle h)
{
    if (!THPVariable_Check(h.ptr())) throw py::type_error("expected a tensor");
    return THPVariable_Unpack(h.ptr());
}

// `plain_call` for a call from Python on these operands (None is none).
bool plain_python_call(std::initializer_list<py::handle> operands)
{
    if (function_mode_watches() || !plain_thread()) return false;
    for (const py::handle h : operands)
        if (!h.is_none() && (!plain_tensor(tensor_of(h)) || subclass_watches(h.ptr()))) return false;
    return true;
}

OptTensor optional_of(py::handle h) { return h.is_none() ? OptTensor() : OptTensor(tensor_of(h)); }

// packed: `codes` are in the packed layout (a single stage)
py::object linear(py::handle x, py::handle codes, py::handle codebook, py::handle bias, int64_t k_repeat, bool packed)
{
    if (!plain_python_call({x, codes, codebook, bias})) return py::none();
    TORCH_CHECK_VALUE(!packed || k_repeat == 1, "linear: additive stages have no packed layout");
    const Tensor &x_t = tensor_of(x), &codes_t = tensor_of(codes), &codebook_t = tensor_of(codebook);
    const OptTensor bias_t = optional_of(bias);
    Tensor y;
    {
        const py::gil_scoped_release no_gil;
        RECORD_FUNCTION("vq_gemm_amd::vq_linear", c10::ArrayRef<const c10::IValue>());
        y = linear_impl(x_t, codes_t, codebook_t, bias_t, k_repeat, packed ? VQGEMM_VARIANT_DECODE_PACKED : VQGEMM_VARIANT_AUTO);
    }
    return py::cast(y);
}

// Whether a layer that holds both layouts of its codes hands the packed one over for x (what is wrong with x the call itself says;
// the kernel of the packed layout takes no operands that begin anywhere).
bool takes_packed(py::handle x_h, py::handle codes_h, py::handle codebook_h, py::handle bias_h)
{
    if (!plain_python_call({x_h, codes_h, codebook_h, bias_h})) return false;
    const Tensor &x = tensor_of(x_h), &codes = tensor_of(codes_h), &codebook = tensor_of(codebook_h);
    const OptTensor bias = optional_of(bias_h);
    if (x.dim() < 1 || codes.dim() != 2 || (codebook.dim() != 2 && codebook.dim() != 3) || !aligned16(codebook)) return false;
    if (bias.has_value() && bias->defined() && (reinterpret_cast<uintptr_t>(bias->data_ptr()) & 7) != 0) return false;
    const int64_t vec = codebook.size(-1), K = codes.size(1) * vec;
    if (K == 0 || x.size(-1) != K) return false;
    const c10::OptionalDeviceGuard guard(x.device());
    return vqgemm_packed_preferred_b(x.numel() / K, K, codes.size(0), (int)vec, (int)codebook.size(-2),
                                     codebook.dim() == 3 ? (int)codebook.size(0) : 1, codes.scalar_type() == at::kByte ? 8 : 16) == 1;
}

py::object gated(py::handle x, py::handle codes, py::handle codebook, py::handle bias)
{
    if (!plain_python_call({x, codes, codebook, bias})) return py::none();
    const Tensor &x_t = tensor_of(x), &codes_t = tensor_of(codes), &codebook_t = tensor_of(codebook);
    const OptTensor bias_t = optional_of(bias);
    Tensor y;
    {
        const py::gil_scoped_release no_gil;
        RECORD_FUNCTION("vq_gemm_amd::vq_gated_linear", c10::ArrayRef<const c10::IValue>());
        y = gated_impl(x_t, codes_t, codebook_t, bias_t);
    }
    return py::cast(y);
}

// ---- the codec ------------------------------------------------------------------------------------------------

// What cabi.encode_b and cabi.dequant_b do on well-formed operands of the current device, without their checks one by one in
// Python (11 of the 12 us of a call on a small matrix); None sends the caller down that path, which says what is wrong.
bool codec_operands(py::handle m_h, py::handle codebook_h, int64_t per_column)
{
    if (!plain_python_call({m_h, codebook_h})) return false;
    const Tensor &m = tensor_of(m_h), &codebook = tensor_of(codebook_h);
    return m.dim() == 2 && m.is_contiguous() && codebook.is_cuda() && codebook.device() == m.device() && codebook.is_contiguous() &&
           codebook.scalar_type() == at::kHalf && (codebook.dim() == 2 || codebook.dim() == 3) && codebook.size(-1) > 0 &&
           m.device().index() == c10::hip::current_device() && (m.size(1) * per_column) % codebook.size(-1) == 0 &&
           (codebook.dim() == 2 || (codebook.size(0) > 0 && m.size(0) % codebook.size(0) == 0));
}

py::object encode(py::handle w_h, py::handle codebook_h)
{
    const Tensor &w = tensor_of(w_h), &codebook = tensor_of(codebook_h);
    if (!codec_operands(w_h, codebook_h, 1) || w.scalar_type() != at::kHalf) return py::none();
    const int64_t N = w.size(0), K = w.size(1), vec = codebook.size(-1), entries = codebook.size(-2);
    const int bits = entries <= 256 ? 8 : 16;
    Tensor codes;
    int rc;
    {
        const py::gil_scoped_release no_gil;
        codes = at::detail::empty_cuda({N, K / vec}, bits == 8 ? at::kByte : at::kUInt16, w.device(), c10::nullopt);
        rc = vqgemm_encode_b(w.data_ptr(), codebook.data_ptr(), codes.data_ptr(), N, K, (int)vec, (int)entries,
                             codebook.dim() == 3 ? (int)codebook.size(0) : 1, bits, stream_of(w));
    }
    if (rc != 0) return py::none();
    return py::cast(codes);
}

py::object dequant(py::handle codes_h, py::handle codebook_h)
{
    const Tensor &codes = tensor_of(codes_h), &codebook = tensor_of(codebook_h);
    const bool u8 = codes.scalar_type() == at::kByte;
    if ((!u8 && codes.scalar_type() != at::kUInt16) || !codec_operands(codes_h, codebook_h, codebook.dim() > 0 ? codebook.size(-1) : 1)) return py::none();
    const int64_t N = codes.size(0), vec = codebook.size(-1), K = codes.size(1) * vec;
    Tensor w;
    int rc;
    {
        const py::gil_scoped_release no_gil;
        w = at::detail::empty_cuda({N, K}, at::kHalf, codes.device(), c10::nullopt);
        rc = vqgemm_dequant_b(codes.data_ptr(), codebook.data_ptr(), w.data_ptr(), N, K, (int)vec, (int)codebook.size(-2),
                              codebook.dim() == 3 ? (int)codebook.size(0) : 1, u8 ? 8 : 16, stream_of(codes));
    }
    if (rc != 0) return py::none();
    return py::cast(w);
}

// ---- the quantiser --------------------------------------------------------------------------------------------

// int32 [books, count] on the host: row g is the start of the g-th permutation of 0 .. n-1 that a generator seeded with `seed` makes
Tensor first_of_permutations(int64_t n, int64_t count, int64_t books, int64_t seed)
{
    TORCH_CHECK_VALUE(count >= 0 && count <= n && n <= (int64_t(1) << 24) && books >= 1, "first_of_permutations: 0 <= count <= n <= 2^24");
    Tensor pick = at::empty({books, count}, at::kInt);
    vq::Mt19937 gen((uint32_t)((uint64_t)seed & 0xffffffffu));
    for (int64_t g = 0; g < books; g++) {
        vq::first_of_permutation(gen, n, count, g + 1 < books, pick.data_ptr<int32_t>() + g * count);
    }
    return pick;
}

// (codes, codebook, squared errors [iters + 1] on the device) of Lloyd iterations from the vectors `pick`, or None where the library
// has no kernel for the codebook's size.  The caller has checked w: fp16 [N, K] on the GPU, contiguous.
py::object kmeans(py::handle w_h, const Tensor &pick, int64_t vec, int64_t entries, int64_t books, int64_t code_bits, int64_t iters)
{
    const Tensor &w = tensor_of(w_h);
    const int64_t N = w.size(0), K = w.size(1);
    TORCH_CHECK_VALUE(w.is_cuda() && w.scalar_type() == at::kHalf && w.is_contiguous() && pick.scalar_type() == at::kInt &&
                          pick.numel() == books * entries && pick.is_contiguous() && vec > 0 && K % vec == 0 && books > 0 && N % books == 0,
                      "kmeans: w fp16 [N, K] on the GPU, pick int32 [books, entries]");
    if (!plain_python_call({w_h})) return py::none();
    const int64_t need = vqgemm_kmeans_workspace_bytes_b(N, K, (int)vec, (int)entries, (int)books, (int)code_bits);
    if (need < 0 || (reinterpret_cast<uintptr_t>(w.data_ptr()) & 7) != 0) return py::none();
    const c10::OptionalDeviceGuard guard(w.device());
    auto on_device = [&](at::IntArrayRef shape, at::ScalarType t) { return at::detail::empty_cuda(shape, t, w.device(), c10::nullopt); };
    Tensor codes, codebook, errors;
    {
        const py::gil_scoped_release no_gil;
        const Tensor pick_d = pick.to(w.device());
        codes = on_device({N, K / vec}, code_bits == 8 ? at::kByte : at::kUInt16);
        codebook = on_device({books, entries, vec}, at::kHalf);
        errors = on_device({iters + 1}, at::kDouble);
        const Tensor ws = on_device({need}, at::kByte);
        check_rc(vqgemm_kmeans_b(w.data_ptr(), pick_d.data_ptr<int32_t>(), codes.data_ptr(), codebook.data_ptr(), errors.data_ptr<double>(), N, K,
                                 (int)vec, (int)entries, (int)books, (int)code_bits, (int)iters, ws.data_ptr(), need, stream_of(w)),
                 "kmeans");
    }
    return py::make_tuple(codes, codebook, errors);
}

}  // namespace

TORCH_LIBRARY(vq_gemm_amd, m)
{
    m.def("vq_linear(Tensor x, Tensor codes, Tensor codebook, Tensor? bias=None) -> Tensor");
    m.def("vq_linear_packed(Tensor x, Tensor codes_packed, Tensor codebook, Tensor? bias=None) -> Tensor");
    m.def("vq_gated_linear(Tensor x, Tensor codes, Tensor codebook, Tensor? bias=None) -> Tensor");
    m.def("silu_mul(Tensor gate_up) -> Tensor");
}

TORCH_LIBRARY_IMPL(vq_gemm_amd, CUDA, m)
{
    m.impl("vq_linear", &vq_linear);
    m.impl("vq_linear_packed", &vq_linear_packed);
    m.impl("vq_gated_linear", &gated_impl);
    m.impl("silu_mul", &silu_mul_impl);
}

TORCH_LIBRARY_IMPL(vq_gemm_amd, AutogradCUDA, m)
{
    m.impl("vq_linear", &with_autograd<vq_linear, kLinear>);
    m.impl("vq_linear_packed", &with_autograd<vq_linear_packed, kLinearPacked>);
    m.impl("vq_gated_linear", &with_autograd<gated_impl, kGated>);
    m.impl("silu_mul", &silu_mul_autograd);
}

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m)
{
    no_torch_function = py::object(py::module_::import("torch._C").attr("_disabled_torch_function_impl")).release().ptr();
    default_device_mode = py::object(py::module_::import("torch.utils._device").attr("DeviceContext")).release().ptr();
    m.def("linear", &linear, "x @ W.T (+ bias) on plain GPU tensors; None where the registered operator is to be called instead");
    m.def("takes_packed", &takes_packed, "whether `linear` does best with the packed layout of the codes");
    m.def("first_of_permutations", &first_of_permutations, py::call_guard<py::gil_scoped_release>(), "the first elements of seeded random permutations");
    m.def("kmeans", &kmeans, "Lloyd iterations on the device; None where the codebook is too large for them");
    m.def("encode", &encode, "nearest-codeword codes; None where cabi.encode_b is to check the operands one by one");
    m.def("dequant", &dequant, "codes and codebook to fp16 likewise");
    m.def("gated", &gated, "silu(gate) * up likewise");
}
