// CPython module behind vpux_plugin_amd.runtime: the operator functions' way from torch tensors to the C ABI.
//
// What bounds a call on a small tensor is the host: the kernel of a FakeQuantize over [1,64,56,56] takes 3 us, a bare
// hipLaunchKernel 2.4 us.  Describing the operands through ctypes and numpy objects took 12 ... 23 us more per call
// (torch.cuda.current_stream() alone 2.9 us); here the tensors' sizes, strides and addresses are read from their C++
// objects, the params blob or the task is laid out on the stack, and the same entry points of
// include/vpx_runtime.h that any other host would call are called.  Nothing is remembered between calls.
#include <torch/csrc/autograd/python_variable.h>
#include <c10/hip/HIPStream.h>

#include <cstring>
#include <vector>

#include "vpx_compiler_utils.h"
#include "vpx_runtime.h"

namespace {

PyObject* g_orders = nullptr;  // name of a layout -> its code (runtime.ORDER)
PyObject* g_ppe = nullptr;     // the type of a task's ppe (runtime.PpeInt)

// What a Python error leaves behind: the exception is set, the call returns null.
struct Raised {};

[[noreturn]] void raise(PyObject* type, const char* text) {
    PyErr_SetString(type, text);
    throw Raised{};
}

const at::Tensor& tensor(PyObject* o) {
    if (Py_TYPE(o) != reinterpret_cast<PyTypeObject*>(THPVariableClass) && !THPVariable_Check(o)) {
        PyErr_Format(PyExc_TypeError, "expected a torch tensor, got %s", Py_TYPE(o)->tp_name);
        throw Raised{};
    }
    return THPVariable_Unpack(o);
}

uint32_t type_code(const at::Tensor& t) {
    switch (t.scalar_type()) {
    case at::kHalf: return VPX_NN_FP16;
    case at::kFloat: return VPX_NN_FP32;
    case at::kByte: return VPX_NN_U8;
    case at::kChar: return VPX_NN_I8;
    case at::kInt: return VPX_NN_I32;
    default: raise(PyExc_KeyError, c10::toString(t.scalar_type()));
    }
}

int64_t integer(PyObject* o) {
    PyObject* i = PyNumber_Index(o);
    if (!i) throw Raised{};
    const int64_t v = PyLong_AsLongLong(i);
    Py_DECREF(i);
    if (v == -1 && PyErr_Occurred()) throw Raised{};
    return v;
}

int32_t integer32(PyObject* o) {
    return (int32_t)integer(o);
}

// An attribute: a whole number, whatever type holds it.
int64_t whole(PyObject* o) {
    PyObject* i = PyIndex_Check(o) ? PyNumber_Index(o) : PyNumber_Long(o);
    if (!i) throw Raised{};
    const int64_t v = PyLong_AsLongLong(i);
    Py_DECREF(i);
    if (v == -1 && PyErr_Occurred()) throw Raised{};
    return v;
}

// A true boolean attribute serialises as int64 -1 (sign-extended i1).
int64_t flag(PyObject* o) {
    const int v = PyObject_IsTrue(o);
    if (v < 0) throw Raised{};
    return v ? -1 : 0;
}

float real(PyObject* o) {
    const double v = PyFloat_AsDouble(o);
    if (v == -1.0 && PyErr_Occurred()) throw Raised{};
    return (float)v;  // beyond float32: infinities
}

void* stream_handle(PyObject* stream) {
    if (stream == Py_None) return c10::hip::getCurrentHIPStream().stream();
    PyObject* h = PyObject_GetAttrString(stream, "cuda_stream");
    if (!h) throw Raised{};
    void* p = PyLong_AsVoidPtr(h);
    Py_DECREF(h);
    if (!p && PyErr_Occurred()) throw Raised{};
    return p;
}

// Layout code of a tensor: None = the logical order is the memory order (NCHW for four dimensions, one hex digit less for
// each one missing), else a code or the name of one.
uint64_t order_code(PyObject* order, int64_t rank) {
    if (order == Py_None) {
        if (rank < 1) raise(PyExc_ValueError, "a tensor without dimensions has no layout");
        uint64_t code = 0;
        for (int64_t i = rank; i >= 1; i--) code = code << 4 | (uint64_t)i;
        return code;
    }
    if (PyUnicode_Check(order)) {
        if (!g_orders) raise(PyExc_RuntimeError, "set_orders was not called");
        PyObject* code = PyDict_GetItemWithError(g_orders, order);
        if (!code) {
            if (!PyErr_Occurred()) PyErr_SetObject(PyExc_KeyError, order);
            throw Raised{};
        }
        order = code;
    }
    const uint64_t code = PyLong_AsUnsignedLongLong(order);
    if (code == (uint64_t)-1 && PyErr_Occurred()) throw Raised{};
    return code;
}

constexpr int kMostTensors = 16, kMostAxes = 32;

// The dims, then the strides in bits, of some operands of a blob, innermost first.
uint8_t* put_shapes(uint8_t* p, const at::Tensor* const* t, int n) {
    for (int i = 0; i < n; i++) {
        const auto sizes = t[i]->sizes();
        for (size_t d = sizes.size(); d-- > 0; p += 4) {
            const int32_t v = (int32_t)sizes[d];
            std::memcpy(p, &v, 4);
        }
    }
    for (int i = 0; i < n; i++) {
        const auto strides = t[i]->strides();
        const int64_t bits = (int64_t)t[i]->element_size() * 8;
        for (size_t d = strides.size(); d-- > 0; p += 8) {
            const int64_t v = strides[d] * bits;
            std::memcpy(p, &v, 8);
        }
    }
    return p;
}

// One launch: the params blob is MemRefData records, attributes, then input dims | input strides | output dims | output
// strides (the layout vpx_create_kernel_params writes).  order: one layout for all tensors, or a tuple with one each.
PyObject* launch_tensors(const char* entry, int n_in, int n, PyObject* const* objects, PyObject* order, const void* attrs, size_t attrs_size,
                         PyObject* stream, bool noalloc) {
    if (n > kMostTensors || n_in < 0 || n_in > n) raise(PyExc_ValueError, "a number of operands that no launch has");
    const bool each = PyTuple_Check(order);
    if (each && PyTuple_GET_SIZE(order) != n) raise(PyExc_ValueError, "one layout per operand, or one for all");
    const at::Tensor* t[kMostTensors];
    vpx_memref_data_t records[kMostTensors];
    vpx_memref_addr_t addrs[kMostTensors];
    size_t levels = 0;
    for (int i = 0; i < n; i++) {
        t[i] = &tensor(objects[i]);
        const int64_t rank = t[i]->dim();
        vpx_memref_data_t& m = records[i];
        m = vpx_memref_data_t{};
        m.isStatic = 1;
        m.numDims = (uint32_t)rank;
        m.dataType = type_code(*t[i]);
        m.dimsOrder = order_code(each ? PyTuple_GET_ITEM(order, i) : order, rank);
        m.location = VPX_LOC_DDR;
        addrs[i] = vpx_memref_addr_t{t[i]->data_ptr(), nullptr, nullptr};
        levels += (size_t)rank;
    }
    uint8_t here[2048];  // (six operands of eight dimensions take 800 bytes)
    std::vector<uint8_t> more;
    const size_t size = (size_t)n * sizeof(vpx_memref_data_t) + attrs_size + levels * (sizeof(int32_t) + sizeof(int64_t));
    if (size > sizeof(here)) more.resize(size);
    uint8_t* const blob = more.empty() ? here : more.data();
    uint8_t* p = blob;
    std::memcpy(p, records, (size_t)n * sizeof(vpx_memref_data_t));
    p += (size_t)n * sizeof(vpx_memref_data_t);
    if (attrs_size) std::memcpy(p, attrs, attrs_size);
    p = put_shapes(p + attrs_size, t, n_in);
    put_shapes(p, t + n_in, n - n_in);
    void* s = stream_handle(stream);
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = (noalloc ? vpx_sw_kernel_launch_noalloc : vpx_sw_kernel_launch)(entry, blob, size, addrs, (uint32_t)n, s);
    Py_END_ALLOW_THREADS
    return PyLong_FromLong(rc);
}

template <class F>
PyObject* guarded(F f) {
    try {
        return f();
    } catch (const Raised&) {
        return nullptr;
    } catch (const python_error&) {
        return nullptr;
    } catch (const std::exception& e) {
        PyErr_SetString(PyExc_RuntimeError, e.what());
        return nullptr;
    }
}

void expect_count(Py_ssize_t n, Py_ssize_t least, Py_ssize_t most) {
    if (n < least || n > most) raise(PyExc_TypeError, "wrong number of arguments");
}

const char* entry_name(PyObject* o) {
    const char* p = PyBytes_AsString(o);
    if (!p) throw Raised{};
    return p;
}

// launch(entry, inputs, layout, attributes, stream, noalloc, tensor ...) -> result code
PyObject* py_launch(PyObject*, PyObject* const* a, Py_ssize_t n) {
    return guarded([&]() -> PyObject* {
        expect_count(n, 7, 6 + kMostTensors);
        char* attrs = nullptr;
        Py_ssize_t size = 0;
        if (PyBytes_AsStringAndSize(a[3], &attrs, &size) < 0) throw Raised{};
        return launch_tensors(entry_name(a[0]), (int)integer(a[1]), (int)(n - 6), a + 6, a[2], attrs, (size_t)size, a[4], PyObject_IsTrue(a[5]) == 1);
    });
}

// fake_quantize(x, in_lo, in_hi, out_lo, out_hi, levels, out, layout, stream) -> result code
PyObject* py_fake_quantize(PyObject*, PyObject* const* a, Py_ssize_t n) {
    return guarded([&]() -> PyObject* {
        expect_count(n, 9, 9);
        const int64_t levels = whole(a[5]);
        PyObject* const t[6] = {a[0], a[1], a[2], a[3], a[4], a[6]};
        return launch_tensors("fake_quantize", 5, 6, t, a[7], &levels, sizeof(levels), a[8], false);
    });
}

// mvn(x, out, across_channels, normalize_variance, eps, layout, stream, noalloc) -> result code
PyObject* py_mvn(PyObject*, PyObject* const* a, Py_ssize_t n) {
    return guarded([&]() -> PyObject* {
        expect_count(n, 8, 8);
        uint8_t attrs[20];
        const int64_t flags[2] = {flag(a[2]), flag(a[3])};
        const float eps = real(a[4]);
        std::memcpy(attrs, flags, 16);
        std::memcpy(attrs + 16, &eps, 4);
        return launch_tensors("mvn1", 1, 2, a, a[5], attrs, sizeof(attrs), a[6], flag(a[7]) != 0);
    });
}

// mvn6(x, out, axes, normalize_variance, eps, eps_mode, scale or None, bias or None, layout, stream) -> result code; axes
// count from the outermost dimension
PyObject* py_mvn6(PyObject*, PyObject* const* a, Py_ssize_t n) {
    return guarded([&]() -> PyObject* {
        expect_count(n, 10, 10);
        const int64_t nd = tensor(a[0]).dim();
        PyObject* t[4] = {a[0]};
        int count = 1;
        int64_t mask = 1 | 8;
        if (a[6] != Py_None) mask |= 2, t[count++] = a[6];
        if (a[7] != Py_None) mask |= 4, t[count++] = a[7];
        t[count++] = a[1];
        PyObject* axes = PySequence_Fast(a[2], "axes: expected a sequence of integers");
        if (!axes) throw Raised{};
        uint8_t attrs[32 + 4 + 8 + 8 * kMostAxes];
        const Py_ssize_t n_axes = PySequence_Fast_GET_SIZE(axes);
        struct Drop {
            PyObject* o;
            ~Drop() { Py_DECREF(o); }
        } drop{axes};
        if (n_axes > kMostAxes) raise(PyExc_ValueError, "too many axes");
        if (nd == 0) raise(PyExc_ZeroDivisionError, "mvn6 over a tensor without dimensions");
        const int64_t head[4] = {INT64_MIN, mask, flag(a[3]), whole(a[5])}, n64 = n_axes;
        const float eps = real(a[4]);
        std::memcpy(attrs, head, 32);
        std::memcpy(attrs + 32, &eps, 4);
        std::memcpy(attrs + 36, &n64, 8);
        for (Py_ssize_t i = 0; i < n_axes; i++) {
            const int64_t axis = ((whole(PySequence_Fast_GET_ITEM(axes, i)) % nd) + nd) % nd, mem = nd - 1 - axis;
            std::memcpy(attrs + 44 + 8 * i, &mem, 8);
        }
        return launch_tensors("mvn6", count - 1, count, t, a[8], attrs, (size_t)(44 + 8 * n_axes), a[9], false);
    });
}

// softmax(x, out, axis, pad, layout, packed, stream) -> result code; axis counts from the outermost dimension
PyObject* py_softmax(PyObject*, PyObject* const* a, Py_ssize_t n) {
    return guarded([&]() -> PyObject* {
        expect_count(n, 7, 7);
        const at::Tensor &x = tensor(a[0]), &out = tensor(a[1]);
        const int64_t rank = x.dim();
        if (rank == 0) raise(PyExc_ZeroDivisionError, "softmax over a tensor without dimensions");
        const int64_t axis = ((integer(a[2]) % rank) + rank) % rank, pad = integer(a[3]);
        uint64_t words[2 + 2 * (VPX_MAX_ND_DIMS + 2)];
        uint32_t count = 2;
        if (PyObject_IsTrue(a[5]) == 1 && rank <= VPX_MAX_ND_DIMS) {
            int64_t dims[VPX_MAX_ND_DIMS], in[VPX_MAX_ND_DIMS], to[VPX_MAX_ND_DIMS] = {};
            for (int64_t d = 0; d < rank; d++) {
                dims[d] = x.size(rank - 1 - d);
                in[d] = x.stride(rank - 1 - d);
            }
            for (int64_t d = 0; d < rank && d < out.dim(); d++) to[d] = out.stride(out.dim() - 1 - d);
            const int rc = vpx_generate_softmax_attr((uint32_t)rank, dims, in, to, rank - 1 - axis, pad, words, &count);
            if (rc) return PyLong_FromLong(rc);
        } else {
            words[0] = (uint64_t)(rank - 1 - axis);
            words[1] = (uint64_t)pad;
        }
        return launch_tensors(x.scalar_type() == at::kFloat ? "softmaxFp32" : "softmax", 1, 2, a, a[4], words, count * sizeof(uint64_t), a[6], false);
    });
}

// quantize(entry, x, out, scale, zero_point, layout, stream, noalloc) -> result code: one scale and zero point, stored as values
// of the floating-point operand's type
PyObject* py_quantize(PyObject*, PyObject* const* a, Py_ssize_t n) {
    return guarded([&]() -> PyObject* {
        expect_count(n, 8, 8);
        const char* entry = entry_name(a[0]);
        const double scale = PyFloat_AsDouble(a[3]);
        if (scale == -1.0 && PyErr_Occurred()) throw Raised{};
        const int64_t zp = integer(a[4]);
        uint64_t words[3];
        uint32_t count = 0;
        const int rc = vpx_get_quant_params_attr(&scale, &zp, 1, type_code(tensor(a[entry[0] == 'q' ? 1 : 2])), words, &count);
        if (rc) return PyLong_FromLong(rc);
        return launch_tensors(entry, 1, 2, a + 1, a[5], words, count * sizeof(uint64_t), a[6], PyObject_IsTrue(a[7]) == 1);
    });
}

// A PpeInt, or a tuple of its fields.
void read_ppe(PyObject* o, vpx_ppe_int_t* ppe) {
    if (!g_ppe) raise(PyExc_RuntimeError, "set_ppe was not called");
    PyObject* made = nullptr;
    if (PyTuple_Check(o)) {
        o = made = PyObject_CallObject(g_ppe, o);
        if (!made) throw Raised{};
    } else {
        const int is = PyObject_IsInstance(o, g_ppe);
        if (is < 0) throw Raised{};
        if (!is) {
            PyErr_Format(PyExc_TypeError, "ppe must be a PpeInt, got %s", Py_TYPE(o)->tp_name);
            throw Raised{};
        }
    }
    Py_buffer view;
    const int rc = PyObject_GetBuffer(o, &view, PyBUF_SIMPLE);
    const bool fits = rc == 0 && view.len == (Py_ssize_t)sizeof(*ppe);
    if (fits) std::memcpy(ppe, view.buf, sizeof(*ppe));
    if (rc == 0) PyBuffer_Release(&view);
    Py_XDECREF(made);
    if (rc < 0) throw Raised{};
    if (!fits) raise(PyExc_TypeError, "a PpeInt of another size");
}

void require(bool ok, const char* text) {
    if (!ok) raise(PyExc_AssertionError, text);
}

// The first n values of a sequence; `exactly`: which has no others.
void read_values(PyObject* o, int32_t* v, Py_ssize_t n, bool exactly) {
    PyObject* f = PySequence_Fast(o, "expected a sequence of integers");
    if (!f) throw Raised{};
    const Py_ssize_t size = PySequence_Fast_GET_SIZE(f);
    if (size < n || (exactly && size > n)) {
        Py_DECREF(f);
        PyErr_Format(exactly ? PyExc_ValueError : PyExc_IndexError, "expected %zd values, got %zd", n, size);
        throw Raised{};
    }
    for (Py_ssize_t i = 0; i < n; i++) {
        const long x = PyLong_AsLong(PySequence_Fast_GET_ITEM(f, i));
        if (x == -1 && PyErr_Occurred()) {
            Py_DECREF(f);
            throw Raised{};
        }
        v[i] = (int32_t)x;
    }
    Py_DECREF(f);
}

// N, H, W, C strides (elements) of an operand that is a view of a larger tensor; a contiguous one leaves them zero.
void view_strides(int64_t* field, const at::Tensor& t) {
    if (!t.is_contiguous())
        for (int i = 0; i < 4; i++) field[i] = t.stride(t.dim() - 4 + i);
}

int run_task(const vpx_nce_task_t& t, PyObject* stream) {
    void* s = stream_handle(stream);
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = vpx_nce_task(&t, s);
    Py_END_ALLOW_THREADS
    return rc;
}

void set_operands(vpx_nce_task_t& t, const at::Tensor& in, const at::Tensor& w, const at::Tensor* table, const at::Tensor& out) {
    t.input = in.data_ptr();
    t.weights = w.data_ptr();
    t.weight_table = table ? (const int32_t*)table->data_ptr() : nullptr;
    t.output = out.data_ptr();
    t.input_type = (int32_t)type_code(in);
    t.weights_type = (int32_t)type_code(w);
    t.output_type = (int32_t)type_code(out);
}

// conv(input, weights, weight_table, out, ppe, zp_in, zp_w, zp_out, strides, pads, stream, groups) -> result code
PyObject* py_conv(PyObject*, PyObject* const* a, Py_ssize_t n) {
    return guarded([&]() -> PyObject* {
        expect_count(n, 12, 12);
        const at::Tensor &in = tensor(a[0]), &w = tensor(a[1]), &table = tensor(a[2]), &out = tensor(a[3]);
        const bool grouped = a[11] != Py_None;
        const int64_t groups = grouped ? integer(a[11]) : 0;
        if (in.dim() < 4 || w.dim() < 4) raise(PyExc_ValueError, "not enough values to unpack (expected 4)");
        if (grouped) {
            require(table.dim() > 0 && out.dim() > 0 && in.size(0) == groups && w.size(0) == groups && table.size(0) == groups && out.size(0) == groups,
                    "every operand of a grouped task has a leading dimension of its groups");
            require(in.is_contiguous() && w.is_contiguous() && table.is_contiguous() && out.is_contiguous(), "the operands of a grouped task are dense");
        }
        vpx_nce_task_t t{};
        t.task_type = VPX_NCE_CONV;
        t.groups = (int32_t)groups;
        set_operands(t, in, w, &table, out);
        t.N = in.size(-4);
        t.H = in.size(-3);
        t.W = in.size(-2);
        t.IC = in.size(-1);
        t.OC = w.size(-4);
        t.kernel_size[0] = (int32_t)w.size(-3);
        t.kernel_size[1] = (int32_t)w.size(-2);
        require(t.IC == w.size(-1), "input and weights have different channel counts");
        read_values(a[8], t.kernel_strides, 2, true);
        read_values(a[9], t.kernel_padding, 4, false);
        t.zp_in = integer32(a[5]);
        t.zp_w = integer32(a[6]);
        t.zp_out = integer32(a[7]);
        read_ppe(a[4], &t.ppe);
        if (!grouped) {
            require(w.is_contiguous() && table.is_contiguous(), "weights and weight table are dense");
            view_strides(t.input_strides, in);
            require(out.is_contiguous() || out.dim() >= 4, "the output has four dimensions");
            view_strides(t.output_strides, out);
        }
        return PyLong_FromLong(run_task(t, a[10]));
    });
}

// matmul(a, b_nk, weight_table, out, ppe, zp_a, zp_b, zp_out, stream) -> out in the task's shape, or a result code: [M,K] x [N,K]
// as the 1x1 convolution of M positions, or [G,M,K] x [G,N,K] as its grouped form
PyObject* py_matmul(PyObject*, PyObject* const* a, Py_ssize_t n) {
    return guarded([&]() -> PyObject* {
        expect_count(n, 9, 9);
        const at::Tensor &x = tensor(a[0]), &b = tensor(a[1]), &table = tensor(a[2]), &out = tensor(a[3]);
        const bool grouped = x.dim() == 3;
        if ((x.dim() != 2 && !grouped) || (grouped ? b.dim() < 2 : b.dim() != 2))
            raise(PyExc_ValueError, "a and b are matrices, or three-dimensional (groups first)");
        const int64_t M = x.size(-2), K = x.size(-1), N = b.size(grouped ? 1 : 0), G = grouped ? x.size(0) : 1;
        if (b.numel() != G * N * K || out.numel() != G * M * N) raise(PyExc_RuntimeError, "a [M,K], b [N,K] and out [M,N] do not fit each other");
        require(b.is_contiguous() && table.is_contiguous(), "b and the weight table are dense");
        vpx_nce_task_t t{};
        t.task_type = VPX_NCE_CONV;
        set_operands(t, x, b, &table, out);
        t.N = t.W = 1;
        t.H = M;
        t.IC = K;
        t.OC = N;
        t.kernel_size[0] = t.kernel_size[1] = t.kernel_strides[0] = t.kernel_strides[1] = 1;
        t.zp_in = integer32(a[5]);
        t.zp_w = integer32(a[6]);
        t.zp_out = integer32(a[7]);
        read_ppe(a[4], &t.ppe);
        if (grouped) {
            require(table.dim() > 0 && table.size(0) == G, "the weight table has a leading dimension of groups");
            require(x.is_contiguous() && out.is_contiguous(), "the operands of a grouped matmul are dense");
            t.groups = (int32_t)G;
        } else {
            // a matrix that is a view of a larger one (out with any dimensions that make one), as [1, rows, 1, columns]
            if (!x.is_contiguous()) view_strides(t.input_strides, x.view({1, M, 1, K}));
            if (!out.is_contiguous()) view_strides(t.output_strides, out.view({1, M, 1, N}));
        }
        const int rc = run_task(t, a[8]);
        if (rc) return PyLong_FromLong(rc);
        return THPVariable_Wrap(grouped ? out.view({G, 1, M, 1, N}) : out.view({1, M, 1, N}));
    });
}

// eltwise(in1, in2, out, ppe, zp_in1, zp_in2, zp_out, subtract, stream) -> result code
PyObject* py_eltwise(PyObject*, PyObject* const* a, Py_ssize_t n) {
    return guarded([&]() -> PyObject* {
        expect_count(n, 9, 9);
        const at::Tensor &in1 = tensor(a[0]), &in2 = tensor(a[1]), &out = tensor(a[2]);
        require(in1.dim() == 4 && in1.sizes() == in2.sizes() && in1.sizes() == out.sizes(), "both inputs and the output have one four-dimensional shape");
        vpx_nce_task_t t{};
        t.task_type = VPX_NCE_ELTWISE;
        t.eltwise_type = PyObject_IsTrue(a[7]) == 1 ? VPX_ELTWISE_SUBTRACT : VPX_ELTWISE_ADD;
        set_operands(t, in1, in2, nullptr, out);
        t.N = in1.size(0);
        t.H = in1.size(1);
        t.W = in1.size(2);
        t.IC = t.OC = in1.size(3);
        t.kernel_size[0] = t.kernel_size[1] = t.kernel_strides[0] = t.kernel_strides[1] = 1;
        t.zp_in = integer32(a[4]);
        t.zp_w = integer32(a[5]);
        t.zp_out = integer32(a[6]);
        read_ppe(a[3], &t.ppe);
        view_strides(t.input_strides, in1);
        view_strides(t.weights_strides, in2);
        view_strides(t.output_strides, out);
        return PyLong_FromLong(run_task(t, a[8]));
    });
}

// stream(stream or None) -> handle as an integer
PyObject* py_stream(PyObject*, PyObject* stream) {
    return guarded([&]() -> PyObject* { return PyLong_FromVoidPtr(stream_handle(stream)); });
}

PyObject* py_set_orders(PyObject*, PyObject* orders) {
    if (!PyDict_Check(orders)) {
        PyErr_SetString(PyExc_TypeError, "expected the dict of layout codes");
        return nullptr;
    }
    Py_INCREF(orders);
    Py_XSETREF(g_orders, orders);
    Py_RETURN_NONE;
}

PyObject* py_set_ppe(PyObject*, PyObject* type) {
    if (!PyType_Check(type)) {
        PyErr_SetString(PyExc_TypeError, "expected the type of a ppe");
        return nullptr;
    }
    Py_INCREF(type);
    Py_XSETREF(g_ppe, type);
    Py_RETURN_NONE;
}

#define FAST(f) (PyCFunction)(void (*)(void)) f
PyMethodDef kMethods[] = {
    {"launch", FAST(py_launch), METH_FASTCALL, "software kernel on tensors"},
    {"fake_quantize", FAST(py_fake_quantize), METH_FASTCALL, "FakeQuantize on tensors"},
    {"mvn", FAST(py_mvn), METH_FASTCALL, "MVN-1 on tensors"},
    {"mvn6", FAST(py_mvn6), METH_FASTCALL, "MVN-6 on tensors"},
    {"softmax", FAST(py_softmax), METH_FASTCALL, "softmax on tensors"},
    {"quantize", FAST(py_quantize), METH_FASTCALL, "quantize / dequantize with one scale"},
    {"conv", FAST(py_conv), METH_FASTCALL, "NCE convolution task"},
    {"matmul", FAST(py_matmul), METH_FASTCALL, "NCE matmul task"},
    {"eltwise", FAST(py_eltwise), METH_FASTCALL, "NCE eltwise task"},
    {"stream", py_stream, METH_O, "handle of a stream, or of the current one"},
    {"set_orders", py_set_orders, METH_O, "names of the layouts"},
    {"set_ppe", py_set_ppe, METH_O, "type of a ppe"},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_binding", "operator calls on torch tensors through libvpx_amd.so", -1, kMethods,
                       nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__binding(void) {
    return PyModule_Create(&kModule);
}
