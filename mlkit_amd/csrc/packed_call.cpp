// A packed layer's call from Python as one native function: the checks that PackedLinear.forward makes, the output's
// allocation and the launch.  Layers of small models wait for nothing but the host: a module call of 896 to 128 values takes 8.1
// us of it through ctypes and 5.0 us through this function (4 of them the launch), the seven layers of such a block 64 and 43 us.
//
// The object keeps the arguments of mk_packed_layer_matvec / _matmul for as long as the layer's five buffers stay where they
// were (their addresses and the types of scales and bias are compared in every call) and answers None, with nothing launched,
// whenever the call is not the plain one: the Python path then does what it always did, errors included.

#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/TracerMode.h>
#include <ATen/core/grad_mode.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>

#include "../../include/mlkit_amd.h"

namespace {

using LayerCall = int (*)(const mk_packed_layer *, const void *, int, void *, int, void *);

constexpr int kBuffers = 5;
const char *const kNames[kBuffers] = {"packed", "scales", "values", "zeros", "bias"};
PyObject *names[kBuffers];

struct PackedCall {
    PyObject_HEAD
    mk_packed_layer layer;
    const void *address[kBuffers];
    int scale_type, bias_type;   // of at::ScalarType; -1: none
    LayerCall matvec, matmul;
};

// The tensor of a buffer that may be None; false for anything else.
bool buffer_of(PyObject *buffers, int index, const at::Tensor **tensor) {
    PyObject *found = PyDict_GetItem(buffers, names[index]);   // borrowed
    *tensor = nullptr;
    if (!found) return false;
    if (found == Py_None) return true;
    if (!THPVariable_Check(found)) return false;
    *tensor = &THPVariable_Unpack(found);
    return true;
}

int code_of(at::ScalarType type) {
    return type == at::kFloat ? MK_F32 : type == at::kHalf ? MK_F16 : type == at::kBFloat16 ? MK_BF16 : -1;
}

// The plain call's output, or null without an error where it is not one.  `product`: mk_packed_layer_matmul, which stands for
// a dense product: nothing may differentiate, batch, record, watch or cast it (the caller has made sure of that).
PyObject *launch(PackedCall *self, PyObject *input, PyObject *buffers, long limit, bool product) {
    if (!THPVariable_CheckExact(input) || !PyDict_Check(buffers)) return nullptr;
    const at::Tensor &x = THPVariable_Unpack(input);
    const int type = code_of(x.scalar_type());
    if (type < 0 || !x.is_cuda() || x.layout() != at::kStrided || !x.has_storage() || x.is_neg() || x.dim() < 1 ||
        x.size(-1) != self->layer.input_width || !x.is_contiguous() || (x.requires_grad() && at::GradMode::is_enabled()))
        return nullptr;
    const int64_t rows = x.numel() / self->layer.input_width;
    if (rows < 1 || rows > limit || (product && type == MK_F32)) return nullptr;
    if (c10::impl::TorchDispatchModeTLS::any_modes_set() || at::impl::torch_function_mode_enabled() ||
        at::tracer::impl::is_dispatch_enabled())
        return nullptr;
    for (int i = 0; i < kBuffers; ++i) {
        const at::Tensor *tensor;
        if (!buffer_of(buffers, i, &tensor) || (tensor ? tensor->const_data_ptr() : nullptr) != self->address[i]) return nullptr;
        if (i == 0 && (!tensor || tensor->device() != x.device())) return nullptr;
        if (i == 1 && (!tensor || static_cast<int>(tensor->scalar_type()) != self->scale_type)) return nullptr;
        if (i == 4 && (tensor ? static_cast<int>(tensor->scalar_type()) : -1) != self->bias_type) return nullptr;
    }
    c10::SmallVector<int64_t, 6> shape(x.sizes().begin(), x.sizes().end());
    shape.back() = self->layer.output_width;
    at::Tensor y = at::empty(shape, x.options());
    const LayerCall call = product ? self->matmul : self->matvec;
    const void *from = x.const_data_ptr();
    void *to = y.mutable_data_ptr(), *stream = c10::hip::getCurrentHIPStream(x.device().index()).stream();
    int status;
    Py_BEGIN_ALLOW_THREADS
    status = call(&self->layer, from, type, to, static_cast<int>(rows), stream);
    Py_END_ALLOW_THREADS
    return status == MK_OK ? THPVariable_Wrap(std::move(y)) : nullptr;
}

template <bool PRODUCT>
PyObject *call_method(PyObject *object, PyObject *const *arguments, Py_ssize_t count) {
    if (count != 3) {
        PyErr_SetString(PyExc_TypeError, "expected (inputs, buffers, row limit)");
        return nullptr;
    }
    const long limit = PyLong_AsLong(arguments[2]);
    if (limit == -1 && PyErr_Occurred()) return nullptr;
    try {
        PyObject *result = launch(reinterpret_cast<PackedCall *>(object), arguments[0], arguments[1], limit, PRODUCT);
        if (result || PyErr_Occurred()) return result;
    } catch (const std::exception &) {   // (out of memory, say: the Python path meets it again and reports it as torch does)
    }
    Py_RETURN_NONE;
}

// PackedCall(layer structure, scale tensor, bias tensor or None, addresses of the two entry points)
PyObject *create(PyTypeObject *type, PyObject *arguments, PyObject *) {
    Py_buffer layer;
    PyObject *scales, *bias;
    unsigned long long matvec, matmul;
    if (!PyArg_ParseTuple(arguments, "y*OOKK", &layer, &scales, &bias, &matvec, &matmul)) return nullptr;
    const bool valid = layer.len == sizeof(mk_packed_layer) && THPVariable_Check(scales) && (bias == Py_None || THPVariable_Check(bias));
    PackedCall *self = valid ? reinterpret_cast<PackedCall *>(type->tp_alloc(type, 0)) : nullptr;
    if (self) {
        memcpy(&self->layer, layer.buf, sizeof(mk_packed_layer));
        const mk_packed_layer &l = self->layer;
        const void *addresses[kBuffers] = {l.packed, l.scales, l.values, l.zeros, l.bias};
        memcpy(self->address, addresses, sizeof(addresses));
        self->scale_type = static_cast<int>(THPVariable_Unpack(scales).scalar_type());
        self->bias_type = bias == Py_None ? -1 : static_cast<int>(THPVariable_Unpack(bias).scalar_type());
        self->matvec = reinterpret_cast<LayerCall>(matvec);
        self->matmul = reinterpret_cast<LayerCall>(matmul);
    } else if (!valid) {
        PyErr_SetString(PyExc_TypeError, "PackedCall(layer, scales, bias, matvec, matmul)");
    }
    PyBuffer_Release(&layer);
    return reinterpret_cast<PyObject *>(self);
}

PyMethodDef methods[] = {
    {"matvec", reinterpret_cast<PyCFunction>(reinterpret_cast<void *>(&call_method<false>)), METH_FASTCALL, "outputs, or None where the call is not a plain one"},
    {"matmul", reinterpret_cast<PyCFunction>(reinterpret_cast<void *>(&call_method<true>)), METH_FASTCALL, "the same for the product of more rows"},
    {nullptr, nullptr, 0, nullptr},
};

PyTypeObject packed_call_type = [] {
    PyTypeObject type = {PyVarObject_HEAD_INIT(nullptr, 0)};
    type.tp_name = "mlkit_amd._packed_call.PackedCall";
    type.tp_basicsize = sizeof(PackedCall);
    type.tp_flags = Py_TPFLAGS_DEFAULT;
    type.tp_methods = methods;
    type.tp_new = create;
    return type;
}();

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_packed_call", nullptr, -1, nullptr, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__packed_call() {
    if (PyType_Ready(&packed_call_type) < 0) return nullptr;
    for (int i = 0; i < kBuffers; ++i)
        if (!(names[i] = PyUnicode_InternFromString(kNames[i]))) return nullptr;
    PyObject *created = PyModule_Create(&module);
    if (!created) return nullptr;
    Py_INCREF(&packed_call_type);
    if (PyModule_AddObject(created, "PackedCall", reinterpret_cast<PyObject *>(&packed_call_type)) < 0) return nullptr;
    return created;
}
