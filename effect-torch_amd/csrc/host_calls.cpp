// The three execute calls of a serving program as a CPython module, from torch tensors straight to the C ABI
// (linear_into, embedding_into, kv_attention_into of quantized.py and kv_cache.py). Describing three or four tensors to
// ctypes - arrays of shapes and strides, a structure, its reference, for every call anew - costs the interpreter
// 8 to 12 us, more than a small launch lasts on the device; read from the tensors' own fields it costs half a
// microsecond.
//
// A call whose arguments are not what these functions read (another tensor type, an element type the ABI does not
// know, no device) returns kNotTaken before anything has happened, and the caller goes through ctypes, which words
// the error.
#include <Python.h>

#include <ATen/ATen.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>

#include "et_hip.h"

namespace {

constexpr long kNotTaken = -1;

bool element_type(at::ScalarType type, int32_t* out) {
    switch (type) {
        case at::kFloat: *out = ET_DTYPE_F32; return true;
        case at::kDouble: *out = ET_DTYPE_F64; return true;
        case at::kHalf: *out = ET_DTYPE_F16; return true;
        case at::kBFloat16: *out = ET_DTYPE_BF16; return true;
        case at::kByte: *out = ET_DTYPE_U8; return true;
        case at::kUInt32: *out = ET_DTYPE_U32; return true;
        case at::kLong: *out = ET_DTYPE_I64; return true;
        default: return false;
    }
}

// A plain strided tensor on the device (None allowed where `optional`).
bool tensor_of(PyObject* object, bool optional, const at::Tensor** out) {
    *out = nullptr;
    if (object == Py_None) return optional;
    if (!THPVariable_Check(object)) return false;
    const at::Tensor& tensor = THPVariable_Unpack(object);
    if (!tensor.defined() || tensor.layout() != at::kStrided || !tensor.is_cuda()) return false;
    *out = &tensor;
    return true;
}

struct Described {
    et_tensor tensor;
    const et_tensor* ref = nullptr;  // null for None
    bool from(PyObject* object, bool optional = false) {
        const at::Tensor* source;
        if (!tensor_of(object, optional, &source)) return false;
        if (source == nullptr) return true;
        if (!element_type(source->scalar_type(), &tensor.dtype)) return false;
        tensor.data = source->storage().data();
        tensor.rank = static_cast<int32_t>(source->dim());
        tensor.shape = reinterpret_cast<const uint64_t*>(source->sizes().data());
        tensor.strides = reinterpret_cast<const uint64_t*>(source->strides().data());
        tensor.offset = static_cast<uint64_t>(source->storage_offset());
        ref = &tensor;
        return true;
    }
};

// Where a contiguous tensor's elements start, and their bytes.
bool span_of(PyObject* object, bool optional, void** data, uint64_t* bytes) {
    const at::Tensor* tensor;
    *data = nullptr;
    *bytes = 0;
    if (!tensor_of(object, optional, &tensor)) return false;
    if (tensor != nullptr) {
        *data = tensor->data_ptr();
        *bytes = static_cast<uint64_t>(tensor->nbytes());
    }
    return true;
}

bool unsigned_of(PyObject* object, uint64_t* out) {
    *out = PyLong_AsUnsignedLongLong(object);
    return !PyErr_Occurred();
}

// A stream handle: None = torch's current stream of the current device.
bool stream_of(PyObject* object, void** out) {
    if (object == Py_None) {
        *out = c10::hip::getCurrentHIPStream().stream();
        return true;
    }
    uint64_t handle;
    if (!unsigned_of(object, &handle)) return false;
    *out = reinterpret_cast<void*>(handle);
    return true;
}

bool address_of(PyObject* object, void** out) {
    uint64_t address = 0;
    if (object != Py_None && !unsigned_of(object, &address)) return false;
    *out = reinterpret_cast<void*>(address);
    return true;
}

template <typename Body>
PyObject* taken(Body&& body) {
    PyObject* result = nullptr;
    try {
        result = body();
    } catch (...) {  // torch's own checks (no device, a tensor without storage)
        result = nullptr;
    }
    if (result == nullptr) {
        PyErr_Clear();
        return PyLong_FromLong(kNotTaken);
    }
    return result;
}

// linear_into(plan, input, weight, bias, destination, workspace, stream, cancel) -> et_status
PyObject* linear_into(PyObject*, PyObject* const* args, Py_ssize_t count) {
    return taken([&]() -> PyObject* {
        void *plan, *workspace, *stream, *cancel;
        uint64_t workspace_bytes;
        Described input, weight, bias, destination;
        if (count != 8 || !address_of(args[0], &plan) || !input.from(args[1]) || !weight.from(args[2]) ||
            !bias.from(args[3], true) || !destination.from(args[4]) || !span_of(args[5], true, &workspace, &workspace_bytes) ||
            !stream_of(args[6], &stream) || !address_of(args[7], &cancel))
            return nullptr;
        int status;
        Py_BEGIN_ALLOW_THREADS;
        status = et_hip_linear_into(static_cast<const et_linear_plan*>(plan), input.ref, weight.ref, bias.ref, destination.ref,
                                    workspace, workspace_bytes, stream, static_cast<const volatile int32_t*>(cancel));
        Py_END_ALLOW_THREADS;
        return PyLong_FromLong(status);
    });
}

// The device status block of a call and the call's et_status.
PyObject* with_status(const at::Tensor& block, int status) {
    PyObject* wrapped = THPVariable_Wrap(block);
    if (wrapped == nullptr) return nullptr;
    return Py_BuildValue("(iN)", status, wrapped);
}

at::Tensor status_block(PyObject* like, uint64_t bytes) {
    return at::empty({static_cast<int64_t>(bytes)}, THPVariable_Unpack(like).options().dtype(at::kByte));
}

// embedding_into(plan, indexes, weight, destination, stream, cancel) -> (et_status, status block)
PyObject* embedding_into(PyObject*, PyObject* const* args, Py_ssize_t count) {
    return taken([&]() -> PyObject* {
        void *plan, *stream, *cancel;
        Described indexes, weight, destination;
        if (count != 6 || !address_of(args[0], &plan) || !indexes.from(args[1]) || !weight.from(args[2]) ||
            !destination.from(args[3]) || !stream_of(args[4], &stream) || !address_of(args[5], &cancel))
            return nullptr;
        const at::Tensor block = status_block(args[3], ET_HIP_STATUS_BYTES);
        void* at = block.data_ptr();
        int status;
        Py_BEGIN_ALLOW_THREADS;
        status = et_hip_embedding_into(static_cast<const et_embedding_plan*>(plan), indexes.ref, weight.ref, destination.ref, at,
                                       stream, static_cast<const volatile int32_t*>(cancel));
        Py_END_ALLOW_THREADS;
        return with_status(block, status);
    });
}

// kv_attention_into(k_slab, v_slab, k_scales, v_scales, block_table, cursors, advances, block_size, max_context,
//                   active_batch, context_window, q, k, v, scale, window, destination, workspace, stream, cancel)
//   -> (et_status, status block)
PyObject* kv_attention_into(PyObject*, PyObject* const* args, Py_ssize_t count) {
    return taken([&]() -> PyObject* {
        if (count != 20) return nullptr;
        et_kv_layer layer = {};
        Described slab, table, cursors, q, k, v, destination;
        uint64_t bytes, workspace_bytes, window;
        void *pointer, *workspace, *stream, *cancel;
        if (!slab.from(args[0]) || slab.tensor.rank != 3) return nullptr;
        layer.slab_dtype = slab.tensor.dtype;
        layer.max_tokens = slab.tensor.shape[0];
        layer.kv_heads = slab.tensor.shape[1];
        layer.head_dim = slab.tensor.shape[2];
        if (!span_of(args[0], false, &layer.k_slab, &bytes) || !span_of(args[1], false, &layer.v_slab, &bytes)) return nullptr;
        if (!span_of(args[2], true, &pointer, &bytes)) return nullptr;
        layer.k_scales = static_cast<float*>(pointer);
        if (!span_of(args[3], true, &pointer, &bytes)) return nullptr;
        layer.v_scales = static_cast<float*>(pointer);
        const at::Tensor* tensor;
        if (!tensor_of(args[4], false, &tensor) || tensor->dim() != 2) return nullptr;
        layer.block_table = static_cast<const uint32_t*>(tensor->data_ptr());
        layer.table_stride = static_cast<uint64_t>(tensor->size(1));
        if (!tensor_of(args[5], false, &tensor)) return nullptr;
        layer.cursors = static_cast<const uint32_t*>(tensor->data_ptr());
        layer.slots = static_cast<uint64_t>(tensor->numel());
        if (!span_of(args[6], false, &pointer, &bytes)) return nullptr;
        layer.advances = static_cast<const uint32_t*>(pointer);
        if (!unsigned_of(args[7], &layer.block_size) || !unsigned_of(args[8], &layer.max_context) ||
            !unsigned_of(args[9], &layer.active_batch) || !unsigned_of(args[10], &layer.context_window))
            return nullptr;
        if (!q.from(args[11]) || !k.from(args[12]) || !v.from(args[13])) return nullptr;
        const double scale = PyFloat_AsDouble(args[14]);
        if (PyErr_Occurred() || !unsigned_of(args[15], &window) || !destination.from(args[16]) ||
            !span_of(args[17], false, &workspace, &workspace_bytes) || !stream_of(args[18], &stream) ||
            !address_of(args[19], &cancel))
            return nullptr;
        const at::Tensor block = status_block(args[16], ET_HIP_KV_STATUS_BYTES(layer.slots > 0 ? layer.slots : 1));
        void* at = block.data_ptr();
        int status;
        Py_BEGIN_ALLOW_THREADS;
        status = et_hip_kv_attention_into(&layer, q.ref, k.ref, v.ref, scale, window, destination.ref, workspace, workspace_bytes, at,
                                          stream, static_cast<const volatile int32_t*>(cancel));
        Py_END_ALLOW_THREADS;
        return with_status(block, status);
    });
}

PyMethodDef kMethods[] = {
    {"linear_into", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(linear_into)), METH_FASTCALL, nullptr},
    {"embedding_into", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(embedding_into)), METH_FASTCALL, nullptr},
    {"kv_attention_into", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(kv_attention_into)), METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "et_host_calls", nullptr, -1, kMethods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit_et_host_calls(void) { return PyModule_Create(&kModule); }
