// The host path of the operators on torch tensors: what ops.py and nn.py do per call -- checks of the tensors against a
// descriptor, the result's allocation, the stream's scratch buffer, the call of the C ABI -- without the interpreter's share of it.
// Layers of a few microseconds are bound by that: of the host's time a forward call with a packed filter took 9.1 us and takes 5.2,
// both gradients of a convolution 22.1 and 14.6, a Dense step 22.1 and 10.4, a convolution with its norm in evaluation 13.3 and 6.2.
//
// Every function answers NotImplemented for a call that is not a plain one -- tensors of another type, shape, device or order
// than the descriptor's, subclasses (of tensors and of descriptors) and wrapped tensors, function and dispatch modes -- and the Python code behind it, which is
// the operators' definition and reports their errors, runs instead.
//
// What is kept between calls: per descriptor (in its own dictionary) its shapes and workspace sizes, checked against the
// descriptor's fields each time; per device and stream one scratch buffer that only grows (captured calls: see scratch).  All
// under the interpreter's lock, which is released around the library's calls.
#include <torch/csrc/python_headers.h>

#include <ATen/core/Tensor.h>
#include <ATen/ops/empty.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <c10/core/GradMode.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPException.h>
#include <c10/hip/HIPGuard.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/DynamicTypes.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cstring>
#include <unordered_map>
#include <vector>

#include "../../include/phx_bn.h"
#include "../../include/phx_qconv.h"

namespace {

// ---- the C ABI, by the addresses of the library that capi.py has loaded ----
#define PHX_HOST_FUNCTIONS(X)                                                                                                   \
    X(phx_qconv2d_workspace_bytes) X(phx_qdense_workspace_bytes) X(phx_qconv2d_fwd) X(phx_qconv2d_fwd_prepacked)               \
    X(phx_qconv2d_fwd_norm) X(phx_qconv2d_bwd_weights) X(phx_qconv2d_bwd_data) X(phx_qconv2d_bwd_data_prepacked)               \
    X(phx_qconv2d_bwd_data_add) X(phx_qconv2d_pack_filters) X(phx_qdense_fwd) X(phx_qdense_bwd) X(phx_qdense_bwd_weights) \
    X(phx_bn_workspace_bytes) X(phx_bn_fwd_train) X(phx_bn_bwd)
struct Library {
#define PHX_FIELD(f) decltype(&::f) f = nullptr;
    PHX_HOST_FUNCTIONS(PHX_FIELD)
#undef PHX_FIELD
} L;

PyObject* g_check = nullptr;       // capi.check(status, name): raises
PyObject* g_capi_dict = nullptr;   // capi's namespace: tuning_generation
PyObject* g_parameter = nullptr;   // torch.nn.Parameter
PyObject* g_conv_type = nullptr;   // ops.Conv2DDescriptor
PyObject* g_dense_type = nullptr;  // ops.DenseDescriptor
PyObject* g_forward_ad = nullptr;  // torch.autograd.forward_ad's namespace: _current_level

struct Names {
#define PHX_HOST_NAMES(X)                                                                                                       \
    X(_host) X(c) X(input_shape) X(filter_shape) X(output_shape) X(bias_shape) X(dtype) X(use_bias) X(real_valued_input)       \
    X(algebra) X(fwd) X(bwd_data) X(layout_key) X(tuning_generation) X(_current_level) X(_parameters) X(_buffers) X(_descs)    \
    X(_packed) X(_pack_pending) X(_forward_hooks) X(_forward_pre_hooks) X(_backward_hooks) X(_backward_pre_hooks) X(forward)   \
    X(training) X(data_format) X(weight) X(bias) X(running_mean) X(running_var) X(eps) X(relu)
#define PHX_FIELD(n) PyObject* n = nullptr;
    PHX_HOST_NAMES(PHX_FIELD)
#undef PHX_FIELD
} N;

PyObject* plain_no() { Py_RETURN_NOTIMPLEMENTED; }

// a reported status becomes the library's exception
bool ok(int status, const char* what) {
    if (status == PHX_OK) return true;
    PyObject* r = PyObject_CallFunction(g_check, "is", status, what);
    Py_XDECREF(r);
    if (r) PyErr_SetString(PyExc_RuntimeError, what);
    return false;
}

template <typename F>
int unlocked(F call) {
    int status;
    Py_BEGIN_ALLOW_THREADS
    status = call();
    Py_END_ALLOW_THREADS
    return status;
}

// no mode that looks at operators or functions
bool no_modes() { return c10::impl::TorchDispatchModeTLS::stack_len() == 0 && at::impl::PythonTorchFunctionTLS::stack_len() == 0; }

// A tensor whose memory the library may read: torch's own type (or a parameter), dense, on the GPU, not wrapped by a transform.
const at::Tensor* plain(PyObject* o) {
    if (Py_TYPE(o) != reinterpret_cast<PyTypeObject*>(THPVariableClass) && reinterpret_cast<PyObject*>(Py_TYPE(o)) != g_parameter) return nullptr;
    const at::Tensor& t = THPVariable_Unpack(o);
    constexpr c10::DispatchKeySet odd({c10::DispatchKey::Python, c10::DispatchKey::PythonTLSSnapshot, c10::DispatchKey::FuncTorchBatched,
                                       c10::DispatchKey::FuncTorchGradWrapper, c10::DispatchKey::Functionalize, c10::DispatchKey::Conjugate,
                                       c10::DispatchKey::Negative, c10::DispatchKey::ZeroTensor, c10::DispatchKey::Batched, c10::DispatchKey::Fake});
    if (!t.defined() || t.key_set().has_any(odd) || !t.is_cuda() || t.layout() != c10::kStrided || !t.has_storage() || !t.is_contiguous()) return nullptr;
    return &t;
}
const at::Tensor* plain(PyObject* o, c10::IntArrayRef shape, c10::ScalarType type, c10::Device device) {
    const at::Tensor* t = plain(o);
    return t && t->scalar_type() == type && t->device() == device && t->sizes() == shape ? t : nullptr;
}

void* address(const at::Tensor* t) { return t ? t->data_ptr() : nullptr; }
size_t bytes_of(const at::Tensor* t) { return t ? (size_t)t->numel() : 0; }

// ---- scratch buffers: grow-only, one per device and stream ----
struct PairHash {
    size_t operator()(const std::pair<int, uintptr_t>& k) const { return k.second * 31 + (size_t)k.first; }
};
struct Buffer {
    at::Tensor memory;
    bool reserved = false;  // asked for in front of a capture (ops.reserve_workspace)
    bool in_graph = false;  // ... and met by one
};
std::unordered_map<std::pair<int, uintptr_t>, Buffer, PairHash>& buffers() {
    static auto* b = new std::unordered_map<std::pair<int, uintptr_t>, Buffer, PairHash>;  // (tensors outlive the runtime's own shutdown)
    return *b;
}
bool holds(const Buffer& b, size_t bytes) { return b.memory.defined() && (size_t)b.memory.numel() >= bytes; }
bool captured(uintptr_t stream) {
    if (!stream) return false;  // (the default stream cannot be)
    hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
    C10_HIP_CHECK(hipStreamIsCapturing(reinterpret_cast<hipStream_t>(stream), &status));
    return status != hipStreamCaptureStatusNone;
}
// A graph replays with the addresses that it was captured with, on any stream and whatever eager calls do meanwhile.  A captured
// call therefore gets memory of its own, from the allocator, which under capture takes it from the graph's pool and gives it to
// later calls of the same capture and stream only.  Nothing of a graph's pool is kept here, and no graph is left with a buffer of
// this table that grows away.  One that was reserved for a capture serves that capture, and is never given back then.
at::Tensor scratch(c10::Device device, uintptr_t stream, size_t bytes, bool reserve = false) {
    Buffer& b = buffers()[{device.index(), stream}];
    const bool capture = captured(stream);
    if (holds(b, bytes) && (!capture || b.reserved)) {
        b.reserved |= reserve;
        b.in_graph |= capture;
        return b.memory;
    }
    at::Tensor memory;
    {
        // (of the stream that works in it: given back, it is that stream's again, behind what is enqueued there)
        const c10::hip::HIPStreamGuard guard(c10::hip::getStreamFromExternal(reinterpret_cast<hipStream_t>(stream), device.index()));
        memory = at::empty({(int64_t)std::max<size_t>(bytes, 1)}, c10::TensorOptions().dtype(c10::kByte).device(device));
    }
    if (capture) return memory;
    if (b.in_graph) {
        static auto* kept = new std::vector<at::Tensor>;
        kept->push_back(b.memory);
        b.in_graph = false;
    }
    b.memory = memory;
    b.reserved |= reserve;
    return memory;
}
uintptr_t current_stream(c10::Device device) { return reinterpret_cast<uintptr_t>(c10::hip::getCurrentHIPStream(device.index()).stream()); }

// ---- what is kept of a descriptor ----
enum { FIELD_C, FIELD_INPUT, FIELD_FILTER, FIELD_OUTPUT, FIELD_DTYPE, FIELD_USE_BIAS, FIELD_BIAS_SHAPE, FIELD_REAL, DESC_FIELDS };
struct Desc {
    PyObject_HEAD
    PyObject* fields[DESC_FIELDS];  // what it was made from (owned; null: not there)
    const void* abi;      // the ctypes structure's memory
    bool dense, bias, real;
    c10::ScalarType type;
    std::vector<int64_t> in, filter, out, bias_shape;
    phx_qconv_desc conv_copy;
    phx_qdense_desc dense_copy;
    long generation;
    size_t workspace[3];
    bool known[3];

    const phx_qconv_desc* conv() const { return static_cast<const phx_qconv_desc*>(abi); }
    const phx_qdense_desc* den() const { return static_cast<const phx_qdense_desc*>(abi); }
};
void desc_dealloc(PyObject* self) {
    Desc* d = reinterpret_cast<Desc*>(self);
    for (PyObject* f : d->fields) Py_XDECREF(f);
    d->in.~vector(); d->filter.~vector(); d->out.~vector(); d->bias_shape.~vector();
    Py_TYPE(self)->tp_free(self);
}
PyTypeObject DescType = {PyVarObject_HEAD_INIT(nullptr, 0)};

bool to_sizes(PyObject* tuple, std::vector<int64_t>& v) {
    if (!tuple || !PyTuple_Check(tuple)) return false;
    v.clear();
    for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(tuple); ++i) {
        const long long e = PyLong_AsLongLong(PyTuple_GET_ITEM(tuple, i));
        if (e == -1 && PyErr_Occurred()) { PyErr_Clear(); return false; }
        v.push_back(e);
    }
    return true;
}

long tuning_generation() {
    PyObject* g = PyDict_GetItem(g_capi_dict, N.tuning_generation);
    return g ? PyLong_AsLong(g) : -1;
}

// The kept part of a descriptor of the quaternion algebra, made (again) where there is none or a field is another object now;
// nullptr: a descriptor of another kind or type.
Desc* desc_of(PyObject* o, bool dense) {
    if (reinterpret_cast<PyObject*>(Py_TYPE(o)) != (dense ? g_dense_type : g_conv_type)) return nullptr;
    PyObject** dictptr = _PyObject_GetDictPtr(o);
    if (!dictptr || !*dictptr) return nullptr;
    PyObject* dict = *dictptr;
    PyObject* fields[DESC_FIELDS] = {PyDict_GetItem(dict, N.c),     PyDict_GetItem(dict, N.input_shape), PyDict_GetItem(dict, N.filter_shape), PyDict_GetItem(dict, N.output_shape),
                                     PyDict_GetItem(dict, N.dtype), PyDict_GetItem(dict, N.use_bias),    PyDict_GetItem(dict, N.bias_shape),   PyDict_GetItem(dict, N.real_valued_input)};
    PyObject* held = PyDict_GetItem(dict, N._host);
    if (held && Py_TYPE(held) == &DescType) {
        Desc* d = reinterpret_cast<Desc*>(held);
        if (d->dense == dense && std::memcmp(d->fields, fields, sizeof(fields)) == 0) return d;
    }
    PyObject* algebra = PyDict_GetItem(dict, N.algebra);
    for (int i = 0; i <= FIELD_USE_BIAS; ++i)
        if (!fields[i]) return nullptr;
    if (!algebra || !PyLong_Check(algebra) || PyLong_AsLong(algebra) != 2 /* ops.QUATERNION */ || !THPDtype_Check(fields[FIELD_DTYPE])) return nullptr;
    Py_buffer view;
    if (PyObject_GetBuffer(fields[FIELD_C], &view, PyBUF_SIMPLE) != 0) { PyErr_Clear(); return nullptr; }
    const void* abi = view.buf;
    const bool size_ok = (size_t)view.len == (dense ? sizeof(phx_qdense_desc) : sizeof(phx_qconv_desc));
    PyBuffer_Release(&view);  // (the structure owns its memory as long as it lives, and this holds it)
    if (!size_ok) return nullptr;
    Desc* d = reinterpret_cast<Desc*>(DescType.tp_alloc(&DescType, 0));
    if (!d) { PyErr_Clear(); return nullptr; }
    new (&d->in) std::vector<int64_t>; new (&d->filter) std::vector<int64_t>; new (&d->out) std::vector<int64_t>; new (&d->bias_shape) std::vector<int64_t>;
    for (int i = 0; i < DESC_FIELDS; ++i) { Py_XINCREF(fields[i]); d->fields[i] = fields[i]; }
    d->abi = abi;
    d->dense = dense;
    d->bias = PyObject_IsTrue(fields[FIELD_USE_BIAS]) == 1;
    d->real = fields[FIELD_REAL] && PyObject_IsTrue(fields[FIELD_REAL]) == 1;
    d->type = reinterpret_cast<THPDtype*>(fields[FIELD_DTYPE])->scalar_type;
    d->generation = -1;
    const bool good = to_sizes(fields[FIELD_INPUT], d->in) && to_sizes(fields[FIELD_FILTER], d->filter) && to_sizes(fields[FIELD_OUTPUT], d->out) &&
                      (!d->bias || to_sizes(fields[FIELD_BIAS_SHAPE], d->bias_shape)) && PyDict_SetItem(dict, N._host, reinterpret_cast<PyObject*>(d)) == 0;
    Py_DECREF(d);  // (the dictionary holds it)
    if (!good) { PyErr_Clear(); return nullptr; }
    return d;
}

size_t workspace_bytes(Desc* d, int pass) {
    const long generation = tuning_generation();
    const void* copy = d->dense ? static_cast<const void*>(&d->dense_copy) : &d->conv_copy;
    const size_t size = d->dense ? sizeof(d->dense_copy) : sizeof(d->conv_copy);
    if (d->generation != generation || std::memcmp(copy, d->abi, size) != 0) {
        std::memcpy(const_cast<void*>(copy), d->abi, size);
        d->generation = generation;
        d->known[0] = d->known[1] = d->known[2] = false;
    }
    if (!d->known[pass]) {
        d->workspace[pass] = d->dense ? L.phx_qdense_workspace_bytes(d->den(), pass) : L.phx_qconv2d_workspace_bytes(d->conv(), pass);
        d->known[pass] = true;
    }
    return d->workspace[pass];
}

at::Tensor result(const Desc* d, const std::vector<int64_t>& shape, c10::Device device) {
    return at::empty(shape, c10::TensorOptions().dtype(d->type).device(device));
}

// The image of `packed` (ops.PackedFilters) for a pass.  False: not for this descriptor, or not a plain tensor (the caller's
// Python code decides what that means); image nullptr: none for the pass.
bool packed_image(const Desc* d, PyObject* packed, bool fwd, const at::Tensor*& image) {
    image = nullptr;
    if (packed == Py_None) return true;
    PyObject** dictptr = _PyObject_GetDictPtr(packed);
    if (!dictptr || !*dictptr) return false;
    PyObject* o = PyDict_GetItem(*dictptr, fwd ? N.fwd : N.bwd_data);
    if (!o) return false;
    if (o == Py_None) return true;
    PyObject* key = PyDict_GetItem(*dictptr, N.layout_key);
    if (!key || !PyTuple_Check(key) || PyTuple_GET_SIZE(key) != 2 || !PyBytes_Check(PyTuple_GET_ITEM(key, 0)) || !PyLong_Check(PyTuple_GET_ITEM(key, 1))) return false;
    // (the descriptor's bytes without has_bias: ops._layout_key)
    constexpr size_t at = offsetof(phx_qconv_desc, has_bias), after = at + sizeof(int32_t);
    const char* bytes = PyBytes_AS_STRING(PyTuple_GET_ITEM(key, 0));
    const char* abi = static_cast<const char*>(d->abi);
    if ((size_t)PyBytes_GET_SIZE(PyTuple_GET_ITEM(key, 0)) != sizeof(phx_qconv_desc) - sizeof(int32_t) || std::memcmp(bytes, abi, at) != 0 ||
        std::memcmp(bytes + at, abi + after, sizeof(phx_qconv_desc) - after) != 0 || PyLong_AsLong(PyTuple_GET_ITEM(key, 1)) != tuning_generation())
        return false;
    image = plain(o);
    return image != nullptr && image->scalar_type() == c10::kByte;
}

// bias (where the descriptor has one); false: not a plain call
bool bias_of(const Desc* d, PyObject* o, c10::Device device, const at::Tensor*& bias) {
    bias = nullptr;
    if (!d->bias) return o == Py_None;
    return !d->real && (bias = plain(o, d->bias_shape, d->type, device)) != nullptr;
}

#define PHX_ARGS(n) if (nargs != n) { PyErr_SetString(PyExc_TypeError, "wrong number of arguments"); return nullptr; }

// conv_fwd(desc, x, w, bias, out, packed)
PyObject* conv_fwd(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    PHX_ARGS(6)
    Desc* d = no_modes() ? desc_of(a[0], false) : nullptr;
    const at::Tensor* x = d ? plain(a[1]) : nullptr;
    if (!x || x->scalar_type() != d->type || x->sizes() != c10::IntArrayRef(d->in)) return plain_no();
    const c10::Device device = x->device();
    const at::Tensor *w = plain(a[2], d->filter, d->type, device), *bias, *image;
    if (!w || !bias_of(d, a[3], device, bias) || !packed_image(d, a[5], true, image)) return plain_no();
    at::Tensor y;
    if (a[4] != Py_None) {
        const at::Tensor* out = plain(a[4], d->out, d->type, device);
        if (!out) return plain_no();
        y = *out;
    } else {
        y = result(d, d->out, device);
    }
    const size_t bytes = workspace_bytes(d, PHX_PASS_FWD);
    const uintptr_t stream = current_stream(device);
    const at::Tensor ws = scratch(device, stream, bytes);
    const phx_stream_t st = reinterpret_cast<phx_stream_t>(stream);
    const phx_qconv_desc c = *d->conv();
    void *px = address(x), *pw = address(w), *pb = address(bias), *pi = address(image), *py = y.data_ptr(), *pws = ws.data_ptr();
    const size_t ni = bytes_of(image);
    const int status = unlocked([&] {
        return pi ? L.phx_qconv2d_fwd_prepacked(&c, st, px, pi, ni, pb, py, pws, bytes) : L.phx_qconv2d_fwd(&c, st, px, pw, pb, py, pws, bytes);
    });
    if (!ok(status, image ? "phx_qconv2d_fwd_prepacked" : "phx_qconv2d_fwd")) return nullptr;
    if (a[4] != Py_None) { Py_INCREF(a[4]); return a[4]; }
    return THPVariable_Wrap(std::move(y));
    END_HANDLE_TH_ERRORS
}

// conv_bwd_weights(desc, x, grad, stream handle or None)
PyObject* conv_bwd_weights(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    PHX_ARGS(4)
    Desc* d = no_modes() ? desc_of(a[0], false) : nullptr;
    const at::Tensor* x = d ? plain(a[1]) : nullptr;
    if (!x || x->scalar_type() != d->type || x->sizes() != c10::IntArrayRef(d->in)) return plain_no();
    const c10::Device device = x->device();
    const at::Tensor* g = plain(a[2], d->out, d->type, device);
    if (!g) return plain_no();
    const uintptr_t stream = a[3] == Py_None ? current_stream(device) : (uintptr_t)PyLong_AsUnsignedLongLong(a[3]);
    if (PyErr_Occurred()) return nullptr;
    at::Tensor dw = result(d, d->filter, device);
    const size_t bytes = workspace_bytes(d, PHX_PASS_BWD_WEIGHTS);
    const at::Tensor ws = scratch(device, stream, bytes);
    const phx_qconv_desc c = *d->conv();
    void *px = address(x), *pg = address(g), *pdw = dw.data_ptr(), *pws = ws.data_ptr();
    const int status = unlocked([&] { return L.phx_qconv2d_bwd_weights(&c, reinterpret_cast<phx_stream_t>(stream), px, pg, pdw, pws, bytes); });
    return ok(status, "phx_qconv2d_bwd_weights") ? THPVariable_Wrap(std::move(dw)) : nullptr;
    END_HANDLE_TH_ERRORS
}

// conv_bwd_data(desc, w, grad, packed, addend)
PyObject* conv_bwd_data(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    PHX_ARGS(5)
    Desc* d = no_modes() ? desc_of(a[0], false) : nullptr;
    const at::Tensor* w = d && !d->real ? plain(a[1]) : nullptr;
    if (!w || w->scalar_type() != d->type || w->sizes() != c10::IntArrayRef(d->filter)) return plain_no();
    const c10::Device device = w->device();
    const at::Tensor *g = plain(a[2], d->out, d->type, device), *image, *addend = nullptr;
    if (!g || !packed_image(d, a[3], false, image) || (a[4] != Py_None && !(addend = plain(a[4], d->in, d->type, device)))) return plain_no();
    at::Tensor dx = result(d, d->in, device);
    const size_t bytes = workspace_bytes(d, PHX_PASS_BWD_DATA);
    const uintptr_t stream = current_stream(device);
    const at::Tensor ws = scratch(device, stream, bytes);
    const phx_stream_t st = reinterpret_cast<phx_stream_t>(stream);
    const phx_qconv_desc c = *d->conv();
    void *pg = address(g), *pw = address(w), *pi = address(image), *pa = address(addend), *pdx = dx.data_ptr(), *pws = ws.data_ptr();
    const size_t ni = bytes_of(image);
    const int status = unlocked([&] {
        return pa   ? L.phx_qconv2d_bwd_data_add(&c, st, pg, pw, pi, ni, pa, pdx, pws, bytes)
               : pi ? L.phx_qconv2d_bwd_data_prepacked(&c, st, pg, pi, ni, pdx, pws, bytes)
                    : L.phx_qconv2d_bwd_data(&c, st, pg, pw, pdx, pws, bytes);
    });
    return ok(status, addend ? "phx_qconv2d_bwd_data_add" : image ? "phx_qconv2d_bwd_data_prepacked" : "phx_qconv2d_bwd_data") ? THPVariable_Wrap(std::move(dx)) : nullptr;
    END_HANDLE_TH_ERRORS
}

// conv_pack(desc, w, packed): packs again into the images of `packed`
PyObject* conv_pack(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    PHX_ARGS(3)
    Desc* d = no_modes() ? desc_of(a[0], false) : nullptr;
    const at::Tensor* w = d ? plain(a[1]) : nullptr;
    const at::Tensor *f, *b;
    if (!w || w->scalar_type() != d->type || w->sizes() != c10::IntArrayRef(d->filter) || a[2] == Py_None || !packed_image(d, a[2], true, f) ||
        !packed_image(d, a[2], false, b) || (!f && !b))
        return plain_no();
    const phx_stream_t st = reinterpret_cast<phx_stream_t>(current_stream(w->device()));
    const phx_qconv_desc c = *d->conv();
    void *pw = address(w), *pf = address(f), *pb = address(b);
    const size_t nf = bytes_of(f), nb = bytes_of(b);
    const int status = unlocked([&] { return L.phx_qconv2d_pack_filters(&c, st, pw, pf, nf, pb, nb); });
    if (!ok(status, "phx_qconv2d_pack_filters")) return nullptr;
    Py_INCREF(a[2]);
    return a[2];
    END_HANDLE_TH_ERRORS
}

// dense_fwd(desc, x, w, bias, out)
PyObject* dense_fwd(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    PHX_ARGS(5)
    Desc* d = no_modes() ? desc_of(a[0], true) : nullptr;
    const at::Tensor* x = d ? plain(a[1]) : nullptr;
    if (!x || x->scalar_type() != d->type || x->sizes() != c10::IntArrayRef(d->in)) return plain_no();
    const c10::Device device = x->device();
    const at::Tensor *w = plain(a[2], d->filter, d->type, device), *bias;
    if (!w || !bias_of(d, a[3], device, bias)) return plain_no();
    at::Tensor y;
    if (a[4] != Py_None) {
        const at::Tensor* out = plain(a[4], d->out, d->type, device);
        if (!out) return plain_no();
        y = *out;
    } else {
        y = result(d, d->out, device);
    }
    const size_t bytes = workspace_bytes(d, PHX_PASS_FWD);
    const uintptr_t stream = current_stream(device);
    const at::Tensor ws = scratch(device, stream, bytes);
    const phx_qdense_desc c = *d->den();
    void *px = address(x), *pw = address(w), *pb = address(bias), *py = y.data_ptr(), *pws = ws.data_ptr();
    const int status = unlocked([&] { return L.phx_qdense_fwd(&c, reinterpret_cast<phx_stream_t>(stream), px, pw, pb, py, pws, bytes); });
    if (!ok(status, "phx_qdense_fwd")) return nullptr;
    if (a[4] != Py_None) { Py_INCREF(a[4]); return a[4]; }
    return THPVariable_Wrap(std::move(y));
    END_HANDLE_TH_ERRORS
}

// conv_bwd / dense_bwd(desc, x, w, grad, whether dx is asked for) -> (dw, dx or None)
template <bool DENSE>
PyObject* both_gradients(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    PHX_ARGS(5)
    Desc* d = no_modes() ? desc_of(a[0], DENSE) : nullptr;
    const at::Tensor* x = d ? plain(a[1]) : nullptr;
    if (!x || x->scalar_type() != d->type || x->sizes() != c10::IntArrayRef(d->in)) return plain_no();
    const c10::Device device = x->device();
    const at::Tensor *w = plain(a[2], d->filter, d->type, device), *g = plain(a[3], d->out, d->type, device);
    const int want = PyObject_IsTrue(a[4]);
    if (want < 0) return nullptr;
    if (!w || !g || (want && d->real)) return plain_no();
    const uintptr_t stream = current_stream(device);
    const phx_stream_t st = reinterpret_cast<phx_stream_t>(stream);
    at::Tensor dw = result(d, d->filter, device), dx;
    if (want) dx = result(d, d->in, device);
    const size_t weights_bytes = workspace_bytes(d, PHX_PASS_BWD_WEIGHTS), data_bytes = want ? workspace_bytes(d, PHX_PASS_BWD_DATA) : 0;
    const at::Tensor ws = scratch(device, stream, std::max(weights_bytes, data_bytes));
    void *px = address(x), *pw = address(w), *pg = address(g), *pdw = dw.data_ptr(), *pdx = want ? dx.data_ptr() : nullptr, *pws = ws.data_ptr();
    int status;
    if constexpr (DENSE) {
        const phx_qdense_desc c = *d->den();
        status = unlocked([&] {
            return pdx ? L.phx_qdense_bwd(&c, st, px, pw, pg, pdw, pdx, pws, std::max(weights_bytes, data_bytes))
                       : L.phx_qdense_bwd_weights(&c, st, px, pg, pdw, pws, weights_bytes);
        });
        if (!ok(status, pdx ? "phx_qdense_bwd" : "phx_qdense_bwd_weights")) return nullptr;
    } else {
        const phx_qconv_desc c = *d->conv();
        bool weights = true;  // (which of the two a status is of)
        status = unlocked([&] {
            const int s = L.phx_qconv2d_bwd_weights(&c, st, px, pg, pdw, pws, weights_bytes);
            if (s != PHX_OK || !pdx) return s;
            weights = false;
            return L.phx_qconv2d_bwd_data(&c, st, pg, pw, pdx, pws, data_bytes);
        });
        if (!ok(status, weights ? "phx_qconv2d_bwd_weights" : "phx_qconv2d_bwd_data")) return nullptr;
    }
    PyObject* po = THPVariable_Wrap(std::move(dw));
    PyObject* pi = want ? THPVariable_Wrap(std::move(dx)) : (Py_INCREF(Py_None), Py_None);
    PyObject* both = po && pi ? PyTuple_Pack(2, po, pi) : nullptr;
    Py_XDECREF(po); Py_XDECREF(pi);
    return both;
    END_HANDLE_TH_ERRORS
}

// ---- batch norm in training ----
bool bn_desc_of(const at::Tensor* x, PyObject* eps, PyObject* momentum, PyObject* relu, phx_bn_desc& b) {
    if (x->dim() < 2 || (x->scalar_type() != c10::kHalf && x->scalar_type() != c10::kFloat) || x->numel() == 0) return false;
    const int64_t rows = x->size(0), c = x->size(1), hw = x->numel() / (rows * c);
    if (rows >= INT32_MAX || c >= INT32_MAX || hw >= INT32_MAX) return false;
    const double e = PyFloat_AsDouble(eps), m = momentum ? PyFloat_AsDouble(momentum) : 0.0;
    const int r = PyObject_IsTrue(relu);
    if (PyErr_Occurred() || r < 0) { PyErr_Clear(); return false; }
    b = phx_bn_desc{x->scalar_type() == c10::kHalf ? PHX_F16 : PHX_F32, (int32_t)rows, (int32_t)c, (int32_t)hw, (float)e, (float)m, r};
    return true;
}

// bn_fwd(x, gamma, beta, running_mean, running_var, eps, momentum, relu, residual) -> (y, mean, invstd)
PyObject* bn_fwd(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    PHX_ARGS(9)
    const at::Tensor* x = no_modes() ? plain(a[0]) : nullptr;
    phx_bn_desc b;
    if (!x || !bn_desc_of(x, a[5], a[6], a[7], b)) return plain_no();
    const c10::Device device = x->device();
    const int64_t c = b.c;
    const at::Tensor* own[4];
    for (int i = 0; i < 4; ++i)
        if (!(own[i] = plain(a[1 + i], {c}, c10::kFloat, device))) return plain_no();
    const at::Tensor* res = nullptr;
    if (a[8] != Py_None && !(res = plain(a[8], x->sizes(), x->scalar_type(), device))) return plain_no();
    const auto params = c10::TensorOptions().dtype(c10::kFloat).device(device);
    at::Tensor y = at::empty(x->sizes(), x->options()), mean = at::empty({c}, params), invstd = at::empty({c}, params);
    const size_t bytes = L.phx_bn_workspace_bytes(&b);
    const uintptr_t stream = current_stream(device);
    const at::Tensor ws = scratch(device, stream, bytes);
    float* po[4];
    for (int i = 0; i < 4; ++i) po[i] = static_cast<float*>(own[i]->data_ptr());
    float *pmean = static_cast<float*>(mean.data_ptr()), *pinv = static_cast<float*>(invstd.data_ptr());
    void *px = address(x), *pr = address(res), *pout = y.data_ptr(), *pws = ws.data_ptr();
    const int status = unlocked([&] { return L.phx_bn_fwd_train(&b, reinterpret_cast<phx_stream_t>(stream), px, pr, po[0], po[1], pout, pmean, pinv, po[2], po[3], pws, bytes); });
    if (!ok(status, "phx_bn_fwd_train")) return nullptr;
    PyObject *py = THPVariable_Wrap(std::move(y)), *pm = THPVariable_Wrap(std::move(mean)), *pi = THPVariable_Wrap(std::move(invstd));
    PyObject* all = py && pm && pi ? PyTuple_Pack(3, py, pm, pi) : nullptr;
    Py_XDECREF(py); Py_XDECREF(pm); Py_XDECREF(pi);
    return all;
    END_HANDLE_TH_ERRORS
}

// bn_bwd(x, dy, gamma, beta, mean, invstd, eps, relu, residual) -> (dx, dgamma, dbeta, dresidual or None)
PyObject* bn_bwd(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    PHX_ARGS(9)
    const at::Tensor* x = no_modes() ? plain(a[0]) : nullptr;
    phx_bn_desc b;
    if (!x || !bn_desc_of(x, a[6], nullptr, a[7], b)) return plain_no();
    const c10::Device device = x->device();
    const int64_t c = b.c;
    const at::Tensor *dy = plain(a[1], x->sizes(), x->scalar_type(), device), *res = nullptr, *own[4];
    if (!dy) return plain_no();
    for (int i = 0; i < 4; ++i)
        if (!(own[i] = plain(a[2 + i], {c}, c10::kFloat, device))) return plain_no();
    if (a[8] != Py_None && !(res = plain(a[8], x->sizes(), x->scalar_type(), device))) return plain_no();
    const auto params = c10::TensorOptions().dtype(c10::kFloat).device(device);
    at::Tensor dx = at::empty(x->sizes(), x->options()), dres, dgamma = at::empty({c}, params), dbeta = at::empty({c}, params);
    if (res) dres = at::empty(x->sizes(), x->options());
    const size_t bytes = L.phx_bn_workspace_bytes(&b);
    const uintptr_t stream = current_stream(device);
    const at::Tensor ws = scratch(device, stream, bytes);
    const float* po[4];
    for (int i = 0; i < 4; ++i) po[i] = static_cast<const float*>(own[i]->data_ptr());
    float *pgamma = static_cast<float*>(dgamma.data_ptr()), *pbeta = static_cast<float*>(dbeta.data_ptr());
    void *p0 = address(x), *p1 = address(res), *p2 = address(dy), *p3 = dx.data_ptr(), *p4 = res ? dres.data_ptr() : nullptr, *pws = ws.data_ptr();
    const int status = unlocked([&] { return L.phx_bn_bwd(&b, reinterpret_cast<phx_stream_t>(stream), p0, p1, p2, po[0], po[1], po[2], po[3], p3, p4, pgamma, pbeta, pws, bytes); });
    if (!ok(status, "phx_bn_bwd")) return nullptr;
    PyObject *px = THPVariable_Wrap(std::move(dx)), *pg = THPVariable_Wrap(std::move(dgamma)), *pb = THPVariable_Wrap(std::move(dbeta)),
             *pr = res ? THPVariable_Wrap(std::move(dres)) : (Py_INCREF(Py_None), Py_None);
    PyObject* all = px && pg && pb && pr ? PyTuple_Pack(4, px, pg, pb, pr) : nullptr;
    Py_XDECREF(px); Py_XDECREF(pg); Py_XDECREF(pb); Py_XDECREF(pr);
    return all;
    END_HANDLE_TH_ERRORS
}

// ---- a convolution and the evaluation-mode norm behind it, by their modules (nn._conv_norm) ----
bool empty_dict(PyObject* dict, PyObject* name) {
    PyObject* d = PyDict_GetItem(dict, name);
    return d && PyDict_Check(d) && PyDict_GET_SIZE(d) == 0;
}
bool unhooked(PyObject* dict) {
    return empty_dict(dict, N._forward_hooks) && empty_dict(dict, N._forward_pre_hooks) && empty_dict(dict, N._backward_hooks) &&
           empty_dict(dict, N._backward_pre_hooks) && !PyDict_GetItem(dict, N.forward);
}
PyObject* member(PyObject* dict, PyObject* table, PyObject* name) {
    PyObject* t = PyDict_GetItem(dict, table);
    return t && PyDict_Check(t) ? PyDict_GetItem(t, name) : nullptr;
}
bool is_plain_tensor_type(PyObject* o) { return Py_TYPE(o) == reinterpret_cast<PyTypeObject*>(THPVariableClass); }

// conv_norm(vars(conv), vars(norm), x, residual or None): the modules' types and the process-wide hooks are the caller's to check.
// NotImplemented as well where the convolution has not met this shape yet, its filter has changed, or the stream is captured.
PyObject* conv_norm(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    PHX_ARGS(4)
    PyObject *conv = a[0], *norm = a[1];
    if (!PyDict_Check(conv) || !PyDict_Check(norm) || !no_modes() || c10::GradMode::is_enabled() || c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::Tracer) ||
        c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::FuncTorchDynamicLayerFrontMode))
        return plain_no();
    PyObject* level = PyDict_GetItem(g_forward_ad, N._current_level);
    if (!level || PyLong_AsLong(level) >= 0) { PyErr_Clear(); return plain_no(); }
    const at::Tensor* x = is_plain_tensor_type(a[2]) ? plain(a[2]) : nullptr;
    if (!x || x->dim() != 4 || !unhooked(conv) || !unhooked(norm) || PyDict_GetItem(norm, N.training) != Py_False ||
        PyDict_GetItem(conv, N._pack_pending) != Py_False)
        return plain_no();
    // (the keys of _descs and _packed: (shape, dtype))
    PyObject* shape = PyTuple_New(4);
    PyObject* key = PyTuple_New(2);
    if (!shape || !key) { Py_XDECREF(shape); Py_XDECREF(key); return nullptr; }
    for (int i = 0; i < 4; ++i) PyTuple_SET_ITEM(shape, i, PyLong_FromLongLong(x->size(i)));
    PyObject* dtype = reinterpret_cast<PyObject*>(torch::getTHPDtype(x->scalar_type()));
    Py_INCREF(dtype);
    PyTuple_SET_ITEM(key, 0, shape);
    PyTuple_SET_ITEM(key, 1, dtype);
    PyObject* pair = member(conv, N._descs, key);
    PyObject* entry = member(conv, N._packed, key);
    Py_DECREF(key);
    if (PyErr_Occurred()) PyErr_Clear();
    if (!pair || !PyTuple_Check(pair) || PyTuple_GET_SIZE(pair) != 2 || !entry || !PyList_Check(entry) || PyList_GET_SIZE(entry) != 2) return plain_no();
    Desc* d = desc_of(PyTuple_GET_ITEM(pair, 0), false);
    if (!d || d->type != x->scalar_type() || x->sizes() != c10::IntArrayRef(d->in) || d->out.size() != 4 || d->conv()->data_format != PHX_NCHW) return plain_no();
    const c10::Device device = x->device();
    const int64_t c = d->out[1], plane = d->out[2] * d->out[3], rows = d->out[0], count = rows * c * plane;
    if (count <= 0 || count >= std::min<int64_t>((int64_t)rows * c << 30, (int64_t)1 << 34) || rows >= INT32_MAX) return plain_no();
    PyObject* wo = member(conv, N._parameters, N.weight);
    const at::Tensor* w = wo && reinterpret_cast<PyObject*>(Py_TYPE(wo)) == g_parameter ? plain(wo, d->filter, d->type, device) : nullptr;
    PyObject* bo = member(conv, N._parameters, N.bias);
    const at::Tensor *bias, *image;
    if (!w || (bo && bo != Py_None && reinterpret_cast<PyObject*>(Py_TYPE(bo)) != g_parameter) || !bias_of(d, bo ? bo : Py_None, device, bias)) return plain_no();
    // the packed image is of this state of the filter
    PyObject* state = PyList_GET_ITEM(entry, 0);
    PyObject* packed = PyList_GET_ITEM(entry, 1);
    if (packed != Py_None) {
        if (!PyTuple_Check(state) || PyTuple_GET_SIZE(state) != 2 || PyLong_AsLongLong(PyTuple_GET_ITEM(state, 0)) != (long long)w->_version() ||
            (uintptr_t)PyLong_AsUnsignedLongLong(PyTuple_GET_ITEM(state, 1)) != reinterpret_cast<uintptr_t>(w->data_ptr())) {
            PyErr_Clear();
            return plain_no();
        }
        if (captured(current_stream(device))) return plain_no();
    }
    if (!packed_image(d, packed, true, image)) return plain_no();
    PyObject* own_o[4] = {member(norm, N._parameters, N.weight), member(norm, N._parameters, N.bias), member(norm, N._buffers, N.running_mean), member(norm, N._buffers, N.running_var)};
    const at::Tensor* own[4];
    for (int i = 0; i < 4; ++i)
        if (!own_o[i] || !(own[i] = plain(own_o[i])) || own[i]->scalar_type() != c10::kFloat || own[i]->device() != device || own[i]->numel() != c) return plain_no();
    const at::Tensor* res = nullptr;
    PyObject* relu_o = PyDict_GetItem(norm, N.relu);
    PyObject* eps_o = PyDict_GetItem(norm, N.eps);
    const int relu = relu_o ? PyObject_IsTrue(relu_o) : -1;
    if (relu < 0 || !eps_o || !PyFloat_Check(eps_o)) { PyErr_Clear(); return plain_no(); }
    if (a[3] != Py_None && (!relu || !is_plain_tensor_type(a[3]) || !(res = plain(a[3], d->out, d->type, device)))) return plain_no();
    const auto f = [](const at::Tensor* t) { return static_cast<const float*>(t->data_ptr()); };
    const phx_output_norm n{f(own[0]), f(own[1]), f(own[2]), f(own[3]), address(res), (float)PyFloat_AS_DOUBLE(eps_o), relu};
    at::Tensor y = result(d, d->out, device);
    const size_t bytes = workspace_bytes(d, PHX_PASS_FWD);
    const uintptr_t stream = current_stream(device);
    const at::Tensor ws = scratch(device, stream, bytes);
    const phx_qconv_desc cd = *d->conv();
    void *px = address(x), *pw = address(w), *pi = address(image), *pb = address(bias), *py = y.data_ptr(), *pws = ws.data_ptr();
    const size_t ni = bytes_of(image);
    const int status = unlocked([&] { return L.phx_qconv2d_fwd_norm(&cd, reinterpret_cast<phx_stream_t>(stream), px, pw, pi, ni, pb, &n, py, pws, bytes); });
    return ok(status, "phx_qconv2d_fwd_norm") ? THPVariable_Wrap(std::move(y)) : nullptr;
    END_HANDLE_TH_ERRORS
}

// workspace(device index, stream handle, bytes, whether for a capture to come) -> the stream's scratch buffer, grown to at least
// that; memory of the capture's own under one (see scratch)
PyObject* workspace(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    PHX_ARGS(4)
    const long device = PyLong_AsLong(a[0]);
    const uintptr_t stream = (uintptr_t)PyLong_AsUnsignedLongLong(a[1]);
    const size_t bytes = (size_t)PyLong_AsUnsignedLongLong(a[2]);
    const int reserve = PyObject_IsTrue(a[3]);
    if (PyErr_Occurred()) return nullptr;
    return THPVariable_Wrap(scratch(c10::Device(c10::DeviceType::CUDA, (c10::DeviceIndex)device), stream, bytes, reserve == 1));
    END_HANDLE_TH_ERRORS
}

// workspace_holds(device index, stream handle, bytes): whether that buffer is there and as large already
PyObject* workspace_holds(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
    PHX_ARGS(3)
    const long device = PyLong_AsLong(a[0]);
    const uintptr_t stream = (uintptr_t)PyLong_AsUnsignedLongLong(a[1]);
    const size_t bytes = (size_t)PyLong_AsUnsignedLongLong(a[2]);
    if (PyErr_Occurred()) return nullptr;
    const auto it = buffers().find({(int)device, stream});
    return PyBool_FromLong(it != buffers().end() && holds(it->second, bytes));
}

// bind(addresses of the C ABI by name, capi's namespace, capi.check, torch.nn.Parameter, forward_ad's namespace, the descriptors' types)
PyObject* bind(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
    PHX_ARGS(7)
#define PHX_FIELD(f)                                                                                         \
    {                                                                                                        \
        PyObject* p = PyDict_GetItemString(a[0], #f);                                                        \
        if (!p) { PyErr_SetString(PyExc_KeyError, #f); return nullptr; }                                     \
        L.f = reinterpret_cast<decltype(L.f)>(PyLong_AsVoidPtr(p));                                          \
        if (PyErr_Occurred()) return nullptr;                                                                \
    }
    PHX_HOST_FUNCTIONS(PHX_FIELD)
#undef PHX_FIELD
    PyObject** kept[6] = {&g_capi_dict, &g_check, &g_parameter, &g_forward_ad, &g_conv_type, &g_dense_type};
    for (int i = 0; i < 6; ++i) { Py_INCREF(a[1 + i]); Py_XDECREF(*kept[i]); *kept[i] = a[1 + i]; }
    Py_RETURN_NONE;
}

#define PHX_METHOD_AS(name, f) {name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(&f)), METH_FASTCALL, nullptr}
#define PHX_METHOD(f) {#f, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(&f)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {PHX_METHOD(bind), PHX_METHOD(conv_fwd), PHX_METHOD(conv_bwd_weights), PHX_METHOD(conv_bwd_data), PHX_METHOD(conv_pack),
                         PHX_METHOD(dense_fwd), PHX_METHOD_AS("conv_bwd", both_gradients<false>), PHX_METHOD_AS("dense_bwd", both_gradients<true>),
                         PHX_METHOD(bn_fwd), PHX_METHOD(bn_bwd), PHX_METHOD(conv_norm),
                         PHX_METHOD(workspace), PHX_METHOD(workspace_holds), {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_phx_host", nullptr, -1, methods};

}  // namespace

PyMODINIT_FUNC PyInit__phx_host(void) {
#define PHX_FIELD(n) if (!(N.n = PyUnicode_InternFromString(#n))) return nullptr;
    PHX_HOST_NAMES(PHX_FIELD)
#undef PHX_FIELD
    DescType.tp_name = "_phx_host.Desc";
    DescType.tp_basicsize = sizeof(Desc);
    DescType.tp_flags = Py_TPFLAGS_DEFAULT;
    DescType.tp_dealloc = desc_dealloc;
    if (PyType_Ready(&DescType) < 0) return nullptr;
    return PyModule_Create(&module);
}
