// bsipytorch_amd._native: the host path of an eager call, in C++.
//
// A small layer's forward is bound by the host: reading the layer's and the keyset's attributes, checking the operands,
// allocating the output and entering the C ABI through ctypes took 13 us of Python for 4 us of GPU work.  The functions
// here do the same for the default configuration on the objects the Python code keeps -- they read the layer's and the
// handles' attributes on every call, so nothing can go stale -- and return None for any call they do not serve; the Python
// path behind them then serves it or raises its errors.  Launches recorded into a graph always take that path.
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/jit/frontend/tracer.h>
#include <torch/version.h>
#include <ATen/EmptyTensor.h>
#include <ATen/ops/zeros.h>
#include <ATen/hip/EmptyTensor.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPGraphsC10Utils.h>
#include <c10/hip/HIPStream.h>

#include <chrono>
#include <cstring>
#include <map>

#include "../../include/bsi_hip.h"

extern char** environ;

namespace {

// Entry points of the library the Python side has loaded (bind()).
struct Library {
    decltype(&bsi_hip_linear_few_rows_out) linear_few_rows_out;
    decltype(&bsi_hip_linear_few_rows_shares) linear_few_rows_shares;
    decltype(&bsi_hip_linear_out) linear_out;
    decltype(&bsi_hip_linear_workspace_bytes_for) linear_workspace_bytes_for;
    decltype(&bsi_hip_dot) dot;
    decltype(&bsi_hip_build_fixed) build_fixed;
    decltype(&bsi_hip_build_fixed_keys) build_fixed_keys;
    decltype(&bsi_hip_ewah_measure) ewah_measure;
    decltype(&bsi_hip_ewah_emit) ewah_emit;
    decltype(&bsi_hip_dot_ewah_batch) dot_ewah_batch;
    decltype(&bsi_hip_dot_ewah_batch_workspace_bytes) dot_ewah_batch_workspace_bytes;
    decltype(&bsi_hip_linear_coop_out) linear_coop_out;
    decltype(&bsi_hip_linear_coop_serves) linear_coop_serves;
    decltype(&bsi_hip_linear_coop_bytes) linear_coop_bytes;
    decltype(&bsi_hip_scalar_query_dot) scalar_query_dot;
    decltype(&bsi_hip_build_measure_rows) build_measure_rows;
    decltype(&bsi_hip_ewah_emit_at) ewah_emit_at;
    decltype(&bsi_hip_scalar_query_host_words) scalar_query_host_words;
} lib;

// The Python side's state (bind()): types of the handles, the workspaces and what is known about shapes.
struct Shared {
    PyObject *keys_type, *batch_type, *hybrid_type;  // PrebuiltBSIKeysCUDA, PrebuiltBSIQueryBatchCUDA, ...HybridCUDA
    PyObject *linear_ws;                   // device index -> {"bytes", "eager": {stream: (buffer, [key, input])}, ...}
    PyObject *reserved, *warmed;           // shapes whose workspace and constants a later capture will find
    PyObject *split_shapes, *attach;       // (device, Q, R, W) -> whether the dot splits; attach_split_scratch
    PyObject *check;                       // raises for a library status
    int few_rows_max, stream_max, split_min;
    int64_t few_rows_lds;
} shared;

// The flags of the process (configure()); off until they have been read, and for configurations the Python path serves.
struct Config {
    bool on = false;
    int bits = 0, core = 0;
    int64_t generation = 0;
} config;

// nn.Module and the layer class as layer_call compares them (bind_layer()).
struct Module {
    PyObject *type, *base, *forward, *call, *global_hooks[4];
} module;

#define NAMES(X)                                                                                                          \
    X(_bsi_keys_cuda) X(_fused) X(_next_bsi_layer) X(_buffers) X(bias) X(collect_stats) X(decimalPlaces) X(fixed) X(Sb) X(W) X(d) \
    X(num_keys) X(decimals) X(layout) X(words) X(ints8) X(ints8_tiled) X(slice_weights) X(bytes) X(eager) X(dot_calls)      \
    X(build_calls) X(dot_query_vectors_total) X(dot_output_elements_total) X(chunk_scales) X(row_scales) X(keys) \
    X(comp_words) X(comp_off) X(comp_len) X(Sa) X(Q) X(forward) X(__call__) X(_compiled_call_impl) X(_forward_hooks)          \
    X(_forward_pre_hooks) X(_backward_hooks) X(_backward_pre_hooks)
struct Names {
#define X(n) PyObject* n;
    NAMES(X)
#undef X
} names;

// The switches that are read on every call, with the value at which they change nothing.
bool switches_at_default() {
    static const struct { const char* name; size_t len; const char* value; } kSwitches[] = {
        {"BSI_TC_DOT=", 11, "1"}, {"BSI_QUERY_FP32=", 15, "0"}, {"BSI_FUSED_LINEAR=", 17, "1"},
        {"BSI_LINEAR_ONE_CALL=", 20, "1"}, {"BSI_QUERY_PACKED=", 17, "1"}, {"BSI_QUERY_CACHE=", 16, "1"}};
    for (char** e = environ; e && *e; ++e) {
        if ((*e)[0] != 'B' || (*e)[1] != 'S' || (*e)[2] != 'I' || (*e)[3] != '_') continue;
        for (const auto& s : kSwitches)
            if (std::strncmp(*e, s.name, s.len) == 0 && std::strcmp(*e + s.len, s.value) != 0) return false;
    }
    return true;
}

// Borrowed reference to dict[name], or nullptr (no error left behind).
PyObject* get(PyObject* dict, PyObject* name) { return PyDict_GetItem(dict, name); }
bool get_int(PyObject* dict, PyObject* name, int64_t* v) {
    PyObject* o = get(dict, name);
    if (o == nullptr || !PyLong_Check(o)) return false;
    *v = PyLong_AsLongLong(o);
    return true;
}
const at::Tensor* get_tensor(PyObject* dict, PyObject* name) {
    PyObject* o = get(dict, name);
    return o != nullptr && THPVariable_Check(o) ? &THPVariable_Unpack(o) : nullptr;
}
void count(PyObject* dict, PyObject* name, int64_t by) {
    int64_t v = 0;
    if (!get_int(dict, name, &v)) return;
    if (PyObject* n = PyLong_FromLongLong(v + by)) {
        PyDict_SetItem(dict, name, n);
        Py_DECREF(n);
    }
}

struct Holder {  // an owned reference
    PyObject* p;
    explicit Holder(PyObject* o = nullptr) : p(o) {}
    ~Holder() { Py_XDECREF(p); }
    Holder(const Holder&) = delete;
    Holder& operator=(const Holder&) = delete;
};

// The null stream cannot be captured; asking about another one takes 0.4 us.
bool capturing(hipStream_t st) {
    if (st == nullptr) return false;
    hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
    return hipStreamIsCapturing(st, &status) != hipSuccess || status != hipStreamCaptureStatusNone;
}
hipStream_t stream_of(const at::Device& device) { return c10::hip::getCurrentHIPStream(device.index()).stream(); }

int dtype_code(at::ScalarType t) {
    switch (t) {
        case at::kFloat: return BSI_DTYPE_F32;
        case at::kHalf: return BSI_DTYPE_F16;
        case at::kBFloat16: return BSI_DTYPE_BF16;
        default: return -1;
    }
}

// What a launch reads of a tensor: address and storage, taken under the interpreter lock.  A tensor found in a Python
// dictionary is only borrowed: once the lock is released (or Python code is called), another thread can put something else in
// its place, or other data into it.
struct Operand {
    c10::Storage storage;
    const void* data = nullptr;
    size_t bytes = 0;
    Operand() = default;
    explicit Operand(const at::Tensor& t) : storage(t.storage()), data(t.const_data_ptr()), bytes(t.nbytes()) {}
    template <typename T>
    const T* as() const { return static_cast<const T*>(data); }
};

// A fixed-bit keyset's attributes as a dot of Q rows needs them.
struct Keys {
    int64_t Sb, W, d, R, decimals;
    int layout, operand_layout;  // of the planes, of `operand`
    bool image;                  // there is an int8 image
    Operand operand, weights;    // operand: planes or image (bsi_ops.key_operand)
};
bool read_keys(PyObject* handle, const at::Device& device, int64_t Q, Keys* k) {
    if (handle == nullptr || reinterpret_cast<PyObject*>(Py_TYPE(handle)) != shared.keys_type) return false;
    Holder attrs(PyObject_GenericGetDict(handle, nullptr));
    if (attrs.p == nullptr) {
        PyErr_Clear();
        return false;
    }
    int64_t layout = 0;
    if (get(attrs.p, names.fixed) != Py_True || !get_int(attrs.p, names.Sb, &k->Sb) || !get_int(attrs.p, names.W, &k->W) ||
        !get_int(attrs.p, names.d, &k->d) || !get_int(attrs.p, names.num_keys, &k->R) ||
        !get_int(attrs.p, names.decimals, &k->decimals) || !get_int(attrs.p, names.layout, &layout))
        return false;
    const at::Tensor* const words = get_tensor(attrs.p, names.words);
    const at::Tensor* const ints8 = get_tensor(attrs.p, names.ints8);
    const at::Tensor* const weights = get_tensor(attrs.p, names.slice_weights);
    if (words == nullptr || weights == nullptr || words->device() != device || weights->device() != device || !weights->is_contiguous() ||
        k->R <= 0 || k->Sb < 2 || k->Sb > 8)
        return false;
    k->layout = k->operand_layout = static_cast<int>(layout);
    k->image = ints8 != nullptr;
    k->weights = Operand(*weights);
    (void)weights->const_data_ptr<float>();  // raises for another type
    const bool use_image = k->image && Q > shared.stream_max;
    k->operand = Operand(use_image ? *ints8 : *words);
    if (use_image) k->operand_layout = get(attrs.p, names.ints8_tiled) == Py_True ? BSI_LAYOUT_INT8_TILED : BSI_LAYOUT_INT8;
    return true;
}

PyObject* int_tuple(std::initializer_list<int64_t> values) {
    PyObject* t = PyTuple_New(static_cast<Py_ssize_t>(values.size()));
    Py_ssize_t i = 0;
    if (t != nullptr)
        for (int64_t v : values) PyTuple_SET_ITEM(t, i++, PyLong_FromLongLong(v));
    return t;
}
bool in_set(PyObject* set, std::initializer_list<int64_t> values) {
    Holder t(int_tuple(values));
    return t.p != nullptr && PySet_Contains(set, t.p) == 1;
}

// Whether a later capture of a few-rows layer will find its workspace and constants (made by the Python side's first call of
// the shape).  The answers of the last shapes are kept: they stay true until the flags are read again.
bool known_few_rows(int device, int64_t rows, int64_t d) {
    struct Known {
        int64_t device, rows, d, generation;
    };
    static Known known[8] = {};
    Known& k = known[(d / 64 + rows + device) & 7];
    if (k.device == device && k.rows == rows && k.d == d && k.generation == config.generation) return true;
    if (!in_set(shared.reserved, {device, rows, d, config.bits}) || !in_set(shared.warmed, {rows, config.bits, device})) return false;
    k = Known{device, rows, d, config.generation};
    return true;
}

// Attaches the split scratch if the launcher splits a dot of this shape; false: the Python side has to find out first.
bool split_scratch(int device, int64_t Q, int64_t R, int64_t W) {
    if (Q < shared.split_min) return true;
    Holder t(int_tuple({device, Q, R, W}));
    PyObject* use = t.p != nullptr ? PyDict_GetItem(shared.split_shapes, t.p) : nullptr;
    if (use == nullptr) return false;
    if (use == Py_True) {
        Holder r(PyObject_CallNoArgs(shared.attach));
        if (r.p == nullptr) {
            PyErr_Clear();
            return false;
        }
    }
    return true;
}

PyObject* fail_status(int rc, const char* what) {
    Holder r(PyObject_CallFunction(shared.check, "is", rc, what));  // raises
    if (r.p != nullptr) PyErr_Format(PyExc_RuntimeError, "%s failed (code %d)", what, rc);
    return nullptr;
}

float scale_inv(int64_t dec_q, int64_t dec_k) {
    double p = 1.0;
    for (int64_t i = 0; i < dec_q + dec_k; ++i) p *= 10.0;
    return static_cast<float>(1.0 / p);
}

// What identifies the query build of a contiguous tensor for keys of Sb slices: its contents (address, shape, type,
// version) and what the build depends on (the generation stands for the process's flags); compared byte by byte.
struct BuildKey {
    const void* data;
    int64_t rows, d, version, generation;
    int32_t dtype, decimals, Sb, unused;
};
BuildKey build_key_of(const at::Tensor& x, int64_t d, int64_t decimals, int64_t Sb) {
    return BuildKey{x.const_data_ptr(), x.numel() / d, d, static_cast<int64_t>(x.unsafeGetTensorImpl()->version_counter().current_version()),
                    config.generation, dtype_code(x.scalar_type()), static_cast<int32_t>(decimals), static_cast<int32_t>(Sb), 0};
}

// build_key(x2d, decimals, Sb) -> bytes, or None for a tensor without a version counter (inference mode), whose contents
// cannot be tracked.
PyObject* build_key(PyObject*, PyObject* args) {
    PyObject* o = nullptr;
    long long decimals = 0, Sb = 0;
    if (!PyArg_ParseTuple(args, "OLL", &o, &decimals, &Sb)) return nullptr;
    HANDLE_TH_ERRORS
    if (!THPVariable_Check(o)) return PyErr_Format(PyExc_TypeError, "build_key: not a tensor");
    const at::Tensor& x = THPVariable_Unpack(o);
    if (x.is_inference() || x.dim() < 1 || x.numel() == 0) Py_RETURN_NONE;
    const BuildKey key = build_key_of(x, x.size(-1), decimals, Sb);
    return PyBytes_FromStringAndSize(reinterpret_cast<const char*>(&key), sizeof(key));
    END_HANDLE_TH_ERRORS
}

// The keys of the layer that runs next (set by quantize_model_bsi), touched by this dot's kernel; nullptr: none.
const void* keys_to_warm(PyObject* layer, int64_t rows, const at::Device& device, size_t* bytes) {
    PyObject* const next = rows > shared.stream_max ? get(layer, names._next_bsi_layer) : nullptr;
    if (next == nullptr || next == Py_None) return nullptr;
    Holder attrs(PyObject_GenericGetDict(next, nullptr));
    PyObject* handle = attrs.p != nullptr ? get(attrs.p, names._bsi_keys_cuda) : nullptr;
    Holder group_keys;
    if (PyObject* g = attrs.p != nullptr ? get(attrs.p, names._fused) : nullptr; g != nullptr && PyTuple_Check(g)) {
        group_keys.p = PyObject_GetAttr(PyTuple_GET_ITEM(g, 0), names.keys);
        handle = group_keys.p;
    }
    PyErr_Clear();
    Keys k;
    if (!read_keys(handle, device, rows, &k)) return nullptr;
    *bytes = k.operand.bytes;
    return k.operand.data;
}

// The areas of launches with the query build inside (2.1 MB each), one for each stream that has made one.  A stream without an
// area takes the ones that no launch has used for kCoopIdle launches back and gets one if fewer than kCoopAreas are left;
// otherwise its layers are two launches, so that streams in turn do not clear an area a call.  forget() gives all back.  An area
// is allocated under its stream, so the allocator reuses it behind the launches on it.  Under the interpreter lock.
constexpr size_t kCoopAreas = 32;
constexpr uint64_t kCoopIdle = 4096;
struct CoopArea {
    at::Tensor memory;
    uint64_t last;  // the last launch that used it
};
auto& coop_areas = *new std::map<std::pair<int, hipStream_t>, CoopArea>;  // never destroyed: the runtime may be gone by then
uint64_t coop_launches = 0;
at::Tensor coop_area(const at::Device& device, hipStream_t st) {
    const std::pair<int, hipStream_t> key(device.index(), st);
    auto found = coop_areas.find(key);
    if (found == coop_areas.end()) {
        for (auto it = coop_areas.begin(); it != coop_areas.end();)
            it = coop_launches - it->second.last > kCoopIdle ? coop_areas.erase(it) : std::next(it);
        if (coop_areas.size() >= kCoopAreas) return at::Tensor();
        at::Tensor memory = at::zeros({static_cast<int64_t>(lib.linear_coop_bytes())}, at::TensorOptions().dtype(at::kByte).device(device));
        found = coop_areas.emplace(key, CoopArea{std::move(memory), 0}).first;
    }
    found->second.last = coop_launches;
    return found->second.memory;
}
PyObject* forget(PyObject*, PyObject*) {
    coop_areas.clear();
    Py_RETURN_NONE;
}

// A Python object that owns a storage.
PyObject* hold(const c10::Storage& storage) {
    return PyCapsule_New(new c10::Storage(storage), nullptr,
                         [](PyObject* o) { delete static_cast<c10::Storage*>(PyCapsule_GetPointer(o, nullptr)); });
}

// linear(layer.__dict__, x) -> the layer's output, or None.
PyObject* linear(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
    if (nargs != 2 || !PyDict_Check(args[0])) {
        PyErr_SetString(PyExc_TypeError, "linear(layer.__dict__, x)");
        return nullptr;
    }
    Holder layer_dict(Py_NewRef(args[0]));
    PyObject* const layer = layer_dict.p;
    if (!config.on || !THPVariable_CheckExact(args[1]) || !switches_at_default()) Py_RETURN_NONE;
    if (PyObject* o = get(layer, names._fused); o != nullptr && o != Py_None) Py_RETURN_NONE;
    if (get(layer, names.collect_stats) != Py_False) Py_RETURN_NONE;
    HANDLE_TH_ERRORS
    at::Tensor x = THPVariable_Unpack(args[1]);
    const int in_code = dtype_code(x.scalar_type());
    if (!x.is_cuda() || x.layout() != at::kStrided || in_code < 0 || x.dim() < 1 || x.numel() == 0) Py_RETURN_NONE;
    const at::Device device = x.device();
    if (device.index() != c10::hip::current_device()) Py_RETURN_NONE;
    const int64_t d = x.size(-1), rows = x.numel() / d;
    Keys k;
    int64_t decimals = 0;
    if (!read_keys(get(layer, names._bsi_keys_cuda), device, rows, &k) || !get_int(layer, names.decimalPlaces, &decimals) ||
        decimals != k.decimals || decimals < 0 || d != k.d)
        Py_RETURN_NONE;
    const int64_t chunks = (k.W + 3) / 4;
    PyObject* const buffers = get(layer, names._buffers);
    if (buffers == nullptr || !PyDict_Check(buffers)) Py_RETURN_NONE;
    Operand bias;
    // A layer without a bias has the buffer, None.  Without the buffer, or with an instance attribute in front of it, self.bias
    // is something else: a parameter, a parametrization.
    PyObject* const bias_object = get(buffers, names.bias);
    if (bias_object == nullptr || get(layer, names.bias) != nullptr) Py_RETURN_NONE;
    if (PyObject* o = bias_object; o != Py_None) {
        if (!THPVariable_Check(o)) Py_RETURN_NONE;
        const at::Tensor& b = THPVariable_Unpack(o);
        if (b.device() != device || b.scalar_type() != at::kFloat || b.dim() != 1 || b.numel() != k.R || !b.is_contiguous())
            Py_RETURN_NONE;
        bias = Operand(b);
    }
    // half-precision output: the kernels that have it (bsi_ops.can_output_half)
    const bool six_tiled = k.Sb == 6 && k.layout == BSI_LAYOUT_TILED16;
    if (in_code != BSI_DTYPE_F32 && !(rows > shared.stream_max ? k.image : six_tiled && chunks <= 32768)) Py_RETURN_NONE;
    hipStream_t const st = stream_of(device);
    if (capturing(st)) Py_RETURN_NONE;

    const bool few = rows <= shared.few_rows_max && six_tiled && k.W % 4 == 0 && chunks * rows * 260 <= shared.few_rows_lds;
    Holder mine;  // the stream's (buffer, slot)
    PyObject* slot = nullptr;
    void* ws = nullptr;
    int64_t ws_bytes = 0;
    const bool own_build = few && lib.linear_few_rows_shares(rows, d, k.R) == 0;
    const at::Tensor coop = !own_build && k.Sb <= 8 && lib.linear_coop_serves(rows, d, k.R, static_cast<int>(decimals), config.bits, k.operand_layout, static_cast<int>(k.Sb))
                           ? coop_area(device, st) : at::Tensor();
    if (few) {
        if (!known_few_rows(device.index(), rows, d)) Py_RETURN_NONE;
    } else {
        Holder index(PyLong_FromLong(device.index()));
        PyObject* record = PyDict_GetItem(shared.linear_ws, index.p);
        if (record == nullptr || !get_int(record, names.bytes, &ws_bytes) ||
            static_cast<size_t>(ws_bytes) <
                lib.linear_workspace_bytes_for(rows, d, config.bits, k.operand_layout, static_cast<int>(k.Sb), k.R, config.core))
            Py_RETURN_NONE;
        if (!coop.defined()) {
            Holder handle(PyLong_FromVoidPtr(st));
            PyObject* const eager = get(record, names.eager);
            mine.p = Py_XNewRef(eager != nullptr ? PyDict_GetItem(eager, handle.p) : nullptr);
            if (mine.p == nullptr || !PyTuple_Check(mine.p) || PyTuple_GET_SIZE(mine.p) != 2 || !THPVariable_Check(PyTuple_GET_ITEM(mine.p, 0)))
                Py_RETURN_NONE;
            ws = THPVariable_Unpack(PyTuple_GET_ITEM(mine.p, 0)).data_ptr();
            slot = PyTuple_GET_ITEM(mine.p, 1);
            if (!PyList_Check(slot) || PyList_GET_SIZE(slot) != 2 || !split_scratch(device.index(), rows, k.R, k.W)) Py_RETURN_NONE;
        }
    }

    if (x.requires_grad()) x = x.detach();
    if (!x.is_contiguous()) x = x.contiguous();
    c10::SmallVector<int64_t, 5> sizes(x.sizes().begin(), x.sizes().end());
    sizes.back() = k.R;
    at::Tensor out = at::detail::empty_cuda(sizes, x.scalar_type(), device, std::nullopt);
    const float inv = scale_inv(decimals, k.decimals);
    const Operand xo(x);
    const void* const xp = xo.data;
    int rc = BSI_OK;
    if (coop.defined()) {
        size_t warm_bytes = 0;
        const void* const warm = keys_to_warm(layer, rows, device, &warm_bytes);
        // under the interpreter lock: launches on an area are in the order of their numbers
        rc = lib.linear_coop_out(xp, in_code, rows, d, static_cast<int>(decimals), config.bits, ++coop_launches, coop.data_ptr(),
                                 k.operand.as<uint64_t>(), k.operand_layout, k.weights.as<float>(), static_cast<int>(k.Sb),
                                 k.R, inv, k.R, bias.as<float>(), out.data_ptr(), in_code, warm, warm_bytes, st);
        if (rc != BSI_OK) return fail_status(rc, "bsi_hip_linear_coop_out");
        if (!few) count(layer, names.build_calls, 1);
    } else if (few) {
        Py_BEGIN_ALLOW_THREADS
        rc = lib.linear_few_rows_out(xp, in_code, rows, d, static_cast<int>(decimals), config.bits,
                                     k.operand.as<uint64_t>(), k.weights.as<float>(), static_cast<int>(k.Sb), k.R, inv, k.R,
                                     bias.as<float>(), out.data_ptr(), in_code, st);
        Py_END_ALLOW_THREADS
        if (rc != BSI_OK) return fail_status(rc, "bsi_hip_linear_few_rows_out");
    } else {
        size_t warm_bytes = 0;
        const void* const warm = keys_to_warm(layer, rows, device, &warm_bytes);
        // a call on the tensor the workspace was last built from skips the build, as in bsi_ops.linear_cuda
        int rebuild = 1;
        Holder key, held;
        if (!x.is_inference()) {
            const BuildKey now = build_key_of(x, d, decimals, k.Sb);
            PyObject* const last = PyList_GET_ITEM(slot, 0);
            if (PyBytes_CheckExact(last) && PyBytes_GET_SIZE(last) == sizeof(now) && std::memcmp(PyBytes_AS_STRING(last), &now, sizeof(now)) == 0) {
                rebuild = 0;
            } else {
                key.p = PyBytes_FromStringAndSize(reinterpret_cast<const char*>(&now), sizeof(now));
                // The storage is held, not the caller's tensor (x.data = other keeps the object and its version and frees the
                // storage): the address is not reused while the build stands for it.
                held.p = hold(xo.storage);
                if (key.p == nullptr || held.p == nullptr) return nullptr;
            }
        }
        if (rebuild != 0) PyList_SetItem(slot, 0, Py_NewRef(Py_None));  // until the build is enqueued
        // under the interpreter lock: another thread must not enqueue a build of its own between the two launches
        rc = lib.linear_out(xp, in_code, rows, d, static_cast<int>(decimals), config.bits, rebuild, ws, static_cast<size_t>(ws_bytes),
                            k.operand.as<uint64_t>(), k.operand_layout, k.weights.as<float>(), static_cast<int>(k.Sb),
                            k.R, inv, k.R, bias.as<float>(), out.data_ptr(), in_code, config.core, warm, warm_bytes, st);
        if (rc != BSI_OK) return fail_status(rc, "bsi_hip_linear_out");
        if (rebuild != 0 && key.p != nullptr) {
            PyList_SetItem(slot, 0, Py_NewRef(key.p));
            PyList_SetItem(slot, 1, Py_NewRef(held.p));
        }
        count(layer, names.build_calls, rebuild);
    }
    count(layer, names.dot_calls, 1);
    count(layer, names.dot_query_vectors_total, rows);
    count(layer, names.dot_output_elements_total, rows * k.R);
    return THPVariable_Wrap(std::move(out));
    END_HANDLE_TH_ERRORS
}

// Whether nn.Module.__call__ would do nothing but call the class's own forward.
bool plain_call(PyObject* self) {
    static PyObject* const kHooks[] = {names._forward_hooks, names._forward_pre_hooks, names._backward_hooks, names._backward_pre_hooks};
    PyTypeObject* const type = Py_TYPE(self);
    if (module.base == nullptr || reinterpret_cast<PyObject*>(type) != module.type || _PyType_Lookup(type, names.forward) != module.forward ||
        _PyType_Lookup(reinterpret_cast<PyTypeObject*>(module.base), names.__call__) != module.call || torch::jit::tracer::isTracing())
        return false;
    // a profiler or debugger of Python frames sees a module by its __call__ and forward
    if (const PyThreadState* const thread = PyThreadState_Get(); thread->c_profilefunc != nullptr || thread->c_tracefunc != nullptr) return false;
    for (PyObject* hooks : module.global_hooks)
        if (PyDict_GET_SIZE(hooks) != 0) return false;
    PyObject** const slot = _PyObject_GetDictPtr(self);
    PyObject* const attrs = slot != nullptr ? *slot : nullptr;
    if (attrs == nullptr || get(attrs, names.forward) != nullptr) return false;
    if (PyObject* o = get(attrs, names._compiled_call_impl); o != nullptr && o != Py_None) return false;
    for (PyObject* name : kHooks) {
        PyObject* const hooks = get(attrs, name);
        if (hooks == nullptr || !PyDict_Check(hooks) || PyDict_GET_SIZE(hooks) != 0) return false;
    }
    return true;
}

// A layer's __call__: a plain call that linear() serves goes straight there (nn.Module.__call__ and the Python forward take
// 0.8 us, a sixth of a small layer's host time); any other is nn.Module's.
PyObject* layer_call(PyObject*, PyObject* const* args, Py_ssize_t nargs, PyObject* kwnames) {
    if (nargs == 2 && kwnames == nullptr && plain_call(args[0])) {
        PyObject* const call[] = {*_PyObject_GetDictPtr(args[0]), args[1]};
        PyObject* const out = linear(nullptr, call, 2);
        if (out != Py_None) return out;
        Py_DECREF(out);
    }
    if (module.base == nullptr) return PyErr_Format(PyExc_RuntimeError, "layer_call before bind_layer");
    Holder base_call(PyObject_GetAttr(module.base, names.__call__));
    return base_call.p != nullptr ? PyObject_Vectorcall(base_call.p, args, nargs, kwnames) : nullptr;
}

// bind_layer(type, nn.Module, global hook dicts): the class whose calls layer_call shortens.
PyObject* bind_layer(PyObject*, PyObject* args) {
    PyObject *type, *base, *hooks[4];
    if (!PyArg_ParseTuple(args, "O!O!(O!O!O!O!)", &PyType_Type, &type, &PyType_Type, &base, &PyDict_Type, &hooks[0], &PyDict_Type,
                          &hooks[1], &PyDict_Type, &hooks[2], &PyDict_Type, &hooks[3]))
        return nullptr;
    PyObject* const forward = _PyType_Lookup(reinterpret_cast<PyTypeObject*>(type), names.forward);
    PyObject* const call = _PyType_Lookup(reinterpret_cast<PyTypeObject*>(base), names.__call__);
    if (forward == nullptr || call == nullptr) return PyErr_Format(PyExc_TypeError, "bind_layer: no forward or no __call__");
    module.type = Py_NewRef(type);
    module.forward = Py_NewRef(forward);
    module.call = Py_NewRef(call);
    for (int i = 0; i < 4; ++i) module.global_hooks[i] = Py_NewRef(hooks[i]);
    module.base = Py_NewRef(base);
    Py_RETURN_NONE;
}

// dot(query_batch, keyset) -> the float32 scores, or None: the plain dot of a fixed-bit batch that carries its int8 image.
PyObject* dot(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
    if (nargs != 2) {
        PyErr_SetString(PyExc_TypeError, "dot(query_batch, keyset)");
        return nullptr;
    }
    if (!config.on || reinterpret_cast<PyObject*>(Py_TYPE(args[0])) != shared.batch_type || !switches_at_default()) Py_RETURN_NONE;
    HANDLE_TH_ERRORS
    Holder attrs(PyObject_GenericGetDict(args[0], nullptr));
    if (attrs.p == nullptr) return nullptr;
    const at::Tensor* const words = get_tensor(attrs.p, names.words);
    const at::Tensor* const weights = get_tensor(attrs.p, names.slice_weights);
    const at::Tensor* const ints8 = get_tensor(attrs.p, names.ints8);
    const at::Tensor* const chunk_scales = get_tensor(attrs.p, names.chunk_scales);
    const at::Tensor* const row_scales = get_tensor(attrs.p, names.row_scales);
    int64_t decimals = 0;
    if (get(attrs.p, names.fixed) != Py_True || words == nullptr || weights == nullptr || ints8 == nullptr || words->dim() != 3 ||
        weights->dim() != 2 || !weights->is_cuda() || !words->is_cuda() || !get_int(attrs.p, names.decimals, &decimals))
        Py_RETURN_NONE;
    const at::Device device = words->device();
    const int64_t Q = words->size(0), Sa = words->size(1), W = words->size(2), chunks = (W + 3) / 4;
    const bool chunked = chunk_scales != nullptr && chunk_scales->numel() > 0;
    const at::Tensor* const scales = chunked ? chunk_scales : row_scales;
    Keys k;
    if (device.index() != c10::hip::current_device() || !read_keys(args[1], device, Q, &k) || k.W != W || k.decimals != decimals ||
        decimals < 0 || Q <= 0 || Sa < 2 || Sa > 8 || weights->size(0) != Q || weights->size(1) != Sa || scales == nullptr ||
        scales->device() != device || scales->scalar_type() != at::kFloat || !scales->is_contiguous() || ints8->device() != device ||
        !ints8->is_contiguous() || ints8->numel() != Q * chunks * 256 || !words->is_contiguous())
        Py_RETURN_NONE;
    if (chunked ? (scales->dim() != 2 || scales->size(0) != Q || W % 4 != 0 || scales->size(1) != chunks) : scales->numel() != Q)
        Py_RETURN_NONE;
    hipStream_t const st = stream_of(device);
    const Operand planes(*words), image(*ints8), factors(*scales);
    if (capturing(st) || !split_scratch(device.index(), Q, k.R, W)) Py_RETURN_NONE;
    at::Tensor out = at::detail::empty_cuda({Q, k.R}, at::kFloat, device, std::nullopt);
    int rc = BSI_OK;
    Py_BEGIN_ALLOW_THREADS
    rc = lib.dot(planes.as<uint64_t>(), image.as<int8_t>(), factors.as<float>(), chunked ? static_cast<int>(chunks) : 1,
                 static_cast<int>(Sa), static_cast<int>(W), k.operand.as<uint64_t>(), k.operand_layout, k.weights.as<float>(),
                 static_cast<int>(k.Sb), k.R, Q,
                 scale_inv(decimals, k.decimals), k.R, out.data_ptr<float>(), nullptr, config.core, nullptr, 0, st);
    Py_END_ALLOW_THREADS
    if (rc != BSI_OK) return fail_status(rc, "bsi_hip_dot");
    return THPVariable_Wrap(std::move(out));
    END_HANDLE_TH_ERRORS
}

// build(x, decimals, planes, image) -> (words [Q, bits, W] or None, chunk or row scales, int8 image or None), or None: the
// fixed-bit query build of a contiguous [Q, d] batch on the current device.
PyObject* build(PyObject*, PyObject* args) {
    PyObject* o = nullptr;
    int decimals = 0, planes = 0, image = 0;
    if (!PyArg_ParseTuple(args, "Oipp", &o, &decimals, &planes, &image)) return nullptr;
    if (!config.on || !THPVariable_CheckExact(o) || decimals < 0 || decimals > 2) Py_RETURN_NONE;
    HANDLE_TH_ERRORS
    const at::Tensor& x = THPVariable_Unpack(o);
    const int code = dtype_code(x.scalar_type());
    if (!x.is_cuda() || code < 0 || x.dim() != 2 || x.numel() == 0 || !x.is_contiguous() ||
        x.device().index() != c10::hip::current_device())
        Py_RETURN_NONE;
    const at::Device device = x.device();
    hipStream_t const st = stream_of(device);
    if (capturing(st)) Py_RETURN_NONE;
    const int64_t Q = x.size(0), d = x.size(1), W = (d + 63) / 64, chunks = (d + 255) / 256;
    const bool chunked = W % 4 == 0;
    at::Tensor words, ints8, scales;
    if (planes) words = at::detail::empty_cuda({Q, config.bits, W}, at::kLong, device, std::nullopt);
    if (image) ints8 = at::detail::empty_cuda({Q, chunks * 256}, at::kChar, device, std::nullopt);
    scales = chunked ? at::detail::empty_cuda({Q, chunks}, at::kFloat, device, std::nullopt)
                     : at::detail::empty_cuda({Q}, at::kFloat, device, std::nullopt);
    const Operand xo(x);
    int rc = BSI_OK;
    Py_BEGIN_ALLOW_THREADS
    rc = lib.build_fixed(xo.data, code, Q, d, decimals, config.bits, chunked ? 1 : 0, 0.0f,
                         planes ? static_cast<uint64_t*>(words.data_ptr()) : nullptr, nullptr, static_cast<float*>(scales.data_ptr()),
                         image ? static_cast<int8_t*>(ints8.data_ptr()) : nullptr, st);
    Py_END_ALLOW_THREADS
    if (rc != BSI_OK) return fail_status(rc, "bsi_hip_build_fixed");
    Holder w(THPVariable_Wrap(std::move(words))), s(THPVariable_Wrap(std::move(scales))), i(THPVariable_Wrap(std::move(ints8)));
    return PyTuple_Pack(3, w.p, s.p, i.p);
    END_HANDLE_TH_ERRORS
}

// build_keys(K, decimals, bits) -> (tiled planes, int8 image, shifts, slice weights, R, d), or None: the one-launch build of a
// contiguous key matrix on the current device.
PyObject* build_keys(PyObject*, PyObject* args) {
    PyObject* o = nullptr;
    int decimals = 0, bits = 0;
    if (!PyArg_ParseTuple(args, "Oii", &o, &decimals, &bits)) return nullptr;
    if (lib.build_fixed_keys == nullptr || bits < 2 || bits > 8 || decimals < 0 || decimals > 2 || !THPVariable_CheckExact(o)) Py_RETURN_NONE;
    HANDLE_TH_ERRORS
    const at::Tensor& x = THPVariable_Unpack(o);
    const int code = dtype_code(x.scalar_type());
    if (!x.is_cuda() || code < 0 || x.dim() != 2 || x.numel() == 0 || !x.is_contiguous() ||
        x.device().index() != c10::hip::current_device())
        Py_RETURN_NONE;
    const at::Device device = x.device();
    hipStream_t const st = stream_of(device);
    if (capturing(st)) Py_RETURN_NONE;
    const int64_t R = x.size(0), d = x.size(1), chunks = (d + 255) / 256;
    at::Tensor words = at::detail::empty_cuda({(R + 15) / 16, chunks, bits, 64}, at::kLong, device, std::nullopt);
    at::Tensor image = at::detail::empty_cuda({R, chunks * 256}, at::kChar, device, std::nullopt);
    at::Tensor shifts = at::detail::empty_cuda({R}, at::kInt, device, std::nullopt);
    at::Tensor weights = at::detail::empty_cuda({R, bits}, at::kFloat, device, std::nullopt);
    const Operand xo(x);
    int rc = BSI_OK;
    Py_BEGIN_ALLOW_THREADS
    rc = lib.build_fixed_keys(xo.data, code, R, d, decimals, bits, static_cast<uint64_t*>(words.data_ptr()),
                              static_cast<int8_t*>(image.data_ptr()), static_cast<int32_t*>(shifts.data_ptr()),
                              static_cast<float*>(weights.data_ptr()), st);
    Py_END_ALLOW_THREADS
    if (rc != BSI_OK) return fail_status(rc, "bsi_hip_build_fixed_keys");
    Holder w(THPVariable_Wrap(std::move(words))), i(THPVariable_Wrap(std::move(image))), s(THPVariable_Wrap(std::move(shifts))),
        f(THPVariable_Wrap(std::move(weights)));
    return Py_BuildValue("OOOOLL", w.p, i.p, s.p, f.p, static_cast<long long>(R), static_cast<long long>(d));
    END_HANDLE_TH_ERRORS
}

// ewah_streams(words [S, W], threshold) -> (stream words, offsets, lengths, flags) of the slices' EWAH encoding, or None.
PyObject* ewah_streams(PyObject*, PyObject* args) {
    PyObject* o = nullptr;
    double threshold = 0.0;
    if (!PyArg_ParseTuple(args, "Od", &o, &threshold)) return nullptr;
    if (lib.ewah_measure == nullptr || !THPVariable_CheckExact(o)) Py_RETURN_NONE;
    HANDLE_TH_ERRORS
    const at::Tensor& words = THPVariable_Unpack(o);
    if (!words.is_cuda() || words.scalar_type() != at::kLong || words.dim() != 2 || words.size(0) < 1 || words.size(0) > INT32_MAX ||
        words.size(1) > INT32_MAX || !words.is_contiguous() || words.device().index() != c10::hip::current_device())
        Py_RETURN_NONE;
    const at::Device device = words.device();
    const int S = static_cast<int>(words.size(0)), W = static_cast<int>(words.size(1));
    hipStream_t const st = stream_of(device);
    if (capturing(st)) Py_RETURN_NONE;
    at::Tensor flags = at::detail::empty_cuda({S}, at::kInt, device, std::nullopt);
    at::Tensor lens = at::detail::empty_cuda({S}, at::kInt, device, std::nullopt);
    at::Tensor off = at::detail::empty_cuda({S}, at::kLong, device, std::nullopt);
    at::Tensor total_host = at::detail::empty_cpu({1}, at::kLong, /*pin_memory=*/true);
    volatile int64_t* const total = static_cast<volatile int64_t*>(total_host.data_ptr());
    *total = -1;
    const Operand wo(words);
    const uint64_t* const w = wo.as<uint64_t>();
    int rc = BSI_OK;
    Py_BEGIN_ALLOW_THREADS
    rc = lib.ewah_measure(w, S, W, threshold, static_cast<int32_t*>(flags.data_ptr()), static_cast<int32_t*>(lens.data_ptr()),
                          static_cast<int64_t*>(off.data_ptr()), const_cast<int64_t*>(total), st);
    // the total arrives while its kernel still runs; the stream is waited for only if it is long in coming
    const auto until = std::chrono::steady_clock::now() + std::chrono::microseconds(200);
    while (rc == BSI_OK && *total < 0 && std::chrono::steady_clock::now() < until) {}
    if (rc == BSI_OK && *total < 0 && hipStreamSynchronize(st) != hipSuccess) rc = BSI_ERR_HIP;
    Py_END_ALLOW_THREADS
    if (rc != BSI_OK) return fail_status(rc, "bsi_hip_ewah_measure");
    at::Tensor streams = at::detail::empty_cuda({static_cast<int64_t>(*total)}, at::kLong, device, std::nullopt);
    if (streams.numel() > 0) {
        Py_BEGIN_ALLOW_THREADS
        rc = lib.ewah_emit(w, S, W, static_cast<const int32_t*>(flags.data_ptr()), static_cast<const uint64_t*>(off.data_ptr()),
                           static_cast<uint64_t*>(streams.data_ptr()), static_cast<int32_t*>(lens.data_ptr()), st);
        Py_END_ALLOW_THREADS
        if (rc != BSI_OK) return fail_status(rc, "bsi_hip_ewah_emit");
    }
    Holder a(THPVariable_Wrap(std::move(streams))), b(THPVariable_Wrap(std::move(off))), c(THPVariable_Wrap(std::move(lens))),
        f(THPVariable_Wrap(std::move(flags)));
    return PyTuple_Pack(4, a.p, b.p, c.p, f.p);
    END_HANDLE_TH_ERRORS
}

// hybrid(x, decimals, threshold) -> (stream words, offsets, lengths, flags, scales, slice weights or None), or None: the
// fixed-bit build of a contiguous [Q, d] batch on the current device, every slice EWAH-encoded.  The host waits for the
// lengths, which arrive a row at a time while the build's kernel still runs: their sum is the size of the streams.  (Emitting ahead of the lengths, into
// memory for the most a batch can need, takes 1 to 1.5 us off a pass of 64 x 2048 or 256 x 4096, adds 3 where the batch compresses and
// has to be emitted again, and the memory that is kept is up to a third more than the streams; not done.)
PyObject* hybrid(PyObject*, PyObject* args) {
    PyObject* o = nullptr;
    int decimals = 0;
    double threshold = 0.0;
    if (!PyArg_ParseTuple(args, "Oid", &o, &decimals, &threshold)) return nullptr;
    if (!config.on || !THPVariable_CheckExact(o) || decimals < 0 || decimals > 2) Py_RETURN_NONE;
    HANDLE_TH_ERRORS
    const at::Tensor& x = THPVariable_Unpack(o);
    const int code = dtype_code(x.scalar_type());
    if (!x.is_cuda() || code < 0 || x.dim() != 2 || x.numel() == 0 || !x.is_contiguous() || x.device().index() != c10::hip::current_device())
        Py_RETURN_NONE;
    const at::Device device = x.device();
    hipStream_t const st = stream_of(device);
    const int64_t Q = x.size(0), d = x.size(1), W = (d + 63) / 64, chunks = (d + 255) / 256, S = Q * config.bits;
    if (W > 1024 || S > 8192 || capturing(st)) Py_RETURN_NONE;  // bsi_hip_build_measure_rows's limits
    const bool chunked = W % 4 == 0;
    at::Tensor words = at::detail::empty_cuda({S, W}, at::kLong, device, std::nullopt);
    at::Tensor scales = chunked ? at::detail::empty_cuda({Q, chunks}, at::kFloat, device, std::nullopt)
                                : at::detail::empty_cuda({Q}, at::kFloat, device, std::nullopt);
    at::Tensor weights;
    if (!chunked) weights = at::detail::empty_cuda({Q, config.bits}, at::kFloat, device, std::nullopt);
    at::Tensor flags = at::detail::empty_cuda({S}, at::kInt, device, std::nullopt);
    at::Tensor lens = at::detail::empty_cuda({S}, at::kInt, device, std::nullopt);
    at::Tensor pinned = at::detail::empty_cpu({Q}, at::kInt, /*pin_memory=*/true);
    volatile int32_t* const host = static_cast<volatile int32_t*>(pinned.data_ptr());
    uint64_t* const w = static_cast<uint64_t*>(words.data_ptr());
    int64_t total = 0;
    for (int64_t q = 0; q < Q; ++q) host[q] = -1;
    int rc = lib.build_measure_rows(x.const_data_ptr(), code, Q, d, decimals, config.bits, chunked ? 1 : 0, threshold, w,
                           static_cast<float*>(scales.data_ptr()), chunked ? nullptr : static_cast<float*>(weights.data_ptr()),
                           static_cast<int32_t*>(flags.data_ptr()), static_cast<int32_t*>(lens.data_ptr()), const_cast<int32_t*>(host), st);
    if (rc != BSI_OK) return fail_status(rc, "bsi_hip_build_measure_rows");
    // The kernel writes into `pinned` until the last length is there: an allocation that fails before that waits for it.
    struct Writing {
        hipStream_t stream;
        bool done;
        ~Writing() {
            if (!done) (void)hipStreamSynchronize(stream);
        }
    } writing{st, false};
    // what can be made before the lengths are here
    at::Tensor off = at::detail::empty_cuda({S}, at::kLong, device, std::nullopt);
    Holder b(THPVariable_Wrap(off)), c(THPVariable_Wrap(lens)), f(THPVariable_Wrap(flags)), s(THPVariable_Wrap(std::move(scales))),
        v(THPVariable_Wrap(std::move(weights)));
    Py_BEGIN_ALLOW_THREADS
    // the stream is waited for only if the lengths are long in coming
    const auto until = std::chrono::steady_clock::now() + std::chrono::microseconds(500);
    bool waited = false;
    for (int64_t q = 0; q < Q && rc == BSI_OK; ++q) {
        while (host[q] < 0 && !waited)
            if (std::chrono::steady_clock::now() > until) {
                waited = true;
                if (hipStreamSynchronize(st) != hipSuccess) rc = BSI_ERR_HIP;
            }
        total += host[q];
    }
    Py_END_ALLOW_THREADS
    writing.done = true;
    if (rc != BSI_OK) return fail_status(rc, "bsi_hip_build_measure_rows");
    at::Tensor streams = at::detail::empty_cuda({total}, at::kLong, device, std::nullopt);
    rc = lib.ewah_emit_at(w, static_cast<int>(S), static_cast<int>(W), static_cast<const int32_t*>(flags.data_ptr()),
                          static_cast<const int32_t*>(lens.data_ptr()), static_cast<int64_t*>(off.data_ptr()),
                          static_cast<uint64_t*>(streams.data_ptr()), st);
    if (rc != BSI_OK) return fail_status(rc, "bsi_hip_ewah_emit_at");
    Holder a(THPVariable_Wrap(std::move(streams)));
    return PyTuple_Pack(6, a.p, b.p, c.p, f.p, s.p, v.p);
    END_HANDLE_TH_ERRORS
}

// dot_streams(hybrid_batch, keyset) -> the float32 scores, or None: the dot of a batch kept as EWAH streams.
PyObject* dot_streams(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
    if (nargs != 2) {
        PyErr_SetString(PyExc_TypeError, "dot_streams(hybrid_batch, keyset)");
        return nullptr;
    }
    if (!config.on || reinterpret_cast<PyObject*>(Py_TYPE(args[0])) != shared.hybrid_type) Py_RETURN_NONE;
    HANDLE_TH_ERRORS
    Holder attrs(PyObject_GenericGetDict(args[0], nullptr));
    if (attrs.p == nullptr) return nullptr;
    const at::Tensor* const streams = get_tensor(attrs.p, names.comp_words);
    const at::Tensor* const off = get_tensor(attrs.p, names.comp_off);
    const at::Tensor* const len = get_tensor(attrs.p, names.comp_len);
    const at::Tensor* const chunk_scales = get_tensor(attrs.p, names.chunk_scales);
    const at::Tensor* const row_scales = get_tensor(attrs.p, names.row_scales);
    const bool chunked = chunk_scales != nullptr && chunk_scales->numel() > 0;
    const at::Tensor* const scales = chunked ? chunk_scales : row_scales;
    int64_t Q = 0, Sa = 0, W = 0, decimals = 0;
    if (streams == nullptr || off == nullptr || len == nullptr || scales == nullptr || !get_int(attrs.p, names.Q, &Q) ||
        !get_int(attrs.p, names.Sa, &Sa) || !get_int(attrs.p, names.W, &W) || !get_int(attrs.p, names.decimals, &decimals))
        Py_RETURN_NONE;
    const at::Device device = streams->device();
    const int64_t chunks = (W + 3) / 4;
    Keys k;
    if (!streams->is_cuda() || device.index() != c10::hip::current_device() || !read_keys(args[1], device, Q, &k) || k.W != W ||
        k.decimals != decimals || decimals < 0 || Q <= 0 || Sa < 2 || Sa > 8 || off->numel() != Q * Sa || len->numel() != Q * Sa ||
        scales->device() != device || !scales->is_contiguous() || (chunked && W % 4 != 0) ||
        scales->numel() != (chunked ? Q * chunks : Q))
        Py_RETURN_NONE;
    hipStream_t const st = stream_of(device);
    const Operand so(*streams), oo(*off), lo(*len), factors(*scales);
    if (capturing(st) || !split_scratch(device.index(), Q, k.R, W)) Py_RETURN_NONE;
    at::Tensor out = at::detail::empty_cuda({Q, k.R}, at::kFloat, device, std::nullopt);
    const size_t need = lib.dot_ewah_batch_workspace_bytes(Q, static_cast<int>(W));
    at::Tensor ws = at::detail::empty_cuda({static_cast<int64_t>(need)}, at::kByte, device, std::nullopt);
    int rc = BSI_OK;
    Py_BEGIN_ALLOW_THREADS
    rc = lib.dot_ewah_batch(so.as<uint64_t>(), oo.as<int64_t>(), lo.as<int32_t>(), static_cast<int>(Sa), static_cast<int>(W),
                            factors.as<float>(), chunked ? static_cast<int>(chunks) : 1, k.operand.as<uint64_t>(), k.operand_layout,
                            k.weights.as<float>(), static_cast<int>(k.Sb), k.R, Q, scale_inv(decimals, k.decimals), k.R, nullptr,
                            static_cast<float*>(out.data_ptr()), nullptr, ws.data_ptr(), need, st);
    Py_END_ALLOW_THREADS
    if (rc != BSI_OK) return fail_status(rc, "bsi_hip_dot_ewah_batch");
    return THPVariable_Wrap(std::move(out));
    END_HANDLE_TH_ERRORS
}

// scalar_query(x, words [R, Sb, W], weights [R, Sb], decimals, threshold, divisor) -> (scores float64 [R] on the host, build
// ns, dot ns, words of the query's stored form), or None: one float32 vector on the current device against decimal keys.
PyObject* scalar_query(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
    if (nargs != 6) {
        PyErr_SetString(PyExc_TypeError, "scalar_query(x, words, weights, decimals, threshold, divisor)");
        return nullptr;
    }
    if (lib.scalar_query_dot == nullptr || !THPVariable_CheckExact(args[0]) || !THPVariable_Check(args[1]) || !THPVariable_Check(args[2])) Py_RETURN_NONE;
    const long decimals = PyLong_AsLong(args[3]);
    const double threshold = PyFloat_AsDouble(args[4]), divisor = PyFloat_AsDouble(args[5]);
    if (PyErr_Occurred()) return nullptr;
    HANDLE_TH_ERRORS
    const at::Tensor &x = THPVariable_Unpack(args[0]), &words = THPVariable_Unpack(args[1]), &weights = THPVariable_Unpack(args[2]);
    if (!x.is_cuda() || x.scalar_type() != at::kFloat || x.dim() != 1 || x.numel() == 0 || !x.is_contiguous() ||
        x.device().index() != c10::hip::current_device())
        Py_RETURN_NONE;
    const at::Device device = x.device();
    const int64_t d = x.size(0), W = (d + 63) / 64;
    if (words.device() != device || words.scalar_type() != at::kLong || words.dim() != 3 || words.size(2) != W || !words.is_contiguous() ||
        words.size(0) == 0 || weights.device() != device || weights.scalar_type() != at::kFloat || !weights.is_contiguous() ||
        weights.numel() != words.size(0) * words.size(1))
        Py_RETURN_NONE;
    hipStream_t const st = stream_of(device);
    if (capturing(st)) Py_RETURN_NONE;
    const int64_t R = words.size(0);
    at::Tensor out = at::detail::empty_cpu({R}, at::kDouble);
    at::Tensor pinned = at::detail::empty_cpu({lib.scalar_query_host_words(R)}, at::kLong, /*pin_memory=*/true);
    int64_t info[4] = {0, 0, 0, 0}, build_ns = 0, dot_ns = 0;
    const Operand xo(x), wo(words), fo(weights);
    const int slices = static_cast<int>(words.size(1));
    int rc = BSI_OK;
    Py_BEGIN_ALLOW_THREADS
    rc = lib.scalar_query_dot(xo.as<float>(), d, static_cast<int>(decimals), threshold, wo.as<uint64_t>(), fo.as<float>(), slices, R,
                              divisor, static_cast<uint64_t*>(pinned.data_ptr()), out.data_ptr<double>(), info, &build_ns, &dot_ns, st);
    Py_END_ALLOW_THREADS
    if (rc != BSI_OK) return fail_status(rc, "bsi_hip_scalar_query_dot");
    Holder scores(THPVariable_Wrap(std::move(out)));
    return Py_BuildValue("OLLL", scores.p, static_cast<long long>(build_ns), static_cast<long long>(dot_ns), static_cast<long long>(info[2]));
    END_HANDLE_TH_ERRORS
}

// configure(bits, core): the process's flags, or configure() to switch the native path off until they are read again.
PyObject* configure(PyObject*, PyObject* args) {
    int bits = 0, core = 0;
    if (!PyArg_ParseTuple(args, "|ii", &bits, &core)) return nullptr;
    config.on = bits != 0;
    config.bits = bits;
    config.core = core;
    ++config.generation;
    Py_RETURN_NONE;
}

bool take(PyObject* from, const char* name, PyObject** to) {
    PyObject* o = PyDict_GetItemString(from, name);
    if (o == nullptr) {
        PyErr_Format(PyExc_KeyError, "bind: %s", name);
        return false;
    }
    Py_INCREF(o);
    Py_XDECREF(*to);
    *to = o;
    return true;
}
template <typename F>
bool entry(PyObject* from, const char* name, F* to) {
    PyObject* o = PyDict_GetItemString(from, name);
    void* p = o != nullptr ? PyLong_AsVoidPtr(o) : nullptr;
    if (p == nullptr) {
        if (!PyErr_Occurred()) PyErr_Format(PyExc_KeyError, "bind: %s", name);
        return false;
    }
    *to = reinterpret_cast<F>(p);
    return true;
}

// bind(entry_points, state, limits): addresses of the library's functions, the Python side's objects, its constants.
PyObject* bind(PyObject*, PyObject* args) {
    PyObject *entries, *state;
    int few, stream, split;
    long long lds;
    if (!PyArg_ParseTuple(args, "O!O!iiiL", &PyDict_Type, &entries, &PyDict_Type, &state, &few, &stream, &split, &lds)) return nullptr;
    if (!entry(entries, "bsi_hip_linear_few_rows_out", &lib.linear_few_rows_out) ||
        !entry(entries, "bsi_hip_linear_few_rows_shares", &lib.linear_few_rows_shares) || !entry(entries, "bsi_hip_linear_out", &lib.linear_out) ||
        !entry(entries, "bsi_hip_linear_workspace_bytes_for", &lib.linear_workspace_bytes_for) || !entry(entries, "bsi_hip_dot", &lib.dot) ||
        !entry(entries, "bsi_hip_build_fixed", &lib.build_fixed) ||
        !entry(entries, "bsi_hip_build_fixed_keys", &lib.build_fixed_keys) || !entry(entries, "bsi_hip_ewah_measure", &lib.ewah_measure) ||
        !entry(entries, "bsi_hip_ewah_emit", &lib.ewah_emit) || !entry(entries, "bsi_hip_dot_ewah_batch", &lib.dot_ewah_batch) ||
        !entry(entries, "bsi_hip_dot_ewah_batch_workspace_bytes", &lib.dot_ewah_batch_workspace_bytes) ||
        !entry(entries, "bsi_hip_build_measure_rows", &lib.build_measure_rows) || !entry(entries, "bsi_hip_ewah_emit_at", &lib.ewah_emit_at) ||
        !entry(entries, "bsi_hip_linear_coop_out", &lib.linear_coop_out) ||
        !entry(entries, "bsi_hip_linear_coop_serves", &lib.linear_coop_serves) ||
        !entry(entries, "bsi_hip_linear_coop_bytes", &lib.linear_coop_bytes) ||
        !entry(entries, "bsi_hip_scalar_query_dot", &lib.scalar_query_dot) ||
        !entry(entries, "bsi_hip_scalar_query_host_words", &lib.scalar_query_host_words) ||
        !take(state, "keys_type", &shared.keys_type) || !take(state, "batch_type", &shared.batch_type) ||
        !take(state, "hybrid_type", &shared.hybrid_type) ||
        !take(state, "linear_ws", &shared.linear_ws) || !take(state, "reserved", &shared.reserved) ||
        !take(state, "warmed", &shared.warmed) || !take(state, "split_shapes", &shared.split_shapes) ||
        !take(state, "attach", &shared.attach) || !take(state, "check", &shared.check))
        return nullptr;
    shared.few_rows_max = few;
    shared.stream_max = stream;
    shared.split_min = split;
    shared.few_rows_lds = lds;
    Py_RETURN_NONE;
}

PyMethodDef methods[] = {
    {"bind", bind, METH_VARARGS, nullptr},
    {"configure", configure, METH_VARARGS, nullptr},
    {"build_key", build_key, METH_VARARGS, nullptr},
    {"build", build, METH_VARARGS, nullptr},
    {"build_keys", build_keys, METH_VARARGS, nullptr},
    {"hybrid", hybrid, METH_VARARGS, nullptr},
    {"ewah_streams", ewah_streams, METH_VARARGS, nullptr},
    {"dot_streams", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(dot_streams)), METH_FASTCALL, nullptr},
    {"linear", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(linear)), METH_FASTCALL, nullptr},
    {"scalar_query", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(scalar_query)), METH_FASTCALL, nullptr},
    {"forget", forget, METH_NOARGS, nullptr},
    {"bind_layer", bind_layer, METH_VARARGS, nullptr},
    {"layer_call", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(layer_call)), METH_FASTCALL | METH_KEYWORDS, nullptr},
    {"dot", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(dot)), METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef definition = {PyModuleDef_HEAD_INIT, "_native", "Host path of eager calls.", -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

// The functions reach into torch's own classes: another torch than the one they were compiled against is refused.
static bool torch_fits() {
    Holder torch(PyImport_ImportModule("torch"));
    Holder version(torch.p != nullptr ? PyObject_GetAttrString(torch.p, "__version__") : nullptr);
    const char* const have = version.p != nullptr && PyUnicode_Check(version.p) ? PyUnicode_AsUTF8(version.p) : nullptr;
    if (have == nullptr) {
        if (!PyErr_Occurred()) PyErr_SetString(PyExc_ImportError, "torch has no version");
        return false;
    }
    const size_t n = std::strlen(TORCH_VERSION);
    if (std::strncmp(have, TORCH_VERSION, n) == 0 && (have[n] == '\0' || have[n] == '+')) return true;
    PyErr_Format(PyExc_ImportError, "built for torch %s, this is %s", TORCH_VERSION, have);
    return false;
}

PyMODINIT_FUNC PyInit__native() {
    if (!torch_fits()) return nullptr;
#define X(n) names.n = PyUnicode_InternFromString(#n);
    NAMES(X)
#undef X
    PyObject* const m = PyModule_Create(&definition);
    // a builtin function does not bind to an instance: the class gets this form of it
    Holder call(m != nullptr ? PyObject_GetAttrString(m, "layer_call") : nullptr);
    Holder method(call.p != nullptr ? PyInstanceMethod_New(call.p) : nullptr);
    if (method.p == nullptr || PyModule_AddObjectRef(m, "layer_call", method.p) != 0) {
        Py_XDECREF(m);
        return nullptr;
    }
    return m;
}
