// The front end of vkop_amd.ops in native code: one Python call from torch tensors to the C ABI.
//
// Everything a call does before its kernels run -- checking the tensor, allocating the results,
// asking for the workspace's size, finding the stream, converting the shape -- took 9 us in Python
// and ctypes on top of the launches, several times the kernels of a small call.  softmax -> top-k
// of one classifier row (kernel 3.8 us): 13.6 us of host time a call, now 4.2, of which the launch
// is about 3; [64,128256] (two launches): 16.5, now 6.9, so that its kernels (14 us) bound it.
// Nothing is computed here and nothing kept between calls but the addresses of the C ABI's
// functions: bind() takes them from the library that vkop_amd.capi has loaded.
#include <Python.h>

#include <cstdarg>
#include <cstring>

#include <ATen/hip/EmptyTensor.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/version.h>

#include "vkop_hip.h"

namespace {

#define VKOP_NATIVE_FUNCTIONS(X)                                                                                       \
    X(last_error) X(softmax_workspace_bytes) X(softmax) X(topk_workspace_bytes) X(topk) X(softmax_topk_workspace_bytes) \
        X(softmax_topk) X(softmax_topk_sampling) X(reduce_max) X(softmax_reduce_max_workspace_bytes) X(softmax_reduce_max)
struct Functions {
#define VKOP_NATIVE_MEMBER(name) decltype(&vkop_hip_##name) name = nullptr;
    VKOP_NATIVE_FUNCTIONS(VKOP_NATIVE_MEMBER)
#undef VKOP_NATIVE_MEMBER
} fn;
PyObject *error_class = nullptr;                             // vkop_amd.capi.VkopHipError(code, message)
PyObject *workspace_class = nullptr;                         // vkop_amd.ops.Workspace
PyObject *name_ptr = nullptr, *name_size = nullptr, *name_get = nullptr;

// A failed Python call inside a function: unwinds to guarded(), which lets the exception set stand.
struct PythonError {};
[[noreturn]] void raise(PyObject *type, const char *fmt, ...) {
    va_list ap;
    va_start(ap, fmt);
    PyErr_FormatV(type, fmt, ap);
    va_end(ap);
    throw PythonError{};
}

// The tensor, its shape and element type as the C ABI takes them.
struct Input {
    at::Tensor x;
    const void *data = nullptr;
    int dtype = 0, ndim = 0, shape[4] = {0, 0, 0, 0};
    explicit Input(PyObject *o) {
        if (!THPVariable_Check(o) || !THPVariable_Unpack(o).is_cuda())
            raise(PyExc_TypeError, "expected a tensor on the GPU (there is no CPU path)");
        const at::Tensor &t = THPVariable_Unpack(o);
        if (t.scalar_type() == at::kFloat) dtype = VKOP_HIP_F32;
        else if (t.scalar_type() == at::kHalf) dtype = VKOP_HIP_F16;
        else {
            PyObject *name = PyObject_GetAttrString(o, "dtype");
            if (name != nullptr) {
                PyErr_Format(PyExc_TypeError, "float32 or float16 expected, got %S", name);
                Py_DECREF(name);
            }
            throw PythonError{};
        }
        if (t.dim() < 1 || t.dim() > 4) raise(PyExc_ValueError, "rank %d outside 1..4", static_cast<int>(t.dim()));
        x = t.is_contiguous() ? t : t.contiguous();
        ndim = static_cast<int>(x.dim());
        for (int d = 0; d < ndim; d++) shape[d] = static_cast<int>(x.size(d));
        data = x.data_ptr();
    }
    // position of `axis` in the shape, negative ones from its end
    int place(long axis) const {
        const long a = axis >= 0 ? axis : axis + ndim;
        if (a < -ndim || a >= ndim) raise(PyExc_IndexError, "axis %ld outside a tensor of rank %d", axis, ndim);
        return static_cast<int>(a >= 0 ? a : a + ndim);  // (what is still negative: refused by the C ABI)
    }
    at::Tensor empty(at::IntArrayRef sizes, at::ScalarType type) const {
        return at::Tensor(at::detail::empty_cuda(sizes, type, x.device(), std::nullopt));
    }
};

long as_long(PyObject *o) {
    PyObject *i = PyNumber_Index(o);  // (whole numbers, those of numpy and one-element tensors too; 2.5 or "2" is a TypeError)
    if (i == nullptr) throw PythonError{};
    const long v = PyLong_AsLong(i);
    Py_DECREF(i);
    if (v == -1 && PyErr_Occurred()) throw PythonError{};
    return v;
}
double as_double(PyObject *o) {
    PyObject *f = PyNumber_Float(o);
    if (f == nullptr) throw PythonError{};
    const double v = PyFloat_AS_DOUBLE(f);
    Py_DECREF(f);
    return v;
}
bool as_bool(PyObject *o) {
    const int v = PyObject_IsTrue(o);
    if (v < 0) throw PythonError{};
    return v != 0;
}

// Scratch memory of at least `need` bytes.  ops.Workspace: its two attributes say what it holds, and its get() is called
// only where that is too little.  Any other object, a class derived from it among them: whatever its get(need) returns.
struct Scratch {
    void *ptr = nullptr;
    size_t size = 0;
    Scratch(PyObject *workspace, size_t need) {
        if (reinterpret_cast<PyObject *>(Py_TYPE(workspace)) == workspace_class) {
            if (need == 0) return;
            size = attribute(workspace, name_size);
            if (size >= need) {
                ptr = reinterpret_cast<void *>(attribute(workspace, name_ptr));
                return;
            }
        }
        PyObject *want = PyLong_FromSize_t(need);
        PyObject *r = want == nullptr ? nullptr : PyObject_CallMethodObjArgs(workspace, name_get, want, nullptr);
        Py_XDECREF(want);
        PyObject *pair = r == nullptr ? nullptr : PySequence_Tuple(r);
        Py_XDECREF(r);
        if (pair == nullptr) throw PythonError{};
        const bool two = PyTuple_GET_SIZE(pair) == 2;
        if (two) {
            ptr = reinterpret_cast<void *>(number(PyTuple_GET_ITEM(pair, 0)));
            size = PyErr_Occurred() ? 0 : number(PyTuple_GET_ITEM(pair, 1));
        }
        Py_DECREF(pair);
        if (!two) raise(PyExc_ValueError, "workspace.get(nbytes): an address and a size expected");
        if (PyErr_Occurred()) throw PythonError{};
    }
    static size_t number(PyObject *v) {  // (an error is left set)
        PyObject *i = v == Py_None ? PyLong_FromLong(0) : PyNumber_Index(v);  // (None: the null pointer, as ctypes has it)
        const size_t n = i == nullptr ? 0 : PyLong_AsSize_t(i);
        Py_XDECREF(i);
        return n;
    }
    static size_t attribute(PyObject *o, PyObject *name) {
        PyObject *v = PyObject_GetAttr(o, name);
        if (v == nullptr) throw PythonError{};
        const size_t n = number(v);
        Py_DECREF(v);
        if (PyErr_Occurred()) throw PythonError{};
        return n;
    }
};

void *stream() { return c10::hip::getCurrentHIPStream().stream(); }

// The interpreter's lock is let go while this lives.
struct Unlocked {
    PyThreadState *state = PyEval_SaveThread();
    Unlocked() = default;
    Unlocked(const Unlocked &) = delete;
    ~Unlocked() { PyEval_RestoreThread(state); }
};

// A C ABI call without the interpreter's lock (a launch may wait for room in the queue).  Its arguments are plain
// values taken before: a tensor without storage (inside torch.vmap, jvp, grad) throws where its pointer is asked for.
template <typename Function, typename... Args> void call(Function function, Args... args) {
    const int rc = [&] {
        const Unlocked unlocked;
        return function(args...);
    }();
    if (rc == VKOP_HIP_OK) return;
    PyObject *e = PyObject_CallFunction(error_class, "is", rc, fn.last_error());
    if (e != nullptr) {
        PyErr_SetObject(error_class, e);
        Py_DECREF(e);
    }
    throw PythonError{};
}

PyObject *tuple_of(std::initializer_list<at::Tensor> tensors) {
    PyObject *t = PyTuple_New(static_cast<Py_ssize_t>(tensors.size()));
    if (t == nullptr) throw PythonError{};
    Py_ssize_t i = 0;
    for (const at::Tensor &x : tensors) {
        PyObject *o = THPVariable_Wrap(x);
        if (o == nullptr) {
            Py_DECREF(t);
            throw PythonError{};
        }
        PyTuple_SET_ITEM(t, i++, o);
    }
    return t;
}

template <typename F> PyObject *guarded(Py_ssize_t given, Py_ssize_t wanted, F &&f) {
    HANDLE_TH_ERRORS
    if (given != wanted) return PyErr_Format(PyExc_TypeError, "%zd arguments expected, got %zd", wanted, given);
    if (fn.topk == nullptr) return PyErr_Format(PyExc_RuntimeError, "bind() has not been called");
    try {
        return f();
    } catch (const PythonError &) {
        return nullptr;
    }
    END_HANDLE_TH_ERRORS
}

// softmax(x, axis, nan_where, nan_value, out or None, workspace) -> out
PyObject *softmax(PyObject *, PyObject *const *a, Py_ssize_t n) {
    return guarded(n, 6, [&]() -> PyObject * {
        const Input in(a[0]);
        const long axis = as_long(a[1]);
        const bool nan_where = as_bool(a[2]);
        const float nan_value = static_cast<float>(as_double(a[3]));
        at::Tensor out;
        void *result = nullptr;
        if (a[4] == Py_None) {
            out = in.empty(in.x.sizes(), in.x.scalar_type());
            result = out.data_ptr();
        } else {
            if (!THPVariable_Check(a[4])) raise(PyExc_TypeError, "out: a tensor expected");
            result = THPVariable_Unpack(a[4]).data_ptr();
        }
        const Scratch ws(a[5], fn.softmax_workspace_bytes(in.dtype, in.shape, in.ndim, static_cast<int>(axis)));
        void *st = stream();
        call(fn.softmax, in.data, result, in.dtype, in.shape, in.ndim, static_cast<int>(axis), nan_where ? 1 : 0, nan_value, ws.ptr,
             ws.size, st);
        if (a[4] == Py_None) return THPVariable_Wrap(out);
        Py_INCREF(a[4]);
        return a[4];
    });
}

// values and indices of a selection of k along an axis
struct Selection {
    at::DimVector sizes;
    at::Tensor values, indices;
    void *value_data = nullptr;
    int32_t *index_data = nullptr;
    Selection(const Input &in, long axis, long k) : sizes(in.x.sizes().begin(), in.x.sizes().end()) {
        sizes[static_cast<size_t>(in.place(axis))] = k;
        if (k < 0) raise(PyExc_RuntimeError, "k = %ld must be at least 1", k);
        values = in.empty(sizes, in.x.scalar_type());
        indices = in.empty(sizes, at::kInt);
        value_data = values.data_ptr();
        index_data = static_cast<int32_t *>(indices.data_ptr());
    }
};

// topk(x, k, axis, largest, sorted, workspace) -> (values, indices)
PyObject *topk(PyObject *, PyObject *const *a, Py_ssize_t n) {
    return guarded(n, 6, [&]() -> PyObject * {
        const Input in(a[0]);
        const long k = as_long(a[1]), axis = as_long(a[2]);
        const bool largest = as_bool(a[3]), sorted = as_bool(a[4]);
        const Selection s(in, axis, k);
        const int ik = static_cast<int>(k), ia = static_cast<int>(axis);
        const Scratch ws(a[5], fn.topk_workspace_bytes(in.dtype, in.shape, in.ndim, ia, ik));
        void *st = stream();
        call(fn.topk, in.data, s.value_data, s.index_data, in.dtype, in.shape, in.ndim, ia, ik, largest ? 1 : 0, sorted ? 1 : 0,
             ws.ptr, ws.size, st);
        return tuple_of({s.values, s.indices});
    });
}

// softmax_topk(x, k, axis, largest, return_probs, workspace) -> (values, indices[, probs])
PyObject *softmax_topk(PyObject *, PyObject *const *a, Py_ssize_t n) {
    return guarded(n, 6, [&]() -> PyObject * {
        const Input in(a[0]);
        const long k = as_long(a[1]), axis = as_long(a[2]);
        const bool largest = as_bool(a[3]), return_probs = as_bool(a[4]);
        const Selection s(in, axis, k);
        at::Tensor probs;
        void *prob_data = nullptr;
        if (return_probs) {
            probs = in.empty(in.x.sizes(), in.x.scalar_type());
            prob_data = probs.data_ptr();
        }
        const int ik = static_cast<int>(k), ia = static_cast<int>(axis);
        const Scratch ws(a[5], fn.softmax_topk_workspace_bytes(in.dtype, in.shape, in.ndim, ia, ik));
        void *st = stream();
        call(fn.softmax_topk, in.data, prob_data, s.value_data, s.index_data, in.dtype, in.shape, in.ndim, ia, ik, largest ? 1 : 0,
             ws.ptr, ws.size, st);
        return return_probs ? tuple_of({s.values, s.indices, probs}) : tuple_of({s.values, s.indices});
    });
}

// the shape without `axis`
at::DimVector without(const Input &in, long axis) {
    at::DimVector sizes;
    const int place = in.place(axis);
    for (int d = 0; d < in.ndim; d++)
        if (d != place) sizes.push_back(in.x.size(d));
    return sizes;
}

// softmax_topk_sampling(x, k, scale, top_p or None, axis, workspace) -> (values, indices[, counts])
PyObject *softmax_topk_sampling(PyObject *, PyObject *const *a, Py_ssize_t n) {
    return guarded(n, 6, [&]() -> PyObject * {
        const Input in(a[0]);
        const long k = as_long(a[1]), axis = as_long(a[4]);
        const float scale = static_cast<float>(as_double(a[2]));
        const bool counted = a[3] != Py_None;
        const float top_p = counted ? static_cast<float>(as_double(a[3])) : 0.f;
        const Selection s(in, axis, k);
        at::Tensor counts;
        int32_t *count_data = nullptr;
        if (counted) {
            counts = in.empty(without(in, axis), at::kInt);
            count_data = static_cast<int32_t *>(counts.data_ptr());
        }
        const int ik = static_cast<int>(k), ia = static_cast<int>(axis);
        const Scratch ws(a[5], fn.softmax_topk_workspace_bytes(in.dtype, in.shape, in.ndim, ia, ik));
        void *st = stream();
        call(fn.softmax_topk_sampling, in.data, s.value_data, s.index_data, count_data, in.dtype, in.shape, in.ndim, ia, ik, scale,
             top_p, ws.ptr, ws.size, st);
        return counted ? tuple_of({s.values, s.indices, counts}) : tuple_of({s.values, s.indices});
    });
}

// softmax_reduce_max(x, axis, workspace) -> out
PyObject *softmax_reduce_max(PyObject *, PyObject *const *a, Py_ssize_t n) {
    return guarded(n, 3, [&]() -> PyObject * {
        const Input in(a[0]);
        const long axis = as_long(a[1]);
        const int ia = static_cast<int>(axis);
        at::Tensor out = in.empty(without(in, axis), in.x.scalar_type());
        void *result = out.data_ptr();
        const Scratch ws(a[2], fn.softmax_reduce_max_workspace_bytes(in.dtype, in.shape, in.ndim, ia));
        void *st = stream();
        call(fn.softmax_reduce_max, in.data, result, in.dtype, in.shape, in.ndim, ia, ws.ptr, ws.size, st);
        return THPVariable_Wrap(out);
    });
}

// reduce_max(x, axis) -> out
PyObject *reduce_max(PyObject *, PyObject *const *a, Py_ssize_t n) {
    return guarded(n, 2, [&]() -> PyObject * {
        const Input in(a[0]);
        const long axis = as_long(a[1]);
        at::Tensor out = in.empty(without(in, axis), in.x.scalar_type());
        void *result = out.data_ptr();
        void *st = stream();
        call(fn.reduce_max, in.data, result, in.dtype, in.shape, in.ndim, static_cast<int>(axis), st);
        return THPVariable_Wrap(out);
    });
}

// bind({name without vkop_hip_: address}, VkopHipError, Workspace)
PyObject *bind(PyObject *, PyObject *const *a, Py_ssize_t n) {
    if (n != 3 || !PyDict_Check(a[0])) return PyErr_Format(PyExc_TypeError, "bind(addresses, error class, workspace class)");
    Functions f;
    auto address = [&](const char *name) -> void * {
        PyObject *v = PyDict_GetItemString(a[0], name);  // (borrowed)
        return v == nullptr ? nullptr : PyLong_AsVoidPtr(v);
    };
#define VKOP_NATIVE_BIND(name)                                                         \
    f.name = reinterpret_cast<decltype(f.name)>(address(#name));                       \
    if (f.name == nullptr) return PyErr_Format(PyExc_ValueError, "no address for " #name);
    VKOP_NATIVE_FUNCTIONS(VKOP_NATIVE_BIND)
#undef VKOP_NATIVE_BIND
    Py_INCREF(a[1]);
    Py_XDECREF(error_class);
    error_class = a[1];
    Py_INCREF(a[2]);
    Py_XDECREF(workspace_class);
    workspace_class = a[2];
    fn = f;
    Py_RETURN_NONE;
}

#define VKOP_NATIVE_METHOD(name) {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(name)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {VKOP_NATIVE_METHOD(bind), VKOP_NATIVE_METHOD(softmax), VKOP_NATIVE_METHOD(topk),
                         VKOP_NATIVE_METHOD(softmax_topk), VKOP_NATIVE_METHOD(softmax_topk_sampling),
                         VKOP_NATIVE_METHOD(softmax_reduce_max), VKOP_NATIVE_METHOD(reduce_max), {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_native", "Native front end of vkop_amd.ops.", -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

#define VKOP_NATIVE_TEXT2(x) #x
#define VKOP_NATIVE_TEXT(x) VKOP_NATIVE_TEXT2(x)
PyMODINIT_FUNC PyInit__native() {
    // (the file's name does not say which interpreter it was built for)
    constexpr char built_for[] = VKOP_NATIVE_TEXT(PY_MAJOR_VERSION) "." VKOP_NATIVE_TEXT(PY_MINOR_VERSION) ".";
    if (std::strncmp(Py_GetVersion(), built_for, sizeof built_for - 1) != 0)
        return PyErr_Format(PyExc_ImportError, "built for Python %sx, this is %s", built_for, Py_GetVersion());
    name_ptr = PyUnicode_InternFromString("ptr");
    name_size = PyUnicode_InternFromString("size");
    name_get = PyUnicode_InternFromString("get");
    if (name_ptr == nullptr || name_size == nullptr || name_get == nullptr) return nullptr;
    PyObject *m = PyModule_Create(&module);
    if (m != nullptr && PyModule_AddStringConstant(m, "torch_version", TORCH_VERSION) != 0) {
        Py_DECREF(m);
        return nullptr;
    }
    return m;
}
