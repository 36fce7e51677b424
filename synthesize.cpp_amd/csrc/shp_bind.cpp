// The calling side of the Python binding, for CPython: an entry point of
// libsynth_hip as a Python callable that takes torch tensors.
//
//   bind(handle, name)  -> callable(arg, ...) -> status
//   describe(tensor)    -> the bytes of its shp_tensor
//
// handle is the loaded library's dlopen handle (ctypes' CDLL._handle), so a
// process may bind any build of the library. Each C parameter is converted
// from its Python argument by its type: a tensor pointer from a torch tensor, a
// BlockTensor or None, numbers from numbers, a stream from its address. A
// BlockTensor and a ctypes ShpTensor are known by an attribute of their class
// (SHP_BLOCKS, SHP_TENSOR), not by the class: a program that loads or reloads the
// Python half twice has two of each, and tensors of both. Two
// entry points start with an array of tensors and its length: there alone a list
// or tuple is taken, of that length. shp_im2col starts with a kernel of which
// only the shape is read: that is a ShpTensor too. The GIL is released while the
// entry point runs.
//
// Why native: filling one descriptor field by field through ctypes takes 4 us
// of Python, ten times an entry point's own host work, and a call has two to
// nineteen of them; here it takes 0.09 us. A prefill layer step of 509 positions
// (one 9.8 us launch) went from 48 us a call to 8.8, the embedding stage (four
// calls) from 82 to 31.

#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <dlfcn.h>

#include <array>
#include <cstring>
#include <exception>
#include <tuple>
#include <utility>
#include <vector>

#include <torch/csrc/autograd/python_variable.h>

#include "synth_hip.h"

namespace {

PyObject * g_data   = nullptr;  // interned attribute names of BlockTensor
PyObject * g_ne0    = nullptr;
PyObject * g_type   = nullptr;
PyObject * g_size   = nullptr;
PyObject * g_blocks = nullptr;  // ... and the class attributes that mark it and ShpTensor
PyObject * g_tensor = nullptr;

// 1 if o's class has the attribute `mark` (as True), 0 if not, -1 with an error set.
int marked(PyObject * o, PyObject * mark) {
    PyObject * v = PyObject_GetAttr(reinterpret_cast<PyObject *>(Py_TYPE(o)), mark);
    if (v == nullptr) {
        if (!PyErr_ExceptionMatches(PyExc_AttributeError)) {
            return -1;
        }
        PyErr_Clear();
        return 0;
    }
    const int yes = v == Py_True ? 1 : 0;
    Py_DECREF(v);
    return yes;
}

// shp_tensor for a torch tensor. Dimensions past the tensor's own have extent
// 1 and the stride of everything below them.
bool from_tensor(PyObject * o, shp_tensor & d) {
    const at::Tensor & t = THPVariable_Unpack(o);
    switch (t.scalar_type()) {
        case at::kFloat:
            d.type = SHP_TYPE_F32;
            break;
        case at::kHalf:
            d.type = SHP_TYPE_F16;
            break;
        case at::kBFloat16:
            d.type = SHP_TYPE_BF16;
            break;
        case at::kInt:
            d.type = SHP_TYPE_I32;
            break;
        case at::kByte:
        case at::kChar:
            d.type = -1;  // raw blocks: the caller names the type
            break;
        default: {
            PyObject * dt = PyObject_GetAttrString(o, "dtype");
            if (dt != nullptr) {
                PyErr_SetObject(PyExc_KeyError, dt);
                Py_DECREF(dt);
            }
            return false;
        }
    }
    const int64_t nd = t.dim();
    if (nd > 4) {
        PyErr_SetString(PyExc_ValueError, "at most 4 dimensions");
        return false;
    }
    const int64_t item = static_cast<int64_t>(t.element_size());
    d.reserved         = 0;
    for (int64_t k = 0; k < 4; ++k) {
        if (k < nd) {
            d.ne[k] = t.size(nd - 1 - k);
            d.nb[k] = static_cast<size_t>(t.stride(nd - 1 - k) * item);
        } else if (k == 0) {  // a scalar
            d.ne[0] = 1;
            d.nb[0] = static_cast<size_t>(item);
        } else {
            d.ne[k] = 1;
            d.nb[k] = d.nb[k - 1] * static_cast<size_t>(d.ne[k - 1]);
        }
    }
    d.data = t.data_ptr();
    return true;
}

bool attr_int(PyObject * o, PyObject * name, int64_t & v) {
    PyObject * a = PyObject_GetAttr(o, name);
    if (a == nullptr) {
        return false;
    }
    v = PyLong_AsLongLong(a);
    Py_DECREF(a);
    return !(v == -1 && PyErr_Occurred() != nullptr);
}

bool to_tensor(PyObject * o, shp_tensor & d) {
    if (THPVariable_Check(o)) {
        if (!from_tensor(o, d)) {
            return false;
        }
        if (d.type == -1) {
            PyObject * dt = PyObject_GetAttrString(o, "dtype");
            if (dt != nullptr) {
                PyErr_SetObject(PyExc_KeyError, dt);
                Py_DECREF(dt);
            }
            return false;
        }
        return true;
    }
    const int block = marked(o, g_blocks);
    if (block < 1) {
        if (block == 0) {
            PyErr_Format(PyExc_TypeError, "expected a tensor, got %s", Py_TYPE(o)->tp_name);
        }
        return false;
    }
    // raw blocks (..., rows, ne0 / ELEMS * BYTES) with a logical row length
    int64_t    ne0 = 0, type = 0, bytes = 0, nd = 0;
    PyObject * raw = PyObject_GetAttr(o, g_data);
    if (raw == nullptr) {
        return false;
    }
    bool ok = THPVariable_Check(raw) && from_tensor(raw, d) && attr_int(o, g_ne0, ne0) && attr_int(o, g_type, type) &&
              attr_int(o, g_size, bytes);
    if (ok) {
        nd = THPVariable_Unpack(raw).dim();
    }
    Py_DECREF(raw);
    if (!ok) {
        if (PyErr_Occurred() == nullptr) {
            PyErr_SetString(PyExc_TypeError, "expected a tensor");
        }
        return false;
    }
    d.type  = static_cast<int32_t>(type);
    d.ne[0] = ne0;
    d.nb[0] = static_cast<size_t>(bytes);
    for (int64_t k = nd < 1 ? 1 : nd; k < 4; ++k) {
        d.nb[k] = d.nb[k - 1] * static_cast<size_t>(d.ne[k - 1]);
    }
    return true;
}

// What an argument's pointer points to while the call runs.
struct Slot {
    shp_tensor              one;
    std::vector<shp_tensor> many;
    std::array<int32_t, 4>  ints;
};

template <class T> struct Arg;

template <> struct Arg<const shp_tensor *> {
    static bool get(PyObject * o, Slot & s, const shp_tensor *& v) {
        v = o == Py_None ? nullptr : &s.one;
        return o == Py_None || to_tensor(o, s.one);
    }
};

// What an entry point's first parameter is beside a tensor.
enum First { kTensor = 0, kArray = 1, kShape = 2 };

// An array of tensors; the entry point reads as many as the parameter after it
// says.
bool array_arg(PyObject * o, PyObject * count, Slot & s, const shp_tensor *& v) {
    if (!PyList_Check(o) && !PyTuple_Check(o)) {
        PyErr_SetString(PyExc_TypeError, "expected a list of tensors");
        return false;
    }
    PyObject * items = PySequence_Tuple(o);  // (a conversion may run Python code: a list could change under it)
    if (items == nullptr) {
        return false;
    }
    const Py_ssize_t n  = PyTuple_GET_SIZE(items);
    const long long  c  = PyLong_AsLongLong(count);
    bool             ok = !(c == -1 && PyErr_Occurred() != nullptr);
    if (ok && c != n) {
        PyErr_Format(PyExc_ValueError, "%zd tensors for a count of %lld", n, c);
        ok = false;
    }
    try {
        s.many.resize(static_cast<size_t>(n));
        for (Py_ssize_t i = 0; ok && i < n; ++i) {
            ok = to_tensor(PyTuple_GET_ITEM(items, i), s.many[static_cast<size_t>(i)]);
        }
    } catch (...) {
        Py_DECREF(items);
        throw;
    }
    Py_DECREF(items);
    v = s.many.data();
    return ok;
}

// A ctypes ShpTensor, for a parameter of which only the shape is read.
bool shape_arg(PyObject * o, Slot & s, const shp_tensor *& v) {
    const int shape = marked(o, g_tensor);
    if (shape < 1) {
        return shape == 0 && Arg<const shp_tensor *>::get(o, s, v);
    }
    Py_buffer b;
    if (PyObject_GetBuffer(o, &b, PyBUF_SIMPLE) != 0) {
        return false;
    }
    const bool ok = b.len == static_cast<Py_ssize_t>(sizeof(shp_tensor));
    if (ok) {
        std::memcpy(&s.one, b.buf, sizeof(s.one));
        v = &s.one;
    } else {
        PyErr_SetString(PyExc_TypeError, "expected a descriptor");
    }
    PyBuffer_Release(&b);
    return ok;
}

template <> struct Arg<shp_tensor *> {
    static bool get(PyObject * o, Slot & s, shp_tensor *& v) {
        v = o == Py_None ? nullptr : &s.one;
        return o == Py_None || to_tensor(o, s.one);
    }
};

template <> struct Arg<float> {
    static bool get(PyObject * o, Slot &, float & v) {
        const double d = PyFloat_AsDouble(o);
        v              = static_cast<float>(d);
        return !(d == -1.0 && PyErr_Occurred() != nullptr);
    }
};

// As ctypes takes integers: any size, the low bits kept.
template <> struct Arg<int64_t> {
    static bool get(PyObject * o, Slot &, int64_t & v) {
        v = static_cast<int64_t>(PyLong_AsUnsignedLongLongMask(o));
        return PyErr_Occurred() == nullptr;
    }
};

template <> struct Arg<int32_t> {
    static bool get(PyObject * o, Slot & s, int32_t & v) {
        int64_t    w  = 0;
        const bool ok = Arg<int64_t>::get(o, s, w);
        v             = static_cast<int32_t>(w);
        return ok;
    }
};

template <> struct Arg<const int32_t *> {
    static bool get(PyObject * o, Slot & s, const int32_t *& v) {
        if (!(PyList_Check(o) || PyTuple_Check(o)) || PySequence_Fast_GET_SIZE(o) != 4) {
            PyErr_SetString(PyExc_TypeError, "expected four integers");
            return false;
        }
        for (Py_ssize_t i = 0; i < 4; ++i) {
            if (!Arg<int32_t>::get(PySequence_Fast_GET_ITEM(o, i), s, s.ints[static_cast<size_t>(i)])) {
                return false;
            }
        }
        v = s.ints.data();
        return true;
    }
};

template <> struct Arg<shp_stream_t> {
    static bool get(PyObject * o, Slot &, shp_stream_t & v) {
        v = o == Py_None ? nullptr : static_cast<shp_stream_t>(PyLong_AsVoidPtr(o));
        return PyErr_Occurred() == nullptr;
    }
};

bool counted(Py_ssize_t got, Py_ssize_t want) {
    if (got != want) {
        PyErr_Format(PyExc_TypeError, "expected %zd arguments, got %zd", want, got);
        return false;
    }
    return true;
}

template <class F, First FIRST> struct Call;

template <First FIRST, class... A> struct Call<shp_status_t (*)(A...), FIRST> {
    template <size_t I> static bool convert_one(PyObject * const * args, Slot & slot, std::tuple<A...> & vals) {
        using T = std::tuple_element_t<I, std::tuple<A...>>;
        if constexpr (I == 0 && FIRST == kArray) {
            return array_arg(args[0], args[1], slot, std::get<0>(vals));
        } else if constexpr (I == 0 && FIRST == kShape) {
            return shape_arg(args[0], slot, std::get<0>(vals));
        } else {
            return Arg<T>::get(args[I], slot, std::get<I>(vals));
        }
    }

    template <size_t... I>
    static bool convert(PyObject * const * args, std::array<Slot, sizeof...(A)> & slots, std::tuple<A...> & vals,
                        std::index_sequence<I...>) {
        return (convert_one<I>(args, slots[I], vals) && ...);
    }

    static PyObject * run(void * fn, PyObject * const * args, Py_ssize_t n) {
        if (!counted(n, sizeof...(A))) {
            return nullptr;
        }
        std::array<Slot, sizeof...(A)> slots;
        std::tuple<A...>               vals{};
        if (!convert(args, slots, vals, std::index_sequence_for<A...>{})) {
            return nullptr;
        }
        shp_status_t st;
        Py_BEGIN_ALLOW_THREADS;
        st = std::apply(reinterpret_cast<shp_status_t (*)(A...)>(fn), vals);
        Py_END_ALLOW_THREADS;
        return PyLong_FromLong(st);
    }
};

// The layer step: its struct's tensors in order, then eps, freq_base, n_dims
// and the stream.
PyObject * run_layer(void * fn, PyObject * const * args, Py_ssize_t n) {
    constexpr Py_ssize_t kTensors = 19;
    if (!counted(n, kTensors + 4)) {
        return nullptr;
    }
    shp_tensor   t[kTensors];
    shp_tensor * p[kTensors];
    for (Py_ssize_t i = 0; i < kTensors; ++i) {
        p[i] = args[i] == Py_None ? nullptr : &t[i];
        if (args[i] != Py_None && !to_tensor(args[i], t[i])) {
            return nullptr;
        }
    }
    Slot           s;
    shp_layer_step step{ p[0],  p[1],  p[2],  p[3],  p[4],  p[5],  p[6],  p[7],  p[8],  p[9], p[10], p[11],
                         p[12], p[13], p[14], p[15], p[16], p[17], p[18], 0.0f,  0.0f,  0,    0 };
    shp_stream_t   stream = nullptr;
    if (!Arg<float>::get(args[kTensors], s, step.eps) || !Arg<float>::get(args[kTensors + 1], s, step.freq_base) ||
        !Arg<int32_t>::get(args[kTensors + 2], s, step.n_dims) ||
        !Arg<shp_stream_t>::get(args[kTensors + 3], s, stream)) {
        return nullptr;
    }
    shp_status_t st;
    Py_BEGIN_ALLOW_THREADS;
    st = reinterpret_cast<decltype(&shp_layer_nongemm_step)>(fn)(&step, stream);
    Py_END_ALLOW_THREADS;
    return PyLong_FromLong(st);
}

using Runner = PyObject * (*) (void *, PyObject * const *, Py_ssize_t);

struct Entry {
    const char * name;
    Runner       run;
};

#define SHP_ENTRY_FIRST(f, first) { #f, &Call<decltype(&f), first>::run }
#define SHP_ENTRY(f) SHP_ENTRY_FIRST(f, kTensor)

const Entry kEntries[] = {
    SHP_ENTRY(shp_get_rows), SHP_ENTRY_FIRST(shp_get_rows_sum, kArray), SHP_ENTRY(shp_rms_norm_mul), SHP_ENTRY(shp_add_rms_norm_mul),
    SHP_ENTRY(shp_rope_ext), SHP_ENTRY(shp_qk_norm_rope), SHP_ENTRY(shp_qk_norm_rope_kv),
    SHP_ENTRY(shp_qk_norm_rope_kv_at), SHP_ENTRY(shp_swiglu), SHP_ENTRY(shp_glu_swiglu), SHP_ENTRY(shp_snake),
    SHP_ENTRY(shp_snake_guarded), SHP_ENTRY(shp_snake_beta), SHP_ENTRY(shp_add_leaky_relu), SHP_ENTRY(shp_add),
    SHP_ENTRY(shp_mul), SHP_ENTRY(shp_div), SHP_ENTRY(shp_sin), SHP_ENTRY(shp_sqr), SHP_ENTRY(shp_cpy),
    SHP_ENTRY(shp_sub), SHP_ENTRY(shp_tanh), SHP_ENTRY(shp_sigmoid), SHP_ENTRY(shp_elu), SHP_ENTRY(shp_gelu_erf),
    SHP_ENTRY(shp_clamp), SHP_ENTRY(shp_norm), SHP_ENTRY(shp_relu), SHP_ENTRY(shp_neg), SHP_ENTRY(shp_step),
    SHP_ENTRY(shp_sqrt), SHP_ENTRY(shp_sum_rows), SHP_ENTRY(shp_mean), SHP_ENTRY(shp_mul_sum_rows),
    SHP_ENTRY(shp_inverse_stft), SHP_ENTRY(shp_harmonic_source), SHP_ENTRY(shp_log_mel), SHP_ENTRY(shp_concat),
    SHP_ENTRY(shp_col2im_1d), SHP_ENTRY(shp_pad), SHP_ENTRY(shp_pad_reflect_1d), SHP_ENTRY(shp_repeat),
    SHP_ENTRY(shp_acc), SHP_ENTRY_FIRST(shp_im2col, kShape), SHP_ENTRY(shp_cont_add_leaky_relu), SHP_ENTRY(shp_soft_max_ext),
    SHP_ENTRY(shp_diag_mask_inf), SHP_ENTRY(shp_soft_max_causal), SHP_ENTRY(shp_exp), SHP_ENTRY(shp_scale_bias),
    SHP_ENTRY_FIRST(shp_sum_scale_leaky_relu, kArray), { "shp_layer_nongemm_step", &run_layer },
};

struct Bound {
    Runner run;
    void * fn;
};

PyObject * call(PyObject * self, PyObject * const * args, Py_ssize_t n) {
    const Bound * b = static_cast<const Bound *>(PyCapsule_GetPointer(self, nullptr));
    if (b == nullptr) {
        return nullptr;
    }
    try {
        return b->run(b->fn, args, n);
    } catch (const std::exception & e) {  // torch refuses a tensor without storage this way
        PyErr_SetString(PyExc_RuntimeError, e.what());
    } catch (...) {
        PyErr_SetString(PyExc_RuntimeError, "unknown C++ exception");
    }
    return nullptr;
}

PyMethodDef kCall = { "entry_point", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(&call)), METH_FASTCALL,
                      nullptr };

PyObject * bind(PyObject *, PyObject * args) {
    unsigned long long handle = 0;
    const char *       name   = nullptr;
    if (!PyArg_ParseTuple(args, "Ks", &handle, &name)) {
        return nullptr;
    }
    for (const Entry & e : kEntries) {
        if (std::strcmp(e.name, name) != 0) {
            continue;
        }
        void * fn = dlsym(reinterpret_cast<void *>(handle), name);
        if (fn == nullptr) {
            break;
        }
        Bound *    b   = new Bound{ e.run, fn };
        PyObject * cap = PyCapsule_New(b, nullptr, [](PyObject * c) {
            delete static_cast<Bound *>(PyCapsule_GetPointer(c, nullptr));
        });
        if (cap == nullptr) {
            delete b;
            return nullptr;
        }
        PyObject * f = PyCFunction_New(&kCall, cap);
        Py_DECREF(cap);
        return f;
    }
    PyErr_Format(PyExc_AttributeError, "no entry point %s", name);
    return nullptr;
}

PyObject * describe(PyObject *, PyObject * o) {
    try {
        shp_tensor d;
        return to_tensor(o, d) ? PyBytes_FromStringAndSize(reinterpret_cast<const char *>(&d), sizeof(d)) : nullptr;
    } catch (const std::exception & e) {
        PyErr_SetString(PyExc_RuntimeError, e.what());
    } catch (...) {
        PyErr_SetString(PyExc_RuntimeError, "unknown C++ exception");
    }
    return nullptr;
}

PyMethodDef kMethods[] = { { "describe", describe, METH_O, "describe(tensor) -> the bytes of its shp_tensor" },
                           { "bind", bind, METH_VARARGS, "bind(handle, name) -> callable" },
                           { nullptr, nullptr, 0, nullptr } };

PyModuleDef kModule = { PyModuleDef_HEAD_INIT, "shp_bind", nullptr, -1, kMethods, nullptr, nullptr, nullptr, nullptr };

}  // namespace

PyMODINIT_FUNC PyInit_shp_bind() {
    g_data   = PyUnicode_InternFromString("data");
    g_ne0    = PyUnicode_InternFromString("ne0");
    g_type   = PyUnicode_InternFromString("TYPE");
    g_size   = PyUnicode_InternFromString("BYTES");
    g_blocks = PyUnicode_InternFromString("SHP_BLOCKS");
    g_tensor = PyUnicode_InternFromString("SHP_TENSOR");
    for (PyObject * name : { g_data, g_ne0, g_type, g_size, g_blocks, g_tensor }) {
        if (name == nullptr) {
            return nullptr;
        }
    }
    return PyModule_Create(&kModule);
}
