// The device entry points that a program calls once per layer or product, without ctypes: a CPython module over include/ftnn.h.
//
// Such a call is two launches at most, 2.2 us of host time each, and on the device it takes 3 to 7 us; ctypes (0.9 us for the
// arguments of a layer) and the checks on its tensors in Python (1.1 us for five) come on top of that, call after call.  Here
// both take 0.2 us.  A call queued behind others, before and now: TBN layer 8 x 128 x 28 x 28 9.8 -> 8.0 us, TNN 256 x 56 x 56
// 9.9 -> 7.9, fully connected layers of 0.5 M weights 9.2 -> 5.9, TNN product 256 x 256 x 4096 5.7 -> 3.7.
//
// Every function takes the arguments of its wrapper in fastertnn_amd/lib.py and returns the library's status, or None where
// an argument is not of the plain kind that it reads itself (an int, a float, a contiguous torch.Tensor on the GPU that is no
// subclass): the wrapper then goes on through ctypes, which converts or refuses it as it always has.
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>

#include <climits>

#include "../../include/ftnn.h"

namespace {

struct Args {
    PyObject* const* v;
    bool good = true;   // every argument so far was a plain one

    int i(int k) {
        if (!PyLong_CheckExact(v[k])) return bad();
        int over = 0;
        const long x = PyLong_AsLongAndOverflow(v[k], &over);
        return over || x < INT_MIN || x > INT_MAX ? bad() : (int)x;
    }
    float f(int k) {
        if (PyFloat_CheckExact(v[k])) return (float)PyFloat_AS_DOUBLE(v[k]);
        return (float)i(k);
    }
    // data of a contiguous device tensor
    char* any(int k, int64_t* bytes = nullptr) {
        if (!THPVariable_CheckExact(v[k])) return bad(), nullptr;
        const at::Tensor& t = THPVariable_Unpack(v[k]);
        if (!t.is_cuda() || !t.is_contiguous()) return bad(), nullptr;
        if (bytes) *bytes = t.numel() * (int64_t)t.element_size();
        return static_cast<char*>(t.data_ptr());
    }
    float* f32(int k) {
        if (!THPVariable_CheckExact(v[k]) || THPVariable_Unpack(v[k]).scalar_type() != at::kFloat) return bad(), nullptr;
        return reinterpret_cast<float*>(any(k));
    }
    const int64_t* words(int k) { return reinterpret_cast<const int64_t*>(any(k)); }
    // N, C, H, W of a layer's input
    bool nchw(int k, int d[4]) {
        if (!THPVariable_CheckExact(v[k])) return bad(), false;
        const at::Tensor& t = THPVariable_Unpack(v[k]);
        if (t.dim() != 4) return bad(), false;
        for (int j = 0; j < 4; j++) {
            if (t.size(j) > INT_MAX) return bad(), false;
            d[j] = (int)t.size(j);
        }
        return true;
    }
    int bad() {
        good = false;
        return 0;
    }
};

// fn(arguments, stream) with N arguments, the lock of the interpreter released around the library
template <Py_ssize_t N, typename F>
PyObject* call(PyObject* const* v, Py_ssize_t n, F&& read) {
    if (n != N) Py_RETURN_NONE;
    int rc = 0;
    try {
        Args a{v};
        auto fn = read(a);
        if (!a.good) Py_RETURN_NONE;
        void* stream = c10::hip::getCurrentHIPStream().stream();
        Py_BEGIN_ALLOW_THREADS
        rc = fn(stream);
        Py_END_ALLOW_THREADS
    } catch (...) {   // a tensor without storage, say: the wrapper meets it again
        Py_RETURN_NONE;
    }
    return PyLong_FromLong(rc);
}

// typ, a, b, n, oh, ow, kn, k, alpha, k_unpack, out
PyObject* mm(PyObject*, PyObject* const* v, Py_ssize_t n) {
    return call<11>(v, n, [](Args& r) {
        return [typ = r.i(0), a = r.words(1), b = r.words(2), n = r.i(3), oh = r.i(4), ow = r.i(5), kn = r.i(6), k = r.i(7),
                alpha = r.f(8), ku = r.i(9), out = r.f32(10)](void* st) { return ftnn_mm(typ, a, b, n, oh, ow, kn, k, ku, alpha, out, st); };
    });
}

// engine, typ, a, b, n, oh, ow, kn, k, alpha, k_unpack, out, scratch
PyObject* mm_engine(PyObject*, PyObject* const* v, Py_ssize_t n) {
    return call<13>(v, n, [](Args& r) {
        int64_t bytes = 0;
        void* scratch = r.any(12, &bytes);
        return [=, e = r.i(0), typ = r.i(1), a = r.words(2), b = r.words(3), n = r.i(4), oh = r.i(5), ow = r.i(6), kn = r.i(7), k = r.i(8),
                alpha = r.f(9), ku = r.i(10), out = r.f32(11)](void* st) {
            return ftnn_mm_engine(e, typ, a, b, n, oh, ow, kn, k, ku, alpha, out, scratch, bytes, st);
        };
    });
}

// engine, typ, a_exp, b_exp, n, oh, ow, kn, k, alpha, k_unpack, out
PyObject* mm_expanded(PyObject*, PyObject* const* v, Py_ssize_t n) {
    return call<12>(v, n, [](Args& r) {
        return [e = r.i(0), typ = r.i(1), a = r.any(2), b = r.any(3), n = r.i(4), oh = r.i(5), ow = r.i(6), kn = r.i(7), k = r.i(8),
                alpha = r.f(9), ku = r.i(10), out = r.f32(11)](void* st) { return ftnn_mm_expanded(e, typ, a, b, n, oh, ow, kn, k, ku, alpha, out, st); };
    });
}

struct Layer {
    int typ, d[4], kn, kh, kw, pad, stride;
    const float *x, *thr;
    float alpha, *y;
};
// typ, x, thr, weights, kn, kh, kw, pad, stride, alpha, ..., out
Layer layer(Args& r, int out) {
    Layer l;
    r.nchw(1, l.d);
    l.typ = r.i(0), l.x = r.f32(1), l.thr = r.f32(2);
    l.kn = r.i(4), l.kh = r.i(5), l.kw = r.i(6), l.pad = r.i(7), l.stride = r.i(8), l.alpha = r.f(9), l.y = r.f32(out);
    return l;
}

// ..., scratch, out
PyObject* conv(PyObject*, PyObject* const* v, Py_ssize_t n) {
    return call<12>(v, n, [](Args& r) {
        return [l = layer(r, 11), w = r.words(3), scratch = r.any(10)](void* st) {
            return ftnn_conv(l.typ, l.x, l.thr, w, l.d[0], l.d[1], l.d[2], l.d[3], l.kn, l.kh, l.kw, l.pad, l.pad, l.stride, l.stride, l.alpha,
                             scratch, l.y, st);
        };
    });
}
PyObject* conv_prepared(PyObject*, PyObject* const* v, Py_ssize_t n) {
    return call<12>(v, n, [](Args& r) {
        return [l = layer(r, 11), w = r.any(3), scratch = r.any(10)](void* st) {
            return ftnn_conv_prepared(l.typ, l.x, l.thr, w, l.d[0], l.d[1], l.d[2], l.d[3], l.kn, l.kh, l.kw, l.pad, l.pad, l.stride, l.stride,
                                      l.alpha, scratch, l.y, st);
        };
    });
}
// ..., out
PyObject* conv_static(PyObject*, PyObject* const* v, Py_ssize_t n) {
    return call<11>(v, n, [](Args& r) {
        return [l = layer(r, 10), w = r.words(3)](void* st) {
            return ftnn_conv_static(l.typ, l.x, l.thr, w, l.d[0], l.d[1], l.d[2], l.d[3], l.kn, l.kh, l.kw, l.pad, l.pad, l.stride, l.stride,
                                    l.alpha, l.y, st);
        };
    });
}

// net handle, x, out, use_graph
PyObject* net_run(PyObject*, PyObject* const* v, Py_ssize_t n) {
    return call<4>(v, n, [](Args& r) {
        void* net = PyLong_CheckExact(r.v[0]) ? PyLong_AsVoidPtr(r.v[0]) : nullptr;
        if (!net) PyErr_Clear(), r.bad();
        return [net, x = r.f32(1), out = r.f32(2), graph = r.i(3)](void* st) { return ftnn_net_run(static_cast<ftnn_net_t*>(net), x, out, graph, st); };
    });
}

#define FTNN_METHOD(name) {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(name)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {FTNN_METHOD(mm),          FTNN_METHOD(mm_engine), FTNN_METHOD(mm_expanded), FTNN_METHOD(conv), FTNN_METHOD(conv_prepared),
                         FTNN_METHOD(conv_static), FTNN_METHOD(net_run),   {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_call", "ftnn device calls without ctypes", -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__call(void) {
    PyObject* const m = PyModule_Create(&module);
    // the torch whose tensors it reads: another one's may lie otherwise in memory
    if (m && PyModule_AddStringConstant(m, "torch_version", FTNN_TORCH) < 0) {
        Py_DECREF(m);
        return nullptr;
    }
    return m;
}
