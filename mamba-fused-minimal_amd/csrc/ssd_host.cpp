// Python extension module `_ssd_host`: from tensors to the C entry points of libssd_gfx950.so without a detour through
// ctypes.  Describing nine tensors as ssd_tensor structs field by field from Python takes longer than the kernels of a
// small call do (13 us a fused call, of 27); here the sizes, strides and pointers are read off the tensor objects.
// Nothing is checked or kept here: shapes are the wrappers' business (ssd_amd/ops.py), everything else the library's.
#include <Python.h>

#include <torch/csrc/autograd/python_variable.h>

#include <string>

#include "../../include/ssd_gfx950.h"

namespace {

struct PyFailure {};      // a Python exception is set

// None -> a struct with a NULL data pointer, as ssd_amd/_lib.py: tensor_arg has it
ssd_tensor tensor(PyObject *o)
{
    ssd_tensor t{};
    if (o == Py_None) return t;
    if (!THPVariable_Check(o)) {
        PyErr_Format(PyExc_TypeError, "expected a tensor or None, got %s", Py_TYPE(o)->tp_name);
        throw PyFailure();
    }
    const at::Tensor &v = THPVariable_Unpack(o);
    switch (v.scalar_type()) {
        case at::kInt: t.dtype = 0; break;
        case at::kFloat: t.dtype = SSD_F32; break;
        case at::kBFloat16: t.dtype = SSD_BF16; break;
        case at::kHalf: t.dtype = SSD_F16; break;
        default:
            PyErr_Format(PyExc_TypeError, "unsupported dtype %s", c10::toString(v.scalar_type()));
            throw PyFailure();
    }
    const auto strides = v.strides();
    if (strides.size() > 5) {
        PyErr_SetString(PyExc_IndexError, "a tensor of more than five dimensions");
        throw PyFailure();
    }
    t.data = v.data_ptr();
    for (size_t i = 0; i < strides.size(); ++i) t.stride[i] = strides[i];
    return t;
}

int64_t number(PyObject *o)
{
    const long long v = PyLong_AsLongLong(o);
    if (v == -1 && PyErr_Occurred()) throw PyFailure();
    return v;
}

void *pointer(PyObject *o)
{
    void *const v = PyLong_AsVoidPtr(o);
    if (!v && PyErr_Occurred()) throw PyFailure();
    return v;
}

double real(PyObject *o)
{
    const double v = PyFloat_AsDouble(o);
    if (v == -1.0 && PyErr_Occurred()) throw PyFailure();
    return v;
}

int32_t size32(int64_t n)
{
    if (n < 0 || n > 0x7fffffffLL) {
        PyErr_SetString(PyExc_OverflowError, "a size beyond 32 bits");
        throw PyFailure();
    }
    return (int32_t)n;
}

const at::Tensor &unpack(PyObject *o, int64_t dim)
{
    if (!THPVariable_Check(o) || THPVariable_Unpack(o).dim() != dim) {
        PyErr_Format(PyExc_TypeError, "expected a tensor of %d dimensions", (int)dim);
        throw PyFailure();
    }
    return THPVariable_Unpack(o);
}

// sizes of x (b,L,H,P), B (b,L,G,N), dt (b,H,C,Q)
ssd_dims dims_of(PyObject *x, PyObject *B, PyObject *dt)
{
    const at::Tensor &xv = unpack(x, 4), &Bv = unpack(B, 4), &dv = unpack(dt, 4);
    return ssd_dims{size32(xv.size(0)), size32(xv.size(1)), size32(xv.size(2)), size32(xv.size(3)),
                    size32(Bv.size(3)), size32(Bv.size(2)), size32(dv.size(3)), size32(dv.size(2))};
}

// Runs f with C++ exceptions (a tensor without storage, say) turned into Python ones.
template <class F>
PyObject *guarded(Py_ssize_t got, Py_ssize_t want, F &&f)
{
    if (got != want) {
        PyErr_Format(PyExc_TypeError, "%zd arguments, %zd expected", got, want);
        return nullptr;
    }
    try {
        return f();
    } catch (const PyFailure &) {
        return nullptr;
    } catch (const std::exception &e) {
        PyErr_SetString(PyExc_RuntimeError, e.what());
        return nullptr;
    } catch (...) {
        PyErr_SetString(PyExc_RuntimeError, "unknown C++ exception");
        return nullptr;
    }
}

// The call itself without the interpreter lock: a launch waits where its queue is full.
template <class F>
int unlocked(F &&f)
{
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = f();
    Py_END_ALLOW_THREADS
    return rc;
}

// x, B, dt, dA_cumsum, seq_idx, states, clamp, stream -> status
PyObject *chunk_state(PyObject *, PyObject *const *a, Py_ssize_t n)
{
    return guarded(n, 8, [&]() -> PyObject * {
        ssd_tensor t[6];
        for (int i = 0; i < 6; ++i) t[i] = tensor(a[i]);
        const ssd_dims d = dims_of(a[0], a[1], a[2]);
        const int clamp = (int)number(a[6]);
        void *const stream = pointer(a[7]);
        return PyLong_FromLong(unlocked([&] { return ssd_chunk_state_fwd(&t[0], &t[1], &t[2], &t[3], &t[4], &t[5], &d, clamp, stream); }));
    });
}

// states, dA_chunk, initial_states, seq_idx, out, final_states, seqlen, chunk_size, stream -> status
PyObject *state_passing(PyObject *, PyObject *const *a, Py_ssize_t n)
{
    return guarded(n, 9, [&]() -> PyObject * {
        ssd_tensor t[6];
        for (int i = 0; i < 6; ++i) t[i] = tensor(a[i]);
        const at::Tensor &s = unpack(a[0], 4);
        const int32_t b = size32(s.size(0)), C = size32(s.size(1)), H = size32(s.size(2)), dim = size32(s.size(3)),
                      L = size32(number(a[6])), Q = size32(number(a[7]));
        void *const stream = pointer(a[8]);
        return PyLong_FromLong(unlocked([&] {
            return ssd_state_passing_fwd(&t[0], &t[1], &t[2], &t[3], &t[4], &t[5], b, C, H, dim, L, Q, stream);
        }));
    });
}

// workspace address and bytes, spin_limit, kernel, chunks_per_item, epoch
ssd_fused_opts opts_of(PyObject *const *a, int32_t *used)
{
    ssd_fused_opts o{};
    o.workspace = pointer(a[0]);
    o.workspace_bytes = (uint64_t)number(a[1]);
    o.spin_limit = (int32_t)number(a[2]);
    o.kernel = (int32_t)number(a[3]);
    o.chunks_per_item = (int32_t)number(a[4]);
    o.epoch = (int32_t)number(a[5]);
    o.used_workspace = used;
    return o;
}

// x, B, dt, dA_cumsum, seq_idx, initial_states, states, out, final_states, clamp, the six of opts_of, stream
// -> (status, used_workspace)
PyObject *fused(PyObject *, PyObject *const *a, Py_ssize_t n)
{
    return guarded(n, 17, [&]() -> PyObject * {
        ssd_tensor t[9];
        for (int i = 0; i < 9; ++i) t[i] = tensor(a[i]);
        const ssd_dims d = dims_of(a[0], a[1], a[2]);
        const int clamp = (int)number(a[9]);
        int32_t used = 0;
        const ssd_fused_opts o = opts_of(a + 10, &used);
        void *const stream = pointer(a[16]);
        const int rc = unlocked([&] {
            return ssd_fused_chunk_state_passing_fwd_ws(&t[0], &t[1], &t[2], &t[3], &t[4], &t[5], &t[6], &t[7], &t[8], &d, clamp, &o, stream);
        });
        return Py_BuildValue("ii", rc, (int)used);
    });
}

// x, B, C, dt, dA_cumsum, seq_idx, initial_states, out, final_states, y, clamp, accumulate, the six of opts_of, stream
// -> (status, used_workspace)
PyObject *fused_scan(PyObject *, PyObject *const *a, Py_ssize_t n)
{
    return guarded(n, 19, [&]() -> PyObject * {
        ssd_tensor t[10];
        for (int i = 0; i < 10; ++i) t[i] = tensor(a[i]);
        const ssd_dims d = dims_of(a[0], a[1], a[3]);
        const int clamp = (int)number(a[10]), accumulate = (int)number(a[11]);
        int32_t used = 0;
        const ssd_fused_opts o = opts_of(a + 12, &used);
        void *const stream = pointer(a[18]);
        const int rc = unlocked([&] {
            return ssd_fused_chunk_state_passing_scan_fwd(&t[0], &t[1], &t[2], &t[3], &t[4], &t[5], &t[6], &t[7], &t[8], &t[9], &d, clamp,
                                                          accumulate, &o, stream);
        });
        return Py_BuildValue("ii", rc, (int)used);
    });
}

// dt, A, dt_bias, dt_out, dA_cumsum, chunk_size, dt_softplus, dt_min, dt_max, stream -> status
PyObject *chunk_cumsum(PyObject *, PyObject *const *a, Py_ssize_t n)
{
    return guarded(n, 10, [&]() -> PyObject * {
        ssd_tensor t[5];
        for (int i = 0; i < 5; ++i) t[i] = tensor(a[i]);
        const at::Tensor &v = unpack(a[0], 3);
        const int32_t b = size32(v.size(0)), L = size32(v.size(1)), H = size32(v.size(2)), Q = size32(number(a[5]));
        const int softplus = (int)number(a[6]);
        const float lo = (float)real(a[7]), hi = (float)real(a[8]);
        void *const stream = pointer(a[9]);
        return PyLong_FromLong(unlocked([&] { return ssd_chunk_cumsum_fwd(&t[0], &t[1], &t[2], &t[3], &t[4], b, L, H, Q, softplus, lo, hi, stream); }));
    });
}

// C, prev_states, dA_cumsum, seq_idx, y, accumulate, stream -> status
PyObject *chunk_scan_states(PyObject *, PyObject *const *a, Py_ssize_t n)
{
    return guarded(n, 7, [&]() -> PyObject * {
        ssd_tensor t[5];
        for (int i = 0; i < 5; ++i) t[i] = tensor(a[i]);
        const at::Tensor &c = unpack(a[0], 4), &s = unpack(a[1], 5), &da = unpack(a[2], 4);
        const ssd_dims d{size32(c.size(0)), size32(c.size(1)), size32(s.size(2)), size32(s.size(3)),
                         size32(c.size(3)), size32(c.size(2)), size32(da.size(3)), size32(s.size(1))};
        const int accumulate = (int)number(a[5]);
        void *const stream = pointer(a[6]);
        return PyLong_FromLong(unlocked([&] { return ssd_chunk_scan_states_fwd(&t[0], &t[1], &t[2], &t[3], &t[4], &d, accumulate, stream); }));
    });
}

// x, B, dt, dA_cumsum, seq_idx, initial_states, out (or None), final_states -> whether the fused call gains from a place for
// fp32 chunk states (arguments it would reject: no, the call itself says so)
PyObject *wants_states(PyObject *, PyObject *const *a, Py_ssize_t n)
{
    return guarded(n, 8, [&]() -> PyObject * {
        ssd_tensor t[8];
        for (int i = 0; i < 8; ++i) t[i] = tensor(a[i]);
        const ssd_dims d = dims_of(a[0], a[1], a[2]);
        return PyBool_FromLong(ssd_query_fused_wants_states(&t[0], &t[1], &t[2], &t[3], &t[4], &t[5], &t[6], &t[7], &d) == 1);
    });
}

#define SSD_METHOD(name) {#name, (PyCFunction)(void (*)(void))name, METH_FASTCALL, nullptr}
PyMethodDef methods[] = {SSD_METHOD(chunk_state), SSD_METHOD(state_passing), SSD_METHOD(fused), SSD_METHOD(fused_scan),
                         SSD_METHOD(chunk_cumsum), SSD_METHOD(chunk_scan_states), SSD_METHOD(wants_states),
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_ssd_host", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__ssd_host(void) { return PyModule_Create(&module); }
