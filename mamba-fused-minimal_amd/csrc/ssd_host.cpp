// Python extension module `_ssd_host`: from tensors to the C entry points of libssd_gfx950.so without a detour through
// ctypes.  Describing nine tensors as ssd_tensor structs field by field from Python takes longer than the kernels of a
// small call do (13 us a fused call, of 27); here the sizes, strides and pointers are read off the tensor objects.
// Nothing is checked or kept here: shapes are the wrappers' business (ssd_amd/ops.py), everything else the library's.
//
// The *_call functions are a wrapper's whole ordinary call in one: plain tensors of the shapes, types and strides that need no
// conversion, outputs allocated here, on the current device and stream.  They return None, and have done nothing, wherever
// anything is out of the ordinary -- other shapes or types, tensor subclasses, several devices, a call that the kernel with a
// kept workspace would serve or that gains from room for chunk states -- and the wrapper goes its general way, which also
// says what is wrong.  A small fused call (2 x 384 tokens x 13 heads) costs the host 12.5 us through the general way and 7 us
// through this one, which is what it takes: its kernel runs 6 us.
#include <Python.h>

#include <torch/csrc/Dtype.h>
#include <torch/csrc/autograd/python_variable.h>

#include <ATen/ops/empty.h>

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

// ---- whole ordinary calls -------------------------------------------------------------------------------------------

struct OutOfTheOrdinary {};      // the general way, then

bool ours(at::ScalarType t) { return t == at::kFloat || t == at::kBFloat16 || t == at::kHalf; }

// A plain dense tensor of `dim` dimensions, none of them empty, on GPU `device`; its last dimension contiguous where asked.
const at::Tensor &plain(PyObject *o, int64_t dim, int64_t device, bool inner = true)
{
    if (!THPVariable_CheckExact(o)) throw OutOfTheOrdinary();
    const at::Tensor &v = THPVariable_Unpack(o);
    if (!v.is_cuda() || v.get_device() != device || v.layout() != at::kStrided || v.dim() != dim || v.numel() == 0 ||
        (inner && v.stride(dim - 1) != 1))
        throw OutOfTheOrdinary();
    return v;
}

void need(bool ok) { if (!ok) throw OutOfTheOrdinary(); }

template <class... N> bool sized(const at::Tensor &v, N... n)
{
    const int64_t want[] = {(int64_t)n...};
    for (size_t i = 0; i < sizeof...(n); ++i)
        if (v.size(i) != want[i]) return false;
    return true;
}

// Memory may have to be mapped, or cached blocks flushed, before an output is there: other Python threads go on meanwhile, as
// they do inside torch.empty.  Where there is none the general way asks again and raises torch.OutOfMemoryError.
at::Tensor made(at::IntArrayRef sizes, at::ScalarType type, const at::Tensor &like)
{
    struct Released {
        PyThreadState *const state = PyEval_SaveThread();
        ~Released() { PyEval_RestoreThread(state); }
    } released;
    try {
        return at::empty(sizes, like.options().dtype(type).requires_grad(false).memory_format(c10::nullopt));
    } catch (const c10::OutOfMemoryError &) {
        throw OutOfTheOrdinary();
    }
}

ssd_tensor described(const at::Tensor &v)
{
    ssd_tensor t{};
    t.dtype = v.scalar_type() == at::kInt ? 0 : v.scalar_type() == at::kFloat ? SSD_F32 : v.scalar_type() == at::kBFloat16 ? SSD_BF16 : SSD_F16;
    t.data = v.data_ptr();
    const auto strides = v.strides();
    for (size_t i = 0; i < strides.size(); ++i) t.stride[i] = strides[i];
    return t;
}

at::ScalarType type_of(PyObject *o)
{
    need(THPDtype_Check(o));
    const at::ScalarType t = ((THPDtype *)o)->scalar_type;
    need(ours(t));
    return t;
}

// seq_idx (b, L) or None
ssd_tensor sequences(PyObject *o, int64_t b, int64_t L, int64_t device)
{
    if (o == Py_None) return ssd_tensor{};
    const at::Tensor &v = plain(o, 2, device, false);
    need(v.scalar_type() == at::kInt && sized(v, b, L));
    return described(v);
}

PyObject *pair_of(const at::Tensor &a, const at::Tensor &b)
{
    PyObject *x = THPVariable_Wrap(a);
    PyObject *y = x ? THPVariable_Wrap(b) : nullptr;
    PyObject *t = y ? PyTuple_Pack(2, x, y) : nullptr;
    Py_XDECREF(x);
    Py_XDECREF(y);
    return t;
}

template <class F>
PyObject *ordinary(Py_ssize_t got, Py_ssize_t want, F &&f)
{
    return guarded(got, want, [&]() -> PyObject * {
        try {
            return f();
        } catch (const OutOfTheOrdinary &) {
            Py_RETURN_NONE;
        }
    });
}

struct Inputs {
    ssd_tensor x, B, dt, dA, seq;
    ssd_dims d;
    const at::Tensor *xv;
};

Inputs inputs(PyObject *Bo, PyObject *xo, PyObject *dto, PyObject *dAo, PyObject *seqo, int64_t device)
{
    const at::Tensor &x = plain(xo, 4, device), &B = plain(Bo, 4, device), &dt = plain(dto, 4, device, false), &dA = plain(dAo, 4, device, false);
    const int64_t b = x.size(0), L = x.size(1), H = x.size(2), G = B.size(2), C = dt.size(2), Q = dt.size(3);
    need(ours(x.scalar_type()) && B.scalar_type() == x.scalar_type() && dt.scalar_type() == at::kFloat && dA.scalar_type() == at::kFloat);
    need(H % G == 0 && B.size(0) == b && B.size(1) == L && sized(dt, b, H, C, Q) && sized(dA, b, H, C, Q) && C == (L + Q - 1) / Q);
    need(b <= INT32_MAX && L <= INT32_MAX && H <= INT32_MAX && x.size(3) <= INT32_MAX && B.size(3) <= INT32_MAX && C <= INT32_MAX && Q <= INT32_MAX);
    return Inputs{described(x), described(B), described(dt), described(dA), sequences(seqo, b, L, device),
                  ssd_dims{(int32_t)b, (int32_t)L, (int32_t)H, (int32_t)x.size(3), (int32_t)B.size(3), (int32_t)G, (int32_t)Q, (int32_t)C}, &x};
}

// B, x, dt, dA_cumsum, out_dtype, initial_states, seq_idx, most (state tile, chunk) pairs, device, stream -> (out, final_states) or None
PyObject *fused_call(PyObject *, PyObject *const *a, Py_ssize_t n)
{
    return ordinary(n, 10, [&]() -> PyObject * {
        const int64_t most = number(a[7]), device = number(a[8]);
        void *const stream = pointer(a[9]);
        // The two refusals that ordinary calls meet return: a throw costs 3 us, and more the first time.  Beyond `most`, the general
        // way's kept workspace may have to grow.
        const at::Tensor &xv = plain(a[1], 4, device);
        if (xv.size(0) * xv.size(2) * ((xv.size(3) + 31) / 32) * plain(a[2], 4, device, false).size(2) > most) Py_RETURN_NONE;
        const at::ScalarType out_type = type_of(a[4]);
        const Inputs in = inputs(a[0], a[1], a[2], a[3], a[6], device);
        const ssd_dims &d = in.d;
        ssd_tensor init{};
        if (a[5] != Py_None) {
            const at::Tensor &v = plain(a[5], 4, device);
            need(ours(v.scalar_type()) && sized(v, d.batch, d.nheads, d.headdim, d.dstate));
            init = described(v);
        }
        // contiguous outputs at a made-up, aligned address, as the allocator will give them
        const int64_t N = d.dstate, P = d.headdim, H = d.nheads, C = d.nchunks;
        void *const somewhere = (void *)(uintptr_t)4096;
        const int code = out_type == at::kFloat ? SSD_F32 : out_type == at::kBFloat16 ? SSD_BF16 : SSD_F16;
        ssd_tensor out{somewhere, code, 0, {C * H * P * N, H * P * N, P * N, N, 1}}, fin{somewhere, SSD_F32, 0, {H * P * N, P * N, N, 1, 0}};
        if (ssd_query_fused_is_plain(&in.x, &in.B, &in.dt, &in.dA, &in.seq, &init, &out, &fin, &d) != 1) Py_RETURN_NONE;
        const at::Tensor out_v = made({d.batch, C, H, P, N}, out_type, *in.xv), fin_v = made({d.batch, H, P, N}, at::kFloat, *in.xv);
        out.data = out_v.data_ptr();
        fin.data = fin_v.data_ptr();
        need(unlocked([&] {
            return ssd_fused_chunk_state_passing_fwd(&in.x, &in.B, &in.dt, &in.dA, &in.seq, &init, nullptr, &out, &fin, &d, 1, stream);
        }) == SSD_OK);
        return pair_of(out_v, fin_v);
    });
}

// B, x, dt, dA_cumsum, seq_idx, states_in_fp32, device, stream -> states or None
PyObject *chunk_state_call(PyObject *, PyObject *const *a, Py_ssize_t n)
{
    return ordinary(n, 8, [&]() -> PyObject * {
        const bool f32 = number(a[5]) != 0;
        const int64_t device = number(a[6]);
        void *const stream = pointer(a[7]);
        const Inputs in = inputs(a[0], a[1], a[2], a[3], a[4], device);
        const ssd_dims &d = in.d;
        const at::Tensor v = made({d.batch, d.nchunks, d.nheads, d.headdim, d.dstate}, f32 ? at::kFloat : in.xv->scalar_type(), *in.xv);
        const ssd_tensor states = described(v);
        need(unlocked([&] { return ssd_chunk_state_fwd(&in.x, &in.B, &in.dt, &in.dA, &in.seq, &states, &d, 1, stream); }) == SSD_OK);
        return THPVariable_Wrap(v);
    });
}

// states, dA_chunk, initial_states, seq_idx, chunk_size (0 without seq_idx), out_dtype (None: that of states), device, stream
// -> (out, final_states) or None
PyObject *state_passing_call(PyObject *, PyObject *const *a, Py_ssize_t n)
{
    return ordinary(n, 8, [&]() -> PyObject * {
        const int64_t Q = number(a[4]), device = number(a[6]);
        void *const stream = pointer(a[7]);
        const at::Tensor &s = plain(a[0], 4, device), &da = plain(a[1], 3, device, false);
        const int64_t b = s.size(0), C = s.size(1), H = s.size(2), dim = s.size(3);
        need(ours(s.scalar_type()) && da.scalar_type() == at::kFloat && sized(da, b, H, C));
        need(b <= INT32_MAX && C <= INT32_MAX && H <= INT32_MAX && dim <= INT32_MAX && Q <= INT32_MAX);
        ssd_tensor init{}, seq{};
        if (a[2] != Py_None) {
            const at::Tensor &v = plain(a[2], 3, device);
            need(ours(v.scalar_type()) && sized(v, b, H, dim));
            init = described(v);
        }
        int64_t L = 0;
        if (a[3] != Py_None) {
            L = plain(a[3], 2, device, false).size(1);
            need(L <= INT32_MAX && Q > 0);
            seq = sequences(a[3], b, L, device);
        }
        const at::ScalarType out_type = a[5] == Py_None ? s.scalar_type() : type_of(a[5]);
        const at::Tensor out_v = made({b, C, H, dim}, out_type, s), fin_v = made({b, H, dim}, at::kFloat, s);
        const ssd_tensor t = described(s), d = described(da), out = described(out_v), fin = described(fin_v);
        need(unlocked([&] {
            return ssd_state_passing_fwd(&t, &d, &init, &seq, &out, &fin, (int32_t)b, (int32_t)C, (int32_t)H, (int32_t)dim, (int32_t)L,
                                         a[3] != Py_None ? (int32_t)Q : 0, stream);
        }) == SSD_OK);
        return pair_of(out_v, fin_v);
    });
}

// dt, A, dt_bias, chunk_size, dt_softplus, dt_min, dt_max, device, stream -> (dA_cumsum, dt_out) or None
PyObject *chunk_cumsum_call(PyObject *, PyObject *const *a, Py_ssize_t n)
{
    return ordinary(n, 9, [&]() -> PyObject * {
        need(PyLong_Check(a[3]));
        const int64_t Q = number(a[3]), device = number(a[7]);
        const int softplus = (int)number(a[4]);
        const float lo = (float)real(a[5]), hi = (float)real(a[6]);
        void *const stream = pointer(a[8]);
        const at::Tensor &dt = plain(a[0], 3, device, false), &A = plain(a[1], 1, device, false);
        const int64_t b = dt.size(0), L = dt.size(1), H = dt.size(2);
        need(ours(dt.scalar_type()) && ours(A.scalar_type()) && A.size(0) == H && Q > 0 && Q <= INT32_MAX);
        need(b <= INT32_MAX && L <= INT32_MAX && H <= INT32_MAX);
        ssd_tensor bias{};
        if (a[2] != Py_None) {
            const at::Tensor &v = plain(a[2], 1, device, false);
            need(ours(v.scalar_type()) && v.size(0) == H);
            bias = described(v);
        }
        const int64_t C = (L + Q - 1) / Q;
        const at::Tensor dt_v = made({b, H, C, Q}, at::kFloat, dt), da_v = made({b, H, C, Q}, at::kFloat, dt);
        const ssd_tensor t = described(dt), At = described(A), out = described(dt_v), da = described(da_v);
        need(unlocked([&] { return ssd_chunk_cumsum_fwd(&t, &At, &bias, &out, &da, (int32_t)b, (int32_t)L, (int32_t)H, (int32_t)Q, softplus, lo, hi, stream); }) ==
             SSD_OK);
        return pair_of(da_v, dt_v);
    });
}

// C, prev_states, dA_cumsum, seq_idx, out_dtype (None: that of C), device, stream -> y or None
PyObject *scan_states_call(PyObject *, PyObject *const *a, Py_ssize_t n)
{
    return ordinary(n, 7, [&]() -> PyObject * {
        const int64_t device = number(a[5]);
        void *const stream = pointer(a[6]);
        const at::Tensor &c = plain(a[0], 4, device), &s = plain(a[1], 5, device), &da = plain(a[2], 4, device, false);
        const int64_t b = c.size(0), L = c.size(1), G = c.size(2), N = c.size(3), C = s.size(1), H = s.size(2), P = s.size(3), Q = da.size(3);
        need(ours(c.scalar_type()) && ours(s.scalar_type()) && da.scalar_type() == at::kFloat);
        need(H % G == 0 && s.size(0) == b && s.size(4) == N && sized(da, b, H, C, Q) && C == (L + Q - 1) / Q);
        need(b <= INT32_MAX && L <= INT32_MAX && H <= INT32_MAX && P <= INT32_MAX && N <= INT32_MAX && C <= INT32_MAX && Q <= INT32_MAX);
        const ssd_tensor seq = sequences(a[3], b, L, device);
        const at::Tensor y = made({b, L, H, P}, a[4] == Py_None ? c.scalar_type() : type_of(a[4]), c);
        const ssd_tensor ct = described(c), st = described(s), dt = described(da), yt = described(y);
        const ssd_dims d{(int32_t)b, (int32_t)L, (int32_t)H, (int32_t)P, (int32_t)N, (int32_t)G, (int32_t)Q, (int32_t)C};
        need(unlocked([&] { return ssd_chunk_scan_states_fwd(&ct, &st, &dt, &seq, &yt, &d, 0, stream); }) == SSD_OK);
        return THPVariable_Wrap(y);
    });
}

#define SSD_METHOD(name) {#name, (PyCFunction)(void (*)(void))name, METH_FASTCALL, nullptr}
PyMethodDef methods[] = {SSD_METHOD(chunk_state), SSD_METHOD(state_passing), SSD_METHOD(fused), SSD_METHOD(fused_scan),
                         SSD_METHOD(chunk_cumsum), SSD_METHOD(chunk_scan_states), SSD_METHOD(wants_states),
                         SSD_METHOD(fused_call), SSD_METHOD(chunk_state_call), SSD_METHOD(state_passing_call), SSD_METHOD(chunk_cumsum_call),
                         SSD_METHOD(scan_states_call),
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_ssd_host", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__ssd_host(void) { return PyModule_Create(&module); }
