// The host path of the Python layer in native code: a CPython module (bitstack_amd/_host.so) over the C ABI.
//
// A decode call is two kernels of 3 to 20 us, and one BitStackLinear.forward spent 25 us on the host in Python (slicing
// the stacked buffers, a dozen property reads per tensor, the workspace table, three context managers, a ctypes call of
// 14 arguments): every call below about 25 us of GPU time ran at the speed of the interpreter.  Here the same checks,
// the output's allocation, the workspace and the launch are one call of METH_FASTCALL.  Whatever is not the ordinary case -
// tensors on the CPU or on two devices, another dtype, non-contiguous tensors, no tokens, no blocks - is answered with None
// and takes the Python path, which converts, or raises its documented errors.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/hip/EmptyTensor.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPGuard.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <map>
#include <memory>
#include <mutex>
#include <utility>
#include <vector>

#include "../../include/bitstack_hip.h"

namespace {

// ---- scratch -----------------------------------------------------------------------------------
// One scratch tensor per (device, stream), grown geometrically.  Kernels on one stream are ordered, so reusing it across
// calls on that stream is safe.  A buffer that is outgrown is never handed back to the allocator: a HIP graph
// captured while it was current has its address baked in, and its replays must keep writing into memory nobody else
// owns.  (A graph captured before a growth still uses the old buffer; it stays correct, it just does not share scratch
// with later eager calls.)  The table lives until the process ends: tensors must not outlive the HIP runtime's tear-down.
// Threads that share a stream share its scratch, and other Python threads run during a call: what a call keeps there between two
// of its kernels is safe because its launches are issued under `launching`.
struct Space {
    at::Tensor buffer;
    std::mutex launching;
};
struct Scratch {
    std::mutex lock;                             // of the table only
    std::map<std::pair<int, hipStream_t>, Space> current;
    std::vector<at::Tensor> retired;
};
Scratch &scratch() {
    static Scratch *s = new Scratch;
    return *s;
}

struct Workspace {
    at::Tensor buffer;
    std::mutex *launching;
    void *data() const { return buffer.mutable_data_ptr(); }
};
// No lock is held through the allocation: it may wait for the device or for the interpreter, and may call back into Python
// (out-of-memory observers, recorded stacks), which may come here again.
Workspace workspace_for(int device, hipStream_t stream, int64_t bytes) {
    Scratch &s = scratch();
    int64_t size = bytes > (1 << 20) ? bytes : (1 << 20);
    {
        std::lock_guard<std::mutex> guard(s.lock);
        Space &space = s.current[{device, stream}];
        const at::Tensor &t = space.buffer;
        if (t.defined() && t.numel() >= bytes) return {t, &space.launching};
        // grow geometrically so that a sequence of slowly growing requests retires few buffers
        if (t.defined() && 2 * t.numel() > size) size = 2 * t.numel();
    }
    at::Tensor fresh = at::empty({size}, at::TensorOptions().dtype(at::kByte).device(at::kCUDA, (c10::DeviceIndex)device));
    std::lock_guard<std::mutex> guard(s.lock);
    Space &space = s.current[{device, stream}];
    at::Tensor &t = space.buffer;
    if (!t.defined() || t.numel() < bytes) {     // (else another thread was quicker on this stream: `fresh` goes back unused)
        if (t.defined()) s.retired.push_back(t);
        t = fresh;
    }
    return {t, &space.launching};
}

// ---- arguments -----------------------------------------------------------------------------------
const at::Tensor *tensor_arg(PyObject *o) { return THPVariable_CheckExact(o) ? &THPVariable_Unpack(o) : nullptr; }

bool plain(const at::Tensor &t, at::ScalarType type, c10::Device dev) {
    return t.scalar_type() == type && t.device() == dev && t.is_contiguous();
}

PyObject *raise_status(int status, const char *what) {
    PyErr_Format(PyExc_RuntimeError, "%s failed with status %d: %s", what, status, bs_error_string(status));
    return nullptr;
}

// The first `blocks` of the stacked buffers of one matrix, if they are what the C ABI takes as they lie.
struct Matrix {
    const uint8_t *q;
    const void *u, *vt;
    int64_t I, M, N, K;
};
bool matrix_args(PyObject *const *a, int64_t blocks, c10::Device dev, Matrix &m) {
    const at::Tensor *q = tensor_arg(a[0]), *u = tensor_arg(a[1]), *vt = tensor_arg(a[2]);
    if (!q || !u || !vt) return false;
    if (!plain(*q, at::kByte, dev) || !plain(*u, at::kHalf, dev) || !plain(*vt, at::kHalf, dev)) return false;
    if (q->dim() != 2 || u->dim() != 3 || vt->dim() != 3) return false;
    m.I = blocks;
    m.M = u->size(1);
    m.K = u->size(2);
    m.N = vt->size(2);
    if (blocks < 1 || blocks > u->size(0) || blocks > vt->size(0) || blocks > q->size(0)) return false;
    if (vt->size(1) != m.K || q->size(1) != (m.M * m.N + 7) / 8) return false;
    m.q = (const uint8_t *)q->const_data_ptr();
    m.u = u->const_data_ptr();
    m.vt = vt->const_data_ptr();
    return m.M > 0 && m.N > 0 && m.M * m.N < ((int64_t)1 << 40) && m.M < INT32_MAX && m.N < INT32_MAX;
}

bool int_arg(PyObject *o, int64_t &v) {
    v = PyLong_AsLongLong(o);
    if (v == -1 && PyErr_Occurred()) return false;
    return true;
}

at::Tensor new_half(at::IntArrayRef sizes, c10::Device dev) {
    return at::Tensor(at::detail::empty_cuda(sizes, at::kHalf, dev, std::nullopt));
}

// The output shape: x's with the last dimension replaced.
c10::SmallVector<int64_t, 6> output_sizes(const at::Tensor &x, int64_t last) {
    c10::SmallVector<int64_t, 6> s(x.sizes().begin(), x.sizes().end());
    s.back() = last;
    return s;
}

// Other Python threads run while a call allocates and launches: with the launch queue full, a launch waits for the device.
// Pointers and sizes are read from the arguments before, and the caller holds the tensors.
struct OtherThreadsRun {
    PyThreadState *state = PyEval_SaveThread();
    OtherThreadsRun() = default;
    OtherThreadsRun(const OtherThreadsRun &) = delete;
    ~OtherThreadsRun() { PyEval_RestoreThread(state); }
};
template <class F>
auto while_others_run(F &&f) {
    OtherThreadsRun scope;
    return f();
}

// A guard only where the tensors' device is not the current one (asking costs less than setting it).
struct DeviceScope {
    c10::hip::OptionalHIPGuard guard;
    explicit DeviceScope(c10::Device dev) {
        if (c10::hip::current_device() != dev.index()) guard.set_index(dev.index());
    }
};

// ---- entry points --------------------------------------------------------------------------------
// Each one's C++ exceptions become the Python errors torch itself raises for them (HANDLE_TH_ERRORS): an allocation that fails is
// torch.OutOfMemoryError, for callers that back off on it.
// forward(qweight, u, vt, blocks, x, bias or None) -> y, or None where the Python path has to take the call
PyObject *host_forward(PyObject *, PyObject *const *a, Py_ssize_t n) {
    if (n != 6) return PyErr_Format(PyExc_TypeError, "forward takes 6 arguments");
    HANDLE_TH_ERRORS
        const at::Tensor *x = tensor_arg(a[4]);
        const at::Tensor *bias = a[5] == Py_None ? nullptr : tensor_arg(a[5]);
        int64_t blocks;
        if (!int_arg(a[3], blocks)) return nullptr;
        Matrix m;
        if (!x || (a[5] != Py_None && !bias) || !x->is_cuda() || x->dim() < 1) Py_RETURN_NONE;
        const c10::Device dev = x->device();
        if (!plain(*x, at::kHalf, dev) || !matrix_args(a, blocks, dev, m)) Py_RETURN_NONE;
        if (x->size(-1) != m.N || x->numel() == 0 || x->numel() / m.N >= INT32_MAX) Py_RETURN_NONE;
        if (bias && (!plain(*bias, at::kHalf, dev) || bias->numel() != m.M)) Py_RETURN_NONE;
        const int T = (int)(x->numel() / m.N);
        const int64_t need = bs_workspace_bytes((int)m.I, (int)m.M, (int)m.N, (int)m.K, T);
        if (need < 0) return raise_status((int)need, "bs_workspace_bytes");
        const void *xp = x->const_data_ptr(), *bp = bias ? bias->const_data_ptr() : nullptr;
        const auto sizes = output_sizes(*x, m.M);
        at::Tensor y;
        const int st = while_others_run([&] {
            DeviceScope scope(dev);
            const hipStream_t stream = c10::hip::getCurrentHIPStream(dev.index()).stream();
            const Workspace ws = workspace_for(dev.index(), stream, need);
            y = new_half(sizes, dev);
            std::lock_guard<std::mutex> launching(*ws.launching);
            return bs_forward(m.q, m.u, m.vt, xp, bp, y.mutable_data_ptr(), (int)m.I, (int)m.M, (int)m.N, (int)m.K, T,
                              ws.data(), ws.buffer.numel(), stream);
        });
        if (st != BS_OK) return raise_status(st, "bs_forward");
        return THPVariable_Wrap(y);
    END_HANDLE_TH_ERRORS
}

// rebuild(qweight, u, vt, blocks) -> w [M, N], or None
PyObject *host_rebuild(PyObject *, PyObject *const *a, Py_ssize_t n) {
    if (n != 4) return PyErr_Format(PyExc_TypeError, "rebuild takes 4 arguments");
    HANDLE_TH_ERRORS
        int64_t blocks;
        if (!int_arg(a[3], blocks)) return nullptr;
        const at::Tensor *u = tensor_arg(a[1]);
        Matrix m;
        if (!u || !u->is_cuda() || !matrix_args(a, blocks, u->device(), m)) Py_RETURN_NONE;
        const c10::Device dev = u->device();
        at::Tensor w;
        const int st = while_others_run([&] {
            DeviceScope scope(dev);
            w = new_half({m.M, m.N}, dev);
            return bs_reconstruct_w(m.q, m.u, m.vt, w.mutable_data_ptr(), (int)m.I, (int)m.M, (int)m.N, (int)m.K,
                                    c10::hip::getCurrentHIPStream(dev.index()).stream());
        });
        if (st != BS_OK) return raise_status(st, "bs_reconstruct_w");
        return THPVariable_Wrap(w);
    END_HANDLE_TH_ERRORS
}

// unpack(qweight [blocks, bytes], blocks, M, N) -> int8 signs [blocks, M, N], or None
PyObject *host_unpack(PyObject *, PyObject *const *a, Py_ssize_t n) {
    if (n != 4) return PyErr_Format(PyExc_TypeError, "unpack takes 4 arguments");
    HANDLE_TH_ERRORS
        const at::Tensor *q = tensor_arg(a[0]);
        int64_t blocks, M, N;
        if (!int_arg(a[1], blocks) || !int_arg(a[2], M) || !int_arg(a[3], N)) return nullptr;
        if (!q || !q->is_cuda() || !plain(*q, at::kByte, q->device()) || q->dim() != 2) Py_RETURN_NONE;
        if (blocks < 1 || blocks > q->size(0) || M < 1 || N < 1 || M >= INT32_MAX || N >= INT32_MAX || M * N % 8 != 0 || q->size(1) != M * N / 8)
            Py_RETURN_NONE;                      // (blocks of whole bytes follow each other without padding)
        const c10::Device dev = q->device();
        const uint8_t *from = (const uint8_t *)q->const_data_ptr();
        at::Tensor s;
        const int st = while_others_run([&] {
            DeviceScope scope(dev);
            s = at::Tensor(at::detail::empty_cuda({blocks, M, N}, at::kChar, dev, std::nullopt));
            return bs_unpack_sign(from, (int8_t *)s.mutable_data_ptr(), blocks * M * N, c10::hip::getCurrentHIPStream(dev.index()).stream());
        });
        if (st != BS_OK) return raise_status(st, "bs_unpack_sign");
        return THPVariable_Wrap(s);
    END_HANDLE_TH_ERRORS
}

// rebuild_from_sign(signs [I, M, N] int8, u, vt, I) -> w [M, N], or None (u and vt may hold more blocks)
PyObject *host_rebuild_from_sign(PyObject *, PyObject *const *a, Py_ssize_t n) {
    if (n != 4) return PyErr_Format(PyExc_TypeError, "rebuild_from_sign takes 4 arguments");
    HANDLE_TH_ERRORS
        const at::Tensor *s = tensor_arg(a[0]), *u = tensor_arg(a[1]), *vt = tensor_arg(a[2]);
        int64_t I;
        if (!int_arg(a[3], I)) return nullptr;
        if (!s || !u || !vt || !u->is_cuda() || s->dim() != 3 || u->dim() != 3 || vt->dim() != 3) Py_RETURN_NONE;
        const c10::Device dev = u->device();
        if (!plain(*s, at::kChar, dev) || !plain(*u, at::kHalf, dev) || !plain(*vt, at::kHalf, dev)) Py_RETURN_NONE;
        const int64_t M = u->size(1), K = u->size(2), N = vt->size(2);
        if (I < 1 || s->size(0) != I || u->size(0) < I || vt->size(0) < I || vt->size(1) != K || s->size(1) != M || s->size(2) != N ||
            M < 1 || N < 1 || M >= INT32_MAX || N >= INT32_MAX)
            Py_RETURN_NONE;
        const int8_t *sp = (const int8_t *)s->const_data_ptr();
        const void *up = u->const_data_ptr(), *vp = vt->const_data_ptr();
        at::Tensor w;
        const int st = while_others_run([&] {
            DeviceScope scope(dev);
            w = new_half({M, N}, dev);
            return bs_reconstruct_w_from_sign(sp, up, vp, w.mutable_data_ptr(), (int)I, (int)M, (int)N, (int)K,
                                              c10::hip::getCurrentHIPStream(dev.index()).stream());
        });
        if (st != BS_OK) return raise_status(st, "bs_reconstruct_w_from_sign");
        return THPVariable_Wrap(w);
    END_HANDLE_TH_ERRORS
}

// linear(x, w, bias or None) -> x @ w^T (+ bias), or None
PyObject *host_linear(PyObject *, PyObject *const *a, Py_ssize_t n) {
    if (n != 3) return PyErr_Format(PyExc_TypeError, "linear takes 3 arguments");
    HANDLE_TH_ERRORS
        const at::Tensor *x = tensor_arg(a[0]), *w = tensor_arg(a[1]);
        const at::Tensor *bias = a[2] == Py_None ? nullptr : tensor_arg(a[2]);
        if (!x || !w || (a[2] != Py_None && !bias) || !x->is_cuda() || x->dim() < 1 || w->dim() != 2) Py_RETURN_NONE;
        const c10::Device dev = x->device();
        if (!plain(*x, at::kHalf, dev) || !plain(*w, at::kHalf, dev)) Py_RETURN_NONE;
        const int64_t M = w->size(0), N = w->size(1);
        if (M < 1 || N < 1 || M >= INT32_MAX || N >= INT32_MAX || x->size(-1) != N || x->numel() == 0 || x->numel() / N >= INT32_MAX) Py_RETURN_NONE;
        if (bias && (!plain(*bias, at::kHalf, dev) || bias->numel() != M)) Py_RETURN_NONE;
        const void *xp = x->const_data_ptr(), *wp = w->const_data_ptr(), *bp = bias ? bias->const_data_ptr() : nullptr;
        const int T = (int)(x->numel() / N);
        const auto sizes = output_sizes(*x, M);
        at::Tensor y;
        const int st = while_others_run([&] {
            DeviceScope scope(dev);
            y = new_half(sizes, dev);
            return bs_linear_f16(xp, wp, bp, y.mutable_data_ptr(), T, (int)M, (int)N, c10::hip::getCurrentHIPStream(dev.index()).stream());
        });
        if (st != BS_OK) return raise_status(st, "bs_linear_f16");
        return THPVariable_Wrap(y);
    END_HANDLE_TH_ERRORS
}

// forward_cat(x [T, N], qweight, u, vt, blocks, qweight, ..) -> y [T, M0 + M1 + ..], or None.  Whether the matrices run as one
// product is asked first, from sizes alone.
PyObject *host_forward_cat(PyObject *, PyObject *const *a, Py_ssize_t n) {
    const int count = (int)(n - 1) / 4;
    if (n < 5 || (n - 1) % 4 != 0 || count > BS_MAX_GROUP) return PyErr_Format(PyExc_TypeError, "forward_cat takes x and four arguments a matrix");
    HANDLE_TH_ERRORS
        const at::Tensor *x = tensor_arg(a[0]);
        if (!x || !x->is_cuda() || x->dim() != 2 || x->size(0) < 1 || x->size(0) >= INT32_MAX || x->size(1) >= INT32_MAX) Py_RETURN_NONE;
        const c10::Device dev = x->device();
        const int T = (int)x->size(0), N = (int)x->size(1);
        bs_matrix mats[BS_MAX_GROUP] = {};
        int64_t blocks[BS_MAX_GROUP], K = 0, rows = 0;
        for (int j = 0; j < count; j++) {
            const at::Tensor *u = tensor_arg(a[1 + 4 * j + 1]);
            if (!u || u->dim() != 3) Py_RETURN_NONE;
            if (!int_arg(a[1 + 4 * j + 3], blocks[j])) return nullptr;
            if (j == 0) K = u->size(2);
            if (u->size(2) != K || u->size(1) >= INT32_MAX || K >= INT32_MAX || blocks[j] > u->size(0)) Py_RETURN_NONE;
            mats[j].I = (int32_t)blocks[j];
            mats[j].M = (int32_t)u->size(1);
            rows += mats[j].M;
        }
        const int64_t need = bs_forward_cat_workspace_bytes(mats, count, N, (int)K, T);
        if (need <= 0 || !plain(*x, at::kHalf, dev)) Py_RETURN_NONE;
        for (int j = 0; j < count; j++) {
            Matrix m;
            if (!matrix_args(a + 1 + 4 * j, blocks[j], dev, m) || m.N != N) Py_RETURN_NONE;
            mats[j].packed = m.q;
            mats[j].u = m.u;
            mats[j].vt = m.vt;
        }
        const void *xp = x->const_data_ptr();
        at::Tensor y;
        const int st = while_others_run([&] {
            DeviceScope scope(dev);
            const hipStream_t stream = c10::hip::getCurrentHIPStream(dev.index()).stream();
            const Workspace ws = workspace_for(dev.index(), stream, need);
            y = new_half({T, rows}, dev);
            std::lock_guard<std::mutex> launching(*ws.launching);
            return bs_forward_cat(mats, count, N, (int)K, xp, T, y.mutable_data_ptr(), ws.data(), ws.buffer.numel(), stream);
        });
        if (st != BS_OK) return raise_status(st, "bs_forward_cat");
        return THPVariable_Wrap(y);
    END_HANDLE_TH_ERRORS
}

// workspace(device index, nbytes) -> the scratch tensor of the device's current stream
PyObject *host_workspace(PyObject *, PyObject *const *a, Py_ssize_t n) {
    if (n != 2) return PyErr_Format(PyExc_TypeError, "workspace takes 2 arguments");
    HANDLE_TH_ERRORS
        int64_t dev, bytes;
        if (!int_arg(a[0], dev) || !int_arg(a[1], bytes)) return nullptr;
        return THPVariable_Wrap(while_others_run([&] {
            return workspace_for((int)dev, c10::hip::getCurrentHIPStream((c10::DeviceIndex)dev).stream(), bytes).buffer;
        }));
    END_HANDLE_TH_ERRORS
}

// hold(device index, nbytes) -> (scratch tensor, key): as workspace(), with the stream's launches kept to this thread until let_go(key)
PyObject *host_hold(PyObject *, PyObject *const *a, Py_ssize_t n) {
    if (n != 2) return PyErr_Format(PyExc_TypeError, "hold takes 2 arguments");
    HANDLE_TH_ERRORS
        int64_t dev, bytes;
        if (!int_arg(a[0], dev) || !int_arg(a[1], bytes)) return nullptr;
        const Workspace ws = while_others_run([&] {
            const Workspace w = workspace_for((int)dev, c10::hip::getCurrentHIPStream((c10::DeviceIndex)dev).stream(), bytes);
            w.launching->lock();
            return w;
        });
        PyObject *t = THPVariable_Wrap(ws.buffer), *key = PyLong_FromVoidPtr(ws.launching), *pair = t && key ? PyTuple_Pack(2, t, key) : nullptr;
        Py_XDECREF(t);
        Py_XDECREF(key);
        if (!pair) ws.launching->unlock();
        return pair;
    END_HANDLE_TH_ERRORS
}
PyObject *host_let_go(PyObject *, PyObject *const *a, Py_ssize_t n) {
    if (n != 1) return PyErr_Format(PyExc_TypeError, "let_go takes 1 argument");
    std::mutex *m = (std::mutex *)PyLong_AsVoidPtr(a[0]);
    if (!m) return PyErr_Occurred() ? nullptr : PyErr_Format(PyExc_ValueError, "let_go takes what hold gave");
    m->unlock();
    Py_RETURN_NONE;
}

// ---- a decode step's launches as one call -----------------------------------------------------------
// The launches between the embedding and the last norm never change between steps: their arguments are laid
// out once (make_steps) and issued in one call (run_steps) - nine kernels per layer at the cost of the launches alone.
// The tensors behind the pointers are kept alive by the caller, who also lays the list out again when one is replaced.
struct Step {
    enum Kind { GROUP, ATTENTION, NORM } kind;
    // GROUP
    std::vector<bs_matrix> mats;
    int N, K, T, epilogue, rms;
    float eps;
    const void *x, *residual;
    void *y;
    // ATTENTION
    const void *qkv, *cos, *sin;
    void *kcache, *vcache, *out;
    const int64_t *pos;
    int B, heads, kv_heads, head_dim, max_len;
    // NORM: y[T, N] = RMSNorm of x with this weight vector
    const void *weight;
};
struct Steps {
    std::vector<Step> list;
    int64_t need = 0;
};
const char *const STEPS = "bitstack_amd.steps";
void free_steps(PyObject *cap) { delete (Steps *)PyCapsule_GetPointer(cap, STEPS); }

// make_steps([("group", address of bs_matrix[n], n, N, K, x, T, eps or None, epilogue, residual or 0, y) |
//             ("attention", qkv, kcache, vcache, cos, sin, pos, out, B, heads, kv_heads, head_dim, max_len) |
//             ("norm", x, weight, y, T, H, eps), ...]) -> handle; every tensor as its address
PyObject *host_make_steps(PyObject *, PyObject *const *a, Py_ssize_t n) {
    if (n != 1 || !PyList_Check(a[0])) return PyErr_Format(PyExc_TypeError, "make_steps takes a list");
    HANDLE_TH_ERRORS
    std::unique_ptr<Steps> steps(new Steps);
    for (Py_ssize_t j = 0; j < PyList_GET_SIZE(a[0]); j++) {
        PyObject *t = PyList_GET_ITEM(a[0], j);
        Step s = {};
        const char *kind = PyTuple_Check(t) && PyTuple_GET_SIZE(t) > 0 ? PyUnicode_AsUTF8(PyTuple_GET_ITEM(t, 0)) : nullptr;
        bool ok = kind != nullptr;
        unsigned long long p[7] = {0, 0, 0, 0, 0, 0, 0};
        if (ok && kind[0] == 'g') {
            PyObject *eps;
            int count;
            s.kind = Step::GROUP;
            ok = PyArg_ParseTuple(t, "sKiiiKiOiKK", &kind, &p[0], &count, &s.N, &s.K, &p[1], &s.T, &eps, &s.epilogue, &p[2], &p[3]) &&
                 count >= 1 && count <= BS_MAX_GROUP;
            if (ok) {
                const bs_matrix *m = (const bs_matrix *)(uintptr_t)p[0];
                s.mats.assign(m, m + count);
                s.rms = eps != Py_None;
                s.eps = s.rms ? (float)PyFloat_AsDouble(eps) : 0.f;
                s.x = (const void *)(uintptr_t)p[1];
                s.residual = (const void *)(uintptr_t)p[2];
                s.y = (void *)(uintptr_t)p[3];
                const int64_t need = bs_forward_group_workspace_bytes(s.mats.data(), count, s.N, s.K, s.T);
                if (need < 0) return raise_status((int)need, "bs_forward_group_workspace_bytes");
                if (need > steps->need) steps->need = need;
            }
        } else if (ok && kind[0] == 'n') {
            s.kind = Step::NORM;
            ok = PyArg_ParseTuple(t, "sKKKiif", &kind, &p[0], &p[1], &p[2], &s.T, &s.N, &s.eps);
            s.x = (const void *)(uintptr_t)p[0];
            s.weight = (const void *)(uintptr_t)p[1];
            s.y = (void *)(uintptr_t)p[2];
        } else if (ok) {
            s.kind = Step::ATTENTION;
            ok = PyArg_ParseTuple(t, "sKKKKKKKiiiii", &kind, &p[0], &p[1], &p[2], &p[3], &p[4], &p[5], &p[6], &s.B, &s.heads, &s.kv_heads,
                                  &s.head_dim, &s.max_len);
            s.qkv = (const void *)(uintptr_t)p[0];
            s.kcache = (void *)(uintptr_t)p[1];
            s.vcache = (void *)(uintptr_t)p[2];
            s.cos = (const void *)(uintptr_t)p[3];
            s.sin = (const void *)(uintptr_t)p[4];
            s.pos = (const int64_t *)(uintptr_t)p[5];
            s.out = (void *)(uintptr_t)p[6];
            const int64_t need = ok ? bs_attention_decode_workspace_bytes(s.B, s.heads, s.kv_heads, s.head_dim, s.max_len) : 0;
            if (need > steps->need) steps->need = need;      // (a shape that is not taken is reported by the call)
        }
        if (!ok || PyErr_Occurred()) {
            if (!PyErr_Occurred()) PyErr_Format(PyExc_ValueError, "make_steps: item %zd is not a launch", j);
            return nullptr;
        }
        steps->list.push_back(std::move(s));
    }
    PyObject *handle = PyCapsule_New(steps.get(), STEPS, free_steps);
    if (handle) steps.release();                 // (the capsule's from here)
    return handle;
    END_HANDLE_TH_ERRORS
}

// run_steps(handle, device index): every launch, in order, on the device's current stream
PyObject *host_run_steps(PyObject *, PyObject *const *a, Py_ssize_t n) {
    if (n != 2) return PyErr_Format(PyExc_TypeError, "run_steps takes 2 arguments");
    HANDLE_TH_ERRORS
        Steps *steps = (Steps *)PyCapsule_GetPointer(a[0], STEPS);
        int64_t index;
        if (!steps || !int_arg(a[1], index)) return nullptr;
        const c10::Device dev(c10::kCUDA, (c10::DeviceIndex)index);
        const char *what = nullptr;
        const int st = while_others_run([&] {
            int st = BS_OK;
            DeviceScope scope(dev);
            const hipStream_t stream = c10::hip::getCurrentHIPStream(dev.index()).stream();
            Workspace ws = workspace_for(dev.index(), stream, steps->need);
            // one launch pair at a time: nothing is kept in the scratch from one to the next
            auto issue = [&](const Step &s) {
                std::lock_guard<std::mutex> launching(*ws.launching);
                if (s.kind == Step::GROUP) {
                    what = "bs_forward_group";
                    return s.rms ? bs_forward_group_rms(s.mats.data(), (int)s.mats.size(), s.N, s.K, s.x, s.T, s.eps, s.epilogue, s.residual,
                                                        s.y, ws.data(), ws.buffer.numel(), stream)
                                 : bs_forward_group(s.mats.data(), (int)s.mats.size(), s.N, s.K, s.x, s.T, s.epilogue, s.residual, s.y,
                                                    ws.data(), ws.buffer.numel(), stream);
                }
                if (s.kind == Step::NORM) {
                    what = "bs_rmsnorm_f16";
                    return bs_rmsnorm_f16(s.x, s.weight, s.y, s.T, s.N, s.eps, stream);
                }
                what = "bs_attention_decode_f16";
                return bs_attention_decode_ws_f16(s.qkv, s.kcache, s.vcache, s.cos, s.sin, s.pos, s.out, s.B, s.heads, s.kv_heads, s.head_dim,
                                                  s.max_len, ws.data(), ws.buffer.numel(), stream);
            };
            for (const Step &s : steps->list) {
                st = issue(s);
                if (st == BS_ERR_WORKSPACE && s.kind == Step::GROUP) {
                    // another kernel has been chosen since (bs_set_decode_kernel): its scratch may be larger
                    ws = workspace_for(dev.index(), stream, bs_forward_group_workspace_bytes(s.mats.data(), (int)s.mats.size(), s.N, s.K, s.T));
                    st = issue(s);
                }
                if (st != BS_OK) break;
            }
            return st;
        });
        if (st != BS_OK) return raise_status(st, what);
        Py_RETURN_NONE;
    END_HANDLE_TH_ERRORS
}

// argmax(x [B, V], out int64 [B] [, pos int64, one element: += 1]) -> True, or None
PyObject *host_argmax(PyObject *, PyObject *const *a, Py_ssize_t n) {
    if (n != 2 && n != 3) return PyErr_Format(PyExc_TypeError, "argmax takes 2 or 3 arguments");
    HANDLE_TH_ERRORS
        const at::Tensor *x = tensor_arg(a[0]), *out = tensor_arg(a[1]), *pos = n == 3 ? tensor_arg(a[2]) : nullptr;
        if (!x || !out || (n == 3 && !pos) || !x->is_cuda() || x->dim() != 2) Py_RETURN_NONE;
        const c10::Device dev = x->device();
        if (!plain(*x, at::kHalf, dev) || !plain(*out, at::kLong, dev) || out->numel() != x->size(0) || x->numel() == 0 ||
            x->size(0) >= INT32_MAX || x->size(1) >= INT32_MAX || (pos && (!plain(*pos, at::kLong, dev) || pos->numel() != 1)))
            Py_RETURN_NONE;
        const void *xp = x->const_data_ptr();
        int64_t *op = (int64_t *)out->mutable_data_ptr(), *pp = pos ? (int64_t *)pos->mutable_data_ptr() : nullptr;
        const int B = (int)x->size(0), V = (int)x->size(1);
        const int st = while_others_run([&] {
            DeviceScope scope(dev);
            return bs_argmax_advance_f16(xp, op, pp, B, V, c10::hip::getCurrentHIPStream(dev.index()).stream());
        });
        if (st != BS_OK) return raise_status(st, "bs_argmax_advance_f16");
        Py_RETURN_TRUE;
    END_HANDLE_TH_ERRORS
}

#define HOST_METHOD(name) {#name, (PyCFunction)(void (*)(void))host_##name, METH_FASTCALL, nullptr}
PyMethodDef methods[] = {HOST_METHOD(forward), HOST_METHOD(rebuild), HOST_METHOD(unpack), HOST_METHOD(rebuild_from_sign), HOST_METHOD(linear), HOST_METHOD(forward_cat), HOST_METHOD(workspace),
                         HOST_METHOD(hold), HOST_METHOD(let_go), HOST_METHOD(argmax), HOST_METHOD(make_steps), HOST_METHOD(run_steps), {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_host", "Native host path over libbitstack_hip.so.", -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__host(void) { return PyModule_Create(&module); }
