// The host side of the kernel calls that a serving step makes once per layer (Ops.decode, Ops.append_decode and
// Ops.write): the argument checks of kushkash_amd/_ops.py and the library call in one native function. In
// Python they cost ~16 us a call, more than the launch of a small step itself (one sequence of 333 tokens: 9 us).
//
// Each function returns the library's code, or NOT_TAKEN for anything that is not the plain, valid case -- a
// tensor subclass or one without storage, a wrong type, shape, stride, device or alignment, an option it does not
// know. The caller then takes its Python path, which makes the same checks and raises the errors. Every pointer is
// read before the GIL is released: data_ptr() throws for a tensor without storage (what torch.vmap passes is of
// type torch.Tensor too), and a thrown exception must find the thread state in place.
#include <Python.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cstdint>

#include "kushkash_amd.h"

namespace {

constexpr long NOT_TAKEN = 1;            // the library's codes are 0 or negative
constexpr int64_t PAGE = 32;

// The entry points, as the public header declares them: a changed argument list does not compile here
using DecodeFn = decltype(&kush_decode_ex);
using AppendDecodeFn = decltype(&kush_append_decode);
using WriteFn = decltype(&kush_write_ex);

// What one Ops is built for
struct Config {
    int64_t D;
    int bits, G, dtype;                  // dtype: the library's code
    at::ScalarType type;
    c10::DeviceIndex device;
    int32_t* sync;
    DecodeFn decode;
    AppendDecodeFn append_decode;
    WriteFn write;
};

const char* const CAPSULE = "kushkash_amd.config";

// A plain tensor on the config's device, or null
const at::Tensor* tensor(const Config& c, PyObject* o) {
    if (!THPVariable_CheckExact(o)) return nullptr;
    const at::Tensor& t = THPVariable_Unpack(o);
    return t.defined() && t.is_cuda() && t.get_device() == c.device && t.layout() == c10::kStrided ? &t : nullptr;
}

const at::Tensor* index32(const Config& c, PyObject* o, int64_t least) {
    const at::Tensor* t = tensor(c, o);
    return t && t->scalar_type() == at::kInt && t->is_contiguous() && t->numel() >= least ? t : nullptr;
}

// k / v rows [rows, H, D], unit dim stride, head stride D
const at::Tensor* rows(const Config& c, PyObject* o, int64_t H) {
    const at::Tensor* t = tensor(c, o);
    return t && t->dim() == 3 && t->size(1) == H && t->size(2) == c.D && t->stride(2) == 1 && t->stride(1) == c.D &&
                   t->scalar_type() == c.type
               ? t
               : nullptr;
}

template <typename T>
T* ptr(const at::Tensor& t) { return static_cast<T*>(t.data_ptr()); }

// The paged cache of H kv heads; block_table of `seqs` rows, `cols` pages each
struct Cache {
    void *cache, *tail;
    const int32_t* table;
    int64_t bs, hs, H, seqs, cols, row;
    bool take(const Config& c, PyObject* oc, PyObject* ot, PyObject* ok) {
        const at::Tensor *tc = tensor(c, oc), *tt = tensor(c, ot), *tk = tensor(c, ok);
        if (!tc || !tt || !tk || tk->dim() != 4 || tc->dim() < 2 || tt->dim() != 2) return false;
        const int64_t e = tc->element_size();
        H = tk->size(1);
        bs = tc->stride(0) * e;
        hs = tc->stride(1) * e;
        seqs = tt->size(0);
        cols = tt->size(1);
        row = tt->stride(0);
        if (tc->size(1) < H || tk->size(2) != PAGE || tk->size(3) != c.D || !tk->is_contiguous() ||
            tk->scalar_type() != c.type || tt->scalar_type() != at::kInt || tt->stride(1) != 1)
            return false;
        cache = tc->data_ptr();
        tail = tk->data_ptr();
        table = ptr<int32_t>(*tt);
        return (((uint64_t)(uintptr_t)cache | (uint64_t)bs | (uint64_t)hs) & 15) == 0;
    }
};

const Config* config(PyObject* o) { return static_cast<const Config*>(PyCapsule_GetPointer(o, CAPSULE)); }

bool integer(PyObject* o, int64_t& x) {
    if (!PyLong_CheckExact(o)) return false;
    int over = 0;
    x = PyLong_AsLongLongAndOverflow(o, &over);
    return over == 0;
}

// args: config, k, v (None: decode alone), q, out, cache, block_table, seq_lens, tail_idx, tail_k, scale, n_splits,
// work, waves, order, rot, sync slots, stream
long decode(PyObject* const* a) {
    const Config& c = *config(a[0]);
    Cache s;
    int64_t ns, waves, slots, stream;
    if (!s.take(c, a[5], a[6], a[9]) || !integer(a[11], ns) || !integer(a[13], waves) || !integer(a[16], slots) ||
        !integer(a[17], stream) || !PyBool_Check(a[15]) || !PyFloat_CheckExact(a[10]))
        return NOT_TAKEN;
    const at::Tensor *q = tensor(c, a[3]), *out = tensor(c, a[4]);
    const int64_t H = s.H;
    if (!q || !out || q->dim() != 3 || q->size(1) != H * c.G || q->size(2) != c.D || !q->is_contiguous() ||
        q->scalar_type() != c.type || out->sizes() != q->sizes() || !out->is_contiguous() || out->scalar_type() != c.type)
        return NOT_TAKEN;
    const int64_t S = q->size(0), rows_ = S * H * ns * c.G;
    const at::Tensor *lens = index32(c, a[7], S), *tidx = index32(c, a[8], S);
    if (!lens || !tidx || s.seqs < S || ns < 1 || ns > (1 << 20) || waves < 0 || waves > 8 || S > INT32_MAX ||
        H > INT32_MAX)
        return NOT_TAKEN;
    float *ml = nullptr, *po = nullptr;
    if (ns > 1) {                                     // merged in the launch, or left to the caller
        const at::Tensor* w = a[12] == Py_None ? nullptr : tensor(c, a[12]);
        if (!w || w->scalar_type() != at::kFloat || !w->is_contiguous() || w->numel() < rows_ * (c.D + 2) ||
            S * H * ((c.G + 15) / 16) > slots)
            return NOT_TAKEN;
        ml = ptr<float>(*w);
        po = ml + 2 * rows_;
    }
    const at::Tensor* order = a[14] == Py_None ? nullptr : index32(c, a[14], S);
    if (a[14] != Py_None && !order) return NOT_TAKEN;
    const int32_t cols = (int32_t)std::min<int64_t>(s.cols, 1 << 30);
    int32_t* const sync = ns > 1 ? c.sync : nullptr;
    const int32_t* const ord = order ? ptr<int32_t>(*order) : nullptr;
    const float scale = (float)PyFloat_AS_DOUBLE(a[10]);
    const int rot = a[15] == Py_True;
    const void* const pq = q->data_ptr();
    void* const pout = out->data_ptr();
    const int32_t *const ptidx = ptr<int32_t>(*tidx), *const plens = ptr<int32_t>(*lens);
    if (a[1] == Py_None) {
        int rc;
        Py_BEGIN_ALLOW_THREADS;
        rc = c.decode(c.D, c.bits, c.G, c.dtype, pq, pout, s.cache, s.bs, s.hs, s.tail, ptidx, s.table, plens, s.row, H,
                      scale, ns, ml, po, S, (void*)stream, cols, sync, waves, ord, rot);
        Py_END_ALLOW_THREADS;
        return rc;
    }
    const at::Tensor *k = rows(c, a[1], H), *v = rows(c, a[2], H);
    if (!k || !v || k->size(0) < S || v->size(0) < S || c.G > 16) return NOT_TAKEN;
    const uint64_t e = k->element_size();
    const void *const pk = k->data_ptr(), *const pv = v->data_ptr();
    const int64_t ks = k->stride(0), vs = v->stride(0);
    if (((uint64_t)(uintptr_t)pk | (uint64_t)(uintptr_t)pv | ks * e | vs * e) & 15) return NOT_TAKEN;
    int rc;
    Py_BEGIN_ALLOW_THREADS;
    rc = c.append_decode(c.D, c.bits, c.G, c.dtype, pq, pout, s.cache, s.bs, s.hs, s.tail, ptidx, s.table, plens, s.row, H,
                         scale, ns, ml, po, S, (void*)stream, pk, pv, ks, vs, cols, sync, waves, ord, rot);
    Py_END_ALLOW_THREADS;
    return rc;
}

// args: config, k, v, query_start_loc, seq_lens, tail_idx, job_seq, job_page, cache, block_table, tail_k, rot, stream:
// the one-launch write (mode 2)
long write(PyObject* const* a) {
    const Config& c = *config(a[0]);
    Cache s;
    int64_t stream;
    const at::Tensor* k = tensor(c, a[1]);
    if (!k || k->dim() != 3 || !integer(a[12], stream) || !PyBool_Check(a[11])) return NOT_TAKEN;
    const int64_t H = k->size(1);
    const at::Tensor* v = rows(c, a[2], H);
    if (!rows(c, a[1], H) || !v || !s.take(c, a[8], a[9], a[10]) || s.H != H) return NOT_TAKEN;
    const at::Tensor *qsl = index32(c, a[3], 0), *lens = index32(c, a[4], 0), *tidx = index32(c, a[5], 0),
                     *js = index32(c, a[6], 1), *jp = index32(c, a[7], 1);
    if (!qsl || !lens || !tidx || !js || !jp || js->numel() != jp->numel() || js->numel() > INT32_MAX || H > INT32_MAX)
        return NOT_TAKEN;
    const void *const pk = k->data_ptr(), *const pv = v->data_ptr();
    const int32_t *const pqsl = ptr<int32_t>(*qsl), *const plens = ptr<int32_t>(*lens), *const ptidx = ptr<int32_t>(*tidx),
                  *const pjs = ptr<int32_t>(*js), *const pjp = ptr<int32_t>(*jp);
    const int64_t ks = k->stride(0), vs = v->stride(0), jobs = js->numel();
    const int rot = a[11] == Py_True;
    int rc;
    Py_BEGIN_ALLOW_THREADS;
    rc = c.write(c.D, c.bits, c.dtype, pk, pv, ks, vs, pqsl, plens, ptidx, pjs, pjp, jobs, 2, s.cache, s.bs, s.hs, s.tail,
                 s.table, s.row, H, (void*)stream, rot);
    Py_END_ALLOW_THREADS;
    return rc;
}

// A tensor without storage throws on its pointer, with the GIL held: not taken either
template <long (*F)(PyObject* const*), int N>
PyObject* entry(PyObject*, PyObject* const* args, Py_ssize_t n) {
    long rc = NOT_TAKEN;
    if (n != N || !PyCapsule_IsValid(args[0], CAPSULE)) {
        PyErr_SetString(PyExc_TypeError, "kushkash_amd._fastcall: bad arguments");
        return nullptr;
    }
    try {
        rc = F(args);
    } catch (...) {
        PyErr_Clear();
    }
    return PyLong_FromLong(rc);
}

// make_config(D, bits, G, dtype code, device index, sync pointer, decode, append_decode, write function addresses)
PyObject* make_config(PyObject*, PyObject* args) {
    long long D, sync, f[3];
    int bits, G, dtype, device;
    if (!PyArg_ParseTuple(args, "LiiiiLLLL", &D, &bits, &G, &dtype, &device, &sync, &f[0], &f[1], &f[2])) return nullptr;
    const at::ScalarType type = dtype == 0 ? at::kFloat : (dtype == 1 ? at::kHalf : at::kBFloat16);
    auto* c = new Config{D, bits, G, dtype, type, (c10::DeviceIndex)device, (int32_t*)sync, (DecodeFn)f[0],
                         (AppendDecodeFn)f[1], (WriteFn)f[2]};
    return PyCapsule_New(c, CAPSULE, [](PyObject* o) { delete static_cast<Config*>(PyCapsule_GetPointer(o, CAPSULE)); });
}

PyMethodDef methods[] = {
    {"make_config", make_config, METH_VARARGS, nullptr},
    {"decode", (PyCFunction)(void (*)(void))entry<decode, 18>, METH_FASTCALL, nullptr},
    {"write", (PyCFunction)(void (*)(void))entry<write, 13>, METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_fastcall", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__fastcall(void) {
    PyObject* m = PyModule_Create(&module);
    if (m) PyModule_AddIntConstant(m, "NOT_TAKEN", NOT_TAKEN);
    if (m) PyModule_AddIntConstant(m, "ABI", KUSH_FASTCALL_ABI);      // the library's revision it was built for
    return m;
}
