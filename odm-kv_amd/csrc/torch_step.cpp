// kvquant._native: the decode step's host path over torch tensors (a CPython extension).
//
// A decode step of one layer is 2 kernel launches of together 18 us at 32k tokens, and a model has the host run it once per
// layer and token: what the host adds (argument checks, views, the output tensor, ctypes, bookkeeping) has to stay below
// that.  In Python these were 20 us of a 31 us layer step; here they are about 2.
#include <Python.h>
#include <structmember.h>
#include <stdlib.h>
#include <string.h>
#include <ATen/ATen.h>
#include <torch/csrc/autograd/python_variable.h>

#include "../../include/odmkv.h"

namespace {

typedef int (*step_fn)(const odmkv_step_t*, const void*, const void*, const void*, int64_t, int64_t, int, void*, float*, void*);

at::ScalarType scalar_of(int code) {
    return code == ODMKV_F16 ? at::kHalf : code == ODMKV_BF16 ? at::kBFloat16 : at::kFloat;
}

struct Step {
    PyObject_HEAD
    odmkv_step_t st;
    step_fn fn;
    PyObject* keep;             // what the block's pointers point into
    long long seq_len;          // tokens the store holds
    long long room;             // exact tokens that can still be appended without touching the host's tables
    long long appended;         // since this object was made
    unsigned long long stream;  // the workspace belongs to it
    int Hkv, device;
    int attends;                // whether an attention call may append its token (the press keeps new tokens exact)
};

PyObject* s_sliding = nullptr; PyObject* s_softcap = nullptr; PyObject* s_aux = nullptr; PyObject* s_scaling = nullptr;

int step_init(PyObject* self_, PyObject* args, PyObject*) {
    Step* self = (Step*)self_;
    unsigned long long fn, store, work, ops, pi_v, cb, cb_host, inv, ws, ws_bytes, stream;
    int B, Hq, Hkv, q_dt, out_dt, device, attends;
    double scaling;
    long long seq_len, room;
    PyObject* keep;
    if (!PyArg_ParseTuple(args, "KKKKKKKKKKKiiiiiidpLLO", &fn, &store, &work, &ops, &pi_v, &cb, &cb_host, &inv, &ws, &ws_bytes, &stream,
                          &B, &Hq, &Hkv, &q_dt, &out_dt, &device, &scaling, &attends, &seq_len, &room, &keep))
        return -1;
    if (!fn || !store || !work || B <= 0 || Hkv <= 0 || Hq % Hkv || q_dt < 0 || q_dt > 2 || out_dt < 0 || out_dt > 2) {
        PyErr_SetString(PyExc_ValueError, "Step: bad arguments");
        return -1;
    }
    self->fn = (step_fn)(uintptr_t)fn;
    odmkv_step_t& s = self->st;
    s.store = (const odmkv_packed_t*)(uintptr_t)store;
    s.work = (const odmkv_worklist_t*)(uintptr_t)work;
    s.pi_k_ops = (const uint16_t*)(uintptr_t)ops;
    s.pi_v = (const float*)(uintptr_t)pi_v;
    s.codebooks = (const float*)(uintptr_t)cb;
    s.codebooks_host = (const float*)(uintptr_t)cb_host;
    s.inv_scales = (const float*)(uintptr_t)inv;
    s.workspace = (void*)(uintptr_t)ws;
    s.workspace_bytes = (size_t)ws_bytes;
    s.B = B; s.Hq = Hq; s.q_dtype = q_dt; s.out_dtype = out_dt; s.scaling = (float)scaling;
    self->stream = stream; self->Hkv = Hkv; self->device = device; self->attends = attends;
    self->seq_len = seq_len; self->room = room; self->appended = 0;
    Py_INCREF(keep);
    Py_XSETREF(self->keep, keep);
    return 0;
}

void step_dealloc(PyObject* self) {
    Py_XDECREF(((Step*)self)->keep);
    Py_TYPE(self)->tp_free(self);
}

bool query_fits(const Step* s, const at::Tensor& q) {
    const odmkv_step_t& st = s->st;
    return q.is_cuda() && q.get_device() == s->device && q.scalar_type() == scalar_of(st.q_dtype) && q.is_contiguous()
           && q.numel() == (int64_t)st.B * st.Hq * ODMKV_HEAD_DIM && q.dim() >= 3 && q.size(0) == st.B && q.size(1) == st.Hq;
}

// Append the last token of keys / values [B, Hkv, n, 128] and attend with query; nullptr and no Python error: this call is
// not what the block was made for, nothing was done.
PyObject* run(Step* s, const at::Tensor& q, const at::Tensor& k, const at::Tensor& v, double scaling, unsigned long long stream) {
    const odmkv_step_t& st = s->st;
    if (s->room <= 0 || (float)scaling != st.scaling || stream != s->stream) return nullptr;
    if (!query_fits(s, q)) return nullptr;
    const at::ScalarType exact = scalar_of(st.store->exact_dtype);
    if (k.dim() != 4 || v.dim() != 4 || k.scalar_type() != exact || v.scalar_type() != exact || !k.is_cuda() || !v.is_cuda()
        || k.get_device() != s->device || v.get_device() != s->device)
        return nullptr;
    const auto ks = k.sizes(), kt = k.strides(), vt = v.strides();
    if (ks != v.sizes() || ks[0] != st.B || ks[1] != s->Hkv || ks[2] < 1 || ks[3] != ODMKV_HEAD_DIM) return nullptr;
    if (kt[3] != 1 || vt[3] != 1 || kt[0] != vt[0] || kt[1] != vt[1]) return nullptr;
    const char* kp = (const char*)k.data_ptr() + (ks[2] - 1) * kt[2] * 2;
    const char* vp = (const char*)v.data_ptr() + (ks[2] - 1) * vt[2] * 2;
    at::Tensor out = at::empty({st.B, 1, st.Hq, ODMKV_HEAD_DIM}, q.options().dtype(scalar_of(st.out_dtype)));
    const int rc = s->fn(&st, q.data_ptr(), kp, vp, kt[0], kt[1], (int)s->seq_len, out.data_ptr(), nullptr, (void*)(uintptr_t)stream);
    if (rc) return PyErr_Format(rc == ODMKV_EHIP ? PyExc_RuntimeError : PyExc_ValueError, "odmkv: decode step failed (code %d)", rc);
    s->seq_len += 1; s->room -= 1; s->appended += 1;
    return THPVariable_Wrap(std::move(out));
}

#define GUARDED(body)                                                  \
    try { body } catch (const std::exception& e) {                     \
        PyErr_SetString(PyExc_RuntimeError, e.what());                 \
        return nullptr;                                                \
    }

// step(query, keys, values, scaling, stream): one new token; [B, 1, Hq, 128], or None if the block does not fit the call
PyObject* step_step(PyObject* self, PyObject* const* a, Py_ssize_t n) {
    if (n != 5 || !THPVariable_Check(a[0]) || !THPVariable_Check(a[1]) || !THPVariable_Check(a[2])) {
        PyErr_SetString(PyExc_TypeError, "step(query, keys, values, scaling, stream)");
        return nullptr;
    }
    const double scaling = PyFloat_AsDouble(a[3]);
    const unsigned long long stream = PyLong_AsUnsignedLongLong(a[4]);
    if (PyErr_Occurred()) return nullptr;
    GUARDED(
        const at::Tensor& k = THPVariable_Unpack(a[1]);
        PyObject* out = k.dim() == 4 && k.size(2) == 1 ? run((Step*)self, THPVariable_Unpack(a[0]), k, THPVariable_Unpack(a[2]), scaling, stream) : nullptr;
        if (!out && !PyErr_Occurred()) Py_RETURN_NONE;
        return out;
    )
}

// attend(query, keys, values, kwargs, stream): an attention call of a model over the store; None: not a call for the block
PyObject* step_attend(PyObject* self, PyObject* const* a, Py_ssize_t n) {
    if (n != 5 || !THPVariable_Check(a[0]) || !THPVariable_Check(a[1]) || !THPVariable_Check(a[2]) || !PyDict_Check(a[3])) {
        PyErr_SetString(PyExc_TypeError, "attend(query, keys, values, kwargs, stream)");
        return nullptr;
    }
    Step* s = (Step*)self;
    if (!s->attends) Py_RETURN_NONE;
    for (PyObject* name : {s_sliding, s_softcap, s_aux}) {
        PyObject* x = PyDict_GetItem(a[3], name);
        if (x && x != Py_None) Py_RETURN_NONE;
    }
    double scaling = 0.08838834764831845;                     // 128 ** -0.5
    PyObject* sc = PyDict_GetItem(a[3], s_scaling);
    if (sc && sc != Py_None) scaling = PyFloat_AsDouble(sc);
    const unsigned long long stream = PyLong_AsUnsignedLongLong(a[4]);
    if (PyErr_Occurred()) return nullptr;
    const char* off = getenv("ODMKV_FUSED_DECODE");
    if (off && strcmp(off, "0") == 0) Py_RETURN_NONE;
    GUARDED(
        const at::Tensor& q = THPVariable_Unpack(a[0]);
        const at::Tensor& k = THPVariable_Unpack(a[1]);
        // one query token, and the dense length (or that of its aliased views) one ahead of the store's
        if (q.dim() != 4 || q.size(2) != 1 || k.dim() != 4 || k.size(2) != s->seq_len + 1 || s->st.q_dtype != s->st.out_dtype) Py_RETURN_NONE;
        PyObject* out = run(s, q, k, THPVariable_Unpack(a[2]), scaling, stream);
        if (!out && !PyErr_Occurred()) Py_RETURN_NONE;
        return out;
    )
}

// look(query, scaling, stream): attention alone, nothing appended; [B, Hq, 128], or None if the block does not fit the call
PyObject* step_look(PyObject* self, PyObject* const* a, Py_ssize_t n) {
    if (n != 3 || !THPVariable_Check(a[0])) {
        PyErr_SetString(PyExc_TypeError, "look(query, scaling, stream)");
        return nullptr;
    }
    const double scaling = PyFloat_AsDouble(a[1]);
    const unsigned long long stream = PyLong_AsUnsignedLongLong(a[2]);
    if (PyErr_Occurred()) return nullptr;
    GUARDED(
        Step* s = (Step*)self;
        const odmkv_step_t& st = s->st;
        const at::Tensor& q = THPVariable_Unpack(a[0]);
        if (!query_fits(s, q) || (float)scaling != st.scaling || stream != s->stream) Py_RETURN_NONE;
        at::Tensor out = at::empty({st.B, st.Hq, ODMKV_HEAD_DIM}, q.options().dtype(scalar_of(st.out_dtype)));
        const int rc = s->fn(&st, q.data_ptr(), nullptr, nullptr, 0, 0, 0, out.data_ptr(), nullptr, (void*)(uintptr_t)stream);
        if (rc) return PyErr_Format(rc == ODMKV_EHIP ? PyExc_RuntimeError : PyExc_ValueError, "odmkv: decode attention failed (code %d)", rc);
        return THPVariable_Wrap(std::move(out));
    )
}

PyMethodDef step_methods[] = {
    {"step", (PyCFunction)(void*)step_step, METH_FASTCALL, nullptr},
    {"look", (PyCFunction)(void*)step_look, METH_FASTCALL, nullptr},
    {"attend", (PyCFunction)(void*)step_attend, METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr}};
PyMemberDef step_members[] = {
    {"seq_len", T_LONGLONG, offsetof(Step, seq_len), READONLY, nullptr},
    {"room", T_LONGLONG, offsetof(Step, room), READONLY, nullptr},
    {"appended", T_LONGLONG, offsetof(Step, appended), READONLY, nullptr},
    {nullptr, 0, 0, 0, nullptr}};

PyTypeObject StepType = {PyVarObject_HEAD_INIT(nullptr, 0)};

PyObject* alias_both(const at::Tensor& keys, const at::Tensor& values, long long length) {
    const at::Tensor* both[2] = {&keys, &values};
    for (const at::Tensor* t : both)
        if (t->dim() != 4 || t->size(2) < 1) return PyErr_Format(PyExc_ValueError, "alias: [B, H, n, D] tensors with a token at least");
    at::Tensor view[2];
    for (int i = 0; i < 2; ++i) {
        const auto z = both[i]->sizes(); const auto r = both[i]->strides();
        view[i] = both[i]->as_strided({z[0], z[1], length, z[3]}, {r[0], r[1], 0, r[3]}, both[i]->storage_offset() + (z[2] - 1) * r[2]);
    }
    PyObject* out = PyTuple_New(2);
    if (out)
        for (int i = 0; i < 2; ++i) PyTuple_SET_ITEM(out, i, THPVariable_Wrap(std::move(view[i])));
    return out;
}

// alias(keys, values, length): [B, H, n, D] each -> stride-0 views [B, H, length, D] of the last token
PyObject* native_alias(PyObject*, PyObject* const* a, Py_ssize_t n) {
    if (n != 3 || !THPVariable_Check(a[0]) || !THPVariable_Check(a[1])) {
        PyErr_SetString(PyExc_TypeError, "alias(keys, values, length)");
        return nullptr;
    }
    const long long length = PyLong_AsLongLong(a[2]);
    if (PyErr_Occurred()) return nullptr;
    GUARDED(
        return alias_both(THPVariable_Unpack(a[0]), THPVariable_Unpack(a[1]), length);
    )
}

PyMethodDef module_methods[] = {
    {"alias", (PyCFunction)(void*)native_alias, METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module_def = {PyModuleDef_HEAD_INIT, "_native", nullptr, -1, module_methods};

}  // namespace

PyMODINIT_FUNC PyInit__native(void) {
    s_sliding = PyUnicode_InternFromString("sliding_window"); s_softcap = PyUnicode_InternFromString("softcap");
    s_aux = PyUnicode_InternFromString("s_aux"); s_scaling = PyUnicode_InternFromString("scaling");
    StepType.tp_name = "kvquant._native.Step";
    StepType.tp_basicsize = sizeof(Step);
    StepType.tp_flags = Py_TPFLAGS_DEFAULT;
    StepType.tp_new = PyType_GenericNew;
    StepType.tp_init = step_init;
    StepType.tp_dealloc = step_dealloc;
    StepType.tp_methods = step_methods;
    StepType.tp_members = step_members;
    if (PyType_Ready(&StepType) < 0) return nullptr;
    PyObject* m = PyModule_Create(&module_def);
    if (!m) return nullptr;
    Py_INCREF(&StepType);
    if (PyModule_AddObject(m, "Step", (PyObject*)&StepType) < 0) { Py_DECREF(&StepType); Py_DECREF(m); return nullptr; }
    return m;
}
