// Native host side of the torch-facing calls (CPython extension, one per process).
//
// A decode step of one layer is 20 to 45 us of GPU work in three to five launches; issued from Python through
// ctypes (some 45 arguments a call, three allocations, three dtype conversions) it took 60 us of host time
// and the GPU waited.  Here a Layer keeps what rarely changes from step to step (plans, cache views,
// widths, layouts, scale); the owner asks it (holds) whether it still is what its attributes say and makes another one
// if not.  One call per layer checks the three tensors that do change, takes scratch from the owner's
// workspace, allocates the output and issues the launches.
//
// Every entry returns None for a call outside the shapes, types and strides it knows.  The Python caller
// then goes its general way, which converts what can be converted and raises where it has to.
//
// What torch throws (out of memory, a tensor without storage, no device) becomes a Python exception at each
// entry: an exception that leaves a C function would end the process.
#include <Python.h>

#include <ATen/ATen.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/utils/object_ptr.h>

#include "../../include/bgtq.h"

namespace {

constexpr int D = BGTQ_HEAD_DIM;
PyObject* g_error = nullptr;          // blockgtq_amd._capi.BgtqError
PyObject* g_note_path = nullptr;      // ops._note_path(layer geometry): warns once where the generic kernel ran
PyObject* g_buf_name = nullptr;       // "_buf"

const at::Tensor* tensor(PyObject* o) { return THPVariable_Check(o) ? &THPVariable_Unpack(o) : nullptr; }

bool as_int(PyObject* o, int64_t& v) {
    if (!PyLong_Check(o)) return false;
    v = PyLong_AsLongLong(o);
    if (v == -1 && PyErr_Occurred()) { PyErr_Clear(); return false; }
    return true;
}

PyObject* fail(const char* what, int rc) {
    PyErr_Format(g_error ? g_error : PyExc_RuntimeError, "%s failed: %s (code %d)", what, bgtq_strerror(rc), rc);
    return nullptr;
}

void* stream_of(const at::Tensor& t) { return (void*)c10::hip::getCurrentHIPStream(t.get_device()).stream(); }

// fp16 or bf16 values of the layer's device, last dim contiguous
bool is_x(const at::Tensor& t, c10::DeviceIndex dev) {
    const auto st = t.scalar_type();
    return (st == at::kHalf || st == at::kBFloat16) && t.is_cuda() && t.get_device() == dev && t.stride(-1) == 1;
}
bool is_index(const at::Tensor& t, c10::DeviceIndex dev, int64_t n) {
    return t.scalar_type() == at::kInt && t.is_cuda() && t.get_device() == dev && t.numel() == n && t.is_contiguous();
}

int default_splits(int B, int n_kv, int64_t T, bool ragged) {
    return (ragged ? bgtq_ragged_splits : bgtq_default_splits)(B, n_kv, (int)(T > 1 ? T : 1));
}

// At least `floats` fp32 values of the workspace object's buffer, grown as ops.Workspace grows it.
// The partial vectors come first and are read 16 bytes at a time (allocations start on 512-byte boundaries).
bool workspace(PyObject* ws, int64_t floats, const at::Tensor& like, at::Tensor& buf) {
    PyObject* o = PyObject_GetAttr(ws, g_buf_name);
    if (!o) return false;
    const at::Tensor* have = tensor(o);
    if (have && have->numel() >= floats && have->device() == like.device()) {
        buf = *have;
        Py_DECREF(o);
        return true;
    }
    Py_DECREF(o);
    buf = at::empty({floats}, like.options().dtype(at::kFloat));
    PyObject* fresh = THPVariable_Wrap(buf);
    if (!fresh) return false;
    const int rc = PyObject_SetAttr(ws, g_buf_name, fresh);
    Py_DECREF(fresh);
    return rc == 0;
}

// ------------------------------------------------------------------------------------------------ Layer
struct Layer {
    PyObject_HEAD
    at::Tensor *plans, *kp, *kn, *vp, *vn, *bk, *bv;
    bgtq_step s;                       // everything that stays from step to step
    int baked;                         // queries arrive rotated
    int64_t capacity;                  // tokens the cache views hold
    int64_t batch;
    c10::DeviceIndex dev;
    int path_seen;
};

void layer_dealloc(PyObject* self) {
    Layer* L = (Layer*)self;
    for (at::Tensor* t : {L->plans, L->kp, L->kn, L->vp, L->vn, L->bk, L->bv}) delete t;
    Py_TYPE(self)->tp_free(self);
}

// Layer(plans, k_packed, k_norms, v_packed, v_norms, k_row_width, norm_width, v_row_width, n_q,
//       k_layout, v_layout, scale, baked, buf_k or None, buf_v or None)
PyObject* layer_new(PyTypeObject* type, PyObject* args, PyObject*) {
    HANDLE_TH_ERRORS
    PyObject *o[7];
    int kw, nw, vw, n_q, kl, vl, baked;
    float scale;
    if (!PyArg_ParseTuple(args, "OOOOOiiiiiifpOO", &o[0], &o[1], &o[2], &o[3], &o[4], &kw, &nw, &vw, &n_q, &kl, &vl,
                          &scale, &baked, &o[5], &o[6])) return nullptr;
    const at::Tensor* t[7];
    for (int i = 0; i < 7; i++) t[i] = tensor(o[i]);
    for (int i = 0; i < 5; i++)
        if (!t[i] || !t[i]->is_cuda()) { PyErr_SetString(PyExc_TypeError, "Layer: the plans and the cache live on the GPU"); return nullptr; }
    if (t[1]->dim() != 4 || t[2]->dim() != 4 || t[3]->dim() != 4 || t[4]->dim() != 3 || t[1]->scalar_type() != at::kByte ||
        t[3]->scalar_type() != at::kByte || t[2]->scalar_type() != at::kHalf || t[4]->scalar_type() != at::kHalf ||
        t[1]->stride(3) != 1 || t[2]->stride(3) != 1 || t[3]->stride(3) != 1 || (!t[5] != !t[6]) ||
        n_q % t[1]->size(1)) {
        PyErr_SetString(PyExc_ValueError, "Layer: cache views have unexpected shapes or types");
        return nullptr;
    }
    Layer* L = (Layer*)type->tp_alloc(type, 0);
    if (!L) return nullptr;
    at::Tensor** dst[7] = {&L->plans, &L->kp, &L->kn, &L->vp, &L->vn, &L->bk, &L->bv};
    THPObjectPtr owner((PyObject*)L);                // (freed should one of the tensors have no storage)
    // (aliases: they keep the storage, and stay what they are if someone gives the tensor another one)
    for (int i = 0; i < 7; i++) *dst[i] = t[i] ? new at::Tensor(t[i]->detach()) : nullptr;
    bgtq_step& s = L->s;
    s = bgtq_step{};
    s.plans = (const bgtq_head_plan*)t[0]->data_ptr();
    s.n_kv = (int)t[1]->size(1);
    s.gqa = n_q / s.n_kv;
    s.k_layout = kl; s.v_layout = vl;
    s.k_packed = t[1]->data_ptr(); s.kp_sb = t[1]->stride(0); s.kp_sh = t[1]->stride(1); s.kp_st = t[1]->stride(2);
    s.k_norms = t[2]->data_ptr();  s.kn_sb = t[2]->stride(0); s.kn_sh = t[2]->stride(1); s.kn_st = t[2]->stride(2);
    s.v_packed = t[3]->data_ptr(); s.vp_sb = t[3]->stride(0); s.vp_sh = t[3]->stride(1); s.vp_st = t[3]->stride(2);
    s.v_norms = t[4]->data_ptr();  s.vn_sb = t[4]->stride(0); s.vn_sh = t[4]->stride(1); s.vn_st = t[4]->stride(2);
    s.k_row_width = kw; s.norm_width = nw; s.v_row_width = vw; s.scale = scale;
    L->baked = baked;
    L->capacity = std::min(std::min(t[1]->size(2), t[2]->size(2)), std::min(t[3]->size(2), t[4]->size(2)));
    s.max_T = (int)L->capacity;
    L->batch = std::min(std::min(t[1]->size(0), t[2]->size(0)), std::min(t[3]->size(0), t[4]->size(0)));
    L->dev = t[1]->get_device();
    if (t[5]) {
        s.win_k = t[5]->data_ptr(); s.win_v = t[6]->data_ptr();
        s.w_sb = t[5]->stride(0); s.w_sh = t[5]->stride(1); s.w_st = t[5]->stride(2);
        s.win_W = (int)t[5]->size(2);
    }
    return owner.release();
    END_HANDLE_TH_ERRORS
}

// Whether o is `have`, or holds it at index li of a leading dimension: the same memory, type, sizes and strides
bool is_view(const at::Tensor* have, PyObject* o, int64_t li) {
    const at::Tensor* t = tensor(o);
    if (!t || !have) return o == Py_None && !have;
    const int64_t more = t->dim() - have->dim();
    if (more != 0 && more != 1) return false;
    if (t->scalar_type() != have->scalar_type() || t->sizes().slice(more) != have->sizes() || t->strides().slice(more) != have->strides()) return false;
    const char* at = (const char*)t->data_ptr() + (more ? li * t->stride(0) * (int64_t)t->element_size() : 0);
    return at == (const char*)have->data_ptr() && (!more || (li >= 0 && li < t->size(0)));
}

// holds(li, the constructor's arguments, tensors of all layers in the place of one layer's where there are such):
// whether this handle is what the constructor would make of them
PyObject* layer_holds(PyObject* self, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    Layer* L = (Layer*)self;
    const bgtq_step& s = L->s;
    if (n != 16) { PyErr_SetString(PyExc_TypeError, "holds() takes a layer index and the arguments of Layer()"); return nullptr; }
    int64_t li, v[6];
    bool same = as_int(a[0], li);
    for (int i = 0; i < 6; i++) same = same && as_int(a[6 + i], v[i]);
    same = same && v[0] == s.k_row_width && v[1] == s.norm_width && v[2] == s.v_row_width && v[3] == (int64_t)s.n_kv * s.gqa &&
           v[4] == s.k_layout && v[5] == s.v_layout;
    const double scale = PyFloat_AsDouble(a[12]);
    if (scale == -1.0 && PyErr_Occurred()) return nullptr;
    const int baked = PyObject_IsTrue(a[13]);
    if (baked < 0) return nullptr;
    same = same && (float)scale == s.scale && baked == L->baked;
    const at::Tensor* have[7] = {L->plans, L->kp, L->kn, L->vp, L->vn, L->bk, L->bv};
    for (int i = 0; i < 7; i++) same = same && is_view(have[i], a[i < 5 ? 1 + i : 9 + i], li);
    return PyBool_FromLong(same);
    END_HANDLE_TH_ERRORS
}

// k, v and (may be null) q of one step into s; false: not for this path
bool take_inputs(const Layer* L, bgtq_step& s, const at::Tensor* q, const at::Tensor* k, const at::Tensor* v) {
    if (!k || !v || k->dim() != 4 || v->dim() != 4 || !is_x(*k, L->dev) || !is_x(*v, L->dev)) return false;
    if (k->scalar_type() != v->scalar_type() || k->sizes() != v->sizes()) return false;
    if (k->size(1) != s.n_kv || k->size(3) != D || k->size(0) > L->batch || k->size(0) < 1 || k->size(2) < 1) return false;
    s.B = (int)k->size(0);
    s.S = (int)k->size(2);
    s.x_dtype = k->scalar_type() == at::kBFloat16 ? BGTQ_X_BF16 : BGTQ_X_FP16;
    s.k = k->data_ptr(); s.k_sb = k->stride(0); s.k_sh = k->stride(1); s.k_ss = k->stride(2);
    s.v = v->data_ptr(); s.v_sb = v->stride(0); s.v_sh = v->stride(1); s.v_ss = v->stride(2);
    if (q) {
        if (q->dim() != 4 || !is_x(*q, L->dev) || q->size(0) != s.B || q->size(1) != (int64_t)s.n_kv * s.gqa || q->size(2) != 1 ||
            q->size(3) != D || q->scalar_type() != k->scalar_type()) return false;
        if (L->baked && q->scalar_type() != at::kHalf) return false;
        s.q = q->data_ptr(); s.q_sb = q->stride(0); s.q_sh = q->stride(1);
    }
    return true;
}

// an int position, or one int32 device value per row
bool take_position(const Layer* L, bgtq_step& s, PyObject* o) {
    int64_t at = 0;
    if (as_int(o, at)) {
        if (at < 0 || at + s.S > L->capacity) return false;
        s.t_pos_scalar = (int)at;
        return true;
    }
    const at::Tensor* t = tensor(o);
    if (!t || !is_index(*t, L->dev, s.B)) return false;
    s.t_pos = t->data_ptr<int32_t>();
    return true;
}

PyObject* finish_step(Layer* L, bgtq_step& s, int64_t T, int64_t n_splits, PyObject* ws, bool windowed) {
    if (T < 0 || T > L->capacity) Py_RETURN_NONE;
    const int64_t n_q = (int64_t)s.n_kv * s.gqa, rows = s.B * n_q;
    if (n_splits <= 0) n_splits = default_splits(s.B, s.n_kv, T, s.seq_lens != nullptr);
    s.T = (int)T;
    s.n_splits = (int)n_splits;
    // [partial vectors | partial lse | rotated queries | with a buffer: its partial, the tokens that leave]
    const int64_t vec = rows * n_splits * D, lse = (rows * n_splits + 3) & ~(int64_t)3, rot = rows * D / 2;
    const int64_t win = windowed ? rows * D + ((rows + 3) & ~(int64_t)3) + (int64_t)s.B * s.n_kv * D : 0;
    at::Tensor buf;
    if (!workspace(ws, vec + lse + rot + win, *L->kp, buf)) return nullptr;
    float* at = buf.data_ptr<float>();
    s.partial_out = at; at += vec;
    s.partial_lse = at; at += lse;
    if (!L->baked || windowed) s.q_rot = at;
    at += rot;
    if (windowed) {
        s.win_out = at; at += rows * D;
        s.win_lse = at; at += (rows + 3) & ~(int64_t)3;
        s.win_old = at;
    } else {
        s.win_k = s.win_v = nullptr;
    }
    at::Tensor out = at::empty({s.B, n_q, 1, D}, L->kp->options().dtype(at::kHalf));
    s.out = out.data_ptr();
    void* st = stream_of(*L->kp);
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = bgtq_decode_step(&s, st);
    Py_END_ALLOW_THREADS
    if (rc != BGTQ_OK) return fail("bgtq_decode_step", rc);
    if (!L->path_seen) {
        L->path_seen = 1;
        PyObject* r = PyObject_CallFunction(g_note_path, "iiLLLii", s.n_kv, s.gqa, (long long)s.kp_st, (long long)s.vp_st,
                                            (long long)s.kn_st, s.k_layout, s.v_layout);
        if (!r) return nullptr;
        Py_DECREF(r);
    }
    return THPVariable_Wrap(std::move(out));
}

// step(q, k, v, t_pos, T, seq_lens or None, n_splits, quant_mode, workspace)
PyObject* layer_step(PyObject* self, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    Layer* L = (Layer*)self;
    int64_t T, n_splits, quant;
    if (n != 9 || !as_int(a[4], T) || !as_int(a[6], n_splits) || !as_int(a[7], quant)) Py_RETURN_NONE;
    bgtq_step s = L->s;
    const at::Tensor* q = tensor(a[0]);
    if (!q || !take_inputs(L, s, q, tensor(a[1]), tensor(a[2])) || !take_position(L, s, a[3])) Py_RETURN_NONE;
    if (a[5] != Py_None) {
        const at::Tensor* lens = tensor(a[5]);
        if (!lens || !is_index(*lens, L->dev, s.B)) Py_RETURN_NONE;
        s.seq_lens = lens->data_ptr<int32_t>();
    }
    s.quant_mode = (int)quant;
    return finish_step(L, s, T, n_splits, a[8], false);
    END_HANDLE_TH_ERRORS
}

// step_window(q, k, v, slot, t_flush, packed_len, buf_len, T, n_splits, quant_mode, workspace)
PyObject* layer_step_window(PyObject* self, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    Layer* L = (Layer*)self;
    int64_t T, n_splits, quant;
    if (n != 11 || !L->bk || !as_int(a[7], T) || !as_int(a[8], n_splits) || !as_int(a[9], quant)) Py_RETURN_NONE;
    bgtq_step s = L->s;
    const at::Tensor* q = tensor(a[0]);
    if (!q || !take_inputs(L, s, q, tensor(a[1]), tensor(a[2])) || s.S != 1) Py_RETURN_NONE;
    const at::Tensor* idx[4];
    for (int i = 0; i < 4; i++) {
        idx[i] = tensor(a[3 + i]);
        if (!idx[i] || !is_index(*idx[i], L->dev, s.B)) Py_RETURN_NONE;
    }
    s.win_slot = idx[0]->data_ptr<int32_t>();
    s.t_pos = idx[1]->data_ptr<int32_t>();
    s.seq_lens = idx[2]->data_ptr<int32_t>();
    s.win_lens = idx[3]->data_ptr<int32_t>();
    s.quant_mode = (int)quant;
    return finish_step(L, s, T, n_splits, a[10], true);
    END_HANDLE_TH_ERRORS
}

// encode(k, v, t_pos, quant_mode) -> True
PyObject* layer_encode(PyObject* self, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    Layer* L = (Layer*)self;
    int64_t quant;
    if (n != 4 || !as_int(a[3], quant)) Py_RETURN_NONE;
    bgtq_step s = L->s;
    if (!take_inputs(L, s, nullptr, tensor(a[0]), tensor(a[1])) || !take_position(L, s, a[2])) Py_RETURN_NONE;
    s.quant_mode = (int)quant;
    void* st = stream_of(*L->kp);
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = bgtq_encode_kv(&s, st);
    Py_END_ALLOW_THREADS
    if (rc != BGTQ_OK) return fail("bgtq_encode_kv", rc);
    Py_RETURN_TRUE;
    END_HANDLE_TH_ERRORS
}

PyMethodDef layer_methods[] = {
    {"holds", (PyCFunction)(void*)layer_holds, METH_FASTCALL, "whether this is the handle of these arguments"},
    {"step", (PyCFunction)(void*)layer_step, METH_FASTCALL, "one decode step of this layer, or None"},
    {"step_window", (PyCFunction)(void*)layer_step_window, METH_FASTCALL, "one decode step in with-buffer mode, or None"},
    {"encode", (PyCFunction)(void*)layer_encode, METH_FASTCALL, "append k and v, True or None"},
    {nullptr, nullptr, 0, nullptr}};

PyTypeObject LayerType = {PyVarObject_HEAD_INIT(nullptr, 0)};

// ------------------------------------------------------------------------------- attention without append
// attend(plans, q_rot (B, n_q, 1, D) or (B, n_q, D), k_packed, k_norms, v_packed, v_norms, T, n_splits,
//        k_layout, v_layout, scale, unrotate, workspace) -> fp16 of q's shape, or None
PyObject* attend(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    int64_t T, n_splits, kl, vl, unrotate;
    if (n != 13 || !as_int(a[6], T) || !as_int(a[7], n_splits) || !as_int(a[8], kl) || !as_int(a[9], vl) ||
        !PyFloat_Check(a[10]) || !as_int(a[11], unrotate)) Py_RETURN_NONE;
    const at::Tensor* t[6];
    for (int i = 0; i < 6; i++) {
        t[i] = tensor(a[i]);
        if (!t[i] || !t[i]->is_cuda()) Py_RETURN_NONE;
    }
    const at::Tensor &plans = *t[0], &q = *t[1], &kp = *t[2], &kn = *t[3], &vp = *t[4], &vn = *t[5];
    for (int i = 0; i < 6; i++)
        if (t[i]->get_device() != q.get_device()) Py_RETURN_NONE;
    const bool four = q.dim() == 4;
    if ((q.dim() != 3 && !(four && q.size(2) == 1)) || q.scalar_type() != at::kHalf || q.stride(-1) != 1 || q.size(-1) != D) Py_RETURN_NONE;
    if (kp.dim() != 4 || kn.dim() != 4 || vp.dim() != 4 || vn.dim() != 3 || kp.scalar_type() != at::kByte || vp.scalar_type() != at::kByte ||
        kn.scalar_type() != at::kHalf || vn.scalar_type() != at::kHalf || kp.stride(3) != 1 || vp.stride(3) != 1 || kn.stride(3) != 1) Py_RETURN_NONE;
    const int64_t B = q.size(0), n_q = q.size(1), n_kv = kp.size(1);
    if (B < 1 || n_kv < 1 || n_q % n_kv || kp.size(2) < T || vp.size(2) < T || T < 0) Py_RETURN_NONE;
    if (n_splits <= 0) n_splits = default_splits((int)B, (int)n_kv, T, false);
    const int64_t vec = B * n_q * n_splits * D;
    at::Tensor buf;
    if (!workspace(a[12], vec + B * n_q * n_splits, q, buf)) return nullptr;
    float *po = buf.data_ptr<float>(), *pl = po + vec;
    at::Tensor out = four ? at::empty({B, n_q, 1, D}, q.options()) : at::empty({B, n_q, D}, q.options());
    void* st = stream_of(q);
    const bgtq_head_plan* P = (const bgtq_head_plan*)plans.data_ptr();
    const int gqa = (int)(n_q / n_kv);
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = bgtq_decode_attn(P, q.data_ptr(), q.stride(0), q.stride(1),
                          kp.data_ptr(), kp.stride(0), kp.stride(1), kp.stride(2), (int)kp.size(3),
                          kn.data_ptr(), kn.stride(0), kn.stride(1), kn.stride(2),
                          vp.data_ptr(), vp.stride(0), vp.stride(1), vp.stride(2), (int)vp.size(3),
                          vn.data_ptr(), vn.stride(0), vn.stride(1), vn.stride(2),
                          nullptr, (int)T, (int)B, (int)n_kv, gqa, (int)n_splits, po, pl, (int)kl, (int)vl,
                          (float)PyFloat_AS_DOUBLE(a[10]), st);
    if (rc == BGTQ_OK)
        rc = bgtq_lse_reduce(P, po, pl, (int)n_splits, nullptr, nullptr, 0, (int)B, (int)n_kv, gqa, (int)unrotate,
                             out.data_ptr(), n_q * D, D, nullptr, st);
    Py_END_ALLOW_THREADS
    if (rc != BGTQ_OK) return fail("bgtq_decode_attn", rc);
    if (bgtq_last_decode_path() == 1) {                     // (the hook warns once per geometry)
        PyObject* r = PyObject_CallFunction(g_note_path, "iiLLLii", (int)n_kv, gqa, (long long)kp.stride(2), (long long)vp.stride(2),
                                            (long long)kn.stride(2), (int)kl, (int)vl);
        if (!r) return nullptr;
        Py_DECREF(r);
    }
    return THPVariable_Wrap(std::move(out));
    END_HANDLE_TH_ERRORS
}

// ------------------------------------------------------------------------------------------ prompt phase
// prompt(plans, q (B, n_q, S, D), rotate_q, k_packed, k_norms, v_packed, v_norms, T, k_row_width, v_row_width,
//        q_pos_offset, is_causal, k_layout, v_layout, scale, unrotate) -> (B, n_q, S, D) fp16, or None
PyObject* prompt(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    int64_t rotate, T, kw, vw, off, causal, kl, vl, unrotate;
    if (n != 16 || !as_int(a[2], rotate) || !as_int(a[7], T) || !as_int(a[8], kw) || !as_int(a[9], vw) || !as_int(a[10], off) ||
        !as_int(a[11], causal) || !as_int(a[12], kl) || !as_int(a[13], vl) || !PyFloat_Check(a[14]) || !as_int(a[15], unrotate)) Py_RETURN_NONE;
    const at::Tensor* t[6];
    const int at6[6] = {0, 1, 3, 4, 5, 6};
    for (int i = 0; i < 6; i++) {
        t[i] = tensor(a[at6[i]]);
        if (!t[i] || !t[i]->is_cuda()) Py_RETURN_NONE;
    }
    const at::Tensor &plans = *t[0], &q = *t[1], &kp = *t[2], &kn = *t[3], &vp = *t[4], &vn = *t[5];
    for (int i = 0; i < 6; i++)
        if (t[i]->get_device() != q.get_device()) Py_RETURN_NONE;
    if (q.dim() != 4 || !is_x(q, q.get_device()) || q.size(3) != D || (!rotate && q.scalar_type() != at::kHalf)) Py_RETURN_NONE;
    if (kp.dim() != 4 || kn.dim() != 4 || vp.dim() != 4 || vn.dim() != 3 || kp.scalar_type() != at::kByte || vp.scalar_type() != at::kByte ||
        kn.scalar_type() != at::kHalf || vn.scalar_type() != at::kHalf || kp.stride(3) != 1 || vp.stride(3) != 1 || kn.stride(3) != 1) Py_RETURN_NONE;
    const int64_t B = q.size(0), n_q = q.size(1), S = q.size(2), n_kv = kp.size(1);
    if (n_kv < 1 || n_q % n_kv || kp.size(2) < T || vp.size(2) < T || kn.size(2) < T || vn.size(2) < T || T < 0 || kp.size(0) < B) Py_RETURN_NONE;
    const int64_t seen = causal ? std::min(T, off + S) : T;      // records that some row sees
    const size_t bytes = bgtq_prompt_workspace_bytes((int)B, (int)n_kv, (int)(n_q / n_kv), (int)S, (int)seen);
    // (the allocator hands the same block out again from call to call, and to nobody else before the launches are done)
    at::Tensor ws = at::empty({(int64_t)bytes}, q.options().dtype(at::kByte));
    at::Tensor out = at::empty({B, n_q, S, D}, q.options().dtype(at::kHalf));
    void* st = stream_of(q);
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = bgtq_prompt_attn((const bgtq_head_plan*)plans.data_ptr(), q.data_ptr(), q.scalar_type() == at::kBFloat16 ? BGTQ_X_BF16 : BGTQ_X_FP16,
                          (int)rotate, q.stride(0), q.stride(1), q.stride(2),
                          kp.data_ptr(), kp.stride(0), kp.stride(1), kp.stride(2), (int)kw,
                          kn.data_ptr(), kn.stride(0), kn.stride(1), kn.stride(2),
                          vp.data_ptr(), vp.stride(0), vp.stride(1), vp.stride(2), (int)vw,
                          vn.data_ptr(), vn.stride(0), vn.stride(1), vn.stride(2),
                          (int)B, (int)n_kv, (int)(n_q / n_kv), (int)S, (int)T, (int)off, (int)causal, (int)kl, (int)vl,
                          (float)PyFloat_AS_DOUBLE(a[14]), (int)unrotate, ws.data_ptr(), bytes,
                          out.data_ptr(), out.stride(0), out.stride(1), out.stride(2), st);
    Py_END_ALLOW_THREADS
    if (rc == BGTQ_EUNSUPPORTED) Py_RETURN_NONE;
    if (rc != BGTQ_OK) return fail("bgtq_prompt_attn", rc);
    return THPVariable_Wrap(std::move(out));
    END_HANDLE_TH_ERRORS
}

// stream(t): the current stream of t's device, as something to compare
PyObject* stream(PyObject*, PyObject* o) {
    HANDLE_TH_ERRORS
    const at::Tensor* t = tensor(o);
    if (!t || !t->is_cuda()) { PyErr_SetString(PyExc_TypeError, "stream(tensor on the GPU)"); return nullptr; }
    return Py_BuildValue("iK", (int)t->get_device(), (unsigned long long)(uintptr_t)stream_of(*t));
    END_HANDLE_TH_ERRORS
}

PyObject* setup(PyObject*, PyObject* const* a, Py_ssize_t n) {
    if (n != 2) { PyErr_SetString(PyExc_TypeError, "setup(error class, path hook)"); return nullptr; }
    Py_INCREF(a[0]);
    Py_INCREF(a[1]);
    Py_XDECREF(g_error);
    Py_XDECREF(g_note_path);
    g_error = a[0];
    g_note_path = a[1];
    Py_RETURN_NONE;
}

PyMethodDef module_methods[] = {
    {"attend", (PyCFunction)(void*)attend, METH_FASTCALL, "decode attention over packed records, or None"},
    {"prompt", (PyCFunction)(void*)prompt, METH_FASTCALL, "prompt-phase attention over packed records, or None"},
    {"stream", (PyCFunction)stream, METH_O, "(device, current stream) of a tensor"},
    {"setup", (PyCFunction)(void*)setup, METH_FASTCALL, "hand over the error class and the hook that notes which kernel ran"},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef module_def = {PyModuleDef_HEAD_INIT, "_bgtq_host", "native host side of blockgtq_amd", -1, module_methods};

}  // namespace

PyMODINIT_FUNC PyInit__bgtq_host(void) {
    LayerType.tp_name = "blockgtq_amd._lib._bgtq_host.Layer";
    LayerType.tp_basicsize = sizeof(Layer);
    LayerType.tp_flags = Py_TPFLAGS_DEFAULT;
    LayerType.tp_new = layer_new;
    LayerType.tp_dealloc = layer_dealloc;
    LayerType.tp_methods = layer_methods;
    if (PyType_Ready(&LayerType) < 0) return nullptr;
    g_buf_name = PyUnicode_InternFromString("_buf");
    PyObject* m = PyModule_Create(&module_def);
    if (!m) return nullptr;
    Py_INCREF(&LayerType);
    PyModule_AddObject(m, "Layer", (PyObject*)&LayerType);
    return m;
}
