// The host side of the calls that a program makes once per layer and token: shapes and strides read, outputs allocated, argument
// blocks filled and the library called from one C function each.  Written out in Python the same steps took longer than the kernels
// of a small call (16 tokens, 8 heads of 128: 4.7 us of dense decoding, 6.6 of an append, 8.2 of an encode besides the launch).
// The callers (ops.py) look up what a codebook or a cache fixes and hand over the addresses of those blocks, which are copied: a
// block may serve several threads.  A function returns its tensors, or the library's status as an int if that is not 0.
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/utils/object_ptr.h>
#include <ATen/ATen.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>

#include "../../include/hqmq_amd.h"

namespace {

const at::Tensor &tensor(PyObject *o) {
    TORCH_CHECK_TYPE(THPVariable_Check(o), "expected a tensor");
    return THPVariable_Unpack(o);
}
template <class T>
T *address(PyObject *o) {
    void *p = PyLong_AsVoidPtr(o);
    if (!p && PyErr_Occurred()) throw python_error();
    return (T *)p;
}
int64_t integer(PyObject *o) {
    const int64_t v = PyLong_AsLongLong(o);
    if (v == -1 && PyErr_Occurred()) throw python_error();
    return v;
}
double number(PyObject *o) {
    const double v = PyFloat_AsDouble(o);
    if (v == -1.0 && PyErr_Occurred()) throw python_error();
    return v;
}
void arguments(Py_ssize_t got, Py_ssize_t want) { TORCH_CHECK_TYPE(got == want, "expected ", want, " arguments, got ", got); }

int dtype_of(const at::Tensor &t) {
    switch (t.scalar_type()) {
        case at::kFloat: return HQMQ_F32;
        case at::kHalf: return HQMQ_F16;
        case at::kBFloat16: return HQMQ_BF16;
        default: TORCH_CHECK_TYPE(false, "unsupported dtype ", t.scalar_type(), " (float32, float16, bfloat16 only)");
    }
    return -1;
}

struct WithoutGil {
    PyThreadState *state = PyEval_SaveThread();
    ~WithoutGil() { PyEval_RestoreThread(state); }
};
// The library is called without the GIL, as ctypes does, on the tensors' device and its current stream.
struct Launch {
    c10::DeviceGuard guard;
    void *stream;
    explicit Launch(const at::Tensor &t) : guard(t.device()), stream((void *)c10::hip::getCurrentHIPStream(t.device().index()).stream()) {}
    template <class F>
    int operator()(F f) {
        WithoutGil release;
        return f(stream);
    }
};

PyObject *none() { Py_RETURN_NONE; }
PyObject *wrap(const at::Tensor &t) { return t.defined() ? THPVariable_Wrap(t) : none(); }
template <class... A>
PyObject *tuple(const A &...t) {
    PyObject *r = PyTuple_New(sizeof...(A));
    if (!r) throw python_error();
    Py_ssize_t i = 0;
    (PyTuple_SET_ITEM(r, i++, wrap(t)), ...);
    return r;
}

// (B, H, T, d_head) with rows of stride 1, on the GPU
at::Tensor rows(const at::Tensor &x) {
    TORCH_CHECK_VALUE(x.dim() == 4, "expected (B, H, T, d_head), got ", x.sizes());
    return x.size(3) > 1 && x.stride(3) != 1 ? x.contiguous() : x;
}
void check_joint(const at::Tensor &x, const at::Tensor &joint) {
    TORCH_CHECK_VALUE(joint.scalar_type() == x.scalar_type() && joint.dim() == 3 && joint.size(0) == x.size(1) && joint.is_contiguous(),
                      "joint must be a contiguous (H, 24S, 4) table in the dtype of x");
}
void fill(hqmq_quantize_args &a, const at::Tensor &x) {
    a.x = x.data_ptr();
    a.x_stride_b = x.stride(0);
    a.x_stride_h = x.stride(1);
    a.x_stride_t = x.stride(2);
    a.B = (int)x.size(0);
    a.T = (int)x.size(2);
}
int median(Launch &go, const at::Tensor &x, double mult, const at::Tensor &ws, void *med, void *thr, void *count) {
    const int dt = dtype_of(x), B = (int)x.size(0), H = (int)x.size(1), T = (int)x.size(2), n = (int)(x.size(3) / 4);
    const int64_t sb = x.stride(0), sh = x.stride(1), st = x.stride(2), bytes = (int64_t)ws.nbytes();
    const void *p = x.data_ptr();
    void *w = ws.data_ptr();
    return go([&](void *stream) {
        return hqmq_med3x_threshold(p, sb, sh, st, dt, B, H, T, n, (float)mult, w, bytes, (float *)med, thr, (int32_t *)count, stream);
    });
}
// room for a median and a threshold nobody asked for, behind the workspace proper (ops._med_workspace)
uint8_t *spare(const at::Tensor &ws, int64_t H) { return (uint8_t *)ws.data_ptr() + ((ws.nbytes() - 12 * H) & -(int64_t)16); }

// codes(x, joint, block, lists, thr or None, want_mask) -> (idx, rq, r_max, mask or None)
PyObject *codes(PyObject *, PyObject *const *o, Py_ssize_t count) {
    HANDLE_TH_ERRORS
    arguments(count, 6);
    const at::Tensor x = rows(tensor(o[0]));
    check_joint(x, tensor(o[1]));
    hqmq_quantize_args a = *address<hqmq_quantize_args>(o[2]);
    const void *lists = address<void>(o[3]);
    fill(a, x);
    const int64_t B = x.size(0), H = x.size(1), T = x.size(2), n = x.size(3) / 4;
    const auto ints = x.options().dtype(at::kInt);
    at::Tensor idx = at::empty({B, H, T, n}, ints), rq = at::empty({B, H, T, n}, ints), scale = at::empty({B, H, T}, x.options()), thr, mask;
    a.idx_out = (int32_t *)idx.data_ptr();
    a.rq_out = (int32_t *)rq.data_ptr();
    a.rmax_out = scale.data_ptr();
    if (o[4] != Py_None) {
        thr = tensor(o[4]).to(x.scalar_type()).contiguous();
        a.thr = thr.data_ptr();
        if (o[5] == Py_True) {
            mask = at::empty({B, H, T, n}, x.options().dtype(at::kBool));        // one byte per chunk, 0 or 1
            a.mask_out = (uint8_t *)mask.data_ptr();
        }
    }
    if (T > 0) {
        const int status = Launch(x)([&](void *stream) { return hqmq_quantize_grid(&a, lists, stream); });
        if (status) return PyLong_FromLong(status);
    }
    return tuple(idx, rq, scale, mask);
    END_HANDLE_TH_ERRORS
}

// fake(x, joint, block, lists, median_mult or None, workspace or None) -> (out, flagged chunks per head or None)
PyObject *fake(PyObject *, PyObject *const *o, Py_ssize_t count) {
    HANDLE_TH_ERRORS
    arguments(count, 6);
    const at::Tensor x = rows(tensor(o[0]));
    check_joint(x, tensor(o[1]));
    hqmq_quantize_args a = *address<hqmq_quantize_args>(o[2]);
    const void *lists = address<void>(o[3]);
    fill(a, x);
    const int64_t H = x.size(1);
    at::Tensor out = at::empty(x.sizes(), x.options()), flagged;
    a.dense_out = out.data_ptr();
    Launch go(x);
    if (o[4] != Py_None) {
        const at::Tensor &ws = tensor(o[5]);
        flagged = at::empty({H}, x.options().dtype(at::kInt));
        uint8_t *room = spare(ws, H);
        const float mult = (float)number(o[4]);
        void *w = ws.data_ptr(), *thr = room + 4 * H;
        const int64_t bytes = (int64_t)ws.nbytes();
        int32_t *counts = (int32_t *)flagged.data_ptr();
        const int status = go([&](void *stream) { return hqmq_quantize_med3x_grid(&a, mult, w, bytes, (float *)room, thr, counts, lists, stream); });
        if (status) return PyLong_FromLong(status);
    } else if (x.size(2) > 0) {
        const int status = go([&](void *stream) { return hqmq_quantize_grid(&a, lists, stream); });
        if (status) return PyLong_FromLong(status);
    }
    return tuple(out, flagged);
    END_HANDLE_TH_ERRORS
}

// med3x(x, mult, workspace, want_count) -> (median, threshold, flagged chunks per head or None)
PyObject *med3x(PyObject *, PyObject *const *o, Py_ssize_t count) {
    HANDLE_TH_ERRORS
    arguments(count, 4);
    const at::Tensor x = rows(tensor(o[0]));
    const int64_t H = x.size(1);
    at::Tensor med = at::empty({H}, x.options().dtype(at::kFloat)), thr = at::empty({H}, x.options()), flagged;
    if (o[3] == Py_True) flagged = at::empty({H}, x.options().dtype(at::kInt));          // written for every head
    Launch go(x);
    const int status = median(go, x, number(o[1]), tensor(o[2]), med.data_ptr(), thr.data_ptr(), flagged.defined() ? flagged.data_ptr() : nullptr);
    if (status) return PyLong_FromLong(status);
    return tuple(med, thr, flagged);
    END_HANDLE_TH_ERRORS
}

// append(k, v, k block, v block, k lists, v lists, t_off, pos or None, median_mult or None, k workspace, v workspace)
//   -> (flagged k chunks per head or None, flagged v chunks per head or None)
PyObject *append(PyObject *, PyObject *const *o, Py_ssize_t count) {
    HANDLE_TH_ERRORS
    arguments(count, 11);
    const at::Tensor x[2] = {rows(tensor(o[0])), rows(tensor(o[1]))};
    hqmq_append_args a[2] = {*address<hqmq_append_args>(o[2]), *address<hqmq_append_args>(o[3])};
    const void *kl = address<void>(o[4]), *vl = address<void>(o[5]);
    const int t_off = (int)integer(o[6]);
    at::Tensor pos, flagged[2];
    if (o[7] != Py_None) pos = tensor(o[7]).to(x[0].device(), at::kInt).contiguous();
    for (int i = 0; i < 2; i++) {
        hqmq_quantize_args &q = a[i].q;
        fill(q, x[i]);
        q.t_off = t_off;
        if (pos.defined()) q.pos = (const int32_t *)pos.data_ptr();
        if (o[8] != Py_None && x[i].size(2) > 0) {
            const at::Tensor &ws = tensor(o[9 + i]);
            const int64_t H = x[i].size(1);
            flagged[i] = at::empty({H}, x[i].options().dtype(at::kInt));       // every path of the library writes all H counts
            uint8_t *room = spare(ws, H);
            a[i].median_mult = (float)number(o[8]);
            a[i].med_workspace = ws.data_ptr();
            a[i].med_workspace_bytes = (int64_t)ws.nbytes();
            a[i].median = (float *)room;
            a[i].thr = room + 4 * H;
            a[i].n_out = (int32_t *)flagged[i].data_ptr();
        }
    }
    const int status = Launch(x[0])([&](void *stream) { return hqmq_append_kv_grid(&a[0], &a[1], kl, vl, stream); });
    if (status) return PyLong_FromLong(status);
    return tuple(flagged[0], flagged[1]);
    END_HANDLE_TH_ERRORS
}

at::Tensor int_rows(const at::Tensor &t) {
    const at::Tensor i = t.scalar_type() == at::kInt ? t : t.to(at::kInt);
    return i.stride(-1) == 1 ? i : i.contiguous();
}
at::Tensor table(const at::Tensor &j) { return j.stride(-1) != 1 || j.stride(1) != 4 ? j.contiguous() : j; }

// dequant(idx, rq, scale, joint, qmax) -> dense
PyObject *dequant(PyObject *, PyObject *const *o, Py_ssize_t count) {
    HANDLE_TH_ERRORS
    arguments(count, 5);
    const at::Tensor idx = int_rows(tensor(o[0])), rq = int_rows(tensor(o[1])), joint = table(tensor(o[3]));
    TORCH_CHECK_VALUE(idx.dim() == 4, "not enough values to unpack (expected 4, got ", idx.dim(), ")");
    const at::Tensor &rs0 = tensor(o[2]);
    const at::Tensor rs = rs0.scalar_type() == joint.scalar_type() ? rs0 : rs0.to(joint.scalar_type());
    const int qmax = (int)integer(o[4]), dt = dtype_of(joint);
    const int64_t B = idx.size(0), H = idx.size(1), T = idx.size(2), n = idx.size(3);
    at::Tensor out = at::empty({B, H, T, 4 * n}, joint.options().device(idx.device()));
    const int32_t *pi = (const int32_t *)idx.data_ptr(), *pr = (const int32_t *)rq.data_ptr();
    const void *ps = rs.data_ptr(), *pj = joint.data_ptr();
    void *po = out.data_ptr();
    const int64_t s[10] = {idx.stride(0), idx.stride(1), idx.stride(2), rq.stride(0), rq.stride(1), rq.stride(2), rs.stride(0), rs.stride(1), rs.stride(2), joint.stride(0)};
    const int K = (int)joint.size(1);
    const int status = Launch(idx)([&](void *stream) {
        return hqmq_dequant(pi, s[0], s[1], s[2], pr, s[3], s[4], s[5], ps, s[6], s[7], s[8], pj, s[9], K, dt, (int)B, (int)H, (int)T, (int)n, qmax, po, stream);
    });
    if (status) return PyLong_FromLong(status);
    return wrap(out);
    END_HANDLE_TH_ERRORS
}

at::Tensor words(PyObject *o, const at::Tensor &like) {
    const at::Tensor &t = tensor(o);
    return t.scalar_type() == at::kInt && t.device() == like.device() && t.is_contiguous() ? t : t.to(like.device(), at::kInt).contiguous();
}
void output(hqmq_attn_args &a, const at::Tensor &Q, const at::Tensor &O) {
    a.Q = Q.data_ptr();
    a.O = O.data_ptr();
    a.o_sb = O.stride(0);
    a.o_sh = O.stride(1);
    a.o_st = O.stride(2);
}

// attn(Q, block, out or None, T_kv, kv_lens, kv_starts, batch_order (each or None), causal, causal_offset, scale or None, n_splits,
//      force_generic, fp8_table_storage, wide_range, kept_workspace, options or None) -> O, or (O, partials or None, n_splits)
//   kept_workspace(bytes, device, "attn") names the buffer that the calls of a stream share;
//   options: (skip_combine, static_scratch, workspace or None, begin event, end event)
PyObject *attn(PyObject *, PyObject *const *o, Py_ssize_t count) {
    HANDLE_TH_ERRORS
    arguments(count, 16);
    const at::Tensor &Q = tensor(o[0]);
    hqmq_attn_args a = *address<hqmq_attn_args>(o[1]);
    const at::Tensor O = o[2] == Py_None ? at::empty_like(Q) : tensor(o[2]);
    output(a, Q, O);
    a.T_kv = (int)integer(o[3]);
    at::Tensor lens, starts, order;
    if (o[4] != Py_None) a.kv_len = (const int32_t *)(lens = words(o[4], Q)).data_ptr();
    if (o[5] != Py_None) a.kv_start = (const int32_t *)(starts = words(o[5], Q)).data_ptr();
    if (o[6] != Py_None) a.batch_order = (const int32_t *)(order = words(o[6], Q)).data_ptr();
    if (PyObject_IsTrue(o[7])) {
        a.causal = 1;
        a.causal_offset = integer(o[8]);
    }
    if (o[9] != Py_None) a.softmax_scale = (float)number(o[9]);
    a.n_splits = (int)integer(o[10]);
    a.force_generic = (int)integer(o[11]);
    a.fp8_table_storage = PyObject_IsTrue(o[12]) ? 1 : 0;
    a.wide_range = PyObject_IsTrue(o[13]) ? 1 : 0;
    bool own_scratch = false;
    at::Tensor ws;
    if (o[15] != Py_None) {
        TORCH_CHECK_TYPE(PyTuple_Check(o[15]) && PyTuple_GET_SIZE(o[15]) == 5, "expected a tuple of five options");
        PyObject *const *opt = &PyTuple_GET_ITEM(o[15], 0);
        a.skip_combine = PyObject_IsTrue(opt[0]) ? 1 : 0;
        own_scratch = PyObject_IsTrue(opt[1]);
        if (opt[2] != Py_None) ws = tensor(opt[2]);
        a.start_event = address<void>(opt[3]);
        a.stop_event = address<void>(opt[4]);
    }
    if (own_scratch) {
        const int status = Launch(Q)([&](void *stream) { return hqmq_attn_fwd_static(&a, stream); });
        return status ? PyLong_FromLong(status) : wrap(O);
    }
    if (a.n_splits <= 0) a.n_splits = hqmq_attn_splits(&a);
    if (a.n_splits > 1) {
        const int64_t bytes = hqmq_attn_workspace_bytes(a.B, a.H_q, a.T_q, 4 * a.n_chunks, a.n_splits);
        if (ws.defined()) {
            if (ws.device() != Q.device()) return PyLong_FromLong(HQMQ_ERR_WORKSPACE);
        } else if (a.skip_combine) {
            ws = at::empty({bytes}, Q.options().dtype(at::kByte));          // the caller's from here on
        } else {
            THPObjectPtr device(PyObject_GetAttrString(o[0], "device")), kept(device ? PyObject_CallFunction(o[14], "LOs", (long long)bytes, device.get(), "attn") : nullptr);
            if (!kept) throw python_error();
            ws = tensor(kept.get());
        }
        a.workspace = ws.data_ptr();
        a.workspace_bytes = (int64_t)ws.nbytes();
    } else ws = at::Tensor();
    const int status = Launch(Q)([&](void *stream) { return hqmq_attn_fwd(&a, stream); });
    if (status) return PyLong_FromLong(status);
    if (!a.skip_combine) return wrap(O);
    THPObjectPtr n(PyLong_FromLong(a.n_splits)), o_out(wrap(O)), ws_out(wrap(ws));
    return PyTuple_Pack(3, o_out.get(), ws_out.get(), n.get());
    END_HANDLE_TH_ERRORS
}

// fused(Q, K idx, rq, scale, joint, V idx, rq, scale, joint, pack block, attention block, bytes of the planes, kv_lens or None,
//       causal, causal_offset, scale or None, n_splits) -> O.  The blocks hold the planes' offsets in place of addresses.
PyObject *fused(PyObject *, PyObject *const *o, Py_ssize_t count) {
    HANDLE_TH_ERRORS
    arguments(count, 17);
    const at::Tensor &Q = tensor(o[0]);
    const auto dt = Q.scalar_type();
    hqmq_pack_args pack = *address<hqmq_pack_args>(o[9]);
    hqmq_attn_args a = *address<hqmq_attn_args>(o[10]);
    Launch go(tensor(o[1]));
    const at::Tensor planes = at::empty({integer(o[11])}, tensor(o[1]).options().dtype(at::kByte));
    uint8_t *base = (uint8_t *)planes.data_ptr();
    const auto at_base = [&](const void *offset) { return base + (uintptr_t)offset; };
    at::Tensor keep[8], most;
    if (dt != at::kHalf) most = at::zeros({2}, planes.options().dtype(at::kInt));
    for (int i = 0; i < 2; i++) {
        const at::Tensor &idx = keep[4 * i] = int_rows(tensor(o[1 + 4 * i])), &rq = keep[4 * i + 1] = int_rows(tensor(o[2 + 4 * i]));
        at::Tensor &rs = keep[4 * i + 2] = tensor(o[3 + 4 * i]);
        if (rs.scalar_type() != dt) rs = rs.to(dt);
        if (rs.sizes() != idx.sizes().slice(0, 3)) rs = rs.expand(idx.sizes().slice(0, 3));
        const at::Tensor &joint = keep[4 * i + 3] = table(tensor(o[4 + 4 * i]));
        hqmq_pack_side &p = pack.side[i];
        hqmq_packed &t = i ? a.V : a.K;
        p.idx = (const int32_t *)idx.data_ptr();
        p.idx_sb = idx.stride(0);
        p.idx_sh = idx.stride(1);
        p.idx_st = idx.stride(2);
        p.rq = (const int32_t *)rq.data_ptr();
        p.rq_sb = rq.stride(0);
        p.rq_sh = rq.stride(1);
        p.rq_st = rq.stride(2);
        p.scale_in = rs.data_ptr();
        p.scale_sb = rs.stride(0);
        p.scale_sh = rs.stride(1);
        p.scale_st = rs.stride(2);
        t.main_plane = p.main_plane = at_base(p.main_plane);
        t.scale_plane = p.scale_plane = at_base(p.scale_plane);
        if (pack.aux_bits) t.aux_plane = p.aux_plane = at_base(p.aux_plane);
        t.joint = joint.data_ptr();
        t.joint_sh = joint.stride(0);
        if (most.defined()) t.scale_max_bits = p.scale_max_bits = (uint32_t *)most.data_ptr() + i;
    }
    int status = go([&](void *stream) { return hqmq_pack_kv(&pack, stream); });
    if (status) return PyLong_FromLong(status);
    const at::Tensor O = at::empty_like(Q);
    output(a, Q, O);
    at::Tensor lens, ws;
    if (o[12] != Py_None) a.kv_len = (const int32_t *)(lens = words(o[12], planes)).data_ptr();
    if (PyObject_IsTrue(o[13])) {
        a.causal = 1;
        a.causal_offset = integer(o[14]);
    }
    if (o[15] != Py_None) a.softmax_scale = (float)number(o[15]);
    a.n_splits = (int)integer(o[16]);
    if (a.n_splits <= 0) a.n_splits = hqmq_attn_splits(&a);
    if (a.n_splits > 1) {
        a.workspace_bytes = hqmq_attn_workspace_bytes(a.B, a.H_q, a.T_q, 4 * a.n_chunks, a.n_splits);
        ws = at::empty({a.workspace_bytes}, planes.options());
        a.workspace = ws.data_ptr();
    }
    // bf16 V scales outside [2^-8, 2^15) need the kernel that guards the fp16 range; only the GPU knows them by now
    status = go([&](void *stream) { return dt == at::kBFloat16 ? hqmq_attn_fwd_guarded(&a, stream) : hqmq_attn_fwd(&a, stream); });
    if (status) return PyLong_FromLong(status);
    return wrap(O);
    END_HANDLE_TH_ERRORS
}

PyMethodDef methods[] = {
    {"attn", (PyCFunction)(void *)attn, METH_FASTCALL, nullptr},       {"fused", (PyCFunction)(void *)fused, METH_FASTCALL, nullptr},
    {"codes", (PyCFunction)(void *)codes, METH_FASTCALL, nullptr},     {"fake", (PyCFunction)(void *)fake, METH_FASTCALL, nullptr},
    {"med3x", (PyCFunction)(void *)med3x, METH_FASTCALL, nullptr},     {"append", (PyCFunction)(void *)append, METH_FASTCALL, nullptr},
    {"dequant", (PyCFunction)(void *)dequant, METH_FASTCALL, nullptr}, {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_native", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__native() { return PyModule_Create(&module); }
