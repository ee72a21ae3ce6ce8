// Native host side of the calls whose shape has been seen before: a CPython extension (module flagattention_amd._host) that
// finds the filled parameter struct of a call by the metadata of its tensors, allocates the outputs and calls the library.
//
// The Python functions (sage_attention/quant.py, sage_attention/attention.py, flash.py) check the arguments of a call, fill the
// parameter struct and register it here under the call's key: every size, stride, dtype and flag that the checks and the
// struct depend on.  A later call with the same key has passed the same checks, so only pointers are written (their
// alignment, the one property of a call that the key does not hold, is looked at every time).  Anything else - a tensor
// subclass, another device than the current one, a key not seen, tensors that require grad - returns None, and the Python
// function takes the call from the start.  Nothing of a call's data is kept.
//
// Host time of a call, Python before -> here: per_block_int8 with smoothing 24.7 -> 6.4 us, sage_attention 12.9 -> 4.0 us, flash_attention 13.6 -> 3.7 us
// (mostly the launches and the allocation of the outputs).
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/ATen.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/version.h>

#include <algorithm>
#include <cstring>
#include <string>
#include <unordered_map>

#include "../../include/sage_attention_hip.h"

namespace {

constexpr size_t kMaxPlans = 64;  // of a thread

// The key of a call: its integers as bytes.
struct Key {
    std::string bytes;
    Key() { bytes.reserve(320); }
    void add(int64_t v) { bytes.append(reinterpret_cast<const char*>(&v), sizeof(v)); }
    void add(const at::Tensor& t) {
        add((int64_t)t.scalar_type());
        const auto s = t.sizes(), st = t.strides();
        add((int64_t)s.size());
        bytes.append(reinterpret_cast<const char*>(s.data()), s.size() * sizeof(int64_t));
        bytes.append(reinterpret_cast<const char*>(st.data()), st.size() * sizeof(int64_t));
    }
    void add(double v) {
        int64_t b;
        std::memcpy(&b, &v, sizeof(b));
        add(b);
    }
};

struct Plan {
    std::string params;      // the library's parameter struct
    int64_t workspace = 0;   // bytes
    bool fused = false;      // (quantizer) sage_smooth_quant_params
};

// Tables of one thread: a parameter struct is written by one thread at a time.  A plan that is used lies in the young table;
// when that is full it becomes the old one, whose plans go unless they are used before the next time.  So sizes that come
// once (the keys of a growing cache) do not push out those that return.
typedef std::unordered_map<std::string, Plan> Table;
thread_local Table t_young, t_old;

void make_room() {
    if (t_young.size() < kMaxPlans / 2) return;
    t_old.swap(t_young);
    t_young.clear();
}

Plan* find(const Key& k) {
    auto it = t_young.find(k.bytes);
    if (it != t_young.end()) return &it->second;
    it = t_old.find(k.bytes);
    if (it == t_old.end()) return nullptr;
    auto node = t_old.extract(it);
    make_room();
    return &t_young.insert(std::move(node)).position->second;
}

// Scratch memory of one call: from the caching allocator, which gives it to the next call on this stream once the launches
// are enqueued.  Not kept between calls: a captured graph holds its address, so under capture it has to come from the
// graph's own memory pool (0.7 us of host time per call).
at::Tensor workspace(const at::Device& dev, int64_t nbytes) {
    return at::empty({std::max<int64_t>(nbytes, 16)}, at::TensorOptions().dtype(at::kByte).device(dev));
}

bool plain(PyObject* o) { return THPVariable_CheckExact(o); }

bool ready(const at::Tensor& t, const at::Device& dev) {
    return t.device() == dev && ((uintptr_t)t.data_ptr() & 15) == 0 && !t.is_neg() && !t.is_conj();
}

bool is_hnd(PyObject* layout, bool& hnd) {
    if (!PyUnicode_Check(layout)) return false;
    if (PyUnicode_CompareWithASCIIString(layout, "HND") == 0) hnd = true;
    else if (PyUnicode_CompareWithASCIIString(layout, "NHD") == 0) hnd = false;
    else return false;
    return true;
}

// true / false / anything else: not handled here
bool is_bool(PyObject* o, bool& v) {
    if (o == Py_True) v = true;
    else if (o == Py_False) v = false;
    else return false;
    return true;
}

at::TensorOptions options(const at::Device& dev, at::ScalarType dt) { return at::TensorOptions().dtype(dt).device(dev); }

PyObject* none() { Py_RETURN_NONE; }

PyObject* pack(std::initializer_list<const at::Tensor*> ts) {
    PyObject* tuple = PyTuple_New((Py_ssize_t)ts.size());
    if (!tuple) return nullptr;
    Py_ssize_t i = 0;
    for (const at::Tensor* t : ts) {
        PyObject* o;
        if (t) o = THPVariable_Wrap(*t);
        else o = Py_NewRef(Py_None);
        if (!o) {
            Py_DECREF(tuple);
            return nullptr;
        }
        PyTuple_SET_ITEM(tuple, i++, o);
    }
    return tuple;
}

template <typename Fn>
PyObject* guarded(Fn&& fn) {
    try {
        return fn();
    } catch (const std::exception& e) {
        PyErr_SetString(PyExc_RuntimeError, e.what());
        return nullptr;
    }
}

PyObject* put(const Key& key, PyObject* params, PyObject* ws, bool fused) {
    Plan plan;
    char* data;
    Py_ssize_t size;
    if (PyBytes_AsStringAndSize(params, &data, &size) < 0) return nullptr;
    plan.params.assign(data, (size_t)size);
    plan.workspace = PyLong_AsLongLong(ws);
    if (PyErr_Occurred()) return nullptr;
    plan.fused = fused;
    make_room();
    t_young[key.bytes] = std::move(plan);
    return none();
}

// ---- quantizer: (q, k, km, blkq, blkk, sm_scale, layout, smooth, want_dot)
struct QuantCall {
    const at::Tensor *q, *k, *km = nullptr;
    bool hnd, smooth, want_dot;
    Key key;
    bool parse(PyObject* const* a, Py_ssize_t n) {
        if (n < 9 || !plain(a[0]) || !plain(a[1])) return false;
        q = &THPVariable_Unpack(a[0]);
        k = &THPVariable_Unpack(a[1]);
        if (a[2] != Py_None) {
            if (!plain(a[2])) return false;
            km = &THPVariable_Unpack(a[2]);
        }
        if (!PyLong_CheckExact(a[3]) || !PyLong_CheckExact(a[4]) || !is_hnd(a[6], hnd) || !is_bool(a[7], smooth) || !is_bool(a[8], want_dot))
            return false;
        key.add((int64_t)1);
        key.add(*q);
        key.add(*k);
        key.add((int64_t)(km != nullptr));
        if (km) key.add(*km);
        key.add((int64_t)PyLong_AsLongLong(a[3]));
        key.add((int64_t)PyLong_AsLongLong(a[4]));
        if (PyErr_Occurred()) {
            PyErr_Clear();
            return false;
        }
        if (a[5] == Py_None) key.add((int64_t)0);
        else if (PyFloat_CheckExact(a[5])) {
            key.add((int64_t)1);
            key.add(PyFloat_AS_DOUBLE(a[5]));
        } else return false;
        key.add((int64_t)(hnd | smooth << 1 | want_dot << 2));
        key.add((int64_t)q->device().index());
        return true;
    }
};

PyObject* quant(PyObject*, PyObject* const* a, Py_ssize_t n) {
    return guarded([&]() -> PyObject* {
        QuantCall c;
        if (!c.parse(a, n)) return none();
        Plan* plan = find(c.key);
        if (!plan) return none();
        const at::Device dev = c.q->device();
        if (!dev.is_cuda() || c10::hip::current_device() != dev.index() || !ready(*c.q, dev) || !ready(*c.k, dev) || (c.km && !ready(*c.km, dev)))
            return none();
        auto* sp = plan->fused ? reinterpret_cast<sage_smooth_quant_params*>(&plan->params[0]) : nullptr;
        sage_quant_params& p = sp ? sp->quant : *reinterpret_cast<sage_quant_params*>(&plan->params[0]);
        const at::Tensor q8 = at::empty(c.q->sizes(), options(dev, at::kChar)), k8 = at::empty(c.k->sizes(), options(dev, at::kChar));
        const at::Tensor qs = at::empty({p.batch, p.heads_q, (p.qo_len + p.blkq - 1) / p.blkq}, options(dev, at::kFloat));
        const at::Tensor ks = at::empty({p.batch, p.heads_kv, (p.kv_len + p.blkk - 1) / p.blkk}, options(dev, at::kFloat));
        p.q.ptr = c.q->data_ptr(); p.k.ptr = c.k->data_ptr(); p.q_int8.ptr = q8.data_ptr(); p.k_int8.ptr = k8.data_ptr();
        p.q_scale = (float*)qs.data_ptr(); p.k_scale = (float*)ks.data_ptr();
        void* stream = c10::hip::getCurrentHIPStream(dev.index()).stream();
        if (!sp) {
            p.km.ptr = c.km ? c.km->data_ptr() : nullptr;
            if (int rc = sage_per_block_int8(&p, stream)) return PyLong_FromLong(rc);
            return pack({&q8, &qs, &k8, &ks, nullptr, nullptr});
        }
        const at::Tensor km = c.hnd ? at::empty({p.batch, p.heads_kv, 1, p.head_dim}, options(dev, c.k->scalar_type()))
                                    : at::empty({p.batch, 1, p.heads_kv, p.head_dim}, options(dev, c.k->scalar_type()));
        at::Tensor dot;
        sp->km_out = km.data_ptr();
        sp->q_dot_km = nullptr;
        if (c.want_dot) {
            dot = at::empty({p.batch, p.heads_q, p.qo_len}, options(dev, at::kFloat));
            sp->q_dot_km = (float*)dot.data_ptr();
        }
        const at::Tensor ws = workspace(dev, plan->workspace);
        sp->workspace = ws.data_ptr();
        if (int rc = sage_per_block_int8_smooth_k(sp, stream)) return PyLong_FromLong(rc);
        return pack({&q8, &qs, &k8, &ks, &km, c.want_dot ? &dot : nullptr});
    });
}

PyObject* put_quant(PyObject*, PyObject* const* a, Py_ssize_t n) {  // + (params, workspace bytes, fused)
    return guarded([&]() -> PyObject* {
        QuantCall c;
        if (n != 12 || !c.parse(a, n)) return none();
        return put(c.key, a[9], a[10], a[11] == Py_True);
    });
}

// ---- SageAttention forward: (q, k, v, q_scale, k_scale, layout, mask, out_dtype, return_lse, causal, shift_mul, shift)
struct AttnCall {
    const at::Tensor *q, *k, *v, *qs, *ks, *mask = nullptr, *shift = nullptr;
    bool hnd, want_lse, causal, natural = false;
    double shift_mul = 0.0;
    at::ScalarType out;
    Key key;
    bool parse(PyObject* const* a, Py_ssize_t n) {
        if (n < 12) return false;
        for (int i = 0; i < 5; i++)
            if (!plain(a[i])) return false;
        q = &THPVariable_Unpack(a[0]); k = &THPVariable_Unpack(a[1]); v = &THPVariable_Unpack(a[2]);
        qs = &THPVariable_Unpack(a[3]); ks = &THPVariable_Unpack(a[4]);
        if (a[6] != Py_None) {
            if (!plain(a[6])) return false;
            mask = &THPVariable_Unpack(a[6]);
        }
        if (!is_hnd(a[5], hnd) || !THPDtype_Check(a[7]) || !is_bool(a[8], want_lse) || !is_bool(a[9], causal)) return false;
        out = reinterpret_cast<THPDtype*>(a[7])->scalar_type;
        if (a[10] != Py_None) {
            if (!PyFloat_CheckExact(a[10])) return false;
            natural = true;
            shift_mul = PyFloat_AS_DOUBLE(a[10]);
            if (a[11] != Py_None) {
                if (!plain(a[11])) return false;
                shift = &THPVariable_Unpack(a[11]);
            }
        }
        key.add((int64_t)2);
        key.add(*q);
        key.add(*k);
        key.add(*v);
        key.add(*qs);
        key.add(*ks);
        key.add((int64_t)(mask != nullptr));
        if (mask) key.add(*mask);
        key.add((int64_t)out);
        key.add((int64_t)(hnd | causal << 1 | natural << 2 | (shift != nullptr) << 3));
        if (shift) key.add(*shift);
        key.add((int64_t)q->device().index());
        return true;
    }
};

PyObject* attn(PyObject*, PyObject* const* a, Py_ssize_t n) {
    return guarded([&]() -> PyObject* {
        AttnCall c;
        if (!c.parse(a, n)) return none();
        Plan* plan = find(c.key);
        if (!plan) return none();
        const at::Device dev = c.q->device();
        if (!dev.is_cuda() || c10::hip::current_device() != dev.index() || !ready(*c.q, dev) || !ready(*c.k, dev) || !ready(*c.v, dev) ||
            c.qs->device() != dev || c.ks->device() != dev || (c.mask && !ready(*c.mask, dev)) ||
            (c.shift && c.shift->device() != dev))
            return none();
        auto& p = *reinterpret_cast<sage_attn_params*>(&plan->params[0]);
        const at::Tensor o = at::empty(c.q->sizes(), options(dev, c.out));
        const at::Tensor lse = c.want_lse ? at::empty({p.batch, p.heads_q, p.qo_len}, options(dev, at::kFloat))
                                          : at::empty({0}, at::TensorOptions().dtype(at::kFloat));
        p.q.ptr = c.q->data_ptr(); p.k.ptr = c.k->data_ptr(); p.v.ptr = c.v->data_ptr(); p.out.ptr = o.data_ptr();
        p.q_scale = (const float*)c.qs->data_ptr(); p.k_scale = (const float*)c.ks->data_ptr();
        p.lse = c.want_lse ? (float*)lse.data_ptr() : nullptr;
        p.mask = c.mask ? c.mask->data_ptr() : nullptr;
        void* stream = c10::hip::getCurrentHIPStream(dev.index()).stream();
        at::Tensor ws;
        if (plan->workspace > 0) ws = workspace(dev, plan->workspace);
        void* wp = plan->workspace > 0 ? ws.data_ptr() : nullptr;
        const int rc = c.natural ? sage_attn_fwd_natural(&p, c.shift ? (const float*)c.shift->data_ptr() : nullptr, (float)c.shift_mul, wp, plan->workspace, stream)
                                 : sage_attn_fwd_ws(&p, wp, plan->workspace, stream);
        if (rc) return PyLong_FromLong(rc);
        return pack({&o, &lse});
    });
}

PyObject* put_attn(PyObject*, PyObject* const* a, Py_ssize_t n) {  // + (params, workspace bytes)
    return guarded([&]() -> PyObject* {
        AttnCall c;
        if (n != 14 || !c.parse(a, n)) return none();
        return put(c.key, a[12], a[13], false);
    });
}

// ---- dense forward: (q, k, v, causal, sm_scale, need_log_normalizer)
struct FlashCall {
    const at::Tensor *q, *k, *v;
    bool causal, need_l;
    Key key;
    bool parse(PyObject* const* a, Py_ssize_t n) {
        if (n < 6 || !plain(a[0]) || !plain(a[1]) || !plain(a[2]) || !is_bool(a[3], causal) || !is_bool(a[5], need_l)) return false;
        q = &THPVariable_Unpack(a[0]); k = &THPVariable_Unpack(a[1]); v = &THPVariable_Unpack(a[2]);
        if (q->requires_grad() || k->requires_grad() || v->requires_grad()) return false;
        key.add((int64_t)3);
        key.add(*q);
        key.add(*k);
        key.add(*v);
        if (a[4] == Py_None) key.add((int64_t)0);
        else if (PyFloat_CheckExact(a[4])) {
            key.add((int64_t)1);
            key.add(PyFloat_AS_DOUBLE(a[4]));
        } else return false;
        key.add((int64_t)causal);
        key.add((int64_t)q->device().index());
        return true;
    }
};

PyObject* flash(PyObject*, PyObject* const* a, Py_ssize_t n) {
    return guarded([&]() -> PyObject* {
        FlashCall c;
        if (!c.parse(a, n)) return none();
        Plan* plan = find(c.key);
        if (!plan) return none();
        const at::Device dev = c.q->device();
        if (!dev.is_cuda() || c10::hip::current_device() != dev.index() || !ready(*c.q, dev) || !ready(*c.k, dev) || !ready(*c.v, dev)) return none();
        auto& p = *reinterpret_cast<sage_flash_params*>(&plan->params[0]);
        const at::Tensor o = at::empty_like(*c.q);
        at::Tensor l;
        if (c.need_l) l = at::empty({p.batch, p.heads_q, p.qo_len}, options(dev, at::kFloat));
        p.q.ptr = c.q->data_ptr(); p.k.ptr = c.k->data_ptr(); p.v.ptr = c.v->data_ptr(); p.out.ptr = o.data_ptr();
        p.log_normalizer = c.need_l ? (float*)l.data_ptr() : nullptr;
        void* stream = c10::hip::getCurrentHIPStream(dev.index()).stream();
        const int rc = plan->workspace > 0 ? sage_flash_attn_fwd_ws(&p, workspace(dev, plan->workspace).data_ptr(), plan->workspace, stream)
                                           : sage_flash_attn_fwd(&p, stream);
        if (rc) return PyLong_FromLong(rc);
        return pack({&o, c.need_l ? &l : nullptr});
    });
}

PyObject* put_flash(PyObject*, PyObject* const* a, Py_ssize_t n) {  // + (params, workspace bytes)
    return guarded([&]() -> PyObject* {
        FlashCall c;
        if (n != 8 || !c.parse(a, n)) return none();
        return put(c.key, a[6], a[7], false);
    });
}

PyMethodDef methods[] = {
    {"quant", (PyCFunction)(void (*)(void))quant, METH_FASTCALL, "outputs of a quantizer call whose plan is known, None, or a status"},
    {"put_quant", (PyCFunction)(void (*)(void))put_quant, METH_FASTCALL, "registers the plan of a quantizer call"},
    {"attn", (PyCFunction)(void (*)(void))attn, METH_FASTCALL, "outputs of a SageAttention call whose plan is known, None, or a status"},
    {"put_attn", (PyCFunction)(void (*)(void))put_attn, METH_FASTCALL, "registers the plan of a SageAttention call"},
    {"flash", (PyCFunction)(void (*)(void))flash, METH_FASTCALL, "outputs of a dense forward call whose plan is known, None, or a status"},
    {"put_flash", (PyCFunction)(void (*)(void))put_flash, METH_FASTCALL, "registers the plan of a dense forward call"},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_host", "native host side of calls whose shape has been seen before", -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__host(void) {
    PyObject* m = PyModule_Create(&module);
    if (m && PyModule_AddStringConstant(m, "torch_version", TORCH_VERSION) < 0) {
        Py_DECREF(m);
        return nullptr;
    }
    return m;
}
