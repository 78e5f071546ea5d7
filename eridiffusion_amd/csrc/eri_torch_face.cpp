/*
 * The per-tensor work of the Python face (eridiffusion_amd/adam8bit.py) in native code: reading the addresses and
 * dtypes of a list of tensors and their gradients, and allocating the tensors an update returns.  A step of an
 * adapter touches 60 to 1,400 tensors for 20 to 90 us of kernel, and the interpreter took about a microsecond per
 * tensor of a list and three per named tensor, so the host was what a step waited for.  Per step, before and after:
 *   1,400 LoRA tensors in a list                          1,547 -> 87 us (the kernel's time)
 *   400 ragged tensors, bf16 and fp32, in a list            445 -> 36 us (the same)
 *   256 short tensors, clipped, gradients at new addresses  349 -> 75 us
 *   60 named tensors, each with a new output                202 -> 61 us (60 allocations; 79 through the dispatcher)
 *
 * Only plain cases are taken here: exact torch.Tensor / torch.nn.Parameter objects with a storage of their own, strided
 * and contiguous, no __torch_function__ mode active, a gradient that the step reads as it is.  Everything else is
 * handed back untouched and goes through the Python code, which is the definition of both calls.
 */
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/EmptyTensor.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/detail/CUDAHooksInterface.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <memory>
#include <vector>

#include "../../include/eri_adam8bit.h"

namespace {

using Held = std::vector<at::Tensor>;
constexpr const char *kHeldName = "eridiffusion_amd.held_tensors";

void held_destroy(PyObject *capsule) { delete static_cast<Held *>(PyCapsule_GetPointer(capsule, kHeldName)); }

/* A Python object that keeps tensors alive; takes the vector over. */
PyObject *held_object(std::unique_ptr<Held> &held) {
    PyObject *c = PyCapsule_New(held.get(), kHeldName, held_destroy);
    if (c) held.release();
    return c;
}

/* The tensor inside a plain tensor object, or null. */
const at::Tensor *plain(PyObject *o) {
    if (!THPVariable_CheckTypeExact(Py_TYPE(o))) return nullptr;
    const at::Tensor &t = THPVariable_Unpack(o);
    return t.defined() && t.layout() == at::kStrided && t.has_storage() && t.is_contiguous() ? &t : nullptr;
}

/* ERI_DTYPE_* of a tensor the optimizers take, or -1. */
int dtype_tag(const at::Tensor &t) {
    return t.scalar_type() == at::kFloat ? ERI_DTYPE_F32 : t.scalar_type() == at::kBFloat16 ? ERI_DTYPE_BF16 : -1;
}

/* Whether a kernel that works on `p` can read t: device memory beside p's, or pinned host memory.  Ordinary host memory
 * in a kernel faults the device. */
bool reachable(const at::Tensor &t, const at::Tensor &p) {
    return t.is_cuda() ? !p.is_cuda() || t.device() == p.device() : t.is_cpu() && t.is_pinned();
}

/* Whether the step reads g as it is: a plain tensor (no subclass where it has a Python object already) of the
 * parameter's dtype, or float32 for a bfloat16 parameter, with an element for each of the parameter's: the launch is
 * sized by the parameter. */
bool grad_as_is(const at::Tensor &g, const at::Tensor &p) {
    PyObject *known = g.unsafeGetTensorImpl()->pyobj_slot()->load_pyobj();
    return (!known || THPVariable_CheckTypeExact(Py_TYPE(known))) && !g.unsafeGetTensorImpl()->is_python_dispatch() && dtype_tag(g) >= 0 &&
           g.layout() == at::kStrided && g.has_storage() && g.is_contiguous() && g.numel() == p.numel() &&
           (g.scalar_type() == p.scalar_type() || (p.scalar_type() == at::kBFloat16 && g.scalar_type() == at::kFloat));
}

/* Whether nothing wants to see or to change the tensors that are made now: no dispatch mode, transform or tracer, no
 * filling of uninitialised memory. */
bool factories_are_plain() {
    if (c10::impl::TorchDispatchModeTLS::any_modes_set()) return false;
    if (c10::impl::tls_local_dispatch_key_set().included_ != c10::default_included_set) return false;
    return !(at::globalContext().deterministicAlgorithms() && at::globalContext().deterministicFillUninitializedMemory());
}

/* Tensors like others, on their devices: what at::empty_strided makes on a device, past the dispatcher. */
struct Outputs {
    const bool direct = factories_are_plain();
    c10::Allocator *const allocator = direct ? at::detail::getCUDAHooks().getCUDADeviceAllocator() : nullptr;
    c10::OptionalDeviceGuard guard;
    at::Tensor like(const at::Tensor &t) {
        if (!direct) return at::empty_strided(t.sizes(), t.strides(), t.options());
        if (guard.current_device() != t.device()) guard.reset_device(t.device());
        return at::detail::empty_strided_generic(t.sizes(), t.strides(), allocator, c10::DispatchKeySet(c10::DispatchKey::CUDA), t.scalar_type());
    }
};

/* What a parameter was when its optimizer was made; handles and states are sized by it. */
struct Made {
    uint64_t numel;
    int64_t dtype_tag;
};

/* bind(params, handles, n[, made]) -> (held, rest): sets data and gradient of the EriParameter at handles[i] from
 * params[i].  `handles` is the address of an array of n pointers; a longer list is an IndexError, before anything is set.
 * `made` is the address of n records: a parameter that has another size or dtype by now, or that kernels cannot reach,
 * is left alone, and so is one with such a gradient.  (Without `made` the caller vouches for that.)  `held` keeps the
 * gradients alive that were read; `rest` lists the indices that were left alone. */
PyObject *face_bind(PyObject *, PyObject *args) {
    PyObject *params;
    unsigned long long handles_addr;
    unsigned long long made_addr = 0;
    Py_ssize_t n_handles;
    if (!PyArg_ParseTuple(args, "O!Kn|K", &PyList_Type, &params, &handles_addr, &n_handles, &made_addr)) return nullptr;
    if (PyList_GET_SIZE(params) > n_handles) {
        PyErr_SetString(PyExc_IndexError, "more parameters than the optimizer was made for");
        return nullptr;
    }
    EriParameter *const *handles = reinterpret_cast<EriParameter *const *>(handles_addr);
    const Made *made = reinterpret_cast<const Made *>(made_addr);
    PyObject *rest = PyList_New(0);
    if (!rest) return nullptr;
    try {
        std::unique_ptr<Held> held(new Held());
        const Py_ssize_t n = PyList_GET_SIZE(params);
        held->reserve((size_t)n);
        const bool general = at::impl::torch_function_mode_enabled();
        for (Py_ssize_t i = 0; i < n; ++i) {
            const at::Tensor *p = general ? nullptr : plain(PyList_GET_ITEM(params, i));
            bool done = false;
            const bool fits = p && (!made || (made[i].numel == (uint64_t)p->numel() && made[i].dtype_tag == dtype_tag(*p) && reachable(*p, *p)));
            if (fits && p->is_leaf()) { // asking for another tensor's gradient warns
                const at::Tensor &g = p->grad();
                void *data = p->data_ptr();
                if (!g.defined()) {
                    done = eri_param_set_data(handles[i], data) == 0 && eri_param_set_grad(handles[i], nullptr) == 0;
                } else if (grad_as_is(g, *p) && (!made || reachable(g, *p))) {
                    done = eri_param_set_data(handles[i], data) == 0 && eri_param_set_grad_typed(handles[i], g.data_ptr(), dtype_tag(g)) == 0;
                    if (done) held->push_back(g);
                }
            }
            if (!done) {
                PyObject *k = PyLong_FromSsize_t(i);
                if (!k || PyList_Append(rest, k) != 0) {
                    Py_XDECREF(k);
                    Py_DECREF(rest);
                    return nullptr;
                }
                Py_DECREF(k);
            }
        }
        PyObject *h = held_object(held);
        if (!h) {
            Py_DECREF(rest);
            return nullptr;
        }
        return Py_BuildValue("NN", h, rest);
    } catch (const std::exception &) {
        Py_DECREF(rest);
        torch::translate_exception_to_python(std::current_exception());
        return nullptr;
    }
}

/* update_many(optimizer, params, grads) -> None if any tensor needs the general path, else (code, outs, held): the new
 * tensors by name, filled by a launch that has been queued if `code` is 0. */
PyObject *face_update_many(PyObject *, PyObject *args) {
    unsigned long long opt_addr;
    PyObject *params, *grads;
    if (!PyArg_ParseTuple(args, "KO!O!", &opt_addr, &PyDict_Type, &params, &PyDict_Type, &grads)) return nullptr;
    if (!PyDict_CheckExact(params) || !PyDict_CheckExact(grads) || at::impl::torch_function_mode_enabled()) Py_RETURN_NONE;
    PyObject *outs = nullptr, *keys = nullptr;
    try {
        std::unique_ptr<Held> held(new Held());
        std::vector<const char *> names;
        std::vector<at::Tensor> ps, gs;
        keys = PyList_New(0); // the names stay valid while the lock is given up below
        if (!keys) return nullptr;
        Py_ssize_t pos = 0;
        PyObject *key, *value;
        while (PyDict_Next(params, &pos, &key, &value)) {
            const char *name = PyUnicode_CheckExact(key) ? PyUnicode_AsUTF8(key) : nullptr;
            PyObject *grad = name ? PyDict_GetItemWithError(grads, key) : nullptr;
            if (!name || (!grad && PyErr_Occurred())) {
                PyErr_Clear();
                Py_DECREF(keys);
                Py_RETURN_NONE;
            }
            if (!grad) continue;
            const at::Tensor *p = plain(value), *g = plain(grad);
            if (!p || !g || !p->is_cuda() || dtype_tag(*p) < 0 || !grad_as_is(*g, *p) || !reachable(*g, *p)) {
                Py_DECREF(keys);
                Py_RETURN_NONE;
            }
            if (PyList_Append(keys, key) != 0) {
                Py_DECREF(keys);
                return nullptr;
            }
            names.push_back(name);
            ps.push_back(*p);
            gs.push_back(*g);
        }
        const size_t k = names.size();
        if (k == 0) {
            Py_DECREF(keys);
            Py_RETURN_NONE;
        }
        std::vector<const void *> p_ptr(k), g_ptr(k);
        std::vector<void *> o_ptr(k);
        std::vector<uint64_t> numel(k);
        std::vector<int32_t> p_tag(k), g_tag(k);
        held->reserve(3 * k);
        outs = PyDict_New();
        if (!outs) {
            Py_DECREF(keys);
            return nullptr;
        }
        std::vector<at::Tensor> fresh(k);
        {
            Outputs made; // its device guard ends before the launch
            for (size_t i = 0; i < k; ++i) fresh[i] = made.like(ps[i]);
        }
        for (size_t i = 0; i < k; ++i) {
            at::Tensor &out = fresh[i];
            p_ptr[i] = ps[i].data_ptr();
            g_ptr[i] = gs[i].data_ptr();
            o_ptr[i] = out.data_ptr();
            numel[i] = (uint64_t)ps[i].numel();
            p_tag[i] = dtype_tag(ps[i]);
            g_tag[i] = dtype_tag(gs[i]);
            PyObject *wrapped = THPVariable_Wrap(out);
            if (!wrapped || PyDict_SetItem(outs, PyList_GET_ITEM(keys, (Py_ssize_t)i), wrapped) != 0) {
                Py_XDECREF(wrapped);
                Py_DECREF(outs);
                Py_DECREF(keys);
                return nullptr;
            }
            Py_DECREF(wrapped);
            held->push_back(std::move(ps[i]));
            held->push_back(std::move(gs[i]));
            held->push_back(std::move(out));
        }
        int rc = 0;
        Py_BEGIN_ALLOW_THREADS
        rc = eri_adam8bit_fn_update_many(reinterpret_cast<EriAdam8bitFn *>(opt_addr), names.data(), p_ptr.data(), g_ptr.data(),
                                         numel.data(), p_tag.data(), g_tag.data(), o_ptr.data(), (uint32_t)k);
        Py_END_ALLOW_THREADS
        Py_DECREF(keys);
        keys = nullptr;
        PyObject *h = held_object(held);
        if (!h) {
            Py_DECREF(outs);
            return nullptr;
        }
        return Py_BuildValue("iNN", rc, outs, h);
    } catch (const std::exception &) { // out of memory reaches Python as torch.OutOfMemoryError, which trainers catch
        Py_XDECREF(keys);
        Py_XDECREF(outs);
        torch::translate_exception_to_python(std::current_exception());
        return nullptr;
    }
}

PyMethodDef methods[] = {{"bind", face_bind, METH_VARARGS, nullptr},
                         {"update_many", face_update_many, METH_VARARGS, nullptr},
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_torch_face", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

} // namespace

extern "C" __attribute__((visibility("default"))) PyObject *PyInit__torch_face(void) { return PyModule_Create(&module); }
