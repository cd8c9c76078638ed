// The eager step of fused_lncc_loss on plain tensors, in C++: argument checks, output allocation, the
// library's launches and the autograd node. Same behaviour as the Python autograd function of
// fused_lncc/__init__.py (which stays for everything else: traced, transformed, unusual or wrong
// arguments, for which step() returns None without doing anything); what it saves is the
// interpreter's share of a small step, in the forward call and, more, in the backward one, where a
// Python node makes the autograd thread take the interpreter lock.
//
// A Python extension module without a link to the HIP library: init() receives the addresses of the C
// ABI's functions and the package's error class from the loader, so that both paths use the one library
// that it loaded and raise the same errors.
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/Exceptions.h>
#include <ATen/ATen.h>
#include <c10/core/DeviceGuard.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>

#include "../../include/fused_lncc.h"

namespace {

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

// The C ABI (include/fused_lncc.h), in the order of init()'s arguments.
struct Api {
    decltype(&fl_validate) validate;
    decltype(&fl_workspace_bytes) workspace_bytes;
    decltype(&fl_lncc_loss_grad) loss_grad;
    decltype(&fl_lncc_loss_grad_pt) loss_grad_pt;
    decltype(&fl_scale_grad) scale_grad;
    decltype(&fl_last_error) last_error;
    PyObject* error;   // FusedLNCCError(code, message)
} api;

int dtype_code(const Tensor& t) {
    return t.scalar_type() == at::kFloat ? FL_F32 : t.scalar_type() == at::kBFloat16 ? FL_BF16 : -1;
}

// The library's refusal as the Python path raises it; called with or without the interpreter lock, on the
// caller's or on an autograd thread (which hands a Python error on to the one that waits for it).
void check(int rc) {
    if (rc == FL_OK) return;
    const std::string msg = api.last_error();
    pybind11::gil_scoped_acquire gil;
    PyObject* text = PyUnicode_DecodeUTF8(msg.data(), (Py_ssize_t)msg.size(), "replace");
    PyObject* e = text ? PyObject_CallFunction(api.error, "iO", rc, text) : nullptr;
    if (e) PyErr_SetObject(api.error, e);
    Py_XDECREF(e);
    Py_XDECREF(text);
    python_error err;
    err.persist();
    throw err;
}

void* stream_of(const Tensor& t) {
    return c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(t.device().index()).stream();
}

// One forward call on contiguous (N, C, D, H, W) tensors: the loss, and the gradients asked for
// (already multiplied by -1/M).
Tensor launch(const Tensor& p, const Tensor& t, int k, double dr, bool need, bool need_t, Tensor& g, Tensor& gt) {
    c10::DeviceGuard guard(p.device());
    const int64_t B = p.size(0) * p.size(1), D = p.size(2), H = p.size(3), W = p.size(4);
    const int code = dtype_code(p);
    const size_t nbytes = api.workspace_bytes(B, D, H, W, k);
    Tensor ws = at::empty({(int64_t)nbytes}, p.options().dtype(at::kByte));
    Tensor loss = at::empty({}, p.options().dtype(at::kFloat));
    if (need) g = at::empty_like(p);
    if (need_t) {
        gt = at::empty_like(t);
        check(api.loss_grad_pt(p.data_ptr(), t.data_ptr(), code, B, D, H, W, k, (float)dr, loss.data_ptr<float>(),
                               g.data_ptr(), gt.data_ptr(), ws.data_ptr(), nbytes, stream_of(p)));
    } else {
        check(api.loss_grad(p.data_ptr(), t.data_ptr(), code, B, D, H, W, k, (float)dr, loss.data_ptr<float>(),
                            need ? g.data_ptr() : nullptr, ws.data_ptr(), nbytes, stream_of(p)));
    }
    return loss;
}

void scale_(Tensor& g, const Tensor& grad_out) {
    Tensor go = grad_out.detach();
    if (go.scalar_type() != at::kFloat || go.device() != g.device()) go = go.to(g.device(), at::kFloat);
    c10::DeviceGuard guard(g.device());
    check(api.scale_grad(g.data_ptr(), dtype_code(g), g.numel(), go.data_ptr<float>(), stream_of(g)));
}

// need: the pred gradient; need_t: the target gradient as well.
struct FusedLNCC : public torch::autograd::Function<FusedLNCC> {
    static Tensor forward(AutogradContext* ctx, const Tensor& p, const Tensor& t, int64_t k, double dr, bool need_t) {
        Tensor g, gt;
        Tensor loss = launch(p, t, (int)k, dr, true, need_t, g, gt);
        // the inputs are saved for a second backward through a retained graph, which recomputes; the
        // gradients are handed out (scaled in place) by the first one
        ctx->save_for_backward({p, t});
        ctx->saved_data["g"] = std::move(g);
        if (need_t) ctx->saved_data["gt"] = std::move(gt);
        ctx->saved_data["k"] = k;
        ctx->saved_data["dr"] = dr;
        ctx->saved_data["t"] = need_t;
        return loss;
    }
    static variable_list backward(AutogradContext* ctx, variable_list grads) {
        const bool need_t = ctx->saved_data["t"].toBool();
        Tensor g, gt;
        auto it = ctx->saved_data.find("g");
        if (it != ctx->saved_data.end()) {
            g = std::move(it->second).toTensor();
            ctx->saved_data.erase("g");
            if (need_t) {
                gt = std::move(ctx->saved_data["gt"]).toTensor();
                ctx->saved_data.erase("gt");
            }
        } else {
            const variable_list in = ctx->get_saved_variables();
            launch(in[0], in[1], (int)ctx->saved_data["k"].toInt(), ctx->saved_data["dr"].toDouble(), true, need_t, g, gt);
        }
        scale_(g, grads[0]);
        if (need_t) scale_(gt, grads[0]);
        return {std::move(g), std::move(gt), Tensor(), Tensor(), Tensor()};
    }
};

// step(pred, target, kernel_size, smooth_dr, target_grad) -> loss, or None where the Python path takes
// over: anything but two plain float32 or bfloat16 GPU tensors of one device, type and 5-d shape that
// the library accepts, or a target that requires grad where pred does not.
PyObject* step(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    if (nargs != 5 || !THPVariable_Check(args[0]) || !THPVariable_Check(args[1])) Py_RETURN_NONE;
    const long k = PyLong_AsLong(args[2]);
    const double dr = PyFloat_AsDouble(args[3]);
    if (PyErr_Occurred()) {   // a kernel size past long: the Python path's refusal
        PyErr_Clear();
        Py_RETURN_NONE;
    }
    const Tensor pred = THPVariable_Unpack(args[0]), target = THPVariable_Unpack(args[1]);
    const int code = dtype_code(pred);
    if (!pred.is_cuda() || pred.device() != target.device() || code < 0 || target.scalar_type() != pred.scalar_type() ||
        pred.dim() != 5 || pred.sizes() != target.sizes() || pred.layout() != at::kStrided || target.layout() != at::kStrided ||
        pred.is_neg() || target.is_neg() || pred._is_zerotensor() || target._is_zerotensor() || k < 0 || k > 1000 ||
        api.validate(code, (int)k, pred.size(0) * pred.size(1), pred.size(2), pred.size(3), pred.size(4)) != FL_OK)
        Py_RETURN_NONE;
    const bool grad_on = at::GradMode::is_enabled();
    const bool need = grad_on && pred.requires_grad();
    const bool need_t = grad_on && args[4] == Py_True && target.requires_grad();
    if (!need && grad_on && target.requires_grad()) Py_RETURN_NONE;   // the node then belongs to the target
    Tensor loss;
    {
        pybind11::gil_scoped_release nogil;
        const Tensor p = pred.contiguous(), t = target.contiguous();
        if (need) {
            loss = FusedLNCC::apply(p, t, (int64_t)k, dr, need_t);
        } else {
            Tensor none, none_t;
            loss = launch(p, t, (int)k, dr, false, false, none, none_t);
        }
    }
    return THPVariable_Wrap(std::move(loss));
    END_HANDLE_TH_ERRORS
}

PyObject* init(PyObject*, PyObject* args) {
    unsigned long long a[6];
    PyObject* error;
    if (!PyArg_ParseTuple(args, "KKKKKKO", &a[0], &a[1], &a[2], &a[3], &a[4], &a[5], &error)) return nullptr;
    Py_INCREF(error);
    Py_XDECREF(api.error);
    api.error = error;
    api.validate = reinterpret_cast<decltype(api.validate)>(a[0]);
    api.workspace_bytes = reinterpret_cast<decltype(api.workspace_bytes)>(a[1]);
    api.loss_grad = reinterpret_cast<decltype(api.loss_grad)>(a[2]);
    api.loss_grad_pt = reinterpret_cast<decltype(api.loss_grad_pt)>(a[3]);
    api.scale_grad = reinterpret_cast<decltype(api.scale_grad)>(a[4]);
    api.last_error = reinterpret_cast<decltype(api.last_error)>(a[5]);
    Py_RETURN_NONE;
}

PyMethodDef methods[] = {
    {"step", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)(void)>(step)), METH_FASTCALL, nullptr},
    {"init", init, METH_VARARGS, nullptr},
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_step", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

// TORCH: the torch that this was compiled against, whose object layouts it uses; FL_VERSION: the C ABI's
// version whose signatures it calls. The loader compares both before init().
PyMODINIT_FUNC PyInit__step(void) {
    PyObject* m = PyModule_Create(&module);
    if (m && (PyModule_AddStringConstant(m, "TORCH", FL_TORCH) < 0 || PyModule_AddIntConstant(m, "FL_VERSION", FL_VERSION) < 0)) {
        Py_DECREF(m);
        return nullptr;
    }
    return m;
}
