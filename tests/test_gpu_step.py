"""The eager step extension against the Python autograd function, call by call: the same bits, the same
gradients handed out, the same refusals; and the calls that are to keep the Python function."""
import contextlib

import pytest
import torch
import torch.utils.checkpoint

import fused_lncc
import workloads as wl
from fused_lncc import _lib, fused_lncc_loss

pytestmark = pytest.mark.gpu
DEV = "cuda"


@contextlib.contextmanager
def python_path(monkeypatch):
    with monkeypatch.context() as m:
        m.setattr(_lib, "_step", False)
        yield


def both(monkeypatch, f):
    """f() through the extension and through the Python function."""
    assert _lib.eager_step() is not None
    got = f()
    with python_path(monkeypatch):
        want = f()
    return got, want


def pair(shape=(2, 2, 9, 20, 24), dtype=torch.float32, seed=3):
    p, t = wl.randn_pair(shape, seed)
    return p.to(dtype).to(DEV), t.to(dtype).to(DEV)


def same(a, b):
    assert (a is None) == (b is None)
    if a is not None:
        assert a.dtype == b.dtype and a.shape == b.shape and a.requires_grad == b.requires_grad and torch.equal(a, b)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("k", [3, 9])
@pytest.mark.parametrize("weight", [1.0, 0.25])
@pytest.mark.parametrize("target_grad", [False, True])
@pytest.mark.parametrize("shape", [(2, 2, 9, 20, 24), (3, 1, 8, 7, 6)])
def test_step(monkeypatch, dtype, k, weight, target_grad, shape):
    def f():
        p, t = pair(shape, dtype)
        p.requires_grad_(True)
        t.requires_grad_(True)
        loss = fused_lncc_loss(p, t, k, 1e-4, target_grad=target_grad)
        (weight * loss).backward()
        return loss.detach(), p.grad, t.grad
    for a, b in zip(*both(monkeypatch, f)):
        same(a, b)


@pytest.mark.parametrize("pg,tg,on", [(False, False, True), (False, True, True), (True, False, False), (True, True, True)])
@pytest.mark.parametrize("target_grad", [False, True])
def test_what_requires_grad(monkeypatch, pg, tg, on, target_grad):
    def f():
        p, t = pair()
        p.requires_grad_(pg)
        t.requires_grad_(tg)
        with torch.set_grad_enabled(on):
            loss = fused_lncc_loss(p, t, 5, target_grad=target_grad)
        if loss.requires_grad:
            loss.backward()
        return loss, p.grad, t.grad
    for a, b in zip(*both(monkeypatch, f)):
        same(a, b)


def test_views_and_non_leaves(monkeypatch):
    def f():
        p, t = pair((1, 4, 10, 12, 14))
        x = p.requires_grad_(True)
        loss = fused_lncc_loss((2 * x).transpose(3, 4), t.transpose(3, 4), 7)   # contiguous copies, through autograd
        loss.backward()
        q = p.detach()[:, 1:3].requires_grad_(True)                             # a view at an offset
        fused_lncc_loss(q, t[:, 1:3], 7).backward()
        return loss.detach(), x.grad, q.grad
    for a, b in zip(*both(monkeypatch, f)):
        same(a, b)


@pytest.mark.parametrize("target_grad", [False, True])
def test_retained_graph_recomputes(monkeypatch, target_grad):
    def f():
        p, t = pair()
        p.requires_grad_(True)
        t.requires_grad_(target_grad)
        loss = fused_lncc_loss(p, t, 7, target_grad=target_grad)
        wrt = (p, t) if target_grad else (p,)
        first = torch.autograd.grad(loss, wrt, retain_graph=True)
        second = torch.autograd.grad(3.0 * loss, wrt)
        with pytest.raises(RuntimeError, match="second time"):
            torch.autograd.grad(loss, wrt)
        return first + second
    for a, b in zip(*both(monkeypatch, f)):
        same(a, b)


def test_inputs_changed_in_place(monkeypatch):
    """The first backward hands out what the forward formed; one that recomputes refuses inputs that
    were changed since."""
    def f():
        p, t = pair()
        x = p.requires_grad_(True) * 1.0
        loss = fused_lncc_loss(x, t, 7)
        t.add_(1.0)
        (g,) = torch.autograd.grad(loss, x, retain_graph=True)
        with pytest.raises(RuntimeError, match="modified by an inplace operation"):
            torch.autograd.grad(loss, x)
        return (g,)
    for a, b in zip(*both(monkeypatch, f)):
        same(a, b)


def test_hooks_create_graph_and_streams(monkeypatch):
    def f():
        seen = []
        p, t = pair()
        p.requires_grad_(True)
        with torch.autograd.graph.saved_tensors_hooks(lambda x: (seen.append(x.shape), x.clone())[1], lambda x: x):
            loss = fused_lncc_loss(p, t, 7)
        torch.autograd.grad(loss, p, retain_graph=True)
        (again,) = torch.autograd.grad(loss, p, create_graph=True)
        s = torch.cuda.Stream()
        s.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(s):
            side = fused_lncc_loss(p, t, 7)
            side.backward()
        torch.cuda.current_stream().wait_stream(s)
        return (torch.tensor(len(seen)), again.detach(), torch.tensor(again.requires_grad), side.detach(), p.grad)
    for a, b in zip(*both(monkeypatch, f)):
        same(a, b)


def checkpointed(reentrant):
    def f():
        p, t = pair()
        p.requires_grad_(True)
        loss = torch.utils.checkpoint.checkpoint(lambda x: fused_lncc_loss(2.0 * x, t, 7), p, use_reentrant=reentrant)
        loss.backward()
        return loss.detach(), p.grad
    return f


def checkpointed_retained():
    """The second backward needs the saved inputs, which the checkpoint forms again."""
    p, t = pair()
    p.requires_grad_(True)
    loss = torch.utils.checkpoint.checkpoint(lambda x: fused_lncc_loss(2.0 * x, t, 7), p, use_reentrant=False)
    return torch.autograd.grad(loss, p, retain_graph=True) + torch.autograd.grad(loss, p)


def anomaly_mode():
    p, t = pair()
    with torch.autograd.detect_anomaly(check_nan=True):
        loss = fused_lncc_loss(p.requires_grad_(True), t, 7)
        loss.backward()
        bad = fused_lncc_loss(p, torch.full_like(t, float("nan")), 7)
        assert torch.isnan(bad).item()
        with pytest.raises(RuntimeError, match="nan values"):
            torch.autograd.grad(bad, p)
    return loss.detach(), p.grad


def inference_mode():
    p, t = pair()
    with torch.inference_mode():
        loss = fused_lncc_loss(p.requires_grad_(True), t, 7)
        assert loss.is_inference() and not loss.requires_grad
        u = t.clone()   # an inference tensor: no graph can save it
    with pytest.raises(RuntimeError, match="Inference tensors cannot be saved"):
        fused_lncc_loss(p, u, 7)
    return (loss.clone(),)


def compiled_autograd():
    from torch._dynamo import compiled_autograd as ca
    p, t = pair()
    loss = fused_lncc_loss(p.requires_grad_(True), t, 7)
    graphs = []
    with ca._enable(lambda gm: (graphs.append(gm), torch.compile(gm, backend="eager"))[1]):
        loss.backward()
    assert len(graphs) == 1
    return loss.detach(), p.grad


@pytest.mark.filterwarnings("ignore:Anomaly Detection:UserWarning", "ignore:Error detected:UserWarning")
@pytest.mark.parametrize("f", [checkpointed(False), checkpointed(True), checkpointed_retained, anomaly_mode, inference_mode,
                               compiled_autograd], ids=lambda f: f.__qualname__.split(".")[0])
def test_autograd_modes(monkeypatch, f):
    for a, b in zip(*both(monkeypatch, f)):
        same(a, b)


def test_threads(monkeypatch):
    """Forward and backward from several threads at once, each with its own inputs."""
    import threading

    def f():
        out = [None] * 4

        def work(i):
            p, t = pair(seed=i)
            p.requires_grad_(True)
            for _ in range(10):
                p.grad = None
                fused_lncc_loss(p, t, 7).backward()
            out[i] = p.grad
        threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
        for th in threads:
            th.start()
        for th in threads:
            th.join()
        return out
    for a, b in zip(*both(monkeypatch, f)):
        same(a, b)


def test_refusals_are_the_python_functions(monkeypatch):
    p, t = pair()
    for bad in (lambda: fused_lncc_loss(p.double(), t.double(), 7), lambda: fused_lncc_loss(p, t.bfloat16(), 7),
                lambda: fused_lncc_loss(p.cpu(), t.cpu(), 7), lambda: fused_lncc_loss(p, t, 11), lambda: fused_lncc_loss(p, t, 2 ** 70 + 1),
                lambda: fused_lncc_loss(p, t.cpu(), 7), lambda: fused_lncc_loss(p[:, :0], t[:, :0], 7)):
        def f():
            with pytest.raises(RuntimeError) as e:
                bad()
            return type(e.value), str(e.value)
        got, want = both(monkeypatch, f)
        assert got == want


def error_of(f):
    with pytest.raises(RuntimeError) as e:
        f()
    return type(e.value), getattr(e.value, "code", None), str(e.value)


def test_library_errors_are_the_python_functions(monkeypatch):
    """What the library itself refuses once the arguments are valid (here, on the host, a forced chunk
    length that makes more workgroups than one launch holds) is a FusedLNCCError with its code."""
    x = torch.zeros(2100000, 1, 2, 1, 1, device=DEV)
    with _lib.dchunk(1):
        got, want = both(monkeypatch, lambda: error_of(lambda: fused_lncc_loss(x, x, 3)))
    assert got == want and got[0] is _lib.FusedLNCCError and got[1] == _lib.FL_E_NULL


def test_library_errors_in_backward_are_the_python_functions(monkeypatch):
    """A device error that the backward's library call reports, on the autograd thread, reaches the
    caller as a FusedLNCCError with its code. (A stand-in for fl_scale_grad that launches nothing.)"""
    import ctypes
    from fused_lncc import _step
    lib = _lib.load()
    real = {n: ctypes.cast(getattr(lib, n), ctypes.c_void_p).value for n in _lib._STEP_API}
    fails = ctypes.CFUNCTYPE(ctypes.c_int, *_lib.SIGNATURES["fl_scale_grad"][1])(lambda *a: _lib.FL_E_DEVICE)

    def f():
        p, t = pair()
        loss = fused_lncc_loss(p.requires_grad_(True), t, 7)
        return error_of(loss.backward)
    assert _lib.eager_step() is not None
    try:
        _step.init(*{**real, "fl_scale_grad": ctypes.cast(fails, ctypes.c_void_p).value}.values(), _lib.FusedLNCCError)
        with monkeypatch.context() as m:
            m.setattr(lib, "fl_scale_grad", fails)
            got, want = both(monkeypatch, f)
    finally:
        _step.init(*real.values(), _lib.FusedLNCCError)
    assert got[:2] == want[:2] == (_lib.FusedLNCCError, _lib.FL_E_DEVICE)


def test_watched_calls_keep_the_python_function(monkeypatch):
    calls = []
    step = _lib.eager_step()
    monkeypatch.setattr(_lib, "_step", lambda *a: (calls.append(1), step(*a))[1])
    p, t = pair()
    fused_lncc_loss(p, t, 7)
    assert len(calls) == 1

    class Mode(torch.overrides.TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    with Mode():
        fused_lncc_loss(p, t, 7)
    with pytest.raises(RuntimeError):
        torch.func.vmap(lambda a, b: fused_lncc_loss(a, b, 7))(p[None], t[None])
    with torch.autograd.forward_ad.dual_level():
        d = torch.autograd.forward_ad.make_dual(p, torch.ones_like(p))
        with pytest.raises((RuntimeError, NotImplementedError)):
            fused_lncc_loss(d, t, 7)
    assert fused_lncc._watched() is False and len(calls) == 1
