"""_call.so against the Python path behind it: the same results, bit for bit, for every form that it takes, and NotImplemented -
hence the Python path's own handling - for the others."""
import ctypes
import subprocess
from pathlib import Path

import pytest
import torch

from ffn_kernel_amd import MaskedFFN, MaskedLinear, build, ops
from helpers import note


class PythonOnly:
    linear_fwd = linear_bwd = ffn_fwd = ffn_bwd = staticmethod(lambda *a: NotImplemented)


class Taken:
    """_call.so, and the names of the functions that took the call."""
    def __init__(self):
        self.names = []

    def __getattr__(self, name):
        def call(*args):
            r = getattr(Taken.module, name)(*args)
            if r is not NotImplemented:
                self.names.append(name)
            return r
        return call


@pytest.fixture
def both(monkeypatch):
    """both(f) -> (f() through _call.so, f() without it, the functions of _call.so that took a call)"""
    Taken.module = ops._native()

    def run(f):
        taken = Taken()
        monkeypatch.setattr(ops, "_native", lambda: taken)
        a = f()
        monkeypatch.setattr(ops, "_native", lambda: PythonOnly)
        b = f()
        return a, b, taken.names
    return run


def test_other_arguments_are_left_to_python():
    call = ops._native()
    x, w, mask = torch.zeros(4, 16, dtype=torch.bfloat16), torch.zeros(8, 16, dtype=torch.bfloat16).T, torch.zeros(4, dtype=torch.bool)
    assert call.linear_fwd(x, w, w, mask, None) is NotImplemented  # no GPU
    assert call.linear_fwd(None, w, w, "mask", None) is NotImplemented
    assert call.linear_fwd(x) is NotImplemented
    assert call.linear_bwd(x, x, w, w, mask, None) is NotImplemented
    assert call.ffn_fwd(x, w, w, w, w, w, w, mask, False, None) is NotImplemented
    assert call.ffn_bwd(x, x, w, w, w, w, w, w, mask, None, None) is NotImplemented


def test_an_exception_out_of_a_foreign_call_finds_the_gil_held(tmp_path):
    so = tmp_path / "call_checks.so"
    subprocess.run(build.call_command(Path(__file__).with_name("call_checks.cpp"), so), check=True, capture_output=True)
    assert ctypes.PyDLL(str(so)).cc_gil_held_after_throw() == 1


def same(a, b):
    a, b = (t if isinstance(t, tuple) else (t,) for t in (a, b))
    assert len(a) == len(b)
    for p, q in zip(a, b):
        assert (p is None) == (q is None)
        if p is not None:
            assert p.shape == q.shape and p.stride() == q.stride() and p.dtype == q.dtype and torch.equal(p, q)


def rnd(dev, r, c, std=1.0):
    return (torch.randn(r, c, device=dev) * std).to(torch.bfloat16)


# Rows as packed; further apart, the last column of a wider tensor's slice; forms that the fast kernels or _call.so do not take:
# columns apart, an unaligned start, a width that is no multiple of 8.
def rows(dev, M, K, form):
    if form == "wide":
        return rnd(dev, M, K + 16)[:, 8:8 + K]
    if form == "columns apart":
        return rnd(dev, M, 2 * K)[:, ::2]
    if form == "unaligned":
        return rnd(dev, M, K + 8)[:, 3:3 + K]
    return rnd(dev, M, K)


@pytest.mark.gpu
@pytest.mark.parametrize("M", [1, 2, 64, 65, 300])
@pytest.mark.parametrize("K,form,taken", [(136, "packed", True), (136, "wide", True), (136, "columns apart", False), (136, "unaligned", False),
                                          (100, "packed", False)])
def test_linear(dev, both, M, K, form, taken):
    note(f"native call: linear M={M} K={K} {form}")
    torch.manual_seed(M + K)
    N = 264
    x, g = rows(dev, M, K, form), rows(dev, M, N, form)
    w1, w2, mask = rnd(dev, N, K, 0.05).T, rnd(dev, N, K, 0.05).T, torch.rand(M, device=dev) < 0.5
    a, b, names = both(lambda: ops.masked_linear_forward(x, w1, w2, mask))
    same(a, b)
    single = M == 1 and form == "columns apart"  # (one row: its columns are still apart)
    assert (names == ["linear_fwd"]) == (taken and not single)
    a, b, names = both(lambda: ops.masked_linear_backward(g, x, w1, w2, mask))
    same(a, b)
    assert (names == ["linear_bwd"]) == (taken and not single)
    # weights as [K, N] rows, a mask with a stride: Python
    same(*both(lambda: ops.masked_linear_forward(x, w1.contiguous(), w2.contiguous(), mask))[:2])
    strided = torch.stack([mask, mask], 1).flatten()[::2]
    same(*both(lambda: ops.masked_linear_forward(x, w1, w2, strided))[:2])
    routing = ops.route(mask)
    same(*both(lambda: ops.masked_linear_forward(x, w1, w2, mask, routing=routing))[:2])


@pytest.mark.gpu
@pytest.mark.parametrize("M,form", [(1, "packed"), (1, "wide"), (64, "wide"), (65, "packed"), (65, "unaligned"), (300, "wide"), (300, "unaligned")])
@pytest.mark.parametrize("h", [200, 320])
def test_ffn(dev, both, M, form, h):
    note(f"native call: ffn M={M} h={h} {form}")
    torch.manual_seed(M + h)
    d = 136
    x, g = rows(dev, M, d, form), rows(dev, M, d, form)
    W = [rnd(dev, *s, 0.05).T for s in ((h, d), (d, h), (h, d)) * 2]
    mask = torch.rand(M, device=dev) < 0.5
    same(*both(lambda: ops.masked_ffn_forward(x, *W, mask))[:2])
    a, b, names = both(lambda: ops.masked_ffn_forward(x, *W, mask, save_pre=True))
    same(a, b)
    assert (names == ["ffn_fwd"]) == (form != "unaligned")
    pre = a[1]
    for p in (None, pre):
        a, b, names = both(lambda: ops.masked_ffn_backward(g, x, *W, mask, pre=p))
        same(a, b)
        assert (names == ["ffn_bwd"]) == (form != "unaligned")


@pytest.mark.gpu
def test_errors_and_devices(dev, both):
    """Wrong arguments raise what they raised, from the same place."""
    x, w, mask = rnd(dev, 70, 64), rnd(dev, 32, 64).T, torch.zeros(70, dtype=torch.bool, device=dev)
    for bad in (lambda: ops.masked_linear_forward(x.float(), w, w, mask), lambda: ops.masked_linear_forward(x, w, w, mask[:-1]),
                lambda: ops.masked_linear_forward(x, w, w[:, :-1], mask), lambda: ops.masked_linear_forward(x, w, w, mask.cpu()),
                lambda: ops.masked_linear_forward(x, w, w, mask, routing=ops.route(mask[:-1]))):
        for native in (Taken(), PythonOnly):
            with pytest.MonkeyPatch.context() as m, pytest.raises(ValueError):
                m.setattr(ops, "_native", lambda: native)
                bad()


@pytest.mark.gpu
def test_current_stream_and_autograd(dev, both):
    note("native call: side stream, autograd")
    torch.manual_seed(5)
    x, Wv, Wt, mask = rnd(dev, 200, 128), rnd(dev, 64, 128, 0.05), rnd(dev, 64, 128, 0.05), torch.rand(200, device=dev) < 0.5
    F = [rnd(dev, *s, 0.05) for s in ((192, 128), (128, 192), (192, 128)) * 2]
    side = torch.cuda.Stream()

    def step(op, weights):
        leaves = [t.clone().requires_grad_() for t in (x, *weights)]
        y = op.apply(leaves[0], *[w.T for w in leaves[1:]], mask)
        return (y.detach(), *torch.autograd.grad(y, leaves, torch.ones_like(y)))

    def on_side(op, weights):
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            r = step(op, weights)
        torch.cuda.current_stream().wait_stream(side)
        return r
    for op, weights in ((MaskedLinear, (Wv, Wt)), (MaskedFFN, F)):
        a, b, names = both(lambda: step(op, weights))
        same(a, b)
        assert len(names) == 2
        same(a, both(lambda: on_side(op, weights))[0])


@pytest.mark.gpu
@pytest.mark.parametrize("unsafe", [True, False])
@pytest.mark.parametrize("M", [2, 300])
def test_outputs_without_memory_are_refused(dev, M, unsafe):
    """Under a mode that makes the call's own tensors fake ones - their address reads as zero, or throws - the call raises, and the
    next one runs."""
    import torch._functorch.config as config
    from torch._subclasses.fake_tensor import FakeTensorMode
    note(f"native call: fake outputs M={M} unsafe={unsafe}")
    x, w, mask = rnd(dev, M, 64), rnd(dev, 32, 64).T, torch.rand(M, device=dev) < 0.5
    before = ops.masked_linear_forward(x, w, w, mask)
    with config.patch(fake_tensor_allow_unsafe_data_ptr_access=unsafe), FakeTensorMode(allow_non_fake_inputs=True):
        with pytest.raises((ValueError, RuntimeError)):
            ops.masked_linear_forward(x, w, w, mask)
    assert torch.equal(ops.masked_linear_forward(x, w, w, mask), before)
