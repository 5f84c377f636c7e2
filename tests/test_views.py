"""Parameters (or gradients) that share memory are never stepped side by side: the driver's own
look at the tensors on the CPU, and on the device the results of one bucket after the other."""

import pytest
import torch
import torch.nn as nn

from muonium_amd import Muon
from muonium_amd.optim import optim as driver

DEV = "cuda"


class Sub(nn.Parameter):
    """A parameter type of a user's own."""


class Opaque(torch.Tensor):
    """A tensor without storage of its own."""

    @staticmethod
    def __new__(cls, t):
        return torch.Tensor._make_wrapper_subclass(cls, t.shape, dtype=t.dtype)

    @classmethod
    def __torch_dispatch__(cls, func, types, args=(), kwargs=None):
        raise RuntimeError("opaque")


def _w(*shape):
    return torch.zeros(*shape)


W = _w(96, 160)
FLAT = _w(2 * 64 * 96)
CASES = [
    ("apart", [_w(4, 8), _w(4, 8), _w(8, 4)], False),
    ("neighbours in one storage", [FLAT[:64 * 96].view(64, 96), FLAT[64 * 96:].view(96, 64)], False),
    ("transpose", [W, W.T], True),
    ("block", [_w(8, 8), W[:48, :80], W], True),
    ("row blocks", [W[:48], W[48:]], False),
    ("blocks that overlap", [W[:49], W[48:]], True),
    ("of a parameter subclass", [Sub(W), Sub(W.T)], True),
    ("empty views", [W[:0], W], False),
    ("no storage", [Opaque(W), _w(4, 8)], True),
]


@pytest.mark.parametrize("tensors, shared", [c[1:] for c in CASES], ids=[c[0] for c in CASES])
def test_shared_memory_is_found(tensors, shared):
    assert driver._share_memory(tensors) is shared


@pytest.mark.parametrize("foreach", [True, False])
@pytest.mark.parametrize("what", ["params", "subclass", "grads", "none"])
def test_plan_of_shared_tensors_is_one_after_the_other(monkeypatch, foreach, what):
    """A planner that puts every bucket on a stream of its own, overruled where memory is shared
    (gradients: by the foreach driver, which writes them)."""
    plans = []
    monkeypatch.setattr(driver, "_concurrent_plan",
                        lambda b, *a: ({i: i for i in range(len(b))}, list(range(len(b)))[::-1]))
    monkeypatch.setattr(driver, "_run_on_streams",
                        lambda b, slots, order, *a, **k: plans.append((slots, order)))
    make = Sub if what == "subclass" else nn.Parameter
    base = torch.randn(96, 160)
    ps = [make(base), make(base.T if what in ("params", "subclass") else torch.randn(160, 96))]
    grad = torch.randn(96, 160)
    ps[0].grad, ps[1].grad = grad, grad.T if what == "grads" else torch.randn(160, 96)
    Muon([{"params": ps}], foreach=foreach).step()
    alone = what in ("params", "subclass") or (what == "grads" and foreach)
    assert plans == [({}, [0, 1])] if alone else plans == [({0: 0, 1: 1}, [1, 0])]


def _steps(shapes, foreach, make=nn.Parameter):
    """Two steps on views of one weight (row and column offset, shape, transposed)."""
    gen = torch.Generator().manual_seed(9)
    w = torch.randn(2048, 1024, generator=gen).to(DEV)
    ps = []
    for r, c, transposed in shapes:
        v = w[:r, :c]
        ps.append(make(v.T if transposed else v))
    opt = Muon([{"params": ps}], lr=0.02, foreach=foreach)
    for _ in range(2):
        for p in ps:
            p.grad = torch.randn(p.shape, generator=gen).to(DEV)
        opt.step()
    torch.cuda.synchronize()
    return w


@pytest.mark.gpu
@pytest.mark.parametrize("make", [nn.Parameter, Sub])
@pytest.mark.parametrize("foreach", [True, False])
@pytest.mark.parametrize("shapes", [
    [(256, 512, False), (256, 512, True), (128, 256, False)],          # common launches' size
    [(2048, 1024, False), (2048, 1024, True), (1024, 768, False)],     # the streams'
    [(256, 512, False), (256, 512, False), (128, 256, False)],         # two of one shape
])
def test_views_are_stepped_one_after_the_other(monkeypatch, shapes, foreach, make):
    if foreach and shapes[0] == shapes[1]:
        pytest.skip("one bucket: the reference stacks its tensors")
    got = _steps(shapes, foreach, make)
    monkeypatch.setattr(driver, "_concurrent_plan", lambda b, a, n: ({}, list(range(len(b)))))
    monkeypatch.setattr(driver, "_per_tensor_runs", lambda p, *a: [[i] for i in range(len(p))])
    assert torch.equal(got, _steps(shapes, foreach, make))
