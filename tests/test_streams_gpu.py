"""The per-parameter driver's same-shape runs on side streams: the results of one run after the
other bit for bit, for each algorithm and momentum format, with a caller's own stream, with a
large run beside small ones, and from several threads at a time."""

import threading

import pytest
import torch
import torch.nn as nn

from muonium_amd import Muon, Muon8bit
from muonium_amd.optim import optim as driver

pytestmark = pytest.mark.gpu
DEV = "cuda"
SHAPES = [(256, 512)] * 2 + [(512, 256)] * 2 + [(130, 300)] + [(384, 1024)] * 3
LARGE = SHAPES + [(4096, 1024)] * 40


def _steps(cls, shapes, seed, plan=True, **kw):
    gen = torch.Generator().manual_seed(seed)
    ps = [nn.Parameter(torch.randn(s, generator=gen).to(DEV)) for s in shapes]
    opt = cls([{"params": ps, **kw}], lr=0.02, foreach=False,
              **({"block_size": 256} if cls is Muon8bit else {}))
    for _ in range(3):
        for p in ps:
            p.grad = torch.randn(p.shape, generator=gen).to(DEV)
        opt.step()
    torch.cuda.current_stream().synchronize()
    return [p.detach().clone() for p in ps]


def _one_after_the_other(monkeypatch):
    monkeypatch.setattr(driver, "_concurrent_plan", lambda b, a, n: ({}, list(range(len(b)))))


@pytest.mark.parametrize("cls, kw, shapes", [
    (Muon, {}, SHAPES), (Muon, {"algorithm": "normuon"}, SHAPES), (Muon8bit, {}, SHAPES),
    (Muon, {}, LARGE)])
def test_runs_on_streams_equal_runs_in_order(monkeypatch, cls, kw, shapes):
    side = torch.cuda.Stream()
    got = _steps(cls, shapes, 3, **kw)
    with torch.cuda.stream(side):
        own = _steps(cls, shapes, 3, **kw)
    _one_after_the_other(monkeypatch)
    want = _steps(cls, shapes, 3, **kw)
    for a, b, c in zip(got, own, want):
        assert torch.equal(a, c) and torch.equal(b, c)


def test_threads_do_not_share_side_streams(monkeypatch):
    out = {}

    def work(seed):
        with torch.cuda.stream(torch.cuda.Stream()):
            out[seed] = _steps(Muon, SHAPES, seed)

    threads = [threading.Thread(target=work, args=(s,)) for s in range(3)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    _one_after_the_other(monkeypatch)
    for seed in range(3):
        for a, b in zip(out[seed], _steps(Muon, SHAPES, seed)):
            assert torch.equal(a, b)
