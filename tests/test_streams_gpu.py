"""The per-parameter driver's same-shape runs on side streams: the results of one run after the
other bit for bit, for each algorithm and momentum format, with a caller's own stream, with a
large run beside small ones, and from several threads at a time."""

import threading

import pytest
import torch
import torch.nn as nn

from muonium_amd import Muon, Muon8bit, _ops
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


def test_a_weight_that_is_a_view_of_another_follows_it(monkeypatch):
    def run():
        gen = torch.Generator().manual_seed(9)
        w = torch.randn(256, 512, generator=gen).to(DEV)
        ps = [nn.Parameter(w), nn.Parameter(w.T), nn.Parameter(w[:128, :256])]
        for p in ps:
            p.grad = torch.randn(p.shape, generator=gen).to(DEV)
        Muon([{"params": ps}], lr=0.02, foreach=False).step()
        return w

    got = run()
    _one_after_the_other(monkeypatch)
    assert torch.equal(got, run())


@pytest.mark.parametrize("shapes", [[(512, 768)] * 2 + [(512, 1024)] * 2 + [(128, 256)],
                                    [(2048, 1024)] * 2 + [(1024, 1536)] * 8 + [(128, 256)]])
def test_runs_before_one_that_fails_are_stepped(monkeypatch, shapes):
    """In common launches (the first set) and on streams."""
    want = _steps(Muon, shapes, 7)
    impl = _ops._fused_step_impl

    def fail(params, *args):
        if params[0].shape == (128, 256) and fail.step == 2:
            raise ValueError("planted")
        fail.step += params[0].shape == (128, 256)
        impl(params, *args)

    fail.step = 0
    monkeypatch.setattr(_ops, "_fused_step_impl", fail)
    gen = torch.Generator().manual_seed(7)
    ps = [nn.Parameter(torch.randn(s, generator=gen).to(DEV)) for s in shapes]
    opt = Muon([{"params": ps}], lr=0.02, foreach=False)
    for i in range(3):
        for p in ps:
            p.grad = torch.randn(p.shape, generator=gen).to(DEV)
        if i < 2:
            opt.step()
        else:
            with pytest.raises(ValueError, match="planted"):
                opt.step()
    for p, w in zip(ps[:-1], want):
        assert torch.equal(p, w)


def test_workspaces_of_a_side_stream_are_one_threads():
    keys = {}

    def work(i):
        stream = driver._side_stream(torch.device(DEV, 0), 0)
        with torch.cuda.stream(stream), _ops.own_workspaces():
            keys[i] = _ops.workspace(torch.device(DEV, 0), torch.bfloat16, 1, 128, 256)[0]
        barrier.wait()

    barrier = threading.Barrier(12)  # (more side streams than torch has distinct ones)
    for round_ in range(2):
        threads = [threading.Thread(target=work, args=(i,)) for i in range(12)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        assert len({w.data_ptr() for w in keys.values()}) == 12
    driver._side_streams.clear()
    driver._side_stream(torch.device(DEV, 0), 0)  # those of ended threads are given back
    assert {k[-1][1] for k in _ops._ws_cache if isinstance(k[-1], tuple)} <= {threading.get_ident()}
