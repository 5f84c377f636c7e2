"""A workspace is one call's from its pre-pass to its last launch, whichever threads call and on
whichever stream: two threads stepping on one stream interleave their launches (a library call
releases the interpreter lock), so neither may write the buffer that the other's iteration reads.
On the CPU, with a library that records the buffers it is given; on the device, threads on one
stream against the same steps one after the other."""

import threading

import pytest
import torch
import torch.nn as nn

from muonium_amd import Muon, Muon8bit, _lib, _ops

DEV = "cuda"


class _Recorder:
    """The library's entry points of a step: sizes from the real library, no launches. A pre-pass
    records its workspace and waits for the other thread's, so both calls are under way there."""

    def __init__(self, real, barrier):
        self.real, self.barrier, self.buffers = real, barrier, {}

    def __getattr__(self, name):
        if name in ("muon_orth_result", "muon_orth_workspace_bytes"):
            return getattr(self.real, name)

        def call(*args):
            if name == "muon_prepass":
                self.buffers.setdefault(threading.get_ident(), []).append(args[12])
                self.barrier.wait(timeout=30)
            return 0

        return call


def _fused(kind):
    t = [torch.zeros(72, 136) for _ in range(3)]
    hp = dict(momentum=0.9, nesterov=True, maximize=False, weight_decay=0.1, cautious_wd=True,
              coeffs=[(3.0, -4.0, 2.0)] * 2, prescale=1.0)
    ratio = [torch.tensor(1.0)]
    if kind == "orthogonalize":
        _ops.orthogonalize(t[:1], hp["coeffs"], prescale=1.0, eps=1e-7, iter_dtype=torch.bfloat16,
                           out_dtype=torch.bfloat16)
    elif kind == "normuon":
        _ops.fused_normuon_step(t[:1], t[1:2], t[2:], [torch.zeros(72, 1)], ratio, 0.1, beta2=0.9,
                                write_back_grad=False, **hp)
    elif kind == "scaled":
        _ops.fused_step(t[:1], t[1:2], t[2:], ratio, 0.1, u_scales=[0.5], write_back_grad=False,
                        **hp)
    else:
        _ops.fused_step(t[:1], t[1:2], t[2:], ratio, 0.1, write_back_grad=False, **hp)


@pytest.mark.parametrize("kind", ["step", "scaled", "normuon", "orthogonalize", "grouped"])
def test_calls_at_the_same_time_have_buffers_of_their_own(monkeypatch, kind):
    lib = _Recorder(_lib.load(), threading.Barrier(2))
    monkeypatch.setattr(_lib, "load", lambda: lib)
    monkeypatch.setattr(_lib, "ensure_device", lambda device: None)
    monkeypatch.setattr(_lib, "stream", lambda device: 0)
    monkeypatch.setattr(_ops, "_check_cuda_contig", lambda ts, what: None)
    monkeypatch.setattr(_ops, "_ws_cache", {})

    def work():
        for _ in range(3):
            if kind == "grouped":
                with _ops.grouped():
                    _fused("step")
                    _fused("normuon")
            else:
                _fused(kind)

    threads = [threading.Thread(target=work) for _ in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    a, b = lib.buffers.values()
    each = 2 if kind == "grouped" else 1  # pre-passes of a call
    assert len(a) == len(b) == 3 * each
    for i in range(0, len(a), each):
        assert len({*a[i:i + each], *b[i:i + each]}) == 2 * each


@pytest.mark.gpu
@pytest.mark.parametrize("cls, shapes, kw", [
    (Muon, [(256, 512)] * 2 + [(130, 300)], {}),                          # common launches
    (Muon, [(256, 512)] * 2 + [(130, 300)], {"algorithm": "normuon"}),
    (Muon, [(2048, 1024)] * 4 + [(1024, 1536)] * 8 + [(128, 256)], {}),   # side streams
    (Muon8bit, [(256, 512), (512, 256)], {"foreach": False}),
    (Muon, [(320, 640)], {}),                                             # one bucket
])
def test_threads_on_one_stream_equal_steps_in_order(cls, shapes, kw):
    def steps(seed):
        gen = torch.Generator().manual_seed(seed)
        ps = [nn.Parameter(torch.randn(s, generator=gen).to(DEV)) for s in shapes]
        opt = cls([{"params": ps, **{k: v for k, v in kw.items() if k != "foreach"}}], lr=0.02,
                  foreach=kw.get("foreach", True), **({"block_size": 256} if cls is Muon8bit else {}))
        for _ in range(6):
            for p in ps:
                p.grad = torch.randn(p.shape, generator=gen).to(DEV)
            opt.step()
        return [p.detach().clone() for p in ps]

    want = {seed: steps(seed) for seed in range(4)}
    out = {}
    stream = torch.cuda.Stream()

    def work(seed):
        with torch.cuda.stream(stream):
            out[seed] = steps(seed)

    threads = [threading.Thread(target=work, args=(s,)) for s in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    for seed in range(4):
        for a, b in zip(out[seed], want[seed]):
            assert torch.equal(a, b)


@pytest.mark.gpu
def test_a_buffer_goes_to_the_next_call_and_is_given_back():
    _ops.release_workspaces()
    dev = torch.device(DEV, 0)
    with _ops.workspace(dev, torch.bfloat16, 2, 128, 256) as (a, cap):
        assert cap == 2
        with _ops.workspace(dev, torch.bfloat16, 1, 128, 256) as (b, _):
            assert a.data_ptr() != b.data_ptr()
    for batch, want in ((1, b), (2, a)):  # the smallest that is large enough
        with _ops.workspace(dev, torch.bfloat16, batch, 128, 256) as (c, _):
            assert c.data_ptr() == want.data_ptr()
    assert sum(len(v) for v in _ops._ws_cache.values()) == 2
    with _ops.workspace(dev, torch.bfloat16, 3, 128, 256) as (_, cap):
        assert cap == 3  # (in the place of the larger of the two)
    assert sum(len(v) for v in _ops._ws_cache.values()) == 2
