"""Small buckets in common launches: bit for bit one bucket at a time, for each algorithm, parameter
type, driver and momentum format; tall and wide, with row blocks, non-contiguous parameters, a
partial tile each, more buckets than one launch takes, and two of the same padded extents."""

import pytest
import torch
import torch.nn as nn

from muonium_amd import Muon, Muon8bit
from muonium_amd.optim import optim as driver

pytestmark = pytest.mark.gpu
DEV = "cuda"
SHAPES = [(128, 256)] * 2 + [(256, 128)] + [(200, 72)] * 2 + [(72, 200)] + [(320, 1000)] + [(129, 130)]
MANY = [(72 + 8 * i, 300 - 8 * i) for i in range(11)]


def _steps(cls, shapes, dtype=torch.float32, foreach=True, strided=False, **kw):
    gen = torch.Generator().manual_seed(5)
    ps = []
    for s in shapes:
        p = torch.randn(s, generator=gen).to(dtype).to(DEV)
        ps.append(nn.Parameter(p.T.contiguous().T if strided else p))
    extra = {"block_size": 8} if cls is Muon8bit else {}
    opt = cls([{"params": ps, **kw}], lr=0.02, foreach=foreach, **extra)
    for _ in range(3):
        for p in ps:
            p.grad = torch.randn(p.shape, generator=gen).to(dtype).to(DEV)
        opt.step()
    out = [p.detach().clone() for p in ps] + [p.grad.clone() for p in ps]
    for p in ps:
        for key in ("momentum_buffer", "variance_neuron"):
            v = opt.state[p].get(key)
            if v is not None:
                out.append((v if isinstance(v, torch.Tensor) else v.codes).clone())
    torch.cuda.synchronize()
    return out


@pytest.mark.parametrize("cls, shapes, kw", [
    (Muon, SHAPES, {}),
    (Muon, SHAPES, dict(dtype=torch.bfloat16)),
    (Muon, SHAPES, dict(dtype=torch.float16, use_cautious_wd=False)),
    (Muon, SHAPES, dict(foreach=False)),
    (Muon, SHAPES, dict(strided=True)),
    (Muon, SHAPES, dict(strided=True, dtype=torch.bfloat16, wd=0.0)),
    (Muon, SHAPES, dict(algorithm="normuon")),
    (Muon, SHAPES, dict(algorithm="normuon", strided=True, foreach=False)),
    (Muon, SHAPES, dict(orthogonalization_strategy="newton_schulz", ns_steps=4)),
    (Muon, [(384, 136), (384, 136), (384, 264)], dict(split_sizes=(128, 256))),
    (Muon, MANY, {}),
    (Muon, [(2, 96, 160), (96, 160), (3, 160, 96)], {}),
    (Muon8bit, [(128, 256), (256, 128), (128, 264)], dict(foreach=False)),
])
def test_group_equals_one_bucket_at_a_time(monkeypatch, cls, shapes, kw):
    used = []
    plan = driver._grouped_plan
    monkeypatch.setattr(driver, "_grouped_plan", lambda *a: used.append(plan(*a)) or used[-1])
    got = _steps(cls, shapes, **kw)
    assert used and all(used)
    monkeypatch.setattr(driver, "_concurrent_plan", lambda b, a, n: ({}, list(range(len(b)))))
    for x, y in zip(got, _steps(cls, shapes, **kw)):
        assert torch.equal(x, y)


def test_large_and_short_buckets_stay_out():
    """More tiles than the common launches take, and iterates of at most 64 rows, stay out of
    them."""
    def plan(shapes):
        buckets = [(torch.device(DEV, 0), None, [torch.empty(s, device=DEV)], None, None)
                   for s in shapes]
        return driver._grouped_plan(buckets, {i: 0 for i in range(len(shapes) - 1)})

    assert plan([(128, 256), (256, 512)])
    assert not plan([(4096, 4096), (4096, 4096)])
    assert not plan([(64, 4096), (128, 256)])
