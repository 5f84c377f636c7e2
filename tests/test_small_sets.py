"""Which small sets of buckets run in common launches, in order and on streams (shapes on the meta
device, the plan reads no data)."""

import pytest
import torch

from muonium_amd import Muon
from muonium_amd.optim import optim as driver
from muonium_amd.optim.algorithms import get_algorithm


def _route(monkeypatch, shapes):
    monkeypatch.setattr(driver, "_compute_units", lambda device: 256)
    monkeypatch.setattr(driver, "_side_stream", lambda device, slot: ("side", slot))
    used = []
    monkeypatch.setattr(driver, "_wait", lambda *a: None)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda d=None: None)

    class on:
        def __init__(self, stream):
            pass

        def __enter__(self):
            used.append("stream")

        def __exit__(self, *exc):
            pass

    class grouped(on):
        def __init__(self):
            pass

        def __enter__(self):
            used.append("group")

    monkeypatch.setattr(torch.cuda, "stream", on)
    monkeypatch.setattr(driver, "grouped", grouped)
    device = torch.device("cuda", 0)
    buckets = [(device, None, [torch.empty(s, device="meta")], None, None) for s in shapes]
    slots, order = driver._concurrent_plan(buckets, get_algorithm("muon"), None)
    ran = []
    driver._run_on_streams(buckets, slots, order, ran.append)
    assert sorted(ran) == list(range(len(shapes)))
    return used[0] if used else "order"


@pytest.mark.parametrize("shapes, route", [
    ([(128, 256), (256, 512)], "group"),
    # one bucket that fills the device by itself
    ([(300, 128, 128), (128, 512), (256, 256)], "group"),
    ([(300, 128, 128), (300, 128, 256), (128, 512), (256, 256)], "stream"),
    # past the bound of common launches
    ([(4, 1024, 1024), (1024, 4096), (2048, 1024)], "stream"),
    # iterates of at most 64 rows: in order, but for the widest
    ([(64, 128), (128, 64), (80, 80)], "order"),
    ([(64, 1024), (128, 512), (256, 256)], "order"),
    ([(64, 32768), (48, 1024)], "order"),
    ([(64, 32769), (48, 1024)], "stream"),
    ([(64, 1024), (6, 2048, 2048), (4, 2048, 4096)], "stream"),
    ([(4096, 4096)], "order"),
])
def test_route_of_a_set(monkeypatch, shapes, route):
    assert _route(monkeypatch, shapes) == route


@pytest.mark.gpu
@pytest.mark.parametrize("foreach", [True, False])
@pytest.mark.parametrize("shapes", [
    [(300, 128, 128), (128, 512), (256, 256)],           # one large bucket: common launches
    [(64, 1024), (128, 512), (256, 256), (40, 100)]])    # short iterates: in order
def test_sets_equal_one_bucket_at_a_time(monkeypatch, shapes, foreach):
    def steps():
        gen = torch.Generator(device="cuda").manual_seed(3)
        ps = [torch.nn.Parameter(torch.randn(s, generator=gen, device="cuda")) for s in shapes]
        opt = Muon([{"params": ps}], lr=0.02, foreach=foreach)
        for _ in range(2):
            for p in ps:
                p.grad = torch.randn(p.shape, generator=gen, device="cuda")
            opt.step()
        return ps

    got = steps()
    monkeypatch.setattr(driver, "_concurrent_plan", lambda b, a, n: ({}, list(range(len(b)))))
    for x, y in zip(got, steps()):
        assert torch.equal(x, y)
