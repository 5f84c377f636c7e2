"""NorMuon's row sums at the edges of their kernels: tall matrices by 8 rows per lane (launches that
fill the device), by 2 and one by one, wide ones by 8 columns and one by one, fewer rows than a
wave takes, ragged ends."""

import pytest
import torch
import torch.nn as nn

from muonium_amd import Muon
from muonium_amd.orthogonalize import foreach_zeropower

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("shape, count", [
    ((4096, 128), 64), ((4104, 72), 60), ((2050, 70), 2), ((2048, 513), 1), ((2049, 71), 2),
    ((130, 66), 3), ((17, 1000), 2), ((16, 1001), 1), ((66, 520), 3), ((100, 100), 1),
    ((2, 70, 1024), 2)])
def test_variance_is_the_mean_square_of_each_row(shape, count):
    """From a zero variance: v = (1 - beta2) mean(U^2) per row (fp32 sums in another order: 1e-5)."""
    gen = torch.Generator(device=DEV).manual_seed(sum(shape))
    ps = [nn.Parameter(torch.randn(shape, generator=gen, device=DEV)) for _ in range(count)]
    gs = [torch.randn(shape, generator=gen, device=DEV) for _ in range(count)]
    for p, g in zip(ps, gs):
        p.grad = g.clone()
    opt = Muon([{"params": ps, "algorithm": "normuon", "muon_beta2": 0.75}], lr=0.01, momentum=0.5,
               nesterov=False, foreach=True)
    opt.step()
    for p, u in zip(ps, foreach_zeropower(gs, strategy="polar_express")):
        want = 0.25 * u.double().square().mean(-1, keepdim=True)
        torch.testing.assert_close(opt.state[p]["variance_neuron"].double(), want, rtol=1e-5, atol=0)
