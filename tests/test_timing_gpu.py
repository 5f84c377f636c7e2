"""The work that the kernel timing books for a step's launches."""

import pytest
import torch

from muonium_amd import Muon, _lib


@pytest.mark.gpu
@pytest.mark.parametrize("algorithm", ["muon", "normuon"])
def test_work_of_common_launches_is_booked(algorithm):
    """The FLOPs that the timing reports for B X are 2 m m n per matrix and iteration, also where the
    last product's launch carries no apply (NorMuon; rows not a multiple of 8 elements)."""
    shapes = [(128, 256), (256, 128), (200, 132)]
    ps = [torch.nn.Parameter(torch.randn(s, device="cuda")) for s in shapes]
    for p in ps:
        p.grad = torch.randn_like(p)
    opt = Muon([{"params": ps, "algorithm": algorithm}], lr=0.02, foreach=True)
    _lib.timing_enable(True)
    opt.step()
    kern = _lib.timing_read()
    _lib.timing_enable(False)
    want = 5 * sum(2.0 * min(s) ** 2 * max(s) for s in shapes)
    assert kern["syrk_xx"][1] == 5  # (common launches)
    assert kern["gemm_bx"][2] + kern["gemm_bx_apply"][2] == pytest.approx(want, rel=1e-9)
