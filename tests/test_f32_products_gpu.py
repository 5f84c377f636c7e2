"""The fp32 products' 64-row tiles: gram_ of whole tiles (M a multiple of 128, K of 64) at its
smallest and at ragged K-tile counts, the shapes just off it (which take the masked kernel), and
a batch against its members alone."""

import pytest
import torch

from helpers import rel_fro
from muonium_amd.kernels.gram import gram
from muonium_amd.orthogonalize.newton_schulz import ns_loop

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B, M, K", [(1, 128, 64), (3, 128, 192), (2, 384, 320), (1, 256, 4096),
                                     (2, 128, 65), (2, 129, 64), (1, 640, 1024)])
def test_gram_fp32(B, M, K):
    """fp32 sums of K products in any order: a relative error of K 2^-24 at most per product sum, well
    below 1e-5 here; the output is symmetric bit for bit."""
    x = torch.randn(B, M, K, generator=torch.Generator().manual_seed(M + K))
    y = gram(x.cuda())
    assert torch.equal(y, y.mT)
    exact = x.double() @ x.double().mT
    assert rel_fro(y.cpu(), exact) <= 1e-5
    assert ((y.cpu().double() - exact).abs() <= K * 2.0 ** -24 * (x.double().abs() @ x.double().abs().mT)).all()


def test_gram_fp32_unaligned_storage():
    """A view one element into its storage is not 16-byte aligned: same values as a copy's."""
    base = torch.randn(1 + 2 * 128 * 64, device="cuda")
    x = base[1:].view(2, 128, 64)
    assert rel_fro(gram(x).cpu(), x.cpu().double() @ x.cpu().double().mT) <= 1e-5


def test_gram_fp32_inf_and_nan_stay_in_their_rows():
    x = torch.randn(128, 128, device="cuda").abs()
    x[5, 7] = float("inf")
    x[9, 3] = float("nan")
    y = gram(x[None])[0].cpu()
    rows = torch.arange(128)
    assert y[9].isnan().all() and y[:, 9].isnan().all()
    assert (y[5][rows != 9] == float("inf")).all()
    assert y[rows[(rows != 5) & (rows != 9)]][:, rows[(rows != 5) & (rows != 9)]].isfinite().all()


def test_fp32_batch_equals_members():
    X = torch.randn(70, 300, 520, generator=torch.Generator().manual_seed(1)).cuda()
    U = ns_loop(X, 5)
    for i in (0, 33, 69):
        assert torch.equal(U[i], ns_loop(X[i:i + 1], 5)[0])
