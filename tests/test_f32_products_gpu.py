"""The fp32 products' 64-row tiles: gram_ of whole tiles (M a multiple of 128, K of 64) at its
smallest and at ragged K-tile counts, the shapes just off it (which take the masked kernel), and
a batch against its members alone."""

import pytest
import torch

from helpers import rel_fro
from muonium_amd.kernels.gram import gram, gram_
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


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("B, M, K", [
    (1, 1, 8), (2, 7, 16), (1, 63, 72), (3, 64, 64), (2, 65, 128), (1, 130, 1336), (4, 100, 40),
    (1, 1000, 8), (40, 200, 136), (2, 1001, 264), (3, 17, 12), (3, 130, 70), (2, 33, 7)])
def test_gram_of_any_extents(B, M, K, dtype):
    """Tiles with partial rows, columns and K (whole 16-byte chunks per row, and rows that are not:
    the element-load kernel), the output between canaries. bf16: one rounding of the fp32 sum."""
    x = torch.randn(B, M, K, generator=torch.Generator().manual_seed(M * K)).to(dtype).cuda()
    n = B * M * M
    store = torch.full((n + 128,), 7.0, dtype=dtype, device="cuda")
    y = store[64:64 + n].view(B, M, M)
    gram_(x, y)
    assert (store[:64] == 7).all() and (store[64 + n:] == 7).all()
    assert torch.equal(y, y.mT)
    xd = x.double()
    exact, mag = xd @ xd.mT, xd.abs() @ xd.abs().mT
    ulp = 2.0 ** -8 if dtype == torch.bfloat16 else 0.0
    assert ((y.double() - exact).abs() <= ulp * exact.abs() + K * 2.0 ** -23 * mag).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_gram_reads_nothing_past_its_rows(dtype):
    """NaN right before and after the input, and in the rows' neighbours, stay out of the sums."""
    B, M, K = 2, 70, 104
    store = torch.full((B * M * K + 512,), float("nan"), dtype=dtype, device="cuda")
    x = store[256:256 + B * M * K].view(B, M, K)
    x.copy_(torch.randn(B, M, K, device="cuda"))
    x[0, 3] = float("nan")
    y = gram(x)
    keep = torch.arange(M, device="cuda") != 3
    assert y[1].isfinite().all() and y[0][keep][:, keep].isfinite().all()
    assert y[0, 3].isnan().all()
