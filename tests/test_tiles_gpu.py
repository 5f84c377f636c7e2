"""The products' tile sizes (256, 128 and 64 rows, chosen by the launch's size) at their edges.

Every tile size sums an element's products in the same order, so a matrix gives the same bits
alone (64-row tiles) as in a batch that fills the device (256-row tiles, packed ones where the last
128 rows are padding); the apply fused into the small tiles' last product gives the post-pass's
parameters bit for bit, for every parameter type, wide and tall, with partial tiles; and the
update stays as close to the 64-bit iteration as the oracle's."""

import pytest
import torch

from helpers import rel_fro
from muonium_amd.orthogonalize import zeropower
from oracle import muon_ref
from test_apply_gpu import _case, _run

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("shape, counts", [
    ((65, 300), (1, 40, 900)), ((128, 128), (1, 300, 1500)), ((129, 520), (1, 30, 700)),
    ((331, 1533), (1, 12, 300)), ((512, 1024), (1, 24, 300)), ((700, 900), (1, 16, 120)),
    ((768, 768), (1, 20, 150)), ((1000, 1100), (1, 12, 80)), ((1408, 2048), (1, 4, 40)),
    ((1100, 700), (1, 12, 100))])
def test_a_matrix_has_the_same_bits_in_any_batch(shape, counts):
    gen = torch.Generator(device=DEV).manual_seed(sum(shape))
    X = torch.randn(counts[-1], *shape, generator=gen, device=DEV).bfloat16()
    ref = None
    for count in counts:
        U = zeropower(X[:count], strategy="polar_express")
        if ref is None:
            ref = U[0].clone()
        assert torch.equal(U[0], ref), count
        if count > 1:
            i = count - 1
            assert torch.equal(U[i], zeropower(X[i:i + 1], strategy="polar_express")[0]), count


@pytest.mark.parametrize("shape, count", [
    ((128, 256), 2), ((200, 136), 3), ((72, 1000), 1), ((1000, 72), 2), ((2, 320, 520), 2),
    ((520, 320), 2), ((640, 648), 1), ((768, 2304), 3), ((2304, 776), 2)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("wd, cautious", [(0.1, True), (0.1, False), (0.0, False)])
def test_apply_in_small_tiles_matches_postpass(shape, count, dtype, wd, cautious):
    p, g, b = _case(shape, count, dtype, seed=sum(shape) + count)
    sides = []
    for fused in (True, False):
        ps, gs, bs = ([t.clone().to(DEV) for t in ts] for ts in (p, g, b))
        _run(ps, gs, bs, fused=fused, wd=wd, cautious=cautious)
        sides.append(ps)
    for x, y, p0 in zip(*sides, p):
        assert torch.equal(x, y)
        assert not torch.equal(x.cpu(), p0)


@pytest.mark.parametrize("shape", [(65, 66), (127, 129), (128, 256), (192, 200), (257, 300),
                                   (300, 257), (640, 641), (385, 1000)])
@pytest.mark.parametrize("strategy", ["newton_schulz", "polar_express"])
def test_update_matches_64_bits_at_tile_edges(shape, strategy):
    """No further from the 64-bit iteration than 1.25 times the bf16 oracle, plus one bf16
    rounding (2e-3)."""
    X = torch.randn(shape, generator=torch.Generator().manual_seed(7)).bfloat16()
    coeffs, prescale = muon_ref.strategy_coeffs(strategy, 5)
    ref = muon_ref.polar_iteration_bf16(X.float(), coeffs, prescale=prescale, eps=1e-7)
    exact = muon_ref.polar_iteration(X.double(), coeffs, prescale=prescale, eps=1e-7)
    got = zeropower(X.to(DEV), strategy=strategy).cpu()
    assert rel_fro(got, exact) <= 1.25 * rel_fro(ref, exact) + 2e-3


@pytest.mark.parametrize("m, n, count", [(2048, 2048, 8), (2048, 2304, 15), (1536, 4352, 13),
                                         (4000, 4096, 2)])
def test_gram_tail_in_small_tiles_has_the_same_bits(m, n, count):
    """Launches of a little more than whole rounds of 256-row tiles (288, 540, 273 and 272 tiles on
    256 compute units): the tiles left over are cut into small ones; each matrix as alone."""
    gen = torch.Generator(device=DEV).manual_seed(m + n)
    X = torch.randn(count, m, n, generator=gen, device=DEV).bfloat16()
    U = zeropower(X, strategy="newton_schulz", steps=2)
    for i in (0, count // 2, count - 1):
        assert torch.equal(U[i], zeropower(X[i:i + 1], strategy="newton_schulz", steps=2)[0]), i
