"""Very wide short iterates (at most 64 rows, at least 65536 columns): the iteration on the
Gram matrix, at the edges of its range (one column below and above the line, ragged widths, one
to 64 rows, tall inputs, 2 to 5 steps, where the result overwrites the iterate or not)."""

import pytest
import torch

from helpers import rel_fro
from muonium_amd import _lib, _ops
from muonium_amd.orthogonalize import foreach_zeropower, zeropower
from muonium_amd.orthogonalize.newton_schulz import ns_loop
from muonium_amd.orthogonalize.polar_express import pe_loop
from oracle import muon_ref

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _x(shape, seed=0):
    return torch.randn(shape, generator=torch.Generator().manual_seed(seed)).bfloat16()


def _check(got, X, strategy, steps):
    """Within the bf16 bar (1e-2) of the oracle's iteration, and no further from the 64-bit
    iteration than 1.25 times the oracle is, plus one bf16 rounding (2e-3)."""
    coeffs, prescale = muon_ref.strategy_coeffs(strategy, steps)
    ref = muon_ref.polar_iteration_bf16(X.float(), coeffs, prescale=prescale, eps=1e-7)
    exact = muon_ref.polar_iteration(X.double(), coeffs, prescale=prescale, eps=1e-7)
    assert rel_fro(got, exact) <= 1.25 * rel_fro(ref, exact) + 2e-3
    assert rel_fro(got, ref) <= 1e-2


@pytest.mark.parametrize("strategy", ["polar_express", "newton_schulz"])
@pytest.mark.parametrize("shape, steps", [
    ((64, 65535), 5), ((64, 65536), 5), ((64, 65537), 2), ((33, 70001), 4), ((70003, 17), 3),
    ((1, 65536), 5), ((2, 63, 66000), 2)])
def test_matches_oracle_and_64_bits(shape, steps, strategy):
    X = _x(shape)
    loop = pe_loop if strategy == "polar_express" else ns_loop
    _check(loop(X.to(DEV), steps, eps=1e-7).cpu(), X, strategy, steps)


def test_a_batch_equals_its_members():
    Xs = [_x((40, 65800), s).to(DEV) for s in range(3)]
    both = foreach_zeropower(Xs, strategy="polar_express")
    for x, u in zip(Xs, both):
        assert torch.equal(u, zeropower(x, strategy="polar_express"))


def test_rank_deficient_zero_and_nan_matrices():
    """Rank 4 of 48 rows (the Gram matrix is singular up to rounding): finite, and as close to 64
    bits as the oracle; a zero matrix stays zero; a NaN makes its own matrix NaN only."""
    g = torch.Generator().manual_seed(3)
    low = (torch.randn(48, 4, generator=g) @ torch.randn(4, 65536, generator=g)).bfloat16()
    nan = _x((48, 65536), 5)
    nan[7, 1234] = float("nan")
    out = torch.stack(foreach_zeropower([t.to(DEV) for t in (low, torch.zeros_like(low), nan)],
                                        strategy="polar_express")).cpu()
    coeffs, prescale = muon_ref.strategy_coeffs("polar_express", 5)
    ref = muon_ref.polar_iteration_bf16(low.float(), coeffs, prescale=prescale, eps=1e-7)
    exact = muon_ref.polar_iteration(low.double(), coeffs, prescale=prescale, eps=1e-7)
    assert rel_fro(out[0], exact) <= 1.25 * rel_fro(ref, exact) + 2e-3
    assert not out[1].any()
    assert out[2].isnan().all()


NS = (3.4445, -4.7750, 2.0315)


def _launches(X, coeffs):
    """The update and the B X launches of its iteration: one on the Gram matrix, one per step where X is
    read each time."""
    x = X.to(DEV)
    _lib.timing_enable(True)
    u = _ops.orthogonalize([x], coeffs, prescale=1.0, eps=1e-7, iter_dtype=torch.bfloat16,
                           out_dtype=torch.bfloat16)[0]
    launches = _lib.timing_read()["gemm_bx"][1]
    _lib.timing_enable(False)
    ref = muon_ref.polar_iteration_bf16(X.float(), coeffs, prescale=1.0, eps=1e-7)
    assert u.isfinite().all()
    assert rel_fro(u.cpu(), ref) <= 1e-2
    return launches


def _first(a, singular=0.25):
    """Coefficients whose first step takes 16 equal singular values (of a unit-norm matrix) to 1."""
    return [(a, (1.0 - a * singular) / singular ** 3, 0.0)] + [NS] * 4


@pytest.mark.parametrize("shape, coeffs, gram", [
    # up to five steps
    ((16, 65536), [NS] * 5, True), ((16, 65536), [NS] * 6, False), ((16, 65536), [NS], False),
    # the squares of all leading coefficients but the last multiply to 2^18 at a = 12.528
    ((16, 65536), _first(12.4), True), ((16, 65536), _first(12.6), False),
    ((16, 65535), [NS] * 5, False), ((65, 65536), [NS] * 2, False)])
def test_many_steps_and_large_coefficients_take_the_streaming_iteration(shape, coeffs, gram):
    """Six steps, and coefficients whose squares multiply past 2^18, stay on the iteration that
    reads X each time (an error of the Gram matrix would grow too far), as do narrower and taller ones."""
    assert _launches(_x(shape), coeffs) == (1 if gram else len(coeffs))
