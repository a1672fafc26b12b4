"""Attention of a few rows of heads that share kv heads (csrc/attention.hip,
attn_group_kernel), which automatic takes by rows times heads of a kv head:
16-query tiles partly, just and more than full, contexts around its 16-position
blocks and 64-position chunks.

Tolerance: an fp32 score is off by a few roundings of its sum of |q k| and an
output by that times |v| plus its own sum's, as test_gpu_attention.py's 5e-5
covers for values in [-1, 1]; the sums here are trees of four- and
eight-product chains, so the bound is a tenth of it."""
import numpy as np
import pytest
import torch

import oracle
from tests import engine, inputs

em = engine.load()
orc = oracle.oracle()
pytestmark = pytest.mark.gpu
TOL = 5e-6


def run(heads, kv_heads, hs, T, rows, pos, q, kc, vc):
    shape = em.attention_shape(heads, kv_heads, hs, T)
    args = [torch.from_numpy(a).cuda() for a in (q, kc, vc)]
    pos_dev = torch.full((1,), pos, dtype=torch.int32, device="cuda")
    got = em.attention(shape, rows, pos_dev, *args)
    again = em.attention(shape, rows, pos_dev, *args)
    assert torch.equal(got.view(torch.int32), again.view(torch.int32))
    return got.cpu().numpy()


def draw(heads, kv_heads, hs, T, rows, seed):
    dim, kv = heads * hs, kv_heads * hs
    return (inputs.uniform((rows, dim + 2 * kv), -2.0, 2.0, seed),
            inputs.uniform((T, kv), -2.0, 2.0, seed + 1), inputs.uniform((T, kv), -1.0, 1.0, seed + 2))


# heads, kv heads, head size, rows, cache: columns 2, 3, 6, 15, 16, 17, 35, 96.
CASES = [(2, 1, 16, 1, 900), (6, 2, 96, 1, 900), (12, 4, 112, 2, 900), (15, 3, 48, 3, 900),
         (32, 8, 128, 4, 900), (32, 8, 128, 4, 1100), (17, 1, 80, 1, 900), (14, 2, 64, 5, 900), (16, 2, 32, 12, 500)]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(map(str, c)))
def test_rows_match_double_reference(case):
    heads, kv_heads, hs, rows, T = case
    q, kc, vc = draw(heads, kv_heads, hs, T, rows, 8300)
    for ctx in (rows, 15, 16, 17, 63, 64, 65, 66, 129, 449, T):
        if ctx < rows:
            continue
        got = run(heads, kv_heads, hs, T, rows, ctx - rows, q, kc, vc)
        want = orc.attention(heads, kv_heads, hs, rows, ctx - rows, q, kc, vc)
        assert np.abs(got - want).max() <= TOL, ctx


def test_values_a_row_does_not_see():
    """An infinite value reaches the rows at and after its position alone."""
    heads, kv_heads, hs, rows, T, pos = 8, 2, 64, 4, 200, 97
    q, kc, vc = draw(heads, kv_heads, hs, T, rows, 8400)
    want = orc.attention(heads, kv_heads, hs, rows, pos, q, kc, vc)
    vc[pos + 2, :hs] = np.inf
    kc[pos + rows:], vc[pos + rows:] = np.nan, np.nan
    got = run(heads, kv_heads, hs, T, rows, pos, q, kc, vc)
    dim = heads // kv_heads * hs  # the first kv head's
    assert np.isinf(got[2:, :dim]).all()
    assert np.abs(got[:2] - want[:2]).max() <= TOL
    assert np.abs(got[2:, dim:] - want[2:, dim:]).max() <= TOL


@pytest.mark.parametrize("hs,at", [(64, 0), (64, 16), (64, 64), (128, 0), (128, 32), (128, 128)])
def test_infinite_keys(hs, at):
    """A key with an infinite component, at the first position of a wave's
    part of a chunk: queries that score +inf there are NaN, those that score
    -inf give it no weight, and both are columns of one tile."""
    heads, kv_heads, rows, T, pos = 16, 2, 2, 1100, 298
    q, kc, vc = draw(heads, kv_heads, hs, T, rows, 8700)
    kc[at, 0] = np.inf
    got = run(heads, kv_heads, hs, T, rows, pos, q, kc, vc)
    with np.errstate(invalid="ignore"):
        want = orc.attention(heads, kv_heads, hs, rows, pos, q, kc, vc)
    nan = np.isnan(want)
    assert nan.any() and not nan[:, :heads // kv_heads * hs].all()
    assert np.array_equal(np.isnan(got), nan)
    assert np.abs(got[~nan] - want[~nan]).max() <= TOL
