"""Prefill attention in 64-row tiles on bf16 MFMA (csrc/attention.hip,
attn_rows_kernel), which automatic takes for grids of a tile per CU and more:
many heads here, so that short contexts reach it.

Tolerance: both products are exact splits summed in fp32, so a score is off by
a few roundings of its sum of |q k| (head_size / 16 + 8 at most, times 2^-24)
and an output by that times |v| plus its own sum's, as test_gpu_attention.py's
5e-5 covers for values in [-1, 1]; the bound here is a tenth of it."""
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


# Head sizes that fill their 32-dim chunks and 80, 112 that do not; rows at
# the least the kernel takes, around a 16-row wave, a tile and two; contexts
# around 32-position blocks, the end of the cache exactly at one and past it.
CASES = [(512, 512, 64), (512, 64, 80), (640, 640, 96), (256, 32, 112), (384, 32, 112), (256, 256, 128)]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(map(str, c)))
@pytest.mark.parametrize("rows,pos", [(32, 0), (33, 1), (47, 17), (64, 0), (64, 33), (65, 30), (130, 7)])
def test_rows_match_double_reference(case, rows, pos):
    heads, kv_heads, hs = case
    T = pos + rows
    q, kc, vc = draw(heads, kv_heads, hs, T, rows, 8100)
    got = run(heads, kv_heads, hs, T, rows, pos, q, kc, vc)
    want = orc.attention(heads, kv_heads, hs, rows, pos, q, kc, vc)
    assert np.abs(got - want).max() <= TOL


def test_small_and_non_finite_values():
    heads, hs, rows, pos = 256, 128, 70, 20
    T = pos + rows + 5
    q, kc, vc = draw(heads, heads, hs, T, rows, 8200)
    # Values whose last terms a bf16 cannot hold: relative precision stays.
    tiny = (vc * np.float32(2.0 ** -115)).astype(np.float32)
    got = run(heads, heads, hs, T, rows, pos, q, kc, tiny)
    want = orc.attention(heads, heads, hs, rows, pos, q, kc, tiny)
    assert np.abs(got - want).max() <= TOL * 2.0 ** -115
    # An infinite value reaches the queries at and after it; positions past
    # the call's rows (uninitialised cache) reach none.
    vc[60, :hs] = np.inf
    kc[T - 5:], vc[T - 5:] = np.nan, np.nan
    got = run(heads, heads, hs, T, rows, pos, q, kc, vc)
    want = orc.attention(heads, heads, hs, rows, pos, q, kc, vc)
    first = 60 - pos  # the first row that sees position 60
    assert np.isinf(got[first:, :hs]).all()
    clean = np.ones_like(got, bool)
    clean[first // 16 * 16:, :hs] = False  # rows of the same 16 may see 0 * inf
    assert np.abs(got[clean] - want[clean]).max() <= TOL


@pytest.mark.parametrize("exponent", [-126, -118, 118, 126])
def test_small_queries_on_large_keys(exponent):
    # Bits that a query's (key's) last term cannot hold below 2^-109, times
    # keys (queries) large enough for scores of order one.
    heads, hs, rows, pos = 256, 128, 70, 20
    T = pos + rows
    q, kc, vc = draw(heads, heads, hs, T, rows, 8500)
    q, kc = q / 2 * np.float32(2.0 ** exponent), kc / 2 * np.float32(2.0 ** -exponent)
    got = run(heads, heads, hs, T, rows, pos, q, kc, vc)
    want = orc.attention(heads, heads, hs, rows, pos, q, kc, vc)
    assert np.abs(got - want).max() <= TOL


@pytest.mark.parametrize("score", [-70.0, -82.0, -86.5, -90.0])
@pytest.mark.parametrize("at", [0, 40])
def test_small_weights_on_large_values(score, at):
    # One position far below the others' scores, its values so large that it
    # is most of every output after it. Its score is off by a few roundings of
    # its size (90 * 2^-24 = 5e-6 each), and so, relatively, is its weight.
    heads, hs, rows, pos = 256, 128, 70, 20
    T = pos + rows
    q, kc, vc = draw(heads, heads, hs, T, rows, 8600)
    q[:], kc[:] = 0.0, 0.0
    q[:, 0:heads * hs:hs] = 16.0
    kc[at, ::hs] = score * np.sqrt(np.float32(hs)) / 16.0
    vc[at] = np.float32(2.0 ** 127) * vc[at]
    got = run(heads, heads, hs, T, rows, pos, q, kc, vc)
    want = orc.attention(heads, heads, hs, rows, pos, q, kc, vc)
    assert (np.abs(got - want) <= 4e-5 * np.abs(want) + TOL).all()
