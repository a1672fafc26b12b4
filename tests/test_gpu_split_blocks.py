"""int8 products at row counts where the exact split takes three 16-row blocks
a workgroup, and around them: whole and ragged last blocks, with k slices and
without, norm, accumulation; against 64-bit products.

Bound per element, times the sum of |a w|: two roundings of 2^-24 for each of
three terms per 32 rows of k at the size of the sums so far, in four waves of
a quarter of the chunks each, and a few more for the waves, slices, scale and
prior C: (3 k / 64 + 24) 2^-24 (a sum is rarely at its largest throughout).
The norm's rounding of each activation adds 4 * 2^-24."""
import numpy as np
import pytest
import torch

import oracle
from tests import engine, inputs

em = engine.load()
orc = oracle.oracle()
pytestmark = pytest.mark.gpu

# Three blocks: (40 .. 48, 4096, 12288) in five slices, (96, 97 rows of 6144
# columns) in two or three, (385 .. 400, 1024, 5632) in one; the rest beside.
SHAPES = [(33, 4096, 12288), (40, 4096, 12288), (48, 4096, 12288), (96, 4096, 6144),
          (97, 4096, 6144), (200, 4096, 6144), (385, 1024, 5632), (400, 1024, 5632),
          (400, 1000, 5632)]


@pytest.mark.parametrize("norm", [False, True], ids=["plain", "norm"])
@pytest.mark.parametrize("shape", SHAPES, ids=str)
def test_blocks(shape, norm):
    m, k, n = shape
    A = inputs.normal((m, k), 1.0, 91)
    w = inputs.uniform((k,), 0.5, 1.5, 92)
    C0 = inputs.normal((m, n), 1.0, 93)
    q, s = orc.quantize_q8(inputs.normal((k, n), 0.02, 94))
    dA, dq, ds, dw = (torch.from_numpy(x).cuda() for x in (A, q, s, w))
    kw = dict(scale=ds, rms_weight=dw if norm else None)
    C = em.matmul(dA, dq, **kw)
    assert torch.equal(C, em.matmul(dA, dq, **kw))
    added = torch.from_numpy(C0.copy()).cuda()
    em.matmul(dA, dq, added, accumulate=True, **kw)
    a = dA.double()
    if norm:
        a = a / torch.sqrt((a * a).mean(1, keepdim=True) + 1e-5) * dw.double()
    b = dq.double() * ds.double()
    want, scale = a @ b, a.abs() @ b.abs()
    bound = (3 * k / 64 + (28 if norm else 24)) * 2.0 ** -24
    assert ((C.double() - want).abs() <= bound * scale).all()
    prior = torch.from_numpy(C0).cuda().double()
    assert ((added.double() - want - prior).abs() <= bound * (scale + prior.abs())).all()
