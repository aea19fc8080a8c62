"""Operator batches: the charge P2M at every source order, batches longer than
one launch's blocks, and outputs that a kernel may add into directly or not
(wider rows, strided, sharing memory with the inputs), against the same calls
item by item or on separate tensors."""
import math

import numpy as np
import pytest
import torch

from fmmgen_amd.codegen.layout import Lsize, Msize

pytestmark = pytest.mark.gpu


def _rand(*shape, seed=0):
    return torch.from_numpy(np.random.default_rng(seed).uniform(-1, 1, shape)).cuda()


def _lib(so, pot, field):
    from fmmgen_amd.operators import Library
    return Library(so, pot, field)


@pytest.mark.parametrize("so,pot,field,order", [(0, True, True, 1), (0, True, True, 12), (1, False, True, 2),
                                                (1, False, True, 8), (2, True, True, 3), (2, True, True, 8)])
def test_charge_p2m(gpu, so, pot, field, order):
    d, q = _rand(65, 3), _rand(65, 1, seed=1)
    out = torch.zeros(65, Msize(order, so), dtype=torch.float64, device="cuda")
    _lib(so, pot, field).P2M(*(d[:, k] for k in range(3)), q, out, order)
    x, y, z = (d[:, k].cpu().numpy() for k in range(3))
    want = [q[:, 0].cpu().numpy() * (-x) ** (g - a) / math.factorial(g - a) * (-y) ** (a - b) / math.factorial(a - b) *
            (-z) ** b / math.factorial(b)
            for g in range(so, order + 1) for a in range(g + 1) for b in range(a + 1)]
    # each value is a product of at most 3 * order + 3 roundings
    np.testing.assert_allclose(out.cpu().numpy(), np.stack(want, 1), rtol=64 * 2.0 ** -52, atol=0)


def test_batch_longer_than_the_launch(gpu):
    n = (1 << 16) + 77
    d, M = 2.0 + _rand(n, 3), _rand(n, Msize(2, 0), seed=1)
    x, y, z = (d[:, k].contiguous() for k in range(3))
    L = torch.zeros(n, Lsize(2, 0), dtype=torch.float64, device="cuda")
    _lib(0, True, True).M2L(x, y, z, M, L, 2)
    for s in (slice(0, 77), slice(n - 77, n)):
        part = torch.zeros(77, Lsize(2, 0), dtype=torch.float64, device="cuda")
        _lib(0, True, True).M2L(x[s], y[s], z[s], M[s], part, 2)
        assert torch.equal(part, L[s])


@pytest.mark.parametrize("op", ["M2M", "M2L", "L2P"])
@pytest.mark.parametrize("order", [3, 10])
def test_outputs_in_every_form(gpu, op, order):
    n, lib = 33, _lib(0, True, True)
    ms = Msize(order, 0)
    nout = 4 if op == "L2P" else ms
    d, a, start = 2.0 + _rand(n, 3), _rand(n, ms, seed=1), _rand(n, nout, seed=2)
    xyz = [d[:, k] for k in range(3)]
    want = torch.zeros(n, nout, dtype=torch.float64, device="cuda")
    getattr(lib, op)(*xyz, a, want, order)
    want += start
    same = start.clone()
    version = same._version
    getattr(lib, op)(*xyz, a, same, order)
    assert torch.equal(same, want) and same._version > version
    wide = torch.cat([start, start], 1)
    getattr(lib, op)(*xyz, a, wide, order)
    assert torch.equal(wide[:, :nout], want) and torch.equal(wide[:, nout:], start)
    rows = torch.zeros(n, 2 * nout, dtype=torch.float64, device="cuda")
    part = rows[:, :nout]
    part.copy_(start)
    getattr(lib, op)(*xyz, a, part, order)
    assert torch.equal(part, want) and not rows[:, nout:].any()
    if nout == ms:  # the output is the next item's input
        mem = torch.cat([a[:1], a])
        keep = mem[1:].clone()
        getattr(lib, op)(*xyz, mem[:-1], mem[1:], order)
        ref = torch.zeros_like(keep)
        getattr(lib, op)(*xyz, torch.cat([a[:1], a])[:-1], ref, order)
        assert torch.equal(mem[1:], keep + ref)
