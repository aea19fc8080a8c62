"""Barnes-Hut walk against the oracle at the edges of its forms: every source
order and output set, the lowest and highest orders, groups of 64 particles that
are not full, and the set sizes where the waves a group change.  Every opening
decision is the reference's, so the sums agree to FP64 rounding (1e-12)."""
import numpy as np
import pytest
import torch

from oracle import oracle as O
from tests import util

pytestmark = pytest.mark.gpu


def _dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


@pytest.mark.parametrize("so,pot,field,order,n", [
    (0, True, True, 1, 1000), (0, True, True, 12, 3001), (0, True, False, 0, 1000), (0, True, False, 12, 3001),
    (0, False, True, 1, 1000), (0, False, True, 7, 3001), (1, False, True, 2, 1000), (1, False, True, 8, 3001),
    (2, True, True, 3, 1000), (2, True, True, 8, 3001),
    (0, True, True, 3, 64 * 512), (0, True, True, 3, 64 * 512 + 1), (0, True, True, 3, 64 * 6144),
    (0, True, True, 3, 64 * 6144 + 1)])
def test_walk_matches_oracle(gpu, so, pot, field, order, n):
    from fmmgen_amd import build_tree
    outsz = int(pot) + 3 * int(field)
    print(f"bh so={so} outputs={outsz} order={order} n={n}", flush=True)
    pos = util.blobs(n, 31)
    S = np.random.default_rng(32).uniform(-1, 1, (n, {0: 1, 1: 3, 2: 6}[so]))
    want = O.OracleTree(pos, S, 32, order, 0.5, source_order=so, outputsize=outsz).compute_field_bh()
    t = build_tree(_dev(pos), _dev(S), n, 32, order, 0.5, source_order=so, potential=pot, field=field)
    F = torch.full((n, outsz), float("nan"), dtype=torch.float64, device="cuda")
    for _ in range(2):
        t.compute_field_bh(F)
        assert util.rel_norm(F.cpu().numpy(), want) < 1e-12
