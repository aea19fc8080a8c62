"""Barnes-Hut walk of dipoles and quadrupoles, and of charges at a high order, on
both sides of the set sizes where the waves a group change (eight to 32768
particles, four to 393216, then one), against the oracle (1e-12: every opening
decision is the reference's)."""
import numpy as np
import pytest
import torch

from oracle import oracle as O
from tests import util

pytestmark = pytest.mark.gpu


def _dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


@pytest.mark.parametrize("so,order,n", [(1, 2, 64 * 512), (1, 2, 64 * 512 + 1), (1, 8, 40000), (2, 3, 64 * 512 + 1),
                                        (2, 8, 40000), (0, 12, 40000), (1, 2, 64 * 6144 + 1), (2, 3, 64 * 6144 + 1),
                                        (0, 8, 64 * 6144 + 1)])
def test_walk_matches_oracle(gpu, so, order, n):
    from fmmgen_amd import build_tree
    outsz = 3 if so == 1 else 4
    print(f"bh so={so} order={order} n={n}", flush=True)
    pos = util.blobs(n, 51)
    S = np.random.default_rng(52).uniform(-1, 1, (n, {0: 1, 1: 3, 2: 6}[so]))
    want = O.OracleTree(pos, S, 32, order, 0.6, source_order=so, outputsize=outsz).compute_field_bh()
    t = build_tree(_dev(pos), _dev(S), n, 32, order, 0.6, source_order=so, potential=so != 1)
    F = torch.full((n, outsz), float("nan"), dtype=torch.float64, device="cuda")
    t.compute_field_bh(F)
    assert util.rel_norm(F.cpu().numpy(), want) < 1e-12
