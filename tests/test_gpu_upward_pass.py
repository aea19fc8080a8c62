"""FP64 upward and downward passes: leaves of one particle, of a staged batch of 32 and around it,
and levels below and above the number of parents, and orders, where M2M and L2L change
their form, through whole evaluations against the oracle (1e-12)."""
import numpy as np
import pytest
import torch

from oracle import oracle as O
from tests import util

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,ncrit,order,so", [(9, 2, 4, 0), (300, 32, 2, 0), (300, 33, 12, 0), (3000, 200, 5, 0),
                                              (3000, 16, 8, 0), (20000, 8, 9, 0), (20000, 8, 10, 0),
                                              (40000, 8, 3, 0), (40000, 8, 3, 1), (5000, 32, 4, 2)])
def test_evaluation_matches_oracle(gpu, n, ncrit, order, so):
    from fmmgen_amd import build_tree
    pos, S = util.blobs(n, 21), np.random.default_rng(22).normal(size=(n, {0: 1, 1: 3, 2: 6}[so]))
    outsz = 3 if so == 1 else 4
    print(f"n={n} ncrit={ncrit} order={order} so={so}", flush=True)
    want = O.OracleTree(pos, S, ncrit, order, 0.5, source_order=so, outputsize=outsz).compute_field_fmm()
    t = build_tree(torch.from_numpy(pos).cuda(), torch.from_numpy(S).cuda(), n, ncrit, order, 0.5, source_order=so,
                   potential=so != 1)
    F = torch.empty(n, outsz, dtype=torch.float64, device="cuda")
    t.compute_field_fmm(F, mode="plain")
    assert util.rel_norm(F.cpu().numpy(), want) <= 1e-12
