"""Near field: leaves cut into many work items and into one, at the sizes where
the cut changes, and coincident particles (infinite potential, undefined field
there, every other particle unaffected), against the oracle's P2P."""
import numpy as np
import pytest
import torch

from oracle import oracle as O
from tests import util

pytestmark = pytest.mark.gpu
P2P = 8


def _dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


@pytest.mark.parametrize("n,ncrit", [(1, 64), (63, 64), (127, 128), (129, 200), (2000, 64), (2000, 8), (9000, 1000),
                                     (60000, 64)])
def test_items_match_oracle(gpu, n, ncrit):
    from fmmgen_amd import build_tree
    pos, q = util.blobs(n, 5), np.random.default_rng(6).uniform(-1, 1, (n, 1))
    want = O.OracleTree(pos, q, ncrit, 3, 0.5).compute_field_fmm(mask=P2P) if n > 1 else np.zeros((1, 4))
    t = build_tree(_dev(pos), _dev(q), n, ncrit, 3, 0.5)
    inf = t.info()
    assert inf["p2p_items"] >= inf["nleaves"]
    F = torch.empty(n, 4, dtype=torch.float64, device="cuda")
    print(f"n={n} ncrit={ncrit} items {inf['p2p_items']} leaves {inf['nleaves']}", flush=True)
    for mode, tol in (("plain", 1e-12), ("f32", 1e-6)):
        t.compute_field_fmm(F, mode=mode, phases=P2P)
        assert util.rel_norm(F.cpu().numpy()[:, 1:], want[:, 1:]) <= tol


def test_coincident_particles(gpu):
    from fmmgen_amd import build_tree
    n = 3000
    pos, q = util.blobs(n, 7), np.random.default_rng(8).uniform(0.5, 1, (n, 1))
    clean = build_tree(_dev(pos), _dev(q), n, 64, 3, 0.5)
    a = torch.empty(n, 4, dtype=torch.float64, device="cuda")
    clean.compute_field_fmm(a, mode="plain", phases=P2P)
    pos2 = np.vstack([pos, pos[:1]])
    q2 = np.vstack([q, [[0.0]]])  # a second particle on the first, without charge: 0 / 0 at the first only
    t = build_tree(_dev(pos2), _dev(q2), n + 1, 64, 3, 0.5)
    F = torch.empty(n + 1, 4, dtype=torch.float64, device="cuda")
    t.compute_field_fmm(F, mode="plain", phases=P2P)
    F = F.cpu().numpy()
    assert np.isposinf(F[n, 0]) and np.isnan(F[n, 1:]).all()  # the charge at zero distance
    assert np.isnan(F[0]).all()                              # the zero charge at zero distance
    assert np.isfinite(F[1:n]).all()
