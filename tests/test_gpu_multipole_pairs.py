"""Dipole and quadrupole pairs: near field and direct sum against the oracle's
sums, at one particle, around the staged chunks of 128 sources, and with
coincident particles (undefined values there only).  FP64 1e-12, FP32 1e-6, as
for the charges."""
import numpy as np
import pytest
import torch

from oracle import oracle as O
from tests import util

pytestmark = pytest.mark.gpu
P2P = 8


def _dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


@pytest.mark.parametrize("so", [1, 2])
@pytest.mark.parametrize("n,ncrit", [(2, 64), (127, 128), (129, 200), (3000, 64)])
def test_pairs_match_oracle(gpu, so, n, ncrit):
    from fmmgen_amd import build_tree, direct_sum
    pot = so == 2
    pos, S = util.blobs(n, 11), np.random.default_rng(12).normal(size=(n, 3 * so))
    outsz = 3 + pot
    want = O.OracleTree(pos, S, ncrit, so + 1, 0.5, source_order=so, outputsize=outsz).compute_field_fmm(mask=P2P)
    t = build_tree(_dev(pos), _dev(S), n, ncrit, so + 1, 0.5, source_order=so, potential=pot)
    F = torch.empty(n, outsz, dtype=torch.float64, device="cuda")
    print(f"so={so} n={n} ncrit={ncrit}", flush=True)
    for mode, tol in (("plain", 1e-12), ("f32", 1e-6)):
        t.compute_field_fmm(F, mode=mode, phases=P2P)
        assert util.rel_norm(F.cpu().numpy()[:, pot:], want[:, pot:]) <= tol
    whole = O.OracleTree(pos, S, n + 1, so + 1, 0.5, source_order=so, outputsize=outsz).compute_field_fmm(mask=P2P)
    tg = torch.arange(n, device="cuda")
    D = direct_sum(_dev(pos), _dev(S), tg, source_order=so, outsz=outsz).cpu().numpy()
    assert util.rel_norm(D, whole) <= 1e-12


@pytest.mark.parametrize("so", [1, 2])
def test_coincident_particles(gpu, so):
    from fmmgen_amd import build_tree, direct_sum
    pot, n = so == 2, 1000
    pos, S = util.blobs(n, 13), np.random.default_rng(14).normal(size=(n, 3 * so))
    pos = np.vstack([pos, pos[:1]])
    S = np.vstack([S, S[:1]])
    t = build_tree(_dev(pos), _dev(S), n + 1, 64, so + 1, 0.5, source_order=so, potential=pot)
    F = torch.empty(n + 1, 3 + pot, dtype=torch.float64, device="cuda")
    out = []
    for mode in ("plain", "f32"):
        t.compute_field_fmm(F, mode=mode, phases=P2P)
        out.append(F.cpu().numpy())
    t.compute_field_bh(F)
    out.append(F.cpu().numpy())
    out.append(direct_sum(_dev(pos), _dev(S), torch.arange(n + 1, device="cuda"), source_order=so,
                          outsz=3 + pot).cpu().numpy())
    for F in out:
        assert np.isnan(F[[0, n]]).all() and np.isfinite(F[1:n]).all()
