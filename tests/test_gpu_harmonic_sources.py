"""The harmonic-layout M2L of dipoles and quadrupoles (multipoles from degree 1
and 2, local expansions to degree p - 1 and p - 2) against the oracle at the
lowest and highest compiled orders, in FP64 and in the mixed modes, and the
automatic choice of the form on both sides of its size limit."""
import numpy as np
import pytest
import torch

from oracle import oracle as O
from tests import util

pytestmark = pytest.mark.gpu


def _set(n, so, seed):
    rng = np.random.default_rng(seed)
    return util.blobs(n, seed), rng.normal(size=(n, {0: 1, 1: 3, 2: 6}[so]))


def _dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


@pytest.mark.parametrize("so,order", [(1, 2), (1, 3), (1, 8), (2, 3), (2, 4), (2, 8)])
def test_harmonic_form_matches_oracle(gpu, so, order):
    from fmmgen_amd import build_tree
    n, pot = 6000, so == 2
    pos, S = _set(n, so, 31 + order)
    Fo = O.OracleTree(pos, S, 32, order, 0.5, source_order=so, outputsize=4 if pot else 3).compute_field_fmm()
    t = build_tree(_dev(pos), _dev(S), n, 32, order, 0.5, source_order=so, potential=pot)
    t.set_m2l_form("harmonic")
    F = torch.empty(n, 4 if pot else 3, dtype=torch.float64, device="cuda")
    # the same sums as the generated operator: 1e-12 in FP64 as for the full
    # form, 1e-6 (field) in FP32 and BF16x3
    for mode, tol in (("plain", 1e-12), ("f32", 1e-6), ("bf16x3", 1e-6)):
        print(f"so={so} order={order} {mode}", flush=True)
        t.compute_field_fmm(F, mode=mode)
        f0 = 1 if pot and mode != "plain" else 0
        assert util.rel_norm(F.cpu().numpy()[:, f0:], Fo[:, f0:]) < tol, mode


@pytest.mark.parametrize("n,order", [(700, 4), (700, 6), (30000, 4)])
@pytest.mark.parametrize("so", [0, 1])
def test_automatic_form_agrees_with_both(gpu, so, n, order):
    """Few groups and many, below and at the order limit; repeated after the
    other form has run, whose expansions it must not read."""
    from fmmgen_amd import build_tree
    pos, S = _set(n, so, 41)
    t = build_tree(_dev(pos), _dev(S), n, 32, order, 0.5, source_order=so, potential=so == 0)
    F = torch.empty(n, 4 if so == 0 else 3, dtype=torch.float64, device="cuda")
    out = []
    for form in ("auto", "full", "harmonic", "auto"):
        t.set_m2l_form(form)
        out.append(t.compute_field_fmm(F, mode="plain").cpu().numpy().copy())
    for o in out[1:]:
        assert util.rel_norm(o, out[0]) < 1e-12
