"""Which operand form of the M2L the automatic choice takes on each side of its
limits: FP64 below order 6 repeats bit for bit, so the form that ran is the one
with the same bits; the mixed modes of dipoles and quadrupoles take the harmonic
form above 2^17 groups, checked against the oracle."""
import numpy as np
import pytest
import torch

from oracle import oracle as O
from tests import util

pytestmark = pytest.mark.gpu
P2P = 8


def _dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def _tree(n, ncrit, order, so, seed=61):
    from fmmgen_amd import build_tree
    pos, S = util.blobs(n, seed), np.random.default_rng(seed + 1).normal(size=(n, {0: 1, 1: 3, 2: 6}[so]))
    return pos, S, build_tree(_dev(pos), _dev(S), n, ncrit, order, 0.5, source_order=so, potential=so != 1)


@pytest.mark.parametrize("so", [0, 1, 2])
@pytest.mark.parametrize("n,few", [(700, True), (30000, False)])
def test_fp64_choice_by_groups(gpu, so, n, few):
    _, _, t = _tree(n, 32, 4, so)
    assert (t.info()["m2l_groups"] < 1 << 14) == few
    out = {}
    for form in ("full", "harmonic", "auto"):
        t.set_m2l_form(form)
        F = torch.empty(n, 3 if so == 1 else 4, dtype=torch.float64, device="cuda")
        out[form] = t.compute_field_fmm(F, mode="plain")
    took, other = ("full", "harmonic") if few else ("harmonic", "full")
    assert torch.equal(out["auto"], out[took]) and not torch.equal(out["auto"], out[other])


@pytest.mark.parametrize("so", [1, 2])
@pytest.mark.parametrize("n,many", [(5000, False), (60000, True)])
@pytest.mark.parametrize("mode", ["f32", "bf16x3"])
def test_mixed_choice_by_groups(gpu, so, n, many, mode):
    pos, S, t = _tree(n, 64, 4, so)
    assert (t.info()["m2l_groups"] >= 1 << 17) == many
    pot = so == 2
    want = O.OracleTree(pos, S, 64, 4, 0.5, source_order=so, outputsize=3 + pot).compute_field_fmm()
    F = torch.empty(n, 3 + pot, dtype=torch.float64, device="cuda")
    print(f"so={so} n={n} {mode} {t.info()['m2l_groups']} groups", flush=True)
    t.compute_field_fmm(F, mode=mode)
    assert util.rel_norm(F.cpu().numpy()[:, pot:], want[:, pot:]) < 1e-6


@pytest.mark.parametrize("pot,field,order", [(True, False, 0), (True, False, 1), (True, True, 1), (False, True, 1)])
@pytest.mark.parametrize("n,form", [(700, "harmonic"), (30000, "auto"), (30000, "full")])
def test_lowest_orders(gpu, pot, field, order, n, form):
    """The automatic form is harmonic on large sets at every order, the lowest ones included."""
    from fmmgen_amd import build_tree
    pos, S = util.blobs(n, 71), np.random.default_rng(72).uniform(-1, 1, (n, 1))
    outsz = int(pot) + 3 * int(field)
    t = build_tree(_dev(pos), _dev(S), n, 32, order, 0.5, potential=pot, field=field)
    t.set_m2l_form(form)
    want = O.OracleTree(pos, S, 32, order, 0.5, outputsize=outsz).compute_field_fmm()
    F = torch.empty(n, outsz, dtype=torch.float64, device="cuda")
    print(f"order {order} n={n} {form}", flush=True)
    t.compute_field_fmm(F, mode="plain")
    assert util.rel_norm(F.cpu().numpy(), want) < 1e-12


@pytest.mark.parametrize("mode,so,order,took", [
    ("f32", 1, 3, "harmonic"), ("f32", 1, 8, "harmonic"), ("f32", 2, 3, "harmonic"),
    ("f32", 2, 5, "harmonic"), ("f32", 2, 6, "full"), ("f32", 2, 7, "harmonic"),
    ("bf16x3", 1, 8, "full"), ("bf16x3", 2, 3, "full"), ("bf16x3", 2, 8, "full"), ("f32", 0, 4, "harmonic"),
    ("bf16x3", 0, 4, "harmonic")])
def test_mixed_choice_by_rounding(gpu, mode, so, order, took):
    """Above the size limit, dipoles and quadrupoles take the harmonic form in the
    mixed modes only where it rounds no worse.  The far field of the automatic form
    is nearer to that of the form it takes (the same roundings but for the order of
    some additions) than to that of the other."""
    n = 60000
    _, _, t = _tree(n, 32, order, so)
    assert t.info()["m2l_groups"] >= 1 << 17
    out = {}
    for form in ("full", "harmonic", "auto"):
        t.set_m2l_form(form)
        F = torch.empty(n, 3 if so == 1 else 4, dtype=torch.float64, device="cuda")
        out[form] = t.compute_field_fmm(F, mode=mode, phases=63 & ~P2P)
    d = {f: (out["auto"] - out[f]).norm().item() for f in ("full", "harmonic")}
    print(f"so={so} order={order} {mode} distance to {d}", flush=True)
    assert min(d, key=d.get) == took
