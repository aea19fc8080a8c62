"""Plain FP64 evaluations of sets whose leaves are cut into several near-field
items, and below order 6 whose M2L tiles are cut into several chunks, give the
same bits every time and agree with the oracle's sums."""
import numpy as np
import pytest
import torch

from oracle import oracle as O
from tests import util

pytestmark = pytest.mark.gpu
P2P = 8


def _dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def _tree(n, ncrit, so, order=3):
    from fmmgen_amd import build_tree
    pot = so != 1
    pos = util.blobs(n, 21)
    S = np.random.default_rng(22).normal(size=(n, {0: 1, 1: 3, 2: 6}[so]))
    return pos, S, build_tree(_dev(pos), _dev(S), n, ncrit, order, 0.5, source_order=so, potential=pot)


def _repeat(t, n, outsz, times, **kw):
    """The first result, after showing that the later ones equal it (with other work between them)."""
    first = None
    for _ in range(times):
        F = torch.full((n, outsz), float("nan"), dtype=torch.float64, device="cuda")
        t.compute_field_fmm(F, mode="plain", **kw)
        if first is None:
            first = F.clone()
        assert torch.equal(F, first)
        t.compute_field_fmm(F, mode="f32")
    return first.cpu().numpy()


@pytest.mark.parametrize("n,ncrit,so", [(129, 200, 0), (2000, 64, 0), (2000, 8, 0), (9000, 1000, 0), (60000, 64, 0),
                                        (9000, 64, 1), (9000, 64, 2)])
def test_near_field_repeats(gpu, n, ncrit, so):
    pos, S, t = _tree(n, ncrit, so)
    outsz = 3 if so == 1 else 4
    print(f"near field so={so} n={n} ncrit={ncrit}", flush=True)
    got = _repeat(t, n, outsz, 8, phases=P2P)
    want = O.OracleTree(pos, S, ncrit, 3, 0.5, source_order=so, outputsize=outsz).compute_field_fmm(mask=P2P)
    assert util.rel_norm(got, want) <= 1e-12


@pytest.mark.parametrize("n,ncrit,so,order,form", [
    (2000, 64, 0, 4, "auto"), (2000, 8, 0, 1, "auto"), (2000, 64, 0, 5, "harmonic"), (700, 64, 0, 5, "full"),
    (30000, 32, 0, 3, "auto"), (30000, 32, 0, 5, "full"), (9000, 64, 1, 2, "auto"), (9000, 64, 1, 5, "harmonic"),
    (9000, 64, 2, 3, "auto"), (9000, 64, 2, 5, "harmonic")])
def test_evaluation_repeats(gpu, n, ncrit, so, order, form):
    pos, S, t = _tree(n, ncrit, so, order)
    t.set_m2l_form(form)
    outsz = 3 if so == 1 else 4
    print(f"so={so} n={n} order={order} {form}: {t.info()['m2l_groups']} groups", flush=True)
    got = _repeat(t, n, outsz, 8)
    want = O.OracleTree(pos, S, ncrit, order, 0.5, source_order=so, outputsize=outsz).compute_field_fmm()
    assert util.rel_norm(got, want) <= 1e-12


@pytest.mark.parametrize("n", [2000, 60000])
def test_small_sets_are_cut_finer_in_fp64(gpu, n):
    """The lists that the tests above are about: the FP32 ones stay as they are
    (their sums depend on the cut)."""
    inf = _tree(n, 64, 0)[2].info()
    print(inf, flush=True)
    # an item a leaf, or a segment of 8192 sources beside a dense cluster
    assert inf["nleaves"] <= inf["p2p_items"] < inf["p2p_items_f64"]
    assert inf["m2l_chunks"] < inf["m2l_chunks_f64"]
