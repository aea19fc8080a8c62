"""FP64 pairs outside the ordinary range of distances: a squared distance that is
subnormal, and one whose inverse cube is, in the near field, the Barnes-Hut
leaves and the direct sum, against the generated operator's formula."""
import numpy as np
import pytest
import torch

from tests import util

pytestmark = pytest.mark.gpu
P2P = 8


def _dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def _evaluations(pos, q, pot, field):
    from fmmgen_amd import build_tree, direct_sum
    n, outsz = len(pos), int(pot) + 3 * int(field)
    t = build_tree(_dev(pos), _dev(q), n, 64, 3, 0.0, potential=pot, field=field)  # theta 0: every pair is a P2P pair
    F = torch.empty(n, outsz, dtype=torch.float64, device="cuda")
    yield "near field", t.compute_field_fmm(F, phases=P2P).cpu().numpy().copy()
    yield "walk", t.compute_field_bh(F).cpu().numpy().copy()
    yield "direct", direct_sum(_dev(pos), _dev(q), torch.arange(n, device="cuda"), outsz=outsz).cpu().numpy()


@pytest.mark.parametrize("pot,field", [(True, True), (True, False)])
def test_subnormal_squared_distance(gpu, pot, field):
    n = 600
    pos, q = util.blobs(n, 3), np.random.default_rng(4).uniform(0.5, 1, (n, 1))
    d = 2.0 ** -518  # d^2 = 2^-1036 is subnormal and exact, 1/d finite
    pos[7], pos[8] = 0.0, (d, 0.0, 0.0)
    for what, F in _evaluations(pos, q, pot, field):
        print(what, F[7], F[8], flush=True)
        # the other particles add less than a rounding of 2^518
        assert np.allclose(F[[7, 8], 0], q[[8, 7], 0] / d, rtol=1e-15, atol=0), what
        if field:  # q r^-3 is infinite, times a zero displacement undefined
            assert F[7, 1] == -np.inf and F[8, 1] == np.inf and np.isnan(F[[7, 8], 2:]).all(), what
        assert np.isfinite(np.delete(F, [7, 8], 0)).all(), what


def test_inverse_cube_below_the_range(gpu):
    """r^-3 = 1e-315, but q r^-2 = 1e-10."""
    n, r, q = 2, 1e105, 1e200
    pos, S = np.array([[0.0, 0.0, 0.0], [r, 0.0, 0.0]]), np.full((n, 1), q)
    for what, F in _evaluations(pos, S, False, True):
        print(what, F, flush=True)
        assert np.allclose(F, [[-q / r / r, 0, 0], [q / r / r, 0, 0]], rtol=1e-14, atol=0), what
