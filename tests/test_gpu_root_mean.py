"""The root centre is the sequential FP64 mean bit for bit (numpy's cumsum adds
in index order, one rounding per addition): run and batch edges, sums that
cross binades and zero, and additions that are all halfway cases, with both
parities of the running sum."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _case(kind, n):
    rng = np.random.default_rng(n)
    if kind == "uniform":
        return rng.random((n, 3))
    if kind == "centred":  # the running sum wanders around zero
        return rng.normal(size=(n, 3)) * rng.lognormal(0, 0.5, (n, 1))
    if kind == "negative":
        return -rng.random((n, 3)) - 1e-3
    if kind == "zeros":
        return np.where(rng.random((n, 3)) < 0.1, 0.0, rng.normal(size=(n, 3)))
    # halfway cases: the sum stays near 2^52 (ulp 1), additions of odd halves
    x = rng.integers(-4, 5, (n, 3)) + 0.5
    x[0] = 2.0 ** 52 * np.array([1.0, 1.5, -1.25])
    return x


@pytest.mark.parametrize("kind,sizes", [
    ("uniform", (1, 2, 255, 256, 257, 16384, 16385, 70001)),
    ("centred", (3, 257, 20000, 300007)),
    ("negative", (511, 40000)),
    ("zeros", (1000, 33000)),
    ("ties", (300, 4000, 4095)),
])
def test_root_centre_is_the_sequential_mean(gpu, kind, sizes):
    from fmmgen_amd import build_tree
    for n in sizes:
        x = np.ascontiguousarray(_case(kind, n))
        print(f"{kind} n={n}", flush=True)
        S = torch.ones(n, 1, dtype=torch.float64, device="cuda")
        t = build_tree(torch.from_numpy(x).cuda(), S, n, 4096, 2, 0.5)
        want = np.cumsum(x, axis=0)[-1] / n
        assert np.array_equal(t.export_cells()[0][0, :3], want), (kind, n)
