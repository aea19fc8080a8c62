"""The root centre is the sequential FP64 mean bit for bit where additions lie
at, one bit above and one bit below a half of the running sum's last place, for
even and odd sums of both signs (numpy's cumsum adds in index order)."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
H = 0.5


@pytest.mark.parametrize("base", [1.5 * 2.0 ** 52, -1.25 * 2.0 ** 52])
@pytest.mark.parametrize("odd", [0, 1])
def test_near_halves(gpu, base, odd):
    from fmmgen_amd import build_tree
    near = [s * np.nextafter(H, to) for s in (1.0, -1.0) for to in (0.0, 1.0)]
    n = 3000  # 12 runs of additions, the first one holding the jump from zero
    rng = np.random.default_rng(5)
    x = np.empty((n, 3))
    for k, one in enumerate(near[:3]):  # the same addition throughout: no parity change hides a wrong one
        x[:, k] = one
    for cols in (x, np.column_stack([np.full(n, near[3])] * 3), rng.choice(near + [H, -H], (n, 3))):
        cols = np.ascontiguousarray(cols)
        cols[0] = base + odd
        print(f"base {base} odd {odd} first additions {cols[1]}", flush=True)
        S = torch.ones(n, 1, dtype=torch.float64, device="cuda")
        t = build_tree(torch.from_numpy(cols).cuda(), S, n, 4096, 2, 0.5)
        want = np.cumsum(cols, axis=0)[-1] / n
        assert np.array_equal(t.export_cells()[0][0, :3], want)
