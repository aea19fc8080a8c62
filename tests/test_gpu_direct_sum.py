"""The direct sum at the target counts where its block shape changes, with
ragged last blocks, targets repeated and out of range, and coincident
particles, against numpy."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _numpy(pos, q, tg):
    out = np.empty((len(tg), 4))
    with np.errstate(divide="ignore", invalid="ignore"):
        for k, i in enumerate(tg):
            d = pos[i] - pos
            r = 1.0 / np.sqrt((d * d).sum(1))
            r[i] = 0.0
            s3 = q * r ** 3
            out[k] = np.append((q * r).sum(), (s3[:, None] * d).sum(0))
    return out


@pytest.mark.parametrize("nt", [1, 7, 511, 512, 767, 768, 1023, 1024, 1027])
@pytest.mark.parametrize("n", [1, 255, 16383, 16384, 20001])
def test_direct_sum(gpu, n, nt):
    from fmmgen_amd import direct_sum
    rng = np.random.default_rng(n * nt)
    pos, q = rng.random((n, 3)), rng.uniform(-1, 1, (n, 1))
    tg = rng.integers(0, n, nt)
    dev = [torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in (pos, q, tg)]
    print(f"n={n} nt={nt}", flush=True)
    F = direct_sum(*dev).cpu().numpy()
    uniq = np.unique(tg)
    want = dict(zip(uniq, _numpy(pos, q[:, 0], uniq)))
    want = np.array([want[i] for i in tg])
    # sums of n terms, each to a few roundings of 1e-16; cancellation bounded by
    # the largest term
    assert np.abs(F - want).max() <= 1e-12 * max(1.0, np.abs(want).max())


@pytest.mark.parametrize("n,nt", [(900, 8), (17000, 600), (17000, 800), (17000, 1100)])
def test_direct_sum_special_targets(gpu, n, nt):
    """Out-of-range targets give NaN rows and leave the others alone; a
    coincident pair gives an infinite potential and an undefined field there."""
    from fmmgen_amd import direct_sum
    rng = np.random.default_rng(nt)
    pos, q = rng.random((n, 3)), rng.uniform(0.5, 1, (n, 1))
    pos[17] = pos[400]
    tg = rng.permutation(np.append(np.arange(nt - 2), (17, 400)))
    tg[3], tg[5] = -1, n
    F = direct_sum(*(torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in (pos, q, tg))).cpu().numpy()
    assert np.isnan(F[[3, 5]]).all()
    ok = np.ones(nt, dtype=bool)
    ok[[3, 5]] = False
    want = _numpy(pos, q[:, 0], tg[ok])
    hit = np.isinf(want[:, 0])
    assert hit.any() == np.isin([17, 400], tg[ok]).any()
    assert np.isposinf(F[ok][hit][:, 0]).all() and np.isnan(F[ok][hit][:, 1:]).all()
    assert np.abs(F[ok][~hit] - want[~hit]).max() <= 1e-12 * np.abs(want[~hit]).max()
