"""The network gradient at the sizes where its split changes: one sample, a
full and a ragged sample tile, the largest batch of a single block and the
smallest of two, ragged and full grids, and batches whose blocks take several
tiles, against the FP64 oracle; repeated calls agree bit for bit."""
import numpy as np
import pytest
import torch

from oracle import mlp_oracle as MO

pytestmark = pytest.mark.gpu


def _f32(a):
    return torch.from_numpy(np.ascontiguousarray(a, dtype=np.float32)).cuda()


@pytest.mark.parametrize("B", [1, 15, 16, 17, 41, 42, 300, 2048, 4097, 8192, 20001])
def test_gradient_matches_oracle(gpu, B):
    from fmmgen_amd import learned as LN
    rng = np.random.default_rng(B)
    X = rng.normal(size=(B, MO.F)).astype(np.float32)
    T = rng.normal(size=(B, MO.O)).astype(np.float32)
    mask = (rng.random((B, MO.O)) < 0.8).astype(np.float32)
    mask[0, 0] = 1.0
    p = MO.init(7).astype(np.float32)
    print(f"gradient of {B} samples", flush=True)
    loss, g = LN.grad(_f32(X), _f32(T), _f32(mask), _f32(p))
    Lo, go = MO.grad(*(a.astype(np.float64) for a in (X, T, mask, p)))
    # FP32 dot products of at most 64 terms a layer, three layers each way, and
    # sums over the batch in runs: some 10^2 roundings of 6e-8 in a chain
    gn = g.cpu().numpy().astype(np.float64)
    assert np.linalg.norm(gn - go) <= 1e-5 * np.linalg.norm(go)
    assert abs(loss.item() - Lo) <= 1e-5 * Lo
    loss2, g2 = LN.grad(_f32(X), _f32(T), _f32(mask), _f32(p))
    assert torch.equal(g, g2) and torch.equal(loss, loss2)


def test_gradient_of_a_fully_masked_batch_is_zero(gpu):
    from fmmgen_amd import learned as LN
    X, T = _f32(np.ones((50, MO.F))), _f32(np.full((50, MO.O), np.nan))
    loss, g = LN.grad(X, T, torch.zeros(50, MO.O, device="cuda"), _f32(MO.init(1)))
    assert loss.item() == 0.0 and not g.any()
