"""Memory kept after the last tree goes back to the device on request, and trees
built afterwards give the same results."""
import gc

import numpy as np
import pytest
import torch

from tests import util

pytestmark = pytest.mark.gpu


def _same(a, b):
    # the order of atomic additions may vary: FP64 rounding only
    return ((a - b).norm() / a.norm()).item() < 1e-13


def test_trim_returns_the_memory(gpu):
    import fmmgen_amd
    n = 200_000
    pos = torch.from_numpy(util.blobs(n, 2)).cuda()
    S = torch.from_numpy(np.random.default_rng(3).uniform(-1, 1, (n, 1))).cuda()
    out = []
    for _ in range(2):
        t = fmmgen_amd.build_tree(pos, S, n, 64, 4, 0.5)
        out.append(t.compute_field_fmm(torch.empty(n, 4, dtype=torch.float64, device="cuda")).clone())
        live = fmmgen_amd.trim_memory()
        again = t.compute_field_fmm(torch.empty(n, 4, dtype=torch.float64, device="cuda"))
        assert live == 0 and _same(again, out[-1])  # a live tree keeps its own
        del t
        gc.collect()
        before = torch.cuda.mem_get_info()[0]
        assert fmmgen_amd.trim_memory(1 << 62) > 0  # the destroyed tree's buffers
        assert fmmgen_amd.trim_memory() == 0
        assert torch.cuda.mem_get_info()[0] > before
    assert _same(*out)
