"""The direct sum at the ends of its ranges: no sources at all (through the C
ABI), and the block forms of dipoles and quadrupoles on both sides of their
target counts, with a coincident pair, against the oracle's sums."""
import ctypes

import numpy as np
import pytest
import torch

from oracle import oracle as O
from tests import util

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("so,outsz", [(0, 4), (0, 1), (0, 3), (1, 3), (2, 4)])
@pytest.mark.parametrize("nt", [1, 767, 768])
def test_no_sources(gpu, so, outsz, nt):
    """Every target is out of range then: NaN rows, and no source is read."""
    from fmmgen_amd import _lib
    buf = torch.zeros(16, dtype=torch.float64, device="cuda")
    tg = torch.from_numpy(np.arange(nt) % 3 - 1).cuda()
    F = torch.zeros(nt, outsz, dtype=torch.float64, device="cuda")
    print(f"no sources: so={so} outputs={outsz} targets={nt}", flush=True)
    p = [ctypes.c_void_p(t.data_ptr()) for t in (buf, tg, F)]
    st = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    _lib.check(_lib.load().fmm_direct_sampled(p[0], p[0], 0, p[1], nt, so, outsz, p[2], st))
    assert torch.isnan(F).all()


@pytest.fixture(scope="module", params=[1, 2])
def large_set(request):
    """Dipoles or quadrupoles with a coincident pair, above the size from which a
    block's targets and threads follow from the target count, and the oracle's sums."""
    so, n = request.param, 17000
    rng = np.random.default_rng(n + so)
    pos, S = rng.random((n, 3)), rng.normal(size=(n, 3 * so))
    pos[17] = pos[400]
    outsz = 4 if so == 2 else 3
    want = O.OracleTree(pos, S, n + 1, so + 1, 0.5, source_order=so, outputsize=outsz).compute_field_fmm(mask=8)
    return so, outsz, pos, S, want


@pytest.mark.parametrize("nt", [7, 511, 512, 767, 768, 1023, 1024, 1100])
def test_multipole_block_forms(gpu, large_set, nt):
    from fmmgen_amd import direct_sum
    so, outsz, pos, S, want = large_set
    tg = np.random.default_rng(nt).permutation(len(pos))[:nt]
    tg[[0, nt // 2, nt - 1]] = 17, 5, 400
    dev = [torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in (pos, S, tg)]
    print(f"so={so} targets={nt}", flush=True)
    F = direct_sum(*dev, source_order=so, outsz=outsz).cpu().numpy()
    hit = np.isin(tg, (17, 400))
    assert np.isnan(F[hit]).all() and np.isnan(want[tg[hit]]).all()
    assert util.rel_norm(F[~hit], want[tg[~hit]]) <= 1e-12
