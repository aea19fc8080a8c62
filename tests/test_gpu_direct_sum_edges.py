"""The direct sum at the ends of its ranges, through the C ABI."""
import ctypes

import numpy as np
import pytest
import torch

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
