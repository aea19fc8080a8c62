"""The gradient's workspace holds the rows its kernels write, and no more: a row of
sums a block, at most 128 of them."""
from fmmgen_amd import _lib


def test_workspace_is_a_row_a_block():
    L = _lib.load()
    row = _lib.MLP_PARAMS + 2
    # blocks of two tiles of 16 samples from 42 samples on, longer runs beyond 128 blocks
    for B, blocks in ((1, 1), (41, 1), (42, 2), (64, 2), (65, 3), (2048, 64), (4096, 128), (4097, 86),
                      (_lib.MLP_NOALLOC_MAX_BATCH, 128), (1 << 20, 128)):
        assert L.fmm_mlp_work_floats(B) == blocks * row, B
    assert L.fmm_mlp_work_floats(0) == 0
