"""Which batch outputs a kernel may add into directly: not those whose memory the
inputs share, by whatever storage they reach it."""
import torch

from fmmgen_amd.operators import _adds_in_place


def test_shared_memory_is_found_through_other_storages():
    buf = torch.zeros(64, dtype=torch.float64)
    out = buf[:40]
    for lo, hi, apart in ((0, 10, False), (30, 50, False), (39, 41, False), (40, 64, True), (48, 64, True)):
        same = buf[lo:hi]
        other = torch.from_dlpack(buf[lo:hi])  # a storage of its own on the same memory
        assert other.data_ptr() == same.data_ptr()
        for inp in (same, other):
            assert _adds_in_place(out, 40, inp) == apart, (lo, hi)
    assert _adds_in_place(out, 40, torch.zeros(100, dtype=torch.float64))
    assert not _adds_in_place(out, 39, torch.zeros(100, dtype=torch.float64))
