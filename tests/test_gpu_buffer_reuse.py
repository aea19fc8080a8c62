"""Buffers kept from earlier trees: trees of other sizes built, evaluated and
destroyed in between, interleaved lifetimes, two threads on streams of their
own, and a build that fails, leave every result as it is in a fresh process
state (the first of each)."""
import gc
import threading

import numpy as np
import pytest
import torch

from tests import util

pytestmark = pytest.mark.gpu


def _inputs(n, seed):
    rng = np.random.default_rng(seed)
    return torch.from_numpy(util.blobs(n, seed)).cuda(), torch.from_numpy(rng.uniform(-1, 1, (n, 1))).cuda()


def _step(n, seed, order, modes=("plain",)):
    from fmmgen_amd import build_tree
    pos, S = _inputs(n, seed)
    t = build_tree(pos, S, n, 32, order, 0.5)
    out = []
    for m in modes:
        F = torch.full((n, 4), float("nan"), dtype=torch.float64, device="cuda")
        out.append(t.compute_field_fmm(F, mode=m).clone())
    return t, out


def _same(a, b):
    # the order of atomic additions varies: FP64 rounding only
    return all(((x - y).norm() / x.norm()).item() < 1e-13 for x, y in zip(a, b))


def test_results_do_not_depend_on_earlier_trees(gpu):
    sizes = [(3000, 1, 4), (40000, 2, 6), (500, 3, 8), (20000, 4, 3)]
    first = [_step(*s)[1] for s in sizes]
    gc.collect()
    for rnd in range(3):
        alive = []
        for s, want in zip(sizes, first):
            t, got = _step(*s)
            assert _same(want, got), (rnd, s)
            alive.append(t)
            if rnd == 1 and len(alive) > 1:
                alive.pop(0)


def test_failing_build_between(gpu):
    from fmmgen_amd import _lib, build_tree
    want = _step(5000, 9, 5)[1]
    p = torch.zeros(100, 3, dtype=torch.float64, device="cuda")  # coincident: deeper than 21 levels
    with pytest.raises(_lib.FmmError):
        build_tree(p, torch.ones(100, 1, dtype=torch.float64, device="cuda"), 100, 8, 3, 0.5)
    assert _same(want, _step(5000, 9, 5)[1])


def test_two_threads_on_their_own_streams(gpu):
    jobs = {0: (9000, 11, 5), 1: (13000, 12, 4)}
    want = {k: _step(*j)[1] for k, j in jobs.items()}
    torch.cuda.synchronize()
    bad = []

    def work(k):
        st = torch.cuda.Stream()
        with torch.cuda.stream(st):
            for _ in range(5):
                t, got = _step(*jobs[k])
                st.synchronize()
                if not _same(want[k], got):
                    bad.append(k)
                del t
    ths = [threading.Thread(target=work, args=(k,)) for k in jobs]
    for th in ths:
        th.start()
    for th in ths:
        th.join()
    assert not bad
