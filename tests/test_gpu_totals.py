"""Totals read without a copy: repeated passes leave the partial sums zero for
the next, and threads that share a context get their own graph's total."""
import threading

import numpy as np
import pytest

import oracle
from acctricnt_amd import graph as G

GRAPHS = [
    lambda: G.from_edges(3, np.array([0, 0, 1]), np.array([1, 2, 2]), name="triangle"),
    lambda: G.from_edges(5, np.array([0, 1]), np.array([1, 2]), name="path"),
    lambda: G.gen_rmat(10, 8, seed=1),
    lambda: G.gen_rmat(17, 16, seed=5),  # with dense sources
]


@pytest.mark.gpu
@pytest.mark.parametrize("threads", (1, 6))
def test_totals(built, threads):
    from acctricnt_amd import cn

    graphs = [f() for f in GRAPHS]
    want = [oracle.triangle_count_bitmap(g) for g in graphs]
    bad = []
    with cn.Context(0) as ctx:

        def work(t):
            for r in range(6):
                i = (t + r) % len(graphs)
                with ctx.upload(graphs[i]) as rg:
                    for _ in range(3):
                        got = rg.triangle_total("forward")
                        if got != want[i]:
                            bad.append((i, got))
                    rg.triangle_launch()
                    rg.compute("forward")
                    total = rg.download()[1]
                    if total != want[i]:
                        bad.append((i, "count", total))

        ts = [threading.Thread(target=work, args=(t,)) for t in range(threads)]
        for t in ts:
            t.start()
        for t in ts:
            t.join()
    assert not bad, bad[:5]
