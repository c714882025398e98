"""Graphs and workspaces on memory that earlier ones of the context gave back
(DevicePool in acc_internal.h): every result of a sequence of uploads of
changing sizes equals the oracle's, on one context and on two contexts from
two threads, with a workspace still running when another graph is uploaded."""
import threading

import numpy as np
import pytest

import oracle
from acctricnt_amd import graph as G

pytestmark = pytest.mark.gpu

SIZES = [3000, 3000, 2999, 3100, 1, 40000, 3000, 39990, 2, 3000]


@pytest.fixture(scope="module")
def graphs(built):
    gs = [G.gen_er(n, 14, seed=n) if n > 2 else G.from_edges(n, [], []) for n in SIZES]
    cnts = [oracle.cn_merge(g) for g in gs]
    return [(g, c, oracle.scan(g, c, "0.3", 2)) for g, c in zip(gs, cnts)]


def rounds(graphs, failures):
    from acctricnt_amd import cn

    try:
        with cn.Context(0) as ctx:
            for relabel in (False, True):
                for g, ref, scan in graphs:
                    with ctx.upload(g, relabel=relabel) as rg, rg.scan_workspace() as ws:
                        ws.run("0.3", 2)
                        with ctx.upload(g) as other:  # while the query runs
                            cnt, _ = other.count_all_edges("bitmap")
                        res = ws.results()
                        assert np.array_equal(cnt, ref)
                        assert res["core_num"] == scan["core_num"] and res["cluster_num"] == scan["cluster_num"]
                        if not relabel:
                            assert np.array_equal(rg.download()[0], ref)
                            assert np.array_equal(res["label"], scan["label"])
    except BaseException as e:  # noqa: BLE001 -- reported by the caller
        failures.append(e)


@pytest.mark.parametrize("threads", [1, 2])
def test_memory_reused(graphs, threads):
    failures = []
    ts = [threading.Thread(target=rounds, args=(graphs, failures)) for _ in range(threads)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not failures, failures
