"""The pair buffer of a workspace on memory that an upload has just given back:
a query runs, a graph with dense sources is uploaded, whose table scratch is as
large as the buffer, and the query's pairs are read; the pairs and the uploaded
graph's counts are right."""
import numpy as np
import pytest

import oracle
from acctricnt_amd import graph as G

pytestmark = pytest.mark.gpu


def test_pairs_after_an_upload(built):
    from acctricnt_amd import cn

    b = G.gen_rmat(17, 16, seed=5)
    # 8 bytes a slot of a, 24 bytes a vertex of b
    a = G.gen_er(3 * b.n // 14, 13, seed=3)
    assert 0.85 < 8 * a.m / (24 * b.n) < 1.02, (a.m, b.n)
    cnt_a, cnt_b, total_b = oracle.cn_merge(a), oracle.cn_bitmap(b), oracle.triangle_count_bitmap(b)
    ref = oracle.scan(a, cnt_a, "0.2", 2)
    with cn.Context(0) as ctx, ctx.upload(a) as ra, ra.scan_workspace() as ws:
        ws.run("0.2", 2)
        want = np.unique(ws.pairs(), axis=0)  # with nothing in between
    for _ in range(3):
        with cn.Context(0) as ctx, ctx.upload(a) as ra, ra.scan_workspace() as ws:
            ws.run("0.2", 2)
            with ctx.upload(b) as rb:
                pairs = ws.pairs()
                cnt, total = rb.count_all_edges("forward")
                assert rb.triangle_total("forward") == total
            res = ws.results()
        assert np.array_equal(cnt, cnt_b) and total == total_b
        assert np.array_equal(res["label"], ref["label"])
        assert np.array_equal(np.unique(pairs, axis=0), want)
