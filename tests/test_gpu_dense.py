"""The dense sources of the forward path (k_dense.hip) against the oracle, at
the sizes where their layout changes: hit matrices around 32, 256, 2048 and
4096 rows (the forms of the summing kernel; larger ones are not kept), (b, a) counters beyond the 2048 in LDS, the
last 16-bit id, packed graphs with and without dense sources, shards, and
the triangle-only pass."""
import numpy as np
import pytest

import bruteforce as BF
import oracle
from acctricnt_amd import graph as G


def band(n, half, holes=0):
    """Vertex v next to v - half .. v + half; holes > 0 drops about 1 / holes of the edges."""
    v = np.arange(n)
    src = np.concatenate([v[: n - k] for k in range(1, half + 1)])
    dst = np.concatenate([v[k:] for k in range(1, half + 1)])
    if holes:
        keep = (src * 7 + dst * 13) % holes != 0
        src, dst = src[keep], dst[keep]
    return G.from_edges(n, src, dst, name=f"band{n}x{half}")


def hub_rows(hubs, leaves):
    """`hubs` sources next to `leaves` later vertices and to the next source:
    every leaf's matrix has `hubs` rows."""
    h = np.arange(hubs)
    src = np.concatenate([np.repeat(h, leaves), h[:-1]])
    dst = np.concatenate([np.tile(hubs + np.arange(leaves), hubs), h[1:]])
    return G.from_edges(hubs + leaves, src, dst, name=f"hubs{hubs}x{leaves}")


@pytest.fixture(scope="module")
def ctx(built):
    from acctricnt_amd import cn

    assert cn.device_count() > 0, "no HIP device visible"
    c = cn.Context(0)
    yield c
    c.close()


GRAPHS = {  # each has more upper slots of dense sources than kDenseMin
    "clique1100": lambda: BF.complete(1100),    # matrices of every size up to 1024 rows
    "clique2300": lambda: BF.complete(2300),    # positions beyond the LDS counters
    "band_holes": lambda: band(5000, 150, holes=3),
    "ids65535": lambda: band(65700, 60),        # the last dense id is 65534
    "rows4090": lambda: hub_rows(4090, 66),     # the largest matrices that are kept
    "rows4200": lambda: hub_rows(4200, 66),     # not kept: counted by atomics
    "rmat17": lambda: G.gen_rmat(17, 16, seed=5),
    "rmat16_unrelabelled": lambda: G.gen_rmat(16, 24, seed=6, relabel=False),
    "chunglu40k": lambda: G.gen_chung_lu(40000, 2.1, 48, 20000, seed=7),
}


@pytest.mark.gpu
@pytest.mark.parametrize("name", sorted(GRAPHS))
def test_dense_graphs(ctx, name):
    g = GRAPHS[name]()
    print(f"[dense] {name} n={g.n} m={g.m}", flush=True)
    ref = oracle.cn_bitmap(g)
    total = oracle.triangle_count_bitmap(g)
    with ctx.upload(g) as rg:
        for chunk in (512, 100):
            rg.set_param("chunk", chunk)
            assert rg.triangle_total("forward") == total
            for raw in (False, True):
                cnt, t = rg.count_all_edges("forward", raw=raw)
                bad = np.nonzero(cnt != ref - (2 if raw else 0))[0]
                assert bad.size == 0, f"{bad.size} slots differ, first {bad[:5]}"
                assert t == total


@pytest.mark.gpu
def test_dense_batch_and_shards(ctx):
    """A packed CSR whose graphs have dense sources or none, before and after
    its partition is set, by replays, and by shares that cut through the
    dense sources."""
    parts = [BF.complete(600), G.gen_er(500, 8, seed=1), G.from_edges(3, [], []), hub_rows(200, 70),
             G.gen_rmat(13, 24, seed=2), band(2000, 100)]
    g, vo = G.pack(parts)
    ref = oracle.cn_bitmap(g)
    totals = [oracle.triangle_count(p) for p in parts]
    with ctx.upload(g) as rg:
        for partition in (False, True):
            if partition:
                rg.set_partition(vo)
            cnt, t = rg.count_all_edges("forward")
            assert np.array_equal(cnt, ref) and t == sum(totals)
            assert rg.triangle_total("forward") == t
        assert rg.graph_totals().tolist() == totals
        rg.capture("forward")
        for raw in (True, False, True):
            assert np.array_equal(rg.count_all_edges("forward", raw=raw)[0], ref - (2 if raw else 0))
            rg.replay()
            cnt, t = rg.download()
            assert np.array_equal(cnt, ref) and t == sum(totals)
            assert rg.graph_totals().tolist() == totals
        for shares in (3, 8):
            acc, tri = np.zeros(g.m, np.int64), 0
            for s in range(shares):
                rg.set_shard(shares, s)
                cnt, t = rg.count_all_edges("forward", raw=True)
                assert rg.triangle_total("forward") == t
                acc += cnt
                tri += t
            assert np.array_equal(acc, ref - 2) and tri == sum(totals)
        rg.set_shard(1, 0)
        assert np.array_equal(rg.count_all_edges("forward")[0], ref)
