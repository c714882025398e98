"""The per-slot SCAN kernels at the borders of their forms, against the
oracle: slot counts of every remainder mod 4 (16-byte groups of slots) and
vertex counts around a 64-vertex word of core bits, core shares on each side of the quarter
that selects CheckHub's order, and exact ties of the similarity with eps, with
and without caller ids."""
import numpy as np
import pytest

import bruteforce as BF
import oracle
from acctricnt_amd import graph as G

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx(built):
    from acctricnt_amd import cn

    assert cn.device_count() > 0, "no HIP device visible"
    c = cn.Context(0)
    yield c
    c.close()


def blocks_and_noise(n, size, noise, seed):
    """Cliques of `size` consecutive ids plus noise random edges."""
    rng = np.random.default_rng(seed)
    v = np.arange(n)
    src = np.concatenate([v[: n - k] for k in range(1, size)] + [rng.integers(0, n, noise)])
    dst = np.concatenate([v[k:] for k in range(1, size)] + [rng.integers(0, n, noise)])
    keep = (src // size == dst // size) | (np.arange(src.size) >= src.size - noise)
    return G.from_edges(n, src[keep], dst[keep], name=f"blocks{n}x{size}+{noise}")


GRAPHS = {
    "n63": lambda: blocks_and_noise(63, 7, 40, 1),
    "n64": lambda: blocks_and_noise(64, 8, 41, 2),
    "n65": lambda: blocks_and_noise(65, 5, 43, 3),
    "n257": lambda: blocks_and_noise(257, 6, 301, 4),
    "few_cores": lambda: blocks_and_noise(20000, 2, 90001, 5),
    "half_cores": lambda: blocks_and_noise(20001, 12, 60000, 6),
    "most_cores": lambda: blocks_and_noise(20002, 30, 30001, 7),
    "cube": lambda: G.from_edges(8, [a for a in range(8) for b in (1, 2, 4) if a < a ^ b],
                                 [a ^ b for a in range(8) for b in (1, 2, 4) if a < a ^ b]),
    "clique7": lambda: BF.complete(7),
    "star2": lambda: BF.star(2),
}


@pytest.mark.parametrize("name", sorted(GRAPHS))
def test_scan_forms(ctx, name):
    g = GRAPHS[name]()
    cnt = oracle.cn_merge(g)
    old = np.random.default_rng(1).permutation(g.n).astype(np.int32)
    with ctx.upload(g) as rg, rg.scan_workspace() as ws:
        for old_id in (None, old):
            rg.set_vertex_ids(old_id)
            for eps in ("0.3", "0.5", "0.7", "1"):
                for mu in (1, 3, 6):
                    want = oracle.scan(g, cnt, eps, mu, old_id=old_id)
                    ws.run(eps, mu)
                    got = ws.results(sim=True, core_count=True)
                    where = f"{name} m={g.m} eps={eps} mu={mu} ids={old_id is not None}"
                    for key in ("label", "cluster_id", "sim", "core_count"):
                        assert np.array_equal(got[key], want[key]), f"{where}: {key}"
                    for key in ("core_num", "cluster_num", "hub_num", "outlier_num"):
                        assert got[key] == want[key], f"{where}: {key}"
