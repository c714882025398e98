"""Wave packs of the forward path, which probe in groups of four elements:
probe lengths around the groups and rows, and ids that differ above bit 23
alone (they share a hash slot), against the oracle."""
import numpy as np
import pytest

import oracle
from acctricnt_amd import graph as G


def cliques(sizes, holes):
    """Disjoint cliques; holes > 0 drops about 1 / holes of the edges."""
    src, dst, base = [], [], 0
    for s in sizes:
        a, b = np.triu_indices(s, 1)
        keep = (a * 7 + b * 13) % holes != 0 if holes else np.ones(len(a), bool)
        src.append(a[keep] + base)
        dst.append(b[keep] + base)
        base += s
    return G.from_edges(base, np.concatenate(src), np.concatenate(dst), name=f"cliques{len(sizes)}_{holes}")


def far_ids(k):
    """A clique of the ids i and 2^24 + i, i < k."""
    ids = np.concatenate([np.arange(k), (1 << 24) + np.arange(k)])
    a, b = np.triu_indices(2 * k, 1)
    return G.from_edges((1 << 24) + k, ids[a], ids[b], name=f"far{k}")


GRAPHS = {
    "edge": lambda: cliques([2], 0),
    "triangle": lambda: cliques([3], 0),
    "every_length": lambda: cliques(list(range(2, 71)) * 2, 0),
    "every_length_holes": lambda: cliques(list(range(2, 71)) * 2, 3),
    "many_small": lambda: cliques([3, 4, 5, 6, 9] * 3000, 0),
    "far_ids": lambda: far_ids(9),
}


@pytest.mark.gpu
@pytest.mark.parametrize("unroll", (1, 2, 4))
@pytest.mark.parametrize("name", sorted(GRAPHS))
def test_packs(built, name, unroll):
    from acctricnt_amd import cn

    g = GRAPHS[name]()
    print(f"[packs] {name} n={g.n} m={g.m} unroll={unroll}", flush=True)
    ref = oracle.cn_bitmap(g)
    with cn.Context(0) as ctx, ctx.upload(g) as rg:
        rg.set_param("fwd_unroll", unroll)
        assert rg.triangle_total("forward") == oracle.triangle_count_bitmap(g)
        cnt, total = rg.count_all_edges("forward")
        assert np.array_equal(cnt, ref)
