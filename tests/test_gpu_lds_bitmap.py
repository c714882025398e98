"""The bitmap path's LDS bitmaps (k_bmp_lds in k_paths.hip) against the oracle:
vertex counts around a 32-id and a 128-id boundary of the bitmap and on both
sides of the limit to HBM bitmaps, lists whose lengths leave every remainder
mod 4 (16-byte groups), the last list of the adjacency array, sources with
more upper slots than one unit, and the counts left by a pass on another
path."""
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


def hubs_and_pairs(n, hubs, seed):
    """`hubs` vertices next to every other vertex in turn and to each other,
    and random pairs: degrees of all remainders, the highest ids in every hub's list."""
    rng = np.random.default_rng(seed)
    src = [np.full(n // (k + 1), k) for k in range(hubs)]
    dst = [n - 1 - np.arange(n // (k + 1)) for k in range(hubs)]
    src.append(rng.integers(0, n, 3 * n))
    dst.append(rng.integers(0, n, 3 * n))
    return G.from_edges(n, np.concatenate(src), np.concatenate(dst), name=f"hubs{n}x{hubs}")


GRAPHS = {
    "clique700": lambda: BF.complete(700),
    "n2047": lambda: hubs_and_pairs(2047, 5, 1),
    "n2048": lambda: hubs_and_pairs(2048, 5, 2),
    "n2049": lambda: hubs_and_pairs(2049, 5, 3),
    "n2177": lambda: hubs_and_pairs(2177, 7, 4),
    "lds_limit": lambda: hubs_and_pairs(1 << 19, 3, 5),
    "past_limit": lambda: hubs_and_pairs((1 << 19) + 1, 3, 6),
    "rmat15": lambda: G.gen_rmat(15, 20, seed=7),
}


@pytest.mark.parametrize("name", sorted(GRAPHS))
def test_lds_bitmap(ctx, name):
    g = GRAPHS[name]()
    print(f"[lds bitmap] {name} n={g.n} m={g.m}", flush=True)
    ref = oracle.cn_bitmap(g)
    total = oracle.triangle_count_bitmap(g)
    with ctx.upload(g) as rg:
        for hash_max, chunk in ((256, 512), (0, 64), (256, 100), (2048, 512)):
            rg.set_param("bmp_hash_max", hash_max)
            rg.set_param("chunk", chunk)
            for raw in (False, True):
                cnt, t = rg.count_all_edges("bitmap", raw=raw)
                bad = np.nonzero(cnt != ref - (2 if raw else 0))[0]
                assert bad.size == 0, f"{bad.size} slots differ, first {bad[:5]}"
                assert t == total
            rg.compute("forward")
