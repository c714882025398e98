"""The autotuner's trials of the counting grid: at an average degree of 16 and
more k_fwd_count takes at most 64 workgroups per compute unit, so a larger
`persist` is a trial of its own only below that degree or beside dense sources,
whose kernel takes it as it is."""
import pytest

from acctricnt_amd import graph as G

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("maker,trials", [
    (lambda: G.gen_er(20000, 24, seed=1), {0, 8, 24}),             # 64, 128 and 256 are one grid
    (lambda: G.gen_er(30000, 8, seed=2), {0, 8, 24, 64, 128}),
    (lambda: G.gen_rmat(17, 16, seed=5), {0, 8, 24, 64, 128}),     # dense sources
], ids=["deg24", "deg8", "dense"])
def test_grid_trials(built, maker, trials):
    from acctricnt_amd import cn

    with cn.Context(0) as ctx, ctx.upload(maker()) as rg:
        rep = rg.tune(forward_only=True)
        tried = {v for _, param, v, _ in rep["trials"] if param == "persist"}
        # where the grids differ, the default 256 is timed again once another value is kept
        assert tried - ({256} if 64 in trials else set()) == trials
