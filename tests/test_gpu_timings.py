"""acc_cn_timings gives every kernel of a pass an entry of its own: the dense
sources' counting apart from the others', and no entry for kernels that a plan
does not launch."""
import pytest

from acctricnt_amd import graph as G

pytestmark = pytest.mark.gpu


def test_kernels_apart(built):
    from acctricnt_amd import cn

    with cn.Context(0) as ctx:
        for maker, dense in ((lambda: G.gen_rmat(17, 16, seed=5), True), (lambda: G.gen_rmat(10, 8, seed=1), False)):
            with ctx.upload(maker()) as rg:
                for _ in range(2):
                    rg.compute("forward", timing=True)
                t = rg.timings()
                want = ["k_init"] + dense * ["k_dense"] + ["k_fwd_count<4>"] + dense * ["k_dense_rows"] + ["k_combine"]
                assert list(t) == want
                assert all(0 < v < 100 for v in t.values()), t
