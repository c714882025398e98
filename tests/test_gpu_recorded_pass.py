"""A counting pass that the caller records from the context's stream into a HIP
graph of their own, as the graph's first pass (nothing that a pass allocates is
there yet) and as a later one: every replay, between other passes, gives the
oracle's counts."""
import ctypes as C

import numpy as np
import pytest

import oracle
from acctricnt_amd import cn, graph as G

pytestmark = pytest.mark.gpu

THREAD_LOCAL = 1


@pytest.fixture(scope="module")
def hip():
    lib = C.CDLL("libamdhip64.so")
    vp = C.c_void_p
    lib.hipStreamBeginCapture.argtypes = [vp, C.c_int]
    lib.hipStreamEndCapture.argtypes = [vp, C.POINTER(vp)]
    lib.hipGraphInstantiate.argtypes = [C.POINTER(vp), vp, vp, vp, C.c_size_t]
    lib.hipGraphLaunch.argtypes = [vp, vp]
    lib.hipGraphExecDestroy.argtypes = [vp]
    lib.hipGraphDestroy.argtypes = [vp]
    return lib


@pytest.mark.parametrize("first", [True, False])
@pytest.mark.parametrize("maker", [lambda: G.gen_rmat(17, 16, seed=5), lambda: G.gen_rmat(12, 8, seed=2)],
                         ids=["dense", "small"])
def test_recorded_by_the_caller(built, hip, maker, first):
    g = maker()
    ref, total = oracle.cn_bitmap(g), oracle.triangle_count_bitmap(g)
    with cn.Context(0) as ctx, ctx.upload(g) as rg:
        if not first:
            rg.compute("forward")
        graph, execution = C.c_void_p(), C.c_void_p()
        assert hip.hipStreamBeginCapture(ctx.stream(), THREAD_LOCAL) == 0
        try:
            rg.compute("forward", raw=True)
        finally:
            rc = hip.hipStreamEndCapture(ctx.stream(), C.byref(graph))
        assert rc == 0
        assert hip.hipGraphInstantiate(C.byref(execution), graph, None, None, 0) == 0
        for k in range(4):
            if k:
                cnt, t = rg.count_all_edges("forward")
                assert np.array_equal(cnt, ref) and t == total
            assert hip.hipGraphLaunch(execution, ctx.stream()) == 0
            cnt, t = rg.download()
            assert np.array_equal(cnt, ref - 2) and t == total
        assert hip.hipGraphExecDestroy(execution) == 0 and hip.hipGraphDestroy(graph) == 0
