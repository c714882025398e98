"""Counting with dense sources where the device has no memory for what only
makes it faster: the hit matrices at the first per-slot pass, and the tables at
the upload.  hipMalloc of that size fails on demand (tests/hip_host/fail_alloc.cpp) in a process of its
own, and every count and total equals the oracle's."""
import os
import subprocess
import sys
import textwrap

import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PROLOGUE = """
import ctypes as C, sys
import numpy as np
fail = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)
fail.fail_alloc_between.argtypes = [C.c_size_t, C.c_size_t]
fail.fail_alloc_real.argtypes = [C.c_void_p]
from acctricnt_amd import _ffi, cn, graph as G
import oracle
fail.fail_alloc_real(C.cast(_ffi.cn_lib().hipMalloc, C.c_void_p))  # the runtime's, a dependency of the library
g = G.gen_rmat(17, 16, seed=5)
ref, total = oracle.cn_bitmap(g), oracle.triangle_count_bitmap(g)

def check(rg):
    for raw in (False, True):
        cnt, t = rg.count_all_edges("forward", raw=raw)
        assert np.array_equal(cnt, ref - (2 if raw else 0)) and t == total
    assert rg.triangle_total("forward") == total
    rg.capture("forward")
    for _ in range(3):
        rg.replay()
        cnt, t = rg.download()
        assert np.array_equal(cnt, ref) and t == total
    acc, tri = np.zeros(g.m, np.int64), 0
    for s in range(3):
        rg.set_shard(3, s)
        cnt, t = rg.count_all_edges("forward", raw=True)
        acc += cnt
        tri += t
    assert np.array_equal(acc, ref - 2) and tri == total
    rg.set_shard(1, 0)
"""


@pytest.fixture(scope="module")
def run(tmp_path_factory, built):
    lib = tmp_path_factory.mktemp("fail_alloc") / "libfail_alloc.so"
    subprocess.run(["g++", "-O1", "-shared", "-fPIC", os.path.join(ROOT, "tests", "hip_host", "fail_alloc.cpp"), "-o",
                    str(lib)], check=True, capture_output=True, text=True)

    def go(program):
        r = subprocess.run([sys.executable, "-c", PROLOGUE + textwrap.dedent(program), str(lib)], cwd=ROOT,
                           capture_output=True, text=True, timeout=100)
        assert r.returncode == 0, r.stdout + r.stderr
    return go


def test_without_hit_matrices(run):
    run("""
    with cn.Context(0) as ctx, ctx.upload(g) as rg:
        before = rg.device_bytes()
        rg.compute("forward")
        hits = rg.device_bytes() - before
        assert hits > 1 << 20
    with cn.Context(0) as ctx, ctx.upload(g) as rg:
        fail.fail_alloc_between(hits, hits + (64 << 10))
        check(rg)
        assert fail.fail_alloc_failed() > 0
        fail.fail_alloc_between(1, 0)
        check(rg)
    """)


def test_without_tables(run):
    run("""
    for size in (16 * g.n, 24 * g.n):  # the vertex records, the tables' scratch
        with cn.Context(0) as ctx:
            fail.fail_alloc_between(size, size + (size >> 2) + (64 << 10))
            with ctx.upload(g) as rg:
                assert fail.fail_alloc_failed() > 0
                fail.fail_alloc_between(1, 0)
                check(rg)
                rg.set_param("chunk", 256)  # the next plan finds memory
                check(rg)
    """)


def test_admission_within_the_budget(run):
    """A served graph is counted with dense sources only where their tables and
    matrices fit the server's budget beside it."""
    run("""
    from acctricnt_amd import serve
    with cn.Context(0) as ctx, ctx.upload(g) as rg:
        before = rg.device_bytes()
        rg.compute("forward")
        hits = rg.device_bytes() - before
    ref_scan = oracle.scan(g, ref, "0.3", 5)
    # the graph and one result slot: 28.3 and 1.1 bytes a slot, 20 and 45 a vertex
    tight = 30 * g.m + 65 * g.n + (4 << 20)
    for budget, asked in ((tight, False), (2 * tight, True)):
        with cn.Context(0) as ctx, serve.Server(ctx, hbm_budget=budget, slots=1) as sv:
            fail.fail_alloc_between(hits, hits + (64 << 10))
            gid = sv.add_graph(g)
            assert (fail.fail_alloc_failed() > 0) == asked
            res = sv.query(gid, "0.3", 5)
            assert np.array_equal(res["label"], ref_scan["label"])
    """)
