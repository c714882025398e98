"""What the host code of libacc_cn.so asks of the HIP runtime, on the CPU: each
test runs a short program over a stand-in runtime (tests/hip_host/fake_hip.cpp)
whose memory is the host's, whose kernels do nothing and which logs the calls."""
import os
import shutil
import subprocess
import sys
import textwrap

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")
pytestmark = pytest.mark.skipif(shutil.which("g++") is None, reason="no host compiler")

PROLOGUE = """
import ctypes as C, sys
import numpy as np
fake = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)
fake.fake_log.restype = C.c_char_p
fake.fake_limit.argtypes = [C.c_size_t]
fake.fake_held.restype = C.c_size_t
fake.fake_fail_new.argtypes = [C.c_long]
from acctricnt_amd import cn, serve
from acctricnt_amd._ffi import AccError
from acctricnt_amd.graph import CSRGraph

def edgeless(n):
    return CSRGraph(np.zeros(n + 1, np.uint32), np.zeros(0, np.int32))

def log():
    return [l.split(" ", 2) for l in fake.fake_log().decode().splitlines()]
"""


@pytest.fixture(scope="module")
def run(tmp_path_factory, built):
    lib = tmp_path_factory.mktemp("hip_host") / "libfake_hip.so"
    subprocess.run(["g++", "-O1", "-g", "-std=c++17", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__", "-I",
                    os.path.join(ROCM, "include"), os.path.join(ROOT, "tests", "hip_host", "fake_hip.cpp"), "-o",
                    str(lib)], check=True, capture_output=True, text=True)

    def go(program):
        r = subprocess.run([sys.executable, "-c", PROLOGUE + textwrap.dedent(program), str(lib)], cwd=ROOT,
                           capture_output=True, text=True, timeout=120)
        assert r.returncode == 0, r.stdout + r.stderr
        return r.stdout
    return go


def test_pairs_wait_for_the_context_stream(run):
    """The pair buffer may be a block whose last use is still queued on the
    context's stream (the scratch of an upload after the query was launched): the
    workspace's stream waits for the context's before the pair kernel writes it."""
    run("""
    with cn.Context(0) as ctx, ctx.upload(edgeless(40)) as a, a.scan_workspace() as ws:
        ws.run("0.5", 2)
        with ctx.upload(edgeless(50)):
            fake.fake_clear()
            ws.pairs()
            calls = log()
        launch = next(i for i, c in enumerate(calls) if c[0] == "launch" and "k_sj_pairs" in c[2])
        stream = calls[launch][1]
        recorded = [c[1] for c in calls[:launch] if c[0] == "record" and int(c[2], 16) == ctx.stream()]
        assert any(c[0] == "wait" and c[1] == stream and c[2] in recorded for c in calls[:launch]), calls
        # and the wait comes after the buffer was taken
        taken = [i for i, c in enumerate(calls) if c[0] == "alloc"]
        waits = [i for i, c in enumerate(calls) if c[0] == "wait"]
        assert all(t < max(waits) for t in taken), calls
    """)


def test_result_slots_take_what_the_pool_holds_idle(run):
    """Freed blocks of the context's graphs are kept for its next ones; where the
    device has no more memory, a serving result slot gets it back from them."""
    run("""
    with cn.Context(0) as ctx:
        ctx.upload(edgeless(1200000)).release()  # leaves blocks far larger than any below
        with serve.Server(ctx, slots=1, streams=1) as sv:
            # room for the graph (1.3 MB at most), not for its result slot (4.4 MB)
            fake.fake_limit(fake.fake_held() + 2500000)
            sv.query(sv.add_graph(edgeless(100000)), "0.5", 2)
    """)


def test_serving_budget_counts_idle_blocks(run):
    """hbm_budget bounds the device memory of a server's graphs, result slots and
    what is kept of evicted graphs, whatever sizes came and went."""
    run("""
    budget = 25 << 20
    with cn.Context(0) as ctx:
        with serve.Server(ctx, hbm_budget=budget, slots=1, streams=1) as sv:
            for n in (1000000, 860000, 740000, 630000, 540000, 460000, 390000, 330000, 280000):
                sv.add_graph(edgeless(n))
                assert fake.fake_held() <= budget, (n, fake.fake_held())
            st = sv.stats()
            assert st["evictions"] and fake.fake_held() >= st["graph_bytes"] + st["slot_bytes"]
    """)


def test_merge_windows_of_small_units(run):
    """Workgroup units with few neighbors take the merge path's small windows,
    whatever the bitmap path makes of them."""
    run("""
    n, deg = 300, 100  # (trusted: every kernel does nothing, so nothing is checked)
    off = np.arange(n + 1, dtype=np.uint32) * deg
    g = CSRGraph(off, np.tile(np.arange(deg, dtype=np.int32), n))
    with cn.Context(0) as ctx, ctx.upload(g, validate=False) as rg:
        fake.fake_clear()
        rg.compute("merge")
        names = [c[2] for c in log() if c[0] == "launch"]
        assert any("k_merge_winILi11E" in k for k in names), names
        assert not any("k_merge_winILi13E" in k for k in names), names
        fake.fake_clear()
        rg.set_param("bmp_hash_max", 0)  # every workgroup unit a hub
        rg.compute("merge")
        names = [c[2] for c in log() if c[0] == "launch"]
        assert any("k_merge_winILi13E" in k for k in names) and not any("k_merge_winILi11E" in k for k in names)
    """)


def test_release_without_host_memory(run):
    """Releasing a graph needs no host memory: no exception leaves the library,
    and what the pool cannot note goes back to the device."""
    run("""
    with cn.Context(0) as ctx:
        held = fake.fake_held()
        rg = ctx.upload(edgeless(100000))
        release, h = rg._lib.acc_graph_release, rg._h
        rg._h = None
        fake.fake_fail_new(0)
        release(h)
        fake.fake_fail_new(-1)
        ctx.upload(edgeless(70000)).release()
    assert fake.fake_held() == held == 0
    """)
