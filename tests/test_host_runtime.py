"""Host code around the kernels: contexts, graphs, results and error paths,
with tests/c/host_runtime.c in the place of the HIP runtime (host memory,
kernels that do nothing, calls that can be made to fail).  Every scenario
below runs in a process of its own."""
import ctypes as C
import os
import subprocess
import sys

import numpy as np
import pytest

from cases import CASES
from libecp_amd import native
from libecp_amd.workloads import plain_small, uneven_batch

HERE = os.path.dirname(os.path.abspath(__file__))
SCENARIOS = {}


def scenario(f):
    SCENARIOS[f.__name__] = f
    return f


def count(name):
    rt = C.CDLL("libamdhip64.so.7")
    rt.hrt_get.restype = C.c_long
    return rt.hrt_get(name.encode())


def make(name, value):
    C.CDLL("libamdhip64.so.7").hrt_set(name.encode(), C.c_long(value))


@scenario
def matrix_before_a_fetch_is_an_error():
    b = native.Batch([plain_small(0)])
    assert b.matrix(0)[0] == -1 and "fetch" in native.last_error()
    b.execute(1)
    assert b.matrix(0)[0] == -1
    b.fetch()
    assert b.matrix(0)[0] == 0
    b.close()
    b = native.Batch([CASES["no_ecp"]()])  # nothing to fetch
    assert b.triplets()[1] == 0 and b.matrix(0)[0] == 0
    b.close()


@scenario
def quadrature_span_is_recorded_by_replays():
    """Two kernels of 100 ticks each between the pair's events, in the eager
    evaluation and in replays; no error is left behind where the runtime
    refuses external event records."""
    make("external_refused", 1)
    b = native.Batch([plain_small(0)])
    b.set_param("fuse", 1)
    b.execute(1)
    assert (b.quadrature_ms(), b.quadrature_samples) == (200.0, 1)
    b.execute(12)
    assert (b.quadrature_ms(), b.quadrature_samples) == (200.0, 8)
    assert C.CDLL("libamdhip64.so.7").hipGetLastError() == 0
    b.close()


def fails(f, *args):
    try:
        f(*args)
    except RuntimeError:
        return True
    return False


@scenario
def failed_calls_of_a_sequence_are_reported():
    """A launch that fails under capture, and a wait between streams."""
    for fuse in (0, 1):
        b = native.Batch([plain_small(0)])
        b.set_param("fuse", fuse)
        b.execute(1)
        make("launch_fail", 1)
        assert fails(b.execute, 2)
        make("launch_fail", 0)
        assert b.execute(2) > 0
        b.close()
        assert count("graphs") == count("execs") == 0
        make("wait_fail", 1)
        b = native.Batch([plain_small(0)])
        b.set_param("fuse", fuse)
        assert fails(b.execute, 1)
        assert fails(b.profile)
        make("wait_fail", 0)
        assert b.execute(1) > 0
        b.close()


@scenario
def graphs_of_a_failed_capture_are_freed():
    for copy in (1, 3):
        b = native.Batch([plain_small(0)])
        b.set_param("fuse", 1)
        make("instantiate_fail", copy)
        assert fails(b.execute, 2)
        assert b.execute(2) > 0
        b.close()
        assert count("graphs") == count("execs") == 0


@scenario
def contexts_are_not_reused_after_a_failed_call():
    m = plain_small(0)
    P = np.eye(m.nao)

    def batch():
        b = native.Batch([m])
        try:
            b.execute(1)
        finally:
            b.close()

    def handle():
        h = native.Handle(m)
        try:
            assert h.contract(P)[0] == 0
        finally:
            h.close()

    for use in (batch, handle):
        use()
        n = count("contexts")
        use()
        assert count("contexts") == n      # taken from the cache
        make("launch_fail", 2)
        assert fails(use)                  # the same one, which is freed
        make("launch_fail", 0)
        assert count("contexts") == n
        use()
        assert count("contexts") == n + 1


@scenario
def idle_contexts_of_batches_stay_below_4_gib():
    """Also one that a handle took and gives back after another batch's came."""
    mols = uneven_batch(0)[:90]
    big = max(mols, key=lambda m: m.nao)

    def batch():
        b = native.Batch(mols)
        b.close()

    batch()
    one, contexts = count("device_bytes"), count("contexts")
    assert 2 << 30 < one < 4 << 30
    h = native.Handle(big)
    h.contract(np.eye(big.nao))
    assert count("contexts") == contexts   # the batch's
    batch()
    h.close()
    assert count("device_bytes") < 4 << 30


@scenario
def batches_take_no_cache_keys_from_handles():
    m = plain_small(0)
    for k in range(9):
        native.Batch([m], tol=1e-12 * (1 + k)).close()

    def handle(tol):
        h = native.Handle(m, tol=tol)
        h.contract(np.eye(m.nao))
        h.close()

    keys = [1e-11 * (2 + k) for k in range(8)]
    for tol in keys:
        handle(tol)
    n = count("contexts")
    for tol in keys:
        handle(tol)
    assert count("contexts") == n


@scenario
def idle_contexts_give_way_when_memory_runs_out():
    """To a batch and to a server whose memory would have been there without
    them."""
    mols = uneven_batch(0)[:12]
    b = native.Batch(mols)
    size = count("device_bytes")
    b.close()
    make("mem_limit", size + (1 << 20))
    b = native.Batch(mols, tol=1e-11)       # another key: a new context
    b.close()
    s = native.Server(slots=1, hbm_budget=size - (32 << 20))
    s.close()
    make("mem_limit", size // 4)
    assert fails(native.Batch, mols)
    make("mem_limit", 0)


@pytest.fixture(scope="module")
def runtime(tmp_path_factory):
    d = tmp_path_factory.mktemp("runtime")
    subprocess.run(["gcc", "-O1", "-shared", "-fPIC", "-Wl,-soname,libamdhip64.so.7", "-o",
                    str(d / "libamdhip64.so.7"), os.path.join(HERE, "c", "host_runtime.c")], check=True)
    return str(d)


@pytest.mark.parametrize("name", sorted(SCENARIOS))
def test_scenario(runtime, name):
    env = dict(os.environ, LD_LIBRARY_PATH=runtime + os.pathsep + os.environ.get("LD_LIBRARY_PATH", ""),
               PYTHONPATH=os.pathsep.join([os.path.dirname(HERE), HERE]))
    p = subprocess.run([sys.executable, "-c", f"import test_host_runtime as t; t.SCENARIOS['{name}']()"],
                       env=env, capture_output=True, text=True, timeout=120)
    assert p.returncode == 0, p.stderr[-3000:]
