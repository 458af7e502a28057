"""A handle in a context that earlier jobs have used: nothing of theirs is
read.  Batches clear their results when they are created; a handle's blocks
are whatever was in the memory until its kernels write them, also those of a
failed integration, which the contraction sums before it reports the code."""
import numpy as np
import pytest

from libecp_amd import native
from libecp_amd.workloads import high_l


def _contract(m, n):
    P = np.random.default_rng(3).standard_normal((m.nao, m.nao))
    h = native.Handle(m, n=n)
    try:
        rc, out = h.contract(P)
        return rc, np.asarray(out)
    finally:
        h.close()


@pytest.mark.gpu
@pytest.mark.parametrize("n", [0, 1])
def test_failed_blocks_of_a_handle(n):
    bad, other = high_l(1003), high_l(1000)
    was = native.cache_enable(True)
    try:
        used = []
        for _ in range(2):
            _contract(other, n)
            used.append(_contract(bad, n))
        native.cache_enable(False)
        fresh = _contract(bad, n)
    finally:
        native.cache_clear()
        native.cache_enable(was)
    assert fresh[0] != 0
    for rc, out in used:
        assert rc == fresh[0] and np.array_equal(out, fresh[1])
