"""libecp_batch_quadrature_ms after graph replays, in whichever HIP runtime
the process has (torch brings its own): the replays run the kernels of the
eager evaluation, so their span is of its size.  (125 us eager and 115 us
replayed on this cluster; a pair that the replays do not record reads the
4 us between two host calls.)"""
import pytest

from libecp_amd import native
from libecp_amd.workloads import medium_cluster


@pytest.mark.gpu
def test_replayed_span_is_of_the_eager_size():
    b = native.Batch([medium_cluster(0)])
    try:
        b.set_param("fuse", 1)
        b.execute(1)
        eager = b.quadrature_ms()
        b.execute(20)
        assert b.quadrature_samples == 1
        replayed = b.quadrature_ms()
        assert b.quadrature_samples == 8
        assert 0.2 * eager < replayed < 2.0 * eager
    finally:
        b.close()
