"""Every value of the launch parameters that choose something gives the bits
of the defaults, out-of-range ones too: fewer than two head levels (the head
always takes levels 0 and 1), no tail, one workgroup a tail, any number of
shares of the type-2 fallback."""
import numpy as np
import pytest

from libecp_amd import native
from libecp_amd.workloads import batch_molecule

pytestmark = pytest.mark.gpu

VALUES = [("t1_head_coop", v) for v in (-3, 0, 1, 2, 3, 8, 14, 15, 40)] + \
         [("t1_tail_grid", v) for v in (0, 1, 7)] + \
         [("fb2_split", v) for v in (-1, 1, 2, 5, 8, 20)] + [("asm2_cache", v) for v in (0, 2)]


def _matrix(m, fuse, name=None, value=0):
    b = native.Batch([m])
    try:
        b.set_param("fuse", fuse)
        if name:
            b.set_param(name, value)
        b.execute(2)
        b.fetch()
        rc, I = b.matrix(0)
        assert rc == 0
        return I
    finally:
        b.close()


@pytest.mark.parametrize("fuse", [0, 1])
@pytest.mark.parametrize("name,value", VALUES)
def test_values_give_the_default_bits(fuse, name, value):
    m = batch_molecule(np.random.default_rng(6), 17)
    assert np.array_equal(_matrix(m, fuse, name, value), _matrix(m, 2))
