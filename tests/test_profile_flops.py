"""Algorithmic FLOPs of the large-grid fallbacks in libecp_batch_profile: one
term per (triplet, channel) with failed entries and per primitive pair, plus
one per failed entry, whatever order a triplet's waves list their entries in.
Alone, a molecule's type-2 passes are split over several waves per triplet;
in a batch of copies that fills the chip, one wave takes a triplet's passes
in turn.  Every term is an integer, so k copies count exactly k times."""
import numpy as np
import pytest

from libecp_amd import native
from libecp_amd.workloads import batch_molecule, high_l

pytestmark = pytest.mark.gpu

MOLECULES = {"f_shells": lambda: batch_molecule(np.random.default_rng(6), 17),
             "g_shells": lambda: high_l(1000, nat=8, n_ecp=2, box=9.0)}


def fallback_flops(mols):
    b = native.Batch(mols)
    try:
        b.execute(1)
        p = b.profile()
        return p["fallback1"][2], p["fallback2"][2], b.triplets()[1]
    finally:
        b.close()


@pytest.mark.parametrize("name", sorted(MOLECULES))
def test_fallback_flops_do_not_depend_on_the_split(name):
    m = MOLECULES[name]()
    f1, f2, nt = fallback_flops([m])
    assert f1 > 0 and f2 > 0
    for _ in range(5):
        assert fallback_flops([m])[:2] == (f1, f2)
    k = 50000 // nt + 1
    assert fallback_flops([m] * k)[:2] == (k * f1, k * f2)
