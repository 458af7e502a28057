"""Device kernels at the edges of their tiles, against the oracle.

Molecules and grids chosen for where the work split of a kernel changes:
a coarser and the finest large grid, contractions
of more than 64 primitive pairs, triplets with a handful and with hundreds of
type-2 entries.  The bar is that of the other parity tests: 1e-10 absolute +
1e-8 relative, widened by the reference algorithm's own rounding floor
(2 |ref - ref_fma|, the oracle compiled with FMA contraction).
"""
import ctypes as C
import os

import numpy as np
import pytest

import ecp_native as E
from libecp_amd import native
from libecp_amd.workloads import build_molecule, plain_small

pytestmark = pytest.mark.gpu


def pairs_81():
    """9-fold contractions: 81 primitive pairs a shell pair, s..d basis, L = 5."""
    return build_molecule(np.random.default_rng(5), nat=3, box=4.0, min_spacing=1.5, ecp_atoms=[1], L=5,
                          ecp_gauss=1, ecp_lmax_basis=2, other_lmax_basis=2, K=9, a_range=(0.02, 300.0))


def entries_5_to_643():
    """s..g basis with L = 5: from 5 to 643 type-2 entries a triplet."""
    return build_molecule(np.random.default_rng(8), nat=2, box=3.0, min_spacing=1.0, ecp_atoms=[0], L=5,
                          ecp_gauss=2, ecp_lmax_basis=4, other_lmax_basis=4, K=2, a_range=(0.2, 30.0))


def entries_few():
    """s and p basis with L = 2: a few type-2 entries a triplet."""
    return build_molecule(np.random.default_rng(9), nat=4, box=4.0, min_spacing=1.0, ecp_atoms=[2], L=2,
                          ecp_gauss=3, ecp_lmax_basis=0, other_lmax_basis=1, K=1, a_range=(0.1, 50.0))


CASES = {"grid_512": (lambda: plain_small(3), 512),
         "grid_2048": (lambda: plain_small(3), 2048), "pairs_81": (pairs_81, 1024),
         "entries_643": (entries_5_to_643, 1024), "entries_few": (entries_few, 1024)}


def _fma_blocks(m, grid):
    lib = C.CDLL(os.path.join(E.ROOT, "oracle", "liboracle_fma.so"))
    lib.orc_init.restype = C.c_void_p
    h = lib.orc_init(C.c_int(m.nat), *E._init_args(m), C.c_int(0), C.c_int(-1), None, C.c_int(grid),
                     C.c_double(1e-12), C.c_double(1e-14), C.c_int(1))
    col = E.Blocks(0)
    rc = lib.orc_calculate(C.c_void_p(h), col.cb, None)
    lib.orc_free(C.c_void_p(h))
    return rc, col


@pytest.mark.parametrize("name", sorted(CASES))
def test_tile_edges_against_oracle(name):
    make, grid = CASES[name]
    m = make()
    h = native.Handle(m, grid=grid)
    try:
        rc, keys, blocks = h.blocks()
    finally:
        h.close()
    rc2, col = E.oracle_blocks(m, grid=grid, options=1)
    _, fma = _fma_blocks(m, grid)
    assert rc == rc2
    assert keys == col.keys
    for k, a, b, f in zip(keys, blocks, col.blocks, fma.blocks):
        a, b, f = np.asarray(a), np.asarray(b), np.asarray(f)
        assert np.all(np.abs(a - b) <= 1e-10 + 1e-8 * np.abs(b) + 2 * np.abs(b - f)), \
            (k, float(np.abs(a - b).max()))


def _flat(out):
    return np.concatenate([np.ravel(np.asarray(x, dtype=float)) for o in out
                           for x in (o if isinstance(o, (tuple, list)) else [o])])


@pytest.mark.parametrize("n", [0, 1])
def test_contract_after_replays(n):
    """A contraction after graph replays gives the bits of one after a first
    evaluation."""
    m = [plain_small(3)]
    rng = np.random.default_rng(2)
    P = [rng.standard_normal((m[0].nao, m[0].nao))]
    outs = []
    for repeats in (1, 3):
        b = native.Batch(m, n=n)
        try:
            b.set_param("fuse", 1)
            b.execute(repeats)
            codes, out, _ = b.contract(P)
        finally:
            b.close()
        assert not codes.any()
        outs.append(_flat(out))
    assert np.array_equal(outs[0], outs[1])
