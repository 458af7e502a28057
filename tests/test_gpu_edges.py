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
from libecp_amd.workloads import batch_molecule, build_molecule, high_l, plain_small

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


def _batch_outputs(mols, n, tune=None):
    """Matrices (n = 0) or contracted gradients, and the parameters seen."""
    b = native.Batch(mols, n=n)
    try:
        params = {k: b.get_param(k) for k in ("fuse", "fb2_split", "t1_tail_grid")}
        for k, v in (tune or {}).items():
            b.set_param(k, v)
        b.execute(3)
        if n == 0:
            b.fetch()
            out = [b.matrix(i) for i in range(len(mols))]
        else:
            rng = np.random.default_rng(1)
            out = b.contract([rng.standard_normal((m.nao, m.nao)) for m in mols])[1]
        return params, out
    finally:
        b.close()


def _flat(out):
    return np.concatenate([np.ravel(np.asarray(x, dtype=float)) for o in out
                           for x in (o if isinstance(o, (tuple, list)) else [o])])


def test_failed_blocks_are_zero_in_a_used_context():
    """A molecule with a failed integration contracts to the same energy and
    code in fresh memory and where another job's blocks were."""
    bad, other = high_l(1003), high_l(1000)
    P = {id(m): [np.random.default_rng(3).standard_normal((m.nao, m.nao))] for m in (bad, other)}

    def energy(m):
        b = native.Batch([m])
        try:
            b.execute(1)
            codes, out, _ = b.contract(P[id(m)])
            return int(codes[0]), out[0]
        finally:
            b.close()

    was = native.cache_enable(False)
    try:
        fresh = energy(bad)
        native.cache_enable(True)
        energy(other)
        used = energy(bad)
    finally:
        native.cache_clear()
        native.cache_enable(was)
    assert fresh[0] != 0
    assert used == fresh


def test_results_before_an_evaluation():
    """A batch that takes another one's context reads zeros until its first
    evaluation."""
    native.cache_clear()
    for m in (plain_small(4), plain_small(3)):
        b = native.Batch([m])
        try:
            b.fetch()
            rc, I = b.matrix(0)
            assert rc == 0 and not I.any()
            b.execute(1)
            b.fetch()
            rc, I = b.matrix(0)
            assert rc == 0 and I.any()
        finally:
            b.close()


def test_batch_in_a_used_context():
    """Batches of rising and falling sizes and both orders in contexts that
    earlier batches of the same tables left (tuned, with their own graphs)
    give the bits and see the parameters of batches in fresh contexts."""
    small, many = [plain_small(3)], [plain_small(i) for i in range(4, 10)]
    seq = [(small, 0), (many, 0), (many[:2], 1), (small, 0), (many, 1), (many[:3], 0)]
    was = native.cache_enable(False)
    try:
        fresh = [_batch_outputs(m, n) for m, n in seq]
        native.cache_enable(True)
        for _ in range(2):
            for (m, n), (params, out) in zip(seq, fresh):
                p, o = _batch_outputs(m, n, {"fuse": 0, "fb2_split": 2, "t1_tail_grid": 512})
                assert p == params
                assert np.array_equal(_flat(o), _flat(out))
    finally:
        native.cache_clear()
        native.cache_enable(was)


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


def _pile(mols, n):
    b = native.Batch(mols, n=n)
    try:
        b.execute(3)
        if n == 0:
            b.fetch()
            return [_flat([b.matrix(i)]) for i in range(len(mols))], b.triplets()[1]
        P = [np.random.default_rng(4).standard_normal((m.nao, m.nao)) for m in mols]
        return [_flat([g]) for g in b.contract(P)[1]], b.triplets()[1]
    finally:
        b.close()


@pytest.mark.parametrize("n", [0, 1])
@pytest.mark.parametrize("name", ["s_to_f", "s_to_g", "few"])
def test_small_job_equals_large_one(name, n):
    """A molecule alone (the type-2 shapes of small jobs) and in a batch of
    copies too large for them: the same bits."""
    m = {"s_to_f": lambda: batch_molecule(np.random.default_rng(6), 17 if n == 0 else 9),
         "s_to_g": lambda: high_l(1000, nat=8 if n == 0 else 5, n_ecp=2, box=9.0),
         "few": entries_few}[name]()
    alone, nt = _pile([m], n)
    assert 0 < nt <= 4096
    copies, many = _pile([m] * (8192 // nt + 1), n)
    assert many > 4096
    for c in copies:
        assert np.array_equal(c, alone[0])
