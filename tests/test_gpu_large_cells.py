"""Structures beyond the bitmap search (262,144 atoms: kept candidates are sorted instead) and beyond the 16-bit keys of the
rows (2,031,616 atoms: neighbours 65,536 indices apart, here four grid planes and both within reach of the centre between
them, share a key and a stretch of the index table).  A periodic repetition of a 4096-atom cell has that cell's energies and
forces atom by atom; the cell itself is checked against the oracle.  Tolerance 1e-10 of the largest: positions of up to
350 A carry 3e-14 A, a relative 1e-13 of forces that change over 0.3 A.  The gather must find every reaction
(no second assembly)."""
import numpy as np
import pytest

from atomnn_amd import synth
from atomnn_amd.nnp import NNP, NNP_ALL_IMAGES, NNP_FORCE, NNP_VACUUM_ENERGY
import oracle_binding as ob

pytestmark = pytest.mark.gpu
A, K, TOL = 2.72, 16, 1e-10
FLAGS = NNP_FORCE | NNP_VACUUM_ENERGY


def repeated(reps):
    """A jittered K^3 grid repeated reps times along x, y, z, in raster order; and each atom's index in the base cell."""
    rng = np.random.default_rng(23)
    jitter, types = rng.uniform(-0.4, 0.4, (K, K, K, 3)), rng.integers(0, 2, (K, K, K)).astype(np.int32)
    ax = [np.arange(K * r) for r in reps]
    g = np.stack(np.meshgrid(*ax, indexing="ij"), -1)
    b = g % K
    base = (b[..., 0] * K + b[..., 1]) * K + b[..., 2]
    pos = A * g + jitter[b[..., 0], b[..., 1], b[..., 2]]
    s = synth.Structure(types.reshape(-1)[base].reshape(-1), np.ascontiguousarray(pos.reshape(-1, 3)),
                        np.diag(A * K * np.array(reps, dtype=float)))
    return s, base.reshape(-1)


@pytest.fixture(scope="module")
def cell(potentials):
    m = NNP.read(potentials["plain4096"])
    s, _ = repeated((1, 1, 1))
    _, Ea, F = m.compute(s, FLAGS)
    _, Eao, Fo = ob.OracleModel(potentials["plain4096"]).compute(s.types, s.pos, s.cell)
    assert np.abs(Ea - Eao).max() <= TOL * np.abs(Eao).max() and np.abs(F - Fo).max() <= TOL * np.abs(Fo).max()
    yield m, s, Ea, F
    m.close()


@pytest.mark.parametrize("reps,atoms", [((4, 4, 4), 262144), ((4, 4, 5), 327680), ((8, 8, 8), 2097152)])
def test_repeated_cell(cell, reps, atoms):
    m, s0, Ea0, F0 = cell
    s, base = repeated(reps)
    assert s.natoms == atoms
    for flags in (FLAGS, FLAGS | NNP_ALL_IMAGES):
        E, Ea, F = m.compute(s, flags)
        info = m.info()
        assert info["reactions_missed"] == 0 and info["assemble_mode"] == 0
        assert np.abs(Ea - Ea0[base]).max() <= TOL * np.abs(Ea0).max()
        assert np.abs(F - F0[base]).max() <= TOL * np.abs(F0).max()
    if atoms == 327680:  # the sort search over a batch
        (_, ea, f), (_, ea0, f0) = m.compute_batch([s, s0], FLAGS)
        assert np.array_equal(ea, Ea) and np.array_equal(ea0, Ea0) and np.array_equal(f0, F0)
        assert m.info()["reactions_missed"] == 0 and np.abs(f - F0[base]).max() <= TOL * np.abs(F0).max()
