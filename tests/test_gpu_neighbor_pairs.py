"""The all-pairs search against the oracle's neighbour lists: cells of one to eight atoms whose images all fall on a few
atoms, skewed and flat ones, lattices with equally near images in exact arithmetic (the first one carries the min
flag), atom counts around a wavefront's 64 and a round's 256, open structures.  Counts, order, indices and min flags are
equal; displacements agree to 1e-11 A, the bound of the other neighbour-list tests.  All of them in one batch give the
energies and forces of the single calls, bit for bit."""
import numpy as np
import pytest

from atomnn_amd import synth
from atomnn_amd.nnp import NNP, NNP_FORCE, NNP_VACUUM_ENERGY
import oracle_binding as ob

pytestmark = pytest.mark.gpu
RC = 6.0


def structures():
    rng = np.random.default_rng(3)
    out = []
    for n in (1, 2, 3, 5, 8):  # random cells, skewed
        c = np.asarray(synth.strained_cell(n, 0.05, 0.2, rng)).reshape(3, 3)
        out.append((n, c, rng.uniform(0, 1, (n, 3)) @ c))
    for basis in ([[0, 0, 0]], [[0, 0, 0], [2, 2, 2]], [[0, 0, 0], [2, 2, 0], [2, 0, 2], [0, 2, 2]]):
        out.append((len(basis), 4.0 * np.eye(3), np.array(basis, dtype=float)))
    out.append((3, np.diag([2.0, 4.0, 32.0]), np.array([[0, 0, 0], [1.0, 2.0, 1.0], [0.5, 1.0, 16.0]])))  # flat
    for n in (31, 63, 64, 65, 128, 255, 256, 257, 300):
        c = np.asarray(synth.strained_cell(n, 0.05, 0.1, rng)).reshape(3, 3)
        out.append((n, c, rng.uniform(0, 1, (n, 3)) @ c))
    for n in (1, 2, 64, 65, 300):
        out.append((n, None, synth.random_positions(n, synth.cubic_cell(n, 0.06), 1.0, 500 + n)))
    return [synth.Structure(np.arange(n, dtype=np.int32) % 2, np.ascontiguousarray(p),
                            None if c is None else np.ascontiguousarray(c)) for n, c, p in out]


@pytest.fixture(scope="module")
def model(potentials):
    m = NNP.read(potentials["plain4096"])
    assert m.rc == RC
    yield m
    m.close()


@pytest.mark.parametrize("k", range(len(structures())))
def test_rows(model, k):
    s = structures()[k]
    got, ref = model.neighbors(s), ob.neighbors(s.types, s.pos, s.cell, RC)
    np.testing.assert_array_equal(got["counts"], ref["counts"])
    np.testing.assert_array_equal(got["index"], ref["index"])
    np.testing.assert_array_equal(got["min"], ref["min"])
    np.testing.assert_allclose(got["r"], ref["r"], rtol=0, atol=1e-11)
    np.testing.assert_allclose(got["d"], ref["d"], rtol=0, atol=1e-11)


def test_one_batch(model):
    strucs = structures()
    flags = NNP_FORCE | NNP_VACUUM_ENERGY
    for s, (Eb, Eab, Fb) in zip(strucs, model.compute_batch(strucs, flags)):
        E, Ea, F = model.compute(s, flags)
        assert np.array_equal(Ea, Eab) and np.array_equal(F, Fb) and np.all(np.isfinite(F))
