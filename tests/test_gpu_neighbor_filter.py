"""The cell-list search's candidate filter against the oracle's neighbour lists: cells whose heights
are at, just above and well above twice the cutoff (with the filter and without it), one to five bins
along an axis (wrapped and unwrapped runs of bins), empty bins, atoms on cell faces and outside the
cell, rows beyond the register batches, batches binned by one workgroup and by several, and a mixed batch.
Counts, order, indices and min flags are equal; displacements agree to 1e-11 A, the bound of the
other neighbour-list tests (positions of some 50 A at 1e-16 relative through a few products)."""
import numpy as np
import pytest

from atomnn_amd import synth
from atomnn_amd.nnp import NNP, NNP_FORCE
import oracle_binding as ob

pytestmark = pytest.mark.gpu
RC = 6.0


@pytest.fixture(scope="module")
def model(potentials):
    m = NNP.read(potentials["plain4096"])
    assert m.rc == RC
    yield m
    m.close()


def check(m, s):
    got, ref = m.neighbors(s), ob.neighbors(s.types, s.pos, s.cell, RC)
    np.testing.assert_array_equal(got["counts"], ref["counts"])
    np.testing.assert_array_equal(got["index"], ref["index"])
    np.testing.assert_array_equal(got["min"], ref["min"])
    np.testing.assert_allclose(got["r"], ref["r"], rtol=0, atol=1e-11)
    np.testing.assert_allclose(got["d"], ref["d"], rtol=0, atol=1e-11)


def structure(n, cell, seed, dmin=1.0, spread=0):
    rng = np.random.default_rng(seed)
    pos = synth.random_positions(n, cell, dmin, seed + 1)
    if spread:  # the same atoms, some in other images of the cell
        pos = pos + rng.integers(-spread, spread + 1, size=(n, 3)) @ cell
    return synth.Structure(rng.integers(0, 2, n).astype(np.int32), pos, cell)


@pytest.mark.parametrize("heights", [(12.0 + 1e-9, 12.001, 12.01), (12.5, 17.9, 18.1), (23.9, 24.1, 30.5),
                                     (13.0, 25.0, 60.0)])
@pytest.mark.parametrize("shear", [0.0, 0.3])
def test_bins_and_heights(model, heights, shear):
    cell = np.diag(heights)
    cell[1, 0] += shear * heights[0]  # heights stay: the added part is along the first vector
    cell[2, 1] += shear * heights[1]
    n = max(256, int(0.03 * np.prod(heights)))
    check(model, structure(n, cell, 11, spread=1))


def test_atoms_on_faces_and_empty_bins(model):
    rng = np.random.default_rng(5)
    L = 36.0
    pos = synth.random_positions(300, np.diag([L, 14.0, 9.0]), 1.0, 6)  # a slab: most bins empty
    pos[:20] = np.round(pos[:20] / 6.0) * 6.0 + rng.normal(0, 1e-13, (20, 3))
    pos = pos[np.unique(np.round(pos, 6), axis=0, return_index=True)[1]]
    check(model, synth.Structure(rng.integers(0, 2, len(pos)).astype(np.int32), pos, np.eye(3) * L))


@pytest.mark.parametrize("n,L", [(600, 13.0), (1500, 17.0), (2200, 22.0)])  # 247, 276 and 187 mean neighbours
def test_rows_beyond_the_register_batches(model, n, L):
    check(model, structure(n, np.eye(3) * L, 21, dmin=0.5))


def test_dense_spot_in_a_thin_cell(model):
    """Mean density below the filter's row bound, but more than 128 entries around a dense spot."""
    rng = np.random.default_rng(8)
    cell = np.eye(3) * 40.0
    pos = np.concatenate([synth.random_positions(1500, cell, 1.0, 9), 20.0 + rng.normal(0.0, 2.2, (150, 3))])
    check(model, synth.Structure(rng.integers(0, 2, len(pos)).astype(np.int32), pos, cell))


@pytest.mark.parametrize("n", [256, 1024, 1025, 4096, 4097, 8193, 12001])
def test_binning_by_one_and_by_several_workgroups(model, n):
    check(model, structure(n, synth.cubic_cell(n, 0.04), 31, dmin=1.5))


@pytest.mark.parametrize("sizes", [(700, 40, 300, 257, 8), (4096, 40, 3000, 257, 2000, 8)])
def test_mixed_batch(model, sizes):
    """A batch of cell-list and all-pairs structures, binned by one and by several workgroups, equals its
    structures one by one."""
    strucs = [structure(n, synth.cubic_cell(n, 0.05), 40 + n, dmin=1.5) for n in sizes]
    for (e, ea, f), s in zip(model.compute_batch(strucs, NNP_FORCE), strucs):
        e1, ea1, f1 = model.compute(s, NNP_FORCE)
        np.testing.assert_array_equal(ea, ea1)
        np.testing.assert_array_equal(f, f1)
