"""Training gradients whose rows go through a bounded buffer (option train_chunk_elems): energy rows tile by tile in
many chunks of a few tiles, with one partly filled, and force rows the same; against the CPU oracle at the training tests'
bar (1e-10 of the loss and of the largest component) and against the call with every row in one buffer (1e-11: the sums of
some 200 rows in another order).  The option also counts on a set that has seen the batch: then the result is that of a
new set under the same option, bit for bit."""
import numpy as np
import pytest

from atomnn_amd import synth
from atomnn_amd.nnp import NNP, Train, LOSS_HUBER
import oracle_binding as ob

pytestmark = pytest.mark.gpu

TOL = 1e-10
SMALL = 1 << 16


@pytest.fixture(scope="module")
def data(potentials):
    rng = np.random.default_rng(8)
    strucs = []
    for k, n in enumerate((1700, 900, 640, 7)):
        cell = synth.cubic_cell(n, 0.05)
        strucs.append(synth.Structure(rng.integers(0, 3, n).astype(np.int32), synth.random_positions(n, cell, 1.8, 90 + k), cell))
    eref = np.array([rng.normal(-3.0, 0.3) * s.natoms for s in strucs])
    path = potentials["mixed64x4096"]
    forces = [rng.normal(0.0, 0.5, (s.natoms, 3)) for s in strucs]
    o = ob.OracleTrain(ob.OracleModel(path), strucs, eref)
    m = NNP.read(path)
    t = Train(m, strucs, eref)
    x = t.params() + rng.normal(0, 0.02, t.nparams())
    # the small buffer holds fewer rows than groups of tiles (32 at most) could do with: tiles go in chunks
    rows = SMALL // max(t.nparams(k) for k in range(3))
    tiles = sum(-(-sum(int((s.types == k).sum()) for s in strucs) // 16) for k in range(3))
    assert 1 < rows < tiles / 32 and tiles % rows
    t.close()
    m.close()
    return path, strucs, eref, forces, x, o.error(x, [0, 1, 2, 3], LOSS_HUBER, 0.05)


def close(a, b, tol):
    return np.abs(np.asarray(a) - b).max() <= tol * np.abs(b).max()


@pytest.mark.parametrize("one_pass", [1, 0])
def test_energy_rows_in_chunks(data, one_pass):
    path, strucs, eref, _, x, (eo, go) = data
    m = NNP.read(path)
    m.set_option("train_one_pass", one_pass)
    t = Train(m, strucs, eref)
    batch = [0, 1, 2, 3]
    e0, g0 = t.error(x, batch, LOSS_HUBER, 0.05)  # every row in one buffer
    m.set_option("train_chunk_elems", SMALL)
    e1, g1 = t.error(x, batch, LOSS_HUBER, 0.05)
    fresh = Train(m, strucs, eref)
    e2, g2 = fresh.error(x, batch, LOSS_HUBER, 0.05)
    assert np.array_equal(e1, e2) and np.array_equal(g1, g2)
    assert not np.array_equal(g1, g0)  # summed in another order
    m.set_option("train_chunk_elems", 1 << 28)
    e3, g3 = t.error(x, batch, LOSS_HUBER, 0.05)
    assert np.array_equal(e0, e3) and np.array_equal(g0, g3)
    for e, g in ((e0, g0), (e1, g1)):
        assert abs(e[0] - eo[0]) <= TOL * abs(eo[0]) and abs(e[1] - eo[1]) <= TOL * abs(eo[1])
        assert close(g, go, TOL)
    assert close(g1, g0, 1e-11)
    fresh.close()
    t.close()
    m.close()


def test_force_rows_in_chunks(data):
    path, strucs, eref, forces, x, _ = data
    m = NNP.read(path)
    t = Train(m, strucs, eref)
    t.set_forces(forces)
    batch = [2, 0, 3]
    e0, g0 = t.error_force(x, batch, LOSS_HUBER, 0.05, beta=0.5)
    m.set_option("train_chunk_elems", SMALL)
    e1, g1 = t.error_force(x, batch, LOSS_HUBER, 0.05, beta=0.5)
    assert np.array_equal(e1, e0)
    assert not np.array_equal(g1, g0) and close(g1, g0, 1e-11)
    t.close()
    m.close()
