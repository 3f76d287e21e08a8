"""Energy-training rows of groups of tiles: one and two hidden layers, widths that are not multiples of 16 and both
sides of 32 and of 64 (the general kernel above), input counts of every operand size and one beyond, one pass with
the structures' own rows and two passes with species rows, groups of one tile, of an odd number and of many; losses
and gradients against the CPU oracle at the training tests' bar (1e-10 of the loss, and of the largest component)."""
import numpy as np
import pytest

from atomnn_amd import synth
from atomnn_amd.nnp import NNP, Train, LOSS_HUBER
import oracle_binding as ob

pytestmark = pytest.mark.gpu

TOL = 1e-10


def structures(sizes, rng):
    out = []
    for k, (na, nb) in enumerate(sizes):
        n = na + nb
        c = synth.cubic_cell(n, 0.05)
        out.append(synth.Structure(np.array([0] * na + [1] * nb, dtype=np.int32), synth.random_positions(n, c, 1.8, 7 + k), c))
    return out


# 2 n_radial + 12 inputs: 16 (one MFMA row tile), 68, 84, 112 and 132
@pytest.mark.parametrize("n_radial,hidden", [(2, [5]), (2, [32]), (2, [33]), (28, [32, 7]), (28, [40, 24]), (36, [64, 64]),
                                             (36, [17, 64]), (36, [20]), (50, [32, 32]), (50, [64]), (50, [64, 64]),
                                             (60, [16]), (2, [65]), (28, [16, 16, 16]), (2, [16, 16])])
@pytest.mark.parametrize("one_pass", [1, 0])
def test_against_the_oracle(tmp_path, n_radial, hidden, one_pass):
    rng = np.random.default_rng(5)
    pot = synth.make_potential(["A", "B"], 5.0, n_radial, [0.02], [1.0, 4.0], [1, -1], hidden, rng)
    path = str(tmp_path / "p.ann")
    pot.write(path)
    # tiles of one row, of 16 and 17, an odd count, a species missing
    strucs = structures([(1, 31), (33, 16), (48, 17), (0, 40), (3, 0), (90, 75)], rng)
    eref = np.array([rng.normal(-3.0, 0.3) * s.natoms for s in strucs])
    m = NNP.read(path)
    m.set_option("train_one_pass", one_pass)
    t = Train(m, strucs, eref)
    o = ob.OracleTrain(ob.OracleModel(path), strucs, eref)
    x = t.params() + rng.normal(0, 0.02, t.nparams())
    for batch in ([0, 1, 2, 3, 4, 5], [5], [4], [3, 0, 3]):
        e, g = t.error(x, batch, LOSS_HUBER, 0.05)
        eo, go = o.error(x, batch, LOSS_HUBER, 0.05)
        assert abs(e[0] - eo[0]) <= TOL * abs(eo[0])
        assert abs(e[1] - eo[1]) <= TOL * abs(eo[1])
        assert np.abs(g - go).max() <= TOL * np.abs(go).max()
    t.close()
    m.close()


@pytest.mark.parametrize("atoms,count", [(700, 13), (4096, 9)])
def test_groups_of_many_tiles_add_up(potentials, atoms, count):
    """More tiles than groups, ragged at the end of each structure's run: the batch's gradient is the sum of the
    structures' (which take groups of two tiles), within the rounding of sums of this length."""
    rng = np.random.default_rng(4)
    strucs = structures([(atoms // 3 + 5 * k, atoms - atoms // 3) for k in range(count)], rng)
    eref = np.array([rng.normal(-3.0, 0.3) * s.natoms for s in strucs])
    m = NNP.read(potentials["plain4096"])
    t = Train(m, strucs, eref)
    x = t.params()
    e, g = t.error(x, list(range(count)), LOSS_HUBER, 0.05)
    parts = [t.error(x, [b], LOSS_HUBER, 0.05) for b in range(count)]
    assert np.allclose(e, sum(p[0] for p in parts), rtol=1e-12)
    assert np.abs(g - sum(p[1] for p in parts)).max() <= 1e-11 * np.abs(g).max()
    t.close()
    m.close()
