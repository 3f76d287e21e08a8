"""The per-centre sums over neighbour entries as matrix products: segments of every length around the four-entry
steps and beyond the registers' 128 entries, more radial functions than one and two operand tiles hold, one to four
angular widths, species counts on both sides of the 16 moment columns; per-atom energies and forces against the oracle
at the FP64 parity bar (1e-10 of the largest component)."""
import numpy as np
import pytest

from atomnn_amd import synth
from atomnn_amd.nnp import NNP, NNP_FORCE, NNP_VACUUM_ENERGY
import oracle_binding as ob

pytestmark = pytest.mark.gpu


def cluster(counts, seed):
    """counts[s] atoms of species s within one cutoff of one another: a segment of every length up to the largest."""
    n = sum(counts)
    types = np.concatenate([np.full(c, s, dtype=np.int32) for s, c in enumerate(counts)])
    rng = np.random.default_rng(seed)
    side = max(4.5, 1.25 * n ** (1 / 3))
    pos = []
    while len(pos) < n:
        p = rng.uniform(0, side, 3)
        if all(np.sum((p - q) ** 2) > 0.8 for q in pos):
            pos.append(p)
    return synth.Structure(types, np.array(pos), None)


@pytest.mark.parametrize("species,n_radial,etas,zetas", [(2, 8, [0.02], [1.0]), (2, 17, [0.02, 0.1], [1.0, 2.0]),
                                                         (3, 33, [0.02], [4.0]), (3, 5, [0.01, 0.05, 0.2, 0.4], [1.0]),
                                                         (1, 16, [0.02], [2.0, 4.0]), (6, 4, [0.02, 0.1], [1.0])])
def test_segment_lengths(tmp_path, species, n_radial, etas, zetas):
    rng = np.random.default_rng(9)
    names = ["A", "B", "C", "D", "E", "F"][:species]
    pot = synth.make_potential(names, 6.0, n_radial, etas, zetas, [1, -1], [12], rng)
    path = str(tmp_path / "p.ann")
    pot.write(path)
    m, o = NNP.read(path), ob.OracleModel(path)
    sizes = [[1], [2], [1, 1], [4, 1], [5, 2], [6, 16], [17, 3], [18, 16], [2, 3, 4]]
    if species <= 3:
        sizes += [[150], [70, 75]]  # rows of more than 128 entries
    for k, c in enumerate(sizes):
        c = (c + [0] * species)[:species] if len(c) <= species else [sum(c)]
        s = cluster(c, 30 + k)
        E, Ea, F = m.compute(s, NNP_FORCE | NNP_VACUUM_ENERGY)
        Eo, Eao, Fo = o.compute(s.types, s.pos, s.cell)
        assert np.abs(Ea - Eao).max() <= 1e-10 * max(1.0, np.abs(Eao).max()), c
        assert np.abs(F - Fo).max() <= 1e-10 * max(1.0, np.abs(Fo).max()), c
    m.close()
