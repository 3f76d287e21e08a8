"""The 32-atom mixed network kernel: hidden widths that are not multiples of 32 (operand columns past a layer read
as zero), growing and shrinking layers, one to three hidden layers, few and many inputs, tiles of 1, 31, 32
and 33 atoms of a species; per-atom energies and forces of the mixed form against the oracle in FP64 within the
form's bounds (1 meV/atom, 20 meV/A RMS), for networks with outputs of order 1 eV."""
import numpy as np
import pytest

from atomnn_amd import synth
from atomnn_amd.nnp import NNP, NNP_FORCE, NNP_PREC_MIXED, NNP_VACUUM_ENERGY
import oracle_binding as ob

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hidden", [[8], [48], [64], [16, 16], [64, 16], [16, 64], [40, 24], [16, 48, 16],
                                    [64, 16, 64], [48, 64, 32]])
@pytest.mark.parametrize("n_radial", [2, 20])
def test_against_the_oracle(tmp_path, hidden, n_radial):
    rng = np.random.default_rng(7)
    pot = synth.make_potential(["A", "B"], 6.0, n_radial, [0.02], [1.0, 4.0], [1, -1], hidden, rng)
    cell = synth.cubic_cell(96, 0.05)
    s = synth.Structure(synth.species_exact(96, [0.5, 0.5], rng), synth.random_positions(96, cell, 2.0, 3), cell)
    path = str(tmp_path / "p.ann")
    synth.precondition(pot, s).write(path)
    m, o = NNP.read(path), ob.OracleModel(path)
    strucs = []
    for na, nb in ((1, 31), (32, 33), (64, 2), (0, 40)):
        n = na + nb
        c = synth.cubic_cell(n, 0.05)
        types = np.array([0] * na + [1] * nb, dtype=np.int32)
        strucs.append(synth.Structure(types, synth.random_positions(n, c, 2.0, 60 + n), c))
    for q in strucs:
        E, Ea, F = m.compute(q, NNP_FORCE | NNP_VACUUM_ENERGY | NNP_PREC_MIXED)
        Eo, Eao, Fo = o.compute(q.types, q.pos, q.cell)
        assert np.abs(Ea - Eao).max() <= 1e-3
        assert np.sqrt(((F - Fo) ** 2).mean()) <= 20e-3
    m.close()
