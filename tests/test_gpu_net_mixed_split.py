"""The mixed networks' split products are worth their name.  With x = hi + lo to BF16 each, an operand is kept to 2^-18 and
the product without lo times lo to 3 * 2^-18 = 1.1e-5, against 2 * 2^-9 = 3.9e-3 for single BF16 products: some 340 times.
On networks of one to three layers with outputs of order 1 eV, and the FP32 descriptors' 1e-6 beside it, that bounds
  per-atom energies   5e-5 eV  (four layers of 1.1e-5)
  forces              1e-4 of their rms  (forward and backward layers), rms
and the three products must be at least 20 times nearer to the oracle than one, in energies and in forces: losing a low part
in any layer, or reading another operand's columns, shows."""
import numpy as np
import pytest

from atomnn_amd import synth
from atomnn_amd.nnp import NNP, NNP_FORCE, NNP_PREC_MIXED, NNP_VACUUM_ENERGY
import oracle_binding as ob

pytestmark = pytest.mark.gpu


def rms(x):
    return float(np.sqrt(np.mean(np.square(x))))


@pytest.mark.parametrize("hidden", [[8], [48], [64], [16, 16], [64, 16], [16, 64], [40, 24], [16, 48, 16],
                                    [64, 16, 64], [48, 64, 32]])
@pytest.mark.parametrize("n_radial", [2, 20])
def test_split_products(tmp_path, hidden, n_radial):
    rng = np.random.default_rng(7)
    pot = synth.make_potential(["A", "B"], 6.0, n_radial, [0.02], [1.0, 4.0], [1, -1], hidden, rng)
    cell = synth.cubic_cell(200, 0.05)
    s = synth.Structure(synth.species_exact(200, [0.5, 0.5], rng), synth.random_positions(200, cell, 2.0, 3), cell)
    path = str(tmp_path / "p.ann")
    synth.precondition(pot, s).write(path)
    m = NNP.read(path)
    _, Eo, Fo = ob.OracleModel(path).compute(s.types, s.pos, s.cell)
    err = {}
    for terms in (3, 1):
        m.set_option("net_bf16_terms", terms)
        _, E, F = m.compute(s, NNP_FORCE | NNP_VACUUM_ENERGY | NNP_PREC_MIXED)
        err[terms] = rms(E - Eo), rms(F - Fo), np.abs(E - Eo).max()
    m.close()
    assert err[3][2] <= 5e-5 * max(1.0, np.abs(Eo).max())
    assert err[3][1] <= 1e-4 * rms(Fo)
    assert 20 * err[3][0] <= err[1][0] and 20 * err[3][1] <= err[1][1]
