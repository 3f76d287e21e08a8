"""Models with zeta in {1, 2, 4, 8, 16} and lambda = +-1 (the pair kernels of powers.hpp) against the oracle:
one to three species, one to four exponents, single levels and all of them, segments of one entry, even and odd
segment lengths, more than 64 entries per centre, open clusters, small cells with repeated images.  FP64:
descriptors, energies and forces within 1e-10 relative, the bound of the other parity tests; mixed
form: 1 meV/atom and 20 meV/A, the precision form's bounds."""
import numpy as np
import pytest

from atomnn_amd import synth
from atomnn_amd.nnp import NNP, NNP_FORCE, NNP_PREC_MIXED, NNP_VACUUM_ENERGY
import oracle_binding as ob

pytestmark = pytest.mark.gpu
TOL = 1e-10

MODELS = [dict(species="A", etas=[0.02], zetas=[16.0]),
          dict(species="AB", etas=[0.005, 0.05], zetas=[1.0, 2.0, 4.0, 16.0]),
          dict(species="AB", etas=[0.001, 0.01, 0.05], zetas=[8.0, 1.0]),
          dict(species="ABC", etas=[0.001, 0.005, 0.02, 0.05], zetas=[2.0, 16.0]),
          dict(species="ABC", etas=[0.01, 0.05], zetas=[8.0], lambdas=[-1])]


def model_path(tmp_path, species, etas, zetas, lambdas=(1, -1)):
    rng = np.random.default_rng(len(etas) * 10 + len(species))
    pot = synth.make_potential(list(species), 6.0, 4, list(etas), list(zetas), list(lambdas), [16, 16], rng)
    cell = synth.cubic_cell(96, 0.05)
    s = synth.Structure(rng.integers(0, len(species), 96).astype(np.int32), synth.random_positions(96, cell, 1.8, 3), cell)
    path = str(tmp_path / "p.ann")
    synth.precondition(pot, s).write(path)
    return path


def structures(nsp):
    rng = np.random.default_rng(77)
    out = []
    for n, rho, dmin, cluster in ((1, 0.05, 1.5, False), (2, 0.05, 1.5, False), (9, 0.05, 1.5, False),
                                  (40, 0.05, 1.5, True), (3, 0.01, 1.5, True), (70, 0.11, 1.3, False),
                                  (300, 0.05, 1.8, False), (280, 0.1, 1.3, False)):
        cell = synth.strained_cell(n, rho, 0.05, rng)
        types = rng.integers(0, nsp, n).astype(np.int32)
        if n == 9:
            types[:] = 0
            types[-1] = nsp - 1
        out.append(synth.Structure(types, synth.random_positions(n, cell, dmin, 500 + n), None if cluster else cell))
    return out


@pytest.mark.parametrize("k", range(len(MODELS)))
def test_against_the_oracle(tmp_path, k):
    path = model_path(tmp_path, **MODELS[k])
    m, o = NNP.read(path), ob.OracleModel(path)
    for s in structures(len(MODELS[k]["species"])):
        Go, G = o.symm(s.types, s.pos, s.cell), m.symm(s)
        assert np.abs(G - Go[:, :G.shape[1]]).max() <= TOL * max(np.abs(Go).max(), 1e-300)
        Eo, Eao, Fo = o.compute(s.types, s.pos, s.cell)
        E, Ea, F = m.compute(s, NNP_FORCE | NNP_VACUUM_ENERGY)
        assert abs(E - Eo) <= TOL * max(abs(Eo), np.abs(Eao).sum())
        if s.natoms > 1:  # one atom and its images: the forces cancel to zero
            assert np.abs(F - Fo).max() <= TOL * np.abs(Fo).max()
        Em, _, Fm = m.compute(s, NNP_FORCE | NNP_VACUUM_ENERGY | NNP_PREC_MIXED)
        assert abs(Em - Eo) / s.natoms <= 1e-3
        assert np.sqrt(((Fm - Fo) ** 2).mean()) <= 20e-3
    m.close()
