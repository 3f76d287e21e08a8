"""Results that reach the caller through the kept page-locked buffers: descriptor tables around the bounds of the parts
they are copied in, at row strides below, at and above the descriptor count (exact); training batches of several
chunks of structures, kept and rebuilt, and calls that alternate between the two entry points and grow (the same
losses and gradients as single calls, within the rounding of the sums)."""
import ctypes

import numpy as np
import pytest

from atomnn_amd import synth
from atomnn_amd.nnp import NNP, Train, LOSS_MSE, _Pinned, lib
import oracle_binding as ob

pytestmark = pytest.mark.gpu


def structure(n, seed):
    rng = np.random.default_rng(seed)
    c = synth.cubic_cell(n, 0.05)
    return synth.Structure(synth.species_exact(n, [0.5, 0.5], rng), synth.random_positions(n, c, 1.8, seed), c)


@pytest.mark.parametrize("parts,extra", [(0, 1), (1, -1), (1, 0), (1, 1), (2, 0), (2, 1), (3, 7)])
def test_descriptor_parts(potentials, parts, extra):
    m = NNP.read(potentials["plain4096"])
    o = ob.OracleModel(potentials["plain4096"])
    nin = m.ninput(0)
    part = (512 << 10) // (8 * ((nin + 15) // 16 * 16))  # about; the sizes around it cover the true one
    s = structure(max(1, parts * part + extra), 3)
    G = m.symm(s)
    Go = o.symm(s.types, s.pos, s.cell)
    assert np.abs(G - Go).max() <= 1e-10 * max(1.0, np.abs(Go).max())
    for ldg in (1, nin - 1, nin + 5, nin + 64):
        out = np.full((s.natoms, ldg), np.nan)
        ps = _Pinned(s)
        assert lib().nnp_symm(m._h, ctypes.byref(ps.c_struct), out.ctypes.data, ldg) == 0
        w = min(ldg, nin)
        assert np.array_equal(out[:, :w], G[:, :w]) and np.all(out[:, w:] == 0)
    m.close()


@pytest.mark.parametrize("cache_atoms", [1 << 20, 0])
def test_training_chunks_and_alternating_calls(potentials, cache_atoms):
    strucs = [structure(4096, 1), structure(37, 2)]
    eref = np.array([-12000.0, -110.0])
    rng = np.random.default_rng(6)
    m = NNP.read(potentials["plain4096"])
    m.set_option("train_cache_atoms", cache_atoms)
    t = Train(m, strucs, eref)
    t.set_forces([rng.normal(0, 0.3, (s.natoms, 3)) for s in strucs])
    x = t.params()
    e1, g1 = t.error_force(x, [0], LOSS_MSE, 1.0, 2.0)
    a1, b1 = t.error(x, [0], LOSS_MSE)
    e2, g2 = t.error_force(x, [1], LOSS_MSE, 1.0, 2.0)
    k = 34  # chunks hold 128k atoms: 32 structures and 2
    for _ in range(2):
        e, g = t.error_force(x, [0] * k + [1], LOSS_MSE, 1.0, 2.0)
        assert np.allclose(e, k * e1 + e2, rtol=1e-11)
        assert np.abs(g - (k * g1 + g2)).max() <= 1e-10 * np.abs(g).max()
        a, b = t.error(x, [0] * k, LOSS_MSE)
        assert np.allclose(a, k * a1, rtol=1e-11)
        assert np.abs(b - k * b1).max() <= 1e-10 * np.abs(b).max()
        # smaller calls after the larger, other parameters, and without the gradient
        y = x + rng.normal(0, 0.02, x.size)
        ey, gy = t.error_force(y, [1], LOSS_MSE, 1.0, 2.0)
        ez, _ = t.error_force(y, [1], LOSS_MSE, 1.0, 2.0, grad=False)
        assert np.array_equal(ey, ez) and not np.array_equal(gy, g2)
        e1b, g1b = t.error_force(x, [0], LOSS_MSE, 1.0, 2.0)
        assert np.array_equal(e1, e1b) and np.array_equal(g1, g1b)
    t.close()
    m.close()
