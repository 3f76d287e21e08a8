"""An energy-training call gives the same errors, bit for bit, with and without the gradient, in one pass and in two and with
the rows in chunks: every kernel adds an output unit's inputs in one order.  Networks that the grouped kernel takes (one
and two tanh layers, widths that are not multiples of 16) and others (three layers, 65 units), six parameter vectors each (a sum
in another order differs in the last place of some)."""
import numpy as np
import pytest

from atomnn_amd import synth
from atomnn_amd.nnp import NNP, Train, LOSS_HUBER, LOSS_MSE

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_radial,hidden", [(2, [5]), (2, [33]), (28, [40, 24]), (36, [64, 64]), (50, [32, 32]),
                                             (2, [16, 16, 16]), (2, [65])])
def test_errors_do_not_depend_on_the_gradient(tmp_path, n_radial, hidden):
    rng = np.random.default_rng(5)
    pot = synth.make_potential(["A", "B"], 5.0, n_radial, [0.02], [1.0, 4.0], [1, -1], hidden, rng)
    path = str(tmp_path / "p.ann")
    pot.write(path)
    strucs = []
    for k, n in enumerate((32, 49, 65, 40, 3, 165, 700)):
        c = synth.cubic_cell(n, 0.05)
        strucs.append(synth.Structure(rng.integers(0, 2, n).astype(np.int32), synth.random_positions(n, c, 1.8, 7 + k), c))
    eref = np.array([rng.normal(-3.0, 0.3) * s.natoms for s in strucs])
    m = NNP.read(path)
    t = Train(m, strucs, eref)
    x0, batch = t.params(), list(range(len(strucs)))
    for k in range(6):
        x, b, loss = x0 + rng.normal(0, 0.02, t.nparams()), batch[k % 3:], (LOSS_MSE, LOSS_HUBER)[k % 2]
        e, _ = t.error(x, b, loss, 0.05, grad=False)
        for one_pass in (1, 0):
            m.set_option("train_one_pass", one_pass)
            assert np.array_equal(t.error(x, b, loss, 0.05)[0], e)
        m.set_option("train_chunk_elems", 1 << 16)
        assert np.array_equal(t.error(x, b, loss, 0.05)[0], e)
        m.set_option("train_chunk_elems", 1 << 28)
        m.set_option("train_one_pass", 1)
    t.close()
    m.close()
