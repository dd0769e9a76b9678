"""The closure network's batch kernels at the edges of their row blocks: 32
rows a wave, ranges of 16 rows that end inside one, batches just over the size
from which the gradients are split, and a small batch after a large one (the
buffers then hold older rows past its end).  Bounds: those of the oracle
comparison at one size (BF16 rounding of activations and gradients)."""
import sys
from pathlib import Path

import numpy as np
import pytest

sys.path.insert(0, str(Path(__file__).resolve().parents[1] / "oracle"))
import mlp_oracle as mo  # noqa: E402
from pennant_amd.closure import Mlp  # noqa: E402

pytestmark = pytest.mark.gpu


def params(seed):
    rng = np.random.default_rng(seed)
    p = rng.normal(0, 0.25, mo.NPARAM).astype(np.float32)
    p[mo.OFF_W1:mo.OFF_W2].reshape(mo.NH, mo.K1)[:, mo.NF + 1:] = 0.0
    return p


def rows(seed, n):
    rng = np.random.default_rng(seed)
    return np.concatenate([rng.normal(0, 1, (n, mo.NF)), rng.uniform(0, 2, (n, mo.NO))], axis=1).astype(np.float32)


def test_gradients_at_row_edges():
    m = Mlp(0)
    p = params(5)
    m.set_params(p)
    for n in (8209, 1041, 1025, 1024, 33, 32, 31, 17, 1):
        t = rows(n, n)
        loss, g = m.loss_grad(t)
        lref, gref = mo.loss_grad(p, t, rounding=True)
        assert abs(loss - lref) <= 1e-4 * abs(lref), n
        for name, a, b in (("W1", mo.OFF_W1, mo.OFF_W2), ("W2", mo.OFF_W2, mo.OFF_B2), ("b2", mo.OFF_B2, mo.OFF_W3),
                           ("W3", mo.OFF_W3, mo.OFF_B3), ("b3", mo.OFF_B3, mo.NPARAM)):
            e = np.linalg.norm(g[a:b] - gref[a:b]) / max(np.linalg.norm(gref[a:b]), 1e-30)
            assert e <= 2e-2, (n, name, e)
        assert np.all(g[mo.OFF_W1:mo.OFF_W2].reshape(mo.NH, mo.K1)[:, mo.NF + 1:] == 0.0), n
    m.close()


def test_inference_and_copies_after_training():
    """The BF16 copies that an Adam step writes are those of the parameters:
    both inference paths after training equal those of a network that is given
    the trained parameters, bit for bit, at sizes around a wave's rows."""
    m = Mlp(2)
    m.train(rows(1, 700), steps=5, batch=333, lr=2e-3, seed=3)
    fresh = Mlp(9)
    fresh.set_params(m.get_params())
    for n in (1, 31, 32, 33, 300):
        x = rows(40 + n, n)[:, :mo.NF].copy()
        for path in (0, 1):
            assert np.array_equal(m.forward(x, path), fresh.forward(x, path)), (n, path)
    m.close()
    fresh.close()
