"""The closure network's batch kernels (forward path 0, loss_grad) on values
that are not finite: relu is max(z, 0) with the number where z is a NaN, so a
row with a NaN feature has no hidden activity, a hidden unit with a NaN weight
has none in any row, and the other rows and units are not touched.  Bounds:
exact where two networks do the same sums, else those of the oracle comparison
(BF16 rounding of activations and gradients)."""
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


def reference(p, t):
    """mo.loss_grad with np.fmax as relu; also the outputs."""
    W1, W2, b2, W3, b3 = mo.unpack(p)
    r = lambda a: mo.bf16(a).astype(np.float64)     # noqa: E731
    t = np.asarray(t, np.float64)
    with np.errstate(invalid="ignore", over="ignore"):
        X, W1r, W2r, W3r = r(mo._inputs(t[:, :mo.NF])), r(W1), r(W2), r(W3)
        H1 = r(np.fmax(X @ W1r.T, 0.0).astype(np.float32))
        H2 = r(np.fmax(H1 @ W2r.T + b2.astype(np.float64), 0.0).astype(np.float32))
        Y = H2 @ W3r.T + b3.astype(np.float64)
        d = Y - t[:, mo.NF:]
        dY = r(2.0 * d / t.shape[0])
        g = np.zeros(mo.NPARAM)
        g[mo.OFF_W3:mo.OFF_B3] = (dY.T @ H2).reshape(-1)
        g[mo.OFF_B3:] = dY.sum(axis=0)
        dZ2 = r(np.where(H2 > 0, dY @ W3r, 0.0))
        g[mo.OFF_W2:mo.OFF_B2] = (dZ2.T @ H1).reshape(-1)
        g[mo.OFF_B2:mo.OFF_W3] = dZ2.sum(axis=0)
        dZ1 = r(np.where(H1 > 0, dZ2 @ W2r, 0.0))
        g[mo.OFF_W1:mo.OFF_W2] = (dZ1.T @ X).reshape(-1)
    return Y, float(np.sum(d * d) / t.shape[0]), g


@pytest.mark.parametrize("n", [5, 32, 47])
def test_forward_rows(n):
    p, x = params(5), rows(n, n)[:, :mo.NF].copy()
    quiet = p.copy()
    quiet[mo.OFF_W1:mo.OFF_W2] = 0.0
    m, q = Mlp(0), Mlp(0)
    m.set_params(p)
    q.set_params(quiet)
    clean = m.forward(x, 0)
    bad = x.copy()
    bad[1, 4] = np.nan
    bad[3, 0] = -np.nan
    bad[4, 7] = np.inf
    y, still = m.forward(bad, 0), q.forward(x, 0)
    for i in range(n):
        if i in (1, 3):
            assert np.array_equal(y[i], still[i]), i
        elif i != 4:
            assert np.array_equal(y[i], clean[i]), i
    ref = reference(p, np.concatenate([bad, np.zeros((n, mo.NO), np.float32)], axis=1))[0][4]
    assert np.array_equal(np.isnan(y[4]), np.isnan(ref))
    assert np.array_equal(np.isinf(y[4]), np.isinf(ref))
    m.close()
    q.close()


@pytest.mark.parametrize("n", [17, 32, 1041])
@pytest.mark.parametrize("where", ["row", "weight", "bias"])
def test_gradients(where, n):
    p, t = params(6), rows(n, n)
    if where == "row":
        t[2, 3] = np.nan                # that feature's column of dW1 is a NaN, nothing else
    elif where == "weight":
        p[mo.OFF_W1 + 5 * mo.K1 + 1] = np.nan
    else:
        p[mo.OFF_B2 + 7] = np.nan
        p[mo.OFF_B2 + 40] = -np.nan
    m = Mlp(0)
    m.set_params(p)
    loss, g = m.loss_grad(t)
    _, lref, gref = reference(p, t)
    assert abs(loss - lref) <= 1e-4 * abs(lref)
    assert np.array_equal(np.isnan(g), np.isnan(gref))
    ok = ~np.isnan(gref)
    for a, b in ((mo.OFF_W1, mo.OFF_W2), (mo.OFF_W2, mo.OFF_B2), (mo.OFF_B2, mo.OFF_W3), (mo.OFF_W3, mo.OFF_B3),
                 (mo.OFF_B3, mo.NPARAM)):
        k = np.arange(a, b)[ok[a:b]]
        if k.size:
            e = np.linalg.norm(g[k] - gref[k]) / max(np.linalg.norm(gref[k]), 1e-30)
            assert e <= 2e-2, (where, n, a, e)
    m.close()
