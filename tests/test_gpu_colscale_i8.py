"""Column pass of the split-int8 form (k_colscale_i8, k_colscale_fin_i8): row
counts around its 512-row chunks, 128-row wave shares and 8-row steps, column
counts around 64, frequency counts around the group of 8.  A wrong column
maximum or diagonal moves E(u) by far more than the bar of the split form
(1e-7 Ha)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("o,v,n,nf", [(1, 1, 1, 1), (1, 7, 3, 9), (3, 43, 64, 8), (4, 32, 65, 7),
                                      (7, 73, 63, 17), (16, 32, 130, 16), (19, 27, 128, 24),
                                      (32, 33, 70, 12)])
def test_split_i8_energy_terms(ctx, o, v, n, nf):
    rng = np.random.default_rng(o * 1000 + v)
    R = rng.standard_normal((o * v, n)) * 0.3 * np.exp(-4.0 * np.arange(n) / n)
    R[rng.integers(0, o * v), rng.integers(0, n)] = 2.5   # a maximum of its own in one column
    eocc, evir = np.sort(rng.uniform(-1.5, -0.3, o)), np.geomspace(0.05, 3.0, v)
    t, w = np.polynomial.legendre.leggauss(nf)
    x, w = (1 + t) / (1 - t), 2 * w / (1 - t) ** 2
    d = (evir[None, :] - eocc[:, None]).ravel()
    e, eu = ctx.ecrpa(R, eocc, evir, x, w, precision="split_i8")
    for k in range(nf):
        p = R.T @ ((4 * d / (d * d + x[k] ** 2))[:, None] * R)
        ref = np.linalg.slogdet(np.eye(n) + p)[1] - np.trace(p)
        assert abs(eu[k] - ref) <= 1e-7, (k, eu[k], ref)
