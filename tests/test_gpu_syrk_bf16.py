"""Split-bf16 Pi product (k_split, k_syrk_bf16): row counts around its 32-row stages and
128-row scaled blocks, orders around its 128-column tiles and 16-column groups,
frequency counts around the split's groups of 8 and grids around the 256-tile rounds of
the XCD order.  The split form stays within its 1e-7 Ha of the host's FP64."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("o,v,n,nf", [(1, 1, 1, 1), (1, 5, 15, 3), (1, 31, 17, 9), (3, 43, 64, 8),
                                      (2, 64, 127, 7), (4, 32, 128, 4), (3, 43, 129, 3),
                                      (6, 64, 255, 17), (6, 43, 257, 43), (9, 71, 385, 27)])
def test_energy_terms(ctx, o, v, n, nf):
    rng = np.random.default_rng(o + v + n)
    R = rng.standard_normal((o * v, n)) * 0.3 * np.exp(-4.0 * np.arange(n) / n)
    R[rng.integers(0, o * v), rng.integers(0, n)] = 2.5   # a scale of its own in one column
    if n > 2:
        R[:, 2] = 0.0                                      # and a column without one
    eocc, evir = np.sort(rng.uniform(-1.5, -0.3, o)), np.geomspace(0.05, 3.0, v)
    t, w = np.polynomial.legendre.leggauss(nf)
    x, w = (1 + t) / (1 - t), 2 * w / (1 - t) ** 2
    d = (evir[None, :] - eocc[:, None]).ravel()
    e, eu = ctx.ecrpa(R, eocc, evir, x, w, precision="split_bf16")
    for k in range(nf):
        p = R.T @ ((4 * d / (d * d + x[k] ** 2))[:, None] * R)
        ref = np.linalg.slogdet(np.eye(n) + p)[1] - np.trace(p)
        assert abs(eu[k] - ref) <= 1e-7, (k, eu[k], ref)
