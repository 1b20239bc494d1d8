"""brpa_gpiug_mo in row chunks of the SYRK (k_syrk_f64, k_syrk_acc): row counts below, at
and above N and around the chunks' 16-row rounding, orders around the 64-column tiles, an
accumulator that is not symmetric, host and device memory.

Tolerance: sums of K products of entries |R| <= 5, each rounded a few times: 4 K u times
the sum of the magnitudes, plus the rounding of the accumulator."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("o,v,n", [(1, 1, 1), (1, 40, 41), (1, 41, 41), (4, 16, 64), (5, 51, 65),
                                   (4, 65, 63), (16, 33, 128), (7, 75, 129), (20, 83, 130), (3, 700, 257)])
def test_chunks(ctx, o, v, n):
    import torch
    rng = np.random.default_rng(o + v + n)
    R, P = rng.uniform(-5, 5, (o * v, n)), rng.standard_normal((n, n))
    eocc, evir = np.sort(rng.uniform(-1.5, -0.3, o)), np.geomspace(0.05, 3.0, v)
    d = (evir[None, :] - eocc[:, None]).ravel()
    c = 4.0 * d / (d * d + 0.7 ** 2)
    ref = P + R.T @ (c[:, None] * R)
    tol = 4 * (o * v + 4) * 2.0 ** -53 * (np.abs(P) + np.abs(R).T @ (c[:, None] * np.abs(R)))
    got = ctx.gpiug_mo(P.copy(), R, eocc, evir, 0.7, 4.0)
    assert np.all(np.abs(got - ref) <= tol)
    Pd = torch.from_numpy(P.copy()).cuda()
    ctx.gpiug_mo(Pd, torch.from_numpy(R).cuda(), eocc, evir, 0.7, 4.0)
    assert np.array_equal(Pd.cpu().numpy(), got)
