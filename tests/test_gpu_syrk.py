"""Pi(u) products (k_syrk_f64) through brpa_thc_piu with a grid point per (a, i), so
that R is any given matrix: orders around its 16 x 16 blocks, 32 x 32 quadrants and
64 x 64 tiles, row counts around its 16-row stages, even and odd orders (16- and
4-byte loads), frequency counts around the group of four, and launches small and
large enough for either of its two forms.

Tolerance: a sum of K rounded products, (K + 4) u sum |c R R|."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _check(ctx, k, n, nf, which):
    rng = np.random.default_rng(1000 * k + 10 * n + nf)
    R = rng.standard_normal((k, n))
    evir, freqs = np.sort(rng.uniform(0.1, 3.0, k)), rng.uniform(0.05, 4.0, nf)
    Pi, R2 = ctx.thc_piu(np.eye(k), np.ones((1, k)), np.ascontiguousarray(R.T),
                         np.array([-0.4]), evir, freqs, want_R=True)
    assert np.array_equal(R2, R)
    d = evir + 0.4
    for w in which:
        c = 4.0 * (d / (d * d + freqs[w] ** 2))
        ref = R.T @ (c[:, None] * R)
        tol = (k + 4) * 2.0 ** -53 * (np.abs(R).T @ (c[:, None] * np.abs(R)))
        assert np.all(np.abs(Pi[w] - ref) <= tol), (k, n, nf, w)
        assert np.array_equal(Pi[w], Pi[w].T)


@pytest.mark.parametrize("n", [1, 2, 15, 16, 17, 32, 33, 63, 64, 65, 66, 127, 130, 200])
@pytest.mark.parametrize("k", [1, 15, 16, 17, 33, 48, 79, 130])
def test_quad_form(ctx, k, n):
    nf = 1 + (k + n) % 6
    _check(ctx, k, n, nf, range(nf))


@pytest.mark.parametrize("k,n,nf", [(1, 3, 4096), (16, 64, 2048), (17, 33, 2047), (31, 66, 677),
                                    (48, 65, 678), (80, 129, 338), (65, 128, 679)])
def test_four_frequency_form(ctx, k, n, nf):
    _check(ctx, k, n, nf, (0, 1, 2, 3, nf // 2, nf - 2, nf - 1))
