"""Diagonal blocks of the blocked Cholesky (k_potrf_diag) through
brpa_ecrpa_analytic: orders around its 16-column panels and 64-column blocks,
matrices that are not positive definite at any place of a panel, and pivots
outside the range of the reciprocal estimate.

Tolerance of the log-det: a backward-stable factor solves A + dA with |dA| <=
N u |A|, and |tr(A^-1 dA)| <= N |A^-1| |dA|, so N^2 u cond(A); the spectra
below lie in [1, 6]."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _pi(n, seed):
    q, _ = np.linalg.qr(np.random.default_rng(seed).standard_normal((n, n)))
    p = (q * np.linspace(0.0, 5.0, n)) @ q.T
    return 0.5 * (p + p.T)


@pytest.mark.parametrize("n", [1, 2, 15, 16, 17, 31, 33, 48, 63, 64, 65, 79, 128, 200])
def test_log_det(ctx, n):
    pis = np.stack([_pi(n, 10 * n + k) for k in range(3)])
    _, eu = ctx.ecrpa_analytic(pis, np.ones(3), np.ones(3))
    for p, e in zip(pis, eu):
        ref = np.linalg.slogdet(np.eye(n) + p)[1] - np.trace(p)
        assert abs(e - ref) <= 6.0 * n * n * 2.0 ** -53 + 1e-15 * abs(ref), (n, e, ref)


@pytest.mark.parametrize("at", [0, 7, 15, 16, 40, 63, 64, 99])
def test_not_positive_definite(ctx, at):
    import brpa
    p = _pi(100, 3)
    p[at, at] = -2.0
    with pytest.raises(brpa.BrpaError) as e:
        ctx.ecrpa_analytic(p[None], np.ones(1), np.ones(1))
    assert e.value.code == 3
    # the same context factors the next matrix
    ctx.ecrpa_analytic(_pi(100, 4)[None], np.ones(1), np.ones(1))


@pytest.mark.parametrize("at", [0, 5, 16, 63, 70])
def test_large_pivot(ctx, at):
    """A pivot above 2^1000, with entries beside it that a factor has to carry."""
    p = _pi(80, 5)
    p[at, :] = p[:, at] = 1e150
    p[at, at] = 1e305
    _, eu = ctx.ecrpa_analytic(p[None], np.ones(1), np.ones(1))
    assert eu[0] == pytest.approx(-1e305, rel=1e-15)
