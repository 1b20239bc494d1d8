"""The blocked Cholesky's launches: one per 64-column step where few matrices are in
the launch (k_chol_step), three where there are many, and a call that changes from one
to the other at an outer panel of 256 columns; ranks of 64 to 192 of the left-looking
part and tiles of the rank-256 update (k_chol_rest) with odd and even orders, one past
and one short of their edges.

Tolerance of the log-det: a backward-stable factor solves A + dA with |dA| <=
N u |A|, and |tr(A^-1 dA)| <= N |A^-1| |dA|, so N^2 u cond(A); the spectra
below lie in [1, 6].  The gradient needs the whole factor; its tolerance is that of
test_gpu_adjoint."""
import numpy as np
import pytest

from brpa import synth
from oracle import adjoint, grid

pytestmark = pytest.mark.gpu


def _pi(n, seed):
    q, _ = np.linalg.qr(np.random.default_rng(seed).standard_normal((n, n)))
    p = (q * np.linspace(0.0, 5.0, n)) @ q.T
    return 0.5 * (p + p.T)


# the last two: more than four work-groups on each of 256 CUs at step 0, fewer at step 4
@pytest.mark.parametrize("n,nf", [(65, 2), (127, 1), (129, 3), (192, 2), (193, 2), (255, 2), (257, 2),
                                  (319, 1), (320, 2), (321, 2), (385, 3), (512, 2), (577, 2),
                                  (449, 200), (578, 120)])
def test_log_det(ctx, n, nf):
    pis = np.stack([_pi(n, 7 * n + k) for k in range(min(nf, 3))])
    ref = np.array([np.linalg.slogdet(np.eye(n) + p)[1] - np.trace(p) for p in pis])
    idx = np.arange(nf) % len(pis)
    _, eu = ctx.ecrpa_analytic(pis[idx], np.ones(nf), np.ones(nf))
    assert np.all(np.abs(eu - ref[idx]) <= 6.0 * n * n * 2.0 ** -53 + 1e-15 * np.abs(ref[idx]))
    # the same matrix gives the same bits wherever it stands in the launch
    assert all(np.unique(eu[idx == k]).size == 1 for k in range(len(pis)))


@pytest.mark.parametrize("n,nf", [(65, 2), (128, 2), (257, 2), (322, 3), (321, 200)])
def test_whole_factor(ctx, n, nf):
    f = synth.make_fragment(3, 40, n, seed=n)
    x, w, _ = grid.freq_grid(f.eocc, f.evir, 12)
    x, w = np.resize(x, nf), np.resize(w, nf)
    got = ctx.ecrpa_grad(f.R, f.eocc, f.evir, x, w)
    for g, r in zip(got, adjoint.ecrpa_grad(f.R, f.eocc, f.evir, x, w)):
        assert np.max(np.abs(g - r)) <= 1e-10 * np.max(np.abs(r))
