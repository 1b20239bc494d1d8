"""E(u) = log det(1 + P) - tr P at small P is as exact as one rounding per step allows: 1 + P, the
sum of the updates added to it, and the square root whose logarithm counts twice.  In units of
2^-53 these have variances 1/3, 1/3 and 4/3 per pivot (uniform, values of 1 to 2), 2 N together;
1.3 times the root of it for the spread of an rms over 128 values and more.  With the updates
added one by one 26 units were left at N = 64."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nfreq,nseed", [(16, 8), (160, 1)])
@pytest.mark.parametrize("n", [20, 33, 64])
def test_small_p(ctx, n, nfreq, nseed):
    o, v, ld = 3, 40, np.longdouble
    eocc, evir = np.linspace(-1.3, -0.7, o), np.linspace(0.2, 1.8, v)
    d = (evir.astype(ld) - eocc.astype(ld)[:, None]).ravel()
    x, w = np.linspace(0.05, 1.5, nfreq), np.full(nfreq, 0.1)
    err = []
    for seed in range(nseed):
        R = np.random.default_rng(seed).standard_normal((o * v, n)) * np.sqrt(0.5 / (o * v * n))
        eu = ctx.ecrpa(R, eocc, evir, x, w)[1]
        for u, e in zip(x.astype(ld), eu):
            P = R.T.astype(ld) @ ((4 * d / (d * d + u * u))[:, None] * R)
            A, ref = P + np.eye(n, dtype=ld), -np.trace(P)
            for k in range(n):
                ref += np.log(A[k, k])
                A[k + 1:, k + 1:] -= np.outer(A[k + 1:, k], A[k, k + 1:]) / A[k, k]
            err.append(float(e - ref) * 2.0 ** 53)
    assert np.sqrt(np.mean(np.square(err))) <= 1.3 * np.sqrt(2 * n)
