"""T^T I T of the T2 amplitudes adds whole frequencies: two of weights +10^6 and -10^6 at one
point cancel exactly, so what remains is the third one's.  The basis moves by about
10^6 eps = 10^-9 and its Ritz values by the square (I has rank NAux = nguess), so 10^-12 of
the largest amplitude bounds the difference; one sum over all frequencies leaves 10^-10."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("budget", [None, "0"])
@pytest.mark.parametrize("o,v,n", [(3, 4, 5), (4, 9, 12), (7, 20, 70)])
def test_cancelling_frequencies(ctx, monkeypatch, budget, o, v, n):
    if budget is not None:
        monkeypatch.setenv("BRPA_WS_BUDGET_GB", budget)
    rng = np.random.default_rng(o)
    R = np.linalg.qr(rng.standard_normal((o * v, n)))[0]
    eo, ev = np.linspace(-1.2, -1.0, o), np.linspace(0.2, 0.4, v)

    def amplitudes(x, w):
        A, V = ctx.t2(R, eo, ev, np.array(x), np.array(w), nguess=n, seed=3, cutoff=1e-10)
        assert len(A) == n
        return np.sort(A)

    a = amplitudes([0.7], [0.5])
    b = amplitudes([0.4, 0.4, 0.7], [1e6, -1e6, 0.5])
    assert abs(a - b).max() <= 1e-12 * abs(a).max()
