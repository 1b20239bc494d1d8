"""FP64 amplitudes with the frequencies stacked into one matrix, in one and in two chunks
(F N NG past 16 M elements), against the CPU oracle on the same guess vectors: NG < o v,
Cholesky-QR basis and (second shape) the eigensolve of the Gram matrix, weights of both
signs.  Tolerances of test_gpu_t2_sosex: 1e-9 relative on T2 and on A."""
import numpy as np
import pytest

from brpa import synth
from oracle import erpa, grid, t2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("o,v,n,nf,ng,neg", [(10, 112, 350, 50, 1050, False), (8, 40, 80, 12, 0, False),
                                             (5, 31, 33, 10, 65, True)])
def test_t2_stacked_frequencies(ctx, o, v, n, nf, ng, neg):
    f = synth.make_fragment(o, v, n, 103)
    x, w, _ = grid.freq_grid(f.eocc, f.evir, 12)
    x, w = np.resize(x, nf), np.resize(w, nf) * (12.0 / nf)   # frequencies repeated
    if neg:
        w[0] = -0.25 * w[0]
    pis = [erpa.gpiug_mo(f.R, f.gaps(), u) for u in x[:12]]
    Pis = [pis[k % 12] for k in range(nf)]
    A_ref, V_ref = t2.t2_v5(f.R, f.gaps(), x, w, Pis, nguess=ng or None, seed=5)
    A, V = ctx.t2(f.R, f.eocc, f.evir, x, w, nguess=ng, seed=5)
    assert len(A) == len(A_ref)
    assert np.max(np.abs(A - A_ref)) <= 1e-9 * np.max(np.abs(A_ref))
    T_ref = (V_ref * A_ref) @ V_ref.T
    T = (V * A) @ V.T
    assert np.max(np.abs(T - T_ref)) <= 1e-9 * np.max(np.abs(T_ref))
