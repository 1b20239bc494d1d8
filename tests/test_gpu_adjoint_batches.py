"""dE/dR and dE/d(eps) with several frequencies per product M_k R^T: all of them (4 tiles
each), and two at a time with one left over (256 tiles each on 512 slots).
Tolerance of test_gpu_adjoint: 1e-10 of the largest element."""
import numpy as np
import pytest

from brpa import synth
from oracle import adjoint, grid

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("o,v,n,nf", [(3, 50, 200, 7), (10, 409, 1000, 5)])
def test_grad_frequency_batches(ctx, o, v, n, nf):
    f = synth.make_fragment(o, v, n, seed=23)
    x, w, _ = grid.freq_grid(f.eocc, f.evir, 12)
    x, w = x[:nf], w[:nf]
    got = ctx.ecrpa_grad(f.R, f.eocc, f.evir, x, w)
    for g, r in zip(got, adjoint.ecrpa_grad(f.R, f.eocc, f.evir, x, w)):
        assert np.max(np.abs(g - r)) <= 1e-10 * np.max(np.abs(r))
