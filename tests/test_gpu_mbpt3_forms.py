"""Final contraction of MBPT3-1: the explicit ov form on X itself (many amplitude
vectors) and the pair forms on a factor of X (few of them), truncated from one set of
amplitudes, on host and device inputs.  Tolerances of test_gpu_mbpt3: 1e-10 relative to
|E| in FP64, 1e-7 Ha in the split-int8 form."""
import numpy as np
import pytest

from brpa import synth
from oracle import erpa, grid, mbpt3, t2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nt", [1, 5, 17, 64, 180])
@pytest.mark.parametrize("prec", ["fp64", "split_i8"])
def test_forms(ctx, nt, prec):
    import torch
    o, v, n = 5, 36, 90
    f = synth.make_fragment(o, v, n, 8)
    x, w, _ = grid.freq_grid(f.eocc, f.evir, 12)
    Pis = [erpa.gpiug_mo(f.R, f.gaps(), xx) for xx in x]
    A, V = t2.t2_v5(f.R, f.gaps(), x, w, Pis, seed=5, nguess=180, cutoff=0.0)
    A, V = A[:nt], np.ascontiguousarray(V[:, :nt])
    ref = mbpt3.mbpt3_1(f.R, V, A, o, v, f.eocc, f.evir)
    tol = 1e-10 * abs(ref) if prec == "fp64" else 1e-7
    assert abs(ctx.mbpt3_1(V, A, f.R, f.eocc, f.evir, precision=prec) - ref) <= tol
    Vd, Rd = torch.from_numpy(V).cuda(), torch.from_numpy(f.R).cuda()
    assert abs(ctx.mbpt3_1(Vd, A, Rd, f.eocc, f.evir, precision=prec) - ref) <= tol
