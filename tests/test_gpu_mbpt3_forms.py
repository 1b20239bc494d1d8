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


@pytest.mark.parametrize("spread,size", [(1e2, 0.1), (1e8, 0.1), (1e2, 30.0), (1e2, 3e3)])
def test_inverses(ctx, spread, size):
    """The inverses of the sign iteration at condition numbers of B where the Cholesky of
    B^T B suffices, needs refinement and breaks down (LU).  A backward-stable solution is
    off by about cond(B) n u; ten times that."""
    o, v, n, nt = 4, 30, 50, 70
    rng = np.random.default_rng(3)
    R = size * rng.standard_normal((o * v, n))
    eocc, evir = -np.geomspace(1e-3, 1e-3 * spread, o)[::-1], np.geomspace(1e-3, 1e-3 * spread, v)
    V = np.linalg.qr(rng.standard_normal((o * v, nt)))[0]
    A = -np.linspace(0.2, 0.01, nt)
    ref = mbpt3.mbpt3_1(R, V, A, o, v, eocc, evir)
    cond = np.linalg.cond(mbpt3.mbpt3_1_matrices(R, V, A, eocc, evir)[1])
    e = ctx.mbpt3_1(V, A, R, eocc, evir)
    assert abs(e - ref) <= (1e-10 + 10 * cond * nt * 2.0 ** -53) * abs(ref)
