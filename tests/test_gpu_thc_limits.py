"""brpa_thc_piu at the ends of its size range: an empty spin block is skipped whatever
ngrid x naux is, a block with orbitals is refused beyond 2^31 elements."""
import ctypes as C

import numpy as np
import pytest

from brpa import _lib

pytestmark = pytest.mark.gpu


def _piu(ctx, Pi, X, g, o, v, n, nf, accumulate):
    """The C entry point: X stands for the three factors, which are not read here."""
    e, p = np.linspace(1.0, 2.0, 8), lambda a: C.c_void_p(a.ctypes.data)
    x = np.ones(nf)
    return ctx._lib.brpa_thc_piu(ctx._h, p(Pi), None, p(X), p(X), p(X), g, o, v, n, p(e), p(e),
                                 p(x), nf, 4.0, accumulate)


@pytest.mark.parametrize("o,v", [(0, 3), (3, 0), (0, 0)])
@pytest.mark.parametrize("g,n", [(16, 8), (1 << 29, 8)])
def test_empty_block(ctx, o, v, g, n):
    Pi = np.full((2, n, n), 7.0)
    assert _piu(ctx, Pi, np.zeros(1), g, o, v, n, 2, 1) == _lib.OK and np.all(Pi == 7.0)
    assert _piu(ctx, Pi, np.zeros(1), g, o, v, n, 2, 0) == _lib.OK and np.all(Pi == 0.0)


def test_refused(ctx):
    assert _piu(ctx, np.zeros((1, 8, 8)), np.zeros(1), 1 << 29, 2, 3, 8, 1, 0) == _lib.ERR_ARG


@pytest.mark.parametrize("o,v,g", [(64, (1 << 18) + 3, 1), (1, 1, (1 << 24) + 77)])
def test_long_launches(ctx, o, v, g):
    """More columns, and more points, of orbital products than one launch's grid covers.
    R is an exact integer here: products of -1, 0 and 1."""
    torch = pytest.importorskip("torch")
    gen = torch.Generator(device="cuda")
    gen.manual_seed(1)
    Xi, Xa, Z = (torch.randint(-1, 2, (s, g), generator=gen, device="cuda").double()
                 for s in (o, v, 1))
    eo, ev, x = -np.arange(o, 0.0, -1.0), np.arange(1.0, v + 1.0), np.array([1.0])
    _, R = ctx.thc_piu(Xa, Xi, Z, eo, ev, x, want_R=True)
    ref = torch.zeros(o, v, dtype=torch.float64, device="cuda")
    for i in range(o):
        ref[i] = (Xa * (Xi[i] * Z[0])).sum(1)
    assert torch.equal(R.view(o, v), ref)
