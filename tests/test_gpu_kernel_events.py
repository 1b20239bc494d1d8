"""Event pairs of the measured kernels: none is left in the context by a call that ran
dense products, so that their number does not grow from call to call (the library's own
kstat_begin tells the index of the next pair)."""
import ctypes as C

import numpy as np
import pytest

import brpa
from brpa import synth

pytestmark = pytest.mark.gpu


def _pending(c):
    begin, drop = getattr(c._lib, "_Z11kstat_beginP8brpa_ctxPm"), getattr(c._lib, "_Z10kstat_dropP8brpa_ctx")
    begin.argtypes, drop.argtypes, drop.restype = [C.c_void_p, C.POINTER(C.c_size_t)], [C.c_void_p], None
    slot = C.c_size_t()
    assert begin(c._h, C.byref(slot)) == 0
    drop(c._h)
    return slot.value


def _calls(o=4, v=30, n=130):
    f = synth.make_fragment(o, v, n, 3)
    x, w = np.linspace(0.1, 2.0, 5), np.ones(5)
    rng = np.random.default_rng(2)

    def amps(nt):
        V = np.ascontiguousarray(np.linalg.qr(rng.standard_normal((o * v, nt)))[0])
        return V, -np.linspace(0.2, 0.01, nt)

    V2, A2 = amps(2)      # few vectors: the pair products
    V60, A60 = amps(60)
    g = 500
    Z = rng.standard_normal((g, g))
    Z = Z + Z.T
    Xi, Y = rng.standard_normal((o, g)), rng.standard_normal((v, g))
    return {
        "ecrpa_grad": lambda c: c.ecrpa_grad(f.R, f.eocc, f.evir, x, w),
        "mbpt3_1 few": lambda c: c.mbpt3_1(V2, A2, f.R, f.eocc, f.evir),
        "mbpt3_1": lambda c: c.mbpt3_1(V60, A60, f.R, f.eocc, f.evir),
        "sosex": lambda c: c.sosex(V60, A60, f.R, o, v),
        "t2": lambda c: c.t2(f.R, f.eocc, f.evir, x, w, seed=1),
        "thc_piu": lambda c: c.thc_piu(Y, Xi, np.ascontiguousarray(Z[:20]), f.eocc, f.evir, x),
        "thc_1b2g": lambda c: c.thc_1b2g(Z, Xi, Y, rng.standard_normal((2000, o, v)),
                                         -np.full(2000, 0.1)),
    }


@pytest.mark.parametrize("name", sorted(_calls()))
def test_none_left(name):
    c = brpa.Context(0)
    try:
        call = _calls()[name]
        for _ in range(2):
            call(c)
            assert _pending(c) == 0
    finally:
        c.close()
