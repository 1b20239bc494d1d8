"""The explicit SOSEX contraction sums in double-double: terms of 2^61 that cancel leave the
small one, in one column and over several (o = 1, exact entries: T(i, b) = T(b, i) = 1 by
pairs of vectors (e_i + e_b), (e_i - e_b) with weights 1/2 and -1/2)."""
import numpy as np
import pytest

from brpa import _lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [(0, 1, 2), (2, 0, 1), (5, 37, 68), (3, 259, 130)])
def test_cancelling_terms(ctx, rows):
    b, big = max(rows) + 1, 2.0 ** 60
    v = b + 1
    R, V = np.zeros((v, 3)), np.zeros((v, 6))
    for k, (i, g) in enumerate(zip(rows, (big, -big, 1.0))):
        R[i, k], R[b, k] = 1.0, g           # G(i, b) = g
        V[i, 2 * k:2 * k + 2] = 1.0
        V[b, 2 * k], V[b, 2 * k + 1] = 1.0, -1.0
    A = np.tile([0.5, -0.5], 3)
    # many vectors, so that the explicit form is the cheaper one at every v
    nt = 4 * v
    V, A = np.pad(V, ((0, 0), (0, nt - 6))), np.pad(A, (0, nt - 6))
    R = np.pad(R, ((0, 0), (0, 4 * v - 3)))
    e = ctx.sosex(V, A, R, 1, v)
    assert ctx.last_kernel_stats(_lib.KERNEL_SOSEX_DOT)[2] == 1
    assert e == -2.0
