"""Split-int8 Pi product (k_syrk_i8_128, k_syrk_i8_64): orders around its 64- and
128-column tiles and 16-column groups, row counts around its 64-row stages and the
128-row padding, and grids around the 256-tile rounds of the XCD order.  Every
variant forms the same integers, so their energies are equal; the split form stays
within its 1e-7 Ha of the FP64 one."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _frag(o, v, n, nf, seed):
    rng = np.random.default_rng(seed)
    R = rng.standard_normal((o * v, n)) * 0.3 * np.exp(-4.0 * np.arange(n) / n)
    t, w = np.polynomial.legendre.leggauss(nf)
    return (R, np.sort(rng.uniform(-1.5, -0.3, o)), np.geomspace(0.05, 3.0, v),
            (1 + t) / (1 - t), 2 * w / (1 - t) ** 2)


@pytest.mark.parametrize("o,v,n,nf", [(1, 5, 15, 3), (2, 32, 64, 5), (3, 43, 127, 4),
                                      (4, 32, 128, 3), (4, 33, 129, 3), (5, 51, 192, 2),
                                      (6, 64, 255, 85), (6, 43, 257, 43), (9, 71, 385, 27)])
def test_variants_and_fp64(o, v, n, nf):
    import brpa
    f = _frag(o, v, n, nf, o + v + n)
    with brpa.Context(0) as ctx:
        e64 = ctx.ecrpa(*f, precision="fp64")[1]
        e8 = ctx.ecrpa(*f, precision="split_i8")[1]
        assert np.max(np.abs(e8 - e64)) <= 1e-7
        # brpa_autotune fails (BRPA_ERR_INTERNAL) unless all variants agree bit for bit
        assert ctx.autotune([f])
        assert np.array_equal(ctx.ecrpa(*f, precision="split_i8")[1], e8)
