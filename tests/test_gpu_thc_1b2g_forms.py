"""brpa_thc_1b2g on both sides of its choice between the fused kernel and the
integrals formed once, against the definition in torch FP64: odd and even grid
sizes, odd ov, one vector, several chunks of 32 vectors.

Tolerance: the sums run over at most 2 G + 2 ov + v + o products, each term of
the definition taken with absolute values."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("o,v,g,nt", [(1, 1, 1, 1), (2, 3, 64, 5), (5, 20, 130, 33),   # fused
                                      (12, 45, 700, 540), (11, 49, 701, 539), (12, 45, 703, 321),
                                      (9, 33, 1000, 297)])                            # explicit
@pytest.mark.parametrize("diag", [False, True])
def test_thc_1b2g(ctx, o, v, g, nt, diag):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(o + g)
    rnd = lambda *s: torch.randn(s, generator=gen, dtype=torch.float64, device="cuda")  # noqa: E731
    X, Y = rnd(o, g), rnd(v, g)
    Zk = rnd(max(2, g // 3), g) * 0.1
    Z, U = (Zk.T @ Zk), rnd(nt, o, v) / np.sqrt(o * v)
    Z = 0.5 * (Z + Z.T)
    A = -0.4 * torch.rand(nt, generator=gen, dtype=torch.float64, device="cuda")
    e1, e2, es, eg, dg = ctx.thc_1b2g(Z, X, Y, U, A, want_diag=diag)
    u = (2 * g + 2 * o * v + v + o) * 2.0 ** -53
    t1 = t2 = b1 = b2 = 0.0
    for m in range(nt):
        M, B = Y.T @ (U[m].T @ X), Y.abs().T @ (U[m].abs().T @ X.abs())
        a = float(A[m])
        s2, s1 = float((Z * M * M).sum()), float((Z * M * M.T).sum())
        c2, c1 = u * float((Z.abs() * B * B).sum()), u * float((Z.abs() * B * B.T).sum())
        assert abs(es[m] + s1 * a) <= c1 * abs(a)
        assert abs(eg[m] + 4 * s2 * a * a) <= 4 * c2 * a * a
        if diag:
            d = torch.diagonal(M).cpu().numpy()
            assert np.max(np.abs(dg[m] - d)) <= (v + o) * 2.0 ** -53 * float(torch.diagonal(B).max())
        t1, t2, b1, b2 = t1 - s1 * a, t2 - 2 * s2 * a * a, b1 + c1 * abs(a), b2 + 2 * c2 * a * a
    assert abs(e1 - 2 * t1) <= 2 * b1 and abs(e2 - 2 * t2) <= 2 * b2
