"""brpa_sosex on both sides of its choice between the explicit ov space and the
pair products, against the contraction written out in torch FP64: sizes below and
around the 128-row GEMM tiles, an ov dimension of two occupied blocks (the second of
one orbital), few amplitude vectors (pair products), the S2 rescaling, host and
device inputs.

Tolerance: each of the K^2 products of entries is formed to (N + NT2) u relative to
its absolute sum, so (N + NT2) u sum |G||T|, doubled for the two summations."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def _inputs(o, v, n, nt, seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    rnd = lambda *s: torch.randn(s, generator=g, dtype=torch.float64, device="cuda")  # noqa: E731
    R = rnd(o * v, n) * 0.3 * torch.exp(-4.0 * torch.arange(n, device="cuda") / n)
    V = rnd(o * v, nt) / np.sqrt(o * v)
    A = -0.45 * torch.exp(-7.0 * torch.arange(nt, dtype=torch.float64, device="cuda") / nt)
    return R, V, A


def _reference(R, V, B, o, v):
    G = (R @ R.T).view(o, v, o, v)
    T = ((V * B) @ V.T).view(o, v, o, v)
    e = bound = 0.0
    for i in range(o):
        p = G[i] * T[:, :, i].transpose(0, 1)      # [a][j][b]
        e += float(p.sum())
        bound += float(p.abs().sum())
    return -e, bound * 2.0 * (R.shape[1] + V.shape[1]) * 2.0 ** -53


@pytest.mark.parametrize("o,v,n,nt", [(1, 1, 1, 1), (1, 5, 3, 2), (3, 7, 9, 15), (5, 26, 64, 90),
                                      (4, 32, 100, 128), (9, 43, 150, 300), (6, 60, 200, 4),
                                      (12, 129, 333, 700), (66, 250, 300, 300)])
@pytest.mark.parametrize("precision", ["fp64", "split_i8"])
def test_sosex_matches_torch(ctx, o, v, n, nt, precision):
    R, V, A = _inputs(o, v, n, nt, 7 * o + v)
    ref, tol = _reference(R, V, A, o, v)
    e = ctx.sosex(V, A, R, o, v, alpha=0.5, precision=precision)
    # the pair products of the split form truncate at 2^-35 of the column maxima
    assert abs(e - 0.5 * ref) <= tol + (1e-7 if precision == "split_i8" else 0.0), (e, 0.5 * ref)


@pytest.mark.parametrize("host", [False, True])
def test_sosex_s2_operator(ctx, host):
    o, v, n, nt = 7, 37, 120, 240
    R, V, A = _inputs(o, v, n, nt, 3)
    ref, tol = _reference(R, V, A / (1.0 - 4.0 * A * A), o, v)
    conv = (lambda t: t.cpu().numpy()) if host else (lambda t: t)
    e = ctx.sosex(conv(V), conv(A), conv(R), o, v, s2_operator=True)
    assert abs(e - ref) <= tol
