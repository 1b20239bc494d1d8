"""k_gemm_f64 with leading dimensions beyond the 32-bit offsets of a tile (2^21 and more):
every form, row and column counts around the 128-row tiles, stages with and without a
remainder.  Integer entries: every sum is exact."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("m,n,k", [(129, 7, 50), (5, 130, 33), (127, 128, 64), (1, 2, 17)])
@pytest.mark.parametrize("ta,tb", [(False, False), (False, True), (True, False), (True, True)])
@pytest.mark.parametrize("odd", [0, 1])
def test_far(ctx, m, n, k, ta, tb, odd):
    rng = np.random.default_rng(m + n + k)
    A = rng.integers(-8, 9, (m, k)).astype(np.float64)
    B = rng.integers(-8, 9, (k, n)).astype(np.float64)

    def dev(x, ld):
        buf = torch.zeros((x.shape[1], ld), dtype=torch.float64, device="cuda")
        buf[:, :x.shape[0]] = torch.from_numpy(np.ascontiguousarray(x.T)).cuda()
        return buf.T[:x.shape[0], :]

    # both far, and each beside an ordinary one
    for fa, fb in ((True, True), (True, False), (False, True)):
        a, b = A.T if ta else A, B.T if tb else B
        C = torch.full((n, m), np.nan, dtype=torch.float64, device="cuda").T
        ctx.dgemm(dev(a, (1 << 21) + odd if fa else a.shape[0] + odd),
                  dev(b, (1 << 22) + odd if fb else b.shape[0] + odd), C, transa=ta, transb=tb)
        assert np.array_equal(C.cpu().numpy(), A @ B)
