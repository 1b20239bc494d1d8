"""Stage counts of the direct-to-LDS GEMM loop (k_gemm_f64): no, one, two and more
full 16-k stages, with and without a last partial one, also as the k ranges of
triangular operands (brpa_dtrtri's corner products).  Integer entries: every
product and sum is exact, so the results are equal."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("k", [1, 2, 15, 16, 17, 31, 32, 33, 47, 48, 49, 63, 64, 66, 80, 113])
@pytest.mark.parametrize("ta,tb", [(False, False), (False, True), (True, False), (True, True)])
def test_stage_counts(ctx, k, ta, tb):
    m, n = 130, 258
    rng = np.random.default_rng(k)
    A = rng.integers(-8, 9, (m, k)).astype(np.float64)
    B = rng.integers(-8, 9, (k, n)).astype(np.float64)

    def dev(x):   # column-major with an even leading dimension
        ld = x.shape[0] + x.shape[0] % 2
        buf = torch.zeros((x.shape[1], ld), dtype=torch.float64, device="cuda")
        buf[:, :x.shape[0]] = torch.from_numpy(np.ascontiguousarray(x.T)).cuda()
        return buf.T[:x.shape[0], :]

    C = torch.full((n, m), np.nan, dtype=torch.float64, device="cuda").T
    ctx.dgemm(dev(A.T if ta else A), dev(B.T if tb else B), C, transa=ta, transb=tb)
    assert np.array_equal(C.cpu().numpy(), A @ B)


@pytest.mark.parametrize("n", [64, 66, 128, 194, 320, 642])
def test_triangular_inverse(ctx, n):
    """Unit upper triangular with entries in {-1, 0, 1} close to the diagonal."""
    rng = np.random.default_rng(n)
    U = np.eye(n) + np.triu(rng.integers(-1, 2, (n, n)), 1) * (np.abs(
        np.subtract.outer(np.arange(n), np.arange(n))) == 7)
    Ud = torch.from_numpy(np.ascontiguousarray(U.T)).cuda().T
    W = torch.empty((n, n), dtype=torch.float64, device="cuda").T
    ctx.dtrtri(Ud, W)
    assert np.array_equal(W.cpu().numpy() @ U, np.eye(n))


@pytest.mark.parametrize("m,n,k", [(1, 1, 1), (127, 129, 31), (128, 128, 33), (129, 255, 48),
                                   (257, 131, 79), (3, 260, 64)])
@pytest.mark.parametrize("ta,tb", [(False, False), (False, True), (True, False), (True, True)])
@pytest.mark.parametrize("off", [0, 1])
def test_odd_leading_dimensions(ctx, m, n, k, ta, tb, off):
    """Odd leading dimensions and operands that are only 8-byte aligned (4 bytes per
    lane), rows and columns around the 128-row tiles."""
    rng = np.random.default_rng(m + k)
    A = rng.integers(-8, 9, (m, k)).astype(np.float64)
    B = rng.integers(-8, 9, (k, n)).astype(np.float64)

    def dev(x):
        ld = x.shape[0] + 1 - x.shape[0] % 2 + 2 * off
        buf = torch.full((x.shape[1] * ld + off,), np.nan, dtype=torch.float64, device="cuda")
        v = buf[off:].view(x.shape[1], ld)
        v[:, :x.shape[0]] = torch.from_numpy(np.ascontiguousarray(x.T)).cuda()
        return v.T[:x.shape[0], :]

    C = torch.full((n, m), np.nan, dtype=torch.float64, device="cuda").T
    ctx.dgemm(dev(A.T if ta else A), dev(B.T if tb else B), C, transa=ta, transb=tb)
    assert np.array_equal(C.cpu().numpy(), A @ B)


def test_far_leading_dimension(ctx):
    """A leading dimension beyond the 32-bit offsets of a tile (2^21 and more)."""
    k, ld = 40, (1 << 21) + 1
    rng = np.random.default_rng(0)
    A = rng.integers(-8, 9, (k, 5)).astype(np.float64)
    B = rng.integers(-8, 9, (k, 3)).astype(np.float64)
    buf = torch.zeros((5, ld), dtype=torch.float64, device="cuda")
    buf[:, :k] = torch.from_numpy(np.ascontiguousarray(A.T)).cuda()
    Bd = torch.from_numpy(np.ascontiguousarray(B.T)).cuda().T
    C = torch.full((3, 5), np.nan, dtype=torch.float64, device="cuda").T
    ctx.dgemm(buf.T[:k, :], Bd, C, transa=True)
    assert np.array_equal(C.cpu().numpy(), A.T @ B)
