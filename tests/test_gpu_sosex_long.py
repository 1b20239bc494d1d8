"""brpa_sosex with more than 2^32 elements of amplitude vectors (explicit form, device
inputs): A_mu nonzero for the last vectors only, so the energy follows from those columns
alone.  Tolerance: (N + NT2) u times the absolute sum, as for the smaller sizes."""
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def test_more_than_2_32_elements(ctx):
    o, v, n, nt, live = 5, 859, 600, 1000000, 40
    k = o * v
    assert k * nt > 1 << 32
    if torch.cuda.mem_get_info()[0] < 150e9:
        pytest.skip("needs 75 GB of device memory and as much headroom")
    gen = torch.Generator(device="cuda")
    gen.manual_seed(7)
    rnd = lambda *s: torch.randn(s, generator=gen, dtype=torch.float64, device="cuda")  # noqa: E731
    R = 0.05 * rnd(k, n)
    # 0 times an element that the scaling missed is not 0: the unused columns hold ones
    V = torch.ones(k, nt, dtype=torch.float64, device="cuda")
    V[:, nt - live:] = rnd(k, live) / k ** 0.5
    A = torch.zeros(nt, dtype=torch.float64, device="cuda")
    A[nt - live:] = -0.4
    G = (R @ R.T).view(o, v, o, v)
    T = ((V[:, nt - live:] * A[nt - live:]) @ V[:, nt - live:].T).view(o, v, o, v)
    ref = bound = 0.0
    for i in range(o):
        p = G[i] * T[:, :, i].transpose(0, 1)
        ref, bound = ref - float(p.sum()), bound + float(p.abs().sum())
    e = ctx.sosex(V, A, R, o, v)
    del V, G, T
    torch.cuda.empty_cache()
    ctx._lib.brpa_ctx_trim(ctx._h)
    assert abs(e - ref) <= 2.0 * (n + nt) * 2.0 ** -53 * bound, (e, ref)
