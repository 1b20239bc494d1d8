"""Calls with a faster form that takes more device scratch run in the other form where the
workspace may not grow that far (BRPA_WS_BUDGET_GB, else 3/4 of the free memory): same
results, and the form that ran as the kernel times tell it.  A context of its own per
case, since a workspace once held is used."""
import ctypes as C
import math

import numpy as np
import pytest

import brpa
from brpa import _lib, synth
from oracle import adjoint, erpa, grid, mbpt3, t2

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

U_ = 2.0 ** -53


@pytest.fixture
def small(monkeypatch):
    """Runs a call on a new context whose workspace may not grow beyond what the call
    cannot do without; returns its result and the launches of one measured kernel."""
    def run(call, kernel):
        monkeypatch.setenv("BRPA_WS_BUDGET_GB", "0")
        c = brpa.Context(0)
        try:
            return call(c), _launches(c, kernel)
        finally:
            c.close()
            monkeypatch.delenv("BRPA_WS_BUDGET_GB")
    return run


def _launches(c, kernel):
    n = C.c_int64()
    assert c._lib.brpa_last_kernel_stats(c._h, kernel, None, None, C.byref(n)) == 0
    return n.value


def _workspace(c, monkeypatch):
    """Bytes of the context's workspace: the largest size that it affords without growing
    (the library's own ws_affords)."""
    affords = getattr(c._lib, "_Z10ws_affordsPK8brpa_ctxm")
    affords.argtypes, affords.restype = [C.c_void_p, C.c_size_t], C.c_bool
    with monkeypatch.context() as m:
        m.setenv("BRPA_WS_BUDGET_GB", "0")
        lo, hi = 0, 1 << 40
        while hi - lo > 1:
            mid = (lo + hi) // 2
            lo, hi = (mid, hi) if affords(c._h, mid) else (lo, mid)
    return lo


def _amplitudes(o, v, n, nt, seed, s2=False):
    rng = np.random.default_rng(seed)
    R = 0.3 * rng.standard_normal((o * v, n)) * np.exp(-4.0 * np.arange(n) / n)
    V = rng.standard_normal((o * v, nt)) / math.sqrt(o * v)
    return R, V, -0.45 * np.exp(-7.0 * np.arange(nt) / nt)


def _sosex(R, V, B, o, v):
    """-sum (aj|bi) T(ai, bj) and (N + NT2) u times its absolute sum, doubled."""
    G = (R @ R.T).reshape(o, v, o, v)
    T = ((V * B) @ V.T).reshape(o, v, o, v)
    p = np.einsum("iajb,jaib->iajb", G, T)
    return -p.sum(), 2.0 * (R.shape[1] + V.shape[1]) * U_ * np.abs(p).sum()


# shapes that take the explicit form where there is memory for it
@pytest.mark.parametrize("o,v,n,nt", [(2, 16, 20, 24), (3, 12, 40, 36), (5, 26, 64, 90),
                                      (6, 33, 97, 190), (9, 65, 150, 300)])
@pytest.mark.parametrize("precision", ["fp64", "split_i8"])
@pytest.mark.parametrize("dev", [False, True])
def test_sosex_pairs(ctx, small, o, v, n, nt, precision, dev):
    R, V, A = _amplitudes(o, v, n, nt, 10 * o + v)
    conv = (lambda x: torch.from_numpy(x).cuda()) if dev else (lambda x: x)
    # the split pair kernel truncates at 2^-35 of the column maxima
    slack = 1e-7 if precision == "split_i8" else 0.0
    # its slices are padded (v to 64): at one of the shapes they take more than the explicit
    # blocks, which then run all the same
    pairs = (precision, n) != ("split_i8", 40)
    for s2, b in ((False, A), (True, A / (1.0 - 4.0 * A * A))):
        ref, tol = _sosex(R, V, b, o, v)
        call = lambda c: c.sosex(conv(V), conv(A), conv(R), o, v, s2_operator=s2,  # noqa: E731
                                 precision=precision)
        e, dots = small(call, _lib.KERNEL_SOSEX_DOT)
        assert (dots == 0) == pairs and abs(e - ref) <= tol + slack, (dots, e, ref)
        e = call(ctx)
        assert _launches(ctx, _lib.KERNEL_SOSEX_DOT) > 0 and abs(e - ref) <= tol, (e, ref)


@pytest.mark.parametrize("precision", ["fp64", "split_i8"])
@pytest.mark.parametrize("signs", ["negative", "both"])
@pytest.mark.parametrize("o,v,n,nt", [(4, 60, 30, 12), (10, 200, 500, 480)])
def test_mbpt3_1_pairs(ctx, small, o, v, n, nt, precision, signs):
    """MBPT3-1 by a factor of X and the pair products, its Cholesky factor, or with
    amplitudes of both signs (X indefinite) the eigenpairs: few vectors, which take it
    anyway, and many where the explicit form's blocks are not affordable."""
    f = synth.make_fragment(o, v, n, 12)
    rng = np.random.default_rng(5)
    V = np.ascontiguousarray(np.linalg.qr(rng.standard_normal((o * v, nt)))[0])
    A = rng.uniform(-0.3, 0.3 if signs == "both" else -0.01, nt)
    Am, Bm = mbpt3.mbpt3_1_matrices(f.R, V, A, f.eocc, f.evir)
    X = mbpt3.lyapunov(Bm, Am)
    ev = np.linalg.eigvalsh(0.5 * (X + X.T))
    assert ev.min() < 0.0 and (ev.max() > 0.0) == (signs == "both")
    ref = -mbpt3.trxk(f.R, V, X, o, v)
    e, dots = small(lambda c: c.mbpt3_1(V, A, f.R, f.eocc, f.evir, precision=precision),
                    _lib.KERNEL_SOSEX_DOT)
    assert dots == 0
    assert abs(e - ref) <= (1e-10 * abs(ref) if precision == "fp64" else 1e-7)
    e = ctx.mbpt3_1(V, A, f.R, f.eocc, f.evir, precision=precision)
    assert (_launches(ctx, _lib.KERNEL_SOSEX_DOT) > 0) == (nt > v / 2)
    assert abs(e - ref) <= (1e-10 * abs(ref) if precision == "fp64" else 1e-7)


def _thc_inputs(o, v, g, nt, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    rnd = lambda *s: torch.randn(s, generator=gen, dtype=torch.float64, device="cuda")  # noqa: E731
    X, Y, Zk = rnd(o, g), rnd(v, g), rnd(max(2, g // 3), g) * 0.1
    Z, U = Zk.T @ Zk, rnd(nt, o, v) / np.sqrt(o * v)
    return 0.5 * (Z + Z.T), X, Y, U, -0.4 * torch.rand(nt, generator=gen, dtype=torch.float64,
                                                       device="cuda")


@pytest.mark.parametrize("o,v,g,nt", [(12, 45, 700, 540), (11, 49, 701, 539)])
def test_thc_1b2g_fused(small, monkeypatch, o, v, g, nt):
    """The workspace tells the form: 128 MB for split k and more in the explicit one."""
    ins = _thc_inputs(o, v, g, nt, o + g)
    Z, X, Y, U, A = ins
    bound = (2 * g + 2 * o * v + v + o) * U_
    fused, explicit, kept = _both(small, monkeypatch, lambda c: c.thc_1b2g(*ins, want_diag=True))
    assert kept[1] - kept[0] >= 128 << 20, kept
    for m in range(nt):
        M, B = Y.T @ (U[m].T @ X), Y.abs().T @ (U[m].abs().T @ X.abs())
        a = float(A[m])
        s1, c1 = float((Z * M * M.T).sum()), bound * float((Z.abs() * B * B.T).sum())
        s2, c2 = float((Z * M * M).sum()), bound * float((Z.abs() * B * B).sum())
        for es, eg in (fused[2:4], explicit[2:4]):
            assert abs(es[m] + s1 * a) <= c1 * abs(a)
            assert abs(eg[m] + 4 * s2 * a * a) <= 4 * c2 * a * a


@pytest.mark.parametrize("o,v,n,g,launches", [(1, 1, 1, 1, 1), (3, 21, 70, 37, 3),
                                              (5, 60, 200, 333, 5), (2, 45, 30, 131073, 4)])
def test_thc_piu_chunks(ctx, small, o, v, n, g, launches):
    """Products of one occupied orbital, and of as many virtual ones as 32 MB hold."""
    gen = torch.Generator(device="cuda")
    gen.manual_seed(g)
    Xi, Xa, Z = (torch.randn(s, g, generator=gen, dtype=torch.float64, device="cuda")
                 for s in (o, v, n))
    eo, ev, x = -np.arange(o, 0.0, -1.0), np.arange(1.0, v + 1.0), np.array([0.3, 2.0])
    call = lambda c: c.thc_piu(Xa, Xi, Z, eo, ev, x, want_R=True)  # noqa: E731
    (Pi, R), ran = small(call, _lib.KERNEL_GEMM_F64)
    assert ran == launches
    Pi0, R0 = call(ctx)
    assert _launches(ctx, _lib.KERNEL_GEMM_F64) == 1
    H = (Xi[:, None, :] * Xa[None, :, :]).reshape(o * v, g)
    ref, tol = H @ Z.T, 2.0 * (g + 2) * U_ * (H.abs() @ Z.abs().T)
    assert bool(((R - ref).abs() <= tol).all()) and bool(((R0 - ref).abs() <= tol).all())
    d = torch.from_numpy(ev[None, :] - eo[:, None]).reshape(-1, 1).cuda()
    for w, u in enumerate(x):
        c = 4.0 * d / (d * d + u * u)
        for P, r in ((Pi, R), (Pi0, R0)):
            bound = 2.0 * (o * v + 4) * U_ * (r.abs().T @ (c * r.abs()))
            assert bool(((P[w] - r.T @ (c * r)).abs() <= bound).all())


def _both(small, monkeypatch, call):
    """The call on a context without room and on one with it, and the bytes of workspace
    that each holds afterwards."""
    kept = []

    def run(c):
        out = call(c)
        kept.append(_workspace(c, monkeypatch))
        return out

    lean, _ = small(run, _lib.KERNEL_GEMM_F64)
    c = brpa.Context(0)
    full = run(c)
    c.close()
    return lean, full, kept


def test_grad_one_frequency_at_a_time(small, monkeypatch):
    """Two frequencies per product take one K x N matrix (33 MB) more."""
    o, v, n, nf = 10, 409, 1000, 5
    f = synth.make_fragment(o, v, n, seed=23)
    x, w, _ = grid.freq_grid(f.eocc, f.evir, 12)
    x, w = x[:nf], w[:nf]
    lean, full, kept = _both(small, monkeypatch,
                             lambda c: c.ecrpa_grad(f.R, f.eocc, f.evir, x, w))
    assert kept[1] - kept[0] >= 30 << 20, kept
    for a, b, r in zip(lean, full, adjoint.ecrpa_grad(f.R, f.eocc, f.evir, x, w)):
        assert max(np.max(np.abs(a - r)), np.max(np.abs(b - r))) <= 1e-10 * np.max(np.abs(r))


def test_mbpt3_1_without_split(small, monkeypatch):
    o, v, n, nt = 6, 40, 90, 70
    f = synth.make_fragment(o, v, n, 12)
    V = np.ascontiguousarray(np.linalg.qr(
        np.random.default_rng(5).standard_normal((o * v, nt)))[0])
    A = -np.linspace(0.3, 0.01, nt)
    ref = mbpt3.mbpt3_1(f.R, V, A, o, v, f.eocc, f.evir)
    lean, full, kept = _both(small, monkeypatch,
                             lambda c: c.mbpt3_1(V, A, f.R, f.eocc, f.evir))
    assert kept[1] - kept[0] >= 128 << 20, kept
    assert max(abs(lean - ref), abs(full - ref)) <= 1e-10 * abs(ref)


@pytest.mark.parametrize("o,v,n,nf,ng,neg", [(8, 40, 80, 12, 0, False), (5, 31, 33, 10, 65, True)])
@pytest.mark.parametrize("precision", ["fp64", "split_i8"])
def test_t2_without_stacks(small, monkeypatch, o, v, n, nf, ng, neg, precision):
    """One frequency per product and no split k; the bounds of the oracle tests."""
    f = synth.make_fragment(o, v, n, 103)
    x, w, _ = grid.freq_grid(f.eocc, f.evir, nf)
    if neg:
        w[0] = -0.25 * w[0]
    Pis = [erpa.gpiug_mo(f.R, f.gaps(), u) for u in x]
    A_ref, V_ref = t2.t2_v5(f.R, f.gaps(), x, w, Pis, nguess=ng or None, seed=5)
    T_ref = (V_ref * A_ref) @ V_ref.T
    lean, full, kept = _both(small, monkeypatch, lambda c: c.t2(
        f.R, f.eocc, f.evir, x, w, nguess=ng, seed=5, precision=precision))
    assert kept[1] - kept[0] >= 128 << 20, kept
    if precision == "split_i8":   # against its own result with the room
        A_ref, T_ref = full[0], (full[1] * full[0]) @ full[1].T
    for A, V in (lean, full):
        assert len(A) == len(A_ref)
        assert np.max(np.abs(A - A_ref)) <= 1e-9 * np.max(np.abs(A_ref))
        assert np.max(np.abs((V * A) @ V.T - T_ref)) <= 1e-9 * np.max(np.abs(T_ref))


def test_sosex_split_i8_pairs_large(ctx, small):
    """The split-int8 pair kernel on a large fragment's own amplitudes (o=64, v=600,
    NAux=3200, 16 frequencies, NT2 = 3 NAux) within 1e-7 Ha of the FP64 explicit form."""
    o, v, n = 64, 600, 3200
    f = synth.make_fragment(o, v, n, synth.BASE_SEED)
    x, w, _ = grid.freq_grid(f.eocc, f.evir, 16)
    R = torch.from_numpy(f.R).cuda()
    A, V = ctx.t2(R, f.eocc, f.evir, x, w, nguess=3 * n, seed=1, device=True)
    e = ctx.sosex(V, A, R, o, v)
    assert _launches(ctx, _lib.KERNEL_SOSEX_DOT) > 0
    ctx._lib.brpa_ctx_trim(ctx._h)
    e8, dots = small(lambda c: c.sosex(V, A, R, o, v, precision="split_i8"), _lib.KERNEL_SOSEX_DOT)
    print("E_x explicit %.10f  split-int8 pairs - explicit %.3e" % (e, e8 - e))
    assert dots == 0 and abs(e8 - e) <= 1e-7
