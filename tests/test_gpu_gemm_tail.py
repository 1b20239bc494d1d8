"""GEMM grids of more than two tiles per CU whose last tiles are split in k
(k_gemm_f64 TAIL, k_gemm_reduce_tail), through the explicit SOSEX form: even and odd
orders, a ragged last tile in the split part, two to four chunks of k.

Tolerance of test_gpu_sosex_explicit: (N + NT2) u sum |G||T|, doubled for the two
summations."""
import pytest

from test_gpu_sosex_explicit import _inputs, _reference

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("o,v,n,nt", [(33, 130, 530, 520), (39, 121, 777, 1031), (33, 132, 800, 1300)])
def test_split_tail(ctx, o, v, n, nt):
    R, V, A = _inputs(o, v, n, nt, o + v)
    ref, tol = _reference(R, V, A, o, v)
    assert abs(ctx.sosex(V, A, R, o, v) - ref) <= tol
