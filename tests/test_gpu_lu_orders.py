"""W = [(I - V Pi)^-1 - I] V by LU over the orders at which the factorisation changes its shape:
the panels' columns per thread (64, 128, 256, 512, 1024, 2048 rows) and width (16, 8), and the
32-wide blocks of the triangular solves.

With V = I the first frequency holds a random matrix, the second a permutation, whose inverse
is exact: it shows every swap.  Tolerance of the first: 16 n eps cond relative to the largest
element, as for any elimination with partial pivoting; the rest of Pi is zero and gives zero."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

EPS = np.finfo(np.float64).eps


@pytest.mark.parametrize("n", [1, 2, 15, 16, 17, 31, 33, 63, 64, 65, 97, 128, 129, 200, 257, 513, 1025, 1100])
def test_orders(n):
    import torch

    from coqui_amd import IAFT, ThcGW

    rng = np.random.default_rng(n)
    ia = IAFT.from_table(1000.0, "1e2.1e-15")
    ctx = ThcGW((1, 1, 1), 2, n, ia)
    eye = np.eye(n)
    A = rng.standard_normal((n, n)) + 1j * rng.standard_normal((n, n))
    P = eye[rng.permutation(n)]
    PiW = torch.zeros((ia.nw_half, 1, n, n), dtype=torch.complex128, device="cuda")
    PiW[0, 0] = torch.from_numpy(eye - A)
    PiW[1, 0] = torch.from_numpy(eye - P)
    ctx.dyson_w(PiW, eye[None].astype(complex))
    ref = np.linalg.inv(A) - eye
    tol = 16 * n * EPS * np.linalg.cond(A)
    assert np.max(np.abs(PiW[0, 0].cpu().numpy() - ref)) <= tol * (1 + np.max(np.abs(ref)))
    assert np.array_equal(PiW[1, 0].cpu().numpy(), P.T - eye)
    assert not torch.any(PiW[2:])
    ctx.close()


@pytest.mark.parametrize("n", [1, 16, 40, 200, 600, 1100])
def test_singular_last_column_is_reported(n):
    import torch

    from coqui_amd import IAFT, ThcGW, ThcgwError

    ia = IAFT.from_table(1000.0, "1e2.1e-15")
    ctx = ThcGW((1, 1, 1), 2, n, ia)
    PiW = torch.zeros((ia.nw_half, 1, n, n), dtype=torch.complex128, device="cuda")
    PiW[0, 0, n - 1, n - 1] = 1.0
    with pytest.raises(ThcgwError) as e:
        ctx.dyson_w(PiW, np.eye(n)[None].astype(complex))
    assert e.value.code == 3
    ctx.close()


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("n", [1, 16, 17, 33, 63, 65, 130, 900])
def test_hermitian_form_orders(n, precision):
    """The same by Cholesky (Hermitian V and Pi), whose triangular leaves are 32 wide in double and
    64 wide in single precision, with one or four vectors per 16 lanes (up to 16384 rows or more).
    M = 1 - L^H Pi L has its eigenvalues in [1, 1 + 1]: its factors lose 16 n eps at most."""
    import torch

    from coqui_amd import IAFT, ThcGW

    rng = np.random.default_rng(n)
    ia = IAFT.from_table(1000.0, "1e2.1e-15")
    ctx = ThcGW((1, 1, 1), 2, n, ia)
    ctx.set_flag(6, 1)
    ctx.set_flag(7, precision)
    a = rng.standard_normal((2, n, n)) + 1j * rng.standard_normal((2, n, n))
    B = a @ np.conj(np.swapaxes(a, 1, 2)) / (4 * n)
    V = B[0] + 0.5 * np.eye(n)
    Pi = -B[1] / np.linalg.norm(B[1], 2) / np.linalg.norm(V, 2)
    PiW = torch.from_numpy(np.broadcast_to(Pi, (ia.nw_half, 1, n, n)).copy()).cuda()
    ctx.dyson_w(PiW, V[None])
    ref = np.linalg.solve(np.eye(n) - V @ Pi, V) - V
    tol = 16 * n * (EPS if precision == 0 else np.finfo(np.float32).eps)
    assert np.max(np.abs(PiW.cpu().numpy() - ref)) <= tol * np.linalg.norm(V, 2)
    ctx.close()
