"""The Dyson step of small orders in registers: W - V = (1 - V Pi)^-1 V - V, Tr(V Pi) and
ln |Re det(1 - V Pi)| over the orders at which the kernel changes its shape, below and above the lines
to the LU form (order 64 for many matrices, 96 for few)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

EPS = np.finfo(np.float64).eps
TABLE = "1e2.1e-15"


def _ctx(kgrid, n):
    from coqui_amd import IAFT, ThcGW

    return ThcGW(kgrid, 2, n, IAFT.from_table(1000.0, TABLE))


def _dev(a):
    import torch

    return torch.from_numpy(np.ascontiguousarray(a, np.complex128)).cuda()


def _solve(A, B, dtype):
    """A^-1 B of stacks of matrices as the LU form does it: A = L U P with pivots among the columns, U with
    a unit diagonal, multiplication by reciprocals, two triangular solves, all in `dtype`."""
    A, X = A.astype(dtype), B.astype(dtype)
    at, n = np.arange(len(A)), A.shape[1]
    cols = np.broadcast_to(np.arange(n), A.shape[:2]).copy()
    for j in range(n):
        p = j + np.argmax(np.abs(A[:, j, j:].real) + np.abs(A[:, j, j:].imag), 1)
        col, c = A[at, :, p], cols[at, p]
        A[at, :, p], cols[at, p] = A[:, :, j], cols[:, j]
        A[:, :, j], cols[:, j] = col, c
        r = np.conj(A[:, j, j]) * (1.0 / (A[:, j, j].real ** 2 + A[:, j, j].imag ** 2))
        A[:, j, j + 1 :] *= r[:, None]
        A[:, j + 1 :, j + 1 :] -= A[:, j + 1 :, j, None] * A[:, j, None, j + 1 :]
        X[:, j] *= r[:, None]
        X[:, j + 1 :] -= A[:, j + 1 :, j, None] * X[:, j, None, :]
    for j in range(n - 1, 0, -1):
        X[:, :j] -= A[:, :j, j, None] * X[:, j, None, :]
    Y = np.empty_like(X)
    Y[at[:, None], cols] = X
    return Y


@pytest.mark.parametrize("size", [1.0, 10.0, 100.0])
@pytest.mark.parametrize("n", [8, 24, 40, 64, 80])
def test_error_no_larger_than_lu(n, size):
    """The mean error of 84 random matrices (V of condition 1e6, |V Pi| about `size`) against extended
    precision stays below 1.2 times that of the same step by LU in double; the mean of 84 fluctuates by a
    few percent.  V and Pi have 20 bits, so that the product V Pi is exact and all of the error is the solve's."""
    rng = np.random.default_rng(n)
    ctx = _ctx((2, 2, 1), n)
    gauss = lambda *s: rng.standard_normal(s) + 1j * rng.standard_normal(s)  # noqa: E731
    U = np.linalg.qr(gauss(4, n, n))[0]
    V = (U * np.logspace(0, -6, n)) @ np.conj(np.swapaxes(U, 1, 2))
    grid = lambda a, step: (np.round(a.real / step) + 1j * np.round(a.imag / step)) * step  # noqa: E731
    V = grid(0.5 * (V + np.conj(np.swapaxes(V, 1, 2))), 2.0**-20)
    Y = gauss(ctx.nw_half, 4, n, n)
    P = grid(-size / n * (Y @ np.conj(np.swapaxes(Y, -1, -2))), size * 2.0**-20)
    A = (np.eye(n) - V.astype(np.clongdouble) @ P.astype(np.clongdouble)).reshape(-1, n, n)
    Vs = np.broadcast_to(V, P.shape).reshape(-1, n, n)
    ref = _solve(A, Vs, np.clongdouble) - Vs
    lu = _solve((np.eye(n) - V @ P).reshape(-1, n, n), Vs, np.complex128) - Vs
    W = _dev(P)
    ctx.dyson_w(W, _dev(V))
    norm = lambda a: np.linalg.norm(a.astype(np.complex128), axis=(1, 2))  # noqa: E731
    err = lambda a: np.mean(norm(a.reshape(-1, n, n) - ref) / norm(ref))  # noqa: E731
    assert err(W.cpu().numpy()) <= 1.2 * err(lu)
    ctx.close()


@pytest.mark.parametrize("n", [1, 7, 24, 33, 64, 81, 96])
def test_weak_coupling_keeps_its_digits(n):
    """V Pi of norm 1e-6: W - V = V Pi V (1 + O(1e-6)) and ln det = -Tr V Pi (1 + O(1e-6)) to 16 n eps of
    themselves, not of V and 1."""
    rng = np.random.default_rng(n)
    ctx = _ctx((1, 1, 1), n)
    gauss = lambda: rng.standard_normal((n, n)) + 1j * rng.standard_normal((n, n))  # noqa: E731
    B, C = gauss(), gauss()
    V = B @ B.conj().T / n + np.eye(n)
    P = -(C @ C.conj().T) / n - np.eye(n)
    P *= 1e-6 / np.linalg.norm(V @ P, 2)
    x = V.astype(np.clongdouble) @ P.astype(np.clongdouble)
    W, p = np.zeros_like(x), x.copy()
    ld = np.longdouble(0.0)
    for k in range(1, 5):  # the series: 1e-24 relative at its end
        W = W + p @ V
        ld = ld - np.trace(p).real / k
        p = p @ x
    Pd = _dev(np.broadcast_to(P, (ctx.nw_half, 1, n, n)))
    tr, got = ctx.dyson_w(Pd, _dev(V[None]), with_terms=True)
    Wd = Pd.cpu().numpy()
    tol = 16 * n * EPS * np.linalg.cond(V)  # V Pi itself is a product in double
    assert np.max(np.abs(Wd - W.astype(np.complex128))) <= tol * float(np.max(np.abs(W)))
    assert np.max(np.abs(tr - complex(np.trace(x)))) <= tol * float(abs(np.trace(x)))
    assert np.max(np.abs(got - float(ld))) <= tol * float(abs(ld))
    ctx.close()


def _check(ctx, A, rows, tol_scale=1.0):
    """Stacks (nw_half, nk, n, n) of A with V = 1: W, trace and determinant of the matrices `rows`."""
    n = A.shape[-1]
    eye = np.eye(n)
    P = _dev(eye - A)
    tr, ld = ctx.dyson_w(P, _dev(np.broadcast_to(eye, (A.shape[1], n, n))), with_terms=True)
    W, a = P.cpu().numpy().reshape(-1, n, n), A.reshape(-1, n, n)
    for b in rows:
        tol = 16 * n * EPS * np.linalg.cond(a[b]) * tol_scale
        ref = np.linalg.inv(a[b]) - eye
        sign, logabs = np.linalg.slogdet(a[b])
        assert np.max(np.abs(W[b] - ref)) <= tol * (1 + np.max(np.abs(ref)))
        assert abs(tr[b] - np.trace(eye - a[b])) <= 16 * n * EPS * np.sum(np.abs(eye - a[b]))
        # ln |Re det|: an error of the phase counts with its tangent
        assert abs(ld[b] - (logabs + np.log(abs(sign.real)))) <= tol * (1 + abs(logabs) + abs(sign.imag / sign.real))


@pytest.mark.parametrize("n", [1, 2, 8, 9, 15, 16, 17, 31, 32, 33, 47, 48, 49, 63, 64, 65, 80, 95, 96, 97, 128])
def test_orders(n):
    """A random matrix (a determinant of any phase), an odd and an even permutation."""
    rng = np.random.default_rng(n)
    ctx = _ctx((1, 1, 1), n)
    A = np.broadcast_to(np.eye(n), (ctx.nw_half, 1, n, n)).astype(np.complex128)
    A[0, 0] = rng.standard_normal((n, n)) + 1j * rng.standard_normal((n, n))
    A[1, 0] = np.eye(n)[np.roll(np.arange(n), 1)]
    A[2, 0] = A[1, 0] @ A[1, 0]
    _check(ctx, A, range(4))
    ctx.close()


@pytest.mark.parametrize("n", [1, 8, 15, 16, 17, 24, 25, 32, 33, 80])
def test_many(n):
    """1344 matrices: one wave each up to order 32, the LU form at order 80."""
    rng = np.random.default_rng(n)
    ctx = _ctx((4, 4, 4), n)
    A = rng.standard_normal((ctx.nw_half, 64, n, n)) + 1j * rng.standard_normal((ctx.nw_half, 64, n, n))
    _check(ctx, A + 2.0 * np.sqrt(n) * np.eye(n), range(0, ctx.nw_half * 64, 7))
    ctx.close()


@pytest.mark.parametrize("n", [20, 72])
def test_chunks_of_any_size_give_the_same_bits(n):
    import torch

    rng = np.random.default_rng(n)
    ctx = _ctx((2, 2, 2), n)
    B = rng.standard_normal((8, n, n)) + 1j * rng.standard_normal((8, n, n))
    V = _dev(B @ np.conj(np.swapaxes(B, 1, 2)) / n)
    P = _dev(np.broadcast_to(-0.3 * V.cpu().numpy(), (ctx.nw_half, 8, n, n)))
    got = []
    for chunk in (0, 5, 8):
        ctx.set_flag(3, chunk)
        W = P.clone()
        got.append((W, *ctx.dyson_w(W, V, with_terms=True)))
    for W, tr, ld in got[1:]:
        assert torch.equal(W, got[0][0])
        assert np.array_equal(tr, got[0][1]) and np.array_equal(ld, got[0][2])
    ctx.close()
