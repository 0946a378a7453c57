"""Updates of the LU form round once at the size of the element: x - l u takes the complex product first.

With u = 2^-53, Re(a b) = 25/16 u - 19/16 u = 3/8 u.  1 - 3/8 u is 1 in double; the two real products subtracted one
after the other give (1 - 25/16 u -> 1 - 2 u), then (1 - 2 u + 19/16 u -> 1 - u).  Every other step of the
elimination is exact, so that the results are too."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

a = (25 / 16 + 19j / 16) * 2.0**-26
b = (1 + 1j) * 2.0**-27


def _step(n, A, V):
    """dyson_w for A = 1 - V Pi in the first frequency; V is its own inverse up to its first order."""
    import torch

    from coqui_amd import IAFT, ThcGW

    ia = IAFT.from_table(1000.0, "1e2.1e-15")
    ctx = ThcGW((1, 1, 1), 2, n, ia)
    eye = np.eye(n)
    Pi = (2 * eye - V) @ (eye - A)
    assert np.array_equal(V @ Pi, eye - A)
    P = torch.zeros((ia.nw_half, 1, n, n), dtype=torch.complex128, device="cuda")
    P[0, 0] = torch.from_numpy(Pi)
    _, ld = ctx.dyson_w(P, np.ascontiguousarray(V[None]), with_terms=True)
    W = P[0, 0].cpu().numpy()
    ctx.close()
    return W, ld[0]


def _eye(n):
    return np.eye(n, dtype=np.complex128)


@pytest.mark.parametrize("n", [100, 200, 520, 1030])
def test_panel(n):
    A = _eye(n)
    A[1, 0], A[0, 1] = a, b
    assert _step(n, A, _eye(n))[1] == 0.0  # ln |1 - a b|


@pytest.mark.parametrize("n", [100, 200])
def test_solve_across_panels(n):
    A = _eye(n)
    A[n - 1, 0], A[0, 1], A[n - 1, 1] = a, b, 1.0
    assert _step(n, A, _eye(n))[0][n - 1, 1].real == -1.0


@pytest.mark.parametrize("n", [100, 200])
def test_forward_solve(n):
    A, V = _eye(n), _eye(n)
    A[1, 0], V[0, 1] = a, b
    assert _step(n, A, V)[0][1, 1].real == 0.0


@pytest.mark.parametrize("n", [100, 200])
def test_backward_solve(n):
    A, V = _eye(n), _eye(n)
    A[0, 1], V[1, 2], V[0, 2] = b, a, 1.0
    assert _step(n, A, V)[0][0, 2].real == 0.0
