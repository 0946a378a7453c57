"""Updates of the Matsubara inverses round once at the size of the element.

X = [[1, 0, b], [0, 1, 1], [a, 1, 1]] with u = 2^-53 and a b = (3/8 + 11/4 i) u leaves the pivot (1 - a b) - 1.
1 - 3/8 u is 1 in double, so that the pivot is -11/4 i u; the two real products 25/16 u and 19/16 u subtracted one
after the other leave -u - 11/4 i u.  With S = 0 every frequency has this X = -F, and G(tau) its inverse times the
sum of a row of the transform."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [3, 17, 40, 64, 70, 96, 100, 128])
def test_inverse(n):
    import torch

    from coqui_amd import IAFT, ThcGW

    ia = IAFT.from_table(100.0, "1e2.1e-15")
    ctx = ThcGW((1, 1, 1), n, 4, ia)
    X = np.eye(n, dtype=np.complex128)
    X[0, 2], X[2, 0] = (1 + 1j) * 2.0**-27, (25 / 16 + 19j / 16) * 2.0**-26
    X[1, 2] = X[2, 1] = 1.0
    zero = torch.zeros(ctx._g(), dtype=torch.complex128, device="cuda")
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()  # noqa: E731
    G, _ = ctx.dyson_g(dev(-X[None, None]), zero, 0.0, S=dev(0.0 * X[None, None]))
    c = np.sum(ia.Ttw_ff * (np.sqrt(2.0) / ia.beta), axis=1)
    t = np.argmax(np.abs(c))
    inv = G.cpu().numpy()[t, 0, 0, 2, 2] / c[t]
    assert abs(inv.imag * 2.75 * 2.0**-53 - 1.0) < 1e-6
    assert abs(inv.real) < 1e-6 * abs(inv.imag)
    ctx.close()
