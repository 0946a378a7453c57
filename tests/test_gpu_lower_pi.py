"""An iteration with a Hermitian G in the resolvent form works on the lower triangles of Pi alone.  The
same steps one at a time work on whole matrices, with the same arithmetic for the lower triangles: the
results are equal to the bit.  Orders around the 16 columns that the tau -> iW transform takes at a
time, every kind of k-grid kernel, and a table whose transform is a GEMM.  The W array, which holds Pi
on the way, starts as NaN: what is not formed must not be read.

An indefinite V has no Cholesky factor and sends every matrix to the LU form, which needs all of Pi;
W = [(1 - V Pi)^-1 - 1] V is then compared with numpy, to 256 n eps of V, which it is a difference of."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

EPS = np.finfo(np.float64).eps
CASES = [
    ((1, 1, 1), 3, 15, "1e2.1e-15"),
    ((1, 1, 1), 4, 16, "1e2.1e-15"),
    ((1, 1, 1), 5, 130, "1e4.1e-15"),
    ((2, 2, 1), 4, 17, "1e2.1e-15"),
    ((2, 2, 2), 4, 33, "1e3.5e-18"),
    ((3, 3, 3), 3, 31, "1e2.1e-15"),
    ((4, 4, 4), 3, 24, "1e2.1e-15"),
]


def _system(orc, kgrid, no, nmu, table, definite):
    import torch

    from coqui_amd import IAFT, ThcGW

    rng = np.random.default_rng(nmu)
    ia, tab = IAFT.from_table(1000.0, table), orc.load_ir(1000.0, None, table=table)
    nk = kgrid[0] * kgrid[1] * kgrid[2]
    gauss = lambda *s: rng.standard_normal(s) + 1j * rng.standard_normal(s)  # noqa: E731
    C = np.linalg.qr(gauss(nk, no, no))[0]
    G = orc.update_G(tab, C, np.sort(rng.uniform(-0.5, 0.5, (nk, no)), axis=1))
    X = 0.5 * gauss(nk, nmu, no) / np.sqrt(2 * nmu)
    B = gauss(nk, nmu, nmu)
    B = B @ np.conj(np.swapaxes(B, 1, 2))
    V = B / np.linalg.norm(B, 2, axis=(1, 2))[:, None, None] + np.eye(nmu)
    if not definite:
        V[:, 0, 0] -= 4.0
    ctx = ThcGW(kgrid, no, nmu, ia)
    ctx.set_flag(6, 2)
    ctx.set_flag(10, 1)
    W = torch.full(ctx._wqt(), complex("nan"), dtype=torch.complex128, device="cuda")
    return ctx, tuple(torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in (G, X, V)), W


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("kgrid,no,nmu,table", CASES)
def test_steps(orc, kgrid, no, nmu, table, precision):
    ctx, (G, X, V), W = _system(orc, kgrid, no, nmu, table, True)
    ctx.set_flag(7, precision)
    S, W, ec = ctx.gw_iteration(G, X, V, with_ec=True, hermitize=True, W_qt=W)
    Pw = ctx.tau_to_w(ctx.pi(G, X))
    ctx.dyson_w(Pw, V)
    W1 = ctx.w_to_tau(Pw)
    assert np.array_equal(W.cpu().numpy(), W1.cpu().numpy())
    assert np.array_equal(S.cpu().numpy(), ctx.sigma(G, W1, X, hermitize=True).cpu().numpy())
    assert ec == ctx.rpa_ec(ctx.tau_to_w(ctx.pi(G, X)), V)
    ctx.close()


@pytest.mark.parametrize("kgrid,no,nmu,table", CASES)
def test_indefinite_v(orc, kgrid, no, nmu, table):
    ctx, (G, X, V), W = _system(orc, kgrid, no, nmu, table, False)
    _, W, _ = ctx.gw_iteration(G, X, V, with_ec=True, hermitize=True, W_qt=W)
    P = ctx.tau_to_w(ctx.pi(G, X))
    v, p = V.cpu().numpy(), P.cpu().numpy()
    eye = np.eye(nmu)
    P[:] = P.new_tensor((np.linalg.inv(eye - v @ p) - eye) @ v)
    ref = ctx.w_to_tau(P).cpu().numpy()
    assert np.max(np.abs(W.cpu().numpy() - ref)) <= 256 * nmu * EPS * np.max(np.abs(v))
    ctx.close()
