"""G(iw) = [(iw_n + mu) S - H0 - F - Sigma(iw_n)]^-1 over the orders at which the inversion changes
its shape: the 16-row blocks of the register kernel, its change of thread grid after order 96
and of method after 128.  Checked through G(tau) and the electron number against numpy.

Tolerance: an inverse by elimination with partial pivoting errs by a small multiple of
n eps cond(X) relative to its largest element; the transforms that follow are sums of some
tens of terms.  16 n eps max cond(X), with cond from numpy."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

EPS = np.finfo(np.float64).eps
TABLE, BETA = "1e2.1e-15", 100.0


def _herm(rng, *shape):
    a = rng.standard_normal(shape) + 1j * rng.standard_normal(shape)
    return 0.5 * (a + np.conj(np.swapaxes(a, -1, -2)))


@pytest.mark.parametrize("with_s", [False, True])
@pytest.mark.parametrize("no", [1, 2, 15, 16, 17, 32, 33, 48, 49, 64, 65, 80, 81, 96, 97, 112, 128, 129])
def test_orders(no, with_s):
    import torch

    from coqui_amd import IAFT, ThcGW

    rng = np.random.default_rng(no + 1000 * with_s)
    ia = IAFT.from_table(BETA, TABLE)
    nk, mu = 2, 0.13
    ctx = ThcGW((1, 1, nk), no, 4, ia)
    F = _herm(rng, 1, nk, no, no) / np.sqrt(no)
    H0 = 0.3 * _herm(rng, 1, nk, no, no) / np.sqrt(no) if with_s else None
    S = np.eye(no) + 0.1 * _herm(rng, 1, nk, no, no) / no if with_s else None
    w = _herm(rng, 1, 1, nk, no, no) / no
    Sig = np.ascontiguousarray(0.05 * (w @ w) * -np.exp(-0.4 * ia.tau)[:, None, None, None, None])
    s2 = np.sqrt(2.0)
    Twt, Ttw = ia.Twt_ff * (BETA / s2), ia.Ttw_ff * (s2 / BETA)
    Sw = np.tensordot(Twt, Sig[:, 0], 1)
    iw = 1j * ia.wn_mesh_f * np.pi / BETA + mu
    Sm = np.broadcast_to(np.eye(no), (nk, no, no)) if S is None else S[0]
    X = iw[:, None, None, None] * Sm - F[0] - Sw - (0.0 if H0 is None else H0[0])
    tol = 16 * no * EPS * float(np.max(np.linalg.cond(X)))
    Gw = np.linalg.inv(X)
    G = np.tensordot(Ttw, Gw, 1)
    n = -2.0 * np.real(ia.T_beta_t_ff @ (Ttw @ (np.einsum("wkij,kji->w", Gw, Sm) / nk)))
    dev = lambda a: None if a is None else torch.from_numpy(np.ascontiguousarray(a, np.complex128)).cuda()  # noqa: E731
    args = dict(H0=dev(H0), S=dev(S))
    g, _ = ctx.dyson_g(dev(F), dev(Sig), mu, **args)
    got = ctx.nelec(dev(F), dev(Sig), mu, **args)
    assert np.max(np.abs(g.cpu().numpy()[:, 0] - G)) <= tol * np.max(np.abs(G))
    assert abs(got - n) <= tol * max(1.0, abs(n))
    ctx.close()


@pytest.mark.parametrize("no", [1, 16, 40, 97, 130])
def test_singular_matrix_is_reported(no):
    """A zero overlap and Hamiltonian make every X zero."""
    import torch

    from coqui_amd import IAFT, ThcGW, ThcgwError

    ia = IAFT.from_table(BETA, TABLE)
    ctx = ThcGW((1, 1, 1), no, 4, ia)
    z = torch.zeros((1, 1, no, no), dtype=torch.complex128, device="cuda")
    sig = torch.zeros((ia.nt, 1, 1, no, no), dtype=torch.complex128, device="cuda")
    with pytest.raises(ThcgwError) as e:
        ctx.dyson_g(z, sig, 0.0, S=z)
    assert e.value.code == 3
    ctx.close()


@pytest.mark.parametrize("n", [1, 7, 8, 9, 15, 16, 17, 24, 25, 31, 32, 33])
def test_many_small_matrices(n):
    """The same kernel with one wave per matrix (order <= 32, 1024 matrices or more): G of 2560
    matrices and W of 1344, equal at every frequency."""
    import torch

    from coqui_amd import IAFT, ThcGW

    rng = np.random.default_rng(n)
    ia = IAFT.from_table(BETA, TABLE)
    nk = 64
    ctx = ThcGW((4, 4, 4), n, n, ia)
    assert ctx.nw_half * nk >= 1024
    F = _herm(rng, 1, nk, n, n) / np.sqrt(n)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a, np.complex128)).cuda()  # noqa: E731
    g, _ = ctx.dyson_g(dev(F), dev(np.zeros((ia.nt, 1, nk, n, n))), 0.13)
    iw = 1j * ia.wn_mesh_f * np.pi / BETA + 0.13
    X = iw[:, None, None, None] * np.eye(n) - F[0]
    G = np.tensordot(ia.Ttw_ff * (np.sqrt(2.0) / BETA), np.linalg.inv(X), 1)
    tol = 16 * n * EPS * float(np.max(np.linalg.cond(X)))
    assert np.max(np.abs(g.cpu().numpy()[:, 0] - G)) <= tol * np.max(np.abs(G))

    eye = np.eye(n)
    A = rng.standard_normal((nk, n, n)) + 1j * rng.standard_normal((nk, n, n))
    P = np.broadcast_to(eye - A, (ctx.nw_half, nk, n, n))
    PiW = dev(P)
    ctx.dyson_w(PiW, dev(np.broadcast_to(eye, (nk, n, n))))
    ref = np.linalg.inv(A) - eye
    tol = 16 * n * EPS * float(np.max(np.linalg.cond(A)))
    assert np.max(np.abs(PiW.cpu().numpy() - ref)) <= tol * (1 + np.max(np.abs(ref)))
    ctx.close()
