"""The chemical potential search without overlap (Hessenberg forms, order <= 128) over the orders at
which its kernels change their shape, for matrices with and without coupling: diagonal ones and
degenerate levels have nothing to reflect in some or all columns.

N(mu) is checked against numpy at the mu that was found.  Tolerance as for the inverses: the
reflections and the elimination are backward stable, 16 n eps max cond(X)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

EPS = np.finfo(np.float64).eps
TABLE, BETA = "1e2.1e-15", 100.0


def _herm(rng, *shape):
    a = rng.standard_normal(shape) + 1j * rng.standard_normal(shape)
    return 0.5 * (a + np.conj(np.swapaxes(a, -1, -2)))


@pytest.mark.parametrize("kind", ["coupled", "diagonal", "degenerate"])
@pytest.mark.parametrize("no", [1, 2, 3, 15, 16, 17, 18, 32, 33, 48, 50, 64, 65, 80, 82, 96, 97, 127, 128, 129])
def test_orders(no, kind):
    import torch

    from coqui_amd import IAFT, ThcGW

    rng = np.random.default_rng(no)
    ia = IAFT.from_table(BETA, TABLE)
    nk = 3
    ctx = ThcGW((1, 1, nk), no, 4, ia)
    F = _herm(rng, 1, nk, no, no) / np.sqrt(no)
    H0 = 0.3 * _herm(rng, 1, nk, no, no) / np.sqrt(no)
    w = _herm(rng, 1, 1, nk, no, no) / no
    Sig = np.ascontiguousarray(0.05 * (w @ w) * -np.exp(-0.4 * ia.tau)[:, None, None, None, None])
    if kind == "diagonal":
        F = F * np.eye(no)
        H0, Sig = None, 0.0 * Sig
    elif kind == "degenerate":
        q = np.linalg.qr(F)[0]
        F = np.ascontiguousarray((q * np.round(np.linspace(-1, 1, no))) @ np.conj(np.swapaxes(q, -1, -2)))
        Sig = 1e-13 * Sig
    dev = lambda a: None if a is None else torch.from_numpy(np.ascontiguousarray(a, np.complex128)).cuda()  # noqa: E731
    target, mu_tol = 0.37 * 2 * no, 1e-6
    mu, got = ctx.update_mu(dev(F), dev(Sig), target, 0.11, H0=dev(H0), mu_tol=mu_tol)
    assert abs(got - target) < mu_tol

    s2 = np.sqrt(2.0)
    Sw = np.tensordot(ia.Twt_ff * (BETA / s2), Sig[:, 0], 1)
    iw = 1j * ia.wn_mesh_f * np.pi / BETA + mu
    X = iw[:, None, None, None] * np.eye(no) - F[0] - Sw - (0.0 if H0 is None else H0[0])
    tr = np.einsum("wkii->w", np.linalg.inv(X)) / nk
    n = -2.0 * np.real(ia.T_beta_t_ff @ ((ia.Ttw_ff * (s2 / BETA)) @ tr))
    tol = 16 * no * EPS * float(np.max(np.linalg.cond(X)))
    assert abs(got - n) <= tol * max(1.0, abs(n))
    assert abs(ctx.nelec(dev(F), dev(Sig), mu, H0=dev(H0)) - got) <= tol * max(1.0, abs(n))
    ctx.close()
