"""Quasiparticle energies over the numbers at which the solver changes its shape: fits of 2 points to
half the frequencies (16 lanes hold one to two points each) and states that do not fill a wave (4 per
wave), near and far roots (bracketing tries 16 steps of 0.01 Ha at a time).

Both sides end at |residual| <= 1e-8 Ha of their own continued fraction; 1e-6 allows for a residual that
is as steep as 1/50 and for an end point that rounding moves by a few halvings."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("weight", [0.03, 0.6])
@pytest.mark.parametrize("nfit", [2, 3, 8, 15, 16, 17, 18])
@pytest.mark.parametrize("nk,no", [(1, 1), (1, 3), (2, 4), (3, 7)])
def test_states(orc, nk, no, nfit, weight):
    import torch

    from coqui_amd import IAFT, ThcGW

    beta, table = 100.0, "1e2.1e-15"
    rng = np.random.default_rng(100 * nfit + 10 * nk + no)
    ia, tab = IAFT.from_table(beta, table), orc.load_ir(beta, None, table=table)
    ctx = ThcGW((1, 1, nk), no, 4, ia)
    E = np.sort(rng.uniform(-0.6, 0.6, (nk, no)), axis=1)
    C = np.linalg.qr(rng.standard_normal((nk, no, no)) + 1j * rng.standard_normal((nk, no, no)))[0]
    H = (C * E[:, None, :]) @ np.conj(np.swapaxes(C, 1, 2))
    # Sigma_nn(iw) = a pole below and one above the levels; its other matrix elements are zero
    g = np.stack([-np.exp(-ia.tau * e) / (1 + np.exp(-beta * e)) for e in (-2.3, 2.1)], axis=1)
    sig = np.einsum("tp,pkn->tkn", g, weight * rng.uniform(0.5, 1.0, (2, nk, no)))
    Sig = np.ascontiguousarray(((C * sig[:, :, None, :]) @ np.conj(np.swapaxes(C, 1, 2)))[:, None])
    args = dict(mu=0.0, nfit=nfit, eta=1e-4, tol=1e-8)
    got = ctx.solve_qp(torch.from_numpy(Sig).cuda(), C, H, E, **args)
    assert np.max(np.abs(got - orc.solve_qp(tab, Sig, C, H, E, **args))) < 1e-6
    ctx.close()
