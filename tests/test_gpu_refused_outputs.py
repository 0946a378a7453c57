"""What a refused iteration leaves in the caller's arrays: Sigma stays to the bit when 1 - V Pi is singular,
Sigma and W when an input is not finite."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _system(kgrid, no, nmu, flags):
    import torch

    from coqui_amd import IAFT, ThcGW

    rng = np.random.default_rng(nmu)
    ctx = ThcGW(kgrid, no, nmu, IAFT.from_table(1000.0, "1e2.1e-15"))
    for f, v in flags.items():
        ctx.set_flag(f, v)
    nk = ctx.nk
    gauss = lambda *s: rng.standard_normal(s) + 1j * rng.standard_normal(s)  # noqa: E731
    C = np.ascontiguousarray(np.linalg.qr(gauss(nk, no, no))[0])
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()  # noqa: E731
    G = ctx.update_G(dev(C), np.tile(np.linspace(-0.4, 0.5, no), (nk, 1)))
    S = torch.full(ctx._g(), 1.5 - 2.5j, dtype=torch.complex128, device="cuda")
    W = torch.full(ctx._wqt(), 0.5 + 3.5j, dtype=torch.complex128, device="cuda")
    V = np.broadcast_to(np.eye(nmu), (nk, nmu, nmu)).astype(np.complex128)
    return ctx, G, dev(gauss(nk, nmu, no)), dev(V), S, W


@pytest.mark.parametrize("flags", [{}, {7: 0, 10: 1}, {2: 1}], ids=["plain", "hermitian-G", "one-pair-per-batch"])
@pytest.mark.parametrize("kgrid,no,nmu", [((1, 1, 1), 3, 8), ((2, 2, 1), 4, 24), ((2, 2, 2), 6, 130)])
def test_singular_leaves_sigma(kgrid, no, nmu, flags):
    import torch

    from coqui_amd import ThcgwError

    ctx, G, X, V, S, W = _system(kgrid, no, nmu, flags)
    S0 = S.clone()
    with pytest.raises(ThcgwError) as e:
        ctx.gw_iteration(G, 1e3 * X, 1e305 * V, Sigma=S, W_qt=W)  # V Pi overflows: no finite pivot
    assert e.value.code == 3
    assert torch.equal(S, S0)
    S1, W1, _ = ctx.gw_iteration(G, X, V, Sigma=S, W_qt=W)  # and the context goes on
    assert torch.isfinite(torch.view_as_real(S1)).all() and torch.isfinite(torch.view_as_real(W1)).all()
    ctx.close()


@pytest.mark.parametrize("flags", [{}, {10: 1}, {6: 1, 7: 1}, {6: 2, 7: 1, 10: 1}, {2: 1}],
                         ids=["plain", "hermitian-G", "mixed", "mixed-resolvent", "one-pair-per-batch"])
@pytest.mark.parametrize("bad", ["G", "X", "V"])
def test_nonfinite_input_leaves_both(bad, flags):
    import torch

    from coqui_amd import ThcgwError

    ctx, G, X, V, S, W = _system((2, 2, 1), 4, 24, flags)
    S0, W0 = S.clone(), W.clone()
    {"G": G, "X": X, "V": V}[bad].view(-1)[-1] = float("nan")
    with pytest.raises(ThcgwError) as e:
        ctx.gw_iteration(G, X, V, Sigma=S, W_qt=W)
    assert e.value.code == 6 and bad + "_" in str(e.value)
    assert torch.equal(S, S0) and torch.equal(W, W0)
    ctx.close()
