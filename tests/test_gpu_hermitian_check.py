"""The check of flag 10 (G(tau, k) Hermitian) sees every element of few large matrices, which several workgroups
share, as of many small ones."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kgrid,no", [((1, 1, 1), 1), ((1, 1, 1), 2), ((1, 1, 1), 63), ((1, 1, 1), 65), ((1, 1, 1), 300),
                                      ((1, 1, 1), 701), ((2, 2, 1), 130), ((4, 4, 4), 5), ((4, 4, 4), 70)])
def test_every_element_is_checked(kgrid, no):
    import torch

    from coqui_amd import IAFT, ThcGW, ThcgwError

    rng = np.random.default_rng(no)
    ctx = ThcGW(kgrid, no, 4, IAFT.from_table(1000.0, "1e2.1e-15"))
    ctx.set_flag(10, 1)
    A = torch.from_numpy(rng.standard_normal((no, no, 2))).cuda()
    A = torch.view_as_complex(A)
    G = (A + A.conj().T).expand(ctx._g()).contiguous()
    X = torch.ones(ctx._x(), dtype=torch.complex128, device="cuda") / no
    ctx.pi(G, X)
    edge = (0, no - 1)
    for t in (0, ctx.nt - 1):
        for k in (0, ctx.nk - 1):
            for i, j in [(i, j) for i in edge for j in edge] + [tuple(rng.integers(0, no, 2)) for _ in range(4)]:
                old = G[t, 0, k, i, j].clone()
                G[t, 0, k, i, j] += 1e-8j
                with pytest.raises(ThcgwError) as e:
                    ctx.pi(G, X)
                assert e.value.code == 1 and "flag 10" in str(e.value)
                G[t, 0, k, i, j] = old
    ctx.pi(G, X)
    ctx.close()
