"""The complex-FP64 products at the edges of their tiles and K chunks: X O X^H (N,N and N,C) and
X^H O X (C,N and N,N) through the projection entry points, against numpy.

The kernel covers a matrix with 64 x 64 tiles whose 32-wide halves are left out where they lie
outside, and takes K in chunks of 8 with a pipelined loop from the fourth full chunk on.  The
bound is the rounding of two complex products of length K, element by element: a real product
of length K errs by at most K eps |A||B|, a complex one by a few of those, three-product
arithmetic included (at most 8 per product), so 8 (2 K + 8) eps (|X||O||X^H|)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

EPS = np.finfo(np.float64).eps


def _cg(rng, *shape):
    return rng.standard_normal(shape) + 1j * rng.standard_normal(shape)


@pytest.mark.parametrize("nmu", [1, 15, 31, 32, 33, 48, 63, 64, 65, 97, 129])
@pytest.mark.parametrize("no", [1, 7, 8, 9, 25, 33, 40, 41, 65])
def test_projection_edges(no, nmu):
    import torch

    from coqui_amd import IAFT, ThcGW

    rng = np.random.default_rng(1000 * no + nmu)
    ctx = ThcGW((1, 2, 1), no, nmu, IAFT.from_table(1000.0, "1e2.1e-15"))
    X, O, P = _cg(rng, 2, nmu, no), _cg(rng, 3, 2, no, no), _cg(rng, 3, 2, nmu, nmu)
    Xh = np.conj(np.swapaxes(X, 1, 2))
    aX = np.abs(X)
    want_p, scale_p = (X @ O) @ Xh, (aX @ np.abs(O)) @ np.swapaxes(aX, 1, 2)
    want_a, scale_a = (Xh @ P) @ X, (np.swapaxes(aX, 1, 2) @ np.abs(P)) @ aX
    Xd, Od, Pd = (torch.from_numpy(a).cuda() for a in (X, O, P))
    try:
        for g3 in (0, 1):
            ctx.set_flag(12, g3)
            got_p = ctx.primary_to_aux(Xd, Od).cpu().numpy()
            got_a = ctx.aux_to_primary(Xd, Pd).cpu().numpy()
            assert np.all(np.abs(got_p - want_p) <= 8 * (2 * no + 8) * EPS * scale_p), (no, nmu, g3)
            assert np.all(np.abs(got_a - want_a) <= 8 * (2 * nmu + 8) * EPS * scale_a), (no, nmu, g3)
    finally:
        ctx.set_flag(12, 0)
        ctx.close()
