"""The general-geometry kernel on both sides of the line between its small groups
(launches of few full groups) and its full ones: the operator
against the oracle, and a two-output sweep with cell scales, on vectors that are only
8-byte aligned, against the same sums formed from it."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim,k,nint", [
    (2, 3, 45), (2, 3, 46), (2, 4, 39), (2, 4, 40), (2, 7, 31), (2, 7, 32), (2, 12, 22), (2, 12, 23),
    (3, 2, 9), (3, 2, 10), (3, 3, 7), (3, 3, 8), (3, 4, 6), (3, 4, 7)])
def test_both_sides(dim, k, nint):
    import torch

    import exwave_amd as X
    print("gen small", dim, k, nint, flush=True)
    om = O.Mesh(dim, nint, 0, O.TRANSFORM_REFERENCE_SINE, 0.1, 3)
    rng = np.random.default_rng(5 * k + dim)
    om.set_material(rng.uniform(0.5, 2, om.n_cells), rng.uniform(0.5, 2, om.n_cells))
    op = X.WaveOperator(X.Context(0), dim, k, om.vertices, om.neighbor, om.rho, om.speed)
    assert not op.is_cartesian
    N = op.n_dofs
    u, b = rng.standard_normal(N), rng.standard_normal(N)
    want = om.apply(k, u)
    scale = rng.uniform(0.5, 2, om.n_cells)
    scale[1::3] = 0.0
    s = np.repeat(scale, N // om.n_cells)

    def dev(a):
        t = torch.zeros(N + 1, dtype=torch.float64, device="cuda")
        t[1:] = torch.from_numpy(a)
        return t[1:]

    a1, a2 = 0.0173, -0.0061
    # the bars of the operator's parity (FP32: scaled by degree above 8)
    for prec, tol in ((X.FP64, 1e-12), (X.FP32, 2e-5 * max(1.0, (k / 8) ** 2))):
        o1, o2 = dev(b), dev(b)
        op.apply_fused(dev(u), b=dev(0 * b), o1=o1, a1=1.0, precision=prec)
        assert np.max(np.abs(o1.cpu().numpy() - want)) <= tol * np.max(np.abs(want))
        o1 = dev(b)
        op.apply_fused(dev(u), b=dev(b), o1=o1, a1=a1, o2=o2, a2=a2, o2_from_o1=True,
                       cell_scale=torch.from_numpy(scale).cuda(), precision=prec)
        on = s != 0
        w1 = b + a1 * s * want
        w2 = w1 + a2 * s * want
        for got, w in ((o1, w1), (o2, w2)):
            assert np.max(np.abs(got.cpu().numpy() - w)[on]) <= tol * np.max(np.abs(want))
            assert np.array_equal(got.cpu().numpy()[~on], b[~on])
