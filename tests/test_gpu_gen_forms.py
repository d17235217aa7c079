"""The operator on general cells on both sides of every line between the form with
one lane per node and the line form (they depend on degree, precision and whether
the launch is a plain sweep; dg_operator_gen.hpp lists them): single sweeps and two-output sweeps
with cell scales and a c operand, on vectors that are only 8-byte aligned, against
the oracle.  Meshes whose last group is part-filled wherever a group has several cells."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

CASES = [(2, 1, 0, 173), (2, 1, 0, 174), (2, 1, 0, 224), (2, 1, 0, 257), (2, 3, 0, 77),
         (2, 3, 0, 95), (2, 3, 0, 179), (2, 4, 0, 34), (2, 4, 0, 35), (2, 4, 0, 77),
         (2, 4, 0, 79), (2, 5, 0, 24), (2, 5, 0, 25), (2, 5, 0, 86), (2, 5, 0, 87),
         (2, 5, 0, 104), (2, 5, 0, 106), (2, 6, 0, 74), (2, 6, 0, 76), (2, 7, 0, 63),
         (2, 7, 0, 65), (2, 7, 0, 85), (2, 8, 0, 54), (2, 8, 0, 57), (2, 9, 0, 54),
         (2, 9, 0, 55), (2, 10, 0, 109), (2, 10, 0, 111), (2, 11, 0, 94), (2, 11, 0, 96),
         (2, 12, 0, 96), (3, 5, 0, 13), (3, 5, 0, 14), (3, 6, 0, 8), (3, 6, 0, 9), (3, 7, 0, 7),
         (3, 7, 0, 8), (3, 8, 0, 12), (3, 8, 0, 13), (3, 9, 0, 3), (2, 3, 1, 78), (2, 3, 1, 123),
         (2, 3, 1, 131), (2, 4, 1, 104), (2, 4, 1, 106), (2, 5, 1, 86), (2, 5, 1, 88),
         (2, 6, 1, 63), (2, 6, 1, 65), (2, 7, 1, 59), (2, 7, 1, 61), (2, 8, 1, 90),
         (2, 8, 1, 92), (2, 9, 1, 127), (2, 9, 1, 129), (2, 11, 1, 109), (2, 11, 1, 111),
         (2, 12, 1, 30), (3, 5, 1, 9), (3, 5, 1, 10), (3, 5, 1, 13), (3, 6, 1, 8), (3, 6, 1, 9),
         (3, 7, 1, 15), (3, 7, 1, 16), (3, 8, 1, 10), (3, 8, 1, 11), (3, 9, 1, 7), (3, 9, 1, 8),
         (2, 1, 0, 154), (2, 1, 0, 155), (2, 3, 0, 128), (2, 3, 0, 129), (2, 4, 0, 71),
         (2, 4, 0, 72), (2, 5, 0, 71), (2, 5, 0, 72), (2, 7, 0, 59), (2, 7, 0, 61), (2, 8, 0, 50),
         (2, 8, 0, 51), (2, 9, 0, 49), (2, 9, 0, 51), (2, 11, 0, 110), (3, 7, 0, 6),
         (3, 8, 0, 11), (2, 3, 1, 129), (2, 5, 1, 71), (2, 5, 1, 72), (2, 8, 1, 79), (2, 8, 1, 80),
         (2, 8, 1, 84), (2, 8, 1, 85), (2, 8, 1, 95), (2, 8, 1, 96), (2, 8, 1, 114), (2, 8, 1, 115),
         (2, 9, 1, 73), (2, 9, 1, 74), (2, 9, 1, 78), (2, 9, 1, 79), (2, 9, 1, 120), (2, 9, 1, 121),
         (2, 11, 1, 98), (2, 11, 1, 99), (3, 8, 1, 9), (3, 9, 1, 6)]


@pytest.mark.parametrize("dim,k,fp32,nint", CASES)
def test_forms(dim, k, fp32, nint):
    import torch

    import exwave_amd as X
    print("gen forms", dim, k, fp32, nint, flush=True)
    om = O.Mesh(dim, nint, 0, O.TRANSFORM_REFERENCE_SINE, 0.1, 3)
    rng = np.random.default_rng(11 * k + dim)
    om.set_material(rng.uniform(0.5, 2, om.n_cells), rng.uniform(0.5, 2, om.n_cells))
    op = X.WaveOperator(X.Context(0), dim, k, om.vertices, om.neighbor, om.rho, om.speed)
    assert not op.is_cartesian
    N = op.n_dofs
    u, b = rng.standard_normal((2, N))
    want = om.apply(k, u)
    scale = rng.uniform(0.5, 2, om.n_cells)
    scale[1::3] = 0.0

    def dev(a):
        t = torch.zeros(N + 1, dtype=torch.float64, device="cuda")
        t[1:] = torch.from_numpy(a)
        return t[1:]

    # the bars of the operator's parity (FP32: scaled by degree above 8)
    prec, tol = (X.FP32, 2e-5 * max(1.0, (k / 8) ** 2)) if fp32 else (X.FP64, 1e-12)
    bar = tol * np.max(np.abs(want))
    o1, o2, s = dev(b), dev(b), np.repeat(scale, N // om.n_cells)
    op.apply(dev(u), o1, precision=prec)
    assert np.max(np.abs(o1.cpu().numpy() - want)) <= bar
    a1, a2 = 0.0173, -0.0061
    op.apply_fused(dev(u), b=dev(u), o1=o1, a1=a1, c=o2, o2=o2, a2=a2,
                   cell_scale=torch.from_numpy(scale).cuda(), precision=prec)
    on = s != 0
    assert np.max(np.abs(o1.cpu().numpy() - (u + a1 * s * want))[on]) <= bar
    assert np.max(np.abs(o2.cpu().numpy() - (b + a2 * s * want))[on]) <= bar
    assert np.array_equal(o2.cpu().numpy()[~on], b[~on])
