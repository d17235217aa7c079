"""The general-geometry kernel's epilogue at the edges of its layouts: cell
counts that leave the last group part-filled, odd numbers of entries per cell
(2D, odd N: the flat copies end in a single entry), vectors that are only 8-byte
aligned, in-place operands, cell scales with inactive cells.  Every output is
checked against the same sum formed from the kernel's own M^-1 A(src): an FMA may
round once less, <= 4 ulp of the largest term; M^-1 A(src) itself, in both
precisions, against the oracle (the bars of the operator's parity)."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

CASES = [(2, 3, 1), (2, 5, 2), (2, 3, 3), (2, 4, 4), (2, 3, 6), (2, 2, 12), (3, 3, 1), (3, 2, 2),
         (3, 3, 3), (3, 3, 4), (3, 2, 5), (3, 2, 6), (3, 2, 7), (3, 2, 8), (3, 1, 9)]


@pytest.mark.parametrize("dim,nint,k", CASES)
@pytest.mark.parametrize("off", [0, 1])
def test_epilogues(dim, nint, k, off):
    import torch

    import exwave_amd as X
    print("gen epilogue", dim, nint, k, off, flush=True)
    om = O.Mesh(dim, nint, 0, O.TRANSFORM_REFERENCE_SINE, 0.1, 3)
    rng = np.random.default_rng(7 * k + dim)
    om.set_material(rng.uniform(0.5, 2, om.n_cells), rng.uniform(0.5, 2, om.n_cells))
    op = X.WaveOperator(X.Context(0), dim, k, om.vertices, om.neighbor, om.rho, om.speed)
    N = op.n_dofs

    def vec(seed=None):
        v = torch.zeros(N + 2, dtype=torch.float64, device="cuda")
        if seed is not None:
            v.copy_(torch.from_numpy(np.random.default_rng(seed).standard_normal(N + 2)))
        return v[off:off + N]

    def near(got, want, *terms):
        if got.numel() == 0:  # (a one-cell mesh has no active cell left)
            return
        big = max(float(t.abs().max()) for t in terms)
        assert float((got - want).abs().max()) <= 4 * 2.3e-16 * big

    src, b, c, kk = vec(1), vec(2), vec(3), vec()
    op.apply(src, kk)
    want, f32 = om.apply(k, src.cpu().numpy()), vec()
    op.apply(src, f32, precision=X.FP32)
    for got, tol in ((kk, 1e-12), (f32, 2e-5 * max(1.0, (k / 8) ** 2))):
        assert np.max(np.abs(got.cpu().numpy() - want)) <= tol * np.max(np.abs(want))
    a1, a2 = 0.37, -1.3
    # the RK stage, o1 over b
    o1, o2 = vec(), vec()
    o1.copy_(b)
    op.apply_fused(src, b=o1, o1=o1, a1=a1, o2=o2, a2=a2, o2_from_o1=True)
    near(o1, b + a1 * kk, b, kk)
    near(o2, (b + a1 * kk) + a2 * kk, b, kk)
    # a c operand, o2 over c
    o1, o2 = vec(), vec()
    o2.copy_(c)
    op.apply_fused(src, b=b, o1=o1, a1=a1, c=o2, o2=o2, a2=a2)
    near(o1, b + a1 * kk, b, kk)
    near(o2, c + a2 * kk, c, kk)
    # cell scales, every third cell inactive
    s = torch.from_numpy(rng.uniform(0.5, 2, om.n_cells)).cuda()
    s[::3] = 0.0
    sc = s.repeat_interleave(N // om.n_cells)
    o1, o2 = vec(5), vec(6)
    w1, w2 = o1.clone(), o2.clone()
    op.apply_fused(src, b=b, o1=o1, a1=a1, o2=o2, a2=a2, o2_from_o1=True, cell_scale=s)
    on = sc != 0
    near(o1[on], (b + a1 * sc * kk)[on], b, 2 * kk)
    near(o2[on], (b + a1 * sc * kk + a2 * sc * kk)[on], b, 4 * kk)
    assert torch.equal(o1[~on], w1[~on]) and torch.equal(o2[~on], w2[~on])


@pytest.mark.parametrize("dim,nint,k", [(2, 5, 1), (2, 5, 3), (3, 3, 1), (3, 3, 2)])
@pytest.mark.parametrize("size", [1e-10, 1.0, 1e11])
def test_fp32_range_of_lengths(dim, nint, k, size):
    """The FP32 operator on meshes of any unit of length: the squares of a face's area
    (1e-42, 1e42 here in 3D) are outside the range of 32 bits, areas and volumes are
    not.  The bar of the FP32 parity tests."""
    import torch

    import exwave_amd as X
    print("gen lengths", dim, nint, k, size, flush=True)
    om = O.Mesh(dim, nint, 0, O.TRANSFORM_REFERENCE_SINE, 0.1, 3)
    V = np.ctypeslib.as_array(om._m.contents.vertices, shape=(om.n_cells, 1 << dim, dim))
    V *= size
    op = X.WaveOperator(X.Context(0), dim, k, om.vertices, om.neighbor, om.rho, om.speed)
    u = np.random.default_rng(3).standard_normal(op.n_dofs)
    want, got = om.apply(k, u), op.new_vector()
    op.apply(torch.from_numpy(u).cuda(), got, precision=X.FP32)
    assert np.max(np.abs(got.cpu().numpy() - want)) <= 2e-5 * np.max(np.abs(want))
