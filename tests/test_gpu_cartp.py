"""Two-output sweeps on many small box cells run dg_operator_cartp_kernel, single
ones dg_operator_cart_kernel.  Both evaluate the same expressions with the same
FMAs, so a fused sweep (o1 = b + a1 k; o2 = o1 + a2 k or c + a2 k) gives the bits of
the single-output sweeps it stands for: at the smallest launches that take the
pair kernel, with a part-filled last group, odd numbers of entries per cell, 8-byte
aligned vectors, every boundary id, varying media, in-place operands, cell
scales with inactive cells, and both operator precisions."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CASES = [(2, 1, 9), (2, 2, 74), (2, 3, 65), (2, 4, 56), (2, 5, 51), (2, 9, 40), (2, 12, 33),
         (3, 1, 5), (3, 2, 13)]
# the smallest launches of the degrees whose line lies higher than these
CASES += [(2, 2, 135), (2, 3, 95), (2, 4, 147), (2, 5, 71), (3, 2, 17), (3, 2, 23)]
FP32_ONLY = [(2, 9, 125), (2, 11, 36), (3, 4, 28), (3, 5, 8), (2, 7, 46), (2, 8, 43), (3, 4, 9), (3, 5, 7)]


@pytest.mark.parametrize("dim,k,n", [(2, 1, 9), (2, 3, 95), (2, 4, 147), (2, 5, 71), (3, 1, 5),
                                     (3, 2, 17)])
@pytest.mark.parametrize("integ", ["LSRK45R2", "LSRK45R3"])
def test_time_step_matches_oracle(dim, k, n, integ):
    """A time step whose stages are such launches, with two outputs and (three
    registers) with three: the bar of the integrators' parity tests, 1e-12."""
    import torch

    import exwave_amd as X
    import oracle as O
    print("cart pairs step", dim, k, n, integ, flush=True)
    om = O.Mesh(dim, n, 0, 0, 0.0, 3)
    rng = np.random.default_rng(9 * k + dim)
    om.set_material(rng.uniform(0.5, 2.0, om.n_cells), rng.uniform(0.5, 2.0, om.n_cells))
    op = X.WaveOperator(X.Context(0), dim, k, om.vertices, om.neighbor, om.rho, om.speed)
    assert op.is_cartesian
    u = rng.standard_normal(op.n_dofs)
    dt = 0.1 / k ** 1.5 * om.min_vertex_distance_over_c
    vn, vnp = u.copy(), np.zeros_like(u)
    om.time_step(k, getattr(O, integ), dt, vn, vnp)
    dn, dnp = torch.from_numpy(u).cuda(), op.new_vector()
    which = getattr(X, integ)
    op.time_step(which, dt, dn, dnp, op.new_vector(max(1, op.work_vectors(which))))
    assert np.max(np.abs(dnp.cpu().numpy() - vnp)) <= 1e-12 * np.max(np.abs(vnp))


@pytest.mark.parametrize("dim,k,n", [(2, 1, 6), (2, 3, 64), (3, 1, 4), (3, 2, 10)])
def test_hanging_step_matches_oracle(dim, k, n):
    """The same on box meshes with hanging faces (the sweep leaves them to
    nc_face_kernel): the bar of the hanging-face parity tests."""
    import torch

    import exwave_amd as X
    import oracle as O
    print("cart pairs hanging", dim, k, n, flush=True)
    rng = np.random.default_rng(9 * k + dim)
    om = O.Mesh.box_refined(dim, n, (rng.uniform(size=(n,) * dim) < 0.5).astype(np.int32), 0, 0.0, 2)
    om.set_material(rng.uniform(0.5, 2.0, om.n_cells), rng.uniform(0.5, 2.0, om.n_cells))
    op = X.WaveOperator(X.Context(0), dim, k, om.vertices, om.neighbor, om.rho, om.speed,
                        hanging=om.hanging)
    u = rng.standard_normal(op.n_dofs)
    dt = 0.1 / k ** 1.5 * om.min_vertex_distance_over_c
    vn, vnp = u.copy(), np.zeros_like(u)
    om.time_step(k, O.LSRK45R2, dt, vn, vnp)
    dn, dnp = torch.from_numpy(u).cuda(), op.new_vector()
    op.time_step(X.LSRK45R2, dt, dn, dnp, op.new_vector(max(1, op.work_vectors(X.LSRK45R2))))
    assert np.max(np.abs(dnp.cpu().numpy() - vnp)) <= 1e-12 * np.max(np.abs(vnp))


@pytest.mark.parametrize("dim,k,n,fp32", [c + (False,) for c in CASES] +
                         [c + (True,) for c in CASES + FP32_ONLY])
def test_pairs_match_staged(dim, k, n, fp32):
    import torch

    import exwave_amd as X
    print("cart pairs", dim, k, n, fp32, flush=True)
    V, nb = X.mesh_hypercube(dim, n, 0, X.TRANSFORM_NONE, 0.0, 2)
    x = V.mean(axis=1)
    nb = np.where(nb < 0, -(1 + (np.arange(len(V)) % 3))[:, None], nb)
    rho, c_ = 1.0 + 0.3 * np.sin(9 * x[:, 0]), 1.5 + 0.4 * np.cos(7 * x[:, -1])
    op = X.WaveOperator(X.Context(0), dim, k, V, nb, rho, c_)
    assert op.is_cartesian
    prec = X.FP32 if fp32 else X.FP64
    N = op.n_dofs

    def vec(off, seed=None):
        v = torch.zeros(N + 2, dtype=torch.float64, device="cuda")
        if seed is not None:
            v.copy_(torch.from_numpy(np.random.default_rng(seed).standard_normal(N + 2)))
        return v[off:off + N]

    a1, a2 = 0.0173, -0.0061
    scale = torch.from_numpy(np.random.default_rng(3).uniform(0.5, 2, op.n_cells)).cuda()
    scale[1::4] = 0.0
    for off in (0, 1):
        for s in (None, scale):
            src, b, c = vec(off, 1), vec(off, 2), vec(off, 3)
            w1, w2, w3 = vec(off, 4), vec(off, 5), vec(off, 5)
            op.apply_fused(src, b=b, o1=w1, a1=a1, cell_scale=s, precision=prec)
            op.apply_fused(src, b=w1, o1=w2, a1=a2, cell_scale=s, precision=prec)
            op.apply_fused(src, b=c, o1=w3, a1=a2, cell_scale=s, precision=prec)
            o1, o2 = vec(off, 4), vec(off, 5)
            if s is None:  # in place, as the RK stages run
                o1.copy_(b)
            op.apply_fused(src, b=o1 if s is None else b, o1=o1, a1=a1, o2=o2, a2=a2,
                           o2_from_o1=True, cell_scale=s, precision=prec)
            assert torch.equal(o1, w1) and torch.equal(o2, w2)
            o1, o2 = vec(off, 4), vec(off, 5)
            if s is None:
                o2.copy_(c)
            op.apply_fused(src, b=b, o1=o1, a1=a1, c=o2 if s is None else c, o2=o2, a2=a2,
                           cell_scale=s, precision=prec)
            assert torch.equal(o1, w1) and torch.equal(o2, w3)
