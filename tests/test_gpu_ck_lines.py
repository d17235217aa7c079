"""The Cauchy-Kowalevski integral on box cells (ader_ck_lines_kernel, one lane per
line, or ader_ck_kernel, one lane per node) against the oracle: cells with a different size in
each direction, varying media, groups that hold several cells with the last one
part-filled, odd numbers of entries per cell, vectors that start on an odd 8 bytes,
with and without the given first derivative, on an interval away from its
expansion time; nothing outside the output's cells is written."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim,k,nint", [
    (2, 1, 5), (2, 2, 5), (2, 3, 3), (2, 4, 5), (2, 5, 3), (2, 7, 3), (2, 9, 3), (2, 11, 2),
    (2, 12, 3), (3, 1, 3), (3, 2, 3), (3, 3, 3), (3, 4, 2), (3, 5, 2), (3, 6, 2), (3, 9, 2),
    (2, 6, 3), (2, 8, 3), (2, 10, 2), (3, 7, 2), (3, 8, 2)])
def test_ck_lines_vs_oracle(dim, k, nint):
    import torch

    import exwave_amd as X
    print("ck lines", dim, k, nint, flush=True)
    om = O.Mesh(dim, nint, 0, 0, 0.0, 2)
    V = np.ctypeslib.as_array(om._m.contents.vertices, shape=(om.n_cells, 1 << dim, dim))
    V *= np.array([1.0, 0.6, 1.7][:dim])
    rng = np.random.default_rng(41)
    om.set_material(rng.uniform(0.5, 2.0, om.n_cells), rng.uniform(0.5, 2.0, om.n_cells))
    op = X.WaveOperator(X.Context(0), dim, k, om.vertices, om.neighbor, om.rho, om.speed)
    assert op.is_cartesian
    N = om.n_dofs(k)
    u, rec = rng.standard_normal(N), rng.standard_normal(N)
    t2, t1, te = 0.011, 0.004, 0.002

    def dev(a, off):
        t = torch.zeros(N + 4, dtype=torch.float64, device="cuda")
        t[off:off + N] = torch.from_numpy(a)
        return t[off:off + N]

    for off in (0, 1):
        for r in (None, rec):
            want = om.ader_ck(k, u, r, t2, t1, te)
            full = torch.full((N + 4,), 7.0, dtype=torch.float64, device="cuda")
            op.ader_ck(dev(u, off), None if r is None else dev(r, 1 - off), t2, t1, te,
                       full[off + 1:off + 1 + N])
            got = full.cpu().numpy()
            # a value is a chain of at most some hundred roundings over terms of the
            # size of the largest entries: far below 1e-12 of the maximum
            assert np.max(np.abs(got[off + 1:off + 1 + N] - want)) <= 1e-12 * np.max(np.abs(want))
            assert np.all(got[:off + 1] == 7.0) and np.all(got[off + 1 + N:] == 7.0)


# (the line form runs from a number of cells on that depends on degree and
# precision: one launch below it and one above, for every degree that has one)
@pytest.mark.parametrize("dim,k,fp32,below,above", [
    (2, 4, 0, 50, 57), (2, 6, 0, 39, 41), (2, 7, 0, 35, 37), (2, 8, 0, 55, 56), (2, 9, 0, 45, 46),
    (2, 10, 0, 45, 46), (2, 11, 0, 35, 36), (3, 3, 0, 6, 7), (3, 4, 0, 7, 8), (3, 6, 0, 7, 8),
    (3, 7, 0, 7, 8), (2, 4, 1, 100, 102), (2, 5, 1, 84, 86), (2, 6, 1, 79, 81), (2, 7, 1, 71, 73),
    (2, 8, 1, 61, 63), (2, 9, 1, 127, 129),
    (3, 4, 1, 12, 13), (3, 6, 1, 10, 11), (3, 7, 1, 9, 10)])
def test_ck_forms_vs_oracle(dim, k, fp32, below, above):
    """Both forms around the line between them; intervals of a tenth of h / k^2, so
    that no term outgrows the state: at most some hundred roundings of the size of
    the largest entry (1e-12, with the FP32 operator 160 x 2^-24 = 1e-5).  (FP32
    stops at degree 9: the tenth derivative of random values, which either form
    holds before the power of the time step scales it, passes 3e38.)"""
    import torch

    import exwave_amd as X
    ctx = X.Context(0)
    for nint in (below, above):
        print("ck forms", dim, k, fp32, nint, flush=True)
        om = O.Mesh(dim, nint, 0, 0, 0.0, 2)
        rng = np.random.default_rng(43)
        om.set_material(rng.uniform(0.5, 2.0, om.n_cells), rng.uniform(0.5, 2.0, om.n_cells))
        op = X.WaveOperator(ctx, dim, k, om.vertices, om.neighbor, om.rho, om.speed)
        u, rec = rng.standard_normal((2, om.n_dofs(k)))
        s = 0.1 / (nint * k * k)
        got = op.new_vector()
        for r in (None, rec * nint):
            want = om.ader_ck(k, u, r, 1.1 * s, 0.4 * s, 0.2 * s)
            op.ader_ck(torch.from_numpy(u).cuda(), None if r is None else torch.from_numpy(r).cuda(),
                       1.1 * s, 0.4 * s, 0.2 * s, got, X.FP32 if fp32 else X.FP64)
            d = np.max(np.abs(got.cpu().numpy() - want))
            assert d <= (1e-5 if fp32 else 1e-12) * np.max(np.abs(want))


@pytest.mark.parametrize("dim,k,n", [(2, 1, 100), (2, 4, 60), (2, 7, 70), (3, 2, 16), (3, 4, 13),
                                     (3, 6, 11)])
def test_ck_lines_fp32_roundings(dim, k, n):
    """The FP32 operator rounds the integral's leading term no more often than the
    kernel of general cells, which runs the same mesh as soon as one vertex is off
    the grid: once when the state is read and once per term that is added.  With
    terms of a few thousandths of each other three roundings count (the third
    derivative's term is below the last bit), a fourth would raise the root mean
    square of the relative error by sqrt(4 / 3) = 1.155: the line is at sqrt(3.5 / 3),
    some tens of standard errors of the 10^5 values from both."""
    import torch

    import exwave_amd as X
    print("ck roundings", dim, k, n, flush=True)
    ctx = X.Context(0)
    V, nb = X.mesh_hypercube(dim, n)
    one = np.ones(V.shape[0])
    W = V.copy()
    W[-1, -1, 0] += 0.1 / n
    g = torch.Generator(device="cuda").manual_seed(7)
    rms = []
    for vertices in (V, W):
        op = X.WaveOperator(ctx, dim, k, vertices, nb, one, one)
        assert op.is_cartesian == (vertices is V)
        r = torch.rand((2, op.n_dofs), generator=g, dtype=torch.float64, device="cuda")
        u = torch.exp2(r[0]) * torch.sign(r[1] - 0.5)
        want, got = op.new_vector(), op.new_vector()
        dt = 2e-3 / (n * k * k)
        op.ader_ck(u, None, dt, 0.0, 0.0, want, X.FP64)
        op.ader_ck(u, None, dt, 0.0, 0.0, got, X.FP32)
        rel = ((got - want) / want).view(V.shape[0], -1)[:-1]
        rms.append(float(rel.square().mean().sqrt()))
    print("rms", rms)
    assert rms[0] <= (3.5 / 3) ** 0.5 * rms[1]
