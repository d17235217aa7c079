"""The output tick's kernels at the edges of their layouts: the preconditioned
solver of exw_post_pressure (a call without iteration counts) against the
oracle's CG and against the plain CG kernel (a call with them), the factored L2
errors and the error of p*, the energy and the projection against the oracle.

Columns per cell of the solver: 3..14 (2D, several cells per wave, cell counts
that leave the last group part-filled), 9..100 in 3D (49 and 64 in one wave, 81
and 100 over two).  Both solvers stop at 1e-13 of the first residual, each in
its own norm: <= 1e-10 of the largest value, as the plain CG's own test."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

POST = [(2, 5, O.TRANSFORM_REFERENCE_SINE, 0.2, 1), (2, 3, O.TRANSFORM_NONE, 0.0, 4),
        (2, 3, O.TRANSFORM_AXIS_2PI, 0.04, 7), (2, 2, O.TRANSFORM_REFERENCE_SINE, 0.2, 12),
        (3, 3, O.TRANSFORM_REFERENCE_SINE, 0.1, 1), (3, 3, O.TRANSFORM_AXIS_2PI, 0.05, 2),
        (3, 2, O.TRANSFORM_NONE, 0.0, 3), (3, 2, O.TRANSFORM_PRODUCT_2PI, 0.05, 4),
        (3, 2, O.TRANSFORM_REFERENCE_SINE, 0.1, 5), (3, 2, O.TRANSFORM_AXIS_2PI, 0.05, 6),
        (3, 2, O.TRANSFORM_REFERENCE_SINE, 0.1, 7), (3, 1, O.TRANSFORM_NONE, 0.0, 8)]


@pytest.fixture(scope="module")
def X():
    import torch
    assert torch.cuda.is_available(), "GPU tests need a GPU"
    import exwave_amd
    exwave_amd.load()
    return exwave_amd


def _setup(X, dim, nint, tr, fac, k):
    om = O.Mesh(dim, nint, 0, tr, fac)
    rng = np.random.default_rng(dim * 100 + k)
    om.set_material(rng.uniform(0.5, 2.0, om.n_cells), rng.uniform(0.5, 2.0, om.n_cells))
    op = X.WaveOperator(X.Context(0), dim, k, om.vertices, om.neighbor, om.rho, om.speed)
    u = om.project(k, O.Exact.reference(dim, 2), 0.3)
    u += 0.05 * rng.standard_normal(u.shape) * np.abs(u).max()
    return om, op, u


@pytest.mark.parametrize("case", POST, ids=lambda c: "d%d_n%d_t%d_k%d" % (c[0], c[1], c[2], c[4]))
def test_post_pcg(X, case):
    import torch
    dim, nint, tr, fac, k = case
    print("post pcg", case, flush=True)
    om, op, u = _setup(X, *case)
    src = torch.from_numpy(u).cuda()
    tmp = torch.zeros_like(src)
    post = torch.zeros(op.n_post, dtype=torch.float64, device="cuda")
    op.post_pressure(src, tmp, post)
    got = post.cpu().numpy()
    want = om.post_pressure(k, u, rel_tol=1e-13, mean_free=True)
    assert np.max(np.abs(got - want)) <= 1e-10 * np.max(np.abs(want))
    its = torch.zeros(om.n_cells, dtype=torch.int32, device="cuda")
    op.post_pressure(src, tmp, post, its)
    assert np.max(np.abs(got - post.cpu().numpy())) <= 1e-10 * np.max(np.abs(want))
    # no flow, no right-hand side: exactly the (zero) cell averages
    src.zero_()
    op.post_pressure(src, tmp, post)
    assert torch.all(post == 0.0)
    # a cell that holds a NaN ends, and says so
    src[0] = float("nan")
    op.post_pressure(src, tmp, post)
    assert torch.isnan(post[: (k + 2) ** dim]).all()


@pytest.mark.parametrize("dim,nint,k", [(2, 10, 3), (2, 10, 4), (3, 4, 2), (3, 3, 4)])
def test_post_pcg_scales(X, dim, nint, k):
    """States that have decayed: down to the bottom of the exponent range every cell
    ends finite and of the state's size (p* is linear in the state while the
    residuals are above EXW_POST_ABS_TOL; below it p* may fall back to the average,
    and products of two residuals underflow from 1e-154 on)."""
    import torch
    print("post scales", dim, nint, k, flush=True)
    om, op, u = _setup(X, dim, nint, O.TRANSFORM_AXIS_2PI, 0.06, k)
    src = torch.from_numpy(u).cuda()
    tmp = torch.zeros_like(src)
    one, post = (torch.zeros(op.n_post, dtype=torch.float64, device="cuda") for _ in range(2))
    op.post_pressure(src, tmp, one)
    top = float(one.abs().max())
    for e in [3, 20, 100] + list(range(138, 172)) + [200, 290]:
        s = 10.0 ** -e
        op.post_pressure(src * s, tmp, post)
        assert torch.isfinite(post).all(), e
        assert float(post.abs().max()) <= 4 * top * s, e
        if e == 3:
            assert float((post - s * one).abs().max()) <= 1e-10 * top * s


@pytest.mark.parametrize("case", POST + [(2, 7, O.TRANSFORM_REFERENCE_SINE, 0.1, 5),
                                         (2, 6, O.TRANSFORM_AXIS_2PI, 0.04, 9)],
                         ids=lambda c: "d%d_n%d_t%d_k%d" % (c[0], c[1], c[2], c[4]))
def test_tick_norms(X, case):
    """The error of p* (tensor passes; direct sums in 2D from degree 5 on), the energy
    and the projection against the oracle: sums of at most 10^5 terms of one sign in
    another order, 1e-12; single evaluations of the modes, 1e-14."""
    import torch
    dim, nint, tr, fac, k = case
    print("tick norms", case, flush=True)
    om, op, u = _setup(X, *case)
    mm = [[1] * dim, [2] + [1] * (dim - 1)]
    e, m = O.Exact.make(dim, mm, [1.0, 0.3]), X.Modes.make(dim, mm, [1.0, 0.3])
    want = om.project(k, e, 0.3)
    got = op.new_vector()
    op.project(m, 0.3, got)
    assert np.max(np.abs(got.cpu().numpy() - want)) <= 1e-14 * np.max(np.abs(want))
    en = om.energy(k, u)
    assert abs(op.energy(torch.from_numpy(u).cuda()) - en) <= 1e-12 * en
    post = np.random.default_rng(k).standard_normal(op.n_post)
    err = om.post_error(k, e, 0.3, post)
    assert abs(op.post_error(m, 0.3, torch.from_numpy(post).cuda()) - err) <= 1e-12 * err


@pytest.mark.parametrize("dim,nint,k", [(2, 5, 1), (2, 3, 6), (2, 2, 12), (3, 3, 1), (3, 3, 4),
                                        (3, 2, 7), (3, 2, 8), (3, 2, 9), (3, 1, 12)])
def test_l2_errors_edges(X, dim, nint, k):
    """Tensor passes in one round of all fields (to 3D k = 7), two and four
    rounds (beyond), several small cells at a time: round-off apart the
    oracle's sums (1e-12: a few ulp per term, errors of the size of the field)."""
    print("l2", dim, nint, k, flush=True)
    import torch
    om, op, u = _setup(X, dim, nint, O.TRANSFORM_REFERENCE_SINE, 0.1, k)
    mm = [[1] * dim, [2] + [1] * (dim - 1)]
    got = op.l2_errors(X.Modes.make(dim, mm, [1.0, 0.3]), 0.7, torch.from_numpy(u).cuda())
    want = om.l2_errors(k, O.Exact.make(dim, mm, [1.0, 0.3]), 0.7, u)
    assert np.allclose(got, want, rtol=1e-12, atol=0), (got, want)
