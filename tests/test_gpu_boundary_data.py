"""The projected boundary data of the collapsed form (products of 1D factors)
against the quadrature kernel, which evaluates the function at every face
point: each boundary function, both sides, corner cells on all boundaries,
one cell per direction, more points than nodes, at a time other than zero,
applies and stages.  1e-12 (FP64) and 2e-6 (FP32) of the largest value, the
bars of the two kernels against each other on periodic meshes."""

import numpy as np
import pytest

torch = pytest.importorskip("torch")

import hyperdeal_amd as H  # noqa: E402

pytestmark = pytest.mark.gpu

FUNCTIONS = [
    (H.FUNC_ZERO, [0.0] * 4),
    (H.FUNC_HYPERRECTANGLE, [0.3, -0.7, 0.2, 0.9]),
    (H.FUNC_CONSTANT_ONE, [0.0] * 4),
    (H.FUNC_SIN_COS, [0.0] * 4),
    (H.FUNC_PRODUCT_SINES, [0.6, 0.1, -0.4, -0.8]),
    (H.FUNC_LANDAU, [0.4, 0.8, 2.0, 0.0]),
    (H.FUNC_LANDAU, [0.4, 0.8, 1.0, 0.0]),
]


@pytest.mark.parametrize("n,px,pv,a", [
    ([3, 2, 2, 3], False, False, [0.7, -0.4, -0.6, 0.3]),
    ([1, 3, 1, 2], False, False, [-0.5, 0.8, 0.4, -0.9]),
    ([2, 3, 3, 2], True, False, [0.7, -0.4, 0.0, 0.3]),
])
@pytest.mark.parametrize("points", [4, 5])
def test_collapsed_matches_quadrature(n, px, pv, a, points):
    for func, prm in FUNCTIONS:
        print("case: boundary data", n, func, prm, points, flush=True)
        mf = H.MatrixFree(2, 2, 3, n, [-1.0, -0.8, -1.5, -1.0],
                          [1.0, 1.1, 1.2, 0.9], periodic_x=px, periodic_v=pv,
                          n_points=points)
        op = H.AdvectionOperation(mf, a, boundary=H.BC_INHOMOGENEOUS,
                                  boundary_function=func, boundary_params=prm)
        u = torch.from_numpy(np.random.default_rng(1).standard_normal(
            mf.n_dofs())).cuda()
        for prec, tol in ((H.FP64, 1e-12), (H.FP32, 2e-6)):
            src = u if prec == H.FP64 else u.float()
            got = []
            for algo in (H.ALGO_QUADRATURE, H.ALGO_COLLAPSED):
                op.set_algorithm(algo)
                dst = op.apply(torch.empty_like(src), src, time=0.37,
                               precision=prec)
                sol, out = u.clone(), torch.empty_like(src)
                op.stage(src, out, sol, 0.37, 0.01, 0.02, precision=prec)
                got.append([t.double().cpu().numpy()
                            for t in (dst, sol, out)])
            for q, c in zip(*got):
                assert np.max(np.abs(q - c)) <= tol * np.max(np.abs(q))
