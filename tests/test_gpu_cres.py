"""The one-pass kernel of 3+3 cells larger than LDS (k = 4, 5) where a block
walks several cells (more cells than resident blocks, an uneven share per
XCD), against the CPU oracle on every cell: apply in both precisions and the
fused FP64 stages that leave and recover the solution, through whole steps.

Bars: FP64 1e-12, FP32 2e-6 of the largest value, as for single cells."""

import numpy as np
import pytest

torch = pytest.importorskip("torch")

import hyperdeal_amd as H  # noqa: E402
import oracle as O  # noqa: E402

pytestmark = pytest.mark.gpu

FORMS = [
    # degree, cells, velocity (both signs, one direction without transport)
    (5, [3, 3, 2, 3, 3, 2], [0.7, -0.4, 0.5, 0.0, -0.9, 0.55]),
    (4, [3, 4, 3, 3, 3, 3], [-0.6, 0.2, -0.8, 0.35, 0.5, -0.7]),
    # few cells: a block per output plane
    (5, [2, 1, 2, 1, 2, 1], [0.7, -0.4, 0.5, 0.3, -0.9, 0.55]),
    (4, [1, 2, 3, 1, 2, 1], [-0.6, 0.2, -0.8, 0.35, 0.0, -0.7]),
    (4, [3, 2, 2, 2, 2, 2], [0.6, 0.2, 0.8, -0.35, 0.5, 0.7]),
]


@pytest.mark.parametrize("k,n,a", FORMS)
def test_many_cells_per_block(k, n, a):
    print("case: one-pass cells", k, n, flush=True)
    P = O.Problem(3, 3, k, n, [0.0] * 6, [1.0] * 6, a)
    mf = H.MatrixFree(3, 3, k, n, [0.0] * 6, [1.0] * 6)
    op = H.AdvectionOperation(mf, a)
    u = np.random.default_rng(7).standard_normal(P.n_dofs)
    ref = P.apply(u)
    src = torch.from_numpy(u).cuda()
    dst = op.apply(torch.empty_like(src), src)
    scale = np.max(np.abs(ref))
    assert np.max(np.abs(dst.cpu().numpy() - ref)) <= 1e-12 * scale
    d32 = op.apply(torch.empty_like(src.float()), src.float(),
                   precision=H.FP32)
    ref32 = P.apply(src.float().double().cpu().numpy())
    assert np.max(np.abs(d32.double().cpu().numpy() - ref32)) <= \
        2e-6 * np.max(np.abs(ref32))
    dt = 0.1 * P.critical_time_step() / k ** 1.5
    sol_ref, ki, ti = u.copy(), P.vector(), P.vector()
    P.lsrk_step("rk45", sol_ref, ki, ti, 0.0, dt)
    for prec, tol in ((H.FP64, 1e-12), (H.FP32, 1e-6)):
        dtype = torch.float64 if prec == H.FP64 else torch.float32
        sol = torch.from_numpy(u).cuda()
        ta = torch.full_like(sol, float("nan"), dtype=dtype)
        tb = torch.full_like(ta, float("nan"))
        H.LowStorageRungeKuttaIntegrator("rk45").perform_time_step(
            op, sol, ta, tb, 0.0, dt, precision=prec)
        assert np.max(np.abs(sol.cpu().numpy() - sol_ref)) <= \
            tol * np.max(np.abs(sol_ref))
