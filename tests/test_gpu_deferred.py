"""FP64 LSRK steps whose stages leave the solution in memory and recover it in
the next stage from their own input, against the CPU oracle: every scheme
(each leaves other stages) on every kernel that takes part (row walk, tile,
late-reading tiles of k = 4, wave-per-group, split, Dirichlet correction,
curved), and vectors off 16 bytes, which take the copying step.

Tolerance 1e-12 of the largest value as for the plain steps: recovering adds
at most |b / a| <= 1 roundings of the solution per stage."""

import numpy as np
import pytest

torch = pytest.importorskip("torch")

import hyperdeal_amd as H  # noqa: E402
import oracle as O  # noqa: E402

pytestmark = pytest.mark.gpu

FORMS = [
    # dims, degree, cells, periodic, deformed
    ((1, 1), 3, [5, 6], True, False),
    ((2, 2), 1, [3, 4, 3, 5], True, False),
    ((2, 2), 2, [3, 2, 3, 3], False, False),
    ((2, 2), 3, [3, 3, 2, 2], True, False),
    ((2, 2), 3, [3, 2, 2, 2], False, False),
    ((2, 2), 4, [2, 3, 2, 2], True, False),
    ((2, 3), 4, [2, 1, 2, 1, 2], True, False),
    ((3, 3), 3, [3, 2, 2, 2, 1, 2], True, False),
    ((2, 2), 3, [3, 2, 2, 3], True, True),
]


@pytest.mark.parametrize("dims,k,n,periodic,deformed", FORMS)
def test_steps_match_oracle(dims, k, n, periodic, deformed):
    print("case: deferred steps", dims, k, n, periodic, deformed, flush=True)
    D = sum(dims)
    a = list(np.random.default_rng(k + D).uniform(-1, 1, D))
    lo, hi = [-1.0] * D, [1.0] * D
    P = O.Problem(dims[0], dims[1], k, n, lo, hi, a, periodic_x=periodic,
                  periodic_v=periodic, func=O.FUNC_HYPERRECTANGLE,
                  func_params=a)
    mf = H.MatrixFree(dims[0], dims[1], k, n, lo, hi, periodic_x=periodic,
                      periodic_v=periodic)
    if deformed:
        P.set_deformation(0.1, 2)
        mf.set_deformation(0.1, 2)
    op = H.AdvectionOperation(mf, a, boundary=H.BC_INHOMOGENEOUS,
                              boundary_function=H.FUNC_HYPERRECTANGLE,
                              boundary_params=a)
    u = np.random.default_rng(2).standard_normal(P.n_dofs)
    dt = 0.1 * P.critical_time_step() / k ** 1.5
    for rk in ("rk33", "rk45", "rk47", "rk59"):
        ref, ki, ti = u.copy(), P.vector(), P.vector()
        for s in range(2):
            P.lsrk_step(rk, ref, ki, ti, s * dt, dt)
        integ = H.LowStorageRungeKuttaIntegrator(rk)
        for shift in (0, 1):
            buf = torch.zeros(P.n_dofs + 1, dtype=torch.float64,
                              device="cuda")
            sol = buf[shift:shift + P.n_dofs]
            sol.copy_(torch.from_numpy(u))
            ta = torch.full_like(buf[:P.n_dofs], float("nan"))
            tb = torch.full_like(ta, float("nan"))
            for s in range(2):
                integ.perform_time_step(op, sol, ta, tb, s * dt, dt)
            err = np.max(np.abs(sol.cpu().numpy() - ref)) / \
                np.max(np.abs(ref))
            assert err <= 1e-12, (rk, shift, err)
