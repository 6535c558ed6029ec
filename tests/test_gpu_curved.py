"""The factorised operator on periodic deformed meshes (hd_curved.hip)
against the CPU oracle's quadrature operator, over the forms it accepts:
spaces of one and two dimensions, node counts that fill a 16-wide tile and
that do not (4, 8, 9, 16, 25 nodes), uneven cell counts with a partial wave,
skew forms, over-integration and collocation, both precisions, fused stages,
and the vectors it leaves to the quadrature kernel.

Tolerances: FP64 1e-12 and FP32 2e-6 of the largest value, the bars of the
quadrature kernel on the same meshes (a row sums at most 25 + 20 products per
space, so reordering moves it by less than 50 roundings)."""

import numpy as np
import pytest

torch = pytest.importorskip("torch")

import hyperdeal_amd as H  # noqa: E402
import oracle as O  # noqa: E402

pytestmark = pytest.mark.gpu

FORMS = [
    # dims, degree, cells, skew, n_points, collocation
    ((1, 1), 1, [3, 5], 0.0, None, False),
    ((1, 1), 3, [17, 9], 0.0, None, False),
    ((1, 1), 4, [5, 6], 0.5, 6, False),
    ((2, 1), 2, [3, 4, 5], 0.0, None, False),
    ((1, 2), 3, [9, 3, 2], 0.3, None, False),
    ((2, 2), 1, [3, 2, 2, 3], 0.0, None, False),
    ((2, 2), 2, [5, 3, 2, 3], 0.5, None, False),
    ((2, 2), 3, [3, 3, 4, 2], 0.0, None, False),
    ((2, 2), 3, [3, 2, 2, 3], 1.0, 5, False),
    ((2, 2), 3, [2, 3, 3, 2], 0.0, None, True),
    ((2, 2), 4, [3, 2, 2, 2], 0.0, None, False),
]


def _pair(dims, k, n, skew, nq, coll, seed):
    D = sum(dims)
    a = list(np.random.default_rng(seed).uniform(-1, 1, D))
    lo, hi = [-1.0] * D, [1.0] * D
    P = O.Problem(dims[0], dims[1], k, n, lo, hi, a, n_points=nq,
                  collocation=coll, skew=skew)
    P.set_deformation(0.1, 2)
    mf = H.MatrixFree(dims[0], dims[1], k, n, lo, hi, n_points=nq,
                      collocation=coll)
    mf.set_deformation(0.1, 2)
    return P, mf, H.AdvectionOperation(mf, a, skew_factor=skew)


def _rel(x, ref):
    return np.max(np.abs(x - ref)) / np.max(np.abs(ref))


@pytest.mark.parametrize("dims,k,n,skew,nq,coll", FORMS)
def test_matches_oracle(dims, k, n, skew, nq, coll):
    print("case: curved", dims, k, n, skew, nq, coll, flush=True)
    P, mf, op = _pair(dims, k, n, skew, nq, coll, seed=k + sum(n))
    u = np.random.default_rng(3).standard_normal(P.n_dofs)
    ref = P.apply(u)
    src = torch.from_numpy(u).cuda()
    dst = op.apply(torch.empty_like(src), src)
    assert _rel(dst.cpu().numpy(), ref) <= 1e-12
    # the quadrature kernel on request, and for vectors off 16 bytes
    q = torch.zeros(P.n_dofs + 1, dtype=torch.float64, device="cuda")
    op.apply(q[1:], src)
    assert _rel(q[1:].cpu().numpy(), ref) <= 1e-12
    s32 = src.float()
    d32 = op.apply(torch.empty_like(s32), s32, precision=H.FP32)
    ref32 = P.apply(s32.double().cpu().numpy())
    assert _rel(d32.double().cpu().numpy(), ref32) <= 2e-6
    # fused stages: sol += b K, out = sol_old + a K, and without an output
    sol0 = torch.from_numpy(np.random.default_rng(4).standard_normal(
        P.n_dofs)).cuda()
    for prec, x, r, tol in ((H.FP64, src, ref, 1e-12),
                            (H.FP32, s32, ref32, 2e-6)):
        for last in (False, True):
            sol, out = sol0.clone(), torch.empty_like(x)
            op.stage(x, None if last else out, sol, 0.0, 0.3, 0.7,
                     precision=prec)
            s0 = sol0.cpu().numpy()
            scale = tol * np.max(np.abs(r))
            assert np.max(np.abs(sol.cpu().numpy() - (s0 + 0.7 * r))) <= scale
            if not last:
                # an FP32 output is rounded once more
                ulp = 0 if prec == H.FP64 else 1.2e-7 * np.max(
                    np.abs(s0 + 0.3 * r))
                assert np.max(np.abs(out.double().cpu().numpy() -
                                     (s0 + 0.3 * r))) <= scale + ulp


@pytest.mark.parametrize("dims,k,n,curved", [
    ((3, 1), 2, [2, 2, 3, 4], False),
    ((1, 1), 1, [270, 270], False),      # tiles mostly empty, many cells
    ((2, 1), 4, [73, 74, 2], True),      # 5,402 x cells
    ((2, 1), 4, [74, 74, 2], False),     # tables of one space above 64 MB
])
def test_other_meshes_take_the_quadrature_kernel(dims, k, n, curved):
    print("case: curved or quadrature", dims, k, n, flush=True)
    P, mf, op = _pair(dims, k, n, 0.0, None, False, seed=8)
    src = torch.from_numpy(np.random.default_rng(3).standard_normal(
        P.n_dofs)).cuda()
    auto = op.apply(torch.empty_like(src), src).cpu().numpy()
    op.set_algorithm(H.ALGO_QUADRATURE)
    quad = op.apply(torch.empty_like(src), src).cpu().numpy()
    assert _rel(auto, quad) <= 1e-12
    assert np.array_equal(auto, quad) != curved


@pytest.mark.parametrize("dims,k,n,zero", [
    ((1, 1), 3, [5, 6], [0]), ((1, 1), 2, [4, 7], [0, 1]),
    ((2, 2), 3, [3, 2, 2, 3], [0, 1]), ((2, 2), 2, [3, 4, 2, 3], [2, 3]),
    ((2, 2), 1, [3, 2, 3, 2], [1, 2]), ((2, 1), 4, [3, 2, 3], [0, 2]),
])
def test_zero_velocities(dims, k, n, zero):
    """Directions, or a whole space, that nothing flows along: their faces
    carry nothing and are skipped."""
    print("case: curved, zero velocities", dims, k, n, zero, flush=True)
    D = sum(dims)
    a = np.random.default_rng(k).uniform(0.2, 1, D)
    a[1::2] *= -1
    a[zero] = 0
    lo, hi = [-1.0] * D, [1.0] * D
    P = O.Problem(dims[0], dims[1], k, n, lo, hi, list(a))
    P.set_deformation(0.1, 2)
    mf = H.MatrixFree(dims[0], dims[1], k, n, lo, hi)
    mf.set_deformation(0.1, 2)
    op = H.AdvectionOperation(mf, list(a))
    u = np.random.default_rng(3).standard_normal(P.n_dofs)
    ref = P.apply(u)
    src = torch.from_numpy(u).cuda()
    for prec, x, tol in ((H.FP64, src, 1e-12), (H.FP32, src.float(), 2e-6)):
        dst = op.apply(torch.empty_like(x), x, precision=prec)
        err = np.abs(dst.double().cpu().numpy() - P.apply(
            x.double().cpu().numpy()))
        assert err.max() <= tol * max(np.abs(ref).max(), 1.0)
