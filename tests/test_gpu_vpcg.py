"""The potential solve on several workgroups (hd_vpcg.hip) against the CPU
oracle's: strips of one row and of several, an uneven last strip, the fewest
strips, one, two and four nodes per thread, meshes that stay on one workgroup, two
operators in turn, and the kernel behind a solve that was given up (its mark set from the host; no
workgroup waits in that case).

Tolerance: CG to 1e-12 of the right-hand side leaves at most cond(A) 1e-12 in
the potential; 1e-8 covers these meshes, as for the one-workgroup solver."""

import ctypes

import numpy as np
import pytest

torch = pytest.importorskip("torch")

import hyperdeal_amd as H  # noqa: E402
import oracle as O  # noqa: E402

pytestmark = pytest.mark.gpu

L = 4 * np.pi
MESHES = [
    # degree, x cells
    (3, [5, 2]),      # two strips of one row
    (1, [7, 6]),      # one workgroup
    (2, [9, 35]),     # one workgroup
    (2, [17, 35]),    # two rows per strip, one in the last
    (3, [4, 96]),     # three rows per strip
    (3, [32, 32]),    # the most cells
    (3, [50, 18]),    # two nodes per thread
    (3, [120, 8]),    # four nodes per thread
]


def _pair(k, nx):
    n = nx + [2, 2]
    lo, hi = [0, 0, -6, -6], [L, 0.8 * L, 6, 6]
    P = O.VlasovPoisson(2, k, n, lo, hi, [1, 1, 6, 6], eps=0.05, kx=0.5)
    mf = H.MatrixFree(2, 2, k, n, lo, hi)
    f = P.interpolate() * (1 + 0.1 * np.random.default_rng(k + nx[0])
                           .standard_normal(P.n_dofs))
    phi, _ = P.poisson_solve(P.rhs(P.density(f)), rel_tol=1e-12)
    return P, mf, f, phi - phi.mean()


def _off(phi, ref):
    phi = phi - phi.mean()
    return np.max(np.abs(phi - ref)) / np.max(np.abs(ref))


@pytest.mark.parametrize("k,nx", MESHES)
def test_potential_matches_oracle(k, nx):
    print("case: strips", k, nx, flush=True)
    P, mf, f, ref = _pair(k, nx)
    op = H.VlasovPoissonOperation(mf, poisson_tol=1e-12)
    op.set_poisson_tolerance(1e-12, 5000)
    fd = torch.from_numpy(f).cuda()
    op.update_field(fd)
    assert _off(op.potential(), ref) <= 1e-8
    it, solves, res = op.solver_stats()
    assert 0 < it < 5000 and solves == 1 and res <= 1e-12
    energy = op.field_energy()
    P.set_potential(op.potential())
    np.testing.assert_allclose(energy, P.energy()[:2], rtol=1e-10)
    # from there to 1e-10: no further iteration (the recurrence's residual
    # drifts from b - A phi by about 400 iterations' roundings, some 1e-12)
    op.set_poisson_tolerance(1e-10, 5000)
    op.update_field(fd)
    assert op.solver_stats()[:2] == (it, 2)


@pytest.mark.parametrize("k,nx", [(3, [4, 96]), (3, [2, 120]), (3, [120, 8]),
                                  (2, [2, 300])])
def test_tolerances_below_rounding(k, nx):
    """A solve asked for less than b - A phi can reach in 64 bits stays at
    what it can reach: at most four times the oracle's residual at 1e-12,
    which is rounding on these meshes (rounding sums in another order: the
    recurrence restated on the CPU ends at 0.7 to 1.4 times plain CG's)."""
    print("case: strips, below rounding", k, nx, flush=True)
    P, mf, f, _ = _pair(k, nx)
    op = H.VlasovPoissonOperation(mf, poisson_tol=1e-12)
    fd = torch.empty(P.n_dofs, dtype=torch.float64, device="cuda")
    for seed in range(4):
        g = f * (1 + 0.1 * np.random.default_rng(seed).standard_normal(
            P.n_dofs))
        fd.copy_(torch.from_numpy(g))
        b = P.rhs(P.density(g))

        def off(phi):
            return np.linalg.norm(b - P.poisson_apply(phi)) / \
                np.linalg.norm(b)
        bar = 4 * off(P.poisson_solve(b, rel_tol=1e-12)[0])
        for tol in (3e-13, 1e-13, 1e-15):
            op.set_poisson_tolerance(tol, 20000)
            op.set_potential(np.zeros(op.x_n_dofs()))
            op.update_field(fd)
            assert off(op.potential()) <= bar, (seed, tol)
        # and from a start that is already there
        op.update_field(fd)
        assert off(op.potential()) <= bar, seed


def test_two_operators_in_turn():
    print("case: strips, two operators", flush=True)
    a, b = _pair(3, [8, 8]), _pair(3, [6, 12])
    ops = [H.VlasovPoissonOperation(m[1], poisson_tol=1e-12) for m in (a, b)]
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    fs = [torch.from_numpy(m[2]).cuda() for m in (a, b)]
    torch.cuda.synchronize()
    for _ in range(4):
        for op, f, s in zip(ops, fs, streams):
            op.set_potential(np.zeros(op.x_n_dofs()))
            op.update_field(f, stream=s)
    torch.cuda.synchronize()
    for op, m in zip(ops, (a, b)):
        assert _off(op.potential(), m[3]) <= 1e-8


class _Solver:
    """The solver of an operator's potential on one workgroup or on strips
    (hd_probe.hip), with inboxes and statistics of its own."""

    def __init__(self, op):
        self.op, self.lib = op, ctypes.CDLL(H.library_path())
        self.lib.hd_probe_strips_bytes.restype = ctypes.c_longlong
        size = self.lib.hd_probe_strips_bytes(op.handle)
        self.comm = torch.empty(size // 8, dtype=torch.int64, device="cuda")
        assert self.lib.hd_probe_strips_reset(op.handle,
                                              self._p(self.comm)) == 0
        self.empty()
        n = op.x_n_dofs()
        self.phi = torch.zeros(n, dtype=torch.float64, device="cuda")
        self.field = torch.empty(2 * n, dtype=torch.float64, device="cuda")
        self.copy = torch.full_like(self.phi, float("nan"))
        self.scale = torch.empty(1, dtype=torch.float64, device="cuda")
        self.image = torch.full((n,), float("nan"), dtype=torch.float32,
                                device="cuda")

    @staticmethod
    def _p(t):
        return ctypes.c_void_p(None if t is None else t.data_ptr())

    def empty(self):
        assert int(self.comm[-1]) == 0 and bool((self.comm[:-1] == -1).all())

    def give_up(self):
        self.comm[:-1] = 5            # what a broken-off launch may leave
        self.comm[-1] = 1

    def _call(self, strips, rho, guess, image, scale, residual):
        stats = torch.zeros(8, dtype=torch.int64, device="cuda")
        p = self._p
        out = (self.image, self.scale, self.copy) if residual else [None] * 3
        torch.cuda.synchronize()
        rc = self.lib.hd_probe_poisson(
            self.op.handle, p(self.comm if strips else None), p(rho),
            p(self.phi), p(self.field), p(guess), p(image), p(scale),
            *[p(x) for x in out], ctypes.c_double(1e-12), 5000, p(stats))
        torch.cuda.synchronize()
        assert rc == 0
        self.empty()
        return stats

    def solve(self, rho, strips=True, guess=None, image=None, scale=None):
        s = self._call(strips, rho, guess, image, scale, False).cpu()
        return dict(its=int(s[0]), weights=s.view(torch.float64)[6:].numpy(),
                    start=float(s.view(torch.float64)[3]))

    def residual(self, rho, strips=True):
        self._call(strips, rho, None, None, None, True)
        return self.image.cpu().numpy(), float(self.scale)


@pytest.mark.parametrize("k,nx", [(3, [6, 5]), (2, [4, 40])])
def test_marked_solve_runs_on_one_workgroup(k, nx):
    print("case: marked solve", k, nx, flush=True)
    P, mf, f, ref = _pair(k, nx)
    s = _Solver(H.VlasovPoissonOperation(mf, poisson_tol=1e-12))
    rho = torch.from_numpy(P.density(f)).cuda()

    def run():
        s.phi.zero_()
        its = s.solve(rho)["its"]
        assert _off(s.phi.cpu().numpy(), ref) <= 1e-8
        return its, s.field.cpu().numpy()

    its, field = run()
    s.give_up()
    its2, field2 = run()
    assert abs(its2 - its) <= max(3, its // 20)
    assert np.max(np.abs(field2 - field)) <= 1e-8 * np.max(np.abs(field))
    run()


# one row per strip, an uneven last strip of several rows, two and four nodes
# per thread
IMAGES = [(3, [5, 7]), (2, [17, 35]), (3, [50, 18]), (3, [120, 8])]


@pytest.mark.parametrize("k,nx", IMAGES)
def test_residual_image_matches_one_workgroup(k, nx):
    """The residual image, its scale and the copy of phi: strips, and the
    kernel behind strips that were given up, against the one-workgroup kernel.
    Tolerances: b - A phi of a random phi to 1e-13 of its rms (sums of 2 (3 N)
    products in another order), pixels to that and one FP32 rounding."""
    print("case: residual image", k, nx, flush=True)
    P, mf, f, _ = _pair(k, nx)
    s = _Solver(H.VlasovPoissonOperation(mf, poisson_tol=1e-12))
    rho = torch.from_numpy(P.density(f)).cuda()
    phi = np.random.default_rng(k).standard_normal(P.n_x_dofs)
    s.phi.copy_(torch.from_numpy(phi))
    ref, scale = s.residual(rho, strips=False)
    for marked in (False, True, False):
        s.image.fill_(float("nan"))
        s.copy.fill_(float("nan"))
        if marked:
            s.give_up()
        img, sc = s.residual(rho)
        assert abs(sc - scale) <= 1e-12 * scale, marked
        assert np.max(np.abs(img - ref)) <= 2.5e-7 * np.max(np.abs(ref))
        assert np.array_equal(s.copy.cpu().numpy(), phi)
        assert np.array_equal(s.phi.cpu().numpy(), phi)


@pytest.mark.parametrize("k,nx", IMAGES)
def test_guess_image_stands_for_its_dofs(k, nx):
    """A guess given as an image starts the solve where the same guess given
    as x values starts it: the weights of phi and the guess and the start's
    residual agree to 1e-9 (the 2 x 2 system's condition, below 1e4 for random
    vectors, times rounding of its sums)."""
    print("case: guess image", k, nx, flush=True)
    P, mf, f, ref = _pair(k, nx)
    s = _Solver(H.VlasovPoissonOperation(mf, poisson_tol=1e-12))
    rho = torch.from_numpy(P.density(f)).cuda()
    r = np.random.default_rng(k)
    phi = torch.from_numpy(r.standard_normal(P.n_x_dofs)).cuda()
    N = k + 1
    # a part of the solution, so that the guess has a weight
    img, _ = H.cnn_dofs_to_image(torch.from_numpy(ref).cuda(), nx[0], nx[1], N)
    img += 0.2 * torch.from_numpy(r.standard_normal(img.shape)).cuda().float()
    scale = torch.full((1,), 0.75, dtype=torch.float64, device="cuda")
    dofs = H.cnn_image_to_dofs(img, scale, nx[0], nx[1], N)
    s.phi.copy_(phi)
    a = s.solve(rho, guess=dofs)
    assert abs(a["weights"][1]) > 1e-4
    s.phi.copy_(phi)
    b = s.solve(rho, guess=torch.zeros_like(dofs), image=img, scale=scale)
    np.testing.assert_allclose(b["weights"], a["weights"], rtol=0,
                               atol=1e-9 * np.abs(a["weights"]).max())
    assert abs(b["start"] - a["start"]) <= 1e-9 * a["start"]
    assert _off(s.phi.cpu().numpy(), ref) <= 1e-8


def test_nan_guess_is_left_out():
    print("case: NaN guess", flush=True)
    P, mf, f, ref = _pair(3, [8, 6])
    s = _Solver(H.VlasovPoissonOperation(mf, poisson_tol=1e-12))
    rho = torch.from_numpy(P.density(f)).cuda()
    plain = s.solve(rho)
    for bad in (float("nan"), float("inf")):
        s.phi.zero_()
        r = s.solve(rho, guess=torch.full_like(s.phi, bad))
        assert list(r["weights"]) == [1.0, 0.0] and r["its"] == plain["its"]
        assert _off(s.phi.cpu().numpy(), ref) <= 1e-8
