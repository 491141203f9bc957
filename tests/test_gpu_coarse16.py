"""GPU: the on-chip coarse levels (16^3, 8^3, 4^3 in one workgroup) against the launches and the
general one-workgroup form where the hierarchy itself starts at 16^3, 8^3 or 4^3 (its finest level then runs there, with a
non-zero iterate and no guard), and with odd sweep counts.  Same operations in the same order:
equality."""
import numpy as np
import pytest

import refbind as R

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def fields(n, dt):
    rng = np.random.default_rng(n)
    d = rng.standard_normal(n ** 3)
    for _ in range(4):
        R.or_nsmooth(d, n)
    rho = R.or_lognormal(n, 1.5, 5)
    u = np.zeros((n ** 3, 5))
    u[:, 0] = rho
    to = lambda a: torch.from_numpy(np.ascontiguousarray(a, dt).ravel()).cuda()  # noqa: E731
    return to(d), to(u), to(rng.standard_normal(n ** 3)), to(1e-3 * rng.standard_normal(n ** 3))


@pytest.mark.parametrize("dt", [np.float64, np.float32])
@pytest.mark.parametrize("n,ng", [(4, 4), (8, 8), (16, 16), (4, 8), (8, 32), (16, 64), (32, 32)])
def test_vcycle_of_a_small_grid(ctx, dt, n, ng):
    print("case small vcycle n=%d ng=%d %s" % (n, ng, dt.__name__), flush=True)
    d, u, rhs, phi = fields(n, dt)
    out = []
    for fused in (16, 0):
        ctx.set_option("coarse_fused_ref", fused)
        try:
            a, b = phi.clone(), rhs.clone()
            st = ctx.multigrid(a, b, d, u, 1.0, 2, ng, nu=5)
        finally:
            ctx.set_option("coarse_fused_ref", 16)
        out.append((a.cpu().numpy(), [(st.r1[l], st.relaxerr[l], st.guard[l]) for l in range(st.nlev)]))
    assert out[0][1] == out[1][1]
    assert np.array_equal(out[0][0], out[1][0])


@pytest.mark.parametrize("mixed,galerkin,nu,nuc", [(0, 1, 1, 1), (1, 1, 3, 4), (0, 0, 3, 5), (1, 0, 1, 2)])
@pytest.mark.parametrize("n", [8, 16, 32])
def test_preconditioner_of_a_small_grid(ctx, n, mixed, galerkin, nu, nuc):
    print("case small solve n=%d mixed=%d galerkin=%d nu=%d" % (n, mixed, galerkin, nu), flush=True)
    d, u, rhs, _ = fields(n, np.float64)
    out = []
    # against the general one-workgroup form: launch by launch, the finest level's mean is removed by the
    # dot products of the mixed solve instead, which rounds otherwise
    for general in (0, 1):
        ctx.set_option("coarse_lds", 1 - general)
        ctx.set_option("galerkin", galerkin)
        try:
            phi = torch.zeros_like(rhs)
            st, ok = ctx.solve(phi, rhs.clone(), d, u, tol=1e-9, max_cycles=200, schedule=1, nu_pre=nu, nu_post=nu,
                               nu_coarse=nuc, mixed=mixed, nu=5, krylov=True)
        finally:
            ctx.set_option("coarse_lds", 1)
            ctx.set_option("galerkin", 1)
        assert ok
        out.append((phi.cpu().numpy(), [st.relres[i] for i in range(st.cycles)]))
    assert out[0][1] == out[1][1]
    assert np.array_equal(out[0][0], out[1][0])


@pytest.mark.parametrize("dt,rhs_exp,rho_exp", [
    (np.float32, -112, 0),      # dividends below 2^-100, quotients and residuals still normal
    (np.float32, -140, 0),      # subnormal right-hand side and iterate
    (np.float32, -60, -127),    # diagonals around the smallest normal number
    (np.float32, -60, -134),    # subnormal diagonals whose reciprocal overflows
    (np.float32, 60, 118),      # large diagonals
    (np.float64, -990, 0), (np.float64, -1065, 0), (np.float64, -500, -1024), (np.float64, -500, -1040),
])
@pytest.mark.parametrize("n", [4, 8, 16])
def test_vcycle_at_the_ends_of_the_number_range(ctx, dt, rhs_exp, rho_exp, n):
    """The on-chip levels divide by way of a reciprocal; the launches divide.  Equality also where that
    reciprocal, the quotient or its residual leaves the normal range."""
    print("case range n=%d %s rhs 2^%d rho 2^%d" % (n, dt.__name__, rhs_exp, rho_exp), flush=True)
    rng = np.random.default_rng(n)
    to = lambda a: torch.from_numpy(np.ascontiguousarray(a, dt).ravel()).cuda()  # noqa: E731
    u = np.zeros((n ** 3, 5))
    u[:, 0] = np.ldexp(R.or_lognormal(n, 0.5, 5), rho_exp)
    d, u, rhs = to(np.zeros(n ** 3)), to(u), to(np.ldexp(rng.standard_normal(n ** 3), rhs_exp))
    out = []
    for fused in (16, 0):
        ctx.set_option("coarse_fused_ref", fused)
        try:
            a, b = torch.zeros_like(rhs), rhs.clone()
            st = ctx.multigrid(a, b, d, u, 1.0, 2, n, nu=5)
        finally:
            ctx.set_option("coarse_fused_ref", 16)
        out.append((a.cpu().numpy(), [(st.r1[l], st.relaxerr[l], st.guard[l]) for l in range(st.nlev)]))
    assert np.isfinite(out[1][0]).all() and np.any(out[1][0])
    assert out[0][1] == out[1][1]
    assert np.array_equal(out[0][0], out[1][0])


@pytest.mark.parametrize("kind,rho_exp", [("fp64", 410), ("mixed", 50), ("batch", 410)])
def test_solve_with_diagonals_past_the_reciprocals_range(ctx, kind, rho_exp):
    """Densities whose operator diagonals exceed the reciprocal form's bound: the solve equals the one with
    the general one-workgroup cycle (option coarse_lds 0)."""
    print("case large density %s" % kind, flush=True)
    n = 32
    d, u, rhs, _ = fields(n, np.float64)
    u = torch.ldexp(u, torch.tensor(rho_exp, device="cuda"))
    out = []
    for general in (0, 1):
        ctx.set_option("coarse_lds", 1 - general)
        try:
            phi = torch.zeros_like(rhs)
            if kind == "batch":
                st, ok = ctx.solve_batch([(phi, rhs.clone(), d, u)], tol=1e-9, max_cycles=200, nu_pre=2, nu_coarse=4, nu=5)
                hist = [st[0].cycles, st[0].relres]
            else:
                st, ok = ctx.solve(phi, rhs.clone(), d, u, tol=1e-9, max_cycles=200, schedule=1, nu_pre=2, nu_post=2,
                                   nu_coarse=4, mixed=kind == "mixed", nu=5, krylov=True)
                hist = [st.relres[i] for i in range(st.cycles)]
        finally:
            ctx.set_option("coarse_lds", 1)
        assert ok
        out.append((phi.cpu().numpy(), hist))
    assert out[0][1] == out[1][1]
    assert np.any(out[0][0]) and np.array_equal(out[0][0], out[1][0])
