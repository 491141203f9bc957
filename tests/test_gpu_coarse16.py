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
