"""GPU: sweeps of a small level that run several colours per launch -- the 32^3 tile sweep (odd and
even counts: its result ends in the other buffer), paired colours at 64^3 -- against the oracle's
colour sweep.  Equality."""
import numpy as np
import pytest

import refbind as R

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def problem(n, dt):
    rng = np.random.default_rng(n)
    d = rng.standard_normal(n ** 3)
    for _ in range(4):
        R.or_nsmooth(d, n)
    u = np.zeros((n ** 3, 5))
    u[:, 0] = R.or_lognormal(n, 1.5, 3)
    G = R.or_metric((2 * d).astype(dt), u.ravel().astype(dt), 5, n, 1.0)
    return rng.standard_normal(n ** 3).astype(dt), rng.standard_normal(n ** 3).astype(dt), G


@pytest.mark.parametrize("dt", [np.float64, np.float32])
@pytest.mark.parametrize("n", [16, 32, 64])
@pytest.mark.parametrize("ns", [1, 2, 3])
def test_sweeps_equal_the_oracle(ctx, n, ns, dt):
    print("case sweeps n=%d ns=%d %s" % (n, ns, dt.__name__), flush=True)
    phi, rhs, G = problem(n, dt)
    got = torch.from_numpy(phi.copy()).cuda()
    ctx.time_sweeps(got, torch.from_numpy(rhs).cuda(), torch.from_numpy(G).cuda(), 1.0, ns)
    R.or_sweep(phi, rhs, G, n, 1.0, ns)
    assert np.array_equal(got.cpu().numpy(), phi)


@pytest.mark.parametrize("ns", [1, 2])
def test_bfloat16_tile_sweeps_equal_the_oracle(ctx, ns):
    print("case bf16 tile sweeps ns=%d" % ns, flush=True)
    n = 32
    phi, rhs, G = problem(n, np.float32)
    Gr = torch.from_numpy(G).bfloat16().float().numpy()
    got = torch.from_numpy(phi.copy()).cuda()
    ctx.time_sweeps_bf16(got, torch.from_numpy(rhs).cuda(), torch.from_numpy(G.astype(np.float64)).cuda(), 1.0, ns)
    R.or_sweep(phi, rhs, Gr, n, 1.0, ns)
    assert np.array_equal(got.cpu().numpy(), phi)


@pytest.mark.parametrize("mixed", [0, 1])
@pytest.mark.parametrize("nu", [1, 2])
def test_paired_galerkin_colours_inside_a_solve(ctx, mixed, nu):
    """A 128^3 Krylov solve sweeps its 64^3 Galerkin level two colours a launch, from zero and from a
    value, forward and reversed: the FP64 solve equals the batched one, which sweeps colour by colour;
    the mixed one (bfloat16 coefficients) reaches the tolerance under the FP64 operator."""
    print("case galerkin pairs mixed=%d nu=%d" % (mixed, nu), flush=True)
    n = 128
    rng = np.random.default_rng(nu)
    u = np.zeros((n ** 3, 5))
    u[:, 0] = R.or_lognormal(n, 1.5, 3)
    to = lambda a: torch.from_numpy(np.ascontiguousarray(a).ravel()).cuda()  # noqa: E731
    rhs, ud, d = rng.standard_normal(n ** 3), to(u), to(np.zeros(n ** 3))
    phi, b = to(np.zeros(n ** 3)), to(rhs)
    _, ok = ctx.solve(phi, b, d, ud, tol=1e-9, max_cycles=200, schedule=1, nu_pre=nu, nu_post=nu, nu_coarse=4,
                      mixed=mixed, nu=5, krylov=True)
    assert ok
    if not mixed:
        phi2, b2 = to(np.zeros(n ** 3)), to(rhs)
        _, ok2 = ctx.solve_batch([(phi2, b2, d, ud)], tol=1e-9, max_cycles=200, nu_pre=nu, nu_coarse=4, nu=5)
        assert ok2 and np.array_equal(phi.cpu().numpy(), phi2.cpu().numpy())
    r = torch.zeros_like(b)
    ctx.residual(r, phi, b, d, ud)
    assert float(r.abs().max()) <= 1.01e-9 * float(b.abs().max())


@pytest.mark.parametrize("n", [512, 1024])
def test_half_sweep_slabs_equal_the_colour_by_colour_order(ctx, n):
    """FP32 sweeps from 512^3 go slab by slab inside a half sweep (two segments of 8 planes a slab, one at
    1024^3); one point per thread (option colour_col = 1) goes colour by colour.  Equality."""
    print("case half-sweep slabs n=%d" % n, flush=True)
    gen = torch.Generator(device="cuda").manual_seed(n)
    draw = lambda k: torch.rand(k, device="cuda", generator=gen)  # noqa: E731
    rhs, G = draw(n ** 3) - 0.5, draw(6 * n ** 3) + 1.0
    a = draw(n ** 3)
    b = a.clone()
    ctx.time_sweeps(a, rhs, G, 1.0, 2)
    try:
        ctx.set_option("colour_col", 1)
        ctx.time_sweeps(b, rhs, G, 1.0, 2)
    finally:
        ctx.set_option("colour_col", 8)
    assert bool(torch.isfinite(a).all()) and torch.equal(a, b)


@pytest.mark.parametrize("mixed", [0, 1])
@pytest.mark.parametrize("nu", [1, 2, 3])
def test_galerkin_tile_sweeps_inside_a_solve(ctx, mixed, nu):
    """A 64^3 Krylov solve whose 32^3 Galerkin level is swept tile by tile (odd and even counts, both
    directions, bfloat16 coefficients when mixed): the FP64 solve equals the batched solve's colour
    launches, the mixed one reaches the tolerance under the FP64 operator."""
    print("case galerkin tile mixed=%d nu=%d" % (mixed, nu), flush=True)
    n = 64
    rng = np.random.default_rng(nu)
    rho = R.or_lognormal(n, 1.5, 3)
    u = np.zeros((n ** 3, 5))
    u[:, 0] = rho
    rhs = rng.standard_normal(n ** 3)
    to = lambda a: torch.from_numpy(np.ascontiguousarray(a).ravel()).cuda()  # noqa: E731
    d, ud = to(np.zeros(n ** 3)), to(u)
    phi, b = to(np.zeros(n ** 3)), to(rhs)
    st, ok = ctx.solve(phi, b, d, ud, tol=1e-9, max_cycles=200, schedule=1, nu_pre=nu, nu_post=nu, nu_coarse=4,
                       mixed=mixed, nu=5, krylov=True)
    assert ok
    if not mixed:
        phi2, b2 = to(np.zeros(n ** 3)), to(rhs)
        _, ok2 = ctx.solve_batch([(phi2, b2, d, ud)], tol=1e-9, max_cycles=200, nu_pre=nu, nu_coarse=4, nu=5)
        assert ok2 and np.array_equal(phi.cpu().numpy(), phi2.cpu().numpy())
    r = torch.zeros_like(b)
    ctx.residual(r, phi, b, d, ud)
    assert float(r.abs().max()) <= 1.01e-9 * float(b.abs().max())


@pytest.mark.parametrize("mixed", [0, 1])
@pytest.mark.parametrize("n,galerkin,nu", [(32, 0, 2), (64, 1, 1), (64, 1, 2), (64, 1, 3), (64, 0, 2), (128, 1, 1),
                                           (128, 1, 2), (128, 1, 3)])
def test_colours_in_one_launch_or_eight(ctx, n, galerkin, nu, mixed):
    """Krylov solves whose 32^3 and 64^3 levels (19-point or Galerkin, bfloat16 coefficients when mixed; from zero
    and from a value, forward and reversed) are swept with several colours a launch, against one
    colour a launch (option colour_fused 0): the same residual after every iteration, the same solution."""
    print("case colours n=%d galerkin=%d nu=%d mixed=%d" % (n, galerkin, nu, mixed), flush=True)
    rng = np.random.default_rng(nu)
    u = np.zeros((n ** 3, 5))
    u[:, 0] = R.or_lognormal(n, 1.5, 3)
    d = rng.standard_normal(n ** 3)
    for _ in range(6):
        R.or_nsmooth(d, n)
    to = lambda a: torch.from_numpy(np.ascontiguousarray(a).ravel()).cuda()  # noqa: E731
    rhs, ud, d = rng.standard_normal(n ** 3), to(u), to(d)
    out = []
    for fused in (1, 0):
        ctx.set_option("colour_fused", fused)
        ctx.set_option("galerkin", galerkin)
        try:
            phi = to(np.zeros(n ** 3))
            st, ok = ctx.solve(phi, to(rhs), d, ud, tol=1e-9, max_cycles=200, schedule=1, nu_pre=nu, nu_post=nu,
                               nu_coarse=4, mixed=mixed, nu=5, krylov=True)
        finally:
            ctx.set_option("colour_fused", 1)
            ctx.set_option("galerkin", 1)
        assert ok
        out.append((phi.cpu().numpy(), [st.relres[i] for i in range(st.cycles)]))
    assert len(out[0][1]) > 3 and out[0][1] == out[1][1]
    assert np.array_equal(out[0][0], out[1][0])
