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
