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
