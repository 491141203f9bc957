"""GPU: the transport step against the oracle on a fluid with momentum and energy, at every tile
shape of the march (16, 32 and 64 wide) and both walk lengths that occur: 4 planes up to 128^3, 32
from 256^3.  Halvings taken together are exact, so the bar is equality."""
import numpy as np
import pytest

import refbind as R

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.mark.parametrize("dt", [np.float64, np.float32])
@pytest.mark.parametrize("n", [16, 32, 64, 128])
def test_transport_of_a_flow_equals_the_oracle(ctx, n, dt):
    print("case transport n=%d %s" % (n, dt.__name__), flush=True)
    rng = np.random.default_rng(n)

    def smooth(amp):
        a = rng.standard_normal(n ** 3)
        for _ in range(3):
            R.or_nsmooth(a, n)
        return a * amp

    rho = np.exp(smooth(8.0))
    u = np.zeros((n ** 3, 5))
    u[:, 0] = rho
    for l in (1, 2, 3):
        u[:, l] = rho * smooth(2.0)
    u[:, 4] = (u[:, 1:4] ** 2).sum(1) / (2 * rho) + 0.1 * rho
    u[: n ** 3 // 3, 1:] = 0.0  # part of the box as the reference starts: at rest and cold
    u = u.ravel().astype(dt)
    d, p = smooth(3.0).astype(dt), smooth(1.0).astype(dt)
    got = torch.from_numpy(u.copy()).cuda()
    ctx.relaxing(got, torch.from_numpy(d).cuda(), torch.from_numpy(p).cuda(), dt=0.7)
    R.or_relaxing(u, d, p, n, dt=0.7)
    assert np.array_equal(got.cpu().numpy(), u)


@pytest.mark.parametrize("dt", [np.float64, np.float32])
def test_transport_by_long_walks_equals_the_oracle(ctx, dt):
    """256^3, where a workgroup walks 32 planes."""
    test_transport_of_a_flow_equals_the_oracle(ctx, 256, dt)
