"""GPU: smoothing at the smallest grids and both walk lengths, and the limiter's diagnostics (combined
on the device) on a mesh where the expansion limiter and the compression gate hold in places.
Smoothing equals the oracle; extremes and counts equal those of the same quantities formed by the
oracle's calcdefp."""
import numpy as np
import pytest

import refbind as R

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.mark.parametrize("dt", [np.float64, np.float32])
@pytest.mark.parametrize("n", [4, 8, 16, 64, 128])
def test_smoothing_equals_the_oracle(ctx, n, dt):
    print("case smoothing n=%d %s" % (n, dt.__name__), flush=True)
    a = np.random.default_rng(n).standard_normal(n ** 3).astype(dt)
    got = torch.from_numpy(a.copy()).cuda()
    for _ in range(2):
        ctx.nsmooth(got)
        R.or_nsmooth(a, n)
        assert np.array_equal(got.cpu().numpy(), a)


@pytest.mark.parametrize("n", [16, 64])
def test_limiter_diagnostics(ctx, n):
    print("case limiter diagnostics n=%d" % n, flush=True)
    rng = np.random.default_rng(n)
    d = rng.standard_normal(n ** 3)
    for _ in range(2):
        R.or_nsmooth(d, n)
    d *= 6.0
    u = np.zeros((n ** 3, 5))
    u[:, 0] = R.or_lognormal(n, 1.0, 9)
    u[:, 1:4] = 0.05 * rng.standard_normal((n ** 3, 3))
    u = u.ravel()
    new = lambda k=n ** 3: np.zeros(k)  # noqa: E731
    # sumorder 2: the order of the device sums (the V-cycle of this mesh amplifies their rounding)
    st_o = R.or_calcdefp(new(), new(), new((n + 2) * n * n), d, u, n, sumorder=2)
    to = lambda a: torch.from_numpy(a).cuda()  # noqa: E731
    st = ctx.calcdefp(to(new()), to(new()), to(new((n + 2) * n * n)), to(d), to(u))
    assert st.nexpand == st_o.nexpand > 0 and st.ncompress == st_o.ncompress > 0
    for f in ("detmin", "detmax", "fluxmin", "fluxmax"):
        assert getattr(st, f) == getattr(st_o, f), f
    assert abs(st.cmax - st_o.cmax) <= 1e-12 * abs(st_o.cmax)  # device acos and cos


@pytest.mark.parametrize("dt", [np.float64, np.float32])
@pytest.mark.parametrize("n,k", [(16, 0), (16, 1), (64, 33)])
def test_limiter_extremes_beside_a_nan(ctx, n, k, dt):
    """A mesh potential that is NaN at one point: the determinant's extremes are those of the other points (of
    a spike two planes away and its mirror images, which the NaN does not reach)."""
    print("case limiter NaN n=%d k=%d %s" % (n, k, dt.__name__), flush=True)
    d = np.zeros((n, n, n), dt)  # [k, j, i]
    d[k, 7, 7] = -1.0            # det = 27 at the spike, and 0 or below around it
    u = np.zeros((n ** 3, 5), dt)
    u[:, 0] = 1.0
    new = lambda m=n ** 3: np.zeros(m, dt)  # noqa: E731
    ref = R.or_calcdefp(new(), new(), new((n + 2) * n * n), d.ravel(), u.ravel(), n, sumorder=2)
    d[k + 2, 7, 7] = np.nan
    to = lambda a: torch.from_numpy(a.ravel()).cuda()  # noqa: E731
    st = ctx.calcdefp(to(new()), to(new()), to(new((n + 2) * n * n)), to(d), to(u))
    assert ref.detmax == 27.0
    assert (st.detmax, st.detmin) == (ref.detmax, ref.detmin)
