"""GPU: the register-pass FFT kernels against the oracle's radix-2 transform, at every remainder of
log2 L by 3, the smallest lines, and arrays that start one element off a 16-byte boundary.  The
butterflies and the recombinations round as the oracle's do, so the bar is equality."""
import numpy as np
import pytest

import refbind as R

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def off(a):
    """Device copy of a that starts one element into its allocation."""
    t = torch.empty(a.size + 1, dtype=torch.from_numpy(a).dtype, device="cuda")[1:]
    t.copy_(torch.from_numpy(a))
    return t


def white(n, dt):
    return np.random.default_rng(n).standard_normal(n ** 3).astype(dt)


@pytest.mark.parametrize("dt", [np.float64, np.float32])
@pytest.mark.parametrize("n", [4, 8, 16, 32, 64, 128])
def test_gradient_and_delta_equal_the_oracle(ctx, n, dt):
    print("case spectral n=%d %s" % (n, dt.__name__), flush=True)
    a = white(n, dt)
    g, d = off(np.zeros(3 * n ** 3, dt)), off(np.zeros(n ** 3, dt))
    ad = off(a)
    ctx.scalar2gradient(ad, g)
    ctx.defp2delta(ad, d)
    assert np.array_equal(g.cpu().numpy(), R.or_gradient(a, n))
    assert np.array_equal(d.cpu().numpy(), np.asarray(R.or_delta(a, n)).ravel())
    assert np.array_equal(ad.cpu().numpy(), a)
    ctx.defp2delta(ad, ad)  # in place
    assert np.array_equal(ad.cpu().numpy(), d.cpu().numpy())


@pytest.mark.parametrize("n", [4, 8, 32, 64])
def test_rlft3_both_ways_equals_the_oracle(ctx, n):
    print("case rlft3 n=%d" % n, flush=True)
    a = white(n, np.float64)
    sq = np.zeros(2 * n * n)
    ad, sd = off(a), off(sq)
    for sign in (1, -1):
        R.or_rlft3(a, sq, n, sign)
        ctx.rlft3(ad, sd, sign)
        assert np.array_equal(ad.cpu().numpy(), a) and np.array_equal(sd.cpu().numpy(), sq)


def test_fields_of_more_than_a_launch_are_refused(ctx):
    """2048^3 points: refused, and the field is left as it was."""
    import mmh_amd
    print("case spectral n=2048 refused", flush=True)
    a = torch.zeros(2048 ** 3, dtype=torch.float32, device="cuda")
    a[12345] = 1.0
    for call in (lambda: ctx.defp2delta(a, a), lambda: ctx.nsmooth(a)):
        with pytest.raises(mmh_amd.MmhError) as e:
            call()
        assert e.value.code == mmh_amd.MMH_EINVAL
    assert float(a[12345]) == 1.0 and int(torch.count_nonzero(a[:1 << 20])) == 1
