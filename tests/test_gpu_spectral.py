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


@pytest.mark.parametrize("n,dt", [(256, np.float64), (256, np.float32), (512, np.float32)])
def test_long_lines_equal_the_oracle(ctx, n, dt):
    """Lines of 128 to 512 points, their workgroups of up to 1024 threads."""
    test_gradient_and_delta_equal_the_oracle(ctx, n, dt)


# ---- lines too long for the oracle's transform of a whole cube: fields that are products of three vectors, so that
# their transforms and derivatives are products of 1-D ones.  The error bound in the 2-norm is t (u + 4 sqrt(2) u)
# < 7 t u for a transform of 2^t points (N. J. Higham, Accuracy and Stability of Numerical Algorithms, theorem
# 24.2) and 6 u more for the recombination: 21 log2(n) u in all three axes.
def separable(n):
    rng = np.random.default_rng(n)
    alt = (-1.0) ** np.arange(n)
    v = [rng.standard_normal(n) for _ in range(3)]
    return [a - (a @ alt) / n * alt for a in v]  # nothing at the Nyquist frequency


class Planes:
    """sum over terms of h[k] g[j] f[i], plane by plane on the device in 64 bits."""

    def __init__(self, *terms):
        self.terms = [[torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in t] for t in terms]

    def __call__(self, k):
        return sum(t[0][k] * t[1][:, None] * t[2][None, :] for t in self.terms)


def distance(got, ref, scale=1.0):
    """2-norms of got - scale ref and of scale ref."""
    d = r = 0.0
    for k in range(got.shape[0]):
        w = scale * ref(k)
        d = d + (got[k] - w).abs().square().sum()
        r = r + w.abs().square().sum()
    return float(d) ** 0.5, float(r) ** 0.5


def device_field(n, ref, dt):
    a = torch.empty(n, n, n, dtype=torch.from_numpy(np.zeros(0, dt)).dtype, device="cuda")
    for k in range(n):
        a[k] = ref(k)
    return a


@pytest.mark.parametrize("dt", [np.float32, np.float64])
def test_derivatives_of_a_separable_field(ctx, dt):
    n = 1024
    print("case spectral separable n=%d %s" % (n, dt.__name__), flush=True)
    f, g, h = separable(n)
    k = np.fft.fftfreq(n, 1.0 / n) * 2 * np.pi / n
    d1 = lambda v: -np.fft.ifft(1j * k * np.fft.fft(v)).real  # noqa: E731  (the transform's sign: exp(+i k x))
    d2 = lambda v: np.fft.ifft(k * k * np.fft.fft(v)).real  # noqa: E731
    eps = 21 * np.log2(n) * float(np.finfo(dt).eps) / 2
    phi = Planes((h, g, f))
    a = device_field(n, phi, dt)
    norm = float(a.double().square().sum()) ** 0.5 if dt == np.float32 else float(a.square().sum()) ** 0.5
    try:
        out = torch.empty(3, n, n, n, dtype=a.dtype, device="cuda")
        ctx.scalar2gradient(a.view(-1), out.view(-1))
        for c, ref in enumerate((Planes((h, g, d1(f))), Planes((h, d1(g), f)), Planes((d1(h), g, f)))):
            d, r = distance(out[c], ref)
            assert d <= eps * (np.pi * norm + r), c
        ctx.defp2delta(a.view(-1), out[0].view(-1))
        d, r = distance(out[0], Planes((h, g, d2(f)), (h, d2(g), f), (d2(h), g, f)))
        assert d <= eps * (3 * np.pi ** 2 * norm + r)
    finally:
        ctx.release_workspace()


@pytest.mark.parametrize("n", [512, 1024, 2048])
def test_rlft3_of_a_separable_field(ctx, n):
    print("case rlft3 separable n=%d" % n, flush=True)
    f, g, h = separable(n)
    F = lambda v: np.conj(np.fft.fft(v))  # noqa: E731
    eps = 21 * np.log2(n) * 2.0 ** -53
    phi = Planes((h, g, f))
    a, sq = device_field(n, phi, np.float64), torch.zeros(2 * n * n, dtype=torch.float64, device="cuda")
    try:
        ctx.rlft3(a.view(-1), sq, 1)
        d, r = distance(torch.view_as_complex(a.view(n, n, n // 2, 2)), Planes((F(h), F(g), F(f)[: n // 2])))
        whole = r * 2 ** 0.5  # with the conjugate half
        assert d <= eps * whole and float(sq.square().sum()) ** 0.5 <= eps * whole
        ctx.rlft3(a.view(-1), sq, -1)
        d, r = distance(a, phi, n ** 3 / 2)
        assert d <= 2 * eps * r
    finally:
        ctx.release_workspace()
