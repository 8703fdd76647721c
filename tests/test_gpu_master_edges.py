"""GPU check of the master synthesis' passes at the sizes where their tiling
changes (one to several row workgroups, partial lag tiles, row 0 / s/2 pairs)
and with the inner limit, against numpy FP64.

Tolerance: the float filter output and two FP32 transforms of at most 11
radix-2 levels (6e-8 each) bound the relative L2 by 1.5e-6; the fit's sums
are of that field's squares, twice that."""
import numpy as np
import pytest

from tests.conftest import rel_l2

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def _want(z, outer, inner, rlim):
    n = z.shape[0]
    f0, fi = n / outer, 5.92 / (2 * np.pi) * n / inner
    k = np.arange(n, dtype=np.float64) - n // 2
    r2 = k[:, None] ** 2 + k[None, :] ** 2
    a = np.exp(-0.5 * r2 / fi / fi) / (r2 + f0 * f0) ** (11.0 / 12.0)
    a[n // 2, n // 2] = 0.0
    if rlim > 0:
        a[np.sqrt(r2) < rlim] = 0.0
    s = np.fft.fft2(np.fft.ifftshift(a * z))
    out, fit = [], []
    for q in (s.real, s.imag):
        c = 0.0
        for lx in (1, 2):
            for ly in (1, 2):
                d = np.mean((q - np.roll(q, (-ly, -lx), (0, 1))) ** 2)
                c += np.log10(d) - 5.0 / 3.0 * np.log10(np.hypot(lx, ly))
        fit.append(10.0 ** (c / 4))
        out.append(q / np.sqrt(fit[-1]))
    return out, fit


@pytest.mark.parametrize("n", [16, 32, 64, 128, 256, 512, 2048])
@pytest.mark.parametrize("rlim", [0.0, 3.5])
@pytest.mark.parametrize("second", [True, False])
def test_master(ctx, n, rlim, second):
    print(f"master {n} rlim {rlim}", flush=True)
    rng = np.random.default_rng(n)
    z = (rng.standard_normal((n, n)) + 1j * rng.standard_normal((n, n))).astype(np.complex64)
    o1, o2, c1, c2 = ctx.make_master(torch.tensor(z, device="cuda"), 0.7 * n, 1.3, rlim=rlim, want_second=second)
    (w1, w2), (f1, f2) = _want(z.astype(np.complex128), 0.7 * n, 1.3, rlim)
    assert abs(c1 / f1 - 1) < 3e-6 and abs(c2 / f2 - 1) < 3e-6
    assert rel_l2(o1.cpu().numpy(), w1) < 3e-6
    if second:
        assert rel_l2(o2.cpu().numpy(), w2) < 3e-6
    else:
        assert o2 is None
