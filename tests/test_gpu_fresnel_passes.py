"""GPU checks of the Fresnel entry points' passes against the same step in
numpy FP64: the column widths and element counts of every grid size (one field
and enough fields to fill the chip), outputs in and out of place, and the z
scan's chunks.

Tolerance: a step is four FP32 transforms of at most 13 radix-2 levels and two
products; with 6e-8 a level, (4 x 13 + 2) x 6e-8 = 3.3e-6 relative L2 even if
every error added up."""
import numpy as np
import pytest

from tests.conftest import rel_l2

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

TOL = 3.3e-6


def _field(shape, seed):
    rng = np.random.default_rng(seed)
    return (1.0 + 0.3 * rng.standard_normal(shape) + 0.3j * rng.standard_normal(shape)).astype(np.complex64)


def _step(x, dx, z, lam):
    n = x.shape[-1]
    k = np.where(np.arange(n) < n // 2, np.arange(n), np.arange(n) - n).astype(np.float64)
    co = np.pi * z * lam / (dx * n) / (dx * n)
    h = np.exp(-1j * co * k * k)
    return np.fft.ifft2(np.fft.fft2(x.astype(np.complex128)) * h[:, None] * h[None, :])


@pytest.mark.parametrize("n,batch", [(16, 1), (16, 200), (32, 3), (64, 31), (64, 32), (128, 15), (128, 17), (256, 7),
                                     (256, 9), (512, 1), (512, 4), (1024, 1), (1024, 2), (2048, 1), (4096, 1),
                                     (8192, 1)])
def test_fresnel_sizes(ctx, n, batch):
    print(f"fresnel {batch} x {n}^2", flush=True)
    x = _field((batch, n, n), n + batch)
    t = torch.tensor(x, device="cuda")
    want = _step(x, 0.01, 1500.0, 0.8e-6)
    got = ctx.fresnel(t, 0.01, 1500.0, 0.8e-6)
    assert rel_l2(got.cpu().numpy(), want) < TOL
    assert np.array_equal(t.cpu().numpy(), x)  # out of place: the input stays
    ctx.fresnel(t, 0.01, 1500.0, 0.8e-6, out=t)
    assert torch.equal(t, got)


@pytest.mark.parametrize("n,sign", [(4096, -1), (4096, 1), (8192, -1), (8192, 1)])
def test_fft_large(ctx, n, sign):
    x = _field((n, n), n)
    got = ctx.fft2d(torch.tensor(x, device="cuda"), sign).cpu().numpy()
    z = x.astype(np.complex128)
    assert rel_l2(got, np.fft.fft2(z) if sign < 0 else np.fft.ifft2(z) * n * n) < TOL


# 256 MB of fields are 8 planes of 2048^2: 9 planes are two chunks
@pytest.mark.parametrize("n,nz", [(16, 1), (64, 5), (512, 3), (2048, 9), (4096, 1)])
def test_cube(ctx, n, nz):
    print(f"cube {nz} x {n}^2", flush=True)
    x = _field((n, n), n + nz)
    amp, pha = ctx.fresnel_cube(torch.tensor(x, device="cuda"), 0.01, -500.0, 900.0, nz, 0.8e-6)
    for k in range(nz):
        want = _step(x, 0.01, -500.0 + 1400.0 * k / nz, 0.8e-6)
        a, p = amp[k].cpu().numpy().astype(np.float64), pha[k].cpu().numpy().astype(np.float64)
        assert rel_l2(a * np.exp(1j * p), want) < TOL
