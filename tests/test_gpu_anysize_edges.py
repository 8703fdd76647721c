"""GPU checks of the one-pass axis transforms at the edges of their plans:
lengths about the powers of two (direct and Bluestein, transforms of 16 to
8192), narrow and wide column tiles, batches, and more lengths than a context
keeps plans for.

Tolerance: a Bluestein axis is two FP32 transforms of at most 13 radix-2
levels and three products; with a rounding of 6e-8 per level and two axes,
2 x (2 x 13 + 3) x 6e-8 = 3.5e-6 relative L2 even if every error added up; a
Fresnel step has twice as many, 7e-6."""
import numpy as np
import pytest

from tests.conftest import rel_l2

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def _rand(shape, seed):
    rng = np.random.default_rng(seed)
    return (rng.standard_normal(shape) + 1j * rng.standard_normal(shape)).astype(np.complex64)


# (batch, n1, n0): columns of 15..17 and 4 (tiles of 16 and 4), rows of every plan size
@pytest.mark.parametrize("shape", [(1, 2, 15), (2, 16, 17), (3, 17, 16), (1, 31, 32), (5, 33, 64), (70, 65, 12),
                                   (1, 129, 500), (2, 512, 513), (300, 48, 20), (1, 1025, 40), (1, 40, 2047),
                                   (1, 2048, 24), (1, 24, 4096), (1, 4095, 6)])
@pytest.mark.parametrize("sign", [-1, 1])
def test_fft_edges(ctx, shape, sign):
    print("fft2d_nm", shape, sign, flush=True)
    x = _rand(shape, sum(shape))
    g = ctx.fft2d_nm(torch.tensor(x, device="cuda"), sign).cpu().numpy()
    z = x.astype(np.complex128)
    want = np.fft.fft2(z) if sign < 0 else np.fft.ifft2(z) * (shape[1] * shape[2])
    assert rel_l2(g, want) < 3.5e-6


def _fresnel(x, dx, z, lam):
    n1, n0 = x.shape[-2:]
    k = lambda n: np.where(np.arange(n) < n // 2, np.arange(n), np.arange(n) - n).astype(np.float64)
    co = np.pi * z * lam / (dx * n0) / (dx * n0)
    h = np.exp(-1j * co * (k(n1)[:, None] ** 2 + k(n0)[None, :] ** 2))
    return np.fft.ifft2(np.fft.fft2(x.astype(np.complex128)) * h)


@pytest.mark.parametrize("shape", [(1, 2, 2), (2, 14, 16), (1, 16, 18), (3, 64, 128), (2, 130, 62), (40, 100, 256),
                                   (1, 512, 600), (1, 1026, 30), (1, 30, 2050), (1, 4096, 16)])
@pytest.mark.parametrize("in_place", [False, True])
def test_fresnel_even_edges(ctx, shape, in_place):
    print("fresnel_nm", shape, flush=True)
    x = _rand(shape, sum(shape) + 1)
    t = torch.tensor(x, device="cuda")
    g = ctx.fresnel_nm(t, 0.02, 3000.0, 1e-6, out=t if in_place else None)
    assert rel_l2(g.cpu().numpy(), _fresnel(x, 0.02, 3000.0, 1e-6)) < 7e-6
    if not in_place:
        assert np.array_equal(t.cpu().numpy(), x)


def test_more_lengths_than_plans(ctx):
    # 70 odd lengths through one context, then the first again (its plan given
    # back in between)
    first = None
    for n in list(range(3, 143, 2)) + [3]:
        x = _rand((4, n), n)
        g = ctx.fft2d_nm(torch.tensor(x, device="cuda"), -1).cpu().numpy()
        assert rel_l2(g, np.fft.fft2(x.astype(np.complex128))) < 3.5e-6
        first = g if first is None else first
    assert np.array_equal(g, first)
