"""atsim_fresnel_nm from and to overlapping memory, as a program that shifts a
ring of fields by one calls it: the same bits as into memory of its own.  Even
and odd sides, the output before and after the input."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.mark.parametrize("n1,n0,batch", [(450, 600, 3), (30, 62, 40), (61, 97, 3), (64, 48, 1)])
@pytest.mark.parametrize("shift", [1, -1, 17])
def test_overlapping_output(ctx, n1, n0, batch, shift):
    print("overlap", n1, n0, batch, shift, flush=True)
    n = batch * n1 * n0
    off = shift if abs(shift) > 1 else shift * n1 * n0 // 2  # 17: not a row
    g = torch.Generator(device="cuda").manual_seed(n + shift)
    x = torch.view_as_complex(torch.randn((n, 2), generator=g, device="cuda"))
    want = ctx.fresnel_nm(x.clone().view(batch, n1, n0), 0.02, 3000.0, 1e-6).cpu().numpy()
    buf = torch.zeros(n + abs(off), dtype=torch.complex64, device="cuda")
    a, b = (0, off) if off > 0 else (-off, 0)
    src = buf[a:a + n].view(batch, n1, n0)
    dst = buf[b:b + n].view(batch, n1, n0)
    src.copy_(x.view(batch, n1, n0))
    got = ctx.fresnel_nm(src, 0.02, 3000.0, 1e-6, out=dst)
    assert np.array_equal(got.cpu().numpy(), want)
