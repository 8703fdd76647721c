"""The sparse block update against the update over every pixel, bit for bit, in
strong turbulence (every block visited) and weak (few): blocks of 20 x 20 to 39 x
39 pixels (one to six rounds of 4 pixels a lane, whole and partial), remainders
from the planes, from the stored map (a field output, sampled layers, layer planes)
and several fields."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def _frames(N, Nout, r0, factored, field, **tuning):
    from atmosphericturbulencesimul_amd.api import Context, Simulation
    cx = Context(0)
    try:
        for k, v in tuning.items():
            cx.set_tuning(k, v)
        L, W, D = 4, 3, 2
        lam = np.linspace(0.6e-6, 2.0e-6, W)
        sc = np.array([[0.5e-6 / m * (1.0 if factored else 1.0 + 1e-3 * l * w) for l in range(L)]
                       for w, m in enumerate(lam)])
        x0 = np.array([[10.3 + 3.7 * d + l for l in range(L)] for d in range(D)])
        s = Simulation(cx, N, Nout, 256, 4000.0 * np.arange(L), np.arange(L), lam, sc, [1, 0, 1], x0, x0[:, ::-1],
                       np.linspace(100.0, 900.0, L), np.linspace(-500.0, 700.0, L), 0.02, 0.001)
        s.synth_masters(7, 400.0, 1.0)
        s.normalize_masters(r0, np.full(L, 0.25))
        f = torch.empty((D, W, N, N), dtype=torch.complex64, device="cuda") if field else None
        out = [t.cpu().numpy() for _ in range(2) for t in s.frame(f)]
        s.close()
        return out
    finally:
        cx.close()


@pytest.mark.parametrize("N,Nout", [(64, 39), (64, 41), (64, 50), (64, 59), (128, 100), (128, 126), (256, 255)])
@pytest.mark.parametrize("r0", [1.5, 8.0])
@pytest.mark.parametrize("kind", ["planes", "map", "field", "layers"])
def test_sparse_update(N, Nout, r0, kind):
    print("block update", N, Nout, r0, kind, flush=True)
    keys = dict(extract_planes=2) if kind == "map" else {}
    args = (N, Nout, r0, kind != "layers", kind == "field")
    got, want = _frames(*args, **keys), _frames(*args, block_apply=2, **keys)
    assert all(np.array_equal(a, b) for a, b in zip(got, want))
    # (in strong turbulence the update has something to change: wavelengths of the
    # block rule whose phases leave (-pi, pi])
    if r0 < 2:
        assert np.abs(got[0][:, [0, 2]]).max() > np.pi
