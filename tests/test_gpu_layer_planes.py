"""Frames whose phase multipliers do not factor: the extraction reads the layers'
phase planes where a frame has them (unpipelined, one pass per gap) and samples
the layers itself elsewhere (pipelined frames, extract_planes 2).  A frame's
outputs are the same bits either way, as atsim_set_tuning promises of
"pipeline"."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def _frames(N, Nout, W, D, rule, field, **tuning):
    from atmosphericturbulencesimul_amd.api import Context, Simulation
    cx = Context(0)
    try:
        for k, v in tuning.items():
            cx.set_tuning(k, v)
        L = 6
        lam = np.linspace(0.6e-6, 2.0e-6, W)
        sc = np.array([[0.5e-6 / m * (1.0 + 1e-3 * l * (w + 1)) for l in range(L)] for w, m in enumerate(lam)])
        sc[:, 2] *= 1.0 + 1e-5  # (no factors with one wavelength too: b_l a_0 rounds)
        x0 = np.array([[10.3 + 3.7 * d + l for l in range(L)] for d in range(D)])
        s = Simulation(cx, N, Nout, max(N, 256), np.array([0.0, 4000.0, 8000.0, 12000.0]), [0, 0, 1, 2, 2, 3], lam, sc,
                       [rule] * W, x0, x0[:, ::-1], np.linspace(100.0, 900.0, L), np.linspace(-500.0, 700.0, L), 0.02,
                       0.001)
        s.synth_masters(7, 400.0, 1.0)
        s.normalize_masters(6.0, np.array([0.4, 0.2, 0.15, 0.1, 0.1, 0.05]))
        f = torch.empty((D, W, N, N), dtype=torch.complex64, device="cuda") if field else None
        out = []
        for _ in range(4):
            pha, amp = s.frame(f)
            out += [pha.cpu().numpy(), amp.cpu().numpy()] + ([f.cpu().numpy()] if field else [])
        s.close()
        return out
    finally:
        cx.close()


# two chunks of the extraction's wavelengths (9), cropped outputs with edges
# inside a tile, both unwrap rules, the field output
@pytest.mark.parametrize("N,Nout,W,D", [(64, 41, 9, 2), (256, 250, 3, 1), (512, 333, 2, 2), (1024, 1024, 5, 1)])
@pytest.mark.parametrize("rule", [0, 1])
@pytest.mark.parametrize("field", [False, True])
def test_same_bits_with_and_without_planes(N, Nout, W, D, rule, field):
    print(f"layer planes N={N} W={W} D={D} rule={rule} field={field}", flush=True)
    want = _frames(N, Nout, W, D, rule, field)
    for tuning in (dict(extract_planes=2), dict(pipeline=1), dict(pipeline=1, graph=1), dict(graph=1, streams=1)):
        for k, (a, b) in enumerate(zip(want, _frames(N, Nout, W, D, rule, field, **tuning))):
            assert np.array_equal(a, b), (tuning, k, int((a != b).sum()))
