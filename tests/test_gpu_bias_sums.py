"""atsim_nn_bias_grad keeps its chunks' sums in FP64 and rounds once: half an ulp
of the result and the FP64 roundings of the magnitudes' sum, and with accumulate
half an ulp of the total more.  One plane per channel and several, sizes about a
workgroup's loads ahead (8 x 256 values in each of 64 chunks)."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.mark.parametrize("S,Cc,P", [(1, 1, 1), (1, 33, 255), (1, 2, 64 * 8 * 256), (1, 3, 64 * 8 * 256 + 1), (3, 5, 1000),
                                    (7, 2, 40000)])
@pytest.mark.parametrize("accumulate", [0, 1])
def test_bias_grad(ctx, S, Cc, P, accumulate):
    print("bias_grad", S, Cc, P, accumulate, flush=True)
    rng = np.random.default_rng(S * Cc + P)
    dy = (rng.standard_normal((S, Cc, P)) * 10.0 ** rng.uniform(-3, 3, (S, Cc, 1))).astype(np.float32)
    was = rng.standard_normal(Cc).astype(np.float32) * 100
    t, db = torch.tensor(dy, device="cuda"), torch.tensor(was, device="cuda")
    torch.cuda.synchronize()
    p = lambda x: C.c_void_p(x.data_ptr())
    ctx._chk(ctx.L.atsim_nn_bias_grad(ctx.h, p(t), p(db), S, Cc, P, accumulate))
    ctx.sync()
    want, mag = dy.astype(np.float64).sum((0, 2)), np.abs(dy).astype(np.float64).sum((0, 2))
    tol = 2.0 ** -24 * np.abs(want) + S * P * 2.0 ** -53 * mag
    if accumulate:
        want = want + was
        tol = tol + 2.0 ** -24 * (np.abs(want) + tol)
    assert np.all(np.abs(db.cpu().numpy().astype(np.float64) - want) <= tol)
