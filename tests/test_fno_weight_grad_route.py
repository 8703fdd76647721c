"""The weight gradient's pass takes chunks of at most 2^24 pixels; a training
step whose pixels are one longer chunk (a multiple of 128 but not of 1 024, such
as 18 frames of 1000^2) goes through the general product instead of being
refused.  On the CPU, with a stand-in library that keeps the pass's own limit."""
import pytest

torch = pytest.importorskip("torch")

import atmosphericturbulencesimul_amd.fno as F  # noqa: E402


class _Lib:
    """the library's limits on the weight gradient; every other call succeeds"""

    def __init__(self):
        self.calls = []

    def __getattr__(self, name):
        def call(*a):
            self.calls.append(name)
            if name == "atsim_nn_weight_bias_grad":
                SP, kc = a[-2:]
                return 0 if 128 <= kc <= 1 << 24 and kc % 128 == 0 and SP % kc == 0 else 3
            return 0
        return call


class _Ctx:
    device = 0
    stream = None
    h = None

    def __init__(self):
        self.L = _Lib()

    def _chk(self, rc):
        if rc:
            raise RuntimeError(f"refused ({rc})")


@pytest.mark.parametrize("SP,own_pass", [(1 << 24, True), ((1 << 24) + 1024, True), ((1 << 24) - 128, True),
                                         ((1 << 24) + 128, False), (18 * 1000 * 1000, False), (2304, True), (100, False)])
def test_long_chunks_take_the_general_product(SP, own_pass):
    ctx = _Ctx()
    net = F.FNO(ctx, 32, 1, 1, width=1, modes=4, blocks=1, hidden=1, device="cpu")
    z = torch.zeros(1).expand(SP)  # one value standing for SP of them: nothing reads it
    ctx.L.calls.clear()
    net._weight_grad(z, z, torch.zeros(1), torch.zeros(1), 1, 1, SP)
    assert ("atsim_nn_weight_bias_grad" in ctx.L.calls) == own_pass
    assert ("atsim_gemm_bf16" in ctx.L.calls) != own_pass
