"""What the Python front end sends to the network's own passes (Ops.*_ok) the
library takes: over sizes about every limit and aligned and misaligned operands,
on the stand-in runtime.  A call that the rules let through and the library
refuses would be an exception in a training step that the general product could
have served."""
from tests import fakehip

_CODE = r'''
import random
from atmosphericturbulencesimul_amd.fno import Ops

c = ctx()
base = ptr(1 << 30, c).value

class T:
    def __init__(self, off=0):
        self.p = base + off
    def data_ptr(self):
        return self.p

rng = random.Random(5)
pick = lambda *v: rng.choice(v)
sent = dict(point=0, dft=0, spectral=0, weight=0, tail=0)
for _ in range(60000):
    Cin, Cout = pick(1, 2, 15, 16, 17, 31, 32, 33, 48, 63, 64, 65), pick(1, 2, 15, 16, 17, 31, 32, 33, 48, 63, 64, 65)
    N = pick(4, 16, 30, 32, 36, 64, 96, 100, 128, 160, 256, 320, 384, 480, 512, 516, 544, 992, 1000, 1024, 1056)
    m = pick(1, 2, 3, 4, 7, 8, 12, 15, 16, 17, 20, 24, 31, 32, 33)
    S = pick(1, 2, 3, 50)
    K2 = pick(0, 0, 2 * m)
    h, out, pre, U, R, B, O = (T(pick(0, 0, 0, 0, 0, 16, 8, 4)) for _ in range(7))
    B, O = T(), T()
    pre = pick(None, pre)
    P = lambda t: None if t is None else t.p
    # a channel map, with the inverse transform (K2) and the next transform (rows)
    use_u = K2 > 0
    tensors = (h, out, pre) + ((U,) if use_u else ())
    if Ops.pointwise_ok(Cout, Cin, N, tensors, K2):
        sent["point"] += 1
        a = (base, Cin, 1, Cout, Cin, h.p, out.p, S * N, N, U.p if use_u else None, K2, base if use_u else None, N, 1, base, P(pre), 1)
        assert L.atsim_nn_pointwise(c, *a) == OK, (Cout, Cin, N, K2, err(c))
        if Ops.rows_ok(Cout, N, m) and K2 in (0, 2 * m) and 2 * m <= N:
            sent["dft"] += 1
            assert L.atsim_nn_map_dft(c, *a, base, 2 * m, 1, m, base) == OK, (Cout, Cin, N, m, err(c))
            if use_u and Cin <= 32:
                assert L.atsim_nn_lift_map_dft(c, base, base, 7, *a, base, 2 * m, 1, m, base) == OK, (Cout, Cin, N, m, err(c))
    if use_u and Cin <= 64 and Ops.pointwise_ok(Cin, Cin, N, (h, U), K2):
        sent["tail"] += 1
        assert L.atsim_nn_tail(c, base, Cin, h.p, S * N, N, U.p, K2, base, N, 1, base, base, base, min(Cout, 64), base, base,
                               pick(1, 2, 16), base) == OK, (Cin, N, K2, err(c))
    if Ops.spectral_ok(Cin, N, m, h, R):
        sent["spectral"] += 1
        assert L.atsim_nn_spectral_fwd(c, h.p, base, 2 * m, 1, base, base, R.p, 0, B.p, O.p, base, Cin, S, N, m) == OK, (Cin, N, m, err(c))
        assert L.atsim_nn_mix_grad(c, B.p, O.p, R.p, Cin, S, m) == OK
        if Ops.rows_ok(Cin, N, m):
            assert L.atsim_nn_spectral_rows(c, base, base, base, R.p, 1, B.p, O.p, base, Cin, S, N, m) == OK, (Cin, N, m, err(c))
    SP = pick(128, 256, 1024, 2304, 6400, 57600, (1 << 24) - 128, 1 << 24, (1 << 24) + 128, (1 << 24) + 1024, 18000000, 100, 130)
    kc = 1024 if SP % 1024 == 0 else SP
    if Ops.weight_grad_ok(Cout, Cin, SP, kc, h, out):
        sent["weight"] += 1
        assert L.atsim_nn_weight_bias_grad(c, h.p, out.p, base, base, base, base, Cout, Cin, SP, kc) == OK, (Cout, Cin, SP, err(c))
    if _ % 500 == 0:
        log()
print(sent)
assert min(sent.values()) > 300, sent
'''


def test_rules_ask_for_no_more_than_the_library_takes(tmp_path):
    print(fakehip.run(tmp_path, _CODE))
