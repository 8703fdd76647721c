"""A context's device memory, events and streams are on the context's device,
whichever device the calling thread has current, and a call leaves the thread's
device as it was.  Two devices of the stand-in runtime: the context is on device
1, every call is made with device 0 current."""
from tests import fakehip

_CODE = r'''
c = ctx(1)
N = 64
p, q = ptr(64 << 20, c), ptr(64 << 20, c)
v = C.c_double()
s = sim(c, N, [0, 1, 2, 3], M=256)
log()

def call(name, *a, rc=OK):
    F.hipSetDevice(0)
    got = getattr(L, name)(*a)
    now = C.c_int(-1)
    F.hipGetDevice(C.byref(now))
    rows = log()
    print(name, got, sorted({r[0] for r in rows}), flush=True)
    assert got == rc, (name, got, err(c))
    assert now.value == 0, f"{name} changed the thread's device"
    wrong = [r for r in rows if r[2] != 1]
    assert not wrong, (name, wrong)
    return rows

made = []
made += call("atsim_fresnel", c, p, q, N, 1, 0.01, 1000.0, 1e-6)        # twiddles, transfer factor
made += call("atsim_fresnel_nm", c, p, q, 48, 30, 1, 0.01, 1000.0, 1e-6)  # line plans, scratch
made += call("atsim_fresnel_nm", c, p, q, 47, 31, 1, 0.01, 1000.0, 1e-6)
made += call("atsim_fft2d_nm", c, p, 61, 97, 2, -1)
made += call("atsim_permut", c, p, 61, 97, 2)
made += call("atsim_fresnel_cube", c, p, q, q, N, 0.01, -100.0, 100.0, 4, 1e-6)
made += call("atsim_make_master", c, p, 128, 50.0, 1.0, 0.0, q, q, None, None)
made += call("atsim_strfn", c, p, 128, 1, 1, C.byref(v))
made += call("atsim_nn_mse_begin", c, p, q, p, 1000)
made += call("atsim_nn_bias_grad", c, p, q, 1, 8, 64, 0)
made += call("atsim_sim_synth_masters", s, 1, (C.c_double * 4)(*[100.0] * 4), (C.c_double * 4)(*[1.0] * 4))
made += call("atsim_sim_stats_enable", s, 1)
made += call("atsim_copy_async", c, 0, p, q, 64)
made += call("atsim_sim_frame", s, p, q, None)
tune(c, pipeline=1)
made += call("atsim_sim_frame", s, p, q, None)                           # second buffer set
tune(c, pipeline=0)
made += call("atsim_sims_frame", C.byref(s), 1, C.byref(p), C.byref(q))
b = np.zeros((3, 3, 2))
dp = lambda a: a.ctypes.data_as(C.POINTER(C.c_double))
made += call("atsim_block_fixup", c, dp(b), 3, dp(np.zeros((3, 3))))
made += call("atsim_sim_autotune", s, p, q, 1, None, 0)
assert {"malloc", "event", "stream", "launch"} <= {r[0] for r in made}
assert sum(r[0] == "malloc" for r in made) >= 12
'''


def test_calls_with_another_device_current(tmp_path):
    print(fakehip.run(tmp_path, _CODE))
