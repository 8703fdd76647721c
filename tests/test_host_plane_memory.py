"""The optional phase planes of a simulation (those of its row passes, and of
every layer for multipliers that do not factor) never cost it, another
simulation or an atsim_malloc the memory: on a stand-in runtime with a limited
device, whatever fits with the column passes' planes alone is accepted.  The
kernels that are launched tell which planes a frame has."""
import pytest

from tests import fakehip

_CODE = r'''
N, SLI = 256, [0, 0, 1, 2, 2, 3]          # groups of 2, 1, 2 and 1 layers, top to bottom 1, 2, 1, 2
KEYS = dict(W=%(W)d, factored=%(factored)s)
PLANE = 8 * N * N

def frame(s, c):
    p = ptr(64, c)
    log()
    assert L.atsim_sim_frame(s, p, p, None) == OK, err(c)
    k = [n.split("<")[0] + ("(PRE)" if n.startswith("k_row_fresnel") and n.endswith("true>") else "")
         + ("(%%s)" %% n[-2] if n.startswith("k_extract") else "") for n in kernels()]
    L.atsim_free(c, p)
    return k

def full(k):      # the frame of a simulation with every plane
    return "k_row_screen" in k and "k_row_fresnel(PRE)" not in k and (KEYS["factored"] or "k_extract(1)" in k)
def columns(k):   # ... with the column passes' planes only
    return ("k_row_screen" not in k and "k_row_fresnel(PRE)" in k
            and ("k_col_screen" in k or "k_col_screen_split" in k) and "k_extract(1)" not in k)

def used(make):
    c = ctx()
    a = F.fake_used()
    s = make(c)
    n = F.fake_used() - a
    L.atsim_sim_destroy(s)
    assert F.fake_used() <= a + (1 << 16), "not all freed"   # (the context keeps its tables)
    L.atsim_ctx_destroy(c)
    return n

all_bytes = used(lambda c: sim(c, N, SLI, **KEYS))
small_bytes = used(lambda c: (tune(c, row_planes=2), sim(c, N, SLI, **KEYS))[1])
extra = all_bytes - small_bytes
# planes: columns (group 1: 2 layers); rows (group 2: 1 layer; with one wavelength
# group 0 too), and of every layer for the extraction
want = (6 if not KEYS["factored"] else 4 if KEYS["W"] == 1 else 3) - 2
print("bytes", all_bytes, small_bytes, "extra planes", extra // PLANE)
assert extra == want * PLANE, (extra, want)
assert used(lambda c: (tune(c, gap_passes=2), sim(c, N, SLI, **KEYS))[1]) == small_bytes

# a device on which the simulation fits with the column passes' planes alone
for slack in (0, extra - 1, extra, 2 * extra - 1):
    c = ctx()
    F.fake_limit(F.fake_used() + small_bytes + slack)
    rc, s = sim_try(c, N, SLI, **KEYS)
    assert rc == OK, (slack, err(c))
    F.fake_limit(1 << 40)
    assert columns(frame(s, c)), slack
    L.atsim_sim_destroy(s)
    L.atsim_ctx_destroy(c)
# and on which it does not
c = ctx()
F.fake_limit(F.fake_used() + small_bytes - 1)
assert sim_try(c, N, SLI, **KEYS)[0] == ENOMEM
assert F.hipGetLastError() == 0
F.fake_limit(1 << 40)
s = sim(c, N, SLI, **KEYS)
assert full(frame(s, c))

# later allocations take the planes back: atsim_malloc ...
F.fake_limit(F.fake_used() + 4096)
p = C.c_void_p()
assert L.atsim_malloc(c, C.byref(p), 4096 + extra) == OK, err(c)
assert L.atsim_malloc(c, C.byref(C.c_void_p()), 1 << 30) == ENOMEM
L.atsim_free(c, p)
assert columns(frame(s, c)) and columns(frame(s, c))
# (they come back when the tuning is set again and there is room)
F.fake_limit(1 << 40)
tune(c, row_planes=1)
assert full(frame(s, c))
# ... another simulation ...
F.fake_limit(F.fake_used() + small_bytes - extra + (1 << 16))
s2 = sim(c, N, SLI, **KEYS)
assert columns(frame(s, c)) and columns(frame(s2, c))
L.atsim_sim_destroy(s2)
F.fake_limit(1 << 40)
# ... the second buffer set of pipelined frames, with and without graphs ...
for graph in (0, 1):
    tune(c, row_planes=1, graph=graph, pipeline=0)
    s3 = sim(c, N, SLI, **KEYS)
    frame(s3, c), frame(s3, c)
    second = KEYS["W"] * 8 * N * N + (2 * PLANE if KEYS["factored"] else 0)
    F.fake_limit(F.fake_used() + max(4096, second + (1 << 16) - extra))
    tune(c, pipeline=1)
    k = frame(s3, c)
    print("pipelined", graph, sorted(set(k)))
    assert ("k_row_screen" in k) != ("k_row_fresnel(PRE)" in k)
    if second > extra:
        assert columns(k)
    F.fake_limit(1 << 40)
    frame(s3, c), frame(s3, c)
    L.atsim_sim_destroy(s3)
tune(c, pipeline=0, graph=0, row_planes=1)
# ... and work space; the context's own block goes first
frame(s, c)
a = F.fake_used()
q = ptr(1 << 20, c)
assert L.atsim_make_master(c, q, 512, 100.0, 1.0, 0.0, q, q, None, None) == OK
kept = F.fake_used() - a - (1 << 20)
F.fake_limit(F.fake_used())
assert L.atsim_malloc(c, C.byref(p), 1 << 20) == OK, err(c)
F.fake_limit(1 << 40)
assert kept > 1 << 20 and full(frame(s, c))

# the keys, between frames
for key, value, kind in (("row_planes", 2, columns), ("row_planes", 0, full), ("gap_passes", 2, None),
                         ("gap_passes", 1, full), ("extract_planes", 2, None), ("extract_planes", 1, full)):
    tune(c, **{key: value})
    k = frame(s, c)
    print(key, value, sorted(set(k)))
    if kind:
        assert kind(k), (key, value, k)
    elif key == "gap_passes":
        assert "k_row_screen" not in k and "k_col_screen" not in k
assert L.atsim_get_tuning(c, b"row_planes") == 1
assert L.atsim_set_tuning(c, b"row_planes", 3) == EINVAL
L.atsim_sim_destroy(s)
L.atsim_ctx_destroy(c)
'''


@pytest.mark.parametrize("W,factored", [(1, True), (3, True), (3, False)])
def test_optional_planes(tmp_path, W, factored):
    print(fakehip.run(tmp_path, _CODE % dict(W=W, factored=factored)))
