"""The kernels that the tuning keys choose, by the names of the launches (the
library's host code on a stand-in runtime, no kernel runs)."""
from tests import fakehip

_COL = r'''
def col(N, W, **keys):
    """the column kernel of a frame with a row and a column pass per gap"""
    c = ctx()
    tune(c, gap_passes=2, streams=1, **keys)
    s = sim(c, N, [0, 1], W=W)
    p = ptr(64, c)
    log()
    assert L.atsim_sim_frame(s, p, p, None) == OK, err(c)
    k = [n for n in kernels() if n.startswith("k_col")]
    assert len(k) == 1, k
    L.atsim_sim_destroy(s)
    L.atsim_ctx_destroy(c)
    print(N, W, keys, k[0])
    return k[0]

'''


# col_e: the elements per thread asked for, wherever that kernel is built
def test_col_e(tmp_path):
    print(fakehip.run(tmp_path, _COL + r'''
for N, cols in ((4096, 4), (8192, 2)):
    for W in (1, 2):
        assert col(N, W, col_e=16).startswith(f"k_col<{N}, 1, 0, {cols}"), N
        for e in (0, 32):
            assert col(N, W, col_e=e).startswith(f"k_col_split<{N}, 1, 0, {2 * cols}, 32"), N
        assert col(N, W, col_c=2).startswith(f"k_col<{N}, 1, 0, 2"), N
for N in (256, 512, 1024, 2048):
    for W in (1, 3):
        assert col(N, W, col_e=16).startswith(f"k_col<{N}, 1, 0, "), N
        assert col(N, W, col_e=32).startswith(f"k_col_split<{N}, 1, 0, 8, 32"), N
        assert col(N, W, col_e=32, col_c=16).startswith(f"k_col_split<{N}, 1, 0, 16, 32"), N
        assert col(N, W, col_e=32, col_c=4).startswith(f"k_col<{N}, 1, 0, 4"), N
assert col(2048, 1).startswith("k_col<2048") and col(2048, 2).startswith("k_col_split<2048")
'''))


# the column passes' widths by size, number of fields and layers of the group
def test_column_widths(tmp_path):
    print(fakehip.run(tmp_path, _COL + r'''
def wide(N, W, D=1):
    c = ctx()
    p = ptr(64, c)
    log()
    assert L.atsim_fft2d(c, p, N, W * D, -1) == OK
    k = [n for n in kernels() if n.startswith("k_col")][0]
    L.atsim_ctx_destroy(c)
    return int(k.split("<")[1].split(">")[0].split(",")[3])

for N in (16, 32, 64, 128):
    for n in (1, 8, 4096):
        assert wide(N, n) == 16, (N, n)
assert [wide(256, n) for n in (1, 7, 8, 63, 64, 4096)] == [4, 4, 8, 8, 16, 16]
assert [wide(512, n) for n in (1, 3, 4, 512)] == [4, 4, 8, 8]
assert [wide(1024, n) for n in (1, 2, 64)] == [4, 8, 8]
assert [wide(2048, n) for n in (1, 2)] == [8, 8]

def screen(N, W, layers):
    """the column pass of a group of that many layers"""
    c = ctx()
    tune(c, streams=1)
    s = sim(c, N, [g for g in range(3) for _ in range(layers)], W=W)
    p = ptr(64, c)
    log()
    assert L.atsim_sim_frame(s, p, p, None) == OK, err(c)
    k = [n for n in kernels() if n.startswith("k_col_screen")]
    assert len(k) == 1, k
    L.atsim_sim_destroy(s)
    L.atsim_ctx_destroy(c)
    return k[0]

for W, most in ((1, 16), (2, 4), (3, 2), (4, 2)):
    for layers in (1, 2, 3, 4, 5, 8, 16):
        want = 4 if layers <= most else 8
        assert screen(1024, W, layers) == f"k_col_screen<1024, {want}>", (W, layers, screen(1024, W, layers))
assert screen(1024, 5, 1) == "k_col_screen<1024, 8>"
assert screen(2048, 1, 4) == "k_col_screen<2048, 8>" and screen(2048, 2, 1).startswith("k_col_screen_split<2048")
assert screen(512, 3, 16) == "k_col_screen<512, 4>" and screen(512, 4, 16) == "k_col_screen<512, 8>"
'''))
