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
