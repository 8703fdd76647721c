"""The kernels that bench.py names for the passes of a frame are the ones the
library launches (its host code on a stand-in runtime), over grid sizes, numbers
of fields, layer groups and tuning keys."""
from tests import fakehip

_CODE = r'''
import bench

def check(N, W, D, lcount, **keys):
    c = ctx()
    tune(c, streams=1, **keys)
    G = len(lcount) - 1
    sli = [g for g in range(G + 1) for _ in range(lcount[G - g])]
    s = sim(c, N, sli, W=W, D=D)
    p = ptr(64, c)
    log()
    assert L.atsim_sim_frame(s, p, p, None) == OK, err(c)
    ran = [n for n in kernels() if n.startswith(("k_row", "k_col"))]
    names = bench.pass_kernels(N, W, D, lcount, lambda k: L.atsim_get_tuning(c, k.encode()))
    one = "col2" in names
    if one:
        assert ran[0] == names["row"], (N, W, D, keys, ran[0], names["row"])
        assert ran[1] == names["col2"], (N, W, D, keys, ran[1], names["col2"])
        assert all(n == names["row2"] for n in ran[2:G:2]), (N, W, D, keys, ran, names)
        if G % 2:
            assert ran[G] == names["col"], (N, W, D, keys, ran[G], names["col"])
    else:
        assert ran[0] == names["row"] and ran[1] == names["col"], (N, W, D, keys, ran, names)
    L.atsim_sim_destroy(s)
    L.atsim_ctx_destroy(c)
    return one

n = 0
for N in (16, 64, 128, 256, 512, 1024, 2048, 4096, 8192):
    for W, D in ((1, 1), (2, 1), (3, 1), (4, 1), (8, 1), (8, 8)):
        for lcount in ([1, 1, 1, 1], [1, 3, 2, 1, 1, 2], [2, 1]):
            for keys in (dict(), dict(gap_passes=2), dict(row_planes=2), dict(col2_e=16), dict(col_e=16),
                         dict(col_e=16, gap_passes=2), dict(col_e=32, gap_passes=2), dict(col_c=8)):
                if keys.get("col_c") and N > 2048:
                    continue
                check(N, W, D, lcount, **keys)
                n += 1
            if 256 <= N <= 2048:
                check(N, W, D, lcount, col2_e=32)
                check(N, W, D, lcount, col_c=16 if N < 2048 else 4)
print(n, "frames")
'''


def test_labels(tmp_path):
    print(fakehip.run(tmp_path, _CODE))
