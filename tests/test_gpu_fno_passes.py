"""GPU checks of the network's fused passes against numpy on the same
BF16-rounded operands (FP64 sums).  The passes accumulate in FP32: at most 64
products per sum and a few roundings after, so 64 ulp of the sum's norm,
4e-6, bounds the relative L2 error."""
import numpy as np
import pytest

from tests.conftest import rel_l2
from tests.test_gpu_fno import bf16

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

TOL = 4e-6


def _dev(*arrays):
    out = [torch.tensor(np.ascontiguousarray(a, np.float32), device="cuda") for a in arrays]
    torch.cuda.synchronize()
    return out


# edges of the 16-channel tiles, the 32-channel steps and the 64-pixel groups
@pytest.mark.parametrize("Cout,Cin,nrows,rowlen", [(1, 1, 1, 4), (2, 64, 3, 60), (16, 32, 5, 64), (17, 33, 2, 68),
                                                   (32, 14, 7, 256), (48, 48, 3, 512), (64, 2, 9, 100)])
@pytest.mark.parametrize("K2", [0, 4, 24, 32, 36, 64])
@pytest.mark.parametrize("act", [0, 1, 2])
def test_pointwise(ctx, Cout, Cin, nrows, rowlen, K2, act):
    from atmosphericturbulencesimul_amd.fno import Ops
    from oracle import fno_ref
    print(f"pointwise {Cout}x{Cin} rows {nrows}x{rowlen} K2 {K2} act {act}", flush=True)
    rng = np.random.default_rng(Cout * 1000 + rowlen + K2)
    W, h = rng.standard_normal((Cin, Cout)), rng.standard_normal((Cin, nrows, rowlen))
    U, F = rng.standard_normal((Cout, nrows, max(K2, 1))), rng.standard_normal((rowlen, max(K2, 1)))
    bias, pre = rng.standard_normal(Cout), rng.standard_normal((Cout, nrows, rowlen))
    tW, th, tU, tF, tb, tp = _dev(W, h, U, F, bias, pre)
    out = torch.empty((Cout, nrows, rowlen), device="cuda")
    torch.cuda.synchronize()
    ops = Ops(ctx)
    assert ops.pointwise_ok(Cout, Cin, rowlen, (th, out, tp, tU), K2)
    # W and F through transposed strides
    ops.pointwise(tW, 1, Cout, Cout, Cin, th, out, nrows, rowlen, tU if K2 else None, K2, tF, 1, K2, tb, tp, act)
    ctx.sync()
    v = np.einsum("ic,irx->crx", bf16(W).astype(np.float64), bf16(h).astype(np.float64))
    if K2:
        v += np.einsum("crk,xk->crx", bf16(U).astype(np.float64), bf16(F).astype(np.float64))
    v += np.float32(bias)[:, None, None]
    want = v if act == 0 else fno_ref.gelu(v) if act == 1 else v * fno_ref.gelu_grad(np.float32(pre).astype(np.float64))
    assert rel_l2(out.cpu().numpy(), want) < TOL
    if act < 2:
        assert rel_l2(tp.cpu().numpy(), v) < TOL


def test_pointwise_refuses_what_it_does_not_take(ctx):
    from atmosphericturbulencesimul_amd.fno import Ops
    ops = Ops(ctx)
    t = torch.zeros(65 * 64 + 4, device="cuda")
    out = torch.empty(65 * 64 + 4, device="cuda")
    assert not ops.pointwise_ok(65, 1, 64, (t, out))
    assert not ops.pointwise_ok(1, 65, 64, (t, out))
    assert not ops.pointwise_ok(8, 8, 63, (t, out))
    assert not ops.pointwise_ok(8, 8, 64, (t[1:], out))
    L = ctx.L
    args = lambda co, ci, h, n: (ctx.h, t.data_ptr(), 1, 1, co, ci, h, out.data_ptr(), 1, n, None, 0, None, 0, 0, None,
                                 None, 0)
    for a in (args(65, 1, t.data_ptr(), 64), args(1, 65, t.data_ptr(), 64), args(8, 8, t.data_ptr(), 63),
              args(8, 8, t.data_ptr() + 4, 64)):
        assert L.atsim_nn_pointwise(*a) == -4  # ATSIM_EUNSUPPORTED


# the transform of out left by the pass that writes it: the spectral path from it
# against the spectral path from out, bit for bit.  Edges of the 16-column tiles
# (8, 9 and 16 modes), of the 64-pixel groups, channels over one tile and one
# step, rows that do not fill the workgroups, the longest rows.
@pytest.mark.parametrize("C,Cin,S,N,m,act,spec", [(1, 1, 1, 32, 1, 0, False), (16, 33, 1, 32, 8, 1, True),
                                                  (17, 32, 2, 96, 9, 2, False), (32, 64, 1, 160, 16, 0, False),
                                                  (32, 32, 5, 64, 16, 1, True), (24, 24, 1, 512, 12, 2, True)])
def test_map_leaves_the_transform_along_x(ctx, C, Cin, S, N, m, act, spec):
    import torch
    from atmosphericturbulencesimul_amd.fno import FNO, Ops
    print(f"map_dft C={C} Cin={Cin} S={S} N={N} m={m} act={act}", flush=True)
    rng = np.random.default_rng(C + N)
    ops = Ops(ctx)
    net = FNO(ctx, N, 2, 2, width=C, modes=m, blocks=1, hidden=4, seed=1)
    f32 = lambda *s: _dev(rng.standard_normal(s))[0]
    W, h, b, pre, U = f32(C, Cin), f32(Cin, S, N, N), f32(C), f32(C, S, N, N), f32(C * S * N, 2 * m)
    kw = dict(U=U, K2=2 * m, F=net.Fxi, sfk=N, sfx=1) if spec else {}
    outs, specs = [], []
    for rows in (False, True):
        out = torch.full((C, S, N, N), np.nan, dtype=torch.float32, device="cuda")
        T = torch.full((C * S * N, 16 * ((m + 7) // 8)), np.nan, dtype=torch.bfloat16, device="cuda") if rows else None
        torch.cuda.synchronize()
        ops.pointwise(W, Cin, 1, C, Cin, h, out, S * N, N, bias=b, pre=pre if act else None, act=act,
                      **kw, **(dict(D=net.Fx, dsk=2 * m, dsn=1, m=m, T=T) if rows else {}))
        B, O = (torch.zeros((C, S, 2 * m, m, 2), dtype=torch.float32, device="cuda") for _ in range(2))
        Us = torch.zeros((C * S * N, 2 * m), dtype=torch.float32, device="cuda")
        torch.cuda.synchronize()
        ops.spectral(out, net.Fx, 2 * m, 1, net.Gre, net.Gim, net.param["R0"], rows, B, O, Us, C, S, N, m, T)
        ctx.sync()
        outs.append(out.cpu().numpy())
        specs.append(B.cpu().numpy())
    assert np.isfinite(outs[0]).all() and np.array_equal(outs[0], outs[1])
    assert np.abs(specs[0]).max() > 0 and np.array_equal(specs[0], specs[1])
    # refused: more channels, more modes, rows of another length
    for C_, m_, N_ in ((33, m, N), (C, 17, N), (C, m, 48), (C, m, 544)):
        assert not ops.rows_ok(C_, N_, m_)
        assert ctx.L.atsim_nn_map_dft(ctx.h, W.data_ptr(), 1, 1, C_, 1, h.data_ptr(), h.data_ptr(), 1, N_, None, 0, None,
                                      0, 0, None, None, 0, net.Fx.data_ptr(), 0, 0, m_, T.data_ptr()) == -4


# a map whose input is lifted in registers against the lift and the map, bit for
# bit: edges of the 16-channel tiles and of one step on both sides
@pytest.mark.parametrize("C,Cl,S,N,m", [(1, 1, 1, 32, 2), (15, 32, 3, 32, 8), (17, 4, 2, 96, 10), (32, 31, 1, 64, 16)])
def test_map_of_a_lift(ctx, C, Cl, S, N, m):
    import torch
    from atmosphericturbulencesimul_amd.fno import FNO, Ops
    print(f"lift C={C} Cl={Cl} S={S} N={N} m={m}", flush=True)
    rng = np.random.default_rng(C + Cl)
    ops = Ops(ctx)
    net = FNO(ctx, N, 2, 2, width=C, modes=m, blocks=1, hidden=4, seed=1)
    f32 = lambda *s: _dev(rng.standard_normal(s))[0]
    L, Lb, W, b, x, U = f32(C, Cl), f32(C), f32(C, C), f32(C), f32(Cl, S, N, N), f32(C * S * N, 2 * m)
    h, o1, o2 = (torch.full((C, S, N, N), np.nan, dtype=torch.float32, device="cuda") for _ in range(3))
    Th, T0, T1, T2 = (torch.zeros((C * S * N, 16 * ((m + 7) // 8)), dtype=torch.bfloat16, device="cuda") for _ in range(4))
    torch.cuda.synchronize()
    rows = dict(D=net.Fx, dsk=2 * m, dsn=1, m=m)
    spec = (U, 2 * m, net.Fxi, N, 1, b, None, 1)
    ops.pointwise(L, Cl, 1, C, Cl, x, h, S * N, N, bias=Lb, T=Th, **rows)
    ops.pointwise(W, C, 1, C, C, h, o1, S * N, N, *spec, T=T1, **rows)
    ops.pointwise(L, Cl, 1, C, Cl, x, None, S * N, N, bias=Lb, T=T0, **rows)
    ops.pointwise(W, C, 1, C, C, x, o2, S * N, N, *spec, T=T2, **rows, L=L, Lb=Lb, Cl=Cl)
    ctx.sync()
    assert np.isfinite(o1.cpu().numpy()).all() and np.array_equal(o1.cpu().numpy(), o2.cpu().numpy())
    assert torch.equal(Th, T0) and torch.equal(T1, T2) and T1.abs().max() > 0


# the fused passes against the general GEMM path, bit for bit: edges of the
# 16-mode tiles, the 32-value steps, channels over one step, odd sample counts
@pytest.mark.parametrize("N,m,width,S,hidden", [(32, 1, 8, 1, 16), (32, 16, 32, 3, 64), (64, 5, 17, 2, 33),
                                                (96, 16, 24, 33, 64), (128, 17, 33, 2, 40), (256, 32, 64, 1, 64),
                                                (160, 20, 48, 17, 32)])
def test_network_matches_the_general_path(ctx, monkeypatch, N, m, width, S, hidden):
    from atmosphericturbulencesimul_amd import fno
    print(f"network N={N} m={m} width={width} S={S} hidden={hidden}", flush=True)
    rng = np.random.default_rng(N + m)
    cin = 5
    x, t = _dev(rng.standard_normal((cin, S, N, N)), rng.standard_normal((2, S, N, N)))

    def step():
        net = fno.FNO(ctx, N, cin, 2, width=width, modes=m, blocks=2, hidden=hidden, seed=3)
        loss = net.loss_and_grads(x, t)
        y = net.forward(x, keep=False)
        ctx.sync()
        return loss, {**{k: v.cpu().numpy() for k, v in net.grad.items()}, "y": y.cpu().numpy()}

    used = []
    spectral = fno.Ops.spectral
    monkeypatch.setattr(fno.Ops, "spectral", lambda self, *a: (used.append(1), spectral(self, *a))[1])
    loss, g = step()
    assert used
    monkeypatch.setattr(fno.Ops, "spectral_ok", staticmethod(lambda *a: False))
    monkeypatch.setattr(fno.Ops, "pointwise_ok", staticmethod(lambda *a: False))
    monkeypatch.setattr(fno.Ops, "weight_grad_ok", staticmethod(lambda *a: False))
    loss0, g0 = step()
    assert loss == loss0
    for k in g0:
        assert np.array_equal(g[k], g0[k]), k


@pytest.mark.parametrize("nb", [1, 2, 127, 128, 129, 512])
@pytest.mark.parametrize("n", [1, 63, 64, 65, 1000])
@pytest.mark.parametrize("accumulate", [0, 1])
def test_reduce_batches_sums_in_order(ctx, nb, n, accumulate):
    rng = np.random.default_rng(nb + n)
    part, out = rng.standard_normal((nb, n)).astype(np.float32), rng.standard_normal(n).astype(np.float32)
    tp, to = _dev(part, out)
    assert ctx.L.atsim_nn_reduce_batches(ctx.h, tp.data_ptr(), to.data_ptr(), nb, n, accumulate) == 0
    ctx.sync()
    want = out.copy() if accumulate else np.zeros(n, np.float32)
    for b in range(nb):
        want = want + part[b]  # float32, ascending
    assert np.array_equal(to.cpu().numpy(), want)


@pytest.mark.parametrize("S,C,P", [(1, 3, 4096), (1, 2, 131072 + 1), (1, 1, 5), (3, 2, 1000)])
def test_bias_grad(ctx, S, C, P):
    rng = np.random.default_rng(P)
    dy = rng.standard_normal((S, C, P)).astype(np.float32)
    t, = _dev(dy)
    db = torch.empty(C, device="cuda")
    torch.cuda.synchronize()
    assert ctx.L.atsim_nn_bias_grad(ctx.h, t.data_ptr(), db.data_ptr(), S, C, P, 0) == 0
    ctx.sync()
    # FP64 chunks rounded to float and 64 of them added: 65 roundings of at most
    # half an ulp of the chunks' magnitudes
    got, want = db.cpu().numpy().astype(np.float64), dy.astype(np.float64).sum((0, 2))
    assert np.all(np.abs(got - want) <= 65 * 2.0 ** -24 * np.abs(dy).astype(np.float64).sum((0, 2)))


# the bias sums made beside the weight gradient: FP64 sums rounded once, so half
# an ulp of the result and the FP64 roundings of the magnitudes' sum
@pytest.mark.parametrize("Cout,Cin,SP,kc", [(1, 1, 128, 128), (16, 17, 3 * 256, 256), (33, 2, 300 * 128, 128),
                                            (64, 64, 2048, 1024)])
def test_weight_and_bias_grad(ctx, Cout, Cin, SP, kc):
    from atmosphericturbulencesimul_amd.fno import Ops
    rng = np.random.default_rng(Cout + SP)
    dy, h = rng.standard_normal((Cout, SP)).astype(np.float32), rng.standard_normal((Cin, SP)).astype(np.float32)
    tdy, th = _dev(dy, h)
    nb = SP // kc
    part, bpart = torch.empty(nb * Cout * Cin, device="cuda"), torch.empty(nb * Cout, dtype=torch.float64, device="cuda")
    gW, gW2, gb = (torch.full((n,), np.nan, device="cuda") for n in (Cout * Cin, Cout * Cin, Cout))
    torch.cuda.synchronize()
    ops = Ops(ctx)
    ops.weight_grad(tdy, th, part, gW, Cout, Cin, SP, kc)
    ops.weight_grad(tdy, th, part, gW2, Cout, Cin, SP, kc, bpart, gb)
    ctx.sync()
    assert np.isfinite(gW.cpu().numpy()).all() and torch.equal(gW, gW2)
    want, mag = dy.astype(np.float64).sum(1), np.abs(dy).astype(np.float64).sum(1)
    assert np.all(np.abs(gb.cpu().numpy() - want) <= 2.0 ** -24 * np.abs(want) + SP * 2.0 ** -53 * mag)


# 1, 32 (one launch) and 33 tensors of sizes about a workgroup
@pytest.mark.parametrize("count", [1, 32, 33])
def test_adam_many_is_adam_of_each(ctx, count):
    from atmosphericturbulencesimul_amd.fno import Ops
    ops = Ops(ctx)
    rng = np.random.default_rng(count)
    sizes = [1, 255, 256, 257, 5000][:count] * (count // 5 + 1)
    sets = [[_dev(*(rng.standard_normal(n) for _ in range(4))) for n in sizes[:count]]]
    for t in sets[0]:
        t[3].abs_()
    sets.append([[x.clone() for x in t] for t in sets[0]])
    torch.cuda.synchronize()
    ops.adam_many([tuple(t) for t in sets[0]], 1e-3, 0.9, 0.999, 1e-8, 3)
    for t in sets[1]:
        ops.adam(*t, 1e-3, 0.9, 0.999, 1e-8, 3)
    ctx.sync()
    for a, b in zip(*sets):
        assert all(torch.equal(x, y) for x, y in zip(a, b))


@pytest.mark.parametrize("n", [1, 1000, 70000])
def test_loss_read_later_is_the_same(ctx, n):
    from atmosphericturbulencesimul_amd.fno import Ops
    ops = Ops(ctx)
    rng = np.random.default_rng(n)
    p, t = _dev(rng.standard_normal(n), rng.standard_normal(n))
    g, g2 = torch.empty_like(p), torch.empty_like(p)
    torch.cuda.synchronize()
    want = ops.mse(p, t, g)
    ops.mse_begin(p, t, g2)
    assert ops.mse_end(n) == want
    ctx.sync()
    assert torch.equal(g, g2)
