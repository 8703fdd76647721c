"""Fourier-neural-operator surrogate of the layer loop (no counterpart in the
reference): a per-layer phase stack -> pupil log-amplitude and diffraction
phase, trained on pairs the simulator generates, served with the plain
Fresnel path as judge and fallback.

Every operation runs in the library's own kernels through the C ABI
(atsim_gemm_bf16 on the matrix cores, atsim_nn_*); torch only holds device
memory, on the library context's stream.

Network and conventions (the same as the FP64 restatement used to check it):
    h0 = Lw x + Lb;  h_{b+1} = act(Wb h_b + Bb + K_b h_b);  y = Q2 GELU(Q1 h + q1b) + q2b
    K_b h = Re IDFT2(R_b(k) DFT2(h)(k)) over ky in [-m, m), kx in [0, m),
    kx > 0 doubled in the inverse (real-input convention), 1/P scaling.
Activations are channel-major over the batch: [C][S][N][N]."""
import ctypes as C
import math

import numpy as np

from . import _lib


def _torch():
    import torch
    return torch


def _p(t):
    return C.c_void_p(t.data_ptr()) if t is not None else None


def on_ctx_stream(fn):
    """run a method with torch's current stream set to the library context's
    stream, so torch allocations and copies are ordered with the kernels"""
    def wrapped(self, *a, **k):
        torch = _torch()
        ctx = self.ctx if hasattr(self, "ctx") else (a[0] if a else k["ctx"])
        with torch.cuda.stream(ctx.stream):
            return fn(self, *a, **k)
    wrapped.__name__ = fn.__name__
    wrapped.__doc__ = fn.__doc__
    return wrapped


class Ops:
    """Thin wrappers of the network entry points of one context."""

    def __init__(self, ctx):
        self.ctx = ctx
        self.L = ctx.L

    def gemm(self, M, N, K, batch, A, a_off, sab, sam, sak, B, b_off, sbb, sbk, sbn, Cm, c_off, scb, scm, scn,
             alpha=1.0, beta=0.0, bias=None, pre=None, gelu=False):
        """C = act(alpha A B + beta C + bias[m]) on float32 tensors with element
        offsets and strides (pre, if given, receives the value before the
        activation); raises before the launch if any operand's last element
        lies outside its tensor"""
        if M > 0 and N > 0 and batch > 0:
            last = lambda off, sb, d: off + (batch - 1) * sb + sum((n - 1) * st for n, st in d)
            if (min(a_off, b_off, c_off) < 0
                    or last(a_off, sab, [(M, sam), (K, sak)]) >= A.numel()
                    or last(b_off, sbb, [(K, sbk), (N, sbn)]) >= B.numel()
                    or last(c_off, scb, [(M, scm), (N, scn)]) >= Cm.numel()
                    or (bias is not None and bias.numel() < M)
                    or (pre is not None and pre.numel() != Cm.numel())):
                raise ValueError(f"gemm operands out of bounds (M {M} N {N} K {K} batch {batch})")
        L = self.L
        pa = C.c_void_p(A.data_ptr() + 4 * a_off)
        pb = C.c_void_p(B.data_ptr() + 4 * b_off)
        pc = C.c_void_p(Cm.data_ptr() + 4 * c_off)
        if bias is None and pre is None and not gelu:
            self.ctx._chk(L.atsim_gemm_bf16(self.ctx.h, M, N, K, batch, alpha, pa, sab, sam, sak, pb, sbb, sbk, sbn,
                                            beta, pc, scb, scm, scn))
        else:
            pp = C.c_void_p(pre.data_ptr() + 4 * c_off) if pre is not None else None
            self.ctx._chk(L.atsim_gemm_bf16_ex(self.ctx.h, M, N, K, batch, alpha, pa, sab, sam, sak, pb, sbb, sbk,
                                               sbn, beta, pc, scb, scm, scn, _p(bias), pp, int(gelu)))

    @staticmethod
    def pointwise_ok(Cout, Cin, rowlen, tensors, K2=0):
        """the sizes and alignments atsim_nn_pointwise takes (K2 > 0: with the
        inverse x transform); the others go through gemm"""
        return (Cout <= 64 and Cin <= 64 and rowlen % 4 == 0
                and all(t.data_ptr() % 16 == 0 for t in tensors if t is not None)
                and (K2 == 0 or (rowlen <= 512 and K2 <= 64 and K2 % 4 == 0)))

    def pointwise(self, W, swm, swk, Cout, Cin, h, out, nrows, rowlen, U=None, K2=0, F=None, sfk=0, sfx=0, bias=None,
                  pre=None, act=0, D=None, dsk=0, dsn=0, m=0, T=None, L=None, Lb=None, Cl=0):
        """out = act(W h [+ U F] [+ bias]) over [C][nrows][rowlen] images; act 0
        identity, 1 GELU (pre keeps its argument), 2 times GELU'(pre).  T: also
        the transform of out along x (table D, m modes), for spectral (out may
        be None); L: the map's input is L h + Lb of Cl channels h"""
        n = nrows * rowlen
        if L is not None and (T is None or U is None or L.numel() < Cin * Cl or Lb.numel() < Cin):
            raise ValueError(f"pointwise lift out of bounds ({Cin} x {Cl} channels)")
        if out is None and T is None:
            raise ValueError("pointwise without an output")
        no = Cout * n if out is None else out.numel()
        if (h.numel() < (Cin if L is None else Cl) * n or no < Cout * n
                or W.numel() <= (Cout - 1) * swm + (Cin - 1) * swk
                or (bias is not None and bias.numel() < Cout) or (pre is not None and pre.numel() != no)
                or (U is not None and (U.numel() < Cout * nrows * K2
                                       or F.numel() <= (K2 - 1) * sfk + (rowlen - 1) * sfx))):
            raise ValueError(f"pointwise operands out of bounds ({Cout} x {Cin} channels, {nrows} rows of {rowlen})")
        if T is not None:
            if (T.numel() < Cout * nrows * 16 * ((m + 7) // 8) or T.element_size() != 2
                    or D.numel() <= (rowlen - 1) * dsk + (2 * m - 1) * dsn):
                raise ValueError(f"pointwise transform out of bounds ({Cout} channels, {nrows} rows, {m} modes)")
            self.ctx._chk(self.L.atsim_nn_lift_map_dft(self.ctx.h, _p(L), _p(Lb), Cl, _p(W), swm, swk, Cout, Cin, _p(h),
                                                       _p(out), nrows, rowlen, _p(U), K2, _p(F), sfk, sfx, _p(bias),
                                                       _p(pre), act, _p(D), dsk, dsn, m, _p(T)))
            return
        self.ctx._chk(self.L.atsim_nn_pointwise(self.ctx.h, _p(W), swm, swk, Cout, Cin, _p(h), _p(out), nrows, rowlen,
                                                _p(U), K2, _p(F), sfk, sfx, _p(bias), _p(pre), act))

    def tail(self, W, C_, h, nrows, rowlen, U, K2, F, sfk, sfx, bias, Q1, q1b, H, Q2, q2b, cout, y):
        """y = Q2 GELU(Q1 (W h + U F + bias) + q1b) + q2b (row-major matrices)"""
        n = nrows * rowlen
        if (h.numel() < C_ * n or y.numel() < cout * n or W.numel() < C_ * C_ or U.numel() < C_ * nrows * K2
                or F.numel() <= (K2 - 1) * sfk + (rowlen - 1) * sfx or bias.numel() < C_ or Q1.numel() < H * C_
                or q1b.numel() < H or Q2.numel() < cout * H or q2b.numel() < cout):
            raise ValueError(f"tail operands out of bounds ({C_}, {H}, {cout} channels, {nrows} rows of {rowlen})")
        self.ctx._chk(self.L.atsim_nn_tail(self.ctx.h, _p(W), C_, _p(h), nrows, rowlen, _p(U), K2, _p(F), sfk, sfx,
                                           _p(bias), _p(Q1), _p(q1b), H, _p(Q2), _p(q2b), cout, _p(y)))

    @staticmethod
    def spectral_ok(C_, N, m, h, R):
        """the sizes and alignments atsim_nn_spectral_fwd takes; the others go
        through gemm"""
        nt, ks = (2 * m + 15) // 16, N // 32
        lds = 2 * (3 * nt * ks * 512 + 32 * ((m + 15) // 16) * (N + 8))
        return (C_ <= 64 and N % 32 == 0 and 2 * m <= N <= 1024 and m <= 32 and lds <= 160 * 1024
                and h.data_ptr() % 16 == 0 and R.data_ptr() % 8 == 0)

    @staticmethod
    def rows_ok(C_, N, m):
        """the sizes at which pointwise takes T and spectral begins from it"""
        return C_ <= 32 and m <= 16 and N % 32 == 0 and N <= 512

    def spectral(self, h, F, sfk, sfn, Gre, Gim, R, adjoint, B, O, U, C_, S, N, m, T=None):
        """B = G (h F), O = R B per mode (adjoint: R^H B), U = G^H O; T: h F as
        pointwise left it"""
        sp = C_ * S * 4 * m * m
        if (h.numel() < C_ * S * N * N or F.numel() <= (N - 1) * sfk + (2 * m - 1) * sfn or Gre.numel() < 2 * m * N
                or Gim.numel() < 2 * m * N or R.numel() < 4 * m * m * C_ * C_ or B.numel() < sp or O.numel() < sp
                or U.numel() < C_ * S * N * 2 * m):
            raise ValueError(f"spectral operands out of bounds ({C_} channels, {S} samples of {N}^2, {m} modes)")
        if T is not None:
            if T.numel() < C_ * S * N * 16 * ((m + 7) // 8):
                raise ValueError(f"spectral rows out of bounds ({C_} channels, {S} samples of {N}^2, {m} modes)")
            self.ctx._chk(self.L.atsim_nn_spectral_rows(self.ctx.h, _p(T), _p(Gre), _p(Gim), _p(R), int(adjoint), _p(B),
                                                        _p(O), _p(U), C_, S, N, m))
            return
        self.ctx._chk(self.L.atsim_nn_spectral_fwd(self.ctx.h, _p(h), _p(F), sfk, sfn, _p(Gre), _p(Gim), _p(R),
                                                   int(adjoint), _p(B), _p(O), _p(U), C_, S, N, m))

    def mix_grad(self, dO, B, dR, C_, S, m):
        """dR = dO B^H per mode over the samples"""
        if min(dO.numel(), B.numel()) < C_ * S * 4 * m * m or dR.numel() < 4 * m * m * C_ * C_:
            raise ValueError("mix_grad: operands too small")
        self.ctx._chk(self.L.atsim_nn_mix_grad(self.ctx.h, _p(dO), _p(B), _p(dR), C_, S, m))

    @staticmethod
    def weight_grad_ok(Cout, Cin, SP, kc, dy, h):
        """the sizes and alignments atsim_nn_weight_grad takes; the others go
        through gemm and reduce"""
        return (Cout <= 64 and Cin <= 64 and kc % 128 == 0 and kc <= 1 << 24 and SP % kc == 0
                and dy.data_ptr() % 16 == 0 and h.data_ptr() % 16 == 0)

    def weight_grad(self, dy, h, part, gW, Cout, Cin, SP, kc, bpart=None, gb=None):
        """gW = dy h^T over SP pixels, in chunks of kc (gb: also the sums of dy)"""
        if (dy.numel() < Cout * SP or h.numel() < Cin * SP or part.numel() < SP // kc * Cout * Cin
                or gW.numel() < Cout * Cin):
            raise ValueError("weight_grad: operands too small")
        if gb is not None and (gb.numel() != Cout or bpart.numel() < SP // kc * Cout or bpart.element_size() != 8):
            raise ValueError("weight_grad: bias operands too small")
        self.ctx._chk(self.L.atsim_nn_weight_bias_grad(self.ctx.h, _p(dy), _p(h), _p(part), _p(gW), _p(bpart), _p(gb),
                                                       Cout, Cin, SP, kc))

    def add_bias_act(self, a, b, bias, pre, y, Cc, P, gelu):
        n = a.numel()
        if any(t is not None and t.numel() != n for t in (b, pre, y)) or (bias is not None and bias.numel() != Cc):
            raise ValueError("add_bias_act: operand sizes differ")
        self.ctx._chk(self.L.atsim_nn_add_bias_act(self.ctx.h, _p(a), _p(b), _p(bias), _p(pre), _p(y), Cc, P,
                                                   a.numel(), int(gelu)))

    def gelu_bwd(self, pre, dy, dx):
        if not pre.numel() == dy.numel() == dx.numel():
            raise ValueError(f"gelu_bwd: sizes {pre.numel()}, {dy.numel()}, {dx.numel()} differ")
        self.ctx._chk(self.L.atsim_nn_gelu_bwd(self.ctx.h, _p(pre), _p(dy), _p(dx), pre.numel()))

    def bias_grad(self, dy, db, Cc, P):
        if dy.numel() != Cc * P or db.numel() != Cc:
            raise ValueError("bias_grad: operand sizes differ")
        self.ctx._chk(self.L.atsim_nn_bias_grad(self.ctx.h, _p(dy), _p(db), 1, Cc, P, 0))

    def mse(self, pred, target, grad, want_loss=True):
        if target.numel() != pred.numel() or (grad is not None and grad.numel() != pred.numel()):
            raise ValueError("mse: operand sizes differ")
        loss = C.c_double()
        self.ctx._chk(self.L.atsim_nn_mse(self.ctx.h, _p(pred), _p(target), _p(grad), pred.numel(),
                                          C.byref(loss) if want_loss else None))
        return loss.value if want_loss else None

    def mse_begin(self, pred, target, grad):
        """queue the loss; mse_end waits for it alone and returns it"""
        if target.numel() != pred.numel() or grad.numel() != pred.numel():
            raise ValueError("mse: operand sizes differ")
        self.ctx._chk(self.L.atsim_nn_mse_begin(self.ctx.h, _p(pred), _p(target), _p(grad), pred.numel()))

    def mse_end(self, n):
        loss = C.c_double()
        self.ctx._chk(self.L.atsim_nn_mse_end(self.ctx.h, n, C.byref(loss)))
        return loss.value

    def reduce(self, part, out, nb, n):
        if part.numel() < nb * n or out.numel() < n:
            raise ValueError("reduce: operands too small")
        self.ctx._chk(self.L.atsim_nn_reduce_batches(self.ctx.h, _p(part), _p(out), nb, n, 0))

    def adam(self, w, g, m, v, lr, b1, b2, eps, step):
        if not w.numel() == g.numel() == m.numel() == v.numel():
            raise ValueError("adam: operand sizes differ")
        self.ctx._chk(self.L.atsim_nn_adam(self.ctx.h, _p(w), _p(g), _p(m), _p(v), w.numel(), lr, b1, b2, eps,
                                           step))


    def adam_many(self, tensors, lr, b1, b2, eps, step):
        """one Adam step on every (w, g, m, v) of tensors"""
        if any(not w.numel() == g.numel() == m.numel() == v.numel() for w, g, m, v in tensors):
            raise ValueError("adam: operand sizes differ")
        k = len(tensors)
        ptrs = [(C.c_void_p * k)(*[t[q].data_ptr() for t in tensors]) for q in range(4)]
        n = (C.c_long * k)(*[t[0].numel() for t in tensors])
        self.ctx._chk(self.L.atsim_nn_adam_many(self.ctx.h, k, *ptrs, n, lr, b1, b2, eps, step))


def init_params(cin, cout, width, modes, blocks, hidden, seed=0):
    """float64 numpy parameters; R_b complex [2m][m][width][width]"""
    rng = np.random.default_rng(seed)
    u = lambda shape, fan: rng.uniform(-1.0, 1.0, shape) / math.sqrt(fan)
    p = {"Lw": u((width, cin), cin), "Lb": u((width,), cin)}
    for b in range(blocks):
        p[f"W{b}"] = u((width, width), width)
        p[f"B{b}"] = u((width,), width)
        sc = 1.0 / (width * width)
        p[f"R{b}"] = sc * (rng.uniform(0, 1, (2 * modes, modes, width, width))
                           + 1j * rng.uniform(0, 1, (2 * modes, modes, width, width)))
    p["Q1"] = u((hidden, width), width)
    p["q1b"] = u((hidden,), width)
    p["Q2"] = u((cout, hidden), hidden)
    p["q2b"] = u((cout,), hidden)
    return p


class FNO:
    """The network on the GPU: parameters, forward, backward, Adam."""

    @on_ctx_stream
    def __init__(self, ctx, N, cin, cout, width=32, modes=16, blocks=4, hidden=64, params=None, seed=0,
                 device=None):
        torch = _torch()
        self.ctx, self.ops = ctx, Ops(ctx)
        self.N, self.cin, self.cout, self.width, self.m, self.blocks, self.hidden = N, cin, cout, width, modes, \
            blocks, hidden
        self.dev = device or f"cuda:{ctx.device}"
        if params is None:
            params = init_params(cin, cout, width, modes, blocks, hidden, seed)
        self.param = {}
        for k, v in params.items():
            a = np.asarray(v)
            if np.iscomplexobj(a):
                a = np.stack([a.real, a.imag], axis=-1)
            self.param[k] = torch.tensor(np.ascontiguousarray(a, np.float32), device=self.dev)
        self.grad = {k: torch.zeros_like(v) for k, v in self.param.items()}
        self.adam_m = {k: torch.zeros_like(v) for k, v in self.param.items()}
        self.adam_v = {k: torch.zeros_like(v) for k, v in self.param.items()}
        self.step = 0
        self._tables()

    # ---------------------------------------------------------------- DFT tables
    def _tables(self):  # called from __init__ (on the context stream)
        torch = _torch()
        N, m = self.N, self.m
        x = np.arange(N)
        kx = np.arange(m)
        ky = np.concatenate([np.arange(m), np.arange(N - m, N)])
        ax = 2 * np.pi * np.outer(x, kx) / N                   # [N][m]
        Fx = np.empty((N, 2 * m))
        Fx[:, 0::2] = np.cos(ax)
        Fx[:, 1::2] = -np.sin(ax)
        ay = 2 * np.pi * np.outer(ky, x) / N                   # [2m][N]
        w = np.where(kx == 0, 1.0, 2.0) / (N * N)
        Fxi = np.empty((2 * m, N))
        Fxi[0::2, :] = (w[:, None] * np.cos(ax.T))
        Fxi[1::2, :] = (-w[:, None] * np.sin(ax.T))
        f = lambda a: torch.tensor(np.ascontiguousarray(a, np.float32), device=self.dev)
        self.Fx, self.Gre, self.Gim, self.Fxi = f(Fx), f(np.cos(ay)), f(-np.sin(ay)), f(Fxi)

    # ---------------------------------------------------------------- building blocks
    def _rows(self, out, R, Cin, S, K2, tensors, adjoint=False):
        """The transform along x that the pass writing out is to leave for the
        spectral path of out with R (adjoint: the backward path's table), as the
        last arguments of Ops.pointwise, if both passes take these sizes"""
        N, m, Cw = self.N, self.m, self.width
        if not (self.ops.rows_ok(Cw, N, m) and self.ops.spectral_ok(Cw, N, m, out, R)
                and self.ops.pointwise_ok(Cw, Cin, N, (out,) + tensors, K2)):
            return {}
        torch = _torch()
        D = (self.Fxi, 1, N) if adjoint else (self.Fx, 2 * m, 1)
        T = torch.empty((Cw * S * N, 16 * ((m + 7) // 8)), dtype=torch.bfloat16, device=self.dev)
        return dict(D=D[0], dsk=D[1], dsn=D[2], m=m, T=T)

    def _pointwise(self, Wt, h, out, Cout, Cin, SP, bias=None, pre=None, gelu=False, rows={}):
        # out[o][q] = act(sum_i W[o][i] h[i][q] + bias[o])
        if self.ops.pointwise_ok(Cout, Cin, self.N, (h, out, pre)):
            self.ops.pointwise(Wt, Cin, 1, Cout, Cin, h, out, SP // self.N, self.N, bias=bias, pre=pre, act=int(gelu),
                               **rows)
            return
        self.ops.gemm(Cout, SP, Cin, 1, Wt, 0, 0, Cin, 1, h, 0, 0, SP, 1, out, 0, 0, SP, 1, bias=bias, pre=pre,
                      gelu=gelu)

    def _pointwise_t(self, Wt, dy, out, Cout, Cin, SP, pre=None, rows={}):
        # out[i][q] = sum_o W[o][i] dy[o][q], times GELU'(pre[i][q]) if pre is given
        if self.ops.pointwise_ok(Cin, Cout, self.N, (dy, out, pre)):
            self.ops.pointwise(Wt, 1, Cin, Cin, Cout, dy, out, SP // self.N, self.N, pre=pre,
                               act=2 if pre is not None else 0, **rows)
            return
        self.ops.gemm(Cin, SP, Cout, 1, Wt, 0, 0, 1, Cin, dy, 0, 0, SP, 1, out, 0, 0, SP, 1)
        if pre is not None:
            self.ops.gelu_bwd(pre, out, out)

    def _weight_grad(self, dy, h, gW, gb, Cout, Cin, SP):
        # gW[o][i] = sum_q dy[o][q] h[i][q] and gb[o] = sum_q dy[o][q], split over K chunks, partials summed in order
        torch = _torch()
        kc = 1024 if SP % 1024 == 0 else SP
        nb = SP // kc
        part = torch.empty((nb, Cout, Cin), dtype=torch.float32, device=self.dev)
        if self.ops.weight_grad_ok(Cout, Cin, SP, kc, dy, h):
            bpart = torch.empty((nb, Cout), dtype=torch.float64, device=self.dev)
            self.ops.weight_grad(dy, h, part, gW, Cout, Cin, SP, kc, bpart, gb)
            return
        self.ops.gemm(Cout, Cin, kc, nb, dy, 0, kc, SP, 1, h, 0, kc, 1, SP, part, 0, Cout * Cin, Cin, 1)
        self.ops.reduce(part, gW, nb, Cout * Cin)
        self.ops.bias_grad(dy, gb, Cout, SP)

    def _spectral(self, h, R, S, T=None):
        """U [C][S][N][2m], the retained spectrum of K h transformed back along y,
        and the retained spectrum B [C][S][2m][m][2] of h (T: h's transform along
        x, from the pass that wrote h)"""
        torch = _torch()
        N, m, Cw = self.N, self.m, self.width
        rows = Cw * S * N
        cs = Cw * S
        B = torch.empty((Cw, S, 2 * m, m, 2), dtype=torch.float32, device=self.dev)
        O = torch.empty_like(B)
        U = torch.empty((rows, 2 * m), dtype=torch.float32, device=self.dev)
        if self.ops.spectral_ok(Cw, N, m, h, R):
            self.ops.spectral(h, self.Fx, 2 * m, 1, self.Gre, self.Gim, R, False, B, O, U, Cw, S, N, m, T)
            return U, B
        T1 = torch.empty((rows, 2 * m), dtype=torch.float32, device=self.dev)
        self.ops.gemm(rows, 2 * m, N, 1, h, 0, 0, N, 1, self.Fx, 0, 0, 2 * m, 1, T1, 0, 0, 2 * m, 1)
        self._cmat_left(self.Gre, self.Gim, T1, B, cs, transpose=False)
        self._mix(R, B, O, S)
        self._cmat_left_inv(O, U, cs)
        return U, B

    def _map_add(self, W, swm, swk, h, U, F, sfk, sfx, out, SP, bias=None, pre=None, act=0, rows={}):
        """out = act(W h + U F + bias): a block's 1x1 map with the inverse x
        transform of its spectral path (U, table F) in the same pass; act as
        Ops.pointwise"""
        N, K2, Cw = self.N, 2 * self.m, self.width
        if self.ops.pointwise_ok(Cw, Cw, N, (h, out, pre, U), K2):
            self.ops.pointwise(W, swm, swk, Cw, Cw, h, out, SP // N, N, U, K2, F, sfk, sfx, bias, pre, act,
                               **rows)
            return
        g = self.ops.gemm
        g(Cw * SP // N, N, K2, 1, U, 0, 0, K2, 1, F, 0, 0, sfk, sfx, out, 0, 0, N, 1)
        g(Cw, SP, Cw, 1, W, 0, 0, swm, swk, h, 0, 0, SP, 1, out, 0, 0, SP, 1, beta=1.0, bias=bias,
          pre=pre if act < 2 else None, gelu=act == 1)
        if act == 2:
            self.ops.gelu_bwd(pre, out, out)

    def _cmat_left(self, Gre, Gim, T, Bout, batch, transpose):
        """Bout[b] (2m x m complex) = G (2m x N complex) T[b] (N x m complex, interleaved columns)"""
        N, m = self.N, self.m
        g = self.ops.gemm
        ts, bs = N * 2 * m, 4 * m * m
        # Bre = Gre Tre - Gim Tim ; Bim = Gre Tim + Gim Tre
        g(2 * m, m, N, batch, Gre, 0, 0, N, 1, T, 0, ts, 2 * m, 2, Bout, 0, bs, 2 * m, 2)
        g(2 * m, m, N, batch, Gim, 0, 0, N, 1, T, 1, ts, 2 * m, 2, Bout, 0, bs, 2 * m, 2, alpha=-1.0, beta=1.0)
        g(2 * m, m, N, batch, Gre, 0, 0, N, 1, T, 1, ts, 2 * m, 2, Bout, 1, bs, 2 * m, 2)
        g(2 * m, m, N, batch, Gim, 0, 0, N, 1, T, 0, ts, 2 * m, 2, Bout, 1, bs, 2 * m, 2, beta=1.0)

    def _cmat_left_inv(self, O, U, batch):
        """U[b] (N x m complex, interleaved) = G^H O[b]: Ure = Gre^T Ore + Gim^T Oim, Uim = Gre^T Oim - Gim^T Ore"""
        N, m = self.N, self.m
        g = self.ops.gemm
        us, os_ = N * 2 * m, 4 * m * m
        g(N, m, 2 * m, batch, self.Gre, 0, 0, 1, N, O, 0, os_, 2 * m, 2, U, 0, us, 2 * m, 2)
        g(N, m, 2 * m, batch, self.Gim, 0, 0, 1, N, O, 1, os_, 2 * m, 2, U, 0, us, 2 * m, 2, beta=1.0)
        g(N, m, 2 * m, batch, self.Gre, 0, 0, 1, N, O, 1, os_, 2 * m, 2, U, 1, us, 2 * m, 2)
        g(N, m, 2 * m, batch, self.Gim, 0, 0, 1, N, O, 0, os_, 2 * m, 2, U, 1, us, 2 * m, 2, alpha=-1.0, beta=1.0)

    def _mix(self, R, B, O, S):
        """O[o][s][k] = sum_i R[k][o][i] B[i][s][k] (complex), one GEMM batch per mode"""
        m, Cw = self.m, self.width
        nm = 2 * m * m
        g = self.ops.gemm
        ra = (2 * Cw * Cw, 2 * Cw, 2)          # sab, sam, sak of R
        bb = (2, S * 2 * nm, 2 * nm)           # sbb, sbk, sbn of B (i, s)
        cc = (2, S * 2 * nm, 2 * nm)
        g(Cw, S, Cw, nm, R, 0, *ra, B, 0, *bb, O, 0, *cc)
        g(Cw, S, Cw, nm, R, 1, *ra, B, 1, *bb, O, 0, *cc, alpha=-1.0, beta=1.0)
        g(Cw, S, Cw, nm, R, 0, *ra, B, 1, *bb, O, 1, *cc)
        g(Cw, S, Cw, nm, R, 1, *ra, B, 0, *bb, O, 1, *cc, beta=1.0)

    def _spectral_backward(self, g_out, R, B, S, dR, T=None):
        """dR (written) from the upstream gradient g_out [C][S][N][N] (T: its
        transform along x, from the pass that wrote it); returns dT1
        [C][S][N][2m], whose product with Fx^T is the gradient of h"""
        torch = _torch()
        N, m, Cw = self.N, self.m, self.width
        rows, cs, nm = Cw * S * N, Cw * S, 2 * m * m
        gm = self.ops.gemm
        if self.ops.spectral_ok(Cw, N, m, g_out, R) and dR.data_ptr() % 8 == 0:
            # the adjoint has the forward path's form: dO = G (g Fxi^T), dB = R^H dO,
            # dT1 = G^H dB
            dO = torch.empty((Cw, S, 2 * m, m, 2), dtype=torch.float32, device=self.dev)
            dB = torch.empty_like(dO)
            dT1 = torch.empty((rows, 2 * m), dtype=torch.float32, device=self.dev)
            self.ops.spectral(g_out, self.Fxi, 1, N, self.Gre, self.Gim, R, True, dO, dB, dT1, Cw, S, N, m,
                              T)
            self.ops.mix_grad(dO, B, dR, Cw, S, m)
            return dT1
        dU = torch.empty((rows, 2 * m), dtype=torch.float32, device=self.dev)
        gm(rows, 2 * m, N, 1, g_out, 0, 0, N, 1, self.Fxi, 0, 0, 1, N, dU, 0, 0, 2 * m, 1)
        dO = torch.empty((Cw, S, 2 * m, m, 2), dtype=torch.float32, device=self.dev)
        # dOre = Gre dUre - Gim dUim ; dOim = Gim dUre + Gre dUim
        self._cmat_left(self.Gre, self.Gim, dU, dO, cs, transpose=False)
        # (the same form as the forward y-DFT: G applied to the interleaved dU)
        dB = torch.empty_like(dO)
        ra_t = (2 * Cw * Cw, 2, 2 * Cw)        # R^T: (i, o) -> sam = 2, sak = 2 Cw
        ob = (2, S * 2 * nm, 2 * nm)
        # dBre = Rre^T dOre + Rim^T dOim ; dBim = Rre^T dOim - Rim^T dOre
        gm(Cw, S, Cw, nm, R, 0, *ra_t, dO, 0, *ob, dB, 0, *ob)
        gm(Cw, S, Cw, nm, R, 1, *ra_t, dO, 1, *ob, dB, 0, *ob, beta=1.0)
        gm(Cw, S, Cw, nm, R, 0, *ra_t, dO, 1, *ob, dB, 1, *ob)
        gm(Cw, S, Cw, nm, R, 1, *ra_t, dO, 0, *ob, dB, 1, *ob, alpha=-1.0, beta=1.0)
        # dRre = dOre Bre^T + dOim Bim^T ; dRim = dOim Bre^T - dOre Bim^T   (contract over s)
        oa = (2, S * 2 * nm, 2 * nm)           # dO as (o, s): sab, sam, sak
        bt = (2, 2 * nm, S * 2 * nm)           # B^T as (s, i): sbb, sbk, sbn
        rc = (2 * Cw * Cw, 2 * Cw, 2)
        gm(Cw, Cw, S, nm, dO, 0, *oa, B, 0, *bt, dR, 0, *rc)
        gm(Cw, Cw, S, nm, dO, 1, *oa, B, 1, *bt, dR, 0, *rc, beta=1.0)
        gm(Cw, Cw, S, nm, dO, 1, *oa, B, 0, *bt, dR, 1, *rc)
        gm(Cw, Cw, S, nm, dO, 0, *oa, B, 1, *bt, dR, 1, *rc, alpha=-1.0, beta=1.0)
        # dT1re = Gre^T dBre + Gim^T dBim ; dT1im = Gre^T dBim - Gim^T dBre  (the inverse-y form)
        dT1 = torch.empty((rows, 2 * m), dtype=torch.float32, device=self.dev)
        self._cmat_left_inv(dB, dT1, cs)
        return dT1

    # ---------------------------------------------------------------- forward / backward
    @on_ctx_stream
    def forward(self, x, keep=True):
        """x [cin][S][N][N] float32 -> y [cout][S][N][N]"""
        torch = _torch()
        N, S = self.N, x.shape[1]
        SP = S * N * N
        Cw, p, ops = self.width, self.param, self.ops
        cache = {"x": x, "S": S}
        first = 0
        h = torch.empty((Cw, S, self.N, self.N), dtype=torch.float32, device=self.dev)
        # nothing is kept: the first image is not written, the lift leaves its
        # transform and block 0's map makes it again from x
        lift = {} if keep or self.blocks < 2 or self.cin > 32 else \
            self._rows(h, p["R1"], self.cin, S, 2 * self.m, (x,))
        if lift and self.ops.spectral_ok(Cw, N, self.m, h, p["R0"]):
            ops.pointwise(p["Lw"], self.cin, 1, Cw, self.cin, x, None, S * N, N, bias=p["Lb"], **lift)
            U, _ = self._spectral(h, p["R0"], S, lift["T"])
            rows = self._rows(h, p["R1"], self.cin, S, 2 * self.m, (x, U))
            ops.pointwise(p["W0"], Cw, 1, Cw, Cw, x, h, S * N, N, U, 2 * self.m, self.Fxi, N, 1, p["B0"], None,
                          1, **rows, L=p["Lw"], Lb=p["Lb"], Cl=self.cin)
            first = 1
        else:
            rows = self._rows(h, p["R0"], self.cin, S, 0, (x,)) if self.blocks > 0 else {}
            self._pointwise(p["Lw"], x, h, Cw, self.cin, SP, bias=p["Lb"], rows=rows)
        for b in range(first, self.blocks):
            # hn = act(W h + K h + B): the 1x1 map adds the spectral path's
            # inverse x transform, its bias and activation in one pass
            U, B = self._spectral(h, p[f"R{b}"], S, rows.get("T"))
            if not keep and b == self.blocks - 1 and self.cout <= 16 and self.hidden <= 64 \
                    and ops.pointwise_ok(Cw, Cw, N, (h, U), 2 * self.m):
                # nothing is kept: the last map and both projections in one pass
                y = torch.empty((self.cout, S, N, N), dtype=torch.float32, device=self.dev)
                ops.tail(p[f"W{b}"], Cw, h, S * N, N, U, 2 * self.m, self.Fxi, N, 1, p[f"B{b}"], p["Q1"], p["q1b"],
                         self.hidden, p["Q2"], p["q2b"], self.cout, y)
                return y
            hn = torch.empty_like(h)
            pre = torch.empty_like(h) if keep else None
            rows = self._rows(hn, p[f"R{b + 1}"], Cw, S, 2 * self.m, (h, pre, U)) if b < self.blocks - 1 else {}
            self._map_add(p[f"W{b}"], Cw, 1, h, U, self.Fxi, N, 1, hn, SP, bias=p[f"B{b}"], pre=pre,
                          act=int(b < self.blocks - 1), rows=rows)
            if keep:
                cache[f"h{b}"], cache[f"pre{b}"], cache[f"B{b}"] = h, pre, B
            h = hn
        cache["hL"] = h
        q1 = torch.empty((self.hidden, S, self.N, self.N), dtype=torch.float32, device=self.dev)
        preq = torch.empty_like(q1) if keep else None
        self._pointwise(p["Q1"], h, q1, self.hidden, Cw, SP, bias=p["q1b"], pre=preq, gelu=True)
        y = torch.empty((self.cout, S, self.N, self.N), dtype=torch.float32, device=self.dev)
        self._pointwise(p["Q2"], q1, y, self.cout, self.hidden, SP, bias=p["q2b"])
        if keep:
            cache["preq"], cache["q1"] = preq, q1
            self.cache = cache
        return y

    @on_ctx_stream
    def loss_and_grads(self, x, t, want_loss=True):
        """forward + backward; gradients land in self.grad; returns the MSE loss
        (None without want_loss, which spares a stream synchronisation)"""
        torch = _torch()
        y = self.forward(x, keep=True)
        c, p, g, ops = self.cache, self.param, self.grad, self.ops
        S = c["S"]
        P = self.N * self.N
        SP = S * P
        Cw, H = self.width, self.hidden
        dy = torch.empty_like(y)
        if want_loss:  # read after the backward pass is queued, so that it does not wait for the host
            ops.mse_begin(y, t, dy)
        else:
            ops.mse(y, t, dy, False)
        self._weight_grad(dy, c["q1"], g["Q2"], g["q2b"], self.cout, H, SP)
        dq1 = torch.empty_like(c["q1"])
        self._pointwise_t(p["Q2"], dy, dq1, self.cout, H, SP, pre=c["preq"])
        self._weight_grad(dq1, c["hL"], g["Q1"], g["q1b"], H, Cw, SP)
        dh = torch.empty_like(c["hL"])
        nb = self.blocks
        rows = self._rows(dh, p[f"R{nb - 1}"], H, S, 0, (dq1,), True) if nb > 0 else {}
        self._pointwise_t(p["Q1"], dq1, dh, H, Cw, SP, rows=rows)
        for b in reversed(range(self.blocks)):
            dpre = dh  # times GELU' already: by the pass that wrote it
            h = c[f"h{b}"]
            self._weight_grad(dpre, h, g[f"W{b}"], g[f"B{b}"], Cw, Cw, SP)
            dhn = torch.empty_like(h)
            dT1 = self._spectral_backward(dpre, p[f"R{b}"], c[f"B{b}"], S, g[f"R{b}"],
                                          rows.get("T"))
            # W^T dpre + dT1 Fx^T, times the GELU' of the block before
            pre = c[f"pre{b - 1}"] if b > 0 else None
            rows = self._rows(dhn, p[f"R{b - 1}"], Cw, S, 2 * self.m, (dpre, pre, dT1), True) if b > 0 else {}
            self._map_add(p[f"W{b}"], 1, Cw, dpre, dT1, self.Fx, 1, 2 * self.m, dhn, SP,
                          pre=pre, act=2 if b > 0 else 0, rows=rows)
            dh = dhn
        self._weight_grad(dh, c["x"], g["Lw"], g["Lb"], Cw, self.cin, SP)
        return ops.mse_end(y.numel()) if want_loss else None

    @on_ctx_stream
    def adam_step(self, lr=1e-3, b1=0.9, b2=0.999, eps=1e-8):
        self.step += 1
        self.ops.adam_many([(self.param[k], self.grad[k], self.adam_m[k], self.adam_v[k]) for k in self.param], lr, b1,
                           b2, eps, self.step)

    @on_ctx_stream
    def params_numpy(self):
        out = {}
        for k, v in self.param.items():
            a = v.cpu().numpy().astype(np.float64)
            if k.startswith("R"):
                a = a[..., 0] + 1j * a[..., 1]
            out[k] = a
        return out

    @on_ctx_stream
    def grads_numpy(self):
        out = {}
        for k, v in self.grad.items():
            a = v.cpu().numpy().astype(np.float64)
            if k.startswith("R"):
                a = a[..., 0] + 1j * a[..., 1]
            out[k] = a
        return out
