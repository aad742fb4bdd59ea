"""Autograd functions over the training kernels (csrc/kernels/train.hip, attention_backward.hip).

Each takes the place of a chain of single torch operations in :mod:`.functional` (forward and backward): activations bf16,
statistics, sums and the gradients of weights fp32, weights either fp32 masters or bf16. Activations are bit for bit those of
the chain. So are, all weights trained, their gradients; ``attention``, ``lora_linear`` and the ``once`` forms, for adapters,
form them in the kernels' own order. Callers ask ``usable`` first; the torch operations stay for the CPU, other types and
sizes, and under transforms that pass functions of this kind by (tracing, functorch, forward-mode). Like the flash attention
that they stand beside they have a first derivative only.
"""
from __future__ import annotations

import math
from typing import Optional, Tuple

import torch
from torch.autograd import Function
from torch.autograd.function import once_differentiable

from .. import ops

BF16 = torch.bfloat16


def usable(x: torch.Tensor, *weights: Optional[torch.Tensor]) -> bool:
    """Whether these functions take bf16 rows x (last dimension 8 to 8,192, a multiple of 8) with fp32 or bf16 weights, which
    the kernels read 16 bytes at a time (rows at other addresses are copied, see _rows)."""
    H = x.shape[-1] if x.dim() else 0
    return (_takes(x) and H % 8 == 0 and 8 <= H <= 8192
            and all(w is None or (w.is_cuda and w.is_contiguous() and w.dtype in (torch.float32, BF16) and _plain(w)
                                  and w.data_ptr() % 16 == 0) for w in weights))


def _plain(t: torch.Tensor) -> bool:
    return type(t) in (torch.Tensor, torch.nn.Parameter)


def _takes(x: torch.Tensor) -> bool:
    """bf16 rows on the GPU, nothing active that these functions would pass by, and no autocast to another type: the torch
    operations between them would change the rows' type."""
    return (x.is_cuda and x.dtype is BF16 and x.numel() > 0 and _plain(x) and not torch.jit.is_tracing() and not torch.compiler.is_compiling()
            and torch._C._functorch.peek_interpreter_stack() is None and torch.autograd.forward_ad._current_level < 0
            and not torch._C._len_torch_dispatch_stack()   # make_fx and other modes that watch the operations
            and (not torch.is_autocast_enabled("cuda") or torch.get_autocast_dtype("cuda") is BF16))


def _rows(t: torch.Tensor) -> torch.Tensor:
    """Contiguous, and at an address that the 16-byte loads take."""
    t = t.contiguous()
    return t if t.data_ptr() % 16 == 0 else t.clone()


class _Linear(Function):
    @staticmethod
    def forward(ctx, x, w, b):
        x2, wb = x.reshape(-1, x.shape[-1]), w.to(BF16)
        ctx.save_for_backward(x2, wb)
        ctx.how = (x.shape, w.dtype, b.dtype)
        return torch.addmm(b.to(BF16), x2, wb.t()).view(*x.shape[:-1], w.shape[0])

    @staticmethod
    @once_differentiable
    def backward(ctx, dy):
        x2, wb = ctx.saved_tensors
        shape, wd, bd = ctx.how
        dy2 = _rows(dy.reshape(-1, dy.shape[-1]))
        dx = (dy2 @ wb).view(shape) if ctx.needs_input_grad[0] else None
        dw = (dy2.t() @ x2).to(wd) if ctx.needs_input_grad[1] else None
        db = ops.kernels().col_sums(dy2).to(BF16).to(bd) if ctx.needs_input_grad[2] else None   # a bf16 bias's gradient
        return dx, dw, db


def linear(x: torch.Tensor, w: torch.Tensor, b: torch.Tensor) -> torch.Tensor:
    """x w^T + b in bf16, w's and b's gradients in their own type (w.shape[0] % 8 == 0)."""
    return _Linear.apply(x, w, b)


class _AddRmsNorm(Function):
    @staticmethod
    def forward(ctx, x, o, w, eps, once):
        ctx.set_materialize_grads(False)
        C = ops.kernels()
        xn, sq = C.rms_sq(_rows(x), None if o is None else _rows(o))
        y, rstd = C.rms_apply(xn, sq.mean(-1), w, eps)
        ctx.save_for_backward(xn, rstd, w)
        ctx.once = once
        return (xn, y) if o is not None else y

    @staticmethod
    @once_differentiable
    def backward(ctx, *grads):
        xn, rstd, w = ctx.saved_tensors
        C, both, dy, want = ops.kernels(), len(grads) == 2, grads[-1], ctx.needs_input_grad[2]
        dxn = grads[0] if both else None
        if dy is None:
            return dxn, dxn, None, None, None
        dy, dxn = _rows(dy), None if dxn is None else _rows(dxn)
        if ctx.once:
            dx, dw = C.rms_bwd(xn, rstd, w, dy, dxn, want)
        else:
            prod, dw = C.rms_prod(dy, xn, w, rstd, want)
            dx = C.rms_dx(dy, xn, w, rstd, prod.sum(-1).reshape(-1), dxn)
        return dx, dx if both else None, dw.to(w.dtype).view_as(w) if want else None, None, None


def rms_norm(x: torch.Tensor, w: torch.Tensor, eps: float, once: bool = False) -> torch.Tensor:
    return _AddRmsNorm.apply(x, None, w, eps, once)


def add_rms_norm(x: torch.Tensor, o: torch.Tensor, w: torch.Tensor, eps: float, once: bool = False) -> Tuple[torch.Tensor, torch.Tensor]:
    """(x + o, its RMS norm times w); once: the gradient in one pass."""
    return _AddRmsNorm.apply(x, o, w, eps, once)


class _ResidualLayerNorm(Function):
    @staticmethod
    def forward(ctx, x, o, g, b, eps):
        s, gf, bf = ops.kernels().add_f32(_rows(x), _rows(o)), g.float(), b.float()
        y, mean, rstd = torch.native_layer_norm(s, s.shape[-1:], gf, bf, eps)
        ctx.save_for_backward(s, mean, rstd, gf, bf)
        ctx.kinds = (g.dtype, b.dtype)
        return y.to(BF16)

    @staticmethod
    @once_differentiable
    def backward(ctx, dy):
        s, mean, rstd, gf, bf = ctx.saved_tensors
        dy = _rows(dy)
        ds = torch.ops.aten.native_layer_norm_backward(dy.float(), s, s.shape[-1:], mean, rstd, gf, bf, [True, False, False])[0].to(BF16)
        dg = db = None
        if ctx.needs_input_grad[2] or ctx.needs_input_grad[3]:
            dg, db = ops.kernels().ln_sums(s, mean, rstd, dy).unbind(0)
            dg, db = dg.to(ctx.kinds[0]), db.to(ctx.kinds[1])
        return ds, ds, dg, db, None


def residual_layer_norm(x, o, g, b, eps: float) -> torch.Tensor:
    """LN(x + o) g + b, the sum in fp32."""
    return _ResidualLayerNorm.apply(x, o, g, b, eps)


class _Gelu(Function):
    @staticmethod
    def forward(ctx, z):
        zr = _rows(z)
        ctx.save_for_backward(zr)
        return ops.kernels().gelu_rows(zr, None)

    @staticmethod
    @once_differentiable
    def backward(ctx, dh):
        return ops.kernels().gelu_rows(ctx.saved_tensors[0], _rows(dh))


def gelu(z: torch.Tensor) -> torch.Tensor:
    """GELU, erf form, computed in fp32."""
    return _Gelu.apply(z)


class _SwiGlu(Function):
    @staticmethod
    def forward(ctx, gu):
        g = _rows(gu)
        ctx.save_for_backward(g)
        return ops.kernels().swiglu_rows(g, None)

    @staticmethod
    @once_differentiable
    def backward(ctx, dh):
        return ops.kernels().swiglu_rows(ctx.saved_tensors[0], _rows(dh))


def swiglu(gu: torch.Tensor) -> torch.Tensor:
    """silu(gate) * up of [gate | up] rows, silu(gate) rounded to bf16."""
    return _SwiGlu.apply(gu)


def swiglu_usable(gu: torch.Tensor) -> bool:
    return _takes(gu) and gu.shape[-1] % 16 == 0


class _Rope(Function):
    @staticmethod
    def forward(ctx, qkv, cs, nr, nh, D):
        ctx.save_for_backward(cs)
        ctx.how = (nr, nh, D)
        return ops.kernels().rope_rows(_rows(qkv.reshape(-1, nh * D)), cs, nr, nh, D, False, False).view(qkv.shape)

    @staticmethod
    @once_differentiable
    def backward(ctx, d):
        return ops.kernels().rope_rows(_rows(d.reshape(-1, d.shape[-1])), ctx.saved_tensors[0], *ctx.how, True, False).view(d.shape), None, None, None, None


def rope(qkv: torch.Tensor, cs: torch.Tensor, nr: int, nh: int, D: int) -> torch.Tensor:
    """Rows of nh heads, the first nr rotated (halves) by the [cos | sin] rows cs [P, D], row t by t % P."""
    return _Rope.apply(qkv, cs, nr, nh, D)


def rope_usable(x: torch.Tensor, D: int) -> bool:
    return _takes(x) and D % 16 == 0


class _Attention(Function):
    @staticmethod
    def forward(ctx, qkv, cs, cu, B, hq, hkv, D, scale):
        r = ops.kernels().rope_rows(_rows(qkv.reshape(-1, (hq + 2 * hkv) * D)), cs, hq + hkv, hq + 2 * hkv, D, False, False)
        q, k, v = _heads(r.view(B, -1, r.shape[1]), hq, hkv, D)
        out, lse = torch.ops.aten._scaled_dot_product_flash_attention(q, k, v, 0.0, True, scale=scale)[:2]
        out = out.transpose(1, 2).reshape(-1, hq * D)
        ctx.save_for_backward(r, out, lse, cs, cu)
        ctx.how = (qkv.shape, hq, hkv, D, scale)
        return out.view(*qkv.shape[:-1], hq * D)

    @staticmethod
    @once_differentiable
    def backward(ctx, dout):
        r, out, lse, cs, cu = ctx.saved_tensors
        shape, hq, hkv, D, scale = ctx.how
        C = ops.kernels()
        d = torch.empty_like(r)
        w = [hq * D, hkv * D, hkv * D]
        l2 = (lse.transpose(0, 1) * math.log2(math.e)).reshape(hq, -1).contiguous()
        C.train_attention_backward(*d.split(w, 1), _rows(dout.reshape(-1, hq * D)), *r.split(w, 1), out, l2, cu, hq, hkv, D, lse.shape[2],
                                   scale)
        C.rope_rows(d, cs, hq + hkv, hq + 2 * hkv, D, True, True)
        return (d.view(shape),) + (None,) * 7


def _heads(qkv, hq, hkv, D):
    return (t.unflatten(-1, (-1, D)).transpose(1, 2) for t in qkv.split([hq * D, hkv * D, hkv * D], -1))


def attention(qkv: torch.Tensor, cs: torch.Tensor, cu: torch.Tensor, hq: int, hkv: int, D: int, scale: float) -> torch.Tensor:
    """Causal attention of qkv [B, S, (hq + 2 hkv) D], q and k rotated as ``rope`` does, whose gradients come from the framework's
    kernel; cu: the sequences' starts [B + 1], int32."""
    return _Attention.apply(qkv, cs, cu, qkv.shape[0], hq, hkv, D, float(scale))


def attention_usable(qkv: torch.Tensor, D: int, hq: int, hkv: int, scale: float) -> bool:
    """Whether ``attention`` takes qkv, and torch would take its flash attention for it (1), whose output that gives."""
    if not (rope_usable(qkv, D) and D in (32, 64, 128) and hkv >= 1 and hq % hkv == 0 and scale > 0):
        return False
    return torch._fused_sdp_choice(*_heads(qkv.detach(), hq, hkv, D), None, 0.0, True, scale=scale, enable_gqa=hq != hkv) == 1


class _CrossEntropySum(Function):
    @staticmethod
    def forward(ctx, logits, y, once):
        lg = _rows(logits)
        ctx.once = once
        if once:
            loss, lse = ops.kernels().ce_fwd(lg, y)
            ctx.save_for_backward(lg, y, lse)
            return loss.sum()
        lp = torch.log_softmax(lg.float(), -1)
        ctx.save_for_backward(lp, y, None)
        return torch.nn.functional.nll_loss(lp, y, reduction="sum")

    @staticmethod
    @once_differentiable
    def backward(ctx, g):
        t, y, lse = ctx.saved_tensors
        return ops.kernels().ce_bwd(t, y, lse, g.float().reshape(1).contiguous()), None, None


def cross_entropy_sum(logits: torch.Tensor, y: torch.Tensor, once: bool = False) -> torch.Tensor:
    """Sum over the rows of the cross entropy of bf16 logits [n, V] (V % 8 == 0) with labels y in [0, V); fp32. once: one pass
    over the logits, kept in bf16, for the probabilities' fp32 logarithms of the other form."""
    return _CrossEntropySum.apply(logits, y, once)


def cross_entropy_usable(logits: torch.Tensor) -> bool:
    return _takes(logits) and logits.shape[-1] % 8 == 0


class _LoraLinear(Function):
    @staticmethod
    def forward(ctx, x, w, a, b, scale):
        x2 = x.reshape(-1, x.shape[-1])
        ab, bb = a.to(BF16), b.to(BF16)
        h = x2 @ ab.t()
        y = x2 @ w.t()
        ops.kernels().add_scaled(y, h @ bb.t(), scale)
        ctx.save_for_backward(x2, w, ab, bb, h)
        ctx.how = (x.shape, scale, a.dtype, b.dtype)
        return y.view(*x.shape[:-1], w.shape[0])

    @staticmethod
    @once_differentiable
    def backward(ctx, dy):
        x2, w, ab, bb, h = ctx.saved_tensors
        shape, scale, ad, bd = ctx.how
        dy2 = dy.reshape(-1, dy.shape[-1])
        dh = (dy2 @ bb).mul_(scale)
        dx = torch.addmm(dy2 @ w, dh, ab).view(shape) if ctx.needs_input_grad[0] else None
        da = (dh.t() @ x2).to(ad) if ctx.needs_input_grad[2] else None
        db = (dy2.t() @ h).to(bd).mul_(scale) if ctx.needs_input_grad[3] else None
        return dx, None, da, db, None


def lora_linear(x: torch.Tensor, w: torch.Tensor, a: torch.Tensor, b: torch.Tensor, scale: float) -> torch.Tensor:
    """x w^T + scale (x a^T) b^T with a frozen bf16 w (w.shape[0] % 8 == 0); the adapter's part of x's gradient joins in the
    accumulator of its second product."""
    return _LoraLinear.apply(x, w, a, b, scale)
