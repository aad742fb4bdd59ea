"""Autograd functions over the training kernels (csrc/kernels/train.hip, attention_backward.hip).

Each takes the place of a chain of single torch operations in :mod:`.functional` (forward and backward): activations bf16,
statistics, sums and the gradients of weights fp32, weights either fp32 masters or bf16. Activations are bit for bit those of
the chain. So are, all weights trained, their gradients and those of matrices; the gradients of norms' weights and of biases
are fp32 sums over the rows in the kernels' own order, and so are those of ``linear``'s matrices over some thousand rows. ``attention``, ``lora_linear`` and the ``once`` forms, for adapters, form
the activations' gradients in that too. Callers ask ``usable`` first; the torch operations stay for the CPU, other types and
sizes, and under transforms that pass functions of this kind by (tracing, functorch, forward-mode). Where a graph of the
backward is asked for (create_graph) the gradients come from torch operations; ``attention``, like the flash attention that it
stands for, has a first derivative only.
"""
from __future__ import annotations

from typing import Optional, Sequence, Tuple

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
    return x.is_cuda and x.dtype is BF16 and x.numel() > 0 and _plain(x) and _undisturbed()


def _undisturbed() -> bool:
    return (not torch.jit.is_tracing() and not torch.compiler.is_compiling()
            and torch._C._functorch.peek_interpreter_stack() is None and torch.autograd.forward_ad._current_level < 0
            and not torch._C._len_torch_dispatch_stack()   # make_fx and other modes that watch the operations
            and (not torch.is_autocast_enabled("cuda") or torch.get_autocast_dtype("cuda") is BF16))


def _rows(t: torch.Tensor) -> torch.Tensor:
    """Contiguous, and at an address that the 16-byte loads take."""
    t = t.contiguous()
    return t if t.data_ptr() % 16 == 0 else t.clone()


def _again(chain, inputs, dy):
    """The inputs' gradients (None where they need none) through torch operations, from tensors that carry the graph of the
    forward: to be differentiated in turn."""
    ins = [t.view_as(t) for t in inputs]
    got = iter(torch.autograd.grad(chain(*ins), [t for t in ins if t.requires_grad], dy, create_graph=True))
    return [next(got) if t.requires_grad else None for t in ins]


class _Linear(Function):
    @staticmethod
    def forward(ctx, x, w, b):
        ctx.save_for_backward(x, w, b)
        return torch.addmm(b, x.reshape(-1, x.shape[-1]), w.t()).view(*x.shape[:-1], w.shape[0])

    @staticmethod
    def backward(ctx, dy):
        x, w, b = ctx.saved_tensors
        if torch.is_grad_enabled():
            return tuple(_again(torch.nn.functional.linear, (x, w, b), dy))
        dy2 = _rows(dy.reshape(-1, dy.shape[-1]))
        dx = (dy2 @ w).view(x.shape) if ctx.needs_input_grad[0] else None
        dw = _weight_grad(dy2, x.reshape(-1, x.shape[-1])) if ctx.needs_input_grad[1] else None
        db = ops.kernels().col_sums(dy2) if ctx.needs_input_grad[2] else None
        return dx, dw, db


def _weight_grad(dy2: torch.Tensor, x2: torch.Tensor) -> torch.Tensor:
    if dy2.dtype is BF16 and x2.dtype is BF16 and ops.weight_grad_covers(dy2.shape[0], dy2.shape[1], x2.shape[1]):
        return ops.kernels().gemm_kn(_rows(dy2), _rows(x2), True)
    return dy2.t() @ x2


def linear(x: torch.Tensor, w: torch.Tensor, b: torch.Tensor) -> torch.Tensor:
    """x w^T + b in bf16, w's and b's gradients in their own type (w.shape[0] % 8 == 0)."""
    return _Linear.apply(x, w.to(BF16), b.to(BF16))


class _HalfCopies(Function):
    @staticmethod
    def forward(ctx, *masters):
        ctx.set_materialize_grads(False)
        out = ops.kernels().half_copies(masters)
        return (*out, *(t.detach() for t in out))

    @staticmethod
    def backward(ctx, *grads):
        n = len(ctx.needs_input_grad)
        two = [[g for g in grads[i::n] if g is not None] if ctx.needs_input_grad[i] else [] for i in range(n)]
        if torch.is_grad_enabled():
            return tuple(sum(g.float() for g in gs) if gs else None for gs in two)
        live = [gs for gs in two if gs]
        got = iter(ops.kernels().half_grads([gs[0] for gs in live], [gs[1] if len(gs) > 1 else None for gs in live]) if live else ())
        return tuple(next(got) if gs else None for gs in two)


def half_copies(masters: Sequence[torch.Tensor]) -> Tuple[Tuple[torch.Tensor, ...], Tuple[torch.Tensor, ...]]:
    """bf16 copies of fp32 masters for two forward passes, a tuple for each: the same values, whose gradients (bf16 each) are
    added up in fp32."""
    out = _HalfCopies.apply(*masters)
    return out[:len(masters)], out[len(masters):]


def half_copies_usable(masters: Sequence[torch.Tensor]) -> bool:
    return len(masters) > 0 and _undisturbed() and all(
        t.is_cuda and t.dtype is torch.float32 and t.device == masters[0].device and t.is_contiguous() and t.data_ptr() % 16 == 0
        and _plain(t) for t in masters)


class _AddRmsNorm(Function):
    @staticmethod
    def forward(ctx, x, o, w, eps, once):
        ctx.set_materialize_grads(False)
        C = ops.kernels()
        xn, sq = C.rms_sq(_rows(x), None if o is None else _rows(o))
        y, rstd = C.rms_apply(xn, sq.mean(-1), w, eps)
        ctx.save_for_backward(x if o is None else xn, rstd, w)
        ctx.how = (eps, once)
        return (xn, y) if o is not None else y

    @staticmethod
    def backward(ctx, *grads):
        xn, rstd, w = ctx.saved_tensors
        C, both, dy, want = ops.kernels(), len(grads) == 2, grads[-1], ctx.needs_input_grad[2]
        eps, once = ctx.how
        dxn = grads[0] if both else None
        if dy is None:
            return dxn, dxn, None, None, None
        if torch.is_grad_enabled():
            def chain(x, w):
                x = x.float()
                return (x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + eps) * w.float()).to(BF16)

            dx, dw = _again(chain, (xn, w), dy)
            dx = dx if dxn is None else dx + dxn
            return dx, dx if both else None, dw, None, None
        xn, dy, dxn = _rows(xn), _rows(dy), None if dxn is None else _rows(dxn)
        if once:
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
        ctx.set_materialize_grads(False)
        s = ops.kernels().add_f32(_rows(x), _rows(o))
        y, mean, rstd = torch.native_layer_norm(s, s.shape[-1:], g, b, eps)
        ctx.save_for_backward(s, mean, rstd, g, b)
        ctx.eps = eps
        return y.to(BF16), s   # an output carries the graph to x and o, for a derivative of the backward

    @staticmethod
    def backward(ctx, dy, more):
        s, mean, rstd, g, b = ctx.saved_tensors
        dg = db = None
        if dy is None:
            ds = more
        elif torch.is_grad_enabled():
            ds, dg, db = _again(lambda s, g, b: torch.nn.functional.layer_norm(s, s.shape[-1:], g, b, ctx.eps).to(BF16), (s, g, b), dy)
            ds = ds if more is None else ds + more
        else:
            dy = _rows(dy)
            ds = torch.ops.aten.native_layer_norm_backward(dy.float(), s, s.shape[-1:], mean, rstd, g, b, [True, False, False])[0]
            ds = ds if more is None else ds + more
            if ctx.needs_input_grad[2] or ctx.needs_input_grad[3]:
                dg, db = ops.kernels().ln_sums(s, mean, rstd, dy).unbind(0)
        ds = None if ds is None else ds.to(BF16)
        return ds, ds, dg, db, None


def residual_layer_norm(x, o, g, b, eps: float) -> torch.Tensor:
    """LN(x + o) g + b, the sum in fp32."""
    return _ResidualLayerNorm.apply(x, o, g.float(), b.float(), eps)[0]


class _Gelu(Function):
    @staticmethod
    def forward(ctx, z):
        ctx.save_for_backward(z)
        return ops.kernels().gelu_rows(_rows(z), None)

    @staticmethod
    def backward(ctx, dh):
        if torch.is_grad_enabled():
            return _again(lambda z: torch.nn.functional.gelu(z.float()).to(BF16), ctx.saved_tensors, dh)[0]
        return ops.kernels().gelu_rows(_rows(ctx.saved_tensors[0]), _rows(dh))


def gelu(z: torch.Tensor) -> torch.Tensor:
    """GELU, erf form, computed in fp32."""
    return _Gelu.apply(z)


class _SwiGlu(Function):
    @staticmethod
    def forward(ctx, gu):
        ctx.save_for_backward(gu)
        return ops.kernels().swiglu_rows(_rows(gu), None)

    @staticmethod
    def backward(ctx, dh):
        if torch.is_grad_enabled():
            return _again(lambda t: torch.nn.functional.silu(t.chunk(2, -1)[0]) * t.chunk(2, -1)[1], ctx.saved_tensors, dh)[0]
        return ops.kernels().swiglu_rows(_rows(ctx.saved_tensors[0]), _rows(dh))


def swiglu(gu: torch.Tensor) -> torch.Tensor:
    """silu(gate) * up of [gate | up] rows, silu(gate) rounded to bf16."""
    return _SwiGlu.apply(gu)


def swiglu_usable(gu: torch.Tensor) -> bool:
    return _takes(gu) and gu.shape[-1] % 16 == 0


class _Rope(Function):
    @staticmethod
    def forward(ctx, qkv, cs, nr, nh, D, back):
        ctx.save_for_backward(cs)
        ctx.how = (nr, nh, D, not back)
        return ops.kernels().rope_rows(_rows(qkv.reshape(-1, nh * D)), cs, nr, nh, D, back, False).view(qkv.shape)

    @staticmethod
    def backward(ctx, d):
        return (_Rope.apply(d, ctx.saved_tensors[0], *ctx.how),) + (None,) * 5


def rope(qkv: torch.Tensor, cs: torch.Tensor, nr: int, nh: int, D: int) -> torch.Tensor:
    """Rows of nh heads, the first nr rotated (halves) by the [cos | sin] rows cs [P, D], row t by t % P."""
    return _Rope.apply(qkv, cs, nr, nh, D, False)


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
        C.train_attention_backward(*d.split(w, 1), _rows(dout.reshape(-1, hq * D)), *r.split(w, 1), out, lse.contiguous(), cu, hq, hkv, D,
                                   lse.shape[2], scale)
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
        ctx.set_materialize_grads(False)
        ctx.once = once
        if once:
            loss, lse = ops.kernels().ce_fwd(_rows(logits), y)
            ctx.save_for_backward(logits, y, lse)
            return loss.sum(), None
        lp = torch.log_softmax(_rows(logits).float(), -1)
        ctx.save_for_backward(lp, y, None)
        return torch.nn.functional.nll_loss(lp, y, reduction="sum"), lp   # an output carries the graph to the logits

    @staticmethod
    def backward(ctx, g, more):
        t, y, lse = ctx.saved_tensors
        if g is not None and more is None and not torch.is_grad_enabled():
            return ops.kernels().ce_bwd(_rows(t) if ctx.once else t, y, lse, g.float().reshape(1).contiguous()), None, None
        p, d = torch.softmax(t.float(), -1) if ctx.once else t.exp(), None
        if g is not None:
            d = g * (p - torch.nn.functional.one_hot(y, t.shape[-1]))
        if more is not None:
            more = more - p * more.sum(-1, keepdim=True)
            d = more if d is None else d + more
        return None if d is None else d.to(BF16), None, None


def cross_entropy_sum(logits: torch.Tensor, y: torch.Tensor, once: bool = False) -> torch.Tensor:
    """Sum over the rows of the cross entropy of bf16 logits [n, V] (V % 8 == 0) with labels y in [0, V); fp32. once: one pass
    over the logits, kept in bf16, for the probabilities' fp32 logarithms of the other form."""
    return _CrossEntropySum.apply(logits, y, once)[0]


def cross_entropy_usable(logits: torch.Tensor) -> bool:
    return _takes(logits) and logits.shape[-1] % 8 == 0


class _FrozenLinear(Function):
    @staticmethod
    def forward(ctx, x, w):
        ctx.save_for_backward(w)
        return x @ w.t()

    @staticmethod
    def backward(ctx, dy):
        w, = ctx.saved_tensors
        if torch.is_grad_enabled():
            return dy @ w, None
        return _input_grad(dy.reshape(-1, w.shape[0]), w).view(*dy.shape[:-1], w.shape[1]), None


def _input_grad(dy2: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    if ops.gemm_kn_covers(dy2.shape[0], w.shape[1], w.shape[0]) and w.is_contiguous() and w.data_ptr() % 16 == 0 and dy2.dtype is BF16:
        return ops.kernels().gemm_kn(_rows(dy2), w, False)
    return dy2 @ w


def frozen_linear(x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    """x w^T with a frozen bf16 w; x's gradient from the framework's own product where that is the faster one."""
    return _FrozenLinear.apply(x, w)


def frozen_linear_usable(x: torch.Tensor, w: torch.Tensor) -> bool:
    return (_takes(x) and x.requires_grad and torch.is_grad_enabled() and w.dim() == 2 and w.device == x.device and w.dtype is BF16
            and not w.requires_grad and _plain(w) and w.is_contiguous() and w.data_ptr() % 16 == 0 and x.shape[-1] == w.shape[1]
            and ops.gemm_kn_covers(x.numel() // w.shape[1], w.shape[1], w.shape[0]))


class _LoraLinear(Function):
    @staticmethod
    def forward(ctx, x, w, a, b, ab, bb, scale):
        x2 = x.reshape(-1, x.shape[-1])
        h = x2 @ ab.t()
        y = x2 @ w.t()
        ops.kernels().add_scaled(y, h @ bb.t(), scale)
        ctx.save_for_backward(x, w, ab, bb, h)
        ctx.how = (scale, a.dtype, b.dtype)
        return y.view(*x.shape[:-1], w.shape[0])

    @staticmethod
    def backward(ctx, dy):
        x, w, ab, bb, h = ctx.saved_tensors
        scale, ad, bd = ctx.how
        if torch.is_grad_enabled():   # the adapter's gradients through its bf16 copies
            dx, da, db = _again(lambda x, a, b: x @ w.t() + ((x @ a.t()) @ b.t()) * scale, (x, ab, bb), dy)
            return dx, None, None, None, da, db, None
        dy2 = dy.reshape(-1, dy.shape[-1])
        need = ctx.needs_input_grad
        if (ops.lora_grads_covers(dy2.shape[0], bb.shape[0], x.shape[-1], bb.shape[1])   # lora.hip; single operations under vmap too
                and _takes(dy) and not torch._C._functorch.is_legacy_batchedtensor(dy)):
            dy2 = _rows(dy2)
            dx = _input_grad(dy2, w) if need[0] else None
            da, db = ops.kernels().lora_grads(dy2, _rows(x.reshape(-1, x.shape[-1])), _rows(h), _rows(ab), _rows(bb), dx, scale,
                                              need[2], need[3])
            return (dx.view(x.shape) if need[0] else None, None, da.to(ad) if need[2] else None, db.to(bd) if need[3] else None,
                    None, None, None)
        dh = (dy2 @ bb).mul_(scale)
        dx = torch.addmm(_input_grad(dy2, w), dh, ab).view(x.shape) if need[0] else None
        da = (dh.t() @ x.reshape(-1, x.shape[-1])).to(ad) if need[2] else None
        db = (dy2.t() @ h).to(bd).mul_(scale) if need[3] else None   # scaled in its own type
        return dx, None, da, db, None, None, None


def lora_linear(x: torch.Tensor, w: torch.Tensor, a: torch.Tensor, b: torch.Tensor, scale: float) -> torch.Tensor:
    """x w^T + scale (x a^T) b^T with a frozen bf16 w (w.shape[0] % 8 == 0); the adapter's gradients come from lora.hip, which adds
    its part of x's to that through w, and of ranks that it does not take from single operations."""
    return _LoraLinear.apply(x, w, a, b, a.to(BF16), b.to(BF16), scale)
