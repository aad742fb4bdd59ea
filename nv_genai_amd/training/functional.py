"""Differentiable forwards for training.

The serving forwards (models/llama.py, models/encoder.py) run packed tokens through the
hand-written gfx950 kernels, which have no backward. Training runs the same weights through
autograd on padded ``[B, S]`` batches:

* matmuls in bf16 (``torch.autocast``) on MFMA via hipBLASLt, fp32 accumulation;
* attention through ``F.scaled_dot_product_attention`` (the flash/memory-efficient backends
  of PyTorch-ROCm), causal for the LLM, key-padding-masked for the encoder; with adapters
  the framework's own kernel gives the flash attention's gradients on the GPU;
* on the GPU norms with their residual, activations, rotation and cross entropy through the functions of
  :mod:`.fused`, elsewhere and for what those do not take through torch operations. All weights trained, a
  step's loss and its gradients of matrices and embeddings are the torch operations' to the bit, but those of an
  encoder's projections over 5,000 rows and more (``ops.weight_grad_covers``): these, the gradients of
  norms' weights and biases, the clipping norm and AdamW's update are fp32 sums in another order, so that weights
  differ by their last bits from the first step on. With adapters the activations keep their bits, and the
  gradients take the forms that are a single pass;
* RMSNorm / LayerNorm / softmax statistics in fp32.

Parameters are taken from the serving model objects by reference (no copy), so a LoRA
adapter trained here merges straight back into a ``LlamaModel`` that the engine serves; full
fine-tuning keeps an fp32 master copy (``trainable_params``).

Reference behaviour: NeMo Megatron GPT SFT/LoRA (models/Gemma/lora.ipynb, sft.ipynb;
``peft_scheme=lora`` on ``attention_qkv``) and Megatron-SBERT fine-tuning
(experimental/synthetic-data-retriever-customization/retriever_customization.ipynb#cell 29).
"""
from __future__ import annotations

from typing import Callable, Dict, List, Optional, Tuple

import torch
import torch.nn.functional as F
from torch.utils.checkpoint import checkpoint as _ckpt

from . import fused

LinearFn = Callable[[torch.Tensor, int, str], torch.Tensor]


def rms_norm(x: torch.Tensor, w: torch.Tensor, eps: float) -> torch.Tensor:
    xf = x.float()
    y = xf * torch.rsqrt(xf.pow(2).mean(-1, keepdim=True) + eps)
    return (y * w.float()).to(x.dtype)


def apply_rope(x: torch.Tensor, cos: torch.Tensor, sin: torch.Tensor) -> torch.Tensor:
    """Rotate-half RoPE. x [B, S, h, D]; cos/sin [B or 1, S, 1, D/2] fp32."""
    h = x.shape[-1] // 2
    x1, x2 = x[..., :h].float(), x[..., h:].float()
    return torch.cat([x1 * cos - x2 * sin, x2 * cos + x1 * sin], dim=-1).to(x.dtype)


def _window_mask(S: int, W: int, device) -> torch.Tensor:
    """[S, S] bool: key j visible to query i iff i - W < j <= i."""
    i = torch.arange(S, device=device)
    d = i[:, None] - i[None, :]
    return (d >= 0) & (d < W)


def llama_hidden(model, ids: torch.Tensor, linear: Optional[LinearFn] = None,
                 params: Optional[Dict] = None, grad_ckpt: bool = False,
                 pos: Optional[torch.Tensor] = None) -> torch.Tensor:
    """ids [B, S] → final-normed hidden [B, S, H] (causal). ``linear(x, layer, name)``
    computes a projection (base weight + adapter); ``params`` overrides the model's tensors
    (fp32 masters for full fine-tuning).

    Every decoder family of ``LlamaConfig`` (the serving model's weights, same semantics as
    models/llama.py): LayerNorm + biases and the non-gated GELU MLP (StarCoder2), GeGLU and
    the scaled embedding (Gemma: its (1 + w) norm scale is already folded into the stored
    weight), sliding-window attention (Mistral v0.1, StarCoder2) and the sparse MoE MLP
    (Mixtral: dense per-expert loop over the routed rows, differentiable through the
    router's top-k weights)."""
    cfg = model.cfg
    P = params or {}
    B, S = ids.shape
    hq, hkv, D = model.hq, model.hkv, model.D
    if pos is None:
        pos = torch.arange(S, device=ids.device).unsqueeze(0).expand(B, S)
    cs = model.cos_sin.to(ids.device)[pos]                        # [B, S, D]
    cos, sin = cs[..., : D // 2].unsqueeze(2), cs[..., D // 2:].unsqueeze(2)
    dt = torch.bfloat16
    layer_norm = cfg.norm == "layer"
    window = cfg.sliding_window if cfg.sliding_window and S > cfg.sliding_window else 0
    amask = None   # made where it is needed
    once = linear is not None

    def W(li, name):
        return P.get((li, name), model.layers[li].get(name) if li >= 0 else None)

    def lin(x, li, name, bias=None):
        y = linear(x, li, name) if linear is not None else x @ W(li, name).to(dt).t()
        b = W(li, bias) if bias else None
        return y if b is None else y + b.to(y.dtype)

    def norm(x, li, name):
        w = W(li, name) if li >= 0 else P.get(name, getattr(model, name))
        if not layer_norm:
            return rms_norm(x, w, cfg.eps)
        b = W(li, name + "_b") if li >= 0 else P.get(name + "_b", getattr(model, name + "_b"))
        return F.layer_norm(x.float(), (x.shape[-1],), w.float(), b.float(), cfg.eps).to(x.dtype)

    def act(g):
        return F.silu(g) if cfg.act == "silu" else F.gelu(g, approximate="tanh")

    def mlp(h, li):
        if cfg.is_moe:
            x2 = h.reshape(-1, h.shape[-1])
            logits = (x2 @ W(li, "router").to(dt).t()).float()
            pr = torch.softmax(logits, -1)
            wk, ids_k = torch.topk(pr, cfg.experts_per_tok, -1)
            wk = wk / wk.sum(-1, keepdim=True)
            w13, w2 = W(li, "w13"), W(li, "w2")
            Fe = w2.shape[2]
            out = torch.zeros(x2.shape, dtype=torch.float32, device=x2.device)
            for e in range(w13.shape[0]):
                tok, slot = torch.where(ids_k == model.expert0 + e)
                if tok.numel() == 0:
                    continue
                gu = x2[tok] @ w13[e].to(dt).t()
                y = (act(gu[:, :Fe]) * gu[:, Fe:]) @ w2[e].to(dt).t()
                out = out.index_add(0, tok, y.float() * wk[tok, slot].unsqueeze(1))
            return out.to(h.dtype).view_as(h)
        gu = lin(h, li, "wgu", "bgu")
        if cfg.gated_mlp:
            if cfg.act == "silu" and fused.swiglu_usable(gu):
                return lin(fused.swiglu(gu), li, "wd", "bd")
            g, u = gu.chunk(2, dim=-1)
            return lin(act(g) * u, li, "wd", "bd")
        return lin(act(gu), li, "wd", "bd")

    emb = P.get("embed", model.embed)
    x = F.embedding(ids, emb).to(dt)
    if cfg.embed_scale != 1.0:
        x = x * torch.tensor(cfg.embed_scale, dtype=dt)

    # rotation rows, and the sequences' starts for the attention whose gradients are the framework's own
    rows = None
    if pos.dim() == 2 and fused.rope_usable(x, D):   # one table for all sequences, or one a token
        rows = cs.expand(len(cs) if cs.shape[1] == S else B, S, D).reshape(-1, D).float().contiguous()
    cu = torch.arange(0, B * S + 1, S, dtype=torch.int32, device=ids.device) if once and rows is not None else None

    def attend(qkv):
        nonlocal amask
        fits = rows is not None and fused.rope_usable(qkv, D)
        if fits and once and not window and fused.attention_usable(qkv, D, hq, hkv, model.scale):
            return fused.attention(qkv, rows, cu, hq, hkv, D, model.scale)
        if fits:
            qkv = fused.rope(qkv, rows, hq + hkv, hq + 2 * hkv, D)
        q, k, v = qkv.split([hq * D, hkv * D, hkv * D], dim=-1)
        q, k, v = q.view(B, S, hq, D), k.view(B, S, hkv, D), v.view(B, S, hkv, D).transpose(1, 2)
        if not fits:
            q, k = apply_rope(q, cos, sin), apply_rope(k, cos, sin)
        q, k = q.transpose(1, 2), k.transpose(1, 2)
        if window and amask is None:
            amask = _window_mask(S, window, ids.device)
        a = F.scaled_dot_product_attention(q, k, v, attn_mask=amask, is_causal=not window, scale=model.scale, enable_gqa=hq != hkv)
        return a.transpose(1, 2).reshape(B, S, hq * D)

    def layer(x, li):
        x = x + lin(attend(lin(norm(x, li, "attn_norm"), li, "wqkv", "bqkv")), li, "wo", "bo")
        return x + mlp(norm(x, li, "mlp_norm"), li)

    def joined(x, d, li, name):
        """(x + d, its norm); d is what the last step leaves to be added."""
        w = W(li, name) if li >= 0 else P.get(name, getattr(model, name))
        if d is not None:
            if fused.usable(x, w) and fused.usable(d) and d.shape == x.shape:
                return fused.add_rms_norm(x, d, w, cfg.eps, once)
            x = x + d   # a projection of another type; the rows from here on may have it too
        return x, fused.rms_norm(x, w, cfg.eps, once) if fused.usable(x, w) else rms_norm(x, w, cfg.eps)

    def layer_joined(x, d, li):
        x, h = joined(x, d, li, "attn_norm")
        x, h = joined(x, lin(attend(lin(h, li, "wqkv", "bqkv")), li, "wo", "bo"), li, "mlp_norm")
        return x, mlp(h, li)

    ckpt = grad_ckpt and torch.is_grad_enabled()
    n = len(model.layers)
    if not layer_norm and x.numel() and fused.usable(
            x, P.get("final_norm", model.final_norm), *(W(li, w) for li in range(n) for w in ("attn_norm", "mlp_norm"))):
        d = None
        for li in range(n):
            x, d = _ckpt(layer_joined, x, d, li, use_reentrant=False) if ckpt else layer_joined(x, d, li)
        return joined(x, d, -1, "final_norm")[1]
    for li in range(n):
        x = _ckpt(layer, x, li, use_reentrant=False) if ckpt else layer(x, li)
    return norm(x, -1, "final_norm")


def lm_loss(model, hidden: torch.Tensor, labels: torch.Tensor, params: Optional[Dict] = None,
            chunk: int = 2048) -> torch.Tensor:
    """Mean next-token cross entropy over positions with ``labels >= 0`` (labels are already
    shifted: labels[b, t] is the target for hidden[b, t]). The vocab projection is chunked
    over tokens so [tokens, 128256] fp32 logits never materialise at once."""
    P = params or {}
    head = P.get("lm_head", P.get("embed") if model.lm_head is model.embed else None)
    head = (head if head is not None else model.lm_head).to(torch.bfloat16)
    h = hidden.reshape(-1, hidden.shape[-1])
    y = labels.reshape(-1)
    keep = (y >= 0).nonzero().squeeze(1)
    h, y = h.index_select(0, keep), y.index_select(0, keep)
    total = h.new_zeros((), dtype=torch.float32)
    for s in range(0, h.shape[0], chunk):
        hs = h[s:s + chunk]
        lg = fused.frozen_linear(hs, head) if fused.frozen_linear_usable(hs, head) else hs @ head.t()
        if fused.cross_entropy_usable(lg):
            if s == 0 and params is None and int(y.max()) >= lg.shape[1]:   # the one-pass form would give NaN
                raise IndexError(f"label {int(y.max())} outside the vocabulary of {lg.shape[1]}")
            total = total + fused.cross_entropy_sum(lg, y[s:s + chunk], params is None)
        else:
            total = total + F.cross_entropy(lg.float(), y[s:s + chunk], reduction="sum")
    return total / max(1, y.numel())


def encoder_embed(model, ids: torch.Tensor, mask: torch.Tensor, params: Optional[Dict] = None,
                  grad_ckpt: bool = False) -> torch.Tensor:
    """ids/mask [B, S] (right padded) → pooled [B, H] fp32 (L2-normalised when configured)."""
    steps = _encoder_steps(model, ids, mask, params, grad_ckpt)
    while True:
        out = next(steps)
        if out is not None:
            return out


def encoder_embed_pair(model, many, few, grad_ckpt: bool = False) -> Tuple[torch.Tensor, torch.Tensor]:
    """``encoder_embed`` of two inputs (ids, mask, params), a layer of the one and a layer of the other in turn; autograd takes a
    backward's layers in turn as well. A step on few tokens (questions) is bound by the host, which launches some 45 kernels a layer
    for each direction: in turn with a step on many (passages) it launches them while the GPU is at those. BERT-large, 4 questions of
    46 tokens and 20 passages of 512: a step 60.0 ms one after the other, 55.3 in turn, of which the GPU is busy 54. On two
    streams a run's losses were now and then not the same to the bit, so they share one."""
    one, two = _encoder_steps(model, *many, grad_ckpt), _encoder_steps(model, *few, grad_ckpt)
    a = b = None
    while a is None:
        a, b = next(one), next(two)
    return a, b


def _encoder_steps(model, ids, mask, params=None, grad_ckpt=False):
    """The steps of ``encoder_embed``: None for each but the last, its result."""
    cfg = model.cfg
    P = params or {}
    B, S = ids.shape
    H, nh, hd = cfg.hidden, cfg.heads, cfg.head_dim
    dt = torch.bfloat16

    def g(li, name):
        return P.get((li, name), model.layers[li][name])

    pos = torch.arange(S, device=ids.device)
    e = (F.embedding(ids, P.get("word", model.word)).float() + P.get("pos", model.pos)[pos].float()
         + P.get("type", model.type)[0].float())
    x = F.layer_norm(e, (H,), P.get("emb_ln_g", model.emb_ln[0]).float(), P.get("emb_ln_b", model.emb_ln[1]).float(),
                     cfg.eps).to(dt)
    amask = mask.bool()[:, None, None, :]

    def lin(x, li, w, b):
        w, b = g(li, w), g(li, b)
        if fused.usable(x, w, b) and w.shape[0] % 8 == 0:
            return fused.linear(x, w, b)
        return F.linear(x, w.to(dt), b.to(dt))

    def add_norm(x, o, li, n):
        w, b = g(li, n + "_g"), g(li, n + "_b")
        if fused.usable(x, w, b):
            return fused.residual_layer_norm(x, o, w, b, cfg.eps)
        return F.layer_norm((x.float() + o.float()), (H,), w.float(), b.float(), cfg.eps).to(dt)

    def layer(x, li):
        q, k, v = (t.view(B, S, nh, hd).transpose(1, 2) for t in lin(x, li, "wqkv", "bqkv").split(H, dim=-1))
        a = F.scaled_dot_product_attention(q, k, v, attn_mask=amask, scale=model.scale)
        x = add_norm(x, lin(a.transpose(1, 2).reshape(B, S, H), li, "wo", "bo"), li, "ln1")
        z = lin(x, li, "wi", "bi")
        h = fused.gelu(z) if fused.usable(z) else F.gelu(z.float()).to(dt)
        return add_norm(x, lin(h, li, "wo2", "bo2"), li, "ln2")

    for li in range(len(model.layers)):
        yield None
        x = _ckpt(layer, x, li, use_reentrant=False) if grad_ckpt and torch.is_grad_enabled() else layer(x, li)
    xf = x.float()
    if cfg.pooling == "cls":
        pooled = xf[:, 0]
    else:
        m = mask.float().unsqueeze(-1)
        pooled = (xf * m).sum(1) / m.sum(1).clamp_min(1.0)
    if cfg.normalize:
        pooled = pooled / pooled.norm(dim=-1, keepdim=True).clamp_min(1e-12)
    yield pooled


def trainable_params(model, kind: str = "llama") -> Dict:
    """fp32 master copies of every weight (full fine-tuning), keyed like ``params``."""
    out: Dict = {}
    if kind == "llama":
        out["embed"], out["final_norm"] = model.embed, model.final_norm
        if getattr(model, "final_norm_b", None) is not None:
            out["final_norm_b"] = model.final_norm_b
        if model.lm_head is not model.embed:   # tied embeddings train through "embed"
            out["lm_head"] = model.lm_head
        for li, L in enumerate(model.layers):
            for n, t in L.items():
                out[(li, n)] = t
    else:
        out.update(word=model.word, pos=model.pos, type=model.type, emb_ln_g=model.emb_ln[0], emb_ln_b=model.emb_ln[1])
        for li, L in enumerate(model.layers):
            for n, t in L.items():
                out[(li, n)] = t
    return {k: v.detach().float().clone().requires_grad_(True) for k, v in out.items()}


# what the encoder's forward takes in bf16 and no other type
_HALF = ("wqkv", "bqkv", "wo", "bo", "wi", "bi", "wo2", "bo2")


def half_params(params: Dict) -> List[Dict]:
    """An encoder's ``params`` for each of the two passes of a step (questions and passages), with the layers' projections in
    bf16, cast once for both and a layer at a time, so that a layer's gradients are there when its backward is done. Where the
    kernel does not take them, or under a mode that watches the operations, they are ``params``, which the passes cast
    themselves. One pass alone has nothing to share: a small decoder's step took 19.0 ms with and without."""
    out = [dict(params), dict(params)]
    for li in sorted({k[0] for k in params if isinstance(k, tuple)}):
        keys = [(li, n) for n in _HALF if (li, n) in params]
        masters = [params[k] for k in keys]
        if fused.half_copies_usable(masters):
            for p, got in zip(out, fused.half_copies(masters)):
                p.update(zip(keys, got))
    return out


def write_back(model, params: Dict, kind: str = "llama") -> None:
    """Copy fp32 masters back into the serving model's bf16 tensors (in place)."""
    with torch.no_grad():
        for k, v in params.items():
            if isinstance(k, tuple):
                model.layers[k[0]][k[1]].copy_(v)
            elif kind == "llama":
                getattr(model, k).copy_(v)
            elif k.startswith("emb_ln"):
                model.emb_ln[0 if k.endswith("g") else 1].copy_(v)
            else:
                getattr(model, k).copy_(v)
