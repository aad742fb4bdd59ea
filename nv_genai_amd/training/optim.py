"""AdamW whose step, with the clipping of the gradients' norm, is a few launches over all tensors (``grad_norm`` and ``adamw``
of csrc/kernels/adamw.hip) instead of a dozen passes of foreach operations. State, groups and checkpoints are those of
``torch.optim.AdamW``; tensors that the kernels do not take go through its step."""
from __future__ import annotations

import inspect
from collections import defaultdict
from typing import Optional, Sequence

import torch

from .. import ops


def _native(t: torch.Tensor) -> bool:
    return t.is_cuda and t.dtype == torch.float32 and t.layout == torch.strided and t.is_contiguous()


class AdamW(torch.optim.AdamW):
    def _covers(self) -> bool:
        if getattr(self, "grad_scale", None) is not None or getattr(self, "found_inf", None) is not None:
            return False   # a GradScaler leaves scaling and skipping to torch's fused step
        dev = None
        for g in self.param_groups:
            if g["amsgrad"] or g["maximize"] or g["capturable"] or g["differentiable"] or isinstance(g["lr"], torch.Tensor):
                return False
            for p in g["params"]:
                if p.grad is None:
                    continue
                dev = dev or p.device
                if p.device != dev or not _native(p) or not _native(p.grad) or type(p.grad) is not torch.Tensor:
                    return False
                st = self.state.get(p)
                if st and not all(n in st and _native(st[n]) for n in ("exp_avg", "exp_avg_sq")):
                    return False
        return dev is not None and not (dev.type == "cuda" and torch.cuda.is_current_stream_capturing())

    @torch.no_grad()
    def step(self, closure=None, max_norm: Optional[float] = None, among: Optional[Sequence[torch.Tensor]] = None):
        """One step; ``max_norm``: first scale all gradients (in place) to that norm, as ``clip_grad_norm_`` does, which where it
        does the work itself adds up the norms in the order of ``among`` (the groups' order otherwise)."""
        loss = None
        if closure is not None:
            with torch.enable_grad():
                loss = closure()
        if not self._covers():
            if max_norm:
                torch.nn.utils.clip_grad_norm_(among or [p for g in self.param_groups for p in g["params"]], max_norm)
            for g in self.param_groups:   # torch's fused step keeps the count beside the weights
                for p in g["params"]:
                    st = self.state.get(p)
                    if st and (g["fused"] or g["capturable"]) and st["step"].device != p.device:
                        st["step"] = st["step"].to(p.device)
            # without the hooks that torch wraps around the base's step: those around this one run already
            inspect.unwrap(torch.optim.AdamW.step, stop=lambda f: not getattr(f, "hooked", False))(self)
            return loss
        C = ops.kernels()
        clip = None
        if max_norm:
            clip = C.grad_norm([p.grad for g in self.param_groups for p in g["params"] if p.grad is not None], float(max_norm))
        for g in self.param_groups:
            ps = [p for p in g["params"] if p.grad is not None]
            for p in ps:
                st = self.state[p]
                if not st:
                    st["step"] = torch.tensor(0.0, dtype=torch.float32)
                    st["exp_avg"], st["exp_avg_sq"] = torch.zeros_like(p), torch.zeros_like(p)
                elif st["step"].is_cuda:   # from a checkpoint of an optimiser that kept it there
                    st["step"] = st["step"].cpu()
            if not ps:
                continue
            torch._foreach_add_([self.state[p]["step"] for p in ps], 1)
            at = defaultdict(list)
            for p in ps:
                at[int(self.state[p]["step"].item())].append(p)
            for step, q in at.items():
                gr, m, v = [p.grad for p in q], [self.state[p]["exp_avg"] for p in q], [self.state[p]["exp_avg_sq"] for p in q]
                C.adamw(q, gr, m, v, clip, float(g["lr"]), float(g["weight_decay"]), float(g["betas"][0]), float(g["betas"][1]),
                        float(g["eps"]), step)
                # the kernel writes through addresses: a graph that saved one of these must see that it changed
                torch.autograd.graph.increment_version(q + m + v + (gr if max_norm else []))
        return loss
