"""The optimiser's behaviour around its step, on the CPU."""
import torch

from nv_genai_amd.training.optim import AdamW


def test_step_hooks_run_once_where_torchs_step_does_the_work():
    # torch wraps the step of every optimiser class of which there is an object: of this one and of its base
    torch.optim.AdamW([torch.nn.Parameter(torch.zeros(2))])
    p = torch.nn.Parameter(torch.ones(3))
    opt, ran = AdamW([p], lr=0.1), []
    opt.register_step_pre_hook(lambda *a: ran.append("pre"))
    opt.register_step_post_hook(lambda *a: ran.append("post"))
    p.grad = torch.ones(3)
    assert not opt._covers()
    opt.step(max_norm=1.0)
    assert ran == ["pre", "post"] and float(opt.state[p]["step"]) == 1.0 and (p < 1).all()


def test_a_training_step_on_the_cpu_keeps_every_bit():
    """Clipping adds the gradients' norms up in the order of the named tensors, not of the optimiser's groups."""
    from nv_genai_amd.training.sft import TrainConfig, Trainer

    g = torch.Generator().manual_seed(0)
    start = {f"p{i}": torch.randn(s, generator=g) for i, s in enumerate(((5,), (7, 3), (4,), (6, 2), (9,), (3, 3)))}
    slope = {n: torch.randn(t.shape, generator=g) for n, t in start.items()}
    a, b = ({n: t.clone().requires_grad_() for n, t in start.items()} for _ in range(2))
    cfg = TrainConfig(lr=1e-2, warmup_steps=0, max_steps=10, global_batch=1, log_every=0)

    def loss(ps):
        return sum((p * slope[n]).sum() for n, p in ps.items())

    tr = Trainer(a, lambda _: loss(a), [None], cfg)
    opt = torch.optim.AdamW([{"params": [p for p in b.values() if p.ndim >= 2], "weight_decay": cfg.weight_decay},
                             {"params": [p for p in b.values() if p.ndim < 2], "weight_decay": 0.0}], lr=cfg.lr, betas=cfg.betas)
    for _ in range(3):
        tr.train_step()
        for group in opt.param_groups:
            group["lr"] = tr.opt.param_groups[0]["lr"]
        opt.zero_grad()
        loss(b).backward()
        torch.nn.utils.clip_grad_norm_(list(b.values()), cfg.grad_clip)
        opt.step()
        assert all(torch.equal(a[n], b[n]) and torch.equal(a[n].grad, b[n].grad) for n in a)
