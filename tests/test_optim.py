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
