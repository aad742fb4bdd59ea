"""The native AdamW step on the GPU against torch's in 64 bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _rel(a, b):
    return ((a.double() - b.double()).norm() / b.double().norm().clamp_min(1e-30)).item()


@pytest.mark.parametrize("max_norm", [None, 0.5, 1e9])
def test_adamw_matches_torch(gpu, max_norm):
    from nv_genai_amd.training.optim import AdamW

    sizes = [(1,), (7, 5), (33_000,), (128, 300), (65_537,)] + [(3, 4)] * 60    # ragged ends, several chunks, two tables
    g = torch.Generator(device="cuda").manual_seed(1)
    ps = [torch.randn(s, device="cuda", generator=g) for s in sizes]
    # the last is a view at an odd address
    ps[-1] = torch.randn(13, device="cuda", generator=g)[1:]
    a, b = [p.clone().requires_grad_() for p in ps], [p.double().requires_grad_() for p in ps]
    a[-1] = torch.nn.Parameter(ps[-1])
    kw = dict(lr=1e-2, betas=(0.9, 0.98))
    oa = AdamW([{"params": a[:3], "weight_decay": 0.1}, {"params": a[3:], "weight_decay": 0.0}], **kw)
    ob = torch.optim.AdamW([{"params": b[:3], "weight_decay": 0.1}, {"params": b[3:], "weight_decay": 0.0}], **kw)
    for step in range(4):
        for i, (p, q) in enumerate(zip(a, b)):
            d = torch.randn(p.shape, device="cuda", generator=g)
            p.grad, q.grad = (None, None) if i == 4 and step == 1 else (d.clone(), d.double())
        assert oa._covers()
        oa.step(max_norm=max_norm)
        if max_norm:
            torch.nn.utils.clip_grad_norm_(b, max_norm)
        ob.step()
        for p, q in zip(a, b):
            assert _rel(p.detach(), q.detach()) < 2e-6
            if p.grad is not None:
                assert _rel(p.grad, q.grad) < 2e-6
    sa, sb = oa.state_dict(), ob.state_dict()
    assert sa["param_groups"][0].keys() == sb["param_groups"][0].keys()
    assert all(float(sa["state"][i]["step"]) == float(sb["state"][i]["step"]) for i in sb["state"])
    again = AdamW([{"params": a[:3], "weight_decay": 0.1}, {"params": a[3:], "weight_decay": 0.0}], **kw)
    again.load_state_dict(sa)
    again.step(max_norm=max_norm)


@pytest.mark.parametrize("max_norm", [None, 1.0])
def test_a_kept_graph_sees_the_step(gpu, max_norm):
    """A backward through a graph that saved the weights raises after the step, as behind torch's."""
    from nv_genai_amd.training.optim import AdamW

    p = torch.nn.Parameter(torch.randn(64, device=gpu))
    opt = AdamW([p], lr=0.1)
    loss = p.pow(3).sum()
    loss.backward(retain_graph=True)
    seen = p.grad._version
    assert opt._covers()
    opt.step(max_norm=max_norm)
    assert (p.grad._version > seen) == (max_norm is not None)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        loss.backward()


@pytest.mark.parametrize("factor", [1.0, float("inf")])
def test_grad_scaler_with_the_fused_form(gpu, factor):
    """A GradScaler hands the scale and the found infinities to a fused optimiser's step."""
    from nv_genai_amd.training.optim import AdamW

    start, got = torch.randn(64, device=gpu), []
    for cls in (AdamW, torch.optim.AdamW):
        p = torch.nn.Parameter(start.clone())
        opt, scaler = cls([p], lr=0.1, fused=True), torch.amp.GradScaler("cuda", init_scale=1024.0)
        for _ in range(2):
            opt.zero_grad()
            scaler.scale((p * torch.linspace(0.0, 1.0, 64, device=gpu)).sum() * factor).backward()
            scaler.step(opt)
            scaler.update()
        got.append((p.detach(), scaler.get_scale()))
    assert torch.equal(got[0][0], got[1][0]) and got[0][1] == got[1][1]
    assert torch.equal(got[0][0], start) == (factor > 1)
