"""Packed and paged attention: rows in and out in whole pieces (attention_varlen.hip, attention_prefill_v2.hip). Each row's result is the same bits wherever its tensors
lie, against 64 bits it is within the kernel's roundings, and nothing else is written."""
import pytest
import torch

pytestmark = pytest.mark.gpu
BF = torch.bfloat16


# ends within a wave's 32 rows, a workgroup's 128 (32 of four heads with four query heads a KV head), a key tile of 64; one tile and two
@pytest.mark.parametrize("D,hq,hkv", [(32, 3, 3), (64, 2, 1), (64, 4, 1), (128, 8, 2), (128, 2, 2)])
@pytest.mark.parametrize("lens", [[1], [31, 33, 64], [65, 127, 2], [129, 200, 63]])
@pytest.mark.parametrize("causal", [False, True])
def test_rows(gpu, D, hq, hkv, lens, causal):
    from nv_genai_amd import ops

    g = torch.Generator("cuda").manual_seed(D + hq + lens[0])
    T, w, scale = sum(lens), hq * D, D ** -0.5
    q, k, v = (torch.randn(T, h * D, device=gpu, generator=g).to(BF) for h in (hq, hkv, hkv))
    cu = torch.tensor([0, *torch.tensor(lens).cumsum(0).tolist()], dtype=torch.int32, device=gpu)
    got = ops.varlen_attention(q, k, v, cu, hq, hkv, D, max(lens), scale, causal)
    at = 0
    for n in lens:
        Q, K, V = (t[at:at + n].view(n, -1, D).transpose(0, 1).double() for t in (q, k, v))
        K, V = K.repeat_interleave(hq // hkv, 0), V.repeat_interleave(hq // hkv, 0)
        S = Q @ K.transpose(1, 2).contiguous() * scale
        P = (S.masked_fill(torch.ones(n, n, device=gpu).triu(1).bool(), float("-inf")) if causal else S).softmax(-1)
        ref = (P @ V).transpose(0, 1).reshape(n, w)
        size = (P @ V.abs()).transpose(0, 1).reshape(n, w)
        # probabilities as bf16 and the result as bf16, 2^-9 each, doubled for the fp32 steps between
        assert ((got[at:at + n].double() - ref).abs() <= 2.0 ** -8 * (size + ref.abs())).all()
        at += n

    def odd(t, by):   # the same rows elsewhere: by values off a 16-byte address, 8 more a row
        s = torch.zeros(T, t.shape[1] + 16, dtype=BF, device=gpu)[:, by:by + t.shape[1]]
        return s.copy_(t)

    for by in (0, 8, 3):
        room = torch.full((T + 1, w + 16), 7.0, dtype=BF, device=gpu)
        ops.varlen_attention(odd(q, by), odd(k, by), odd(v, by), cu, hq, hkv, D, max(lens), scale, causal, out=room[:T, by:by + w])
        assert torch.equal(room[:T, by:by + w], got)
        room[:T, by:by + w] = 7.0
        assert (room == 7.0).all()


def _pages(gpu, lens, ctxs, hq, hkv, seed):
    D, T, B = 128, sum(lens), len(lens)
    g = torch.Generator("cuda").manual_seed(seed)
    rn = lambda *s: torch.randn(*s, device=gpu, generator=g).to(BF)  # noqa: E731
    pages = [(c + 63) // 64 for c in ctxs]
    q, kc, vc = rn(T, hq * D), rn(sum(pages), hkv, 64, D), rn(sum(pages), hkv, D, 64)
    bt = torch.zeros(B, max(pages), dtype=torch.int32)
    for i, n in enumerate(pages):
        bt[i, :n] = torch.arange(n) + sum(pages[:i])
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=gpu)  # noqa: E731
    return pages, q, kc, vc, bt.to(gpu), i32([0, *torch.tensor(lens).cumsum(0).tolist()]), i32(ctxs)


# one group of waves and two by size, the old kernel among them (impl 0), and each by name (2 and 3); the same by a list of items, more
# than there are workgroups, so that one takes several in turn; one to four heads a workgroup; chunks of prompts, whose keys lie before them
@pytest.mark.parametrize("how", [0, 2, 3, "items 1", "items 2"])
@pytest.mark.parametrize("hq,hkv", [(8, 2), (4, 2), (2, 2)])
@pytest.mark.parametrize("lens,ctxs", [([1], [1]), ([31, 64, 33], [31, 70, 200]), ([200, 129], [200, 400]), ([700] * 12, [700] * 12)])
def test_paged_rows(gpu, hq, hkv, lens, ctxs, how):
    from nv_genai_amd import ops

    D, T, B = 128, sum(lens), len(lens)
    pages, q, kc, vc, bt, cu, cl = _pages(gpu, lens, ctxs, hq, hkv, T + hq)
    items = torch.from_numpy(ops.plan_prefill_items(cu.tolist(), ctxs, 0, B, hq, hkv)).to(gpu)
    n_items = torch.tensor([len(items)], dtype=torch.int32, device=gpu)

    def run(q, out):
        if isinstance(how, int):
            ops.kernels().prefill_attention(out, q, None, None, kc, vc, bt, cu, cl, hq, hkv, D, max(lens), D ** -0.5, True, 0, how, 1.0, 1.0)
        else:
            ops.kernels().prefill_attention_worklist(out, q, kc, vc, bt, cu, cl, hq, hkv, D ** -0.5, True, 0, items, n_items, 3, int(how[-1]), 2,
                                                     1.0, 1.0)
        return out

    got = run(q, torch.empty(T, hq * D, dtype=BF, device=gpu))
    at = 0
    for n, c, p in zip(lens, ctxs, [sum(pages[:i]) for i in range(B)]):
        m = (c + 63) // 64
        K = kc[p:p + m].transpose(1, 2).reshape(-1, hkv, D)[:c].transpose(0, 1).double().repeat_interleave(hq // hkv, 0)
        V = vc[p:p + m].permute(0, 3, 1, 2).reshape(-1, hkv, D)[:c].transpose(0, 1).double().repeat_interleave(hq // hkv, 0)
        S = q[at:at + n].view(n, -1, D).transpose(0, 1).double() @ K.transpose(1, 2).contiguous() * D ** -0.5
        P = S.masked_fill(torch.ones(n, c, device=gpu).triu(c - n + 1).bool(), float("-inf")).softmax(-1)
        flat = lambda x: x.transpose(0, 1).reshape(n, -1)  # noqa: E731
        ref = flat(P @ V)
        assert ((got[at:at + n].double() - ref).abs() <= 2.0 ** -8 * (flat(P @ V.abs()) + ref.abs())).all()
        at += n
    for by in (0, 8, 3):
        wide = torch.zeros(T, hq * D + 16, dtype=BF, device=gpu)[:, by:by + hq * D].copy_(q)
        room = torch.full((T + 1, hq * D + 16 + by), 7.0, dtype=BF, device=gpu)
        assert torch.equal(run(wide, room[:T, by:by + hq * D]), got)
        room[:T, by:by + hq * D] = 7.0
        assert (room == 7.0).all()


@pytest.mark.parametrize("by", [0, 8, 3])
def test_out_is_written_in_place(gpu, by):
    """Rows that no item covers are another kernel's, which may write them at the same time: no copy of the output is made, wherever it lies."""
    from nv_genai_amd import ops

    D, hq, hkv, lens = 128, 4, 2, [70, 33]
    T, w = sum(lens), hq * D
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=gpu)  # noqa: E731
    _, q, kc, vc, bt, cu, cl = _pages(gpu, lens, lens, hq, hkv, by)
    k, v = (torch.randn(T, hkv * D, device=gpu).to(BF) for _ in range(2))
    items, n = i32([[0, 0], [0, 1]]), i32([2])   # the first sequence alone
    room = torch.full((T, w + 16 + by), 7.0, dtype=BF, device=gpu)
    out, C = room[:, by:by + w], ops.kernels()
    calls = {2: lambda: C.prefill_attention_worklist(out, q, kc, vc, bt, cu, cl, hq, hkv, D ** -0.5, True, 0, items, n, 3, 1, 2, 1.0, 1.0),
             1: lambda: C.prefill_attention_worklist(out, q, kc, vc, bt, cu, cl, hq, hkv, D ** -0.5, True, 0, items, n, 3, 1, 1, 1.0, 1.0),
             "pages": lambda: C.prefill_attention(out, q, None, None, kc, vc, bt, cu, cl, hq, hkv, D, 70, D ** -0.5, True, 0, 2, 1.0, 1.0),
             "packed": lambda: C.prefill_attention(out, q, k, v, None, None, None, cu, None, hq, hkv, D, 70, D ** -0.5, True, 0, 0, 1.0, 1.0)}
    for name, call in calls.items():
        room.fill_(7.0)
        before = torch.cuda.memory_stats()["allocation.all.allocated"]
        call()
        assert torch.cuda.memory_stats()["allocation.all.allocated"] == before, name
        if name in (1, 2):
            assert bool((out[70:] == 7).all()) and not bool((out[:70] == 7).all())
        assert bool((room[:, :by] == 7).all()) and bool((room[:, by + w:] == 7).all())
