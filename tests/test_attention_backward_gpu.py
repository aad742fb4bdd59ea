"""Gradients of packed causal attention (attention_backward.hip) against 64 bits, where its tiles, halves and stores have their edges."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu
BF = torch.bfloat16


# one wave and two for 32 rows (sequences up to 64 tokens and above); ends within a tile's first and second half, a wave's 32 rows, the
# workgroup's 128, and rows past the end of all of these; parts of a KV head's queries (few workgroups) and all of them (many)
@pytest.mark.parametrize("D,hq,hkv,lens", [(128, 4, 1, [64, 1, 31]), (128, 4, 1, [65, 33, 64]), (128, 4, 2, [97, 96, 95, 1]), (128, 2, 2, [127, 128, 129, 160]),
                                           (128, 8, 2, [300, 193, 5]), (128, 40, 20, [130] * 7), (64, 4, 2, [129, 31, 128]), (32, 6, 3, [257, 64])])
def test_edges(gpu, D, hq, hkv, lens):
    from nv_genai_amd import ops

    g = torch.Generator("cuda").manual_seed(D + len(lens))
    T, G, scale = sum(lens), hq // hkv, D ** -0.5
    w = [hq * D, hkv * D, hkv * D]
    qkv = torch.randn(T, sum(w), device=gpu, generator=g).to(BF)
    do = torch.randn(T, hq * D, device=gpu, generator=g).to(BF)
    out, lse = torch.empty(T, hq * D, dtype=torch.float64, device=gpu), torch.empty(hq, T, device=gpu)
    ref = torch.empty(T, sum(w), dtype=torch.float64, device=gpu)
    bound = torch.empty_like(ref)
    at = 0
    for n in lens:
        rows = slice(at, at + n)
        q, k, v = (t.view(n, -1, D).transpose(0, 1).double() for t in qkv[rows].split(w, 1))
        k, v, d = k.repeat_interleave(G, 0), v.repeat_interleave(G, 0), do[rows].view(n, hq, D).transpose(0, 1).double()
        S = (q @ k.transpose(1, 2).contiguous() * scale).masked_fill(torch.ones(n, n, device=gpu).triu(1).bool(), -math.inf)
        P = S.softmax(-1)
        o = P @ v
        dP = d @ v.transpose(1, 2).contiguous()
        delta = (o * d).sum(-1, keepdim=True)
        dS = P * (dP - delta)
        # P and dS enter the products as bf16 (an ulp, 2^-8, for their rounding and that of the fp32 sums before it), delta comes of an
        # output in bf16, and the result is bf16
        e = 2.0 ** -8
        off = e * (dS.abs() + P * (o * d).abs().sum(-1, keepdim=True) * 2)
        t = lambda x: x.transpose(1, 2).contiguous()  # noqa: E731
        fold = lambda x: x.view(hkv, G, n, D).sum(1)  # noqa: E731
        flat = lambda x: x.transpose(0, 1).reshape(n, -1)  # noqa: E731
        ref[rows] = torch.cat([flat(dS @ k * scale), flat(fold(t(dS) @ q) * scale), flat(fold(t(P) @ d))], 1)
        bound[rows] = torch.cat([flat(off @ k.abs() * scale), flat(fold(t(off) @ q.abs()) * scale), flat(fold(e * t(P) @ d.abs()))], 1)
        out[rows], lse[:, rows] = flat(o), (S.logsumexp(-1) * math.log2(math.e)).float()
        at += n
    cu = torch.tensor([0, *torch.tensor(lens).cumsum(0).tolist()], dtype=torch.int32, device=gpu)
    got = torch.full((T + 1, sum(w)), 7.0, dtype=BF, device=gpu)
    ops.kernels().train_attention_backward(*got[:T].split(w, 1), do, *qkv.split(w, 1), out.to(BF), lse, cu, hq, hkv, D, max(lens), scale)
    assert ((got[:T].double() - ref).abs() <= bound + 2.0 ** -8 * (ref.abs() + bound)).all()
    assert (got[T] == 7).all()   # nothing is written past the last row


@pytest.mark.parametrize("B,S,D,hq,hkv", [(1, 1, 128, 2, 1), (3, 65, 128, 4, 2), (2, 33, 64, 3, 3)])
def test_log_sums_by_sequence(gpu, B, S, D, hq, hkv):
    """Natural logarithms [B, Hq, S] give the bits of what they are turned into."""
    from nv_genai_amd import ops

    g = torch.Generator("cuda").manual_seed(S)
    w = [hq * D, hkv * D, hkv * D]
    rn = lambda *s: torch.randn(*s, device=gpu, generator=g)  # noqa: E731
    qkv, do, out, lse = rn(B * S, sum(w)).to(BF), rn(B * S, hq * D).to(BF), rn(B * S, hq * D).to(BF), 30 + rn(B, hq, S)
    cu = torch.arange(B + 1, dtype=torch.int32, device=gpu) * S
    got = []
    for how in (lse, (lse.transpose(0, 1) * math.log2(math.e)).reshape(hq, -1).contiguous()):
        d = torch.empty_like(qkv)
        ops.kernels().train_attention_backward(*d.split(w, 1), do, *qkv.split(w, 1), out, how, cu, hq, hkv, D, S, D ** -0.5)
        got.append(d)
    assert torch.equal(*got)


@pytest.mark.parametrize("D", [64, 128])
def test_rows_far_apart(gpu, D):
    """Rows 2^25 values apart, beyond a tile's 32-bit addresses, give the bits of rows one behind the other."""
    from nv_genai_amd import ops

    T, step = 3, 1 << 25
    g = torch.Generator("cuda").manual_seed(D)
    rn = lambda *s: torch.randn(*s, device=gpu, generator=g)  # noqa: E731
    near = [rn(T, D).to(BF) for _ in range(4)]   # q, k, v, dout
    out, lse = rn(T, D).to(BF), 30 + rn(1, T)
    cu = torch.tensor([0, T], dtype=torch.int32, device=gpu)
    room = torch.empty((T - 1) * step + 4 * D, dtype=BF, device=gpu)
    far = [torch.as_strided(room, (T, D), (step, 1), i * D).copy_(t) for i, t in enumerate(near)]
    got = []
    for max_len in (64, 65):
        for q, k, v, do in (near, far):
            d = torch.empty(T, 3 * D, dtype=BF, device=gpu)
            ops.kernels().train_attention_backward(*d.split(D, 1), do, q, k, v, out, lse, cu, 1, 1, D, max_len, D ** -0.5)
            got.append(d)
    assert torch.equal(got[0], got[1]) and torch.equal(got[2], got[3])


def test_log_sums_by_sequence_are_of_one_length(gpu):
    from nv_genai_amd import ops

    T, D = 8, 64
    t = [torch.zeros(T, D, dtype=BF, device=gpu) for _ in range(8)]
    lse = torch.zeros(2, 1, 4, device=gpu)   # two sequences of 4 tokens; these are of 3 and 5
    cu = torch.tensor([0, 3, 8], dtype=torch.int32, device=gpu)
    with pytest.raises(RuntimeError, match="S tokens each"):
        ops.kernels().train_attention_backward(*t, lse, cu, 1, 1, D, 5, D ** -0.5)
