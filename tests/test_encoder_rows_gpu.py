"""Encoder forwards of few rows: up to 32 with the attention of one sequence inside a projection, above them LDS tiles of 32 and 64
features, with one group of waves and two."""
import pytest
import torch

from nv_genai_amd import ops

pytestmark = pytest.mark.gpu


def _exact(m, ids, cu):
    d = lambda t: t.double()  # noqa: E731
    ln = lambda x, g, b: torch.nn.functional.layer_norm(x, (x.shape[-1],), d(g), d(b), m.cfg.eps)  # noqa: E731
    out = []
    for lo, hi in zip(cu[:-1], cu[1:]):
        n = hi - lo
        if n == 0:
            continue
        x = ln(d(m.word)[ids[lo:hi].long()] + d(m.pos)[:n] + d(m.type)[0], *m.emb_ln)
        for L in m.layers:
            q, k, v = ((x @ d(L["wqkv"]).t() + d(L["bqkv"])).view(n, 3, m.cfg.heads, -1).permute(1, 2, 0, 3)).contiguous()
            p = torch.softmax(q @ k.transpose(1, 2).contiguous() * m.cfg.head_dim ** -0.5, -1)
            a = (p @ v).transpose(0, 1).reshape(n, -1)
            x = ln(x + a @ d(L["wo"]).t() + d(L["bo"]), L["ln1_g"], L["ln1_b"])
            h = torch.nn.functional.gelu(x @ d(L["wi"]).t() + d(L["bi"]))
            x = ln(x + h @ d(L["wo2"]).t() + d(L["bo2"]), L["ln2_g"], L["ln2_b"])
        out.append(x)
    return torch.cat(out)


@pytest.mark.parametrize("H,heads,F", [(128, 2, 256), (192, 6, 448), (384, 12, 1536), (768, 12, 3072), (1024, 16, 4096), (1024, 8, 8192)])
@pytest.mark.parametrize("lens", [[1], [5], [16], [17], [19], [32], [3, 1, 20], [32, 0], [33], [64, 1],
                                  [60, 64, 9], [50] * 5, [64] * 5])
def test_rows_forward(gpu, H, heads, F, lens):
    """Head sizes 32, 64 and 128, K ranges that the waves share unevenly, one tile of rows and two, one sequence and several.
    Against 64 bits, beside the same layers step by step: their roundings to bf16 are the same but for the sums before the
    norms (fp32 here), so the error is the steps' to within chance (a fifth at 128 values of one row)."""
    from nv_genai_amd.models.config import EncoderConfig
    from nv_genai_amd.models.encoder import EncoderModel

    m = EncoderModel(EncoderConfig(name="t", vocab_size=500, hidden=H, layers=3, heads=heads, ffn=F, max_position=64), gpu, seed=H)
    g = torch.Generator(gpu).manual_seed(7)
    for L in m.layers:   # biases and norms as of a trained model
        for n in ("bqkv", "bo", "bi", "bo2", "ln1_b", "ln2_b"):
            L[n].normal_(0, 0.1, generator=g)
        for n in ("ln1_g", "ln2_g"):
            L[n].normal_(1, 0.1, generator=g)
    T = sum(lens)
    cu = [0]
    for n in lens:
        cu.append(cu[-1] + n)
    ids = torch.randint(0, 500, (T,), generator=g, device=gpu, dtype=torch.int32)
    pos = torch.cat([torch.arange(n) for n in lens]).int().to(gpu)
    t = (ids, pos, torch.tensor(cu, dtype=torch.int32, device=gpu), max(lens))
    assert ops.encoder_covers(m.word, m.layers, heads, (m.pos, m.type, *m.emb_ln))

    def hidden():
        return ops.encoder_forward(t[0], t[1], None, t[2], t[3], m.word, m.pos, m.type, m.emb_ln, m.layers, heads, m.cfg.eps, m.scale)

    got, want = hidden(), _exact(m, ids, cu)
    e = torch.nn.functional
    x = ops.layernorm((e.embedding(ids.long(), m.word) + e.embedding(pos.long(), m.pos) + m.type[0]).contiguous(), *m.emb_ln, m.cfg.eps)
    for L in m.layers:
        qkv = torch.addmm(L["bqkv"], x, L["wqkv"].t())
        a = ops.varlen_attention(qkv[:, :H], qkv[:, H:2 * H], qkv[:, 2 * H:], t[2], heads, heads, H // heads, t[3], m.scale, causal=False)
        x = ops.layernorm(torch.addmm(L["bo"], a, L["wo"].t()), L["ln1_g"], L["ln1_b"], m.cfg.eps, resid=x)
        h = ops.bias_gelu_(x @ L["wi"].t(), L["bi"])
        x = ops.layernorm(torch.addmm(L["bo2"], h, L["wo2"].t()), L["ln2_g"], L["ln2_b"], m.cfg.eps, resid=x)
    err = lambda y: ((y.double() - want).norm() / want.norm()).item()  # noqa: E731
    assert err(got) <= 1.2 * err(x), (err(got), err(x))
    assert torch.equal(got, hidden())


# each tile with rows and features that do not fill it; above 1,024 rows the smallest, the last of hidden 1,024 and of 768 with LDS
# tiles, K slices of each count
@pytest.mark.parametrize("H,heads,F,T", [(384, 12, 1536, 1025), (384, 12, 1536, 2047), (128, 2, 256, 4100), (768, 12, 3072, 2276),
                                         (1024, 16, 4096, 1280), (1024, 16, 4096, 1281), (384, 12, 1536, 9001), (1024, 16, 4096, 301),
                                         (1024, 16, 4096, 513), (1024, 16, 4096, 1001), (192, 6, 448, 700), (768, 12, 3072, 511)])
def test_many_rows_forward(gpu, H, heads, F, T):
    test_rows_forward(gpu, H, heads, F, [64] * (T // 64) + [T % 64])


# rows at which both ways were timed: the last with the LDS tiles ahead, the first with the library's products ahead
@pytest.mark.parametrize("H,tiles,library", [(128, 20_000, 36_000), (192, 12_288, 20_480), (256, 8_192, 14_000), (320, 8_000, 12_288),
                                             (384, 6_144, 9_600), (448, 4_096, 7_000), (512, 3_500, 4_608), (576, 2_048, 3_584), (640, 2_048, 3_500),
                                             (704, 1_792, 2_560), (768, 1_700, 1_900), (896, 1_408, 1_700), (1024, 1_100, 1_340), (1536, 1_024, 1_025)])
def test_tiles_end_where_the_library_is_faster(gpu, H, tiles, library):
    assert tiles <= ops.kernels().encoder_tile_rows(H) < library


def test_norms_read_ahead_what_the_caches_hold(gpu):
    """The next product's weights, of the sizes that gain from it: what lies beyond them would be read twice."""
    f = ops.kernels().norm_reads_ahead
    for M in (1, 32):
        assert f(M, 4096, 1024, False) and f(M, 8192, 2048, False) and not f(M, 10240, 2560, False) and not f(M, 16384, 4096, False)
    for M, most, beyond in ((33, 1280, 1408), (512, 1280, 1408), (513, 1024, 1152), (1024, 1024, 1152)):
        assert f(M, 4 * most, most, True) and not f(M, 4 * beyond, beyond, True) and not f(M, 32768, 8192, True)
    assert not f(19, 1536, 448, False) and not f(19, 448, 1536, False) and f(19, 1152, 384, False)


def test_no_hidden_size_jumps(gpu):
    """Neighbouring sizes (64 apart) take the tiles up to neighbouring row counts: neither product nor quotient of rows and size jumps."""
    rows = {H: ops.kernels().encoder_tile_rows(H) for H in range(64, 4097, 64)}
    assert all(rows[H] >= rows[H + 64] >= rows[H] * (H / (H + 64)) ** 2 - 1 for H in range(64, 4096, 64) if H >= 128)


@pytest.mark.parametrize("H,heads,F", [(1024, 16, 4096), (768, 12, 3072), (384, 12, 1536)])
@pytest.mark.parametrize("more", [0, 1])
def test_forward_on_both_sides_of_the_line(gpu, H, heads, F, more):
    T = ops.kernels().encoder_tile_rows(H) + more
    test_rows_forward(gpu, H, heads, F, [64] * (T // 64) + [T % 64])


# the library's products, with the up projection, its bias and GELU in one kernel from 3,072 rows on: tiles of rows that are full, hold one
# row, or take a second round of workgroups; features that it does not take
@pytest.mark.parametrize("H,heads,F,T,one", [(1024, 16, 4096, 3071, False), (1024, 16, 4096, 3072, True), (1024, 16, 4096, 3329, True), (768, 12, 3072, 4097, True),
                                             (1024, 16, 4096, 4865, True), (768, 12, 2944, 4097, False)])
def test_forward_above_the_tiles(gpu, H, heads, F, T, one):
    assert T > ops.kernels().encoder_tile_rows(H) and ops.kernels().gemm_nt_gelu_covers(T, F, H) == one
    test_rows_forward(gpu, H, heads, F, [64] * (T // 64) + [T % 64])


def test_rows_of_another_sequence_do_not_mix(gpu):
    """A token outside the table gives its own sequence NaN and no other; infinities in one stay there."""
    from nv_genai_amd.models.config import encoder_config
    from nv_genai_amd.models.encoder import EncoderModel

    m = EncoderModel(encoder_config("encoder-tiny"), gpu, seed=2)
    ids = torch.arange(20, dtype=torch.int32, device=gpu)
    ids[15] = 10 ** 6
    pos, cu = torch.cat([torch.arange(12), torch.arange(8)]).int().to(gpu), torch.tensor([0, 12, 20], dtype=torch.int32, device=gpu)
    got = m.forward(ids, pos, cu, 12)
    assert torch.isfinite(got[0]).all() and torch.isnan(got[1]).all()
    alone = m.forward(ids[:12].contiguous(), pos[:12].contiguous(), cu[:2].contiguous(), 12)
    assert ((got[0] - alone[0]).norm() / alone[0].norm()).item() < 2e-2   # other kernels, three roundings of 2^-9 a layer
    assert torch.isnan(m.forward(ids[12:].contiguous(), pos[12:].contiguous(), (cu[1:] - 12).contiguous(), 8)).all()
