"""Decode attention at the edges of its tiles: 16 positions a tile, 8 or 16 waves taking tiles in turn, 1, 2 or 4 heads a
workgroup, workgroups of a KV head dealt to one XCD or not."""
import numpy as np
import pytest
import torch

from bitstack_amd import _lib
from bitstack_amd.utils import inference_utils as IU


def test_positions_are_cut_where_the_cache_is_long_and_the_heads_are_few():
    parts = lambda *shape: _lib.lib().bs_attention_decode_workspace_bytes(*shape) > 0
    for B, heads, kv, line in ((1, 32, 8, 1100), (4, 32, 8, 1100), (1, 6, 3, 1100), (1, 32, 32, 1000), (1, 8, 8, 1000), (2, 6, 2, 1000)):
        assert [parts(B, heads, kv, 128, n) for n in (1, 512, line - 1, line, 8192)] == [False, False, False, True, True]
    assert parts(16, 32, 8, 128, 4096) and not parts(17, 32, 8, 128, 4096)      # more than 128 workgroups fill the chip


@pytest.mark.gpu
@pytest.mark.parametrize("B,heads,kv", [(1, 32, 8), (2, 6, 2), (9, 32, 8), (9, 32, 32), (17, 32, 16), (17, 32, 8), (33, 32, 8)])
def test_attention_at_tile_edges(B, heads, kv):
    d, max_len = 128, 272
    g = torch.Generator().manual_seed(B * 100 + heads + kv)
    k = torch.randn(B, kv, max_len, d, generator=g).half()
    v = torch.randn(B, kv, max_len, d, generator=g).half()
    qkv = torch.randn(B, (heads + 2 * kv) * d, generator=g).half()
    cos, sin = torch.ones(max_len, d // 2).half().cuda(), torch.zeros(max_len, d // 2).half().cuda()   # the rotation is exact
    q = qkv[:, :heads * d].double().view(B, kv, heads // kv, d)
    kn, vn = qkv[:, heads * d:(heads + kv) * d].view(B, kv, d), qkv[:, (heads + kv) * d:].view(B, kv, d)
    kd, vd = k.cuda(), v.cuda()
    for at in (0, 1, 15, 16, 17, 127, 128, 129, 255, 256, 257, max_len - 1):
        print(f"attention B={B} heads={heads} kv={kv} at={at}", flush=True)
        kc, vc = kd.clone(), vd.clone()
        kc[:, :, at + 1:] = float("nan")        # what lies behind the position is not read
        vc[:, :, at:] = float("nan")
        got = IU.attention_decode_hip(qkv.cuda(), kc, vc, cos, sin, torch.tensor([at], device="cuda"), heads, kv)
        ks, vs = k[:, :, :at + 1].double().clone(), v[:, :, :at + 1].double().clone()
        ks[:, :, at], vs[:, :, at] = kn.double(), vn.double()
        p = torch.softmax(torch.matmul(q, ks.transpose(2, 3)) / d ** 0.5, -1)
        ref = torch.matmul(p, vs).reshape(B, heads * d).numpy()
        assert torch.equal(kc[:, :, at].cpu(), kn) and torch.equal(vc[:, :, at].cpu(), vn)
        assert torch.equal(kc[:, :, :at].cpu(), k[:, :, :at]) and torch.equal(vc[:, :, :at].cpu(), v[:, :, :at])
        # one rounding to fp16; scores of size up to 5 in fp32 sums of 128 terms move the weights by at most 2^-14 of themselves
        bound = np.abs(ref) * 2.0 ** -11 + np.abs(vs.numpy()).max() * 2.0 ** -14 + 2.0 ** -25
        assert (np.abs(got.double().cpu().numpy() - ref) <= bound).all()


@pytest.mark.gpu
@pytest.mark.parametrize("B,heads,kv,max_len", [(1, 32, 8, 4096), (1, 32, 8, 1100), (1, 6, 2, 4100), (3, 8, 4, 2050), (2, 16, 16, 1024), (16, 32, 8, 1130)])
def test_attention_over_split_positions(B, heads, kv, max_len):
    """Few heads over a long cache: the positions in parts (up to 16 of them, most without a position early on)."""
    d = 128
    g = torch.Generator(device="cuda").manual_seed(B + heads + max_len)
    k = torch.randn(B, kv, max_len, d, generator=g, device="cuda").half()
    v = torch.randn(B, kv, max_len, d, generator=g, device="cuda").half()
    qkv = torch.randn(B, (heads + 2 * kv) * d, generator=g, device="cuda").half()
    cos, sin = torch.ones(max_len, d // 2).half().cuda(), torch.zeros(max_len, d // 2).half().cuda()
    q = qkv[:, :heads * d].double().view(B, kv, heads // kv, d)
    kn, vn = qkv[:, heads * d:(heads + kv) * d].view(B, kv, d), qkv[:, (heads + kv) * d:].view(B, kv, d)
    for at in (0, 16, 511, 512, 513, 768, 769, 1000, max_len - 1):
        print(f"split attention B={B} heads={heads} kv={kv} max_len={max_len} at={at}", flush=True)
        kc, vc = k.clone(), v.clone()
        kc[:, :, at:] = float("nan")
        vc[:, :, at:] = float("nan")
        got = IU.attention_decode_hip(qkv, kc, vc, cos, sin, torch.tensor([at], device="cuda"), heads, kv).double()
        ks, vs = k[:, :, :at + 1].double(), v[:, :, :at + 1].double()
        ks[:, :, at], vs[:, :, at] = kn.double(), vn.double()
        p = torch.softmax((q.unsqueeze(3) * ks.unsqueeze(2)).sum(-1) / d ** 0.5, -1)
        ref = (p.unsqueeze(-1) * vs.unsqueeze(2)).sum(3).reshape(B, heads * d)
        assert torch.equal(kc[:, :, at], kn) and torch.equal(vc[:, :, at], vn)
        bound = ref.abs() * 2.0 ** -11 + vs.abs().max() * 2.0 ** -14 + 2.0 ** -25      # as above
        assert bool(((got - ref).abs() <= bound).all())
    for at in (-1, max_len):                     # outside of the cache: zeros
        assert not IU.attention_decode_hip(qkv, kc, vc, cos, sin, torch.tensor([at], device="cuda"), heads, kv).any()


@pytest.mark.gpu
@pytest.mark.parametrize("B,heads,kv,max_len,at", [(1, 32, 8, 272, 100), (2, 6, 2, 272, 33), (9, 32, 8, 272, 250), (17, 32, 8, 272, 128), (33, 32, 8, 272, 200),
                                                   (1, 32, 8, 2100, 1500), (1, 6, 2, 2100, 1500), (2, 16, 16, 2100, 700)])
def test_an_infinite_value_stays_infinite(B, heads, kv, max_len, at):
    """Values of +inf and -inf in the cache (the first and the last row of it among them) and in this step's own row: the dimensions they
    stand in come out as their sign, all others as if they were not there; one of each sign in a dimension makes NaN."""
    print(f"infinite values B={B} heads={heads} kv={kv} max_len={max_len} at={at}", flush=True)
    d, inf = 128, float("inf")
    g = torch.Generator(device="cuda").manual_seed(at + heads)
    k = torch.randn(B, kv, max_len, d, generator=g, device="cuda").half()
    v = torch.randn(B, kv, max_len, d, generator=g, device="cuda").half()
    qkv = torch.randn(B, (heads + 2 * kv) * d, generator=g, device="cuda").half()
    vn = qkv[:, (heads + kv) * d:].view(B, kv, d)
    v[:, :, 0, 3], v[:, 0, 20, 7], v[:, :, at - 1, 64], vn[:, :, 127] = inf, -inf, inf, -inf
    v[:, :, 5, 90], v[:, :, at - 2, 90] = inf, -inf
    cos, sin = torch.ones(max_len, d // 2).half().cuda(), torch.zeros(max_len, d // 2).half().cuda()
    q, kn = qkv[:, :heads * d].double().view(B, kv, heads // kv, d), qkv[:, heads * d:(heads + kv) * d].view(B, kv, d)
    got = IU.attention_decode_hip(qkv, k.clone(), v.clone(), cos, sin, torch.tensor([at], device="cuda"), heads, kv).double().view(B, kv, -1, d)
    ks, vs = k[:, :, :at + 1].double(), v[:, :, :at + 1].double()
    ks[:, :, at], vs[:, :, at] = kn.double(), vn.double()
    p = torch.softmax((q.unsqueeze(3) * ks.unsqueeze(2)).sum(-1) / d ** 0.5, -1)
    ref = (p.unsqueeze(-1) * vs.unsqueeze(2)).sum(3)
    assert torch.equal(got.isnan(), ref.isnan()) and bool(ref[..., 90].isnan().all())
    assert torch.equal(got.isinf(), ref.isinf()) and torch.equal(got[ref.isinf()], ref[ref.isinf()]) and int(ref.isinf().sum()) >= 3 * B * heads
    rest = ref.isfinite()
    # one rounding to fp16; scores of size up to 5 in fp32 sums of 128 terms move the weights by at most 2^-14 of themselves
    bound = ref.abs() * 2.0 ** -11 + float(vs[vs.isfinite()].abs().max()) * 2.0 ** -14 + 2.0 ** -25
    assert bool(((got - ref).abs() <= bound)[rest].all())
