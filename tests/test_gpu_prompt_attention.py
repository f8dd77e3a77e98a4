"""The prompt pass's attention kernel where it can go wrong: both numbers of queries per wave, positions around the edges of its stages of 64 and tiles of 16 and 32,
workgroups that are not full, groups of heads that do not fit its four waves, and values that are not finite behind a query."""
import pytest
import torch

from bitstack_amd.utils import inference_utils as IU

pytestmark = pytest.mark.gpu


def inputs(B, n, heads, kv, max_len):
    g = torch.Generator(device="cuda").manual_seed(n + heads)
    q = torch.randn(B * n, heads * 128, generator=g, device="cuda").half()
    kc, vc = (torch.randn(B, kv, max_len, 128, generator=g, device="cuda").half() for _ in range(2))
    kc[:, :, n:], vc[:, :, n:] = float("nan"), float("nan")          # not read
    return q, kc, vc


# up to 400 workgroups of 32 queries per wave: 16 (the first line), more: 32
@pytest.mark.parametrize("B,n,heads,kv", [(1, 47, 3, 1), (1, 48, 5, 1), (2, 63, 7, 7), (1, 66, 10, 2), (1, 127, 6, 2), (1, 129, 1, 1), (1, 900, 8, 8),
                                          (16, 31, 128, 32), (8, 64, 128, 64), (8, 65, 64, 64), (4, 95, 128, 128), (3, 257, 96, 32), (8, 130, 40, 8), (12, 191, 24, 24)])
def test_against_float64(B, n, heads, kv):
    print(f"prompt attention B={B} n={n} heads={heads} kv={kv}", flush=True)
    d, rep = 128, heads // kv
    assert (B * kv * -(-(rep * -(-n // 32)) // 4) > 400) == (B > 2)
    q, kc, vc = inputs(B, n, heads, kv, n + 3)
    got = IU.attention_prefill_hip(q, kc, vc, n).double().view(B, n, kv, rep, d)
    qd = q.double().view(B, n, kv, rep, d).permute(0, 2, 3, 1, 4)
    kd, vd = (c[:, :, :n].double().unsqueeze(2).expand(B, kv, rep, n, d).contiguous() for c in (kc, vc))
    s = torch.matmul(qd, kd.transpose(-1, -2).contiguous()) / d ** 0.5
    s = s.masked_fill(torch.ones(n, n, device="cuda").triu(1).bool(), float("-inf"))
    ref = torch.matmul(torch.softmax(s, -1), vd).permute(0, 3, 1, 2, 4)
    # one rounding of the result, and one of every softmax weight (2^-11 of itself at most, weights sum to one; those below
    # 2^-14 of the largest lose up to 2^-25 of it each)
    bound = ref.abs() * 2.0 ** -11 + vd.abs().max() * (2.0 ** -11 + n * 2.0 ** -25)
    assert bool(((got - ref).abs() <= bound).all())
    assert float((got - ref).norm() / ref.norm()) < 6e-4


@pytest.mark.parametrize("B,heads,kv", [(1, 4, 2), (16, 64, 32)])
def test_values_behind_a_query(B, heads, kv):
    # a position that is not finite leaves the queries of the 32-position tiles before its own alone, and reaches every query from its own on
    n = 140
    q, kc, vc = inputs(B, n, heads, kv, n)
    want = IU.attention_prefill_hip(q, kc, vc, n).view(B, n, heads, 128)
    for at in (32, 40, 64, 96, 139):
        v = vc.clone()
        v[:, :, at, 5] = float("inf")
        k = kc.clone()
        k[:, :, at] = float("nan")
        for kk, vv, dim in ((kc, v, 5), (k, vc, 0)):
            got = IU.attention_prefill_hip(q, kk, vv, n).view(B, n, heads, 128)
            tile = at // 32 * 32
            assert torch.equal(got[:, :tile], want[:, :tile]), at
            assert not bool(got[:, at:, :, dim].isfinite().any()), at
