"""The kernels between the linears of a prompt pass, against float64 (one rounding to fp16) or the plain kernel."""
import pytest
import torch

from bitstack_amd import BitStackLinear
from bitstack_amd.utils import inference_utils as IU
from bitstack_amd.utils.synthetic import synthetic_layer

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,n,heads,kv,d,max_len", [(1, 1, 2, 1, 128, 1), (2, 5, 32, 8, 128, 9), (3, 7, 4, 4, 64, 7), (1, 3, 5, 1, 16, 4),
                                                    (2, 3, 3, 3, 6, 5), (2, 33, 6, 2, 256, 40), (1, 2, 2, 2, 24, 2)])
def test_rope_store(B, n, heads, kv, d, max_len):
    g = torch.Generator(device="cuda").manual_seed(d + n)
    q, k, v = (torch.randn(B * n, h * d, generator=g, device="cuda").half() for h in (heads, kv, kv))
    ang = torch.rand(max_len, d // 2, generator=g, device="cuda") * 6.28
    cos, sin = ang.cos().half(), ang.sin().half()
    kc, vc = (torch.full((B, kv, max_len, d), 7.0, device="cuda").half() for _ in range(2))
    rot = q.clone()
    IU.rope_store_hip(rot, k, v, cos, sin, kc, vc, n)

    def want(x, h):
        x = x.double().view(B, n, h, d)
        c, s = (t[:n].double().view(1, n, 1, d // 2) for t in (cos, sin))
        a, b = x[..., :d // 2], x[..., d // 2:]
        return torch.cat([a * c - b * s, b * c + a * s], -1)

    # one rounding to fp16, and sums of two products of size up to 2^3 in fp32
    def check(got, ref):
        assert bool(((got.double() - ref).abs() <= ref.abs() * 2.0 ** -11 + 2.0 ** -20).all())
    check(rot.view(B, n, heads, d), want(q, heads))
    check(kc[:, :, :n].transpose(1, 2), want(k, kv))
    assert torch.equal(vc[:, :, :n].transpose(1, 2), v.view(B, n, kv, d))
    assert bool((kc[:, :, n:] == 7).all()) and bool((vc[:, :, n:] == 7).all())


@pytest.mark.parametrize("count", [1, 7, 8, 9, 2047, 2048, 2049, 5 * 14336])
def test_silu_mul(count):
    g = torch.Generator(device="cuda").manual_seed(count)
    a, b = (torch.randn(count, generator=g, device="cuda").half() * 4 for _ in range(2))
    ref = a.double() * torch.sigmoid(a.double()) * b.double()
    up = b.clone()
    y = IU.silu_mul_hip(a, up)
    assert y.data_ptr() == a.data_ptr() and torch.equal(up, b)
    # one rounding (subnormal below 2^-14), and 2^-20 for exp, quotient and product in fp32
    assert bool(((y.double() - ref).abs() <= ref.abs() * (2.0 ** -11 + 2.0 ** -20) + 2.0 ** -25).all())


@pytest.mark.parametrize("T,H", [(1, 8), (3, 2048), (2, 2056), (5, 4096), (2, 16384)])
def test_add_rmsnorm(T, H):
    g = torch.Generator(device="cuda").manual_seed(H)
    x, add = (torch.randn(T, H, generator=g, device="cuda").half() for _ in range(2))
    w = torch.rand(H, generator=g, device="cuda").half()
    x0, want = x.clone(), x + add
    s, y = IU.add_rmsnorm_hip(x, add, w, 1e-5)
    assert torch.equal(s, want) and torch.equal(x, x0) and s.data_ptr() == add.data_ptr()
    assert torch.equal(y, IU.rmsnorm_hip(want, w, 1e-5))


def test_norms_refuse_weights_and_outputs_of_another_size():
    x, w = torch.zeros(3, 512, device="cuda").half(), torch.ones(512, device="cuda").half()
    for call in (lambda: IU.rmsnorm_hip(x, w[:256], 1e-5), lambda: IU.add_rmsnorm_hip(x, x.clone(), w[:8], 1e-5),
                 lambda: IU.rmsnorm_hip(x, w, 1e-5, out=x[:2]), lambda: IU.rmsnorm_hip(x, w, 1e-5, out=torch.zeros(3, 512, device="cuda"))):
        with pytest.raises(ValueError):
            call()
    assert IU.rmsnorm_hip(x, w.view(1, 512), 1e-5).shape == x.shape


@pytest.mark.parametrize("B,n,heads,kv,max_len", [(1, 1, 4, 1, 1), (2, 15, 8, 2, 20), (1, 16, 6, 3, 16), (3, 17, 5, 5, 40), (1, 31, 32, 8, 31),
                                                  (2, 32, 8, 8, 33), (1, 33, 12, 4, 64), (2, 64, 4, 2, 64), (1, 65, 4, 4, 70), (1, 517, 8, 2, 600)])
def test_attention_prefill(B, n, heads, kv, max_len):
    print(f"prompt attention B={B} n={n} heads={heads} kv={kv}", flush=True)
    d, rep = 128, heads // kv
    g = torch.Generator(device="cuda").manual_seed(n + heads)
    q = torch.randn(B * n, heads * d, generator=g, device="cuda").half()
    kc, vc = (torch.randn(B, kv, max_len, d, generator=g, device="cuda").half() for _ in range(2))
    kc[:, :, n:], vc[:, :, n:] = float("nan"), float("nan")          # not read
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
    # and not far from the error of one rounding over the whole
    assert float((got - ref).norm() / ref.norm()) < 6e-4


@pytest.mark.parametrize("T,N,shapes", [(129, 256, [(2, 64), (1, 40)]), (200, 1024, [(3, 512), (2, 128), (1, 128)]), (300, 136, [(2, 72), (2, 72)]),
                                        (257, 4096, [(2, 4096), (3, 1024), (1, 1024)]), (140, 4096, [(1, 8184), (2, 8184)])])
def test_forward_cat_is_the_matrices_side_by_side(T, N, shapes):
    mods, x = [], None
    for j, (I, M) in enumerate(shapes):
        q, u, vt, xj = synthetic_layer(M, N, I, T, seed=j, device="cuda")
        x = xj if x is None else x
        mod = BitStackLinear(0, N, M, 16, False, False, "cuda", fused_level=5)
        mod.w_bit, mod.qweight, mod.u, mod.vt = I, q, u, vt
        mods.append(mod)
    x = x.view(T, N).contiguous()
    y = IU.forward_cat_hip(mods, x)
    assert y is not None and y.shape == (T, sum(M for _, M in shapes))
    want = torch.cat([m(x) for m in mods], 1).double()
    # the same weights and fp32 sums, in another order at most: a last bit of fp16 here and there
    assert bool(((y.double() - want).abs() <= want.abs() * 2.0 ** -10 + want.abs().max() * 2.0 ** -13).all())
    if N % 128 == 0:                                                     # (other column counts are rebuilt for any token count)
        assert IU.forward_cat_hip(mods, x[:8].contiguous()) is None
    mods[0].bias = torch.zeros(shapes[0][1], device="cuda").half()
    assert IU.forward_cat_hip(mods, x) is None


def test_forward_cat_decides_from_sizes_before_it_touches_the_blocks(monkeypatch):
    def mods(rows, N, blocks=2):
        out = []
        for M in rows:
            q, u, vt, _ = synthetic_layer(M, N, blocks, 1, device="cuda")
            mod = BitStackLinear(0, N, M, 16, False, False, "cuda", fused_level=5)
            mod.w_bit, mod.qweight, mod.u, mod.vt = blocks, q, u, vt
            out.append(mod)
        return out
    small, wide = mods((512, 256), 1024), mods((6152, 6152), 8192)              # (wide: 192 MiB of weights, beyond every limit)
    x, xw = torch.randn(300, 1024, device="cuda").half(), torch.randn(300, 8192, device="cuda").half()
    want = IU.forward_cat_hip(small, x)
    monkeypatch.setattr(IU, "MatrixGroup", None)
    monkeypatch.setattr(BitStackLinear, "_stacked", None)
    assert IU.forward_cat_hip(small, x[:5].contiguous()) is None and IU.forward_cat_hip(wide, xw) is None
    assert torch.equal(IU.forward_cat_hip(small, x), want)
    for bad in (x.float(), x.view(1, 300, 1024), x.t().contiguous().t(), x[:, :1016].contiguous(), x[:0], x.cpu()):
        assert IU.forward_cat_hip(small, bad) is None
    for blocks in (0, 3):                                                        # none, and more than are stacked
        small[0].w_bit = blocks
        assert IU.forward_cat_hip(small, x) is None
    small[0].w_bit = 2
    small[1].vt = small[1].vt.float()
    assert IU.forward_cat_hip(small, x) is None


def test_column_slices_as_operands():
    B, n, heads, kv, d, width = 2, 33, 4, 2, 128, 72
    g = torch.Generator(device="cuda").manual_seed(5)
    qkv = torch.randn(B * n, (heads + 2 * kv) * d, generator=g, device="cuda").half()
    cos, sin = (torch.rand(40, d // 2, generator=g, device="cuda").half() for _ in range(2))
    caches = [torch.zeros(B, kv, 40, d, device="cuda").half() for _ in range(4)]
    q, k, v = qkv.split((heads * d, kv * d, kv * d), 1)
    qc, kc, vc = (t.contiguous() for t in (q, k, v))
    IU.rope_store_hip(qc, kc, vc, cos, sin, caches[0], caches[1], n)
    IU.rope_store_hip(q, k, v, cos, sin, caches[2], caches[3], n)
    assert torch.equal(q, qc) and torch.equal(caches[0], caches[2]) and torch.equal(caches[1], caches[3])
    assert torch.equal(IU.attention_prefill_hip(q, caches[2], caches[3], n), IU.attention_prefill_hip(qc, caches[0], caches[1], n))
    both = torch.randn(5, 2 * width, generator=g, device="cuda").half()
    a, b = both.chunk(2, 1)
    assert torch.equal(IU.silu_mul_hip(a, b), IU.silu_mul_hip(a.contiguous(), b.contiguous()))
