"""Every build of the dense product's pipeline (gemm_pipe.hip) that a forward or linear_f16_hip runs: each tile, in one piece and cut into parts, at each number of stages; as many k-steps as
stages, one fewer and up to twice as many, and in parts every remainder of them; ragged tokens and features.  Each case names the tile, parts and stages that it is there for, and is
checked to have them."""
import pytest
import torch

from bitstack_amd import _lib
from bitstack_amd.utils import inference_utils as IU
from bitstack_amd.utils.synthetic import synthetic_layer

# (tile, parts, stages): (tokens, out features, in features) behind a rebuilt weight
REBUILT = {
    ((64, 64), 1, 4): [(33, 17, 192), (49, 17, 256), (33, 17, 320), (49, 17, 384), (33, 17, 448), (49, 17, 512)],
    ((64, 128), 1, 3): [(50, 17, 128), (65, 2497, 192), (163, 16440, 256), (161, 16385, 320)],
    ((64, 128), 1, 4): [(65, 8462, 256), (65, 8317, 320), (65, 8435, 384), (33, 16667, 448), (66, 8274, 512)],
    ((64, 128), 8, 3): [(2, 5584, 6080), (2, 6760, 5056)],
    ((64, 128), 11, 3): [(2, 4352, 7744)],
    ((64, 128), 12, 4): [(2, 1400, 24256), (2, 1344, 25152), (2, 1472, 22848), (2, 1952, 17344)],
    ((96, 128), 1, 2): [(65, 16399, 64), (65, 16765, 128), (65, 16947, 192), (403, 10881, 256)],
    ((96, 128), 1, 4): [(66, 16550, 256), (65, 16415, 320), (65, 17367, 384), (65, 16932, 448), (67, 16745, 512)],
    ((96, 128), 4, 2): [(65, 12416, 2752)],
    ((96, 128), 12, 2): [(65, 4576, 7360)],
    ((96, 128), 8, 4): [(68, 3024, 11200)],
    ((96, 128), 12, 4): [(66, 1392, 24448), (66, 1520, 22208), (65, 1288, 26624)],
    ((128, 128), 1, 2): [(99, 16437, 64), (100, 16675, 128), (97, 16515, 192)],
    ((128, 128), 1, 4): [(97, 16468, 256), (97, 16771, 320), (98, 16469, 384), (97, 16548, 448), (97, 16539, 512)],
    ((128, 128), 6, 2): [(621, 2096, 19904), (595, 2120, 16384)],
    ((128, 128), 12, 4): [(97, 1888, 18048), (98, 1584, 22208), (101, 2464, 13824), (99, 2048, 17152)],
    ((128, 192), 1, 3): [(483, 10911, 128), (194, 18228, 192), (193, 16578, 256), (196, 16425, 320), (193, 16388, 384)],
    ((128, 192), 4, 3): [(66, 10888, 3328), (69, 12264, 2816)],
    ((128, 192), 8, 3): [(67, 5952, 5888)],
    ((128, 256), 1, 2): [(293, 16945, 64), (295, 16639, 128), (294, 16662, 192), (293, 16898, 256)],
    ((128, 256), 1, 3): [(293, 16680, 576)],
    ((128, 256), 6, 3): [(100, 8752, 3904)],
    ((128, 256), 12, 3): [(98, 4296, 8512), (101, 5016, 7360)],
    ((160, 128), 1, 2): [(129, 16709, 64), (129, 16760, 128)],
    ((160, 128), 1, 3): [(130, 16423, 192), (129, 16547, 256), (131, 16609, 320), (131, 16593, 384)],
    ((160, 128), 8, 3): [(129, 2816, 12480), (132, 3872, 8704)],
    ((160, 128), 12, 3): [(130, 1944, 17856)],
    ((160, 256), 1, 3): [(393, 16389, 192), (388, 16465, 256), (388, 16460, 320), (386, 17223, 384)],
    ((160, 256), 8, 3): [(130, 6200, 6016), (130, 6560, 6208)],
    ((160, 256), 12, 3): [(130, 4392, 8256)],
    ((192, 128), 1, 3): [(484, 8843, 128), (328, 11020, 192), (161, 18127, 256), (162, 16819, 320), (161, 16761, 384)],
    ((192, 128), 8, 3): [(162, 3648, 9408)],
    ((192, 128), 12, 3): [(162, 1512, 22848), (161, 1296, 26880)],
    ((192, 192), 1, 3): [(1036, 7228, 128), (518, 13078, 192), (524, 13257, 256), (648, 10894, 320), (513, 13548, 384)],
    ((192, 192), 4, 3): [(130, 11000, 3136)],
    ((192, 192), 8, 3): [(130, 5968, 5952)],
    ((192, 192), 11, 3): [(147, 4392, 7744)],
    ((192, 256), 1, 2): [(389, 16929, 64), (385, 17069, 128), (805, 9884, 192), (801, 9911, 256)],
    ((192, 256), 12, 2): [(556, 1736, 19904), (526, 1472, 23680)],
    ((224, 128), 1, 3): [(386, 13243, 128), (401, 13199, 192), (385, 13342, 256), (393, 12527, 320), (388, 12572, 384)],
    ((224, 128), 6, 3): [(195, 4520, 7488)],
    ((224, 128), 8, 3): [(193, 3216, 11008)],
    ((224, 128), 12, 3): [(200, 2200, 15552)],
    ((224, 256), 1, 2): [(582, 16456, 64), (590, 16744, 128), (586, 16814, 192), (591, 16745, 256)],
    ((224, 256), 3, 2): [(195, 16720, 3008)],
    ((224, 256), 8, 2): [(194, 6544, 8576)],
    ((256, 128), 1, 3): [(3658, 2055, 128), (679, 10820, 192), (692, 10825, 256), (689, 10766, 320), (691, 10762, 384)],
    ((256, 128), 3, 3): [(230, 10784, 3328)],
    ((256, 128), 12, 3): [(237, 2656, 21440), (249, 2632, 12992)],
    ((256, 192), 1, 2): [(988, 10889, 64), (971, 11061, 128), (963, 11085, 192), (967, 10936, 256)],
    ((256, 192), 4, 2): [(453, 5672, 6784)],
    ((256, 192), 8, 2): [(451, 2848, 12992)],
    ((256, 256), 1, 2): [(673, 16597, 64), (675, 17010, 128), (676, 16738, 192), (684, 16634, 256)],
    ((256, 256), 12, 2): [(483, 2168, 18112), (508, 2120, 17664)],
}
# ... and of linear_f16_hip, whose 128 x 128 tiles have two workgroups on a CU too
LINEAR = {
    ((64, 64), 1, 4): [(131, 1001, 192), (309, 1021, 320)],
    ((128, 128), 1, 4): [(1000, 4090, 256), (600, 5001, 448)],
    ((128, 128), 1, 2): [(1152, 4096, 256), (1151, 4090, 320), (1030, 4000, 1024), (500, 5303, 64), (1000, 4090, 192)],
    ((128, 256), 1, 2): [(500, 14333, 64), (755, 8066, 512)],
    ((128, 256), 1, 3): [(500, 14333, 576), (755, 8066, 640), (512, 14336, 704)],
    ((256, 256), 1, 2): [(1000, 14333, 64), (2047, 8185, 192)],
}
FLAT = [(rebuilt, *key, *dims) for rebuilt, table in ((True, REBUILT), (False, LINEAR)) for key, cases in table.items() for dims in cases]


def test_the_cases_have_the_builds_they_are_there_for():
    for rebuilt, tile, parts, stages, *dims in FLAT:
        assert _lib.dense_plan(*dims, rebuilt) == (*tile, parts, stages), (rebuilt, dims)
    steps = {}
    for _, tile, parts, stages, T, M, N in FLAT:
        steps.setdefault((tile, parts > 1, stages), set()).add(-(-N // 64 // parts) % stages)
    assert all(len(rest) == stages for (_, _, stages), rest in steps.items()), steps


def close(y, x, w, bias):
    want, size = torch.nn.functional.linear(x, w, bias), torch.nn.functional.linear(x.abs(), w.abs(), None if bias is None else bias.abs())
    # y is rounded to fp16 once (2^-11 of it, 2^-25 where it is subnormal); either side's fp32 sums of N products are off by up to N 2^-24 of the sum of their sizes
    bound = want.abs() * 2.0 ** -11 + 2.0 ** -25 + 2 * (x.shape[1] + 1) * 2.0 ** -24 * size
    return bool(((y.float() - want).abs() <= bound).all())


@pytest.mark.gpu
@pytest.mark.parametrize("rebuilt,tile,parts,stages,T,M,N", FLAT)
def test_build(rebuilt, tile, parts, stages, T, M, N):
    print(f"dense build rebuilt={rebuilt} tile={tile} parts={parts} stages={stages} T={T} M={M} N={N}", flush=True)
    assert _lib.dense_plan(T, M, N, rebuilt) == (*tile, parts, stages)
    dev = torch.device("cuda")
    g = torch.Generator(device=dev).manual_seed(T + M + N)
    bias = (torch.randn(M, device=dev, generator=g) * 0.05).half() if T % 2 else None
    if not rebuilt:
        x, w = torch.randn(T, N, device=dev, generator=g).half(), (torch.randn(M, N, device=dev, generator=g) * 0.05).half()
        y = IU.linear_f16_hip(x, w, bias)
    else:
        q, u, vt, x = synthetic_layer(M, N, 1, T, seed=T + M + N, device=dev, signed_factors=True)
        u, x = (u * 20).half(), x.reshape(T, N)
        L = _lib.lib()
        _lib.check(L.bs_set_prefill_kernel(_lib.PREFILL_REBUILD), "bs_set_prefill_kernel")
        try:
            assert L.bs_forward_path(1, M, N, 16, T) == 0
            y = IU.bitstack_forward_hip(q, u, vt, x, bias)
        finally:
            L.bs_set_prefill_kernel(_lib.PREFILL_AUTO)
        w = IU.unpack_and_reconstruct_w_hip(q, u, vt)
    assert close(y.reshape(T, M), x.float(), w.float(), None if bias is None else bias.float())


# (tokens, out features, in features) of a large tile, and a block of it (256 tokens, 5200 features) that is small enough for linear_f16_kernel's tile of 64 x 64 in steps of 128: another
# kernel's products of the same operands
@pytest.mark.gpu
@pytest.mark.parametrize("T,M,N,tile", [(2048, 14336, 4096, (256, 256)), (2047, 14335, 4160, (256, 256)), (500, 14333, 4096, (128, 256)), (600, 5300, 4096, (128, 128))])
def test_large_tiles_against_the_other_kernel(T, M, N, tile):
    print(f"dense tiles against the other kernel T={T} M={M} N={N}", flush=True)
    assert _lib.dense_plan(T, M, N)[:3] == (*tile, 1) and _lib.dense_plan(T, M, N)[3] > 0
    assert _lib.dense_plan(256, 5200, N) == (64, 64, 1, 0) and _lib.linear_plan(256, 5200, N)[2] == 128
    g = torch.Generator(device="cuda").manual_seed(T + M)
    x, w = torch.randn(T, N, device="cuda", generator=g).half(), (torch.randn(M, N, device="cuda", generator=g) * 0.05).half()
    y = IU.linear_f16_hip(x, w, None)
    for t, m in ((0, 0), (T - 256, M - 5200)):
        small = IU.linear_f16_hip(x[t:t + 256].contiguous(), w[m:m + 5200].contiguous(), None).float()
        part = y[t:t + 256, m:m + 5200].float()
        # the same products added in two orders, each up to N 2^-24 of their sizes off, and rounded once each
        size = x[t:t + 256].float().abs() @ w[m:m + 5200].float().abs().T
        assert bool(((part - small).abs() <= 2.0 ** -10 * small.abs() + 2.0 ** -24 + 2 * N * 2.0 ** -24 * size).all())
