"""The dense product's tiles and pipeline depths (gemm_pipe.hip) where they can go wrong: every tile that linear_choice has, with one workgroup per CU and, where that
is another number of stages, two; ragged tokens and features; fewer k-steps than stages, and every remainder of them."""
import pytest
import torch

from bitstack_amd import _lib
from bitstack_amd.utils import inference_utils as IU
from bitstack_amd.utils.synthetic import synthetic_layer

# tokens, out features, in features: the tile that the estimates choose
CASES = [(131, 102, 64), (131, 102, 128), (133, 104, 192), (155, 301, 704), (190, 250, 832),      # 64 x 64
         (3592, 269, 576),                                                                       # 64 x 64, two per CU
         (131, 2100, 64), (225, 538, 128), (1907, 127, 64), (140, 4101, 1472),                   # 64 x 128
         (166, 16559, 128), (184, 16644, 192),                                                   # 64 x 128, two
         (133, 11089, 64), (412, 5775, 128), (2097, 1135, 192), (161, 17104, 64), (885, 5508, 128),   # 96 x 128, two
         (201, 11259, 64), (452, 7623, 128), (1052, 3278, 320),                                  # 128 x 128
         (587, 9521, 64), (229, 17211, 384), (291, 17105, 64), (626, 11220, 128),                # 128 x 192, 128 x 256
         (133, 16586, 64), (555, 6582, 128), (4142, 2422, 1472), (830, 10798, 2112),             # 160 x 128, two
         (393, 16603, 192), (3200, 3048, 320), (783, 19869, 320),                                # 160 x 256
         (329, 13161, 128), (844, 5824, 320), (4909, 1542, 128), (1158, 6896, 320),              # 192 x 128, 192 x 192
         (399, 13236, 64), (865, 7758, 128), (613, 16648, 64), (2311, 5611, 128),                # 224 x 128, 224 x 256
         (3817, 2123, 64), (4189, 1916, 128)]                                                    # 256 x 128


@pytest.mark.gpu
@pytest.mark.parametrize("T,M,N", CASES)
def test_tile_and_depth(T, M, N):
    print(f"dense stages T={T} M={M} N={N}", flush=True)
    dev = torch.device("cuda")
    q, u, vt, x = synthetic_layer(M, N, 1, T, seed=T + M + N, device=dev, signed_factors=True)
    u = (u * 20).half()
    bias = (torch.randn(M, generator=torch.Generator().manual_seed(T)) * 0.05).half().to(dev) if T % 2 else None
    L = _lib.lib()
    _lib.check(L.bs_set_prefill_kernel(_lib.PREFILL_REBUILD), "bs_set_prefill_kernel")
    try:
        y = IU.bitstack_forward_hip(q, u, vt, x, bias)
        assert torch.equal(IU.bitstack_forward_hip(q, u, vt, x, bias), y)
    finally:
        L.bs_set_prefill_kernel(_lib.PREFILL_AUTO)
    w = IU.unpack_and_reconstruct_w_hip(q, u, vt).float()
    xf = x.float().reshape(T, N)
    want, size = torch.nn.functional.linear(xf, w, None if bias is None else bias.float()), torch.nn.functional.linear(xf.abs(), w.abs())
    # y is rounded to fp16 once (2^-11 of it, 2^-25 where it is subnormal); either side's fp32 sums of N products are off by up to N 2^-24 of the sum of their sizes
    bound = want.abs() * 2.0 ** -11 + 2.0 ** -25 + 2 * (N + 1) * 2.0 ** -24 * (size + (0 if bias is None else bias.float().abs()))
    assert bool(((y.float().reshape(T, M) - want).abs() <= bound).all())
