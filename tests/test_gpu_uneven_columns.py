"""Column counts that are multiples of 128 but not of 512 on the decode kernels (their last chunk is partial): one to four
tokens on every kernel that takes them, the last chunk holding one, two and three lane groups, rows that end a tile,
small ranks and a bias, against the float64 oracle."""
import numpy as np
import pytest
import torch

from bitstack_amd import _lib
from bitstack_amd.utils import inference_utils as IU
from bitstack_amd.utils.synthetic import synthetic_layer
from oracle import c_oracle as C

# (blocks, out features, in features, rank)
CASES = [(1, 16, 384, 16), (3, 130, 896, 16), (2, 512, 1152, 16), (4, 1000, 1664, 5), (2, 1024, 2176, 16), (5, 300, 1280, 16),
         (3, 4096, 11008, 16), (2, 2048, 5504, 7)]


def test_a_partial_chunk_is_taken_where_it_adds_at_most_a_third():
    L = _lib.lib()
    assert [n for n in range(128, 2049, 128) if L.bs_decode_kernel(2, 256, n, 16, 1) == 0] == [128, 256, 640]
    assert L.bs_decode_kernel(8, 4096, 11008, 16, 1) == _lib.DECODE_MX and L.bs_decode_kernel(1, 1024, 1152, 16, 1) == _lib.DECODE_F16


@pytest.mark.gpu
@pytest.mark.parametrize("T", [1, 2, 3, 4])
@pytest.mark.parametrize("I,M,N,K", CASES)
def test_decode_with_a_partial_last_chunk(I, M, N, K, T):
    print(f"uneven columns I={I} M={M} N={N} K={K} T={T}", flush=True)
    dev = torch.device("cuda")
    q, u, vt, x = synthetic_layer(M, N, I, T, k=K, seed=I + N + T, signed_factors=True)
    u = (u * 20).half()
    bias = (torch.randn(M, generator=torch.Generator().manual_seed(N)) * 0.05).half() if (I + T) % 2 else None
    want = C.forward_f64(q.numpy(), u.numpy(), vt.numpy(), x.numpy())
    if bias is not None:
        want = want + bias.numpy().astype(np.float64)
    args = (q.to(dev), u.to(dev), vt.to(dev), x.to(dev), None if bias is None else bias.to(dev))
    L = _lib.lib()
    for mode in (_lib.DECODE_AUTO, _lib.DECODE_F16) + ((_lib.DECODE_MX,) if T <= 2 else ()):
        _lib.check(L.bs_set_decode_kernel(mode), "bs_set_decode_kernel")
        try:
            assert L.bs_decode_kernel(I, M, N, K, T) == mode or mode == _lib.DECODE_AUTO
            y = IU.bitstack_forward_hip(*args)
            _lib.workspace(dev, 1).fill_(0xFF)
            assert torch.equal(IU.bitstack_forward_hip(*args), y)
        finally:
            L.bs_set_decode_kernel(_lib.DECODE_AUTO)
        d = np.abs(y.cpu().numpy().astype(np.float64) - want)
        assert d.max() <= 1e-2 * np.abs(want).max() and d.mean() <= 1e-3 * np.abs(want).mean(), (mode, d.max(), d.mean())
