"""The large tiles of the dense product behind a rebuilt weight (gemm_pipe.hip) where they can go wrong: ragged tokens and
features, an odd number of k-steps, features that are no multiple of 8 (outputs through LDS), the contracted range in
parts (the last one shorter), against torch's fp16 product of the same rebuilt weight."""
import pytest
import torch

from bitstack_amd import _lib
from bitstack_amd.utils import inference_utils as IU
from bitstack_amd.utils.synthetic import synthetic_layer

# (tokens, out features, in features, parts are expected)
CASES = [(130, 4104, 8256, True), (20, 4104, 8256, True), (509, 4096, 14336, True), (2049, 4096, 8256, None),
         (1400, 14336, 4096, False), (900, 5120, 5120, False), (1400, 4096, 4096, False), (1399, 4091, 4160, False),
         (700, 3000, 2560, False), (259, 20001, 576, False), (5000, 7169, 192, False)]


def test_scratch_for_parts_follows_the_shape():
    L = _lib.lib()
    for T, M, N, parts in CASES:
        extra = int(L.bs_workspace_bytes(9, M, N, 16, T)) - (M * N * 2 + 255) // 256 * 256
        assert 0 <= extra <= M * N * 2 + 256
        if parts is not None:
            assert (extra > 0) == parts, (T, M, N, extra)


@pytest.mark.gpu
@pytest.mark.parametrize("T,M,N,parts", CASES)
def test_product_behind_the_rebuild(T, M, N, parts):
    print(f"dense pipe T={T} M={M} N={N}", flush=True)
    dev = torch.device("cuda")
    q, u, vt, x = synthetic_layer(M, N, 9, T, seed=T + M, device=dev, signed_factors=True)
    u = (u * 20).half()
    bias = (torch.randn(M, generator=torch.Generator().manual_seed(T)) * 0.05).half().to(dev) if T % 2 else None
    L = _lib.lib()
    assert int(L.bs_forward_path(9, M, N, 16, T)) == _lib.PATH_REBUILD or T < 97
    _lib.check(L.bs_set_prefill_kernel(_lib.PREFILL_REBUILD), "bs_set_prefill_kernel")
    try:
        y = IU.bitstack_forward_hip(q, u, vt, x, bias)
        ws = _lib.workspace(dev, int(L.bs_workspace_bytes(9, M, N, 16, T)))
        ws.fill_(0xFF)                                    # NaN in every partial sum that would not be written
        assert torch.equal(IU.bitstack_forward_hip(q, u, vt, x, bias), y)
    finally:
        L.bs_set_prefill_kernel(_lib.PREFILL_AUTO)
    want = torch.nn.functional.linear(x.float(), IU.unpack_and_reconstruct_w_hip(q, u, vt).float(), None if bias is None else bias.float())
    d = (y.float() - want).abs()
    assert float(d.max()) <= 2e-3 * float(want.abs().max()) and float(d.mean()) <= 5e-4 * float(want.abs().mean())
