"""Equal rows of one dense product have equal outputs, wherever they lie: words that share a row of the weight get the same logit, and a token that occurs twice in a call gets the same
result twice."""
import pytest
import torch

from bitstack_amd import _lib
from bitstack_amd.utils import inference_utils as IU

# tokens, out features, in features, the tile: every width of the few-token kernel, one and two blocks of tokens, rows of more than 32 lines
FEW = [(8, 4096, 4096, (32, 16)), (8, 5120, 4096, (32, 32)), (3, 16000, 2048, (32, 64)), (16, 12800, 4104, (32, 64)), (24, 4000, 6152, (32, 16)), (32, 5120, 4096, (32, 32)), (17, 12801, 2056, (32, 64))]
# several tiles of tokens and of features on every XCD, up to 512 tokens on 16 Mi weights and more: 128 x 128 with one and two workgroups per CU, 128 x 256, 256 x 256, 64 x 64
MORE = [(300, 8192, 4096, (128, 128)), (512, 8704, 2048, (128, 128)), (500, 14336, 2048, (128, 256)), (512, 20500, 1024, (256, 256)), (140, 5000, 4096, (64, 64))]
CASES = FEW + MORE


@pytest.mark.gpu
@pytest.mark.parametrize("T,M,N,tile", CASES)
def test_equal_rows_have_equal_outputs(T, M, N, tile):
    print(f"equal rows T={T} M={M} N={N}", flush=True)
    assert _lib.linear_plan(T, M, N)[:2] == tile
    g = torch.Generator(device="cuda").manual_seed(T + M + N)
    kinds, rows = (T + 1) // 2, 7 * M // 16 + 3     # (many different outputs: a sum in another order seldom rounds to another fp16 number)
    x = torch.randn(kinds, N, device="cuda", generator=g).half()[torch.arange(T, device="cuda") % kinds].contiguous()
    w = torch.randn(rows, N, device="cuda", generator=g).half()[torch.arange(M, device="cuda") % rows].contiguous()
    y = IU.linear_f16_hip(x, w, None)
    assert torch.equal(y, y[torch.arange(T, device="cuda") % kinds][:, torch.arange(M, device="cuda") % rows])
