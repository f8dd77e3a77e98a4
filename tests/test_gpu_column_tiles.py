"""The column kernel at every number of token tiles: what a token gets does not depend on how many others there are, bit for bit (the columns are
dealt and summed by the matrix's sizes alone)."""
import pytest
import torch

from bitstack_amd import _lib
from bitstack_amd.utils import inference_utils as IU
from bitstack_amd.utils.synthetic import synthetic_layer

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("I,M,N", [(6, 2817, 4224), (1, 20737, 640)])
def test_tokens_do_not_depend_on_their_number(I, M, N):
    q, u, vt, x = (t.cuda() for t in synthetic_layer(M, N, I, 128, seed=I + N, signed_factors=True))
    u, x = (u * 20).half(), x.view(128, N)
    bias = torch.randn(M, device="cuda").half()
    assert _lib.tile_kernel([(I, M)], N, 16, 128)[0] == _lib.TILE_COLUMN
    whole = IU.bitstack_forward_hip(q, u, vt, x, bias).view(128, M)
    for T in (49, 64, 65, 79, 80, 81, 96, 97, 111, 112, 113, 127):
        assert _lib.tile_kernel([(I, M)], N, 16, T)[0] == _lib.TILE_COLUMN
        assert torch.equal(IU.bitstack_forward_hip(q, u, vt, x[:T].contiguous(), bias).view(T, M), whole[:T]), T


def test_seven_blocks_up_to_six_token_tiles():
    """Seven blocks are taken up to 96 tokens, on four, five and six token tiles (six: held to float64 with the tile kernel's tests)."""
    I, M, N = 7, 2815, 4352
    q, u, vt, x = (t.cuda() for t in synthetic_layer(M, N, I, 96, seed=I + N, signed_factors=True))
    u, x = (u * 20).half(), x.view(96, N)
    whole = IU.bitstack_forward_hip(q, u, vt, x, None).view(96, M)
    for T in (50, 64, 65, 79, 80, 81):
        assert _lib.tile_kernel([(I, M)], N, 16, T)[0] == _lib.TILE_COLUMN
        assert torch.equal(IU.bitstack_forward_hip(q, u, vt, x[:T].contiguous(), None).view(T, M), whole[:T]), T
