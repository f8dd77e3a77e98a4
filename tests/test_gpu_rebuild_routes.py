"""One weight whatever it is made from and by: the rank-16 tile kernel (``tile.hip``) for packed signs, the strip-wise kernel (``reconstruct.hip``) for int8
signs and for factors the tile kernel cannot read, bit for bit; and the same sum in float64 within one rounding."""
import numpy as np
import pytest
import torch

from bitstack_amd import _lib
from bitstack_amd.utils import inference_utils as IU
from bitstack_amd.utils import pack_utils as PU
from bitstack_amd.utils.synthetic import synthetic_layer
from oracle import bitstack_oracle as O

pytestmark = pytest.mark.gpu


# blocks and widths of every kind of group the tile kernel has, last rows and columns that fill no tile, runs of one tile; and shapes it declines
@pytest.mark.parametrize("I,M,N,taken", [(8, 1025, 4096, True), (3, 6144, 1408, True), (4, 4000, 2176, True), (1, 14336, 1024, False), (1, 14336, 4096, True), (16, 3001, 1152, True), (10, 3333, 2048, True),
                                         (2, 10743, 896, False), (2, 100, 128, False)])
def test_same_weight_by_every_route(I, M, N, taken):
    print(f"I={I} M={M} N={N}", flush=True)
    q, u, vt, _ = synthetic_layer(M, N, I, 1, seed=I + M, signed_factors=True)
    u, vt = (u * 20).half(), (vt * 20).half()
    assert (_lib.tile_kernel([(I, M)], N, 16, 4096)[0] == _lib.TILE_REBUILD) == taken
    qd, ud, vd = q.cuda(), u.cuda(), vt.cuda()
    w = IU.unpack_and_reconstruct_w_hip(qd, ud, vd)
    sign = torch.stack([PU.unpack_sign_hip(qd[i], torch.Size([M, N])) for i in range(I)])
    assert torch.equal(w.view(torch.int16), IU.reconstruct_w_hip(sign, ud, vd).view(torch.int16))
    # u on 8 bytes only: the strip-wise kernel, from packed signs
    room = torch.empty(ud.numel() + 4, dtype=torch.float16, device="cuda")
    shifted = room[4:].view_as(ud).copy_(ud)
    assert shifted.data_ptr() % 16 == 8
    assert torch.equal(w.view(torch.int16), IU.unpack_and_reconstruct_w_hip(qd, shifted, vd).view(torch.int16))
    exact = O.reconstruct_w_exact(q.numpy(), u.numpy(), vt.numpy())
    # half a step of the result, and 16 I sums in fp32 whose terms are at most the sum of their sizes
    size = sum(np.abs(u[i].double().numpy()) @ np.abs(vt[i].double().numpy()) for i in range(I))
    assert np.all(np.abs(w.cpu().double().numpy() - exact) <= np.spacing(np.abs(exact).astype(np.float16)).astype(np.float64) / 2 * 1.001 + 16 * I * 2.0 ** -23 * size)
