"""Groups of matrices of ranks 4 to 15 on the tile kernel: the same bits as rank 16 with factors of zero behind them, with the norm's sums and each epilogue, u on an address that is
only 8-byte aligned."""
import pytest
import torch

from bitstack_amd import _lib
from bitstack_amd.utils import inference_utils as IU
from bitstack_amd.utils.synthetic import synthetic_layer

# (blocks, out features) of the matrices, in features, tokens: one, two and three token tiles, partial row tiles, waves without columns, every width
GROUPS = [([(3, 8192), (2, 1024), (3, 1000)], 8192, 8), ([(6, 1100), (4, 1100)], 4096, 20), ([(2, 11008), (2, 11008)], 4096, 32), ([(5, 3000), (3, 500), (4, 77)], 2176, 40),
          ([(1, 28672), (5, 28672)], 1152, 16), ([(3, 2100), (2, 2100), (9, 2100), (1, 300)], 2048, 13)]


def test_the_groups_run_on_the_tile_kernel():
    for layers, N, T in GROUPS:
        taken = _lib.tile_kernel(layers, N, 16, T)
        assert taken[0] == _lib.TILE_FORWARD
        for K in (4, 6, 8, 11, 15):
            assert _lib.small_rank_kernel(layers, N, K, T) == taken, (layers, N, K, T)


@pytest.mark.gpu
@pytest.mark.parametrize("K", [4, 6, 8, 11, 15])
@pytest.mark.parametrize("layers,N,T", GROUPS)
def test_group_is_the_padded_one(layers, N, T, K):
    print(f"small rank group {layers} N={N} T={T} K={K}", flush=True)
    mats, padded = [], []
    for j, (I, M) in enumerate(layers):
        q, u, vt, x = (t.cuda() for t in synthetic_layer(M, N, I, T, k=K, seed=100 * j + K, signed_factors=True))
        bias = torch.randn(M, device="cuda").half()
        odd = torch.empty(u.numel() + 8, dtype=torch.half, device="cuda")[4:4 + u.numel()].view(u.shape).copy_(u * 20)
        assert odd.data_ptr() % 16 == 8
        pad_u, pad_vt = torch.zeros(I, M, 16, dtype=torch.half, device="cuda"), torch.zeros(I, 16, N, dtype=torch.half, device="cuda")
        pad_u[:, :, :K], pad_vt[:, :K] = odd, vt
        mats.append((q, odd, vt, bias))
        padded.append((q, pad_u, pad_vt, bias))
    group, want = IU.MatrixGroup(mats), IU.MatrixGroup(padded)
    residual = torch.randn(T, sum(M for _, M in layers), device="cuda").half()
    cases = [(_lib.EPI_NONE, None), (_lib.EPI_RESIDUAL, residual)] + ([(_lib.EPI_SWIGLU, None)] if len(layers) == 2 and layers[0][1] == layers[1][1] else [])
    for epilogue, more in cases:
        for eps in (None, 1e-5):
            y = IU.bitstack_forward_group_hip(want, x, epilogue, more, rms_eps=eps)
            assert bool(y.isfinite().all())
            assert torch.equal(IU.bitstack_forward_group_hip(group, x, epilogue, more, rms_eps=eps), y), (epilogue, eps)
