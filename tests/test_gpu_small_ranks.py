"""Ranks 4 to 15 on the tile and column kernels: the same bits as rank 16 with factors of zero behind them, whichever halves the pieces of a u row start at, and
nothing read from beyond the factors."""
import pytest
import torch

from bitstack_amd import _lib
from bitstack_amd.utils import inference_utils as IU
from bitstack_amd.utils import pack_utils as PU
from bitstack_amd.utils.synthetic import synthetic_layer

# blocks, out features, in features, tokens: every width and token tile of the tile kernel, whole and partial tiles and column groups, waves without columns; the column kernel
FORWARD = [(3, 1, 384, 5), (5, 65, 1152, 8), (2, 8200, 1152, 8), (3, 33, 256, 17), (4, 100, 640, 33), (10, 70, 640, 47), (2, 16400, 2048, 20), (16, 65, 1280, 12), (7, 4100, 3072, 48)]
FROM_8 = [(3, 1, 384, 5), (3, 33, 256, 17)]          # one tile of three blocks: the strip kernel's below rank 8
COLUMN = [(6, 2817, 4224, 50), (1, 20737, 640, 128), (8, 2815, 4352, 64), (3, 2850, 4096, 100)]
REBUILD = [(8, 1025, 4096), (3, 6144, 1408), (4, 4000, 2176), (16, 3001, 1152)]


def test_the_cases_reach_their_kernels():
    for cases, kind in ((FORWARD, _lib.TILE_FORWARD), (COLUMN, _lib.TILE_COLUMN), ([c + (4096,) for c in REBUILD], _lib.TILE_REBUILD)):
        for I, M, N, T in cases:
            taken = _lib.tile_kernel([(I, M)], N, 16, T)
            assert taken[0] == kind
            for K in range(1, 17):
                assert _lib.small_rank_kernel([(I, M)], N, K, T) == (taken if (8 if (I, M, N, T) in FROM_8 else 4) <= K < 16 else (_lib.TILE_NONE, [0])), (I, M, N, T, K)


def factors(I, M, N, T, K):
    """Signs, factors of rank K with NaN on both sides of them in memory, the same padded to rank 16, x."""
    q, u, vt, x = (t.cuda() for t in synthetic_layer(M, N, I, T, k=K, seed=I + M + K, signed_factors=True))
    u = (u * 20).half()

    def between_nans(t):
        room = torch.full((t.numel() + 128,), float("nan"), dtype=t.dtype, device="cuda")
        return room[64:64 + t.numel()].view(t.shape).copy_(t)

    pad_u, pad_vt = torch.zeros(I, M, 16, dtype=torch.half, device="cuda"), torch.zeros(I, 16, N, dtype=torch.half, device="cuda")
    pad_u[:, :, :K], pad_vt[:, :K] = u, vt
    return q, between_nans(u), between_nans(vt), pad_u, pad_vt, x


@pytest.mark.gpu
@pytest.mark.parametrize("I,M,N,T,K", [c + (K,) for c in FORWARD + COLUMN for K in (4, 5, 6, 7, 8, 9, 11, 12, 15) if K >= 8 or c not in FROM_8])
def test_forward_is_the_padded_one(I, M, N, T, K):
    print(f"ranks I={I} M={M} N={N} T={T} K={K}", flush=True)
    q, u, vt, pad_u, pad_vt, x = factors(I, M, N, T, K)
    bias = torch.randn(M, device="cuda").half()
    want = IU.bitstack_forward_hip(q, pad_u, pad_vt, x, bias)
    assert bool(want.isfinite().all())
    assert torch.equal(IU.bitstack_forward_hip(q, u, vt, x, bias), want)


@pytest.mark.gpu
@pytest.mark.parametrize("I,M,N", REBUILD)
@pytest.mark.parametrize("K", [4, 5, 7, 8, 10, 13, 14, 15])
def test_rebuild_is_the_padded_one_from_either_kind_of_signs(I, M, N, K):
    print(f"ranks I={I} M={M} N={N} K={K}", flush=True)
    q, u, vt, pad_u, pad_vt, _ = factors(I, M, N, 1, K)
    want = IU.unpack_and_reconstruct_w_hip(q, pad_u, pad_vt)
    assert torch.equal(IU.unpack_and_reconstruct_w_hip(q, u, vt).view(torch.int16), want.view(torch.int16))
    sign = torch.stack([PU.unpack_sign_hip(q[i], torch.Size([M, N])) for i in range(I)])
    assert torch.equal(IU.reconstruct_w_hip(sign, u, vt).view(torch.int16), want.view(torch.int16))


@pytest.mark.gpu
@pytest.mark.parametrize("K", [4, 7, 8, 11])
@pytest.mark.parametrize("T", [8, 40, 64])
def test_rows_that_are_not_finite(T, K):
    N, shapes = (640, [(3, 100), (2, 4100)]) if T < 49 else (4224, [(3, 2817)])
    for I, M in shapes:
        q, u, vt, _, _, x = factors(I, M, N, T, K)
        clean = IU.bitstack_forward_hip(q, u, vt, x, None).view(T, M)
        for row in (0, 37, M - 1):
            for rank in {0, min(7, K - 1), min(8, K - 1), K - 1}:
                bad = u.clone()
                bad[I - 1, row, rank] = float("inf")
                y = IU.bitstack_forward_hip(q, bad, vt, x, None).view(T, M)
                keep = torch.arange(M, device="cuda") != row
                assert not bool(y[:, row].isfinite().any()) and torch.equal(y[:, keep], clean[:, keep]), (row, rank)
