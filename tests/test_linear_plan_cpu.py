"""bs_linear_plan names the k-step, and the partial last one, of the kernel that bs_linear_f16 runs; bs_dense_plan the tile, the parts and the stages of either dense product."""
import ctypes
import random

import pytest

from bitstack_amd import _lib

# tokens, out features, in features: tile, k-step, whether the last one is partial
PLANS = [
    # 64 x 64: linear_pipe_kernel's steps of 64, where N is a multiple of them
    (140, 1024, 4160, (64, 64, 64, 0)), (140, 1024, 4096, (64, 64, 64, 0)), (190, 5000, 2112, (64, 64, 64, 0)), (256, 6080, 3072, (64, 64, 64, 0)), (640, 3000, 1088, (64, 64, 64, 0)),
    # otherwise linear_f16_kernel's of 128
    (256, 6144, 4096, (64, 64, 128, 0)), (256, 6144, 4160, (64, 64, 128, 1)), (140, 1024, 4104, (64, 64, 128, 1)), (140, 6208, 3136, (64, 64, 128, 1)),
    # the larger tiles' and few tokens'
    (1024, 4096, 4160, (128, 128, 64, 0)), (512, 14336, 4096, (128, 256, 64, 0)), (2048, 14336, 4096, (256, 256, 64, 0)), (2048, 14336, 4128, (256, 256, 32, 0)),
    (64, 8192, 4160, (128, 64, 64, 0)), (64, 4096, 4160, (128, 32, 128, 1)), (8, 4096, 4096, (32, 16, 0, 0))]


@pytest.mark.parametrize("T,M,N,plan", PLANS)
def test_the_step_of_the_kernel_that_runs(T, M, N, plan):
    assert _lib.linear_plan(T, M, N) == plan


def test_the_kernel_of_the_small_tiles_is_the_faster_one():
    """Products timed on both kernels (us, linear_f16_kernel / linear_pipe_kernel)."""
    for dims in [(256, 5120, 2048), (256, 5120, 3072), (256, 5120, 8192), (140, 6144, 14336), (256, 6144, 3072), (256, 6656, 5120), (320, 5600, 5120),   # 17.4 / 19.4, 23.8 / 29.2, 54.5 / 63.8, 87.9 / 102.9, 25.3 / 29.6, 43.7 / 49.1, 43.0 / 48.1
                 (190, 7214, 4096), (160, 5870, 4096)]:                                                                                                   # 34.7 / 37.2, 29.3 / 32.3
        assert _lib.dense_plan(*dims) == (64, 64, 1, 0), dims
    for dims in [(256, 3000, 4096), (256, 4096, 8192), (190, 5000, 14336), (200, 7600, 4096), (320, 5152, 1792), (350, 3755, 1536), (140, 6144, 1024), (448, 4108, 4096)]:   # 24.5 / 20.6 ... 41.8 / 34.3
        assert _lib.dense_plan(*dims) == (64, 64, 1, 4), dims


def test_dense_plan_of_linear_f16_is_its_tile():
    for T, M, N, plan in PLANS:
        bt, bf, parts, stages = _lib.dense_plan(T, M, N)
        assert (bt, bf, parts) == plan[:2] + (1,)
        assert (stages >= 2) == (N % 64 == 0 and plan[2] == 64 and bt * bf != 128 * 64)      # (linear_f16_kernel has its tile of 128 x 64 in steps of 64 too)


def test_dense_plan_behind_a_rebuilt_weight_fits_the_scratch():
    rng, cut = random.Random(5), 0
    for _ in range(400):
        T, M, N = rng.randint(129, 4000), 8 * rng.randint(64, 3500), 128 * rng.randint(4, 200)
        bt, bf, parts, stages = _lib.dense_plan(T, M, N, rebuilt=True)
        assert stages in (2, 3, 4) and stages * (bt + bf) * 128 <= 160 << 10
        weight = (M * N * 2 + 255) // 256 * 256
        room = _lib.lib().bs_workspace_bytes(4, M, N, 16, T) - weight
        assert room >= (parts * T * M * 4 if parts > 1 else 0) and (parts > 1 or room == 0)
        cut += parts > 1
    assert 40 < cut < 360


def test_dense_plan_refuses_what_linear_plan_refuses():
    v = [ctypes.byref(ctypes.c_int()) for _ in range(4)]
    L = _lib.lib()
    assert L.bs_dense_plan(0, 64, 64, 0, *v) == L.bs_dense_plan(4, 0, 64, 1, *v) == L.bs_dense_plan(4, 64, -8, 1, *v) == -2
    assert L.bs_dense_plan(4, 64, 64, 0, None, *v[1:]) == L.bs_dense_plan(4, 64, 64, 1, *v[:3], None) == -1
    assert _lib.dense_plan(4, 64, 100) == _lib.dense_plan(4, 64, 100, rebuilt=True) == (0, 0, 1, 0)


# out of whole calls timed cut and in one piece (us, cut / in one): sums beyond what the cache holds, estimates that are level, and clear gains
IN_ONE = [(2515, 9480, 12800), (2247, 5080, 19712),                                                          # 597 / 540, 467 / 398
          (1722, 6936, 22272), (1362, 8824, 17408), (2056, 8200, 17536), (1130, 10592, 22400), (1497, 5768, 16256)]  # 585 / 493, 480 / 427, 638 / 567, 627 / 551, 311 / 268
CUT = [(1400, 4096, 14336), (509, 4096, 14336), (1017, 3248, 22528), (479, 3048, 28416), (706, 5344, 28032)]       # 186 / 211, 123 / 149, 173 / 249, 140 / 220, 266 / 340


def test_the_range_is_cut_where_that_was_faster():
    for dims in IN_ONE:
        assert _lib.dense_plan(*dims, rebuilt=True)[2] == 1, dims
    for dims in CUT:
        assert _lib.dense_plan(*dims, rebuilt=True)[2] > 1, dims


def test_the_tile_is_the_faster_one():
    """Whole calls timed on the tile that is not to be taken and on the one that is (us)."""
    for dims, other in [((2254, 4592, 2176), (256, 192)), ((3753, 2784, 3968), (256, 192)), ((687, 13264, 1920), (256, 192)),                  # 59.1 / 55.7, 93.7 / 88.6, 63.0 / 58.0
                        ((3120, 3188, 24576), (160, 128)), ((1324, 14438, 10368), (160, 128)), ((874, 10870, 4480), (160, 128)),              # 510 / 450, 536 / 465, 125 / 116
                        ((1994, 545, 9088), (64, 64)), ((1428, 1315, 14464), (64, 64)), ((313, 11067, 17664), (64, 128)), ((303, 11116, 15232), (64, 128))]:   # 62.2 / 52.6, 122 / 94, 356 / 302, 301 / 259
        assert _lib.dense_plan(*dims, rebuilt=True)[:2] != other, dims
    for dims in [(401, 8284, 1536), (404, 8240, 1920), (257, 11188, 3072)]:                                                                   # (shorter rows) 37.2 / 33.3, 39.2 / 36.3, 63.0 / 57.8
        assert _lib.dense_plan(*dims, rebuilt=True)[:2] == (64, 128), dims
