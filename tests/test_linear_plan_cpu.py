"""bs_linear_plan names the k-step, and the partial last one, of the kernel that bs_linear_f16 runs."""
import pytest

from bitstack_amd import _lib

# tokens, out features, in features: tile, k-step, whether the last one is partial
PLANS = [
    # 64 x 64: linear_pipe_kernel's steps of 64, where N is a multiple of them, up to 256 workgroups, beyond 384, and up to 3072 columns
    (140, 1024, 4160, (64, 64, 64, 0)), (140, 1024, 4096, (64, 64, 64, 0)), (190, 5000, 2112, (64, 64, 64, 0)), (256, 6144, 3072, (64, 64, 64, 0)), (640, 3000, 1088, (64, 64, 64, 0)),
    # otherwise linear_f16_kernel's of 128
    (256, 6144, 4096, (64, 64, 128, 0)), (256, 6144, 4160, (64, 64, 128, 1)), (140, 1024, 4104, (64, 64, 128, 1)), (140, 6208, 3136, (64, 64, 128, 1)),
    # the larger tiles' and few tokens'
    (1024, 4096, 4160, (128, 128, 64, 0)), (512, 14336, 4096, (128, 256, 64, 0)), (2048, 14336, 4096, (256, 256, 64, 0)), (2048, 14336, 4128, (256, 256, 32, 0)),
    (64, 8192, 4160, (128, 64, 64, 0)), (64, 4096, 4160, (128, 32, 128, 1)), (8, 4096, 4096, (32, 16, 0, 0))]


@pytest.mark.parametrize("T,M,N,plan", PLANS)
def test_the_step_of_the_kernel_that_runs(T, M, N, plan):
    assert _lib.linear_plan(T, M, N) == plan
