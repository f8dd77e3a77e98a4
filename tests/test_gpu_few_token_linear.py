"""The dense product of up to 32 tokens (``linear_skinny_kernel``) at the edges of its lines, workgroups and token blocks, against float64."""
import pytest
import torch

from bitstack_amd import _lib
from bitstack_amd.utils import inference_utils as IU

# (tokens, out features, in features, features per workgroup): contracted ranges of less than a line, of fewer lines than waves, that end inside a
# line and inside its first half; features that fill no workgroup; each width of one
CASES = [(1, 1, 8, 16), (3, 17, 24, 16), (16, 33, 72, 16), (17, 100, 512, 16), (32, 5119, 1000, 16), (15, 5121, 456, 32), (17, 5120, 4104, 32), (32, 12287, 200, 32),
         (1, 12289, 520, 64), (16, 12300, 1032, 64), (17, 12288, 576, 64), (31, 32003, 40, 64), (8, 4096, 6136, 16), (2, 3, 65528, 16)]


@pytest.mark.gpu
@pytest.mark.parametrize("T,M,N,features", CASES)
def test_few_tokens_match_float64(T, M, N, features):
    print(f"few tokens T={T} M={M} N={N}", flush=True)
    assert _lib.linear_plan(T, M, N) == (32, features, 0, 0)
    g = torch.Generator(device="cuda").manual_seed(T + M + N)
    x = torch.randn(T, N, device="cuda", generator=g).half()
    w = torch.randn(M, N, device="cuda", generator=g).half()
    bias = torch.randn(M, device="cuda", generator=g).half() if T % 2 else None
    if M > 1:
        w[1, 0] = float("inf")                       # behind the last column of row 0
    y = IU.linear_f16_hip(x, w, bias).double()
    want, size = x.double() @ w.double().t(), x.double().abs() @ w.double().abs().t()
    if bias is not None:
        want, size = want + bias.double(), size + bias.double().abs()
    if M > 1:
        assert not torch.isfinite(y[:, 1]).any()
        y[:, 1] = want[:, 1] = size[:, 1] = 0
    # N products added in float32 (2^-24 of the sum of magnitudes each, in whatever order), rounded once
    bound = want.abs() * 2.0 ** -11 + size * (N + 9) * 2.0 ** -24 + 2.0 ** -25
    assert ((y - want).abs() <= bound).all()


# both sides of every change of width: one round of 256 workgroups of 16 features, rounds of 32 against rounds of 64
ROUNDS = [(5, 4096, 1032, 16), (8, 4097, 1032, 32), (32, 5119, 1096, 32), (3, 8192, 1024, 32), (3, 8193, 1024, 64), (20, 16384, 1032, 64), (20, 16385, 1032, 32),
          (1, 24577, 1024, 64), (16, 32769, 1024, 32), (17, 4097, 952, 32), (32, 4096, 952, 16)]


def test_a_round_that_is_nearly_empty_is_avoided():
    """A few rows more than a round holds take no second one where a wider workgroup needs none."""
    for T, M, N, features in ROUNDS:
        assert _lib.linear_plan(T, M, N) == (32, features, 0, 0), (T, M, N)
    for T in (1, 8, 17, 32):
        for M in (4189, 5000, 8192, 8400, 12287, 13000, 16384):
            assert -(-M // _lib.linear_plan(T, M, 4096)[1]) <= 256, (T, M)


@pytest.mark.gpu
@pytest.mark.parametrize("T,M,N,features", ROUNDS)
def test_either_side_of_a_change_of_width(T, M, N, features):
    test_few_tokens_match_float64(T, M, N, features)
