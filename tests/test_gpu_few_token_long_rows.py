"""The dense product of up to 32 tokens on rows of about 32 lines and more, 64 and 32 features to a workgroup, with and without a partial last line, against float64."""
import pytest

from test_gpu_few_token_linear import test_few_tokens_match_float64 as match_float64

CASES = [(1, 12289, 2040, 64), (8, 16000, 4104, 64), (16, 12300, 1984, 64), (16, 16000, 2112, 64), (17, 12800, 4104, 64), (32, 12801, 2040, 64), (32, 16000, 8192, 64), (9, 5120, 4104, 32), (31, 5121, 1992, 32)]


@pytest.mark.gpu
@pytest.mark.parametrize("T,M,N,features", CASES)
def test_long_rows(T, M, N, features):
    match_float64(T, M, N, features)
