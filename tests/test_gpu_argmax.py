"""The greedy token and the next position in one launch: rows around the number of values a workgroup asks for at a time."""
import numpy as np
import pytest
import torch

from bitstack_amd import _lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,V", [(1, 7), (1, 8), (2, 8192), (1, 8200), (1, 32767), (3, 32768), (2, 32776), (1, 65541)])
def test_argmax_and_advance(B, V):
    x = torch.randn(B, V, generator=torch.Generator().manual_seed(V)).half()
    for at in (0, V // 2, V - 1):                       # the largest value there and, a lower index, nowhere else
        y = x.clone()
        y[:, at] = 60000.0
        out, pos = torch.full((B,), -1, dtype=torch.int64, device="cuda"), torch.tensor(41, device="cuda")
        assert _lib.host().argmax(y.cuda(), out, pos)
        assert out.tolist() == [at] * B and int(pos) == 42
        assert _lib.host().argmax(x.cuda(), out) and int(pos) == 42
        assert out.tolist() == [int(np.argmax(r)) for r in x.float().numpy()]
    assert _lib.host().argmax(x.cuda(), out, torch.zeros(2, dtype=torch.int64, device="cuda")) is None
    assert _lib.host().argmax(x.cuda(), out, torch.zeros(1, dtype=torch.int32, device="cuda")) is None
