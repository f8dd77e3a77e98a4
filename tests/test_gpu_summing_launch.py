"""The summing launch four outputs at a time against one at a time (which an output off an 8-byte boundary takes): the same bits.  One to sixteen partial sums per
output, matrices side by side whose rows end inside a workgroup, every epilogue, with and without the RMS scale."""
import pytest
import torch

from bitstack_amd import _lib
from bitstack_amd.utils import inference_utils as IU
from bitstack_amd.utils.synthetic import synthetic_layer

pytestmark = pytest.mark.gpu


# (blocks, out features) of each matrix, in features, tokens
GROUPS = [([(2, 4100), (3, 1024), (1, 1500)], 4096, 40), ([(3, 14336), (2, 14336)], 1024, 16), ([(3, 14336), (2, 14336)], 1024, 40), ([(1, 28672)], 896, 5), ([(4, 4100)], 10240, 48), ([(3, 4096)], 14336, 37),
          ([(2, 4096)], 16384, 33), ([(9, 5000)], 4096, 48), ([(2, 12288)], 1408, 17), ([(8, 16388)], 2048, 8)]


@pytest.mark.parametrize("layers,N,T", GROUPS)
def test_four_at_a_time_gives_the_same_bits(layers, N, T):
    print(f"{layers} N={N} T={T}", flush=True)
    mats = []
    for j, (I, M) in enumerate(layers):
        q, u, vt, x = (t.cuda() for t in synthetic_layer(M, N, I, T, seed=I + M + N, signed_factors=True))
        mats.append((q, (u * 20).half(), vt, torch.randn(M, device="cuda").half() if j % 2 == 0 else None))
    x, grp = x.view(T, N), IU.MatrixGroup(mats)
    width = sum(M for _, M in layers)
    cases = [(_lib.EPI_NONE, width), (_lib.EPI_RESIDUAL, width)]
    if len(layers) == 2:
        cases.append((_lib.EPI_SWIGLU, layers[0][1]))
    for epilogue, w in cases:
        residual = torch.randn(T, w, device="cuda").half() if epilogue == _lib.EPI_RESIDUAL else None
        for eps in (None, 1e-5):
            room = torch.full((T * w + 2,), float("nan"), dtype=torch.float16, device="cuda")
            one = IU.bitstack_forward_group_hip(grp, x, epilogue, residual, out=room[2:].view(T, w), rms_eps=eps)
            room = torch.full((T * w + 8,), float("nan"), dtype=torch.float16, device="cuda")
            four = IU.bitstack_forward_group_hip(grp, x, epilogue, residual, out=room[4:-4].view(T, w), rms_eps=eps)
            assert one.data_ptr() % 8 == 4 and four.data_ptr() % 8 == 0
            assert bool(torch.isfinite(one).all()) and torch.equal(one, four), (epilogue, eps)
            assert bool(room[:4].isnan().all()) and bool(room[-4:].isnan().all())


@pytest.mark.parametrize("I,M,N,T", [(5, 14336, 4096, 100), (2, 12036, 1152, 128), (1, 2816, 4224, 127)])
def test_many_tokens(I, M, N, T):
    L = _lib.lib()
    q, u, vt, x = (t.cuda() for t in synthetic_layer(M, N, I, T, seed=I + M + N, signed_factors=True))
    bias = torch.randn(M + 4, device="cuda").half()
    need = L.bs_workspace_bytes(I, M, N, 16, T)
    ws = torch.empty(need, dtype=torch.uint8, device="cuda")
    got = []
    for at in (4, 2):                                    # halves: y and bias on an 8-byte boundary, and off it
        room = torch.full((T * M + 8,), float("nan"), dtype=torch.float16, device="cuda")
        y, b = room[at:at + T * M], torch.empty(M + 4, dtype=torch.float16, device="cuda")[at:at + M].copy_(bias[:M])
        _lib.check(L.bs_forward(q.data_ptr(), u.data_ptr(), vt.data_ptr(), x.data_ptr(), b.data_ptr(), y.data_ptr(), I, M, N, 16, T, ws.data_ptr(), need,
                                torch.cuda.current_stream().cuda_stream), "bs_forward")
        got.append(y.clone())
        assert bool(room[:at].isnan().all()) and bool(room[at + T * M:].isnan().all())
    assert bool(torch.isfinite(got[0]).all()) and torch.equal(got[0], got[1])
