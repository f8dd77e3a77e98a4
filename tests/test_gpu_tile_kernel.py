"""The tile kernel (rank 16, one to 48 tokens) at the edges of its tiles, against the float64 oracle and against the strip kernel, which
takes the same call when u lies 8 bytes off a 16-byte boundary."""
import ctypes
import os
import re
import shutil
import subprocess

import numpy as np
import pytest
import torch

from bitstack_amd import _lib
from bitstack_amd.utils import inference_utils as IU
from bitstack_amd.utils.synthetic import synthetic_layer
from oracle import c_oracle as C

CSRC = os.path.join(os.path.dirname(_lib.LIB_PATH))
# (blocks, out features, in features, tokens): rows about whole tiles of 32, columns that leave waves without any, both sides of the block
# limits of 1024, 512 and 256 columns per workgroup, whole and partial column groups of each, one, two and three token tiles
CASES = [(3, 1, 384, 5), (5, 1, 128, 16), (3, 32, 128, 16), (3, 33, 256, 17), (3, 31, 384, 48), (3, 64, 640, 1), (4, 100, 640, 33), (5, 65, 1152, 8), (2, 8200, 1152, 8),
         (3, 8224, 2176, 7), (4, 8191, 1024, 6), (1, 16400, 640, 40), (2, 8193, 1664, 32), (7, 130, 896, 16), (8, 200, 512, 9), (8, 97, 640, 33),
         (9, 256, 768, 8), (10, 70, 640, 47), (10, 128, 1024, 40), (13, 300, 384, 5), (15, 129, 1024, 24), (16, 33, 384, 16), (16, 65, 1280, 1),
         (1, 1892, 2176, 16), (1, 4183, 1024, 20), (2, 16400, 2048, 20), (1, 5877, 640, 2), (4, 8300, 2176, 16), (1, 3334, 1152, 48), (1, 16385, 1280, 48), (7, 4100, 3072, 48)]


def _runs_on(kind, layers, N, T):
    """The columns per workgroup of each matrix, of a call that has to run on `kind` of the tile kernel."""
    got, columns = _lib.tile_kernel(layers, N, 16, T)
    assert got == kind, (layers, N, T, got)
    return columns


def test_the_cases_reach_every_width():
    """Which kernel a call runs on follows from its sizes: every list below reaches what it is there for."""
    reached = {(_runs_on(_lib.TILE_FORWARD, [c[:2]], c[2], c[3])[0], (c[3] + 15) // 16) for c in CASES}
    assert reached == {(w, tt) for w in (1024, 512, 256) for tt in (1, 2, 3)}
    whole = {(w[0], c[2] % w[0] == 0) for c in CASES for w in [_runs_on(_lib.TILE_FORWARD, [c[:2]], c[2], c[3])]}
    assert whole == {(w, f) for w in (1024, 512, 256) for f in (False, True)}
    assert {(w[0], c[2] % w[0] == 0) for c in REBUILDS for w in [_runs_on(_lib.TILE_REBUILD, [c[:2]], c[2], 130)]} == whole
    for T in (3, 4):
        for cases in (TWO_TERMS, LARGE_WEIGHTS, EVERY_SIZE):
            assert {_runs_on(_lib.TILE_TWO_TERMS, [c[:2]], c[2], T)[0] for c in cases} == {1024, 512, 256}
        for cases in (TWO_TERM_GROUPS,):
            assert {w for layers, N in cases for w in _runs_on(_lib.TILE_TWO_TERMS, layers, N, T)} == {1024, 512, 256}
    for c in COLUMNS:
        _runs_on(_lib.TILE_COLUMN, [c[:2]], c[2], c[3])


def _args(I, M, N, T, off):
    """Inputs on the GPU; `off`: u starts 8 bytes off a 16-byte boundary."""
    q, u, vt, x = synthetic_layer(M, N, I, T, seed=I + N + T, signed_factors=True)
    u = (u * 20).half()
    want = C.forward_f64(q.numpy(), u.numpy(), vt.numpy(), x.numpy())
    q, u, vt, x = (t.cuda() for t in (q, u, vt, x))
    if off:
        room = torch.empty(u.numel() + 4, dtype=u.dtype, device="cuda")
        room[4:] = u.flatten()
        u = room[4:].view(u.shape)
        assert u.data_ptr() % 16 == 8
    return (q, u, vt, x, None), want


@pytest.mark.gpu
@pytest.mark.parametrize("I,M,N,T", CASES)
def test_edges(I, M, N, T):
    print(f"tile kernel I={I} M={M} N={N} T={T}", flush=True)
    _runs_on(_lib.TILE_FORWARD, [(I, M)], N, T)
    args, want = _args(I, M, N, T, False)
    y = IU.bitstack_forward_hip(*args)
    _lib.workspace(torch.device("cuda"), 1).fill_(0xFF)          # nothing is read from scratch that the call has not written
    assert torch.equal(IU.bitstack_forward_hip(*args), y)
    d = np.abs(y.cpu().numpy().astype(np.float64) - want)
    assert d.max() <= 1e-2 * np.abs(want).max() and d.mean() <= 1e-3 * np.abs(want).mean(), (d.max(), d.mean())
    other = IU.bitstack_forward_hip(*_args(I, M, N, T, True)[0])
    # The same weights in fp32, their blocks added in the same order, and rounded to fp16 (2^-11 of a weight where the two sums straddle a
    # rounding boundary, for few of them), then fp32 sums over the columns in another order and one rounding to fp16 each.
    w = IU.unpack_and_reconstruct_w_hip(*args[:3])
    size = torch.matmul(args[3].double().abs(), w.double().abs().t().contiguous())
    assert bool(((y.double() - other.double()).abs() <= y.double().abs() * 2.0 ** -10 + size * 2.0 ** -12).all())


@pytest.mark.gpu
@pytest.mark.parametrize("T", [1, 8, 20, 40])
def test_non_finite_inputs(T):
    """An infinity or NaN in u, vt or x reaches the outputs it has a part in and no others."""
    I, M, N = 3, 100, 640
    (q, u, vt, x, _), _ = _args(I, M, N, T, False)
    clean = IU.bitstack_forward_hip(q, u, vt, x, None)
    for value in (float("inf"), float("nan")):
        bad = u.clone()
        bad[1, 37, 3] = value
        y = IU.bitstack_forward_hip(q, bad, vt, x, None)
        assert not torch.isfinite(y[..., 37]).any()
        keep = torch.arange(M, device="cuda") != 37
        assert torch.equal(y[..., keep], clean[..., keep])
        bad = x.clone()
        bad.view(T, N)[T - 1, 130] = value
        y = IU.bitstack_forward_hip(q, u, vt, bad, None).view(T, M)
        assert not torch.isfinite(y[T - 1]).any() and torch.equal(y[:T - 1], clean.view(T, M)[:T - 1])
        bad = vt.clone()
        bad[2, 5, 200] = value
        assert not torch.isfinite(IU.bitstack_forward_hip(q, u, bad, x, None)).any()


@pytest.mark.gpu
@pytest.mark.parametrize("T", [8, 40])
@pytest.mark.parametrize("N", [1024, 2176])
def test_groups_of_unlike_matrices_are_the_single_calls(N, T):
    """Matrices of other heights and block counts in one launch: what each computes alone, up to the order of the column groups' sums."""
    L = _lib.lib()
    layers = [(1, 700), (8, 33), (3, 1000), (5, 64)]
    _runs_on(_lib.TILE_FORWARD, layers, N, T)
    x = synthetic_layer(8, N, 1, T, seed=3)[3].cuda()
    mats = (_lib.bs_matrix * len(layers))()
    keep, alone = [], []
    for j, (I, M) in enumerate(layers):
        q, u, vt, _ = (t.cuda() for t in synthetic_layer(M, N, I, T, seed=j, signed_factors=True))
        keep.append((q, u, vt))
        mats[j] = _lib.bs_matrix(q.data_ptr(), u.data_ptr(), vt.data_ptr(), None, I, M)
        alone.append((IU.bitstack_forward_hip(q, u, vt, x, None).view(T, M), IU.unpack_and_reconstruct_w_hip(q, u, vt)))
    rows = sum(M for _, M in layers)
    y = torch.empty(T, rows, dtype=torch.half, device="cuda")
    need = L.bs_forward_group_workspace_bytes(ctypes.byref(mats), len(layers), N, 16, T)
    ws = torch.full((need,), 0xFF, dtype=torch.uint8, device="cuda")
    _lib.check(L.bs_forward_group(ctypes.byref(mats), len(layers), N, 16, x.data_ptr(), T, 0, None, y.data_ptr(), ws.data_ptr(), need,
                                  torch.cuda.current_stream().cuda_stream), "bs_forward_group")
    at = 0
    for (I, M), (ref, w) in zip(layers, alone):
        part = y[:, at:at + M].double()
        at += M
        size = torch.matmul(x.double().view(T, N).abs(), w.double().abs().t().contiguous())
        assert bool(((part - ref.double()).abs() <= ref.double().abs() * 2.0 ** -10 + size * 2.0 ** -13).all()), (I, M)


@pytest.mark.skipif(not os.path.exists(shutil.which("hipcc") or "/opt/rocm/bin/hipcc"), reason="hipcc not available")
@pytest.mark.parametrize("source", ["tile.hip", "column.hip"])
def test_the_tile_kernels_keep_everything_in_registers(source, tmp_path):
    asm = tmp_path / "k.s"
    subprocess.run([shutil.which("hipcc") or "/opt/rocm/bin/hipcc", "--offload-arch=gfx950", "-O3", "-std=c++17", "-Xclang", "-target-feature", "-Xclang",
                    "-packed-fp32-ops", "-S", "--cuda-device-only", os.path.join(CSRC, source), "-o", str(asm)], check=True, capture_output=True)
    sizes = re.findall(r"\.private_segment_fixed_size:\s+(\d+)", asm.read_text())
    assert sizes and set(sizes) == {"0"}, sizes


# rows about whole tiles, whole and partial column groups of each width, block counts on both sides of the widths' limits, runs of one and of many tiles
REBUILDS = [(1, 11601, 1152), (2, 8200, 1152), (3, 20000, 384), (4, 8193, 2176), (5, 4100, 1664), (8, 9000, 1024), (13, 33, 128), (11, 9000, 768), (16, 1000, 1280),
            (16, 31, 256), (1, 8257, 2048), (1, 4183, 2048)]


@pytest.mark.gpu
@pytest.mark.parametrize("I,M,N", REBUILDS)
def test_rebuilt_weight(I, M, N):
    print(f"rebuild I={I} M={M} N={N}", flush=True)
    (q, u, vt, _, _), _ = _args(I, M, N, 1, False)
    # a forward of more than 128 tokens leaves it at the start of its scratch
    L, T = _lib.lib(), 130
    x, y = torch.ones(T, N, dtype=torch.half, device="cuda"), torch.empty(T, M, dtype=torch.half, device="cuda")
    need = L.bs_workspace_bytes(I, M, N, 16, T)
    assert L.bs_forward_path(I, M, N, 16, T) == _lib.PATH_REBUILD and need >= M * N * 2
    _runs_on(_lib.TILE_REBUILD, [(I, M)], N, T)
    guard = torch.full((need // 2 + 64,), 7.0, dtype=torch.half, device="cuda")
    _lib.check(L.bs_forward(q.data_ptr(), u.data_ptr(), vt.data_ptr(), x.data_ptr(), None, y.data_ptr(), I, M, N, 16, T, guard.data_ptr(), need,
                            torch.cuda.current_stream().cuda_stream), "bs_forward")
    assert bool((guard[need // 2:] == 7.0).all())
    w = guard[:M * N].view(M, N)
    # float64 from the same factors: I fp32 additions of sums of 16 exact products, and one rounding to fp16
    sign = ((q.view(I, M, N // 8, 1) >> torch.arange(7, -1, -1, device="cuda", dtype=torch.uint8)) & 1).reshape(I, M, N)
    want = torch.zeros(M, N, dtype=torch.float64, device="cuda")
    size = torch.zeros_like(want)
    for i in range(I):
        p = u[i].double() @ vt[i].double()
        want += torch.where(sign[i].bool(), p, -p)
        size += u[i].double().abs() @ vt[i].double().abs()
    assert bool(((w.double() - want).abs() <= want.abs() * 2.0 ** -11 + size * (I + 16) * 2.0 ** -24 + 2.0 ** -25).all())


@pytest.mark.gpu
def test_rebuilt_weights_of_several_matrices_in_one_launch():
    """bs_forward_cat rebuilds its matrices together: the rows of each are what the matrix gives alone."""
    L = _lib.lib()
    N, T, layers = 1024, 200, [(3, 4100), (6, 700), (1, 1300)]
    x = synthetic_layer(8, N, 1, T, seed=3)[3].cuda()
    mats, keep = (_lib.bs_matrix * len(layers))(), []
    for j, (I, M) in enumerate(layers):
        keep.append([t.cuda() for t in synthetic_layer(M, N, I, T, seed=j, signed_factors=True)[:3]])
        mats[j] = _lib.bs_matrix(*(t.data_ptr() for t in keep[-1]), None, I, M)
    need = L.bs_forward_cat_workspace_bytes(ctypes.byref(mats), len(layers), N, 16, T)
    assert need > 0
    _runs_on(_lib.TILE_REBUILD, layers, N, T)
    rows = sum(M for _, M in layers)
    ws = torch.full((need,), 0xFF, dtype=torch.uint8, device="cuda")
    y = torch.empty(T, rows, dtype=torch.half, device="cuda")
    _lib.check(L.bs_forward_cat(ctypes.byref(mats), len(layers), N, 16, x.data_ptr(), T, y.data_ptr(), ws.data_ptr(), need,
                                torch.cuda.current_stream().cuda_stream), "bs_forward_cat")
    w = ws[:rows * N * 2].view(torch.half).view(rows, N)
    at = 0
    for (I, M), (q, u, vt) in zip(layers, keep):
        alone = IU.unpack_and_reconstruct_w_hip(q, u, vt)
        # the same products added up in the same order, once by the matrix instruction and once behind it: a weight's rounding apart, rarely
        d = (w[at:at + M].double() - alone.double()).abs()
        assert bool((d <= alone.double().abs() * 2.0 ** -10 + 2.0 ** -23).all()) and float((d > 0).double().mean()) < 1e-2
        at += M


# (blocks, out features, in features) at three and four tokens: each width, whole and partial column groups, rows about whole tiles
TWO_TERMS = [(2, 8300, 512), (3, 4100, 1024), (4, 4163, 512), (5, 2081, 1536), (2, 3735, 3584), (2, 12993, 1024), (10, 3001, 512), (12, 4096, 512), (16, 2100, 1536)]
LARGE_WEIGHTS = [(2, 16001, 1024), (4, 4163, 512), (6, 4100, 1536), (12, 4096, 512)]
EVERY_SIZE = [(2, 16001, 1024), (4, 4163, 512), (6, 4100, 1536), (16, 2100, 1536)]


@pytest.mark.gpu
@pytest.mark.parametrize("T", [3, 4])
@pytest.mark.parametrize("I,M,N", TWO_TERMS)
def test_three_and_four_tokens(I, M, N, T):
    """Two fp16 terms per weight: nothing but y is rounded, so it stands no further from float64 than the factor-through kernel."""
    print(f"two terms I={I} M={M} N={N} T={T}", flush=True)
    L = _lib.lib()
    _runs_on(_lib.TILE_TWO_TERMS, [(I, M)], N, T)
    args, want = _args(I, M, N, T, False)
    size = np.abs(args[3].cpu().numpy().astype(np.float64)) @ np.abs(IU.unpack_and_reconstruct_w_hip(*args[:3]).cpu().numpy().astype(np.float64)).T
    y = IU.bitstack_forward_hip(*args)
    _lib.workspace(torch.device("cuda"), 1).fill_(0xFF)
    assert torch.equal(IU.bitstack_forward_hip(*args), y)
    d = np.abs(y.cpu().numpy().astype(np.float64) - want)
    error = np.linalg.norm(d) / np.linalg.norm(want)
    for mode in (_lib.DECODE_F16, None):                 # the other kernel: pinned, and by u's alignment
        if mode is not None:
            _lib.check(L.bs_set_decode_kernel(mode), "bs_set_decode_kernel")
        try:
            other = IU.bitstack_forward_hip(*(args if mode is not None else _args(I, M, N, T, True)[0])).cpu().numpy().astype(np.float64)
        finally:
            L.bs_set_decode_kernel(_lib.DECODE_AUTO)
        assert error <= 1.02 * np.linalg.norm(other - want) / np.linalg.norm(want)
    # one rounding of y; the weights to 2^-21, their fp32 sums over I blocks and y's over the columns, 32 at a time: 40 additions at most on the way
    assert bool((d <= np.abs(want) * 2.0 ** -11 + size * 2.0 ** -18 + 2.0 ** -25).all())


@pytest.mark.gpu
@pytest.mark.parametrize("T", [3, 4])
def test_three_and_four_tokens_with_non_finite_inputs_and_large_weights(T):
    I, M, N = 3, 2800, 1024
    (q, u, vt, x, _), _ = _args(I, M, N, T, False)
    u, vt, x = u * 0 + 1, vt * 0 + 1, x * 0 + 1
    q = torch.full_like(q, 0xFF)                         # weights: 16 per block
    bad = u.clone()
    bad[1, 37, 3] = float("inf")
    y = IU.bitstack_forward_hip(q, bad, vt, x, None)
    keep = torch.arange(M, device="cuda") != 37
    assert bool(torch.isposinf(y[..., 37]).all()) and bool((y[..., keep] == 48.0 * N).all())
    bad[1, 37, 3] = float("nan")
    y = IU.bitstack_forward_hip(q, bad, vt, x, None)
    assert bool(torch.isnan(y[..., 37]).all()) and bool((y[..., keep] == 48.0 * N).all())
    # a weight beyond fp16's range stays what it is: 16 * 80 * 80 = 102400 in one block
    big = u.clone()
    big[0, 5, :] = 80.0
    w_vt = vt.clone()
    w_vt[0] = 80.0
    z = torch.zeros_like(x)
    z[..., 9] = 0.25
    y = IU.bitstack_forward_hip(q, big, w_vt, z, None)
    assert bool((y[..., 5] == 0.25 * (102400 + 32)).all()), y[..., 5]


@pytest.mark.gpu
@pytest.mark.parametrize("T", [3, 4])
@pytest.mark.parametrize("I,M,N", LARGE_WEIGHTS)
def test_three_and_four_tokens_with_weights_beyond_fp16(I, M, N, T):
    """Weights of either sign on both sides of 65504 and of 131008, where two fp16 terms end, and far beyond: y is a finite fp16 number and has to be
    right, in rows beside each other and alone in their tile, and every other row keeps its bits."""
    print(f"large weights I={I} M={M} N={N} T={T}", flush=True)
    (q, u, vt, x, _), _ = _args(I, M, N, T, False)
    x = (x.float() * 2.0 ** -20).half()
    vt[0], u[0] = 448.0, 0.0                             # a weight of block 0 is 7168 u[0, row, 0], of random sign
    clean = IU.bitstack_forward_hip(q, u, vt, x, None)
    rows = [3, 4, 5, 37, 40, 64, 71, M - 2]
    for row, value in zip(rows, (9.0, -9.5, 18.0, -18.5, 28.0, -28.0, 20000.0, -20000.0)):
        u[0, row] = value
    y = IU.bitstack_forward_hip(q, u, vt, x, None)
    keep = torch.ones(M, dtype=torch.bool, device="cuda")
    keep[rows] = False
    assert torch.equal(y[..., keep], clean[..., keep])
    sign = ((q.view(I, M, N // 8, 1)[:, rows] >> torch.arange(7, -1, -1, device="cuda", dtype=torch.uint8)) & 1).reshape(I, len(rows), N)
    w = torch.zeros(len(rows), N, dtype=torch.float64, device="cuda")
    for i in range(I):
        p = u[i, rows].double() @ vt[i].double()
        w += torch.where(sign[i].bool(), p, -p)
    assert float(w.min()) < -1e8 and float(w.max()) > 1e8
    xd = x.view(T, N).double()
    want, size = xd @ w.t().contiguous(), xd.abs() @ w.abs().t().contiguous()
    # one rounding of y; fp32 sums of I blocks and over the columns (32 at a time), weights to 2^-21
    assert bool(((y.view(T, M)[:, rows].double() - want).abs() <= want.abs() * 2.0 ** -11 + size * 2.0 ** -15 + 2.0 ** -25).all())
    # infinite weights stay infinite and keep their sign, a NaN stays one, and their neighbours keep their bits
    ones, x = torch.full_like(q, 0xFF), x.abs() + 2.0 ** -14
    u[0, 36:39] = 0.0
    clean = IU.bitstack_forward_hip(ones, u, vt, x, None).view(T, M)
    u[0, 36], u[0, 37], u[0, 38] = float("inf"), float("-inf"), float("nan")
    y = IU.bitstack_forward_hip(ones, u, vt, x, None).view(T, M)
    assert bool((y[:, 36] == float("inf")).all()) and bool((y[:, 37] == float("-inf")).all()) and bool(y[:, 38].isnan().all())
    assert torch.equal(y[:, :36], clean[:, :36]) and torch.equal(y[:, 39:], clean[:, 39:])


@pytest.mark.gpu
@pytest.mark.parametrize("T", [3, 4])
@pytest.mark.parametrize("I,M,N", EVERY_SIZE)
def test_three_and_four_tokens_with_weights_of_every_size(I, M, N, T):
    """Rows with weights from about 0.1 down to 1e-9 beside each other: the second term holds what the first one leaves of a small weight too, so no row stands further
    from float64 than the rounding of its y."""
    print(f"weights of every size I={I} M={M} N={N} T={T}", flush=True)
    (q, u, vt, x, _), _ = _args(I, M, N, T, False)
    power = torch.arange(M, device="cuda") % 14
    u = (u.float() * 2.0 ** 6 * torch.pow(4.0, -power.float()).view(1, M, 1)).half()
    x = (x.float() * 2.0 ** 9).half()
    want = torch.from_numpy(C.forward_f64(q.cpu().numpy(), u.cpu().numpy(), vt.cpu().numpy(), x.cpu().numpy())).cuda().view(T, M)
    y = IU.bitstack_forward_hip(q, u, vt, x, None).view(T, M).double()
    for p in range(14):
        # One rounding of y to fp16, and of the weights at most 2^-12 at random (below 2^-24, where the first term is nothing), so 2^-12 of y too: the
        # two add up as squares.  The fp32 sums are a hundredth of that.
        d, rounding = (y - want)[:, power == p].norm(), (want.half().double() - want)[:, power == p].norm()
        lost = (2.0 ** -21 if p < 5 else 2.0 ** -12) * want[:, power == p].norm()
        assert d <= 1.01 * torch.hypot(rounding, lost), (p, float(d / rounding))


# groups at three and four tokens, as a decoder has them: q, k and v, gate and up, of each width
TWO_TERM_GROUPS = [([(6, 4096), (6, 1024), (7, 1024)], 4096), ([(6, 8200), (7, 8200)], 2560), ([(3, 16001), (4, 16001)], 1024), ([(3, 8193), (2, 8193)], 2048), ([(12, 4097), (10, 4097)], 1536)]


@pytest.mark.gpu
@pytest.mark.parametrize("T", [3, 4])
@pytest.mark.parametrize("epilogue", ["none", "rms", "rms residual", "rms swiglu", "swiglu"])
@pytest.mark.parametrize("layers,N", TWO_TERM_GROUPS)
def test_groups_at_three_and_four_tokens(layers, N, epilogue, T):
    """The sums of squares of x for the RMS scale, the residual and SwiGLU behind the weights in two terms, against float64."""
    print(f"two-term group {layers} N={N} {epilogue} T={T}", flush=True)
    L = _lib.lib()
    _runs_on(_lib.TILE_TWO_TERMS, layers, N, T)
    swiglu, residual, eps = "swiglu" in epilogue, "residual" in epilogue, 1e-5
    if swiglu:
        layers = layers[:2] if layers[0][1] == layers[1][1] else [layers[0], layers[0]]
        _runs_on(_lib.TILE_TWO_TERMS, layers, N, T)
    x = synthetic_layer(8, N, 1, T, seed=T)[3].cuda().view(T, N)
    xd, want, size = x.double(), [], []
    mats, keep = (_lib.bs_matrix * len(layers))(), []
    for j, (I, M) in enumerate(layers):
        q, u, vt, _ = (t.cuda() for t in synthetic_layer(M, N, I, T, seed=10 + j, signed_factors=True))
        u = (u * 20).half()
        keep.append((q, u, vt))
        mats[j] = _lib.bs_matrix(q.data_ptr(), u.data_ptr(), vt.data_ptr(), None, I, M)
        sign = ((q.view(I, M, N // 8, 1) >> torch.arange(7, -1, -1, device="cuda", dtype=torch.uint8)) & 1).reshape(I, M, N)
        w = torch.zeros(M, N, dtype=torch.float64, device="cuda")
        for i in range(I):
            p = u[i].double() @ vt[i].double()
            w += torch.where(sign[i].bool(), p, -p)
        del sign
        want.append(xd @ w.t().contiguous())
        size.append(xd.abs() @ w.abs().t().contiguous())
    scale = torch.rsqrt(xd.pow(2).mean(1, keepdim=True) + eps) if "rms" in epilogue else torch.ones(T, 1, dtype=torch.float64, device="cuda")
    want, size = [v * scale for v in want], [v * scale for v in size]
    # a sum: one rounding of y, weights to 2^-21 and fp32 sums (40 additions at most on the way), the scale to 2^-21
    bound = [v.abs() * 2.0 ** -11 + z * 2.0 ** -18 + 2.0 ** -25 for v, z in zip(want, size)]
    rows = sum(M for _, M in layers)
    res = torch.randn(T, rows, device="cuda").half() if residual else None
    if swiglu:
        rows = layers[0][1]
        gate, up = want
        act = gate * torch.sigmoid(gate)
        # silu's slope is at most 1.1, its value at most its argument's; act and the product are rounded once each, the exponential is good to 2^-20
        off = 1.1 * bound[0] + act.abs() * 1.01 * 2.0 ** -11 + 2.0 ** -25
        want, bound = act * up, off * (up.abs() + bound[1]) + act.abs() * bound[1]
        bound += want.abs() * 1.01 * 2.0 ** -11 + 2.0 ** -25
    else:
        want, bound = torch.cat(want, 1), torch.cat(bound, 1)
        if residual:
            want = want + res.double()
            bound += want.abs() * 1.01 * 2.0 ** -11
    y = torch.full((T, rows), float("nan"), dtype=torch.half, device="cuda")
    need = L.bs_forward_group_workspace_bytes(ctypes.byref(mats), len(layers), N, 16, T)
    ws = torch.full((need + 256,), 0xFF, dtype=torch.uint8, device="cuda")
    code = _lib.EPI_SWIGLU if swiglu else _lib.EPI_RESIDUAL if residual else _lib.EPI_NONE
    stream = torch.cuda.current_stream().cuda_stream
    args = (code, res.data_ptr() if residual else None, y.data_ptr(), ws.data_ptr(), need, stream)
    if "rms" in epilogue:
        _lib.check(L.bs_forward_group_rms(ctypes.byref(mats), len(layers), N, 16, x.data_ptr(), T, eps, *args), "bs_forward_group_rms")
    else:
        _lib.check(L.bs_forward_group(ctypes.byref(mats), len(layers), N, 16, x.data_ptr(), T, *args), "bs_forward_group")
    assert bool((ws[need:] == 0xFF).all())
    worst = ((y.double() - want).abs() / bound).max()
    assert bool(worst <= 1.0), float(worst)


# 49 to 128 tokens: the column kernel from 11 Mi weights on.  Both sides of its token tiles and block limits, rows about whole workgroups of 256,
# half a span of columns at the end, one span and many per workgroup
COLUMNS = [(1, 11300, 1024, 49), (2, 12033, 1024, 64), (8, 2816, 4096, 64), (8, 2817, 4224, 50), (3, 30977, 384, 65), (7, 2815, 4352, 96), (5, 90200, 128, 80),
           (6, 11265, 1152, 97), (6, 4000, 4096, 128), (4, 257, 45056, 127), (1, 20737, 640, 128), (5, 8191, 5760, 100)]


@pytest.mark.gpu
@pytest.mark.parametrize("I,M,N,T", COLUMNS)
def test_columns_edges(I, M, N, T):
    """Against float64 from the same rounded weights, and against the kernels that take the call when u is off a 16-byte boundary."""
    print(f"column kernel I={I} M={M} N={N} T={T}", flush=True)
    L = _lib.lib()
    assert L.bs_forward_path(I, M, N, 16, T) in (_lib.PATH_WALKED, _lib.PATH_PANEL)
    _runs_on(_lib.TILE_COLUMN, [(I, M)], N, T)
    q, u, vt, x = (t.cuda() for t in synthetic_layer(M, N, I, T, seed=I + N + T, signed_factors=True))
    u = (u * 20).half()
    bias = torch.randn(M, device="cuda").half()
    need = L.bs_workspace_bytes(I, M, N, 16, T)
    guard = torch.full((need // 2 + 64,), float("nan"), dtype=torch.half, device="cuda")
    y = torch.full((T, M), float("nan"), dtype=torch.half, device="cuda")
    _lib.check(L.bs_forward(q.data_ptr(), u.data_ptr(), vt.data_ptr(), x.data_ptr(), bias.data_ptr(), y.data_ptr(), I, M, N, 16, T, guard.data_ptr(), need,
                            torch.cuda.current_stream().cuda_stream), "bs_forward")
    assert bool(guard[need // 2:].isnan().all())
    room = torch.empty(u.numel() + 4, dtype=u.dtype, device="cuda")
    room[4:] = u.flatten()
    other = IU.bitstack_forward_hip(q, room[4:].view(u.shape), vt, x, bias).view(T, M)
    # Rounded weights: 2^-11 of a weight where the two fp32 sums straddle a rounding boundary, for few of them; then fp32 sums over the columns
    # and one rounding to fp16.
    w = IU.unpack_and_reconstruct_w_hip(q, u, vt)
    xd = x.view(T, N).double()
    want = torch.matmul(xd, w.double().t().contiguous()) + bias.double()
    size = torch.matmul(xd.abs(), w.double().abs().t().contiguous()) + bias.double().abs()
    bound = want.abs() * 2.0 ** -10 + size * 2.0 ** -12
    assert bool(((y.double() - want).abs() <= bound).all()) and bool(((other.double() - want).abs() <= bound).all())


@pytest.mark.gpu
@pytest.mark.parametrize("I,M,N,T", [(3, 30800, 384, 60), (2, 2900, 4096, 128)])
def test_columns_with_non_finite_inputs(I, M, N, T):
    """An infinity or NaN in u, vt or x reaches the outputs it has a part in and no others, and an infinite weight stays one beside the columns
    that a half span at the end does not have."""
    q, u, vt, x = (t.cuda() for t in synthetic_layer(M, N, I, T, seed=3, signed_factors=True))
    clean = IU.bitstack_forward_hip(q, u, vt, x, None).view(T, M)
    keep = torch.arange(M, device="cuda") != 37
    for value in (float("inf"), float("nan")):
        bad = u.clone()
        bad[1, 37, 3] = value
        y = IU.bitstack_forward_hip(q, bad, vt, x, None).view(T, M)
        assert not torch.isfinite(y[:, 37]).any() and torch.equal(y[:, keep], clean[:, keep])
        bad = x.clone()
        bad.view(T, N)[T - 1, 130] = value
        y = IU.bitstack_forward_hip(q, u, vt, bad, None).view(T, M)
        assert not torch.isfinite(y[T - 1]).any() and torch.equal(y[:T - 1], clean[:T - 1])
        bad = vt.clone()
        bad[1, 5, 200] = value
        assert not torch.isfinite(IU.bitstack_forward_hip(q, u, bad, x, None)).any()
    big, ones, pos = u.clone(), torch.full_like(q, 0xFF), vt.abs() + 0.01
    big[0, 37, 3] = float("inf")
    y = IU.bitstack_forward_hip(ones, big, pos, x.abs() + 0.01, None).view(T, M)
    assert bool((y[:, 37] == float("inf")).all())
