"""The sparse kernel (one to three tokens, the sign bits as the index operand of the sparse matrix instruction) at the edges of its units,
against float64: nothing but y is rounded."""
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

# (blocks, out features, in features, rank, tokens): rows about whole tiles of 16 and workgroups of 128, 256 and 512, column groups of 128
# that leave a unit's lanes without columns, one unit per workgroup and several, ranges that end inside a row of units, ranks below 16
CASES = [(1, 1, 512, 16, 2), (3, 17, 512, 16, 2), (2, 129, 1024, 5, 3), (5, 700, 1536, 16, 3), (14, 1300, 512, 16, 1), (5, 2100, 1024, 11, 1), (1, 4097, 4096, 16, 1), (3, 1025, 4096, 1, 3), (2, 14336, 2048, 16, 2),
         (1, 14300, 4096, 16, 1), (16, 1000, 3584, 12, 3), (3, 4096, 4096, 16, 3), (2, 16, 128, 7, 2), (3, 100, 384, 3, 1), (4, 2053, 2176, 16, 1), (2, 4096, 11008, 16, 2),
         (6, 3000, 1408, 16, 1), (1, 20001, 896, 16, 2), (8, 5000, 5504, 9, 1), (1, 40000, 640, 16, 1)]


def test_which_calls_the_sparse_kernel_serves():
    for I, M, N, K, T in CASES:
        assert _lib.sparse_kernel([(I, M)], N, K, T), (I, M, N, K, T)
        assert _lib.forward_kernel_name(I, M, N, K, T) == "gemv_sparse_kernel"
    # every height of a workgroup at every token count
    reached = {(_lib.decode_plan(I, M, N, 16, T)[1], T) for T in (1, 2, 3) for I, M, N in ((2, 2048, 2048), (2, 4096, 4096), (1, 14336, 4096), (1, 28672, 4096))}
    assert reached == {(r, t) for r in (1, 2, 4) for t in (1, 2, 3)}
    for I, M, N, K, T in [(8, 14336, 4096, 16, 1), (8, 14336, 4096, 16, 2), (2, 14336, 4096, 16, 4), (1, 5877, 640, 16, 1), (1, 1024, 4096, 16, 1), (4, 4096, 11008, 16, 3), (2, 64, 72, 16, 1), (2, 64, 128, 16, 5)]:
        assert not _lib.sparse_kernel([(I, M)], N, K, T), (I, M, N, K, T)
    L = _lib.lib()
    try:
        L.bs_set_decode_kernel(_lib.DECODE_F16)
        assert not _lib.sparse_kernel([(3, 4096)], 4096, 16, 1) and _lib.forward_kernel_name(3, 4096, 4096, 16, 1).startswith("gemv_kernel")
    finally:
        L.bs_set_decode_kernel(_lib.DECODE_AUTO)


# Calls that other kernels are quicker on, and neighbours that they are not (us sparse / tile or strip kernel): many partial sums per output (few rows of many columns), a
# unit that is mostly empty (up to 256 columns), long stacks of three tokens
LEFT_TO_OTHERS = [(8, 144, 26112, 16, 3), (8, 55, 30720, 16, 3), (8, 260, 30208, 16, 3), (10, 4882, 8192, 16, 3),       # 17.1 / 11.1, 14.9 / 9.6, 24.2 / 16.3, 45.3 / 41.5
                  (16, 20204, 128, 16, 2), (8, 28, 27392, 16, 2), (8, 320, 27520, 16, 2), (8, 71, 29824, 8, 2)]         # 20.8 / 15.7, 12.4 / 8.8, 17.8 / 15.2, 14.8 / 12.1
KEPT = [(4, 4096, 4096, 16, 3), (8, 4096, 4096, 16, 3), (3, 718, 4608, 16, 3), (4, 4096, 11008, 16, 1), (8, 4096, 11008, 16, 2), (2, 20000, 1408, 16, 2), (4, 21114, 4736, 16, 2), (3, 27415, 256, 16, 1)]


def test_calls_that_are_quicker_elsewhere_are_left_there():
    for I, M, N, K, T in LEFT_TO_OTHERS:
        assert not _lib.sparse_kernel([(I, M)], N, K, T), (I, M, N, K, T)
        kind = _lib.tile_kernel([(I, M)], N, K, T)[0]
        assert kind == (_lib.TILE_NONE if K != 16 else _lib.TILE_TWO_TERMS if T == 3 else _lib.TILE_FORWARD), (I, M, N, K, T)
        assert _lib.lib().bs_workspace_bytes(I, M, N, K, T) <= 64 << 20
    for I, M, N, K, T in KEPT:
        assert _lib.sparse_kernel([(I, M)], N, K, T) and _lib.tile_kernel([(I, M)], N, K, T)[0] == _lib.TILE_NONE, (I, M, N, K, T)


def test_the_decode_plan_is_the_sparse_kernels_wherever_it_serves():
    for I, M, N, K, T in CASES + [(4, 4096, 11008, 16, 1)]:
        waves, R, grid, kmax = _lib.decode_plan(I, M, N, K, T)
        units = I * -(-M // (128 * R)) * -(-N // 512) if R else 0
        assert waves == 8 and R in (1, 2, 4) and grid == min(units, 256) and 1 <= kmax <= -(-N // 512), (I, M, N, K, T)
    # the strip and tile kernels' calls, and the strip kernel's below the sparse one's sizes
    for I, M, N, K, T in [(4, 4096, 11008, 16, 3), (4, 4096, 11008, 16, 8), (1, 5877, 640, 16, 1), (4, 4096, 4096, 16, 40)]:
        assert _lib.decode_plan(I, M, N, K, T) == (0, 0, 0, 0), (I, M, N, K, T)


@pytest.mark.parametrize("M,N,K,T,mx,sparse,path", [
    # a block of vt, or x, reaches 2^31 bytes: not the kernels that address it with 32-bit offsets; 2^32: not gemv_kernel either
    (1, 1 << 28, 16, 1, False, False, _lib.PATH_REBUILD), (1, (1 << 27) - 512, 16, 1, False, False, _lib.PATH_DECODE_F16), (1, 1 << 27, 16, 1, False, False, _lib.PATH_REBUILD),
    (1, (1 << 26) - 512, 16, 1, True, True, _lib.PATH_DECODE_F16), (1, 1 << 26, 16, 1, False, False, _lib.PATH_DECODE_F16), (1, (1 << 30) - 512, 1, 1, True, True, _lib.PATH_DECODE_F16),
    (1, 1 << 29, 1, 2, True, False, _lib.PATH_DECODE_F16), (1, 1 << 29, 1, 3, False, False, _lib.PATH_DECODE_F16), (1, (1 << 30) - 512, 2, 2, False, False, _lib.PATH_DECODE_F16)])
def test_columns_beyond_32_bit_offsets(M, N, K, T, mx, sparse, path):
    assert _lib.sparse_kernel([(1, M)], N, K, T) == sparse
    L = _lib.lib()
    assert L.bs_forward_path(1, M, N, K, T) == path and L.bs_workspace_bytes(1, M, N, K, T) > 0
    try:
        L.bs_set_decode_kernel(_lib.DECODE_MX)
        assert (L.bs_decode_kernel(1, M, N, K, T) == _lib.DECODE_MX) == mx
    finally:
        L.bs_set_decode_kernel(_lib.DECODE_AUTO)


@pytest.mark.skipif(not os.path.exists(shutil.which("hipcc") or "/opt/rocm/bin/hipcc"), reason="hipcc not available")
def test_the_sparse_kernel_keeps_everything_in_registers(tmp_path):
    asm, source = tmp_path / "k.s", os.path.join(os.path.dirname(_lib.LIB_PATH), "gemv_sparse.hip")
    subprocess.run([shutil.which("hipcc") or "/opt/rocm/bin/hipcc", "--offload-arch=gfx950", "-O3", "-std=c++17", "-Xclang", "-target-feature", "-Xclang",
                    "-packed-fp32-ops", "-S", "--cuda-device-only", source, "-o", str(asm)], check=True, capture_output=True)
    sizes = re.findall(r"\.private_segment_fixed_size:\s+(\d+)", asm.read_text())
    assert sizes and set(sizes) == {"0"}, sizes


def _layer(I, M, N, K, T):
    q, u, vt, x = synthetic_layer(M, N, I, T, k=K, seed=I + M + N + T, signed_factors=True)
    u = (u * 20).half()
    want = torch.from_numpy(C.forward_f64(q.numpy(), u.numpy(), vt.numpy(), x.numpy())).view(T, M)
    size = torch.from_numpy(C.forward_f64(np.full_like(q.numpy(), 0xFF), u.abs().numpy(), vt.abs().numpy(), x.abs().numpy())).view(T, M)
    return q.cuda(), u.cuda(), vt.cuda(), x.cuda(), want.cuda(), size.cuda()


@pytest.mark.gpu
@pytest.mark.parametrize("I,M,N,K,T", CASES)
def test_edges(I, M, N, K, T):
    print(f"sparse kernel I={I} M={M} N={N} K={K} T={T}", flush=True)
    assert _lib.sparse_kernel([(I, M)], N, K, T)
    q, u, vt, x, want, size = _layer(I, M, N, K, T)
    bias = torch.randn(M, device="cuda").half() if (M + T) % 2 else None
    L = _lib.lib()
    need = L.bs_workspace_bytes(I, M, N, K, T)
    guard = torch.full((need + 256,), 0xFF, dtype=torch.uint8, device="cuda")        # nothing is read from scratch that the call has not written
    room = torch.empty(u.numel() + 4, dtype=u.dtype, device="cuda")                  # u 8 bytes off a 16-byte boundary
    room[4:] = u.flatten()
    y = torch.full((T, M), float("nan"), dtype=torch.half, device="cuda")
    for _ in range(2):
        _lib.check(L.bs_forward(q.data_ptr(), room[4:].data_ptr(), vt.data_ptr(), x.data_ptr(), None if bias is None else bias.data_ptr(), y.data_ptr(), I, M, N, K, T,
                                guard.data_ptr(), need, torch.cuda.current_stream().cuda_stream), "bs_forward")
    assert bool((guard[need:] == 0xFF).all())
    assert torch.equal(IU.bitstack_forward_hip(q, u, vt, x, bias).view(T, M), y)
    if bias is not None:
        want, size = want + bias.double(), size + bias.double().abs()
    # One rounding of y; exact products; fp32 sums over a unit's 16 operands of 32 columns, the units of a range, 16 ranks and the slots: fewer than
    # 2^10 additions on the way, whose errors are random: 2^-18 of the sum of the magnitudes is five times their largest here.
    assert bool(((y.double() - want).abs() <= want.abs() * 2.0 ** -11 + size * 2.0 ** -18 + 2.0 ** -25).all())


# Several units per workgroup, so that the loop over them, its two register sets and LDS buffers, u at a crossing and the slots that a finished row leaves empty are
# reached: every (row tiles per wave, tokens), two to six units, ranges that start and end within a row of units and run over one, two and three of them
SEVERAL = [(5, 1100, 5632, 16, 1), (4, 1100, 11008, 16, 1), (4, 3001, 8192, 9, 1), (5, 28001, 896, 16, 1), (5, 5001, 11008, 16, 1),
           (5, 1100, 5632, 11, 2), (5, 1100, 11008, 16, 2), (5, 9000, 1408, 16, 2), (7, 28001, 896, 13, 2), (4, 28001, 1408, 16, 2),
           (7, 1100, 8192, 16, 3), (4, 4097, 8192, 16, 3), (7, 5001, 5632, 11, 3), (7, 4097, 5632, 11, 3), (3, 28001, 3584, 16, 3)]


def test_the_cases_of_several_units_are_that():
    heights, lengths, rows, inside = set(), set(), set(), 0
    for I, M, N, K, T in SEVERAL:
        assert _lib.sparse_kernel([(I, M)], N, K, T), (I, M, N, K, T)
        waves, R, grid, kmax = _lib.decode_plan(I, M, N, K, T)
        chunks = -(-N // 512)
        q, rem = divmod(I * -(-M // (128 * R)) * chunks, grid)
        heights.add((R, T))
        for w in range(grid):
            begin, end = w * q + min(w, rem), (w + 1) * q + min(w + 1, rem)
            lengths.add((T, min(end - begin, 4)))
            rows.add((T, (end - 1) // chunks - begin // chunks + 1))
            inside += begin % chunks != 0 and end % chunks != 0 and (end - 1) // chunks > begin // chunks
    assert heights == {(r, t) for r in (1, 2, 4) for t in (1, 2, 3)} and inside >= 100
    assert lengths >= {(t, n) for t in (1, 2, 3) for n in (2, 3, 4)} and rows >= {(t, n) for t in (1, 2, 3) for n in (1, 2)} and max(n for _, n in rows) >= 3


@pytest.mark.gpu
@pytest.mark.parametrize("I,M,N,K,T", SEVERAL)
def test_several_units(I, M, N, K, T):
    test_edges(I, M, N, K, T)                        # (the bound's count of additions covers six units of a range, and 7 x 22 slots)


@pytest.mark.gpu
@pytest.mark.parametrize("N,T", [(2560, 2), (3584, 3)])
def test_a_group_of_several_units(N, T):
    """Two to four units per workgroup on four row tiles per wave, more on fewer, and a rank below 16: the bound of test_edges."""
    layers, K = [(3, 9000), (2, 20001), (5, 700)], 11
    assert _lib.sparse_kernel(layers, N, K, T) and sum(I * -(-M // 512) for I, M in layers) * (N // 512) > 2 * 256
    parts = [_layer(I, M, N, K, T) for I, M in layers]
    group, x = IU.MatrixGroup([p[:3] + (None,) for p in parts]), parts[0][3]
    want, size = [], []
    for q, u, vt, _, _, _ in parts:                  # (all of them on the first one's x)
        q, u, vt, xc = (t.cpu().numpy() for t in (q, u, vt, x))
        want.append(torch.from_numpy(C.forward_f64(q, u, vt, xc)).view(T, -1))
        size.append(torch.from_numpy(C.forward_f64(np.full_like(q, 0xFF), np.abs(u), np.abs(vt), np.abs(xc))).view(T, -1))
    want, size = torch.cat(want, 1).cuda(), torch.cat(size, 1).cuda()
    print(f"group of several units N={N} T={T}", flush=True)
    y = IU.bitstack_forward_group_hip(group, x)
    assert torch.equal(y, IU.bitstack_forward_group_hip(group, x))
    assert bool(((y.double() - want).abs() <= want.abs() * 2.0 ** -11 + size * 2.0 ** -18 + 2.0 ** -25).all())


# One token from 8 to 12 MiB of sign bytes: many partial sums per output go to the block-scaled kernel, with half as many (us sparse / block-scaled: 15.7 / 12.2, 14.8 / 12.9,
# 13.2 / 11.6, 14.8 / 13.1); whole matrices do not, nor below 8 MiB
MANY_SUMS = [(16, 355, 15872), (14, 323, 15872), (9, 925, 11776), (8, 425, 26112)]


def test_many_partial_sums_go_to_the_block_scaled_kernel():
    for I, M, N in MANY_SUMS:
        assert not _lib.sparse_kernel([(I, M)], N, 16, 1) and _lib.lib().bs_decode_kernel(I, M, N, 16, 1) == _lib.DECODE_MX, (I, M, N)
    for I, M, N in [(4, 4096, 4096), (5, 4096, 4096), (3, 1792, 14336), (2, 14336, 2560), (16, 255, 15872), (16, 258, 14848)]:
        assert _lib.sparse_kernel([(I, M)], N, 16, 1), (I, M, N)
    assert not _lib.sparse_kernel([(1, 1627), (8, 297)], 17920, 16, 1) and _lib.sparse_kernel([(2, 4096), (3, 1024)], 4096, 16, 1)


@pytest.mark.gpu
@pytest.mark.parametrize("I,M,N", MANY_SUMS)
def test_many_partial_sums(I, M, N):
    """Within what three fp6 terms of vt * x (2^-12 of a block's largest) and one rounding of y allow."""
    print(f"many partial sums I={I} M={M} N={N}", flush=True)
    q, u, vt, x, want, size = _layer(I, M, N, 16, 1)
    y = IU.bitstack_forward_hip(q, u, vt, x, None).view(1, M)
    assert bool(((y.double() - want).abs() <= want.abs() * 2.0 ** -10 + size * 2.0 ** -11).all())


@pytest.mark.gpu
@pytest.mark.parametrize("I,M,N,K,T", LEFT_TO_OTHERS)
def test_calls_left_to_others(I, M, N, K, T):
    """u on a 16-byte boundary and off it, as a call of one matrix and as a group of one, twice: within what one rounding of the weight and one of y allow."""
    print(f"left to others I={I} M={M} N={N} K={K} T={T}", flush=True)
    q, u, vt, x, want, size = _layer(I, M, N, K, T)
    room = torch.empty(u.numel() + 4, dtype=u.dtype, device="cuda")
    room[4:] = u.flatten()
    ys = [IU.bitstack_forward_hip(q, f, vt, x, None).view(T, M) for f in (u, room[4:].view(u.shape), u)]
    ys.append(IU.bitstack_forward_group_hip(IU.MatrixGroup([(q, u, vt, None)]), x))
    assert torch.equal(ys[0], ys[2]) and torch.equal(ys[0], ys[3])
    assert all(bool(((y.double() - want).abs() <= want.abs() * 2.0 ** -10 + size * 2.0 ** -11).all()) for y in ys)


@pytest.mark.gpu
@pytest.mark.parametrize("I,M,N,K,T", [(3, 1024, 4096, 16, 3), (4, 2053, 2176, 16, 2), (2, 300, 640, 6, 1)])
def test_non_finite_inputs(I, M, N, K, T):
    """An infinity or NaN in u, vt or x reaches the outputs it has a part in and no others."""
    assert _lib.sparse_kernel([(I, M)], N, K, T)
    q, u, vt, x, _, _ = _layer(I, M, N, K, T)
    clean = IU.bitstack_forward_hip(q, u, vt, x, None).view(T, M)
    keep = torch.arange(M, device="cuda") != 37
    for value in (float("inf"), float("nan")):
        bad = u.clone()
        bad[1, 37, 3] = value
        y = IU.bitstack_forward_hip(q, bad, vt, x, None).view(T, M)
        assert not torch.isfinite(y[:, 37]).any() and torch.equal(y[:, keep], clean[:, keep])
        for col in (0, 130, N - 1):
            bad = x.clone()
            bad.view(T, N)[T - 1, col] = value
            y = IU.bitstack_forward_hip(q, u, vt, bad, None).view(T, M)
            assert not torch.isfinite(y[T - 1]).any() and torch.equal(y[:T - 1], clean[:T - 1])
            bad = vt.clone()
            bad[I - 1, K - 1, col] = value
            assert not torch.isfinite(IU.bitstack_forward_hip(q, u, bad, x, None)).any()


@pytest.mark.gpu
@pytest.mark.parametrize("I,M,N,K,T", [(4, 2053, 2176, 16, 2), (2, 300, 640, 6, 1), (3, 100, 384, 3, 1), (2, 16, 128, 7, 2), (2, 1024, 4096, 16, 1)])
def test_an_infinite_result_stays_one(I, M, N, K, T):
    """One infinity in vt, in the first columns and in the last ones (which a unit that is wider than what is left of the row may not repeat): y is
    infinite with the sign that float64 gives, and no NaN."""
    assert _lib.sparse_kernel([(I, M)], N, K, T)
    q, u, vt, x, _, _ = _layer(I, M, N, K, T)
    u[u == 0], x[x == 0] = 1.0, 1.0
    for col in (0, N - 9, N - 8, N - 3, N - 1):
        bad = vt.clone()
        bad[I - 1, K - 1, col] = float("inf")
        y = IU.bitstack_forward_hip(q, u, bad, x, None).view(T, M).cpu()
        want = torch.from_numpy(C.forward_f64(q.cpu().numpy(), u.cpu().numpy(), bad.cpu().numpy(), x.cpu().numpy())).view(T, M)
        assert bool(want.isinf().all()) and torch.equal(y.double(), want), col


@pytest.mark.gpu
@pytest.mark.parametrize("T", [1, 2, 3])
@pytest.mark.parametrize("layers,N", [([(3, 4096), (1, 1024), (2, 1024)], 1024), ([(2, 700), (1, 33), (3, 3000), (1, 64)], 1024), ([(2, 2816), (3, 2816)], 1664)])
def test_groups_with_the_epilogues(layers, N, T):
    """Matrices in one launch: side by side against float64, then with the RMS scale of x, a residual and SwiGLU against what that gave."""
    if T == 3 and N % 512:
        pytest.skip("the tile kernel's")
    assert _lib.sparse_kernel(layers, N, 16, T)
    parts = [_layer(I, M, N, 16, T) for I, M in layers]
    x, group = parts[0][3], IU.MatrixGroup([p[:3] + (None,) for p in parts])
    refs = [C.forward_f64(*(t.cpu().numpy() for t in p[:3]), x.cpu().numpy()) for p in parts]
    alone = torch.cat([torch.from_numpy(r).view(T, -1) for r in refs], 1).cuda()
    # one rounding to fp16 each, and fp32 sums (2^-18 of the magnitudes' sum, here below 2^-14 of the largest result)
    close = lambda a, b, bits: bool(((a.double() - b).abs() <= b.abs() * 2.0 ** -bits + b.abs().max() * 2.0 ** -14).all())
    got = IU.bitstack_forward_group_hip(group, x)
    assert close(got, alone, 10)
    scale = torch.rsqrt(x.double().pow(2).mean(1, keepdim=True) + 1e-5)
    assert close(IU.bitstack_forward_group_hip(group, x, rms_eps=1e-5), alone * scale, 9)
    res = torch.randn(T, sum(m for _, m in layers), device="cuda").half()
    assert close(IU.bitstack_forward_group_hip(group, x, epilogue=_lib.EPI_RESIDUAL, residual=res), res.double() + got.double(), 10)
    if len(layers) == 2:
        a, b = got[:, :layers[0][1]].double(), got[:, layers[0][1]:].double()
        assert close(IU.bitstack_forward_group_hip(group, x, epilogue=_lib.EPI_SWIGLU), a * torch.sigmoid(a) * b, 8)


@pytest.mark.gpu
@pytest.mark.parametrize("layers,N,T", [([(16, 4096)], 14336, 1), ([(8, 14336)], 4096, 1), ([(3, 9000), (2, 20000)], 1408, 2)])
def test_a_group_follows_the_pinned_kernel(layers, N, T):
    """Another kernel pinned after a group's first call needs other scratch: it is asked for again."""
    parts = [_layer(I, M, N, 16, T) for I, M in layers]
    group, x, L = IU.MatrixGroup([p[:3] + (None,) for p in parts]), parts[0][3], _lib.lib()
    want = torch.cat([p[4] for p in parts], 1) if len(layers) == 1 else None
    size, ys = torch.cat([p[5] for p in parts], 1), []
    try:
        for mode in (_lib.DECODE_AUTO, _lib.DECODE_F16, _lib.DECODE_MX, _lib.DECODE_AUTO):
            L.bs_set_decode_kernel(mode)
            with torch.cuda.stream(torch.cuda.Stream()):         # scratch of its own: the smallest there is
                ys.append(IU.bitstack_forward_group_hip(group, x))
            torch.cuda.synchronize()
    finally:
        L.bs_set_decode_kernel(_lib.DECODE_AUTO)
    assert torch.equal(ys[0], ys[3])
    want = ys[0].double() if want is None else want
    # vt * x, or the weight, rounded to fp16 once, and y
    assert all(bool(((y.double() - want).abs() <= want.abs() * 2.0 ** -10 + size * 2.0 ** -11).all()) for y in ys)
