"""The native host path (csrc/host.cpp) and the Python path behind it give the same results, and each call
that is not the ordinary case is left to the Python path."""
import pytest
import torch

from bitstack_amd import BitStackLinear, _lib
from bitstack_amd.utils import inference_utils as IU
from bitstack_amd.utils.synthetic import synthetic_layer


def layer(I, M, N, T, dev, bias=True):
    q, u, vt, x = synthetic_layer(M, N, I, T, seed=I + T, device=dev)
    mod = BitStackLinear(0, N, M, 16, False, False, dev, fused_level=5)
    mod.w_bit, mod.qweight, mod.u, mod.vt = I, q, u, vt
    if bias:
        mod.bias = (torch.randn(M, generator=torch.Generator().manual_seed(3)) * 0.1).half().to(dev)
    return mod, x


def test_unusual_arguments_are_left_to_python():
    mod, x = layer(2, 16, 64, 3, "cpu")
    H = _lib.host()
    assert H.forward(mod.qweight, mod.u, mod.vt, 2, x, mod.bias) is None          # CPU tensors
    assert H.rebuild(mod.qweight, mod.u, mod.vt, 2) is None
    assert H.linear(x, x, None) is None
    assert H.forward(None, None, None, 2, x, None) is None
    with pytest.raises(RuntimeError, match="HIP device"):
        mod(x)
    with pytest.raises(TypeError):
        H.forward(mod.qweight)


@pytest.mark.gpu
@pytest.mark.parametrize("I,M,N,T", [(1, 16, 512, 2), (3, 200, 1024, 5), (2, 100, 72, 3), (3, 256, 512, 130)])
def test_native_and_python_paths_agree(I, M, N, T):
    mod, x = layer(I, M, N, T, torch.device("cuda"))
    H = _lib.host()
    x3 = x.view(1, T, N).requires_grad_()
    y = mod(x3)
    assert y.shape == (1, T, M) and not y.requires_grad
    assert H.forward(mod.qweight, mod.u, mod.vt, I, x, mod.bias) is not None
    # the same call through a layout that only the Python path takes (columns of a wider tensor)
    wide = torch.zeros(T, N + 8, dtype=torch.float16, device=x.device)
    wide[:, :N] = x
    assert H.forward(mod.qweight, mod.u, mod.vt, I, wide[:, :N], mod.bias) is None
    assert torch.equal(y[0], IU.bitstack_forward_hip(mod.qweight, mod.u, mod.vt, wide[:, :N], mod.bias))
    # fewer blocks than are stacked
    mod.set_bit(1)
    assert torch.equal(mod(x), IU.bitstack_forward_hip(mod.qweight[:1], mod.u[:1], mod.vt[:1], x, mod.bias))
    mod.set_bit(I)
    w = IU.unpack_and_reconstruct_w_hip(mod.qweight, mod.u, mod.vt)
    assert torch.equal(w, mod._rebuilt())
    assert torch.equal(IU.linear_f16_hip(x, w), IU.linear_f16_hip(wide[:, :N], w))


@pytest.mark.gpu
def test_scratch_is_one_tensor_per_stream_and_outgrown_ones_stay():
    dev = torch.device("cuda")
    a = _lib.workspace(dev, 1 << 20)
    assert _lib.workspace(dev, 1000).data_ptr() == a.data_ptr()
    with torch.cuda.stream(torch.cuda.Stream()):
        b = _lib.workspace(dev, 1000)
        assert b.data_ptr() != a.data_ptr()
    big = _lib.workspace(dev, 2 * a.numel() + 1)
    assert big.numel() > 2 * a.numel() and big.data_ptr() != a.data_ptr()


def test_the_host_module_has_no_thread_local_storage():
    """A module with a TLS segment that is never touched slows every thread-local access of the process (glibc before 2.39)."""
    import struct
    _lib.host()
    data = open(_lib.host().__file__, "rb").read()
    offset, size, count = struct.unpack_from("<Q", data, 32)[0], *struct.unpack_from("<HH", data, 54)
    kinds = [struct.unpack_from("<I", data, offset + k * size)[0] for k in range(count)]
    assert 1 in kinds and 7 not in kinds      # PT_LOAD, PT_TLS


@pytest.fixture
def little_memory():
    """One GiB of GPU memory beyond what is reserved."""
    torch.cuda.empty_cache()
    total = torch.cuda.get_device_properties(0).total_memory
    torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + (1 << 30)) / total)
    yield
    torch.cuda.set_per_process_memory_fraction(1.0)


@pytest.mark.gpu
def test_an_allocation_that_fails_is_torchs_out_of_memory_error(little_memory):
    dev = torch.device("cuda")
    H = _lib.host()
    x, w = torch.zeros(1 << 16, 128, device=dev).half(), torch.zeros(1 << 15, 128, device=dev).half()
    before = _lib.workspace(dev, 1)
    with pytest.raises(torch.OutOfMemoryError):
        H.linear(x, w, None)                                                      # 4 GiB of output
    for _ in range(3):
        with pytest.raises(torch.OutOfMemoryError):
            _lib.workspace(dev, before.numel() + (4 << 30))
    assert _lib.workspace(dev, 1).data_ptr() == before.data_ptr()                 # ... and the scratch is what it was
    q, u, vt = torch.zeros(1, (1 << 15) * 16, dtype=torch.uint8, device=dev), torch.zeros(1, 1 << 15, 16, device=dev).half(), torch.zeros(1, 16, 128, device=dev).half()
    with pytest.raises(torch.OutOfMemoryError):
        H.forward(q, u, vt, 1, x, None)
    with pytest.raises(torch.OutOfMemoryError):
        H.unpack(torch.zeros(4, (1 << 29) // 8, dtype=torch.uint8, device=dev), 4, 1 << 20, 512)


@pytest.mark.gpu
def test_scratch_can_be_asked_for_while_it_is_being_allocated(little_memory):
    """An out-of-memory observer runs inside the allocation: what it calls may want scratch too."""
    dev = torch.device("cuda")
    have = _lib.workspace(dev, 1)
    got = []
    torch._C._cuda_attach_out_of_memory_observer(lambda *args: got.append(_lib.workspace(dev, 1).data_ptr()) if not got else None)
    with pytest.raises(torch.OutOfMemoryError):
        _lib.workspace(dev, have.numel() + (4 << 30))
    assert got == [have.data_ptr()]


@pytest.mark.gpu
def test_threads_grow_the_scratch_of_one_stream_together():
    import threading
    dev = torch.device("cuda")
    with torch.cuda.stream(torch.cuda.Stream()):
        stream = torch.cuda.current_stream()
        sizes, tensors = [], []
        def grow(k):
            with torch.cuda.stream(stream):
                for j in range(1, 40):
                    n = (1 << 20) + 4096 * j * (k + 1)
                    t = _lib.workspace(dev, n)
                    sizes.append(t.numel() >= n)
                    tensors.append(t)
        threads = [threading.Thread(target=grow, args=(k,)) for k in range(6)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        assert all(sizes) and len(sizes) == 6 * 39
        assert len({t.data_ptr() for t in tensors}) <= 8 and _lib.workspace(dev, 1).data_ptr() == max(tensors, key=lambda t: t.numel()).data_ptr()


def _calls(dev):
    """name -> a call of each entry point that launches."""
    mod, x = layer(2, 512, 1024, 2, dev)
    H = _lib.host()
    w = mod._rebuilt()
    sign = H.unpack(mod.qweight, 2, 512, 1024)
    out = torch.zeros(2, dtype=torch.long, device=dev)
    y = torch.empty(2, 1024, dtype=torch.float16, device=dev)
    weight = torch.ones(1024, dtype=torch.float16, device=dev)
    steps = H.make_steps([("norm", x.data_ptr(), weight.data_ptr(), y.data_ptr(), 2, 1024, 1e-5)])
    return {"forward": lambda: H.forward(mod.qweight, mod.u, mod.vt, 2, x, mod.bias), "rebuild": lambda: H.rebuild(mod.qweight, mod.u, mod.vt, 2),
            "unpack": lambda: H.unpack(mod.qweight, 2, 512, 1024), "rebuild_from_sign": lambda: H.rebuild_from_sign(sign, mod.u, mod.vt, 2),
            "linear": lambda: H.linear(x, w, None), "argmax": lambda: H.argmax(x, out), "workspace": lambda: H.workspace(dev.index, 1),
            "run_steps": lambda: (H.run_steps(steps, dev.index), y, weight)}


@pytest.mark.gpu
@pytest.mark.parametrize("name", ["forward", "rebuild", "unpack", "rebuild_from_sign", "linear", "argmax", "workspace", "run_steps"])
def test_other_threads_run_during_a_call(name):
    import sys
    import threading
    import time
    call = _calls(torch.device("cuda", torch.cuda.current_device()))[name]
    call()
    torch.cuda.synchronize()
    ran = []
    interval = sys.getswitchinterval()
    thread = threading.Thread(target=lambda: (time.sleep(0.05), ran.append(1)))
    thread.start()
    try:
        sys.setswitchinterval(1000.0)            # from here a thread that computes keeps the interpreter until it lets go of it
        end = time.perf_counter() + 0.15
        while time.perf_counter() < end:
            pass
        assert not ran                           # (waiting for the interpreter since its sleep ended)
        for _ in range(20000):
            call()
            if ran:
                break
        seen = bool(ran)                         # (a synchronisation lets go of it too)
    finally:
        sys.setswitchinterval(interval)
    thread.join()
    assert seen


@pytest.mark.gpu
def test_threads_that_share_a_stream_do_not_mix_their_scratch():
    import threading
    dev = torch.device("cuda")
    calls = []
    for I, M, N, T in ((3, 2048, 4096, 1), (2, 1024, 2048, 4), (2, 500, 640, 20), (3, 256, 512, 130)):
        mod, x = layer(I, M, N, T, dev)
        wide = torch.zeros(T, N + 8, dtype=torch.float16, device=dev)
        wide[:, :N] = x
        calls += [lambda mod=mod, x=x: mod(x), lambda mod=mod, x=wide[:, :N]: mod(x)]          # native, Python path
    mods = [layer(2, M, 1024, 200, dev, bias=False) for M in (512, 128)]
    calls.append(lambda: IU.forward_cat_hip([m for m, _ in mods], mods[0][1]))
    group = IU.MatrixGroup.from_modules([m for m, _ in mods])
    few = mods[0][1][:3].contiguous()
    calls.append(lambda: IU.bitstack_forward_group_hip(group, few))
    g = torch.Generator(device="cuda").manual_seed(1)
    qkv, cache = torch.randn(1, 48 * 128, generator=g, device=dev).half(), torch.randn(2, 1, 8, 2048, 128, generator=g, device=dev).half()
    cos, pos = torch.rand(2048, 64, generator=g, device=dev).half(), torch.full((1,), 2000, device=dev)
    calls.append(lambda: IU.attention_decode_hip(qkv, cache[0], cache[1], cos, cos, pos, 32, 8))
    want = [call() for call in calls]
    wrong, total = [], []

    def hammer(k):
        for _ in range(100):
            y = calls[k]()
            total.append(1)
            if not torch.equal(y, want[k]):
                wrong.append(k)
    threads = [threading.Thread(target=hammer, args=(k,)) for k in range(len(calls))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong and len(total) == 100 * len(calls)


@pytest.mark.gpu
def test_the_streams_launches_are_let_go_when_a_call_fails():
    dev = torch.device("cuda")
    with pytest.raises(RuntimeError):
        with _lib.scratch(dev, 16) as ws:
            assert ws.numel() >= 16
            _lib.check(_lib.lib().bs_forward(None, None, None, None, None, None, 1, 16, 512, 16, 1, _lib.ptr(ws), ws.numel(), _lib.stream_ptr(dev)), "bs_forward")
    mod, x = layer(1, 16, 512, 1, dev)
    assert mod(x).shape == (1, 16)
    with pytest.raises((ValueError, OverflowError, TypeError)):
        _lib.host().let_go(0)
