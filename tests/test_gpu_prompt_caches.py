"""A prompt pass over caches of another type or layout attends to k and v as they were computed, not to what such a cache keeps."""
import pytest
import torch

from bitstack_amd.utils.llama_decode import LlamaShape, PROJ, SyntheticLlamaDecoder

pytestmark = pytest.mark.gpu
SHAPE = LlamaShape(layers=2, hidden=512, intermediate=1024, heads=4, kv_heads=2, vocab=500)


def decoder():
    return SyntheticLlamaDecoder(SHAPE, {f"layer.{L}.{p}": 2 for L in range(2) for p in PROJ}, 24, "cuda", seed=5, batch=2)


def rel(a, b):
    return float((a.double() - b.double()).norm() / b.double().norm())


@pytest.mark.parametrize("kind", ["narrower", "wider", "dimensions apart", "wider k and v"])
def test_attention_sees_k_and_v_as_computed(kind):
    a, b = decoder(), decoder()
    prompt = torch.arange(2 * 20, device="cuda").view(2, 20)
    attended = []                                # what o_proj of the first layer is given
    for dec in (b, a):
        dec.lin[0][PROJ[3]].register_forward_pre_hook(lambda m, args: attended.append(args[0].clone()))
    b.prefill(prompt)
    if kind == "wider k and v":
        for row in a.lin:
            for p in PROJ[:3]:
                row[p].register_forward_hook(lambda m, args, out: out.float())
    else:
        to = {"narrower": lambda t: t.to(torch.float8_e4m3fn), "wider": lambda t: t.float(),
              "dimensions apart": lambda t: t.transpose(3, 4).contiguous().transpose(3, 4)}[kind]
        a.kcache, a.vcache = to(a.kcache), to(a.vcache)
    a.prefill(prompt)
    # fp16 roundings at other places (every operation of the rotation is rounded here)
    assert rel(attended[1], attended[0]) < 1e-3 and rel(a.logits, b.logits) < 3e-3
    for mine, ref in ((a.kcache, b.kcache), (a.vcache, b.vcache)):
        stored = mine.float()
        # the first layer's k and v are the same but for those roundings, an 8-bit cache keeps four bits of them
        assert rel(stored[0], ref[0].float()) < (0.04 if kind == "narrower" else 1e-3)
