"""A decoder whose norm weight, caches, tables or position are replaced between steps: step_fused() works on the tensors that
are in place when it is called, as a decoder that had them from the beginning, bit for bit."""
import pytest
import torch

from bitstack_amd.utils.llama_decode import LlamaShape, PROJ, SyntheticLlamaDecoder

pytestmark = pytest.mark.gpu
SHAPE = LlamaShape(layers=2, hidden=512, intermediate=1024, heads=4, kv_heads=2, vocab=1000)
CONFIG = {f"layer.{L}.{p}": 2 for L in range(2) for p in PROJ}
LEN = 24


def decoder(max_len=LEN):
    return SyntheticLlamaDecoder(SHAPE, CONFIG, max_len, "cuda", seed=3, batch=2)


def step(dec, token, pos):
    dec.token.fill_(token)
    dec.pos.fill_(pos)
    dec.step_fused()
    return dec.logits.clone(), dec.kcache.clone(), dec.vcache.clone()


def fill(shape, seed, scale=0.1):
    return (torch.randn(shape, generator=torch.Generator(device="cuda").manual_seed(seed), device="cuda") * scale).half()


def replacements():
    caches = (2, 2, 2, LEN, 128)
    wide = fill((2, 2) + caches[1:], 5)                          # a layer contiguous, the layers apart
    strided = fill((1024,), 6, 1.0)
    return {
        "norm": lambda d: {"final_norm": fill((512,), 1, 1.0)},
        "norm strided": lambda d: {"final_norm": strided[::2]},
        "keys": lambda d: {"kcache": fill(caches, 2)},
        "values": lambda d: {"vcache": fill(caches, 3)},
        "tables": lambda d: {"cos": fill((LEN, 64), 4, 1.0), "sin": fill((LEN, 64), 7, 1.0)},
        "layers apart": lambda d: {"kcache": wide[:, 0], "vcache": wide[:, 1]},
        "longer": lambda d: {n: getattr(decoder(2 * LEN), n) for n in ("kcache", "vcache", "cos", "sin")},
        "position without a dimension": lambda d: {"pos": torch.zeros((), dtype=torch.long, device="cuda")},
    }


@pytest.mark.parametrize("what", ["norm", "norm strided", "keys", "values", "tables", "layers apart", "longer", "position without a dimension"])
def test_a_step_uses_the_tensors_that_are_in_place(what):
    a, b = decoder(), decoder()
    step(a, 7, 3)
    kept = [a.final_norm, a.kcache, a.vcache, a.cos, a.sin, a.pos]      # (what a stale address would read stays allocated)
    for dec in (a, b):
        for name, t in replacements()[what](dec).items():
            if name in ("kcache", "vcache") and what != "longer":       # (what the earlier step has stored is not compared)
                t[:, :, :, 3] = 0
            setattr(dec, name, t)
    if what not in ("keys", "values", "layers apart", "longer"):
        b.kcache.copy_(a.kcache)
        b.vcache.copy_(a.vcache)
    elif what in ("keys", "values"):
        other = "vcache" if what == "keys" else "kcache"
        getattr(b, other).copy_(getattr(a, other))
    for token, pos in ((11, 4), (12, 5)):
        for got, want in zip(step(a, token, pos), step(b, token, pos)):
            assert torch.equal(got, want)
    assert len(kept) == 6


def test_what_the_step_cannot_read_is_refused():
    dec = decoder()
    step(dec, 7, 3)
    for name, t, error in (("kcache", dec.kcache.view(torch.int16), ValueError), ("vcache", dec.vcache[:, :, :, :16], ValueError),
                           ("vcache", dec.vcache[:1], ValueError), ("cos", dec.cos[:16], ValueError), ("sin", dec.sin.float(), ValueError),
                           ("pos", torch.zeros(2, dtype=torch.long, device="cuda"), ValueError), ("pos", dec.pos.int(), ValueError),
                           ("final_norm", dec.final_norm.float(), TypeError), ("final_norm", dec.final_norm[:256], ValueError)):
        good = getattr(dec, name)
        setattr(dec, name, t)
        with pytest.raises(error):
            dec.step_fused()
        setattr(dec, name, good)
    dec.step_fused()
