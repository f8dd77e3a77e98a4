"""The prompt pass keeps away from what a module has returned: a hook that records a linear's output finds there what the linear
computed, and everything a call of the module does besides is done."""
import types

import pytest
import torch

from bitstack_amd import BitStackLinear
from bitstack_amd.utils.llama_decode import LlamaShape, PROJ, SyntheticLlamaDecoder

pytestmark = pytest.mark.gpu


def decoder(hidden, batch, heads, length):
    shape = LlamaShape(layers=2, hidden=hidden, intermediate=2 * hidden, heads=heads, kv_heads=heads // 2, vocab=500)
    return SyntheticLlamaDecoder(shape, {f"layer.{L}.{p}": 2 for L in range(2) for p in PROJ}, length, "cuda", seed=5, batch=batch)


def linears(dec):
    return [m for row in dec.lin for m in row.values()]


# few tokens and many (one product for q, k and v), one position of one sequence, heads of another size
@pytest.mark.parametrize("hidden,batch,heads,n", [(512, 2, 4, 5), (512, 2, 4, 200), (512, 1, 4, 1), (256, 1, 4, 9)])
@pytest.mark.parametrize("how", ["hook", "global", "forward"])
def test_recorded_outputs_stay_what_the_modules_computed(hidden, batch, heads, n, how):
    dec, plain = (decoder(hidden, batch, heads, n) for _ in range(2))
    prompt = torch.randint(0, 500, (batch, n), device="cuda", generator=torch.Generator(device="cuda").manual_seed(n))
    plain.prefill(prompt)
    seen = []
    record = lambda mod, args, out: seen.append((mod, args[0], args[0].clone(), out, out.clone()))
    handles = []
    if how == "hook":
        handles = [m.register_forward_hook(record) for m in linears(dec)]
    elif how == "global":
        handles = [torch.nn.modules.module.register_module_forward_hook(lambda m, a, o: record(m, a, o) if isinstance(m, BitStackLinear) else None)]
    else:
        def forward(self, x):
            out = BitStackLinear.forward(self, x)
            record(self, (x,), out)
            return out
        for m in linears(dec):
            m.forward = types.MethodType(forward, m)
    try:
        dec.prefill(prompt)
    finally:
        for h in handles:
            h.remove()
    assert [m for m, *_ in seen] == linears(dec)
    for m, x, x_then, out, out_then in seen:
        assert torch.equal(out, out_then) and torch.equal(x, x_then)
    # q, k and v alone are summed in another order than as one product: a last bit of fp16 here and there
    rel = lambda a, b: float((a.double() - b.double()).norm() / b.double().norm())
    assert rel(dec.logits, plain.logits) < 2e-3 and rel(dec.kcache, plain.kcache) < 2e-3


def test_a_hook_that_takes_itself_off_keeps_its_tensor():
    dec, seen, handles = decoder(512, 2, 4, 7), [], {}

    def once(mod, args, out):
        seen.append((out, out.clone()))
        handles[mod].remove()
    for m in linears(dec):
        handles[m] = m.register_forward_hook(once)
    dec.prefill(torch.arange(14, device="cuda").view(2, 7))
    assert len(seen) == len(linears(dec)) and all(torch.equal(a, b) for a, b in seen)


def test_a_hook_may_return_another_tensor():
    dec, plain = decoder(512, 2, 4, 12), decoder(512, 2, 4, 12)
    prompt = torch.arange(24, device="cuda").view(2, 12)
    plain.prefill(prompt)
    row = dec.lin[0]
    row[PROJ[1]].register_forward_hook(lambda m, a, o: o.t().contiguous().t())
    row[PROJ[3]].register_forward_hook(lambda m, a, o: torch.cat([o, o], 1)[:, :o.shape[1]])     # rows apart
    row[PROJ[4]].register_forward_hook(lambda m, a, o: o.t().contiguous().t())
    dec.prefill(prompt)
    assert float((dec.logits.double() - plain.logits.double()).norm() / plain.logits.double().norm()) < 5e-3
