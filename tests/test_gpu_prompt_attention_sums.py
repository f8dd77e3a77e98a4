"""The softmax denominator of the prompt pass's attention is the fp32 sum of the fp32 weights.  Weights of one size, whose roundings to fp16 all err the same way, show it: the sum of
the rounded ones is up to 2^-11 of itself away, which is more than the one rounding of the result."""
import math

import pytest
import torch

from bitstack_amd.utils import inference_utils as IU

D, N_POS = 128, 512


def half(v):
    return torch.tensor(v, dtype=torch.float64).half().double().item()


def ulp(v):
    return 2.0 ** (math.floor(math.log2(v)) - 10)


def bound(want, i):
    # the result's rounding to fp16; a weight's base-2 exponent, up to 8, is rounded three times (2^-24 of it each, ln 2 of that in the weight) and the
    # exponential once; i + 1 weights added in fp32 in whatever order
    return 0.5 * ulp(want) + want * (3 * 8 * 2.0 ** -24 + (i + 2) * 2.0 ** -24)


def cases():
    """{i: a}: query i scores -a / sqrt(128) against positions 1 .. i and 0 against position 0, whose v is 1 where the others' is 0, so its result is 1 / (1 + i p).  The ones where
    the rounded weights' sum would end beyond the bound."""
    found = {}
    for k in range(16 * 8, 16 * 56):
        a = k / 16                                   # (an fp16 number)
        p = math.exp(-a / math.sqrt(D))
        for i in range(16 + k % 16, N_POS, 16):
            want = 1.0 / (1.0 + i * p)
            if abs(half(1.0 / (1.0 + i * half(p))) - want) > bound(want, i) + 0.1 * ulp(want):
                found[i] = a
    return found


def test_there_are_cases():
    assert len(cases()) >= 200


@pytest.mark.gpu
@pytest.mark.parametrize("B,heads,kv", [(1, 4, 2), (4, 64, 16)])               # 16 and 32 queries per wave
def test_the_denominator_is_the_sum_of_the_weights(B, heads, kv):
    print(f"prompt attention sums B={B} heads={heads}", flush=True)
    q, k, v = torch.zeros(B, N_POS, heads, D), torch.zeros(B, kv, N_POS, D), torch.zeros(B, kv, N_POS, D)
    k[:, :, 1:, 0] = -1.0
    v[:, :, 0, 0] = 1.0
    for i, a in cases().items():
        q[:, i, :, 0] = a
    q, k, v = (t.half().cuda() for t in (q.view(B * N_POS, heads * D), k, v))
    out = IU.attention_prefill_hip(q, k, v, N_POS).double().cpu().view(B, N_POS, heads, D)
    for i, a in cases().items():
        want = 1.0 / (1.0 + i * math.exp(-a / math.sqrt(D)))
        assert bool(((out[:, i, :, 0] - want).abs() <= bound(want, i)).all()), (i, a)
