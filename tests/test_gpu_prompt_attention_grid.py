"""The prompt pass's attention takes as many sequences as memory holds: more workgroups than one grid may have along x become several launches."""
import pytest
import torch

from bitstack_amd.utils import inference_utils as IU


@pytest.mark.gpu
def test_more_sequences_than_a_grid_holds():
    B, heads = (1 << 24) // 32 + 3, 32               # 2^24 workgroups of 256 threads are one grid too many
    print(f"prompt attention B={B} heads={heads}", flush=True)
    q, k = (torch.ones(1, device="cuda", dtype=torch.half).expand(B * heads * 128).contiguous() for _ in range(2))
    v = torch.randint(-(1 << 15), 1 << 15, (B, heads, 1, 128), dtype=torch.int16, device="cuda") & 0x3FFF       # (positive fp16 numbers below 2)
    out = IU.attention_prefill_hip(q.view(B, heads * 128), k.view(B, heads, 1, 128), v.view(torch.half), 1)
    assert torch.equal(out.view(torch.int16), v.view(B, heads * 128))     # one position: its v
