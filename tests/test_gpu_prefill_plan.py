"""Prefill chunks on both sides of the split plan's lines, against FP32 attention in torch: tiles that
do not fill the GPU unsplit (their heavy tiles divided between workgroups that may sit on different
CUs), ragged last tiles, two to many splits; scores that keep raising the running maximum."""

import math

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("gain", [1.0, 6.0])
@pytest.mark.parametrize("kv", ["bf16", "fp8"])
@pytest.mark.parametrize("tokens,start", [(17, 0), (391, 0), (1300, 0), (1900, 300), (1000, 1000), (1024, 4096), (64, 4000), (33, 9001)])
def test_chunks_across_the_split_plan(tokens, start, kv, gain):
    from layover_amd.kernels import fp8, hip_decode
    from layover_amd.kernels.hip_prefill import paged_prefill_attention_hip

    heads, groups, layers = 8, 4, 2
    blocks = -(-(start + tokens) // 16)
    pool = torch.randn(blocks, 2, layers, heads, 16, 128, device="cuda").to(torch.bfloat16)
    # Later keys score higher, so that the maximum is raised all along the walk.
    pool[:, 0] *= torch.linspace(0.3, gain, blocks, device="cuda").to(torch.bfloat16).view(-1, 1, 1, 1, 1)
    order = torch.randperm(blocks, device="cuda")
    held = torch.empty_like(pool)
    held[order] = pool
    read = held
    if kv == "fp8":
        read = hip_decode.Fp8KVPool.empty(blocks, layers, heads, 16, 128, "cuda")
        ids = torch.arange(blocks, dtype=torch.int32, device="cuda")
        fp8.quantize_blocks(held, ids, read.records, read.layout)
        fp8.dequantize_blocks(read.records, ids, held, read.layout)
        pool = held[order]
    q = torch.randn(heads * groups, tokens, 128, device="cuda").to(torch.bfloat16)
    out = paged_prefill_attention_hip(q, read, 1, order.to(torch.int32), start, groups)
    again = paged_prefill_attention_hip(q, read, 1, order.to(torch.int32), start, groups)
    assert torch.equal(out, again)
    k, v = (pool[:, kind, 1].permute(1, 0, 2, 3).reshape(heads, -1, 128)[:, : start + tokens].double() for kind in (0, 1))
    seen = torch.arange(start + tokens, device="cuda")[None, :] <= torch.arange(start, start + tokens, device="cuda")[:, None]
    for head in range(heads):
        kt = k[head].t().contiguous()
        for h in range(head * groups, (head + 1) * groups):
            weights = torch.softmax((q[h].double() @ kt / math.sqrt(128)).masked_fill(~seen, -math.inf), dim=-1)
            expected, mean_v = weights @ v[head], weights @ v[head].abs()
            # The result's rounding to BF16, and each weight's (2^-9 of the weighted mean of |v|).
            allowed = 2.0**-8 * expected.abs() + 2.0**-8 * mean_v + 1e-4
            assert bool(((out[h].double() - expected).abs() <= allowed).all()), (h, float((out[h].double() - expected).abs().max()))
