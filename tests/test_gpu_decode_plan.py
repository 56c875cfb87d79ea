"""Decode on both sides of the one-split rule, with rows much shorter than the table and full ones, against
FP64 attention in torch: the split kernel's own output for batches that fill the GPU, and splits whose
sizes are no power of two."""

import math

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kv", ["bf16", "fp8"])
@pytest.mark.parametrize("batch,width", [(1, 16), (1, 17), (5, 13), (12, 44), (24, 112), (23, 112), (24, 113), (3, 375), (70, 90), (65, 30), (97, 33), (130, 60), (260, 66)])
def test_decode_across_the_split_plan(batch, width, kv):
    from layover_amd.kernels import fp8, hip_decode

    heads, groups, layers = 8, 4, 1
    lengths = [width * 16] + [1 + (i * 7919) % (width * 16) for i in range(batch - 1)]
    blocks = sum(-(-n // 16) for n in lengths)
    pool = torch.randn(blocks, 2, layers, heads, 16, 128, device="cuda").to(torch.bfloat16)
    read = pool
    if kv == "fp8":
        read = hip_decode.Fp8KVPool.empty(blocks, layers, heads, 16, 128, "cuda")
        ids = torch.arange(blocks, dtype=torch.int32, device="cuda")
        fp8.quantize_blocks(pool, ids, read.records, read.layout)
        fp8.dequantize_blocks(read.records, ids, pool, read.layout)
    order, table = torch.randperm(blocks, dtype=torch.int32), torch.zeros(batch, width, dtype=torch.int32)
    at = 0
    for row, n in enumerate(lengths):
        mine = order[at : at + -(-n // 16)]
        at += len(mine)
        table[row, : len(mine)] = mine
    q = torch.randn(batch, heads * groups, 128, device="cuda").to(torch.bfloat16)
    out = hip_decode.paged_decode_attention_hip_trusted(q, read, 0, table.cuda(), torch.tensor(lengths, dtype=torch.int32, device="cuda"), groups)
    for row, n in enumerate(lengths):
        k, v = (pool[:, kind, 0].index_select(0, table[row, : -(-n // 16)].long().cuda()).permute(1, 0, 2, 3).reshape(heads, -1, 128)[:, :n].double()
                for kind in (0, 1))
        scores = (q[row].double().view(heads, groups, 128) @ k.transpose(1, 2).contiguous()) / math.sqrt(128)
        weights = torch.softmax(scores, dim=-1)
        expected, mean_v = weights @ v, weights @ v.abs()
        # BF16 rounding of the result; FP8 pools round each weight to BF16 too.
        allowed = 2.0**-8 * expected.abs() + (2.0**-8 * mean_v if kv == "fp8" else 0.0) + 1e-4
        error = (out[row].double().view(heads, groups, 128) - expected).abs()
        assert bool((error <= allowed).all()), (row, n, float(error.max()))
