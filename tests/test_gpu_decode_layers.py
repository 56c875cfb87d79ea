"""Decode launches of several layers (LK_DECODE_LAYERS) against one call per layer: the same pool bytes
after the token writes, the same outputs up to the order of the partial sums, for queries packed or
spaced between layers, one split and several, either pool, and a shape that runs layer by layer."""

import pytest
import torch

from layover_amd.kernels import _lib, hip_decode

pytestmark = pytest.mark.gpu

CASES = [
    # lengths, table width, first layer, layers, rows between layers, head_dim, groups
    ([1], 1, 0, 5, 1, 128, 4),
    ([16, 17, 1000], 64, 1, 4, 4, 128, 4),  # one split: written by the split kernel
    ([1023, 1024, 1], 64, 0, 2, 3, 128, 12),  # one split, too many heads for that
    ([3000, 40], 200, 2, 3, 8, 128, 2),
    ([2100] * 9, 132, 0, 5, 9, 128, 8),
    ([300, 31], 20, 1, 3, 2, 64, 4),  # the tiled kernel, layer by layer
]


@pytest.mark.parametrize("kv", ["bf16", "fp8"])
@pytest.mark.parametrize("lengths,width,first,count,rows,dim,groups", CASES, ids=[f"{len(c[0])}x{c[0][0]}d{c[5]}" for c in CASES])
def test_layers_in_one_launch_equal_one_call_per_layer(kv, lengths, width, first, count, rows, dim, groups):
    from layover_amd.kernels import fp8

    batch, layers, heads = len(lengths), 5, 2
    blocks = sum(-(-n // 16) for n in lengths)
    pool = torch.randn(blocks, 2, layers, heads, 16, dim, device="cuda").to(torch.bfloat16)
    if kv == "fp8":
        held = hip_decode.Fp8KVPool.empty(blocks, layers, heads, 16, dim, "cuda")
        fp8.quantize_blocks(pool, torch.arange(blocks, dtype=torch.int32, device="cuda"), held.records, held.layout)
        pool, twin = held, hip_decode.Fp8KVPool(held.records.clone(), layers, heads, 16, dim)
    else:
        twin = pool.clone()
    packed = torch.zeros(batch, 3 + width, dtype=torch.int32)
    ids = torch.randperm(blocks, dtype=torch.int32)
    for b, n in enumerate(lengths):
        mine, ids = ids[: -(-n // 16)], ids[-(-n // 16) :]
        packed[b, 3 : 3 + len(mine)] = mine
        packed[b, :3] = torch.tensor([mine[(n - 1) // 16], (n - 1) % 16, n])
    packed = packed.cuda()
    q = torch.randn(count, rows, heads * groups, dim, device="cuda").to(torch.bfloat16)[:, :batch]
    k, v = (torch.randn(count, rows, heads, dim, device="cuda").to(torch.bfloat16)[:, :batch] for _ in range(2))
    args = (packed[:, 3:], packed[:, 2], groups, packed[:, 0], packed[:, 1])
    together, apart = torch.empty(q.shape, dtype=q.dtype, device="cuda"), torch.empty(q.shape, dtype=q.dtype, device="cuda")
    hip_decode.run_kernel_append_layers(q, pool, first, *args, k, v, together)
    for i in range(count):
        hip_decode.run_kernel_append(q[i].contiguous(), twin, first + i, *args, k[i].contiguous(), v[i].contiguous(), apart[i])
    storage, twin_storage = (p.records if kv == "fp8" else p for p in (pool, twin))
    assert torch.equal(storage.view(torch.uint8), twin_storage.view(torch.uint8))
    # Splits of another size scale and round the weights otherwise: each result is off by at most the
    # weights' relative rounding (2^-17 as a pair of BF16s, 2^-9 as one, for FP8 pools) of the weighted
    # mean of |v|, below 1 here but for rows of a few tokens (N(0, 1) has 0.8), whose 4 at most is
    # allowed for. Then each is rounded to BF16 once.
    a, b = together.double(), apart.double()
    mean_v = torch.tensor([4.0 if n < 100 else 1.0 for n in lengths], device="cuda").view(1, -1, 1, 1)
    allowed = 2.0**-7 * b.abs() + 2 * (2.0**-9 if kv == "fp8" else 2.0**-17) * mean_v
    assert bool(((a - b).abs() <= allowed).all()), float((a - b).abs().max())


def test_layers_that_do_not_exist_are_refused():
    lib = _lib.load()
    shape = _lib.DecodeShape(2, 8, 2, 128, 5, 16, 3, 4, _lib.LK_BF16, _lib.LK_BF16, 0.1, 0, 0, 3 << 8 | 2 << 16)
    assert lib.lk_paged_decode_workspace(shape) == 0  # layers 3, 4 and 5 of 5
    shape.flags = 2 << 8 | 1 << 16  # fewer rows than the batch
    assert lib.lk_paged_decode_workspace(shape) == 0
    shape.flags = 2 << 16  # rows without layers
    assert lib.lk_paged_decode_workspace(shape) == 0
    shape.flags = 2 << 8 | 2 << 16
    assert lib.lk_paged_decode_workspace(shape) > 0
    word = torch.zeros(4, dtype=torch.int32, device="cuda")
    assert lib.lk_paged_decode_static(shape, word.data_ptr(), word.data_ptr(), word.data_ptr(), word.data_ptr(), word.data_ptr(), None) == _lib.LK_ERR_INVALID


def test_padding_rows_are_zero_whatever_batch_came_before():
    """Steps of batches 4, 3, 1, 2 and 3 on one graph set: the padding rows' inputs are zeros in each."""
    from layover_amd.config import ModelConfig
    from layover_amd.kv.decode_graphs import DecodeAttentionGraphs
    from layover_amd.kv.paged_cache import BlockTable, PagedKVCache

    cfg = ModelConfig(num_hidden_layers=2, num_attention_heads=8, num_key_value_heads=2, head_dim=128)
    cache = PagedKVCache(cfg, 12, device="cuda")
    graphs = DecodeAttentionGraphs(cache, 8, sizes=(1, 2, 4), max_tokens=32)
    free = [b for b in range(12) if b not in graphs.scratch_blocks]
    for batch in (4, 3, 1, 2, 3):
        q = torch.randn(2, batch, 8, 128, device="cuda").to(torch.bfloat16)
        k = torch.randn(2, batch, 2, 128, device="cuda").to(torch.bfloat16)
        out = graphs.run([BlockTable(free[i : i + 1], i + 1) for i in range(batch)], q, k, k)
        size = graphs.size_for(batch)
        assert out.shape == (2, batch, 8, 128) and torch.equal(graphs.q[:, :batch], q)
        for buffer in (graphs.q, graphs.k_new, graphs.v_new):
            assert not buffer[:, batch:size].any()
