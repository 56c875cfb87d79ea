"""The generic decode kernel (decode_split_generic) against the float64 oracle: head_dims that are no
multiple of 8, and pools, records and queries too loosely aligned for the matrix-core kernels; each pool
and query format, blocks of few and many slots, one split and several, runs of tokens that leave waves
without any."""

import numpy as np
import pytest
import torch

from oracle import oracle

pytestmark = pytest.mark.gpu

LAYERS, HEADS = 3, 2
# head_dim, slots, groups, lengths, whether in several splits; pools of the last shapes start one element past alignment.
SHAPES = [
    (31, 16, 4, [1, 3, 17, 3000], True),
    (31, 7, 1, [2, 500], True),
    (31, 7, 1, [2, 63], False),
    (255, 16, 2, [30, 64], False),
    (100, 16, 4, [5, 700, 2049], True),
    (100, 200, 2, [199, 200, 201, 1500], True),
    (255, 4, 3, [9, 1333], True),
    (64, 16, 4, [4, 1300], True),
    (128, 16, 4, [33, 1300], True),
    (128, 16, 8, [7, 200], False),
]


def _moved(tensor, elements):
    room = torch.empty(tensor.numel() + elements, dtype=tensor.dtype, device="cuda")
    view = room[elements:].view(tensor.shape)
    view.copy_(tensor)
    return view


@pytest.mark.parametrize("kv", ["bf16", "fp32", "fp8"])
@pytest.mark.parametrize("head_dim,slots,groups,lengths,several", SHAPES, ids=[f"d{s[0]}s{s[1]}x{s[3][-1]}" for s in SHAPES])
def test_generic_decode_matches_the_oracle(kv, head_dim, slots, groups, lengths, several):
    from layover_amd.kernels.hip_decode import Fp8KVPool, decode_shape, paged_decode_attention_hip, workspace_bytes

    rng = np.random.default_rng(head_dim + slots)
    width = max(-(-n // slots) for n in lengths)
    blocks = len(lengths) * width
    bits = oracle.bf16_bits(rng.standard_normal((blocks, 2, LAYERS, HEADS, slots, head_dim), dtype=np.float32))
    table = rng.permutation(blocks).reshape(len(lengths), width).astype(np.int32)
    q = oracle.bf16_bits(rng.standard_normal((len(lengths), HEADS * groups, head_dim)).astype(np.float32))
    for row, length in enumerate(lengths):  # nothing past a length may be read into the result
        if length % slots:
            bits[table[row, length // slots], :, :, :, length % slots :] = 0x7FC0
    odd = head_dim % 8 == 0  # a shape of the matrix-core kernels, at an address they do not take
    if kv == "fp8":
        group, count, ids = slots * head_dim, 2 * LAYERS * HEADS, np.arange(blocks)
        records = oracle.quantize_records(bits, ids, group, count)
        oracle.dequantize_records(records, ids, bits, group, count)
        rows = torch.from_numpy(records.reshape(blocks, -1)).cuda()
        pool = Fp8KVPool(_moved(rows, 1) if odd else rows, LAYERS, HEADS, slots, head_dim)
    else:
        pool = torch.from_numpy(bits.view(np.int16)).cuda().view(torch.bfloat16)
        pool = pool.float() if kv == "fp32" else pool
        pool = _moved(pool, 1) if odd and kv == "bf16" else pool
    expected = oracle.decode_attention(q, bits, 1, table, np.array(lengths, dtype=np.int32), groups)
    table_gpu, lens_gpu = torch.from_numpy(table).cuda(), torch.tensor(lengths, dtype=torch.int32, device="cuda")
    for q_dtype in (torch.bfloat16, torch.float32):
        if odd and kv == "fp32" and q_dtype == torch.float32:
            continue  # four bytes suffice the tiled kernel
        q_gpu = torch.from_numpy(q.view(np.int16)).cuda().view(torch.bfloat16).to(q_dtype)
        if odd and q_dtype == torch.bfloat16:
            q_gpu = _moved(q_gpu, 1)
        shape = decode_shape(q_gpu, pool, 1, table_gpu, groups, lens_gpu)
        assert (workspace_bytes(shape) > len(lengths) * HEADS * groups * (head_dim + 2) * 4) == several
        got = paged_decode_attention_hip(q_gpu, pool, 1, table_gpu, lens_gpu, groups).double().cpu().numpy()
        assert np.isfinite(got).all()
        # The result's own rounding (2^-9 of it in BF16) and FP32 arithmetic: a sum of n terms and a
        # dot product of head_dim ones, each term within 2^-24 of values that are about 1.
        rounding = 2.0**-8 * np.abs(expected) if q_dtype == torch.bfloat16 else 0.0
        allowed = rounding + 2.0**-24 * 4 * (head_dim + 64)
        assert (np.abs(got - expected) <= allowed).all(), (q_dtype, np.abs(got - expected).max())
