"""The tiled decode kernel (layover_amd/csrc/decode_tiles.h) against the float64 oracle: every head_dim
class and its remainders, block sizes that divide a 16-token tile, straddle it and exceed it, one to
many query heads per KV head, each pool and query format, one split and several."""

import numpy as np
import pytest
import torch

from oracle import oracle

pytestmark = pytest.mark.gpu

# head_dim, slots, groups, lengths: class edges (8/32/40/64/72/128/136/256 dims), tiles that end
# inside a block and blocks inside a tile, more than 16 query heads (two chunks), rows of one token, the
# matrix-core kernel's shape with the pools that it does not take (FP32, unaligned records).
SHAPES = [
    (8, 16, 1, [1, 16, 33]),
    (24, 16, 2, [1, 384, 2300]),
    (32, 1, 4, [1, 17, 300]),
    (40, 5, 3, [4, 5, 6, 501]),
    (64, 16, 4, [15, 16, 17, 3000]),
    (64, 32, 8, [1, 31, 32, 4100]),
    (72, 24, 5, [23, 700]),
    (128, 16, 20, [1, 130, 1100]),
    (128, 8, 16, [7, 8, 9, 2050]),
    (128, 16, 4, [33, 3100, 5000]),
    (136, 16, 2, [47, 260]),
    (256, 16, 9, [1, 2100]),
    (256, 64, 1, [63, 64, 65, 900]),
]


def _case(head_dim, slots, groups, lengths, seed):
    rng = np.random.default_rng(seed)
    kv_heads, layers = 2, 3
    width = max(-(-n // slots) for n in lengths)
    blocks = len(lengths) * width
    pool = oracle.bf16_bits(rng.standard_normal((blocks, 2, layers, kv_heads, slots, head_dim), dtype=np.float32))
    table = rng.permutation(blocks).reshape(len(lengths), width).astype(np.int32)
    q = oracle.bf16_bits(rng.standard_normal((len(lengths), kv_heads * groups, head_dim)).astype(np.float32))
    for row, length in enumerate(lengths):  # nothing past a length may be read into the result
        if length % slots:
            pool[table[row, length // slots], :, :, :, length % slots :] = 0x7FC0
    return q, pool, table, np.array(lengths, dtype=np.int32)


def _bf16(bits):
    return torch.from_numpy(bits.view(np.int16)).cuda().view(torch.bfloat16)


def _run(q, pool, table, lens, groups):
    from layover_amd.kernels.hip_decode import paged_decode_attention_hip

    return paged_decode_attention_hip(q, pool, 1, torch.from_numpy(table).cuda(), torch.from_numpy(lens).cuda(), groups).double().cpu().numpy()


@pytest.mark.parametrize("kv", ["bf16", "fp32", "fp8"])
@pytest.mark.parametrize("head_dim,slots,groups,lengths", SHAPES, ids=[f"d{s[0]}s{s[1]}g{s[2]}" for s in SHAPES])
def test_tiled_decode_matches_the_oracle(kv, head_dim, slots, groups, lengths):
    from layover_amd.kernels.hip_decode import Fp8KVPool

    q, bits, table, lens = _case(head_dim, slots, groups, lengths, seed=head_dim + slots)
    if kv == "fp8":
        group, count = slots * head_dim, 2 * 3 * 2
        ids = np.arange(bits.shape[0])
        records = oracle.quantize_records(bits, ids, group, count)
        oracle.dequantize_records(records, ids, bits, group, count)
        pool = Fp8KVPool(torch.from_numpy(records.reshape(len(ids), -1)).cuda(), 3, 2, slots, head_dim)
    else:
        pool = _bf16(bits) if kv == "bf16" else _bf16(bits).float()
    expected = oracle.decode_attention(q, bits, 1, table, lens, groups)
    for q_dtype in (torch.bfloat16, torch.float32):
        if (head_dim, slots, kv) == (128, 16, "bf16") and groups <= 16:
            continue  # decode_split_mfma's
        got = _run(_bf16(q).to(q_dtype), pool, table, lens, groups)
        assert np.isfinite(got).all()
        # The result's own rounding (2^-9 of it in BF16) and FP32 arithmetic: a sum of n terms and a
        # dot product of head_dim ones, each term within 2^-24 of values that are about 1.
        rounding = 2.0**-8 * np.abs(expected) if q_dtype == torch.bfloat16 else 0.0
        allowed = rounding + 2.0**-24 * 4 * (head_dim + 64)
        assert (np.abs(got - expected) <= allowed).all(), (q_dtype, np.abs(got - expected).max())


@pytest.mark.parametrize("exponent", [-130, -100, 100, 118])
def test_tiled_fp8_decode_of_far_shifts_is_exact(exponent):
    """Groups whose shift is far from 0 are decoded with it, as the record format defines."""
    from layover_amd.kernels.hip_decode import Fp8KVPool

    q, bits, table, lens = _case(64, 16, 2, [40, 300], seed=3)
    values = oracle.bf16_to_float(bits)
    values[:, 1] *= np.float32(2.0 ** (exponent // 2)) * np.float32(2.0 ** (exponent - exponent // 2))
    bits = oracle.bf16_bits(np.where(np.isnan(values), 1.0, values).astype(np.float32))
    ids = np.arange(bits.shape[0])
    records = oracle.quantize_records(bits, ids, 1024, 12)
    oracle.dequantize_records(records, ids, bits, 1024, 12)
    pool = Fp8KVPool(torch.from_numpy(records.reshape(len(ids), -1)).cuda(), 3, 2, 16, 64)
    expected = oracle.decode_attention(q, bits, 1, table, lens, 2)
    got = _run(_bf16(q), pool, table, lens, 2)
    # BF16 rounding of the result; below FP32's normals each of the 300 terms may be lost whole.
    scale = np.abs(oracle.bf16_to_float(bits)[:, 1]).max()
    assert (np.abs(got - expected) <= 2.0**-8 * np.abs(expected) + 2.0**-16 * scale + 300 * 2.0**-126).all()


@pytest.mark.parametrize("kv", ["bf16", "fp32"])
@pytest.mark.parametrize("head_dim,slots", [(64, 16), (40, 5), (128, 8), (256, 16)])
def test_tiled_weights_meet_values_of_any_size(kv, head_dim, slots):
    """A weight that underflows to zero hides a V near BF16's largest value, one of about 2^-104 scales a V
    of 2^104 to about 1, and an infinity in a visible row comes out as that infinity, whatever the
    weight it meets."""
    length = 333
    width = -(-length // slots)
    rng = np.random.default_rng(head_dim)
    # All of a token's K equal kappa and q is all ones: scores are kappa sqrt(head_dim), in nats.
    nats = 0.5 * rng.standard_normal(width * slots).astype(np.float32)
    hidden, small, infinite, small_infinite = 40, 100, 200, 310  # tokens
    nats[hidden], nats[small], nats[small_infinite] = -320.0, -72.0, -72.0
    k = np.repeat((nats / np.sqrt(head_dim))[:, None], head_dim, axis=1)
    v = rng.standard_normal((width * slots, head_dim)).astype(np.float32)
    v[hidden] = 2.0**127
    v[small] = 2.0**104
    v[infinite, 0], v[infinite, head_dim - 1] = np.inf, -np.inf
    v[small_infinite, 3] = -np.inf
    pool = np.zeros((width, 2, 3, 2, slots, head_dim), dtype=np.float32)
    for kind, rows in enumerate((k, v)):
        pool[:, kind, 1] = rows.reshape(width, 1, slots, head_dim)
    bits, q = oracle.bf16_bits(pool), oracle.bf16_bits(np.ones((1, 4, head_dim), dtype=np.float32))
    table, lens = np.arange(width, dtype=np.int32).reshape(1, width), np.array([length], dtype=np.int32)
    expected = oracle.decode_attention(q, bits, 1, table, lens, 2)
    assert np.isinf(expected[..., [0, 3, head_dim - 1]]).all() and np.isfinite(np.delete(expected, [0, 3, head_dim - 1], axis=-1)).all()
    got = _run(_bf16(q), _bf16(bits) if kv == "bf16" else _bf16(bits).float(), table, lens, 2)
    infinities = np.isinf(expected)
    assert np.array_equal(got[infinities], expected[infinities])
    # BF16 rounding of the result and FP32 arithmetic as above; the small weight's own error is 2^-24 of
    # its exponent, about 104.
    error, size = np.abs(got[~infinities] - expected[~infinities]), np.abs(expected[~infinities])
    assert (error <= 2.0**-8 * size + 2.0**-24 * 4 * (head_dim + 64)).all(), error.max()


@pytest.mark.parametrize("kv,offset", [("bf16", 2), ("fp32", 1), ("fp8", 4)])
@pytest.mark.parametrize("head_dim,slots,groups", [(24, 16, 2), (64, 16, 4), (128, 8, 16)])
def test_tiled_decode_of_4_byte_aligned_pools_and_queries(kv, offset, head_dim, slots, groups):
    """Pools and queries that start 4 bytes past a 16-byte boundary give the same bits."""
    from layover_amd.kernels.hip_decode import Fp8KVPool

    def shifted(tensor, elements):
        room = torch.empty(tensor.numel() + elements, dtype=tensor.dtype, device="cuda")
        view = room[elements:].view(tensor.shape)
        view.copy_(tensor)
        assert view.data_ptr() % 16 == 4
        return view

    q, bits, table, lens = _case(head_dim, slots, groups, [1, 40, 1300], seed=head_dim)
    if kv == "fp8":
        ids = np.arange(bits.shape[0])
        records = torch.from_numpy(oracle.quantize_records(bits, ids, slots * head_dim, 12).reshape(len(ids), -1)).cuda()
        pools = [Fp8KVPool(r, 3, 2, slots, head_dim) for r in (records, shifted(records, offset))]
    else:
        pool = _bf16(bits) if kv == "bf16" else _bf16(bits).float()
        pools = [pool, shifted(pool, offset)]
    for q_gpu, q_offset in ((_bf16(q), 2), (_bf16(q).float(), 1)):
        expected = _run(q_gpu, pools[0], table, lens, groups)
        assert np.isfinite(expected).all()
        assert np.array_equal(_run(shifted(q_gpu, q_offset), pools[1], table, lens, groups), expected)
