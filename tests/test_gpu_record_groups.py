"""Records of every group size class of the vector record kernels, byte for byte against the oracle:
side-by-side groups that fill their lanes or leave some idle, one to eight loads a lane, more groups than
a wave takes and fewer, stages aligned to 4 bytes only, and values that need the integer codec."""

import numpy as np
import pytest
import torch

from oracle import oracle

pytestmark = pytest.mark.gpu


def _check(group, groups, count, offset, special):
    from layover_amd.kernels import fp8

    rng = np.random.default_rng(group + groups)
    blocks = count + 2
    bits = oracle.bf16_bits((rng.standard_normal((blocks, groups, group)) * 2.0 ** rng.integers(-6, 7, (blocks, groups, 1))).astype(np.float32))
    if special:
        spots = rng.random(bits.shape)
        for low, pattern in ((0.000, 0x7F80), (0.004, 0xFFC1), (0.008, 0x0001), (0.012, 0x8000), (0.016, 0x7F7F), (0.020, 0x0080)):
            bits[(spots >= low) & (spots < low + 0.004) & (rng.random((blocks, groups, 1)) < 0.5)] = pattern
        bits[0, 0] = 0x0003  # a group of subnormals
        bits[1, groups - 1] = 0x0081 + rng.integers(0, 100, group)  # shift below -126
    layout = fp8.Fp8Layout(group, groups)
    ids = rng.permutation(blocks)[:count].astype(np.int32)
    pool = torch.from_numpy(bits.view(np.int16)).cuda().view(torch.bfloat16)
    nbytes = count * layout.record_bytes
    room = torch.full((offset + nbytes + 64,), 0xA5, dtype=torch.uint8, device="cuda")
    stage = room[offset : offset + nbytes + 16]
    fp8.quantize_blocks(pool, torch.from_numpy(ids).cuda(), stage, layout)
    expected = oracle.quantize_records(bits, ids, group, groups)
    assert np.array_equal(stage[:nbytes].cpu().numpy(), expected), (groups, count, offset)
    assert bool((room[:offset] == 0xA5).all()) and bool((room[offset + nbytes :] == 0xA5).all())
    restored = np.full_like(bits, 0x1234)
    target = torch.from_numpy(restored.view(np.int16)).cuda().view(torch.bfloat16)
    fp8.dequantize_blocks(stage, torch.from_numpy(ids).cuda(), target, layout)
    oracle.dequantize_records(expected, ids, restored, group, groups)
    assert np.array_equal(target.view(torch.int16).cpu().numpy().view(np.uint16), restored), (groups, count, offset)


@pytest.mark.parametrize("special", [False, True], ids=["ordinary", "special"])
@pytest.mark.parametrize("group", [8, 24, 32, 128, 248, 256, 384, 504, 512, 520, 1024, 1032, 2040, 2056, 3000, 4096, 4104])
def test_record_group_sizes_are_bit_exact(group, special):
    for groups, count, offset in ((2, 1, 0), (6, 5, 4), (64, 3, 16), (10, 7, 2)):
        _check(group, groups, count, offset, special)


@pytest.mark.parametrize("special", [False, True], ids=["ordinary", "special"])
@pytest.mark.parametrize("group", [8, 24, 104, 128, 248, 256, 384])
def test_many_small_record_groups_are_bit_exact(group, special):
    """Totals around those from which small groups take the vector kernels (4,096 groups; 2^19 values decoding, 2^20
    encoding)."""
    for values, offset in ((4112 * group, 0), (1 << 19, 0), ((1 << 19) + 514 * group, 4), (1 << 20, 4)):
        _check(group, 514, -(-values // (514 * group)), offset, special)
