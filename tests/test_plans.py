"""The host-side choice of kernels, tiles and splits, without a GPU."""
import ctypes
import random

import pytest

import llaisys_amd as L
from llaisys_amd.libllaisys import LIB_LLAISYS

DTS = {"f32": L.DataType.F32, "bf16": L.DataType.BF16, "f16": L.DataType.F16}


# kernels of a prefill: the generic launches, 32- and 16-query MFMA blocks, the vector kernel with 4 and 8
# loads per step
GENERIC, K32, K16, GROUP, GROUP8 = range(5)


def attention_route(seq, total, nh, nkvh, d, int8, dt):
    """(kernel, chunks, keys per chunk, blocks, q heads per block, INT8 cache dequantized first)"""
    out = (ctypes.c_int * 6)()
    LIB_LLAISYS.llaisysTestAttentionRoute(*(ctypes.c_size_t(x) for x in (seq, total, nh, nkvh, d)), int(int8), int(DTS[dt]), out)
    return tuple(out)


@pytest.mark.parametrize("int8", [False, True])
@pytest.mark.parametrize("dt", ["bf16", "f16"])
@pytest.mark.parametrize("d", [64, 128])
def test_prefill_row_offsets_fit_32_bits(d, dt, int8):
    """The prefill kernel addresses the rows of one 1 KB load (512 / head_dim keys) by 32-bit offsets:
    more kv heads than that allows go to the kernel that addresses each row by itself."""
    rows, seq = 512 // d, 2048
    for nkvh in (1, 3, 1 << 12, (1 << 20) + 1, 3 << 20, (1 << 22) - 1, 1 << 22, 6 << 20, 1 << 24):
        if attention_route(seq, seq, nkvh, nkvh, d, int8, dt)[0]:
            assert rows * nkvh * 2 * d < 1 << 32, nkvh
    assert attention_route(seq, seq, 12, 2, d, int8, dt)[0]


# seq, total, nh, nkvh, d, dt: few steps and few heads per kv head, where a 32-query block's fixed cost
# counts, then calls long or wide enough for it
SHORT = [((16, 16, 16, 16, 128, "bf16"), K16, 1), ((100, 100, 32, 8, 128, "bf16"), K16, 2), ((400, 600, 32, 8, 128, "bf16"), K16, 4),
         ((64, 112, 8, 4, 128, "bf16"), K16, 2), ((33, 33, 20, 4, 128, "bf16"), K16, 1), ((16, 16, 16, 16, 64, "bf16"), GROUP, 1),
         ((32, 240, 8, 4, 64, "bf16"), GROUP, 2), ((16, 496, 16, 16, 64, "bf16"), GROUP8, 1), ((16, 16, 4, 4, 128, "f16"), GROUP, 1),
         ((2048, 2048, 12, 2, 128, "bf16"), K32, 2), ((64, 1664, 16, 16, 128, "bf16"), K32, 1), ((400, 400, 16, 16, 128, "bf16"), K32, 1),
         ((100, 100, 16, 16, 64, "bf16"), K32, 1), ((16, 16, 12, 2, 64, "bf16"), K32, 2), ((300, 1500, 12, 2, 128, "f16"), K32, 2)]


@pytest.mark.parametrize("shape, kernel, heads", SHORT)
def test_short_prefills_take_the_faster_kernel(shape, kernel, heads):
    """Measured on both sides of the line; 100 queries of 32 / 8 heads take 8.3 us in blocks of 32 queries and
    6.2 us in blocks of 16."""
    route = attention_route(*shape[:5], False, shape[5])
    assert (route[0], route[4]) == (kernel, heads)


def test_prefill_kernel_and_cut_are_the_same_for_codes():
    """INT8 calls sum as dequantizing and attending does, so they take the same kernel, cut alike."""
    rng = random.Random(2)
    for _ in range(4000):
        nkvh, group = rng.choice([1, 2, 3, 4, 8, 16, 32]), rng.choice([1, 2, 3, 4, 5, 6, 7, 8, 16])
        seq, past = int(16 * 2 ** rng.uniform(0, 8)), rng.choice([0, int(2 ** rng.uniform(0, 15))])
        total = rng.choice([seq + past, max(1, seq // 2)])
        for d in (64, 128):
            for dt in ("bf16", "f16"):
                shape = (seq, total, nkvh * group, nkvh, d)
                assert attention_route(*shape, False, dt)[:5] == attention_route(*shape, True, dt)[:5], (shape, dt)
