"""The host-side choice of kernels, tiles and splits, without a GPU."""
import ctypes

import pytest

import llaisys_amd as L
from llaisys_amd.libllaisys import LIB_LLAISYS

DTS = {"f32": L.DataType.F32, "bf16": L.DataType.BF16, "f16": L.DataType.F16}


def attention_route(seq, total, nh, nkvh, d, int8, dt):
    """(taken by the MFMA prefill, chunks, keys per chunk, blocks)"""
    out = (ctypes.c_int * 4)()
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
