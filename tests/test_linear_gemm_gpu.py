"""The tiled linear kernels (linear_gemm.hip) at the edges of their tiles and of their split of K,
against the oracle's restatement of the reference linear.  Tolerance: numerics.assert_linear_close."""
import threading
import zlib

import numpy as np
import pytest

import llaisys_amd as L
import oracle
from numerics import assert_exact, assert_linear_close
from test_linear_gpu import AMD, DTS, dev, linear, sample

pytestmark = pytest.mark.gpu

# rows, in_features, out_features: row tiles of 32 / 64 / 128 and one more, channel tiles of 64
# and one less / more, K of one chunk, one stage, a ragged last stage, and split over blocks
F32_EDGES = [(2, 4, 1), (32, 32, 64), (33, 36, 65), (64, 1536, 63), (65, 100, 130), (128, 4100, 66),
             (129, 1540, 31), (5, 8960, 257), (1, 8964, 33), (1, 1540, 70)]


@pytest.mark.parametrize("shape", F32_EDGES, ids=lambda s: "x".join(map(str, s)))
def test_f32_tiles(shape):
    rows, in_f, out_f = shape
    rng = np.random.default_rng(zlib.crc32(repr(shape).encode()))
    x, w, b = (sample(rng, s, "f32", sc) for s, sc in (((rows, in_f), 1.0), ((out_f, in_f), 0.05), ((out_f,), 1.0)))
    got = linear(x, w, b, "f32")
    assert_linear_close(got, oracle.linear(x, w, b), x, w, f"f32 {shape}")
    assert_exact(linear(x, w, b, "f32"), got, "repeat")


def test_split_k_under_capture_without_workspace(monkeypatch):
    """A linear that would split K, captured where the scratch may not grow, runs unsplit."""
    monkeypatch.setenv("LLAISYS_GRAPH_WORKSPACE_BYTES", "0")
    rng = np.random.default_rng(5)
    x, w = sample(rng, (8, 8960), "f32"), sample(rng, (1024, 8960), "f32", 0.05)
    zeros, errors = np.zeros((8, 1024), np.float32), []

    def body():  # a fresh thread: its own scratch, not grown yet
        try:
            tx, tw, out = dev(x), dev(w), L.Tensor((8, 1024), DTS["f32"], **AMD)
            graph = L.Graph.capture()
            L.Ops.linear(out, tx, tw)
            graph.end()
            linear(x, w, None, "f32")  # eager, split: the scratch grows beside the graph
            for _ in range(3):
                out.load(zeros.ctypes.data)
                graph.launch()
                L.RuntimeAPI(L.DeviceType.AMD).device_synchronize()
                assert_linear_close(out.numpy(), oracle.linear(x, w, None), x, w, "captured")
        except BaseException as e:  # re-raised in the test thread
            errors.append(e)

    th = threading.Thread(target=body)
    th.start()
    th.join()
    if errors:
        raise errors[0]
