"""The tiled linear kernels (linear_gemm.hip) at the edges of their tiles and of their split of K,
against the oracle's restatement of the reference linear.  Tolerance: numerics.assert_linear_close."""
import ctypes
import threading
import zlib

import numpy as np
import pytest

import llaisys_amd as L
import oracle
from llaisys_amd.hostfmt import f32_to_bf16
from llaisys_amd.libllaisys import LIB_LLAISYS
from numerics import assert_exact, assert_linear_close
from test_norm_linear_gpu import Case
from test_linear_gpu import AMD, DTS, dev, int8_weights, linear, linear_w8a16, sample

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


# rows, in_features, out_features through the public calls: the 64-row tile with its deep stages (first and
# last row count, K of one chunk pair, a ragged last stage, split), then what the expected launch time
# picks as the rows grow, mostly 64 x 64 tiles, split and not, and larger ones over a few stages, with
# ragged channels or rows (test_each_tile has every tile over many stages)
EDGES = [(17, 16, 64), (64, 144, 63), (37, 1552, 130), (64, 8960, 66), (65, 16, 65), (96, 208, 300), (128, 8960, 192),
         (161, 1552, 2000), (300, 4112, 140), (300, 64, 9002), (800, 80, 9001), (1024, 2064, 770), (1500, 96, 1531),
         (2047, 48, 9003), (3999, 112, 1540), (2048, 64, 18000)]


@pytest.mark.parametrize("dt", ["bf16", "f16"])
@pytest.mark.parametrize("shape", EDGES, ids=lambda s: "x".join(map(str, s)))
def test_16_bit_tiles(shape, dt):
    """Dense against the oracle, and W8A16 with unit scales over the same codes bit for bit (one
    order of the sums); W8A16 with scales and bias against the oracle."""
    rows, in_f, out_f = shape
    rng = np.random.default_rng(zlib.crc32(repr((shape, dt)).encode()))
    x, b = sample(rng, (rows, in_f), dt), sample(rng, (out_f,), dt)
    codes, scale = int8_weights(rng, out_f, in_f)
    w = f32_to_bf16(codes.astype(np.float32)) if dt == "bf16" else codes.astype(np.float16)
    some = slice(None) if rows * in_f * out_f < 1 << 30 else np.r_[:70, rows // 2:rows // 2 + 140, rows - 70:rows]
    xs = x[some]
    got = linear(x, w, b, dt)
    assert_linear_close(got[some], oracle.linear(xs, w, b), xs, w, f"{dt} {shape}")
    assert_exact(linear_w8a16(x, codes, np.ones(out_f, np.float32), b, dt), got, "unit scales")
    assert_linear_close(linear_w8a16(x, codes, scale, b, dt)[some], oracle.linear_w8a16(xs, codes, scale, b), xs, codes,
                        f"w8a16 {dt} {shape}", w_scale=scale)


@pytest.mark.parametrize("dt", ["bf16", "f16", "f32"])
@pytest.mark.parametrize("rows, in_f, out_f", [(2, 64, 100), (3, 1536, 2000), (16, 4112, 4100), (5, 272, 33),
                                               (17, 528, 90), (64, 2064, 33), (100, 1536, 131), (300, 528, 1000),
                                               (1100, 144, 4500)])
def test_swiglu_epilogue_equals_separate_ops(rows, in_f, out_f, dt):
    """rms_norm -> gate / up -> swiglu with the swiglu in the linear's epilogue (or in its split
    reduction) equals the three ops on the two halves of the weight, bit for bit."""
    for int8 in (False, True):
        if int8 and (dt == "f32" or in_f % 16):
            continue
        c = Case(rows, in_f, out_f, dt, int8, True, bias=True, res=True, seed=rows)
        got, h = c.fused()
        want, _, h_want = c.composed()
        assert_exact(h, h_want, "residual")
        assert_exact(got, want, f"int8={int8}")


# GemmTile: weight rows, activation rows and k per stage; the 256 x 128 tile is for INT8 weights only, and
# dense weights take 192 x 256 in stages of 32
TILES = {"64x64deep": (0, 64, 64, 128), "64x64": (1, 64, 64, 64), "128x64": (2, 128, 64, 64), "128x128": (3, 128, 128, 64),
         "192x128": (4, 192, 128, 64), "256x128": (5, 256, 128, 64), "192x256": (6, 192, 256, 64)}
# stages of the tile's k, what the last one lacks, splits: fewer stages than the ring of LDS tiles holds (2 to
# 5), as many, one more, odd and even counts beyond; ranges of K that start past 0, the last one short
STAGES = [(1, 48, 1), (2, 0, 1), (3, 16, 1), (4, 0, 1), (5, 32, 1), (8, 0, 1), (9, 16, 1), (4, 16, 2), (9, 0, 2), (19, 48, 3)]


def on_tile(tile, x, w, scale, bias, dt, swiglu, splits, ws):
    """The rows of x through `tile`, K in `splits` ranges (llaisysTestLinearTile)."""
    n = w.shape[0] // 2 if swiglu else w.shape[0]
    tx, tw, out = dev(x, DTS[dt]), dev(w, None if scale is not None else DTS[dt]), L.Tensor((x.shape[0], n), DTS[dt], **AMD)
    ts, tb = None if scale is None else dev(scale), None if bias is None else dev(bias, DTS[dt])
    ptr = lambda t: ctypes.c_void_p(None if t is None else t.data_ptr())
    got = LIB_LLAISYS.llaisysTestLinearTile(ptr(out), ptr(tx), ptr(tw), ptr(ts), ptr(tb), *(ctypes.c_size_t(v) for v in (*x.shape, n)),
                                            int(swiglu), int(DTS[dt]), tile, ctypes.c_size_t(splits), ptr(ws),
                                            ctypes.c_size_t(ws.shape()[0] * 4))
    assert got == splits, (tile, got)
    return out.numpy()


@pytest.mark.parametrize("dt", ["bf16", "f16"])
@pytest.mark.parametrize("int8", [False, True], ids=["dense", "int8"])
@pytest.mark.parametrize("name", TILES)
def test_each_tile(name, int8, dt):
    """Every tile against the oracle, and its swiglu epilogue (in the tile, or in the sum over splits) bit
    for bit against the two halves on the same tile."""
    tile, bw, bx, ks = TILES[name]
    if name == "256x128" and not int8:
        return
    rng = np.random.default_rng(zlib.crc32(repr((name, int8, dt)).encode()))
    ws = L.Tensor((8 << 20,), DTS["f32"], **AMD)
    for stages, lacks, splits in STAGES:
        rows, n, k = bx + int(rng.integers(1, 40)), bw + 2 * int(rng.integers(1, 40)), stages * ks - lacks
        x, b = sample(rng, (rows, k), dt), sample(rng, (2 * n,), dt)
        what = f"{name} {rows}x{k}x{n} / {splits}"
        if int8:
            w, scale = int8_weights(rng, 2 * n, k)
            gate, up = ((w[h], scale[h], b[h]) for h in (slice(n), slice(n, None)))
            want = oracle.linear_w8a16(x, *gate)
        else:
            w, scale = sample(rng, (2 * n, k), dt, 0.05), None
            gate, up = ((w[h], None, b[h]) for h in (slice(n), slice(n, None)))
            want = oracle.linear(x, gate[0], gate[2])
        y = [on_tile(tile, x, *half, dt, False, splits, ws) for half in (gate, up)]
        assert_linear_close(y[0], want, x, gate[0], what, **({"w_scale": gate[1]} if int8 else {}))
        out = L.Tensor((rows, n), DTS[dt], **AMD)
        L.Ops.swiglu(out, dev(y[0], DTS[dt]), dev(y[1], DTS[dt]))
        assert_exact(on_tile(tile, x, w, scale, b, dt, True, splits, ws), out.numpy(), "swiglu " + what)


def in_new_thread(body):
    """body() in a thread of its own: its own scratch, not grown yet"""
    result, errors = [], []

    def run():
        try:
            result.append(body())
        except BaseException as e:  # re-raised in the test thread
            errors.append(e)

    th = threading.Thread(target=run)
    th.start()
    th.join()
    if errors:
        raise errors[0]
    return result[0]


def test_scratch_grows_by_half_at_least():
    """Prompts of a row more each find the scratch grown a few times, not at every one (a growth waits for
    the device)."""
    size = LIB_LLAISYS.llaisysTestWorkspaceBytes
    size.restype = ctypes.c_size_t

    def body():
        x, w = dev(np.zeros((64, 8960), np.float16)), dev(np.zeros((1536, 8960), np.float16))
        sizes = set()
        for rows in range(17, 65):
            L.Ops.linear(L.Tensor((rows, 1536), DTS["f16"], **AMD), x.slice(0, 0, rows), w)
            sizes.add(size(0))
        L.RuntimeAPI(L.DeviceType.AMD).device_synchronize()
        return sizes

    sizes = in_new_thread(body)
    assert 1 < len(sizes) <= 5, sizes


@pytest.mark.parametrize("dt", ["bf16", "f32"])
def test_split_k_is_the_same_in_a_graph(monkeypatch, dt):
    """With the scratch a capture reserves by itself a linear splits as it does outside; with room for its
    own partial sums but not for those of gate and up in one launch, neither that launch nor the
    linear on one half splits."""
    rng = np.random.default_rng(6)
    rows, in_f, out_f = 64, 8960, 512
    x, w = sample(rng, (rows, in_f), dt), sample(rng, (out_f, in_f), dt, 0.05)

    def captured(reserve):
        if reserve is None:
            monkeypatch.delenv("LLAISYS_GRAPH_WORKSPACE_BYTES", raising=False)
        else:
            monkeypatch.setenv("LLAISYS_GRAPH_WORKSPACE_BYTES", str(reserve))
        tx, tw, out = dev(x, DTS[dt]), dev(w, DTS[dt]), L.Tensor((rows, out_f), DTS[dt], **AMD)
        graph = L.Graph.capture()
        L.Ops.linear(out, tx, tw)
        graph.end()
        for _ in range(2):
            graph.launch()
            L.RuntimeAPI(L.DeviceType.AMD).device_synchronize()
        return out.numpy()

    eager = in_new_thread(lambda: linear(x, w, None, dt))
    assert_exact(in_new_thread(lambda: captured(None)), eager, "default reserve")
    unsplit = in_new_thread(lambda: captured(0))
    assert not np.array_equal(unsplit, eager)  # a shape that splits, seen in its bits
    own = 32 * rows * out_f * 4
    assert_exact(in_new_thread(lambda: captured(own)), unsplit, "its own partial sums only")


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
