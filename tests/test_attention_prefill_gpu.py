"""The prefill attention (attnPrefill, attnPrefill16 and short calls on attnGroup) at the edges of its tiles, against the oracle: both
16-bit types, both head dims, cache in the type and in INT8.  Tolerance: assert_attention_close."""
import zlib

import numpy as np
import pytest

import llaisys_amd as L
import oracle
from numerics import _as_f32 as as_f32
from numerics import assert_attention_close, assert_exact
from test_attention_gpu import AMD, DTS, attend, dev, sample

pytestmark = pytest.mark.gpu

# seq, total, nh, nkvh, d: one query block, one key over a step of 128 and over a split of 32, the last
# query block of one query, even and odd groups (two heads / two query blocks per block), keys split
# over blocks (few and many chunks), more queries than keys (the early ones wrap and see every key)
EDGES = [(16, 16, 2, 1, 64), (33, 129, 4, 2, 128), (64, 97, 3, 1, 64), (65, 160, 5, 5, 128), (97, 384, 12, 2, 64),
         (16, 4100, 12, 2, 128), (31, 20000, 3, 3, 64), (300, 200, 4, 2, 128), (130, 100, 3, 1, 64),
         # bf16 on the 16-query kernel: one tile of 64 keys and one key more, an odd count of tiles (one wave set
         # has one less), 1, 2 and 4 heads per block, queries past a block and wrapping queries; then
         # attnGroup with 8 loads per step, and keys split over its blocks
         (16, 64, 5, 1, 128), (17, 65, 8, 1, 128), (48, 129, 2, 2, 128), (270, 300, 32, 8, 128), (100, 60, 8, 2, 128),
         (60, 400, 4, 4, 64), (24, 300, 8, 4, 64), (40, 1100, 2, 1, 64)]


@pytest.mark.parametrize("dt", ["bf16", "f16"])
@pytest.mark.parametrize("shape", EDGES, ids=lambda s: "x".join(map(str, s)))
def test_prefill_tiles(dt, shape):
    seq, total, nh, nkvh, d = shape
    rng = np.random.default_rng(zlib.crc32(repr((dt, shape)).encode()))
    q, k, v = sample(rng, (seq, nh, d), dt), sample(rng, (total, nkvh, d), dt), sample(rng, (total, nkvh, d), dt)
    scale = 1.0 / np.sqrt(d)
    got = attend(q, k, v, scale, dt)
    assert_attention_close(got, oracle.self_attention(q, k, v, scale), v, f"{dt} {shape}")
    assert_exact(attend(q, k, v, scale, dt), got, "repeat")
    # INT8: dequantized into the workspace, or converted in the tiles: the bits of the composition
    (kq, ks), (vq, vs) = oracle.quantize_int8(k), oracle.quantize_int8(v)
    tq, t8 = dev(q, DTS[dt]), [dev(a) for a in (kq, ks, vq, vs)]
    out, ref = (L.Tensor((seq, nh, d), DTS[dt], **AMD) for _ in range(2))
    L.Ops.self_attention_int8kv(out, tq, *t8, scale)
    kd, vd = (L.Tensor((total, nkvh, d), DTS[dt], **AMD) for _ in range(2))
    L.Ops.dequantize_int8_pair(kd, t8[0], t8[1], vd, t8[2], t8[3])
    L.Ops.self_attention(ref, tq, kd, vd, scale)
    assert_exact(out.numpy(), ref.numpy(), "int8 vs dequantize + attend")


@pytest.mark.parametrize("dt", ["bf16", "f16"])
def test_small_weights_keep_their_share(dt):
    """One key with nearly all of the weight and many with 2^-15 of it each: their sum still counts
    (the weights enter the matrix product as two 16-bit parts)."""
    d, total = 64, 1024
    rng = np.random.default_rng(3)
    q = np.zeros((16, 2, d), np.float32)
    q[..., 0] = 1.0
    k = np.zeros((total, 1, d), np.float32)
    k[0, 0, 0] = 15 * np.log(2)
    v = (1 + rng.random((total, 1, d))).astype(np.float32)
    to = {"bf16": lambda x: (x.view(np.uint32) >> 16).astype(np.uint16), "f16": lambda x: x.astype(np.float16)}[dt]
    q, k, v = to(q), to(k), to(v)
    got = attend(q, k, v, 1.0, dt)
    assert_attention_close(got, oracle.self_attention(q, k, v, 1.0), v, dt)


def test_no_alloc_prefill_over_a_split_cache():
    """Keys split over blocks, the caches too large for the fixed scratch beside the partials: the
    codes are converted in the tiles, with the bits of the allocating entry point."""
    seq, total, nh, nkvh, d = 40, 30000, 12, 2, 128
    rng = np.random.default_rng(9)
    q, k, v = sample(rng, (seq, nh, d), "bf16"), sample(rng, (total, nkvh, d), "bf16"), sample(rng, (total, nkvh, d), "bf16")
    (kq, ks), (vq, vs) = oracle.quantize_int8(k), oracle.quantize_int8(v)
    tq, t8 = dev(q, DTS["bf16"]), [dev(a) for a in (kq, ks, vq, vs)]
    out, ref = (L.Tensor((seq, nh, d), DTS["bf16"], **AMD) for _ in range(2))
    L.Ops.self_attention_int8kv(ref, tq, *t8, 0.0883883)
    L.Ops.self_attention_int8kv_noalloc(out, tq, *t8, 0.0883883)
    assert_exact(out.numpy(), ref.numpy(), "no alloc")


def _bits(x, dt):
    """f32 values (infinities and NaN among them) in the storage type."""
    x = np.float32(x)
    return {"bf16": lambda: np.uint16(x.view(np.uint32) >> 16), "f16": lambda: np.float16(x), "f32": lambda: x}[dt]()


def visible_attention(q, k, v, scale):
    """The oracle over each query's own keys alone."""
    seq, total = q.shape[0], k.shape[0]
    rows = [oracle.self_attention(q[i:i + 1], k[:total - seq + i + 1], v[:total - seq + i + 1], scale) for i in range(seq)]
    return np.concatenate(rows)


# seq, total, nh, nkvh: the diagonal within one step, rows past the cache in a part-filled tile, an odd
# group's two query blocks, and keys split over blocks
NON_FINITE = [(40, 40, 4, 2), (33, 201, 3, 1), (40, 200, 12, 2), (40, 1100, 2, 1)]


@pytest.mark.parametrize("int8", [False, True], ids=["plain", "int8"])
@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("dt", ["bf16", "f16"])
@pytest.mark.parametrize("shape", NON_FINITE, ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("value", [np.inf, -np.inf, np.nan])
def test_non_finite_v_reaches_only_queries_that_see_it(value, shape, dt, d, int8):
    """An infinite or NaN V element of a later token leaves earlier queries as they were (the tiles hold
    keys that a query does not see), and an infinite one that is seen gives an infinity, not NaN."""
    seq, total, nh, nkvh = shape
    rng = np.random.default_rng(zlib.crc32(repr((shape, dt, d)).encode()))
    q, k, v = sample(rng, (seq, nh, d), dt), sample(rng, (total, nkvh, d), dt), sample(rng, (total, nkvh, d), dt)
    scale = float(np.float32(1.0 / np.sqrt(d)))
    late = total - seq // 2  # seen by the second half of the queries
    if int8:
        (kq, ks), (vq, vs) = oracle.quantize_int8(k), oracle.quantize_int8(v)
        vs[late, 0] = value  # the whole row, zero codes NaN
        k, v = (oracle.dequantize_int8(c, s, q.dtype) for c, s in ((kq, ks), (vq, vs)))
    else:
        v[late, 0, [3, d - 1]] = _bits(value, dt)
        v[0, nkvh - 1, 17] = _bits(value, dt)  # what rows past the cache are read from
    want = visible_attention(q, k, v, scale)
    tq, out = dev(q, DTS[dt]), L.Tensor((seq, nh, d), DTS[dt], **AMD)
    if int8:
        L.Ops.self_attention_int8kv(out, tq, *(dev(a) for a in (kq, ks, vq, vs)), scale)
        got = out.numpy()
    else:
        got = attend(q, k, v, scale, dt)
    finite = np.where(np.isfinite(as_f32(v)), v, np.zeros_like(v))  # for the tolerance's max |v|
    assert_attention_close(got, want, finite, f"{dt} {shape} d{d}")
    got, want = as_f32(got), as_f32(want)
    assert_exact(np.where(np.isinf(got), got, 0), np.where(np.isinf(want), want, 0), "infinities")


# seq, total, nh, nkvh, d: prefill in one piece and with the keys split over few and many blocks, decode
# in one piece and split, head_dim 64, and one that the scalar kernel takes
BAD_SCORES = [(40, 40, 4, 2, 128), (33, 1100, 3, 1, 64), (16, 9000, 2, 1, 128), (5, 40, 4, 2, 128), (2, 3000, 12, 2, 128),
              (3, 700, 4, 2, 64), (7, 40, 4, 2, 24)]


@pytest.mark.parametrize("dt", ["bf16", "f16", "f32"])
@pytest.mark.parametrize("shape", BAD_SCORES, ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("value", [np.inf, np.nan])
def test_non_finite_k_gives_nan_where_the_reference_does(value, shape, dt):
    """A NaN or +Inf score makes its query's output NaN (not 0), a -Inf score weighs nothing, and
    queries before the key are as they were, whether or not the keys are split over blocks."""
    seq, total, nh, nkvh, d = shape
    rng = np.random.default_rng(zlib.crc32(repr((shape, dt)).encode()))
    q, k, v = sample(rng, (seq, nh, d), dt), sample(rng, (total, nkvh, d), dt), sample(rng, (total, nkvh, d), dt)
    k[total - (seq + 1) // 2, 0, 9] = _bits(value, dt)
    scale = 1.0 / np.sqrt(d)
    assert_attention_close(attend(q, k, v, scale, dt), visible_attention(q, k, v, scale), v, f"{dt} {shape}")
