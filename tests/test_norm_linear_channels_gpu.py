"""rms_norm -> projection of one row over more channels than the chip holds waves (two channels per
wave, INT8 weights and plain 16-bit projections): equal to the separate ops bit for bit, with the
last wave's second channel, or all of it, past the end."""
import pytest

from numerics import assert_exact
from test_norm_linear_gpu import Case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", ["bf16", "f16"])
@pytest.mark.parametrize("N, int8, swiglu", [(8193, True, False), (8194, True, True), (8195, True, True), (8193, False, False),
                                             (8198, False, False), (8193, False, True)])
def test_two_channels_per_wave(N, int8, swiglu, dt):
    c = Case(1, 1536, N, dt, int8, swiglu, bias=True, res=True, seed=N)
    got, h = c.fused()
    want, _, h_want = c.composed()
    assert_exact(h, h_want, "residual")
    assert_exact(got, want, f"N={N} int8={int8} swiglu={swiglu}")
