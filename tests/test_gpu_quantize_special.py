"""bfloat16 blocks with infinities, NaNs and subnormals beside ordinary values: the packed
route of finite blocks and the float route of the others give the bits of the float32
quantizer on the same values, along rows and columns, in 1x32 blocks and 32x32 tiles."""

import pytest
import torch

from tests._util import announce

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tiles", [False, True])
@pytest.mark.parametrize("kind", ["inf", "nan", "both", "subnormal", "largest"])
def test_special_blocks_are_the_float32_quantizers(lib, kind, tiles):
    from bux_amd import grouped_mxfp8
    g = torch.Generator(device="cuda").manual_seed(110)
    x = torch.randn(160, 96, generator=g, device="cuda").to(torch.bfloat16)
    at = torch.rand(x.shape, generator=g, device="cuda")
    if kind in ("inf", "both"):
        x[at < 0.01] = torch.inf
        x[at > 0.99] = -torch.inf
    if kind in ("nan", "both"):
        x[(at > 0.5) & (at < 0.51)] = torch.nan
    if kind == "subnormal":
        x = (x * 2.0**-130).to(torch.bfloat16)
    if kind == "largest":
        x[at < 0.05] = torch.finfo(torch.bfloat16).max
    announce("special blocks", kind, tiles)
    got = grouped_mxfp8.quantized_twice(x, tiles=tiles)
    want = grouped_mxfp8.quantized_twice(x.float(), tiles=tiles)
    torch.cuda.synchronize()
    for a, b in zip(got, want):
        assert torch.equal(a.scales, b.scales) and torch.equal(a.values, b.values)


def _special(x, kind, g):
    """x with a hundredth of its values infinite or NaN, or all of them subnormal."""
    at = torch.rand(x.shape, generator=g, device="cuda")
    if kind == "subnormal":
        return (x * 2.0**-130).to(torch.bfloat16)
    if kind in ("inf", "both"):
        x[at < 0.005] = torch.inf
        x[(at > 0.005) & (at < 0.01)] = -torch.inf
    if kind in ("nan", "both"):
        x[at > 0.99] = torch.nan
    if kind == "largest":
        x[at < 0.05] = torch.finfo(torch.bfloat16).max
    return x


def _same(got, want):
    for a, b in zip(got, want):
        assert torch.equal(a.scales, b.scales) and torch.equal(a.values, b.values)


@pytest.mark.parametrize("rows", ["first", "all"])
@pytest.mark.parametrize("kind", ["inf", "nan", "both", "subnormal", "largest"])
def test_special_rows_by_index_are_the_float32_quantizers(lib, kind, rows):
    """Rows read by index, some of them outside the tokens, the last ones past `filled`."""
    from bux_amd import grouped_mxfp8
    g = torch.Generator(device="cuda").manual_seed(111)
    t, k, d = 70, 3, 160
    x = _special(torch.randn(t, d, generator=g, device="cuda").to(torch.bfloat16), kind, g)
    index = torch.randperm(t * k, generator=g, device="cuda").int()
    index[5], index[60] = -1, t * k
    filled = torch.tensor([150 if rows == "first" else t * k], dtype=torch.int32, device="cuda")
    announce("special rows by index", kind, rows)
    got, want = (grouped_mxfp8.quantized_twice(v, filled, True, index, k, 256) for v in (x, x.float()))
    torch.cuda.synchronize()
    _same(got, want)


@pytest.mark.parametrize("gated", [True, False])
@pytest.mark.parametrize("kind", ["inf", "nan", "both", "subnormal", "largest"])
def test_special_activations_are_the_float32_quantizers(lib, kind, gated):
    """The quantizing activation and its gradient: the copies of the bfloat16 values that the
    plain kernels give, quantized by the float route."""
    from bux_amd import grouped_mxfp8, moe
    g = torch.Generator(device="cuda").manual_seed(112)
    m, f, p = 130, 96, 2 if gated else 1
    projected = _special(torch.randn(m, f, p, generator=g, device="cuda").to(torch.bfloat16), kind, g)
    dh = _special(torch.randn(m, f, generator=g, device="cuda").to(torch.bfloat16), kind, g)
    w = torch.rand(m, generator=g, device="cuda").to(torch.bfloat16)
    filled = torch.tensor([m - 9], dtype=torch.int32, device="cuda")
    ffn = moe.Ffn()
    announce("special activations", kind, gated)
    got = moe.weighted_units_quantized(ffn, projected, w, filled, 256)[:2]
    h = moe.weighted_units(ffn, projected, w, filled)
    want = grouped_mxfp8.quantized_twice(h.float(), filled, height=256)
    back = moe.weighted_units_backward_quantized(ffn, projected, w, dh, filled, 256)[:2]
    dp = moe.weighted_units_backward(ffn, projected, w, dh, filled)[0].reshape(m, f * p)
    torch.cuda.synchronize()
    _same(got, want)
    _same(back, grouped_mxfp8.quantized_twice(dp.float(), filled, height=256))
    if kind in ("inf", "nan", "both"):
        assert not bool(h.isfinite().all()) and not bool(dp.isfinite().all())
