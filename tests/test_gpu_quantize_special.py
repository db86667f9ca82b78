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
