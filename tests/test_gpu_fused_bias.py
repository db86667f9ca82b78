"""The rows GEMM's bias epilogue against the bias added as an op of its own, to the bit, over
whole, half and partial tiles, empty groups, rows past the groups and the kernel for groups
of few rows; and the biased token sums, whose experts are found a token at once, against
float64 at every k around its kernels' 4 and 8 picks."""

import numpy as np
import pytest
import torch

from tests._util import announce
from tests.test_gpu_small_groups import _codes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("sizes,k,n", [([300, 0, 129, 256], 256, 512), ([700, 90], 128, 516),
                                       ([256, 100, 511], 384, 36), ([3, 0, 40] + [1] * 60, 256, 132)])
def test_rows_with_a_bias(lib, sizes, k, n, dtype):
    from bux_amd import grouped_mxfp8, moe
    rng = np.random.default_rng(100)
    filled = sum(sizes)
    m = filled + 30
    gs = torch.tensor(sizes, dtype=torch.int32, device="cuda")
    offsets = torch.tensor([0, *np.cumsum(sizes)], dtype=torch.int32, device="cuda")
    a, b = _codes(rng, (m, k)), _codes(rng, (len(sizes), n, k))
    bias = (torch.randn(len(sizes), n, device="cuda") * 100).to(dtype)
    tiles = grouped_mxfp8.tiles_of(gs, m, m)
    announce("rows with a bias", sizes[:4], k, n, dtype)
    got = grouped_mxfp8.rows(a, b, gs, dtype, tiles=tiles, bias=bias)
    plain = grouped_mxfp8.rows(a, b, gs, dtype, tiles=tiles)
    expert = torch.repeat_interleave(torch.arange(len(sizes), device="cuda"), gs.long())
    want = plain.clone()
    want[:filled] += bias[expert]
    torch.cuda.synchronize()
    assert torch.equal(got, want) and not torch.equal(got, plain)
    assert (got[filled:] == 0).all()
    if n % 8 == 0:
        assert torch.equal(got, moe.add_expert_bias(plain, bias, offsets))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("k,experts,width", [(1, 1, 8), (3, 64, 264), (4, 65, 2880), (5, 200, 2056),
                                             (8, 128, 1024), (9, 70, 264)])
def test_biased_token_sums(lib, k, experts, width, dtype):
    from bux_amd import moe
    g = torch.Generator(device="cuda").manual_seed(101)
    t = 37
    idx = torch.randint(-1, experts + 1, (t, k), generator=g, device="cuda").int()  # some in no expert
    s = moe.sort_by_expert(idx, experts)
    y, bias = (torch.randn(*shape, generator=g, device="cuda").to(dtype)
               for shape in ((t * k, width), (experts, width)))
    w = torch.randn(t * k, generator=g, device="cuda").to(dtype)
    inverse = s.inverse.view(t, k).clone()
    inverse[0, 0] = t * k  # a row outside y adds nothing
    announce("biased token sums", k, experts, width, dtype)
    got = moe.sum_by_token_biased(y, inverse, bias, s.offsets, w)
    torch.cuda.synchronize()
    expert = idx.long().clamp(0, experts - 1)
    inside = (idx >= 0) & (idx < experts)
    inside[0, 0] = False
    rows = inverse.long().clamp(max=t * k - 1)
    part = (bias[expert] * w[rows][..., None]).double() * inside[..., None]
    there = torch.ones(t, k, 1, device="cuda", dtype=torch.float64)
    there[0, 0] = 0
    both = [(y[rows].double() * there).sum(1), part.sum(1)]
    # each float32 sum of k terms, then (bfloat16) its rounding and the total's
    unit = 2.0**-8 if dtype == torch.bfloat16 else 2.0**-23
    size = (y[rows].double() * there).abs().sum(1) + part.abs().sum(1)
    bound = k * 2.0**-24 * size + unit * (both[0].abs() + both[1].abs()) + unit * sum(both).abs()
    assert bool(((got.double() - sum(both)).abs() <= bound).all())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("width", [8, 504, 520, 1024, 1536, 2560, 2880, 3072, 4104, 6400])
def test_token_sums_of_any_width(lib, width, dtype):
    """The workgroups' waves, 1 to 4 or 6, and the columns' end in them: the sums with and
    without biases of rows whose values their sums hold exactly."""
    from bux_amd import moe
    g = torch.Generator(device="cuda").manual_seed(102)
    t, k, e = 19, 3, 7
    idx = torch.randint(0, e, (t, k), generator=g, device="cuda").int()
    s = moe.sort_by_expert(idx, e)
    y, bias = (torch.randint(-8, 9, shape, generator=g, device="cuda").to(dtype)
               for shape in ((t * k, width), (e, width)))
    w = torch.randint(1, 3, (t * k,), generator=g, device="cuda").to(dtype)
    inverse = s.inverse.view(t, k)
    announce("token sums", width, dtype)
    plain = moe.sum_by_token(y, inverse)
    biased = moe.sum_by_token_biased(y, inverse, bias, s.offsets, w)
    torch.cuda.synchronize()
    want = y[inverse.long()].sum(1)
    assert torch.equal(plain, want)
    assert torch.equal(biased, want + (bias[idx.long()] * w[inverse.long()][..., None]).sum(1))


def test_the_biased_case_of_few_rows_takes_its_kernel(lib):
    from tests.test_abi import _direct
    assert _direct(lib, 103 + 30, 63, 132) == 1 and _direct(lib, 685 + 30, 4, 512) == 0


@pytest.mark.parametrize("fmt", ["mxfp8", "compute"])
def test_a_strided_up_bias_is_refused(lib, fmt):
    """Every other expert's biases of a larger tensor: refused where the bias rides the GEMM
    as where it is an op of its own."""
    from bux_amd import moe
    t, k, e, d, f = 16, 2, 4, 128, 64
    g = torch.Generator(device="cuda").manual_seed(103)
    z, up, down = ((torch.randn(*s, generator=g, device="cuda") * 0.1).bfloat16()
                   for s in ((t, d), (e, d, f, 2), (e, f, d)))
    idx = torch.randint(0, e, (t, k), generator=g, device="cuda").int()
    w = torch.full((t, k), 0.5, device="cuda").bfloat16()
    biases = torch.randn(2 * e, f, 2, generator=g, device="cuda").bfloat16()
    announce("a strided up bias", fmt)
    moe.experts_forward(z, idx, w, up, down, fmt=fmt, up_bias=biases[::2].contiguous())
    with pytest.raises(ValueError, match="contiguous"):
        moe.experts_forward(z, idx, w, up, down, fmt=fmt, up_bias=biases[::2])
    torch.cuda.synchronize()
