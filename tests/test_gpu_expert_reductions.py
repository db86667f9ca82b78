"""The sums over rows of the experts' norm (its gain's and bias's gradients) and of the
biases' gradients, against float64, at row counts around what a workgroup and a wave take:
one and several rows a norm workgroup with a remainder, experts of none, one and more rows
than the 16 waves' four in flight. Each float32 sum of n terms is held within n 2^-24 of
the sum of its terms' magnitudes, the bound of any order of additions, and the terms
themselves within 2^-20 (a float32 mean and rsqrt)."""

import pytest
import torch

from tests._util import announce

pytestmark = pytest.mark.gpu


def _offsets(sizes):
    return torch.tensor([0, *torch.tensor(sizes).cumsum(0).tolist()], dtype=torch.int32, device="cuda")


@pytest.mark.parametrize("sizes,d", [([700, 0, 323], 256), ([1025], 2056), ([2000, 500, 1, 77], 4104),
                                     ([3], 8192)])
def test_norm_parameter_gradients(lib, sizes, d):
    from bux_amd import moe
    g = torch.Generator(device="cuda").manual_seed(90)
    m = sum(sizes)
    y, dy, w = (torch.randn(*s, generator=g, device="cuda") for s in ((m, d), (m, d), (m,)))
    scale, bias = (torch.randn(d, generator=g, device="cuda") for _ in range(2))
    order = torch.arange(m, dtype=torch.int32, device="cuda")
    norm = moe.ExpertNorm("layernorm", bias=True)
    announce("norm parameter gradients", sizes, d)
    dv, dw, d_scale, d_bias = moe.expert_norm_backward(dy, order, 1, y, _offsets(sizes), norm, scale,
                                                       bias, w)
    torch.cuda.synchronize()
    y64, g64 = y.double(), dy.double() * w.double()[:, None]
    u = y64 - y64.mean(-1, keepdim=True)
    xn = u * torch.rsqrt(u.square().mean(-1, keepdim=True) + norm.eps)
    for got, terms in ((d_scale, g64 * xn), (d_bias, g64)):
        err = (got.double() - terms.sum(0)).abs()
        assert bool((err <= (m * 2.0**-24 + 2.0**-20) * terms.abs().sum(0)).all())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("sizes,width", [([1, 0, 15, 16, 17], 256), ([63, 64, 65, 129, 500], 264),
                                         ([0, 1000], 8)])
def test_expert_sums(lib, sizes, width, dtype):
    from bux_amd import moe
    g = torch.Generator(device="cuda").manual_seed(91)
    m = sum(sizes) + 5  # rows in no expert add to none
    x = torch.randn(m, width, generator=g, device="cuda").to(dtype)
    index = torch.randperm(m, generator=g, device="cuda").int()
    index[0] = -1  # a row of 0
    w = torch.randn(m, generator=g, device="cuda").to(dtype)
    announce("expert sums", sizes, width, dtype)
    got = moe.expert_sums(x, _offsets(sizes), index, 1, w)
    torch.cuda.synchronize()
    rows = (x[index.long().clamp(min=0)] * w[:, None]).double()  # products rounded to the dtype
    rows[0] = 0
    start = 0
    for e, size in enumerate(sizes):
        part = rows[start:start + size]
        start += size
        err = (got[e].double() - part.sum(0)).abs()
        assert bool((err <= size * 2.0**-24 * part.abs().sum(0)).all())


@pytest.mark.parametrize("m,d", [(1023, 256), (1024, 256), (1025, 256), (2049, 2056), (65537, 8)])
def test_norm_gradients_of_every_row(lib, m, d):
    """dv and the weights' gradients are a row's own, whichever workgroup takes it: the bits
    of calls on parts of the rows."""
    from bux_amd import moe
    g = torch.Generator(device="cuda").manual_seed(92)
    y, dy, w = (torch.randn(*s, generator=g, device="cuda") for s in ((m, d), (m, d), (m,)))
    scale = torch.randn(d, generator=g, device="cuda")
    norm = moe.ExpertNorm("rmsnorm")

    def backward(lo, hi):
        order = torch.arange(hi - lo, dtype=torch.int32, device="cuda")
        return moe.expert_norm_backward(dy[lo:hi], order, 1, y[lo:hi], _offsets([hi - lo]), norm, scale,
                                        None, w[lo:hi])[:2]

    announce("norm gradients of every row", m, d)
    got = backward(0, m)
    cuts = [0, *range(500, m, 500), m]
    parts = [backward(lo, hi) for lo, hi in zip(cuts, cuts[1:])]
    torch.cuda.synchronize()
    for i in range(2):
        assert torch.equal(got[i], torch.cat([p[i] for p in parts]))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("sizes,width", [([7, 0, 8, 15, 33, 1], 520), ([32] * 6, 1288),
                                         ([31, 32, 33, 100, 0, 17] * 20, 1288), ([40, 41] * 64, 1032)])
def test_expert_sums_in_each_form(lib, sizes, width, dtype):
    """Few rows an expert (8 waves of 512 columns), and many in more workgroups than the 512
    up to which 16 waves take 256 columns: around a turn of the waves and the columns' ends."""
    test_expert_sums(lib, sizes, width, dtype)
