"""The "compute" GEMMs on a tile list made once give the bits of those that make their own,
in bfloat16 and float32, on the tiled and the any-shape kernels, and refuse a list made for
other dimensions."""

import numpy as np
import pytest
import torch

from tests._util import announce

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("sizes,m,k,n", [([300, 0, 77, 500], 900, 64, 264), ([5, 0, 3], 10, 45, 37),
                                         ([0, 0], 64, 32, 32), ([513] + [3] * 40, 700, 128, 128)])
def test_listed_gemms_are_the_others(lib, sizes, m, k, n, dtype):
    from bux_amd import grouped, grouped_mxfp8
    g = torch.Generator(device="cuda").manual_seed(120)
    gs = torch.tensor(sizes, dtype=torch.int32, device="cuda")
    x, w, dy = (torch.randn(*s, generator=g, device="cuda").to(dtype)
                for s in ((m, k), (len(sizes), k, n), (m, n)))
    tiles = grouped_mxfp8.tiles_of(gs, m, m)
    announce("listed compute GEMMs", sizes[:4], m, k, n, dtype)
    pairs = [(grouped.dot(x, w, gs), grouped.dot(x, w, gs, tiles=tiles)),
             (grouped.dot(dy, w, gs, transposed=True), grouped.dot(dy, w, gs, transposed=True, tiles=tiles)),
             (grouped.weight_grad(x, dy, gs), grouped.weight_grad(x, dy, gs, tiles=tiles))]
    torch.cuda.synchronize()
    for own, listed in pairs:
        assert torch.equal(own, listed)
    with pytest.raises(ValueError):
        grouped.dot(x, w, gs, tiles=grouped_mxfp8.tiles_of(gs, m + 128, m))
    with pytest.raises(ValueError):
        grouped.weight_grad(x, dy, gs, tiles=grouped_mxfp8.tiles_of(torch.cat([gs, gs]), m, m))


@pytest.mark.parametrize("kind", ["bfloat16", "float32", "any shape", "mxfp8"])
def test_a_contract_on_a_list_of_more_rows(lib, kind):
    """A contract takes the rows below its own m of a list made for more: the bits of the
    starts that its own prologue caps."""
    from bux_amd import grouped, grouped_mxfp8
    g = torch.Generator(device="cuda").manual_seed(121)
    m, d, f = 384, 72, 264
    if kind == "any shape":
        d, f = 45, 37
    gs = torch.tensor([100, 0, 250, 700, 5], dtype=torch.int32, device="cuda")
    longer = grouped_mxfp8.tiles_of(gs, 2048, 2048)
    dtype = torch.float32 if kind == "float32" else torch.bfloat16
    announce("contract on a longer list", kind)
    if kind == "mxfp8":
        x, dy = (torch.randn(m, c, generator=g, device="cuda").to(dtype) for c in (96, 160))
        a, b = (grouped_mxfp8.quantized_twice(v, rows=False)[1] for v in (x, dy))
        own, listed = (grouped_mxfp8.contract(a, b, gs, tiles=t) for t in (None, longer))
    else:
        x, dy = (torch.randn(m, c, generator=g, device="cuda").to(dtype) for c in (d, f))
        own, listed = (grouped.weight_grad(x, dy, gs, tiles=t) for t in (None, longer))
    torch.cuda.synchronize()
    assert torch.equal(own, listed)
    assert bool((own[:1] != 0).any()) and not own[4].any()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("k,n", [(64, 264), (45, 37)])
def test_a_list_of_other_dimensions_is_refused_by_the_kernel(lib, k, n, dtype):
    """Through the C ABI, which sees a list's size alone: the GEMM writes nothing and sets
    the list's status word."""
    from bux_amd import grouped_mxfp8, kernels
    m, groups = 200, 3
    gs = torch.tensor([100, 40, 60], dtype=torch.int32, device="cuda")
    x, w, dy, y, dw = (torch.full(s, 3.0, device="cuda", dtype=dtype)
                       for s in ((m, k), (groups, k, n), (m, n), (m, n), (groups, k, n)))
    twin = "_f32" if dtype == torch.float32 else ""
    p, s = kernels.ptr, kernels.stream()
    announce("lists of other dimensions", k, n, dtype)
    lists = {"rows": (gs, m + 56, m), "contract": (torch.cat([gs, gs]), m, m)}
    for kind, args in lists.items():
        made = grouped_mxfp8.tiles_of(*args)
        call = getattr(lib, f"bux_bf16_grouped_{kind}_listed{twin}")
        size = made.buffer.numel()
        rc = (call(p(x), p(w), 0, groups, m, n, k, p(y), p(made.buffer), size, s) if kind == "rows"
              else call(p(x), p(dy), groups, m, k, n, p(dw), p(made.buffer), size, s))
        torch.cuda.synchronize()
        status = made.buffer[:20].view(torch.int32)[4].item()
        assert rc == 0 and status == 1  # BUX_LIST_REFUSED
    assert bool((y == 3).all()) and bool((dw == 3).all())
