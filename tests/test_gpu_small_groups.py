"""The MXFP8 GEMMs' float32 epilogue and the rows GEMM for groups of few rows, at the
edges of their tiles, against each other: every output of either kernel is the same
float32 sum, so a bfloat16 output is its float32 twin's rounding to the bit, and a call
that goes to one rows kernel gives the other's bits. (Their values against the oracle's
float64 sums: tests/test_gpu_gemm.py, whose cases take both kernels.)"""

import numpy as np
import pytest
import torch

from tests._util import announce

pytestmark = pytest.mark.gpu


def _codes(rng, shape):
    from bux_amd import grouped_mxfp8
    *lead, r, k = shape
    values = rng.integers(0, 120, (*lead, k // 64, r, 64), np.uint8) | rng.choice(
        np.array([0, 128], np.uint8), (*lead, k // 64, r, 64))
    scales = rng.integers(118, 132, (*lead, k // 128, r, 4), np.uint8)
    return grouped_mxfp8.Tiled(torch.from_numpy(values).cuda(), torch.from_numpy(scales).cuda())


# sizes, k, n: groups at and over a block of 32 rows, one of a whole tile and more, empty
# ones, rows past the groups; n off the waves' 32 and 64 columns; K of one pair, of an odd
# number of them, of fewer than are in flight
SMALL = [
    ([1] + [0] * 31, 128, 4),
    ([5, 0, 32, 33, 1] + [0] * 45, 256, 132),
    ([0, 300] + [1] * 60, 384, 260),
    ([64, 31, 0, 7] + [2] * 60, 1152, 96),
    ([3] * 128, 640, 1540),  # waves of 64 columns
    ([0] * 20 + [240], 896, 160),
]


@pytest.mark.parametrize("sizes,k,n", SMALL)
def test_rows_of_few_rows_are_the_tiled_kernels(lib, sizes, k, n):
    from bux_amd import grouped_mxfp8
    rng = np.random.default_rng(70)
    groups, filled = len(sizes), sum(sizes)
    m = filled + 3
    assert m <= 16 * groups
    far = 32 * groups + 1  # rows enough for the tiled kernel
    a = _codes(rng, (far, k))
    few = grouped_mxfp8.Tiled(a.values[:, :m].contiguous(), a.scales[:, :m].contiguous())
    b = _codes(rng, (groups, n, k))
    gs = torch.tensor(sizes, dtype=torch.int32, device="cuda")
    announce("rows of few rows", sizes[:5], k, n)
    got = [grouped_mxfp8.rows(few, b, gs, dt) for dt in (torch.bfloat16, torch.float32)]
    want = [grouped_mxfp8.rows(a, b, gs, dt) for dt in (torch.bfloat16, torch.float32)]
    torch.cuda.synchronize()
    for g, w in zip(got, want):
        assert torch.equal(g, w[:m])
        assert (g[filled:] == 0).all()
    assert torch.equal(got[0], got[1].to(torch.bfloat16))


# group sizes, n (or d and f): whole tiles, half tiles, partial ones, columns of a multiple
# of 4 alone
@pytest.mark.parametrize("sizes,k,n", [([300, 5, 129, 256], 256, 256), ([700, 90], 128, 516),
                                       ([256, 100, 511], 384, 36), ([1030], 128, 700)])
def test_float32_outputs_round_to_the_bfloat16_ones(lib, sizes, k, n):
    from bux_amd import grouped_mxfp8
    rng = np.random.default_rng(71)
    m = -(-sum(sizes) // 128) * 128
    gs = torch.tensor(sizes, dtype=torch.int32, device="cuda")
    a, b = _codes(rng, (m, k)), _codes(rng, (len(sizes), n, k))
    at, bt = _codes(rng, (k + 4, m)), _codes(rng, (n, m))
    announce("float32 outputs", sizes, k, n)
    rows = [grouped_mxfp8.rows(a, b, gs, dt) for dt in (torch.bfloat16, torch.float32)]
    dw = [grouped_mxfp8.contract(at, bt, gs, dt) for dt in (torch.bfloat16, torch.float32)]
    torch.cuda.synchronize()
    for b16, f32 in (rows, dw):
        assert torch.equal(b16, f32.to(torch.bfloat16))
    assert bool((dw[1] != 0).any(-1).all()) and bool((rows[1][:sum(sizes)] != 0).any(-1).all())


@pytest.mark.parametrize("sizes,k,n", [c for c in SMALL if len(c[0]) < 128] + [([3] * 64, 640, 1540)])
def test_the_two_rows_kernels_each_take_their_call(lib, sizes, k, n):
    """The comparison above, with the library's own rule saying that the call of few rows
    takes rows_direct_kernel and the other the tiled one."""
    from tests.test_abi import _direct
    groups, m = len(sizes), sum(sizes) + 3
    assert _direct(lib, m, groups, n) == 1 and _direct(lib, 32 * groups + 1, groups, n) == 0
    test_rows_of_few_rows_are_the_tiled_kernels(lib, sizes, k, n)


# groups of a block of rows, of two, of more, in part and whole; a tile and a second one
CROWDED = [33, 64, 65, 0, 1, 300, 31, 32, 128, 97] + [2] * 54


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("k,n", [(128, 2308), (256, 2304), (384, 2500), (640, 2308)])
def test_waves_of_two_blocks_are_the_tiled_kernel(lib, k, n, dtype):
    """K of one pair to five, columns off the waves' 64, with and without a bias."""
    from bux_amd import grouped_mxfp8
    from tests.test_abi import _direct
    rng = np.random.default_rng(72)
    groups, filled = len(CROWDED), sum(CROWDED)
    m, far = filled + 3, 32 * groups + 1
    assert _direct(lib, m, groups, n) == 2 and _direct(lib, far, groups, n) == 0
    a = _codes(rng, (far, k))
    few = grouped_mxfp8.Tiled(a.values[:, :m].contiguous(), a.scales[:, :m].contiguous())
    b = _codes(rng, (groups, n, k))
    gs = torch.tensor(CROWDED, dtype=torch.int32, device="cuda")
    bias = (torch.randn(groups, n, device="cuda") * 100).to(dtype)
    announce("waves of two blocks", k, n, dtype)
    for added in (None, bias):
        got, want = (grouped_mxfp8.rows(x, b, gs, dtype, tiles=grouped_mxfp8.tiles_of(gs, rows, rows),
                                        bias=added) for x, rows in ((few, m), (a, far)))
        torch.cuda.synchronize()
        assert torch.equal(got, want[:m])
        assert (got[filled:] == 0).all() and bool((got[:filled] != 0).any(-1).all())
