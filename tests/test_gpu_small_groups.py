"""The MXFP8 GEMMs' float32 epilogue at the edges of its tiles: both dtypes store the same
float32 sums, so a bfloat16 output is its float32 twin's rounding to the bit. (The values
against the oracle's float64 sums: tests/test_gpu_gemm.py.)"""

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
