"""The layer's sort (bux_moe_permute_layer) against its parts: the sort against the
oracle's, the sorted weights and the tile list against picked_weights and tiles_of, all to
the bit, at the edges of its one-workgroup kernel (4096 and 8192 picks, 900 bins) and of the waves'
segments in it."""

import numpy as np
import pytest
import torch

from oracle import moe as omoe
from tests._util import announce, to_gpu

pytestmark = pytest.mark.gpu

# picks a token, tokens, experts
CASES = [(1, 1, 1), (8, 8, 128), (1, 63, 4), (4, 256, 899), (5, 205, 900), (3, 341, 8), (8, 1024, 128), (8, 512, 128),
         (1, 8193, 128), (1, 4097, 128), (2, 600, 1000), (7, 1171, 256), (8, 16384, 128)]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("k,t,e", CASES)
def test_the_layers_sort_is_its_parts(lib, k, t, e, dtype):
    from bux_amd import grouped_mxfp8, moe
    rng = np.random.default_rng(80)
    n = t * k
    idx = rng.integers(-1, e + 1, (t, k)).astype(np.int32)  # some picks outside the experts
    if n > 40:
        idx.reshape(-1)[: n // 2] = rng.integers(0, max(1, e // 3))  # one expert of many rows
        rng.shuffle(idx.reshape(-1))
    weights = torch.randn(t, k, device="cuda").to(dtype)
    height = grouped_mxfp8.whole(n)
    announce("layer sort", k, t, e, dtype)
    s, row_weights, listed = moe.sort_for_layer(to_gpu(idx), e, weights, height)
    tiles = grouped_mxfp8.tiles_of(s.sizes, height, n)
    bare, none = moe.sort_for_layer(to_gpu(idx), e, weights, None)[::2]
    torch.cuda.synchronize()
    want = omoe.sort_by_expert(idx, e)
    np.testing.assert_array_equal(s.order.cpu().numpy(), want.order)
    np.testing.assert_array_equal(s.inverse.cpu().numpy(), want.inverse)
    np.testing.assert_array_equal(s.sizes.cpu().numpy(), want.sizes)
    np.testing.assert_array_equal(s.offsets.cpu().numpy()[:e], want.offsets)
    assert int(s.offsets[e]) == want.sizes.sum()
    assert none is None and all(torch.equal(a, b) for a, b in zip(s, bare))
    assert torch.equal(row_weights, weights.reshape(-1)[s.order.long()])
    # the list: header and starts, then (256-byte aligned) the records
    head, records = 64 + 4 * (e + 2), -(-(64 + 4 * (e + 2)) // 256) * 256
    got, made = listed.buffer.cpu().numpy(), tiles.buffer.cpu().numpy()
    assert listed[1:] == tiles[1:] and got.size == made.size
    np.testing.assert_array_equal(got[:head], made[:head])
    np.testing.assert_array_equal(got[records:], made[records:])


def test_weights_other_than_one_a_pick(lib):
    """A non-contiguous view is read as its values; picks past the weights weigh 0."""
    from bux_amd import moe
    idx = to_gpu(np.array([[1, 0], [0, 1], [1, 1]], np.int32))
    w = torch.arange(1, 7, device="cuda").to(torch.bfloat16)
    announce("layer sort, strided and short weights")
    _, strided, _ = moe.sort_for_layer(idx, 2, w.view(2, 3).T, None)
    _, short, _ = moe.sort_for_layer(idx, 2, w[:4], None)
    torch.cuda.synchronize()
    assert strided.tolist() == [4, 2, 1, 5, 3, 6]  # order 1, 2, 0, 3, 4, 5 of 1 4 2 5 3 6
    assert short.tolist() == [2, 3, 1, 4, 0, 0]


@pytest.mark.parametrize("n", [64, 1000, 4097, 8192])
def test_picks_of_few_experts(lib, n):
    """All the picks with one expert, and in runs of two: a wave's 64 picks in a bin or two,
    in the one-workgroup kernel with one to eight turns a wave and a last one in part."""
    from bux_amd import moe
    announce("layer sort, picks of few experts", n)
    for idx in (np.full((n, 1), 5, np.int32), (np.arange(n, dtype=np.int32)[:, None] // 37) % 2 + 3):
        weights = torch.randn(n, 1, device="cuda")
        s, row_weights, _ = moe.sort_for_layer(to_gpu(idx), 8, weights, None)
        torch.cuda.synchronize()
        want = omoe.sort_by_expert(idx, 8)
        np.testing.assert_array_equal(s.order.cpu().numpy(), want.order)
        np.testing.assert_array_equal(s.inverse.cpu().numpy(), want.inverse)
        np.testing.assert_array_equal(s.sizes.cpu().numpy(), want.sizes)
        assert torch.equal(row_weights, weights.reshape(-1)[s.order.long()])


@pytest.mark.parametrize("dtype", [torch.float16, torch.int32, torch.float64])
def test_weights_of_other_dtypes_are_refused(lib, dtype):
    from bux_amd import moe
    idx = to_gpu(np.array([[1, 0]], np.int32))
    announce("layer sort, weights of another dtype", dtype)
    with pytest.raises(TypeError, match="weights"):
        moe.sort_for_layer(idx, 2, torch.ones(1, 2, dtype=dtype, device="cuda"), None)
