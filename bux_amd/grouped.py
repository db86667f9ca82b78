"""The grouped GEMMs of the "compute" precision (no MXFP8) on MI355X.

Mirrors ``grouped.dot`` and ``grouped.weight_grad``
(src/bux/architecture/experts/grouped.py:90-146): float32 sums, out in the operands'
dtype (bfloat16, or float32 for a layer in float32), the rows past the groups 0.
"""

import torch

from bux_amd import _lib
from bux_amd.grouped_mxfp8 import TileList
from bux_amd.kernels import lib, ptr, require, stream, workspace


def _f32(name: str, *tensors: torch.Tensor) -> bool:
    """Whether the operands are float32 (all), not bfloat16 (all)."""
    kinds = {t.dtype for t in tensors}
    if kinds == {torch.float32}:
        return True
    if kinds == {torch.bfloat16}:
        return False
    raise TypeError(f"{name}: bfloat16 or float32 operands, one dtype, not {kinds}")


def dot(x: torch.Tensor, w: torch.Tensor, sizes: torch.Tensor, transposed: bool = False,
        tiles: TileList | None = None) -> torch.Tensor:
    """Return each group's rows of x times its matrix: x (m, k) and w (g, k, n), or
    with `transposed` w (g, n, k) and x w[g]^T; in x's dtype (bfloat16 or float32, w
    the same). tiles: `grouped_mxfp8.tiles_of(sizes, m, m)`, made once for a step's GEMMs;
    None to make it here."""
    require(x, w, sizes)
    f32 = _f32("dot", x, w)
    m, k = x.shape
    groups = w.shape[0]
    n = w.shape[1] if transposed else w.shape[2]
    if (w.shape[2] if transposed else w.shape[1]) != k:
        raise ValueError(f"dot: x {tuple(x.shape)}, w {tuple(w.shape)}, transposed={transposed}")
    y = torch.empty(m, n, dtype=x.dtype, device=x.device)
    if tiles is not None:
        if (tiles.groups, tiles.m, tiles.height) != (groups, m, m):
            raise ValueError(f"dot: a tile list for {tiles.groups} groups, m={tiles.m}, "
                             f"height={tiles.height}, not {groups}, {m}, {m}")
        rows = lib().bux_bf16_grouped_rows_listed_f32 if f32 else lib().bux_bf16_grouped_rows_listed
        _lib.check(rows(ptr(x), ptr(w), int(transposed), groups, m, n, k, ptr(y), ptr(tiles.buffer),
                        tiles.buffer.numel(), stream()))
        return y
    ws = workspace(lib().bux_bf16_grouped_rows_workspace_size(groups, m), x.device)
    rows = lib().bux_bf16_grouped_rows_f32 if f32 else lib().bux_bf16_grouped_rows
    _lib.check(rows(ptr(x), ptr(w), int(transposed), ptr(sizes), groups, m, n, k, ptr(y), ptr(ws),
                    ws.numel(), stream()))
    return y


def weight_grad(x: torch.Tensor, dy: torch.Tensor, sizes: torch.Tensor,
                tiles: TileList | None = None) -> torch.Tensor:
    """Return ``x[rows of g]^T dy[rows of g]`` for each group g, (g, k, n), in x's dtype
    (bfloat16 or float32, dy the same). tiles: a tile list of the same sizes, as `dot`'s,
    or of more rows: those past x's add nothing."""
    require(x, dy, sizes)
    f32 = _f32("weight_grad", x, dy)
    m, k = x.shape
    n = dy.shape[1]
    groups = sizes.shape[0]
    dw = torch.empty(groups, k, n, dtype=x.dtype, device=x.device)
    if tiles is not None:
        if tiles.groups != groups:
            raise ValueError(f"weight_grad: a tile list for {tiles.groups} groups, not {groups}")
        contract = (lib().bux_bf16_grouped_contract_listed_f32 if f32
                    else lib().bux_bf16_grouped_contract_listed)
        _lib.check(contract(ptr(x), ptr(dy), groups, m, k, n, ptr(dw), ptr(tiles.buffer),
                            tiles.buffer.numel(), stream()))
        return dw
    ws = workspace(lib().bux_bf16_grouped_contract_workspace_size(groups), x.device)
    contract = lib().bux_bf16_grouped_contract_f32 if f32 else lib().bux_bf16_grouped_contract
    _lib.check(contract(ptr(x), ptr(dy), ptr(sizes), groups, m, k, n, ptr(dw), ptr(ws), ws.numel(),
                        stream()))
    return dw
