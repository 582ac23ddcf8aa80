"""Calls that have to be refused before a kernel sees them: the checks run on
the host, so CPU tensors reach them."""
from __future__ import annotations

import types

import pytest
import torch


def _blocked(n, m):
    v = lambda k: torch.zeros(k, dtype=torch.float16)
    return types.SimpleNamespace(w_blk=torch.zeros((m + 15) // 16, (n + 127) // 128, 2048, dtype=torch.uint8), mx=v(m),
                                 rx=v(m), my=v(n), ry=v(n), bias=None, in_features=n, out_features=m)


@pytest.mark.parametrize("nx,nm,ny,nr", [(1, 2, 2, None), (2, 2, 1, None), (2, 1, 2, None), (2, 2, 2, 1), (5, 5, 5, None),
                                         (0, 0, 0, None)])
def test_mm8_rows_refuses_uneven_lists(nx, nm, ny, nr):
    """As many inputs, outputs and residuals as products: the library reads one
    pointer of each array for every product."""
    from rwkv7mi.native_quant_mm8 import mm8_rows_multi_into

    x, y = torch.zeros(100, 128, dtype=torch.float16), torch.zeros(100, 32, dtype=torch.float16)
    with pytest.raises(ValueError, match="1..4 problems"):
        mm8_rows_multi_into([x] * nx, [_blocked(128, 32)] * nm, [y] * ny, residuals=None if nr is None else [y] * nr)


@pytest.mark.parametrize("rows", [8, 300])
def test_dense_group_of_uneven_lists_runs_one_by_one(rows):
    from rwkv7mi.model import DenseLinear

    lins = [DenseLinear(torch.zeros(32, 64, dtype=torch.float16)) for _ in range(3)]
    xs = [torch.zeros(rows, 64, dtype=torch.float16)] * 2
    outs = [torch.zeros(rows, 32, dtype=torch.float16)] * 3
    assert DenseLinear.apply_group(lins, xs, outs) is False
