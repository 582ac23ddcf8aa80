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


@pytest.fixture
def dense_calls(monkeypatch):
    """The dense products' library calls, recorded instead of run."""
    from rwkv7mi import _lib, model

    calls = []
    monkeypatch.setattr(_lib, "require_gpu", lambda *t, name: None)
    monkeypatch.setattr(_lib, "stream_of", lambda t: 0)
    monkeypatch.setattr(_lib, "call", lambda name, *args: calls.append(args))
    return calls


def test_dense_multi_refuses_residuals_the_kernel_would_misread(dense_calls):
    from rwkv7mi.fused_lora import dense_multi

    x, w, y = torch.zeros(4, 64), torch.zeros(32, 64), torch.zeros(4, 32)
    run = lambda res, out=y, k=1: dense_multi([(x, w, None, out, 0)] * k, 4, res)
    for bad in (torch.zeros(4, 32, dtype=torch.float16), torch.zeros(1, 32), torch.zeros(32, 4).t(),
                torch.zeros(4, 32, device="meta")):
        with pytest.raises(ValueError, match="residual"):
            run([bad])
    with pytest.raises(ValueError, match="residual"):
        run([y], torch.zeros(4, 64)[:, :32])
    with pytest.raises(ValueError, match="residual"):
        run([y], k=2)
    assert not dense_calls
    run([y])
    run([None])
    run(None)
    assert len(dense_calls) == 3


def test_dense_linear_residual_forms_go_through_torch(dense_calls, monkeypatch):
    """A residual or an output that the kernel's epilogue cannot take is added
    by torch, which handles strides and refuses another device or a partial
    overlap; an output over x's memory is not written during the product."""
    from rwkv7mi.model import DenseLinear

    torch_add, added = torch.add, []
    monkeypatch.setattr(torch, "add", lambda *a, **k: (added.append(a), torch_add(*a, **k))[1])
    lin = DenseLinear(torch.zeros(32, 32))
    x = torch.zeros(4, 32)
    buf = torch.zeros(5, 32)
    for out, res in ((torch.zeros(4, 64)[:, :32], torch.ones(4, 32)), (x, torch.ones(4, 32)), (torch.zeros(4, 32),
                     torch.ones(1, 32))):
        n = len(added)
        lin.apply(x, out, residual=res)
        assert len(added) == n + 1
    for out, res in ((torch.zeros(4, 32), torch.ones(4, 32, device="meta")), (buf[:4], buf[1:])):
        with pytest.raises(RuntimeError):
            lin.apply(torch.zeros(4, 32), out, residual=res)
    n = len(added)
    y = torch.zeros(4, 32)
    lin.apply(x, y, residual=y)
    lin.apply(x, y, residual=torch.ones(32, 4).t())
    assert len(added) == n  # in the kernel


@pytest.mark.parametrize("name", ["w_blk", "mx", "ry"])
def test_mm8_linear_reads_its_tensors_where_they_are(monkeypatch, name):
    """A module whose packed tensors were reassigned as parameters runs."""
    from rwkv7mi import _lib, native_quant_mm8 as Q

    seen = []
    monkeypatch.setattr(_lib, "require_gpu", lambda *t, name: None)
    monkeypatch.setattr(Q, "_linear_into", lambda *a: seen.append(a) or True)
    b = _blocked(128, 32)
    mod = Q.MM8Linear.from_packed(b.w_blk, b.mx, b.rx, b.my, b.ry, 128, 32)
    setattr(mod, name, torch.nn.Parameter(getattr(mod, name), requires_grad=False))
    mod(torch.zeros(4, 128, dtype=torch.float16))
    for got, want in zip(seen[0][1:6], ("w_blk", "mx", "rx", "my", "ry")):
        assert got is getattr(mod, want)


def test_mm8_reserve_hook_grows_the_slots_a_call_uses(monkeypatch):
    """4096 -> 16384 (2^26 weights): above 64 rows the middle-row kernel and its
    own slot, the tile GEMM's beside it for calls that stay on that one."""
    from rwkv7mi import native_quant_mm8 as Q

    grown = {}
    monkeypatch.setattr(Q._ws, "reserve", lambda device, need, slot, **k: grown.__setitem__(slot, need))
    n, m = 4096, 16384
    b = _blocked(n, m)
    mod = Q.MM8Linear.from_packed(b.w_blk, b.mx, b.rx, b.my, b.ry, n, m)
    for rows in (17, 64, 65, 256):
        grown.clear()
        mod.rwkv7_reserve_workspace(rows)
        form, need = Q._linear_plan(rows, n, m, Q._lib.F16, 0)[:2]
        assert (form == 2) == (rows > 64)
        assert grown[Q._FORM_SLOT[form]] == need == mod.rwkv7_workspace_bytes(rows)
        assert grown["mm8g"] == Q.mm8_gemm_workspace_bytes(1, rows, n, m)
    mod.mx = mod.mx.float()  # fp32 metadata: fp32 activations, the tile GEMM
    assert mod.rwkv7_workspace_bytes(100) == Q.mm8_gemm_workspace_bytes(1, 100, n, m)


@pytest.mark.parametrize("rows,slot", [(200, "mm8g"), (300, "mm8p")])
@pytest.mark.parametrize("route", ["one", "many"])
def test_mm8_middle_rows_ready_a_capture_at_other_row_counts(monkeypatch, rows, slot, route):
    """An eager call grows the slot of the form beside it: a graph captured
    later at 64 or 1500 rows runs that form and cannot grow it itself."""
    from rwkv7mi import _lib, native_quant_mm8 as Q

    grown = {}

    def reserve(device, need, slot="mm8", **k):
        grown[slot] = need
        return torch.empty(need, dtype=torch.uint8, device="meta")

    monkeypatch.setattr(Q._ws, "reserve", reserve)
    monkeypatch.setattr(_lib, "require_gpu", lambda *t, name: None)
    monkeypatch.setattr(_lib, "stream_of", lambda t: 0)
    monkeypatch.setattr(_lib, "call", lambda *a: None)
    n, m = 4096, 16384
    b = _blocked(n, m)
    x, y = torch.zeros(rows, n, dtype=torch.float16), torch.zeros(rows, m, dtype=torch.float16)
    if route == "one":
        assert Q._linear_into(x, b.w_blk, b.mx, b.rx, b.my, b.ry, None, None, y, 0)
    else:
        Q.mm8_many_rows_into([x], [b], [y])
    assert "mm8r" in grown
    want = Q.mm8_gemm_workspace_bytes(1, rows, n, m) if slot == "mm8g" else Q.mm8_prefill_workspace_bytes(1, n, m)
    assert grown[slot] == want


def test_w4_asks_for_its_scratch_once_a_shape(monkeypatch):
    """One library call a product: the size query is kept by the sizes."""
    from rwkv7mi import _lib, sm70_quant as W

    asked, calls = [], []

    class Lib:
        @staticmethod
        def rwkv7mi_w4_workspace_bytes(*a):
            asked.append(a)
            return 0

    monkeypatch.setattr(_lib, "require_gpu", lambda *t, name: None)
    monkeypatch.setattr(_lib, "stream_of", lambda t: 0)
    monkeypatch.setattr(_lib, "load", lambda: Lib)
    monkeypatch.setattr(_lib, "call", lambda *a: calls.append(a))
    x, q, s = torch.zeros(3, 256), torch.zeros(48, 128, dtype=torch.uint8), torch.zeros(48, 2)
    W._w4_scratch.cache_clear()
    try:
        for _ in range(5):
            W.w4_groupwise_linear(x, q, s, 48, 256)
        W.w4_affine_groupwise_linear(x, q, s, s, 48, 256)
    finally:
        W._w4_scratch.cache_clear()  # (filled by the stand-in library)
    assert len(calls) == 6 and [a[4] for a in asked] == [0, 1]
