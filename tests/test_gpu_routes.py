"""The kernels that calls run on at the lines of the dispatch rules that the
library decides without a trace on the host."""
from __future__ import annotations

import pytest
import torch

from graph_routes import kernels

pytestmark = pytest.mark.gpu
F16, BF16 = torch.float16, torch.bfloat16


def _r(*shape, dt=F16, scale=1.0):
    return torch.randn(*shape, device="cuda", dtype=dt) * scale


@pytest.mark.parametrize("rows,K,N,kernel", [(17, 768, 768, "w4g_kernel"), (64, 1024, 4096, "w4g_kernel"),
                                             (48, 1024, 16384, "w4g_kernel"), (96, 1024, 1024, "w4g_kernel"),
                                             (97, 1024, 16384, "w4m_kernel"), (17, 512, 65536, "w4m_kernel")])
def test_w4_few_rows(rows, K, N, kernel):
    from rwkv7mi.sm70_quant import w4_groupwise_linear

    q = torch.randint(0, 256, (N, K // 2), device="cuda", dtype=torch.uint8)
    s = torch.rand(N, K // 128, device="cuda").to(F16) * 0.02
    x = _r(rows, K)
    out = torch.empty(rows, N, device="cuda", dtype=F16)
    launches = (rows + 63) // 64 if kernel == "w4g_kernel" else 1
    assert kernels(lambda: w4_groupwise_linear(x, q, s, N, K, out=out)) == [kernel] * launches


@pytest.mark.parametrize("rows,D,seq", [
    (7000, 768, False), (9000, 768, True), (12500, 768, True), (8000, 1024, False), (12000, 1024, True),
    (10240, 2048, False), (13000, 2048, True), (17000, 2048, False), (17000, 768, True), (32768, 1536, True),
])
def test_lora_one_launch_or_pair(rows, D, seq):
    from rwkv7mi.fused_lora import fused_wavg_lora

    ranks = (64, 64, 128, 32)
    x = _r(rows, D)
    dn, up = [_r(r, D, scale=0.02) for r in ranks], [_r(D, r, scale=0.02) for r in ranks]
    got = kernels(lambda: fused_wavg_lora(x, x, x, x, *dn, *up, None, None, None, None))
    assert got == (["lora_seq_kernel"] if seq else ["lora_mid_kernel", "lora_out_kernel"])


def _dense(rows, K, Ns, dt):
    from rwkv7mi.fused_lora import dense_multi

    x = _r(rows, K, dt=dt)
    probs = [(x, _r(n, K, dt=dt, scale=0.05), None, torch.empty(rows, n, device="cuda", dtype=dt), 0) for n in Ns]
    got = kernels(lambda: dense_multi(probs, rows))
    step = 2.0 ** -11 if dt == F16 else 2.0 ** -8  # one rounding of the output, fp32 sums
    for _, W, _, y, _ in probs:
        ref = x.double() @ W.double().t()
        assert bool(((y.double() - ref).abs() <= step * ref.abs() + 2e-5 * ref.abs().max()).all())
    return got


@pytest.mark.parametrize("Ns,dt,kernel", [((2048,), F16, "dense_gemv_kernel"), ((768, 768), F16, "dense_gemv_kernel"),
                                          ((3072,), F16, "dense_tile_kernel"), ((768, 768), BF16, "dense_tile_kernel")])
def test_dense_two_rows(Ns, dt, kernel):
    assert _dense(2, 768, Ns, dt) == [kernel]


@pytest.mark.parametrize("rows,K,Ns,dt,kernel", [
    (5, 768, (32768,), F16, "dense_kernel"), (12, 1024, (16380,) + (8,), F16, "dense_kernel"),
    (16, 512, (65536,), F16, "dense_kernel"), (13, 768, (32768,), F16, "dense_tile_kernel"),
    (5, 768, (32768,), BF16, "dense_tile_kernel"), (5, 1536, (32768,), F16, "dense_tile_kernel"),
    (4, 768, (32768,), F16, "dense_tile_kernel"),
])
def test_dense_few_rows_of_many_short_outputs(rows, K, Ns, dt, kernel):
    assert _dense(rows, K, Ns, dt) == [kernel]


@pytest.mark.parametrize("T,H,dt,two", [(320, 64, F16, False), (400, 64, F16, True), (1500, 64, torch.float32, True),
                                        (2000, 64, torch.float32, False), (2000, 48, torch.float32, True),
                                        (4200, 64, F16, False), (4200, 64, BF16, True)])
def test_scan_one_launch_or_two(T, H, dt, two):
    from rwkv7mi import dplr_chunk_scan

    k = torch.nn.functional.normalize(_r(1, T, H, 64, dt=torch.float32), dim=-1).to(dt)
    w = torch.full((1, T, H, 64), 0.6, device="cuda")
    st = torch.zeros(1, H, 64, 64, device="cuda")
    got = kernels(lambda: dplr_chunk_scan(_r(1, T, H, 64, dt=dt), w, k, k, k, k.abs(), st))
    assert set(got) == ({"wkv7_chunk_kernel", "wkv7_chain_kernel"} if two else {"wkv7_chunk_kernel"})
