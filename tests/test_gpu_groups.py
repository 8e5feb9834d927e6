"""The MFMA skeleton that gives the groups of a workgroup a share of K each: every element type and operand order at
sizes cut by every edge (rows, columns, K tails of part of a 16-byte chunk, one K tile for several groups, an odd number of
result columns), with the tiles asked for by RX_GEMM_G and with those the planner picks."""
import re

import numpy as np
import pytest

from _harness import contraction_err, dot_bound, gpu_run, oracle_run
from _loader import load_pkg
from oracle import stablehlo_interp as I
from test_gpu_dot import cw_tol, dot_module

pytestmark = pytest.mark.gpu

ORDERS = [(True, True), (True, False), (False, True), (False, False)]
# M, N, K in units of the type's elements per dword; tile = BM,BN,WM,WN,KG,S
SHAPES = [((13, 70, 777), "16,16,1,1,8,4"), ((67, 130, 65), "64,64,2,2,2,3"), ((101, 77, 131), "32,64,2,2,4,2"), ((200, 33, 1000), "128,64,2,2,1,2"),
          ((97, 99, 260), "96,96,2,2,1,3"), ((40, 300, 129), "16,32,1,1,4,3"), ((250, 161, 80), "160,128,2,2,1,2")]
CASES = [(dt, shape, tile, o) for dt in ("f32", "f64", "bf16", "f16", "f8E4M3FN") for i, (shape, tile) in enumerate(SHAPES) for o in (ORDERS[i % 4], ORDERS[(i + 1) % 4])]


@pytest.mark.parametrize("dt,shape,tile,order", CASES)
def test_every_edge_with_a_given_tile(rx, client, monkeypatch, dt, shape, tile, order):
    unit = {"f32": 1, "f64": 1, "bf16": 2, "f16": 2, "f8E4M3FN": 4}[dt]     # operand rows are whole dwords
    M, N, K = (v * unit for v in shape)
    out = {"f8E4M3FN": "f32"}.get(dt, dt)
    text, sa, sb = dot_module(M, N, K, dt, out, *order)
    monkeypatch.setenv("RX_GEMM_G", tile)
    monkeypatch.setenv("RX_SPLIT_K", "0")
    src = rx.compile_offline(text, with_source=True)
    assert re.search(r"rx_gemm_body_g<rx_el_\w+, %s, " % tile.replace(",", ", "), src), src[:500]
    a, b = (I.tensor(np.random.default_rng(s).normal(size=z), dt) for s, z in ((0, sa), (1, sb)))
    got, exe = gpu_run(rx, client, text, [a, b])
    assert len(exe.launches()) == 1
    ref = oracle_run(text, [a, b], hifi=True)
    assert contraction_err(got[0].a, ref[0].a, dot_bound(text, [a, b])) <= cw_tol(dt, out)


@pytest.mark.parametrize("dt,M,N,K,order,batch", [("f32", 1001, 777, 153, (True, False), 0), ("f64", 129, 515, 301, (False, True), 0), ("bf16", 1, 4096, 784, (True, False), 0),
                                                   ("bf16", 29, 10, 2048, (True, False), 0), ("f8E4M3FN", 6, 4096, 512, (True, True), 0), ("f32", 77, 65, 131, (True, True), 5),
                                                   ("bf16", 60, 68, 130, (False, False), 3), ("f32", 3, 4096, 784, (True, False), 0)])
def test_the_tiles_the_planner_picks(rx, client, dt, M, N, K, order, batch):
    out = {"f8E4M3FN": "f32"}.get(dt, dt)
    text, sa, sb = dot_module(M, N, K, dt, out, *order, batch)
    assert "rx_gemm_body_g<" in load_pkg().compile_offline(text, with_source=True)
    a, b = (I.tensor(np.random.default_rng(s).normal(size=z), dt) for s, z in ((2, sa), (3, sb)))
    got, exe = gpu_run(rx, client, text, [a, b])
    assert len(exe.launches()) == 1
    ref = oracle_run(text, [a, b], hifi=True)
    assert contraction_err(got[0].a, ref[0].a, dot_bound(text, [a, b])) <= cw_tol(dt, out)


def test_rows_past_an_edge_do_not_leak_into_others(rx, client):
    """Infinities in the row after a K tail and in the rows past the last tile's edge stay in their own rows."""
    text, sa, sb = dot_module(70, 66, 131, "f32", "f32", True, True)
    a, b = np.random.default_rng(4).normal(size=sa).astype(np.float32), np.random.default_rng(5).normal(size=sb).astype(np.float32)
    a[17], b[40] = np.inf, np.inf
    got, _ = gpu_run(rx, client, text, [I.Tensor(a, "f32"), I.Tensor(b, "f32")])
    fin = np.isfinite(got[0].a)
    assert not fin[17].any() and not fin[:, 40].any()
    assert fin[np.arange(70) != 17][:, np.arange(66) != 40].all()
