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


X_TILES = ["128,128,2,2,1,1,1", "128,128,2,2,2,1,1", "128,256,2,4,1,1,1", "256,128,4,2,1,1,1", "64,64,2,1,2,1,1"]
# edges of both dimensions and of K inside a vector, one K tile for each of two groups, whole tiles, batches
X_SHAPES = [(129, 260, 77, 0), (300, 131, 1030, 0), (128, 256, 64, 0), (70, 515, 96, 0), (130, 66, 131, 3)]


def x_fits(tile, order):
    bm, bn, wm, wn = (int(v) for v in tile.split(",")[:4])
    return (order[0] or bm * 2 % (wm * wn * 64) == 0) and (order[1] or bn * 2 % (wm * wn * 64) == 0)


@pytest.mark.parametrize("tile,shape,order", [(t, s, o) for t in X_TILES for i, s in enumerate(X_SHAPES) for o in (ORDERS[i % 4], ORDERS[(i + 1) % 4]) if x_fits(t, o)])
def test_f32_operands_split_into_bf16(rx, client, monkeypatch, tile, shape, order):
    """Componentwise within what two roundings of the sum per 32 k and the terms left out allow, (K / 16 + 2) 2^-24 of |A| . |B|."""
    M, N, K, batch = shape
    text, sa, sb = dot_module(M, N, K, "f32", "f32", *order, batch)
    monkeypatch.setenv("RX_GEMM_G", tile)
    monkeypatch.setenv("RX_SPLIT_K", "0")
    assert "rx_gemm_body_x<" in rx.compile_offline(text, with_source=True)
    a, b = (I.tensor(np.random.default_rng(s).normal(size=z), "f32") for s, z in ((6, sa), (7, sb)))
    got, exe = gpu_run(rx, client, text, [a, b])
    ref = oracle_run(text, [a, b], hifi=True)
    assert contraction_err(got[0].a, ref[0].a, dot_bound(text, [a, b])) <= (K / 16 + 2) * 2.0 ** -24


@pytest.mark.parametrize("order", ORDERS)
def test_numbers_that_do_not_split_into_bf16(rx, client, monkeypatch, order):
    """Infinities, NaN, numbers that round to infinity in bf16, subnormals: as the f32 MFMAs of the general path have them."""
    M, N, K = 140, 130, 70
    text, sa, sb = dot_module(M, N, K, "f32", "f32", *order)
    rng = np.random.default_rng(8)
    A, B = rng.normal(size=(M, K)).astype(np.float32), rng.normal(size=(N, K)).astype(np.float32)
    A[3, 5], A[4, 6], A[5, 69], A[131, 7], B[129, 0] = np.inf, -np.inf, np.nan, np.float32(3.4e38), np.inf
    B[:, 7] *= np.float32(1e-3)                       # finite sums with the largest numbers
    A[20:24] = rng.normal(size=(4, K)) * 1e-36        # bits below what bf16 holds
    A[24:28] = rng.normal(size=(4, K)) * 1e-40        # subnormal
    A[28], A[28, 1], B[40, :] = 0, 1e-37, 0           # one tiny product alone
    B[40, 1] = 1 + 2.0 ** -20
    a, b = (I.Tensor(np.ascontiguousarray(x if kc else x.T), "f32") for x, kc in ((A, order[0]), (B, order[1])))
    out = {}
    for tile in ("0", "128,128,2,2,1,1,1", "128,128,2,2,2,1,1"):
        monkeypatch.setenv("RX_GEMM_G", tile)
        assert ("rx_gemm_body_x<" in rx.compile_offline(text, with_source=True)) == (tile != "0")
        out[tile] = gpu_run(rx, client, text, [a, b])[0][0].a
    ref = out.pop("0")
    with np.errstate(all="ignore"):
        exact = A.astype(np.float64) @ B.astype(np.float64).T
        bound = np.abs(A).astype(np.float64) @ np.abs(B).astype(np.float64).T
    for got in out.values():
        assert np.array_equal(np.isnan(got), np.isnan(ref)) and np.array_equal(np.isposinf(got), np.isposinf(ref)) and np.array_equal(np.isneginf(got), np.isneginf(ref))
        fin = np.isfinite(ref)
        # a rounding per product and K 2^-149 for sums that are subnormal
        assert (np.abs(got[fin].astype(np.float64) - exact[fin]) <= bound[fin] * (K + 2) * 2.0 ** -24 + K * 2.0 ** -149).all()


def test_large_f32_products_take_the_split(rx):
    for (m, n, k, order) in ((4096, 4096, 4096, ORDERS[1]), (2048, 2048, 2048, ORDERS[3]), (2000, 3000, 500, ORDERS[0])):
        assert "rx_gemm_body_x<" in rx.compile_offline(dot_module(m, n, k, "f32", "f32", *order)[0], with_source=True)
    assert "rx_gemm_body_g<" in rx.compile_offline(dot_module(777, 1001, 1531, "f32", "f32", True, False)[0], with_source=True)


# A rounding is at most u, and u / sqrt(3) in the mean square, of the sum that it rounds.  Sums of n positive terms from zero
# are rounded n times, at a third of their square in the mean, and m such sums in one result average out: sqrt(n / 3 m) of that.
# Up to eight rows: n = 32 (f64 16, 16-bit operands 4 MFMAs), in totals with more bits, fewer than 24 sums nowhere here, and the
# rounding of the result; the sums of four before them add a third of u: 0.8 u.  More rows: n = 512, m = 8, in totals
# of the same type: 2.9 u.
@pytest.mark.parametrize("dt,M,N,K,units", [("f32", 2, 1024, 25088, 0.8), ("f32", 6, 4096, 4096, 0.8), ("f32", 3, 4096, 784, 0.8), ("f32", 1, 2048, 4096, 0.8),
                                            ("f64", 3, 512, 4096, 0.8), ("f64", 6, 1024, 784, 0.8), ("bf16", 2, 1024, 4096, 0.8), ("bf16", 6, 1000, 25088, 0.8),
                                            ("f32", 16, 4096, 4096, 2.9)])
def test_long_sums_of_one_sign(rx, client, monkeypatch, dt, M, N, K, units):
    """The error of few rows against a matrix does not grow with K (2-norm, operands uniform in [0, 1))."""
    out = {"bf16": "f32"}.get(dt, dt)
    text, sa, sb = dot_module(M, N, K, dt, out, True, False)
    a, b = (I.tensor(np.random.default_rng(s).random(size=z), dt) for s, z in ((9, sa), (10, sb)))
    got, exe = gpu_run(rx, client, text, [a, b])
    assert exe.launches()[0]["kind"].startswith("gemm")
    wide = np.longdouble if dt == "f64" else np.float64
    exact = a.a.astype(wide) @ b.a.astype(wide)
    err = np.sqrt(((got[0].a - exact) ** 2).sum() / (exact ** 2).sum())
    assert err <= 1.25 * units * 2.0 ** (-53 if dt == "f64" else -24), err


@pytest.mark.parametrize("M,N,K,order", [(6, 4096, 512, (True, True)), (1, 1024, 4096, (True, False)), (1024, 8, 1000, (False, True))])
def test_e4m3_products_of_few_rows_sum_as_f32(rx, client, M, N, K, order):
    """2-norm error against 64 bits: four roundings per 128 k of sums of either sign, at half of their square in the mean, and
    that of the result, each u / sqrt(3) in the mean square: u (the f8 MFMA's sums: 250 u)."""
    text, sa, sb = dot_module(M, N, K, "f8E4M3FN", "f32", *order)
    assert "rx_el_f8b" in rx.compile_offline(text, with_source=True)
    a, b = (I.tensor(np.clip(np.random.default_rng(s).normal(size=z) * 80, -448, 448), "f8E4M3FN") for s, z in ((11, sa), (12, sb)))
    got, _ = gpu_run(rx, client, text, [a, b])
    x, y = a.a.astype(np.float64), b.a.astype(np.float64)
    exact = (x if order[0] else x.T) @ (y.T if order[1] else y)
    err = np.sqrt(((got[0].a - exact) ** 2).sum() / (exact ** 2).sum())
    assert err <= 1.5 * 2.0 ** -24, err


def test_every_e4m3_code_of_a_matrix_against_a_row(rx, client):
    """Row n holds code n mod 256 alone, at k = n: its product with ones is the code's value, NaN where that is."""
    N, K = 1024, 1024
    text, sa, sb = dot_module(1, N, K, "f8E4M3FN", "f32", True, True)
    assert "rx_el_f8b" in rx.compile_offline(text, with_source=True)
    w = np.zeros((N, K), dtype=np.uint8)
    w[np.arange(N), np.arange(N)] = np.arange(N) % 256
    b = I.Tensor.from_bytes(w.tobytes(), "f8E4M3FN", sb)
    got, _ = gpu_run(rx, client, text, [I.tensor(np.ones(sa), "f8E4M3FN"), b])
    assert np.array_equal(got[0].a[0], b.a[np.arange(N), np.arange(N)], equal_nan=True)


BIG_X_TILES = ["128,128,2,2,1,1,1", "128,128,2,2,2,1,1", "128,256,2,4,1,1,1", "256,128,4,2,1,1,1"]


@pytest.mark.parametrize("tile,order,batch", [(t, [o for o in ORDERS if x_fits(t, o)][j], 3 * j) for t in BIG_X_TILES for j in (0, 1)])
def test_tiny_numbers_where_they_matter_and_where_not(rx, client, monkeypatch, tile, order, batch):
    """Numbers with bits below what bf16 holds, in a product of several tiles and many K tiles: beside numbers of ordinary size
    they change nothing and no tile is contracted again (the same bits as with numbers that do split in their place); rows
    and columns of nothing else come out as exactly as all others."""
    M, N, K = 300, 290, 1030
    text, sa, sb = dot_module(M, N, K, "f32", "f32", *order, batch)
    monkeypatch.setenv("RX_GEMM_G", tile)
    monkeypatch.setenv("RX_SPLIT_K", "0")
    assert "rx_gemm_body_x<" in rx.compile_offline(text, with_source=True)
    rng = np.random.default_rng(13)
    lead = (batch,) if batch else ()
    A, B = rng.normal(size=lead + (M, K)).astype(np.float32), rng.normal(size=lead + (N, K)).astype(np.float32)

    def run(a, b):
        a, b = (np.ascontiguousarray(x if kc else np.swapaxes(x, -1, -2)) for x, kc in ((a, order[0]), (b, order[1])))
        return gpu_run(rx, client, text, [I.Tensor(a, "f32"), I.Tensor(b, "f32")])[0][0].a.copy()

    a0, a1, b0, b1 = A.copy(), A.copy(), B.copy(), B.copy()
    for x0, x1 in ((a0, a1), (b0, b1)):
        x0[..., ::40, 7], x1[..., ::40, 7] = np.float32(1.2345678e-33), np.float32(2.0 ** -109)
        x0[..., 5, 1029], x1[..., 5, 1029] = np.float32(-1e-41), 0
    # one sum whose ordinary terms cancel, in the K tiles of either of two groups
    b0[..., 70, :] = b1[..., 70, :] = 0
    for x in (a0, a1):
        x[..., 60, [0, 1, 32, 33]] = 3, -3, 5, -5
        x[..., 60, 9] = np.float32(1.2345678e-33) if x is a0 else 0
    for x in (b0, b1):
        x[..., 70, [0, 1, 9, 32, 33]] = 1
    one, two = run(a0, b0), run(a1, b1)
    assert (one[..., 60, 70] == np.float32(1.2345678e-33)).all() and (two[..., 60, 70] == 0).all()
    two[..., 60, 70] = one[..., 60, 70]
    assert np.array_equal(one, two)
    a0[..., 20:24, :] *= np.float32(1e-36)
    a0[..., 290, :] *= np.float32(1e-40)
    b0[..., 150, :] *= np.float32(1e-35)
    b0[..., 40, :] = 0
    got = run(a0, b0).astype(np.float64)
    exact = np.matmul(a0.astype(np.float64), np.swapaxes(b0, -1, -2).astype(np.float64))
    bound = np.matmul(np.abs(a0).astype(np.float64), np.swapaxes(np.abs(b0), -1, -2).astype(np.float64))
    # one rounding per product where a tile is contracted in f32, and K 2^-149 for sums that are subnormal
    assert (np.abs(got - exact) <= bound * (K + 2) * 2.0 ** -24 + K * 2.0 ** -149).all()
    a0[..., 299, 3] = np.inf
    got = run(a0, b0)
    assert not np.isfinite(got[..., 299, :]).any() and np.isfinite(got[..., :299, :]).all()


# K is no whole number of K tiles, of 16-byte chunks or of slices, N odd (f32) or two more than a vector
SLICED = [("f32", 21, 35, 20001), ("f32", 101, 203, 20001), ("bf16", 20, 34, 20002), ("bf16", 100, 202, 20002), ("f16", 20, 34, 20002), ("f16", 100, 202, 20002), ("f8E4M3FN", 20, 36, 20004)]


@pytest.mark.parametrize("dt,M,N,K,order", [c + (o,) for c in SLICED for o in ORDERS])
def test_slices_of_ragged_products(rx, client, dt, M, N, K, order):
    """K cut into slices of a workgroup's groups where nothing divides anything: the last slices' tiles lie past K."""
    out = {"f8E4M3FN": "f32"}.get(dt, dt)
    text, sa, sb = dot_module(M, N, K, dt, out, *order)
    a, b = (I.tensor(np.random.default_rng(s).normal(size=z), dt) for s, z in ((14, sa), (15, sb)))
    got, exe = gpu_run(rx, client, text, [a, b])
    slices = int(re.search(r"kind=gemm_\w+ grid=\d+x(\d+)x1", exe.report()).group(1))
    assert slices > 1 and K % slices and exe.launches()[1]["kind"].startswith("reduce")
    ref = oracle_run(text, [a, b], hifi=True)
    assert contraction_err(got[0].a, ref[0].a, dot_bound(text, [a, b])) <= cw_tol(dt, out)


def test_the_terms_that_the_split_leaves_out(rx, client, monkeypatch):
    """Constant operands whose left-out terms m l + l m + l l are largest, 1.98 2^-25 of every product and all of one sign."""
    M, N, K = 256, 256, 256
    text, sa, sb = dot_module(M, N, K, "f32", "f32", True, True)
    monkeypatch.setenv("RX_GEMM_G", "128,128,2,2,1,1,1")
    assert "rx_gemm_body_x<" in rx.compile_offline(text, with_source=True)
    x = np.float32(1 + 2.0 ** -8 - 2.0 ** -17)
    got, _ = gpu_run(rx, client, text, [I.Tensor(np.full(sa, x), "f32"), I.Tensor(np.full(sb, x), "f32")])
    exact = K * np.float64(x) ** 2
    # 2^-24 left out, and two roundings per 32 k of sums that are half the result in the mean
    assert np.abs(got[0].a / exact - 1).max() <= 2.0 ** -24 * (1 + K / 32)
