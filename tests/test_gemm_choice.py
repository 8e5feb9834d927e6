"""Which MFMA skeleton a product is planned on and that its kernel compiles, without a device."""
import re

import pytest

from _loader import load_pkg
from test_gpu_dot import dot_module

rx = load_pkg()


def skeleton(*args):
    m = re.search(r"(rx_gemm_body\w*)<([^\n]*)>\(A, B, epi", rx.compile_offline(dot_module(*args)[0], with_source=True))
    return m.group(1) if m else None


# (K + 64) rows of 4 M bytes reach 2^32 at M = 2^23 (K = 64): below it the body with split operands, from it on another one
@pytest.mark.parametrize("tall,other,k", [(6_000_000, 128, 64), (8_388_600, 128, 64), (6_000_000, 256, 80)])
def test_f32_products_of_a_tall_matrix_compile(tall, other, k):
    assert skeleton(tall, other, k, "f32", "f32", False, True) == "rx_gemm_body_x"
    assert skeleton(other, tall, k, "f32", "f32", True, False) == "rx_gemm_body_x"


def test_f32_products_past_the_offset_bound_compile():
    assert skeleton(8_388_608, 128, 64, "f32", "f32", False, True) not in (None, "rx_gemm_body_x", "rx_gemm_body_g")
    assert skeleton(128, 8_388_608, 64, "f32", "f32", True, False) not in (None, "rx_gemm_body_x", "rx_gemm_body_g")


def test_one_stage_serves_one_tile(monkeypatch):
    """A tile asked for with one LDS stage is refused (the planner's own is taken) where a group has more than one K tile."""
    def text(k, spec):
        monkeypatch.setenv("RX_GEMM_G", spec)
        return rx.compile_offline(dot_module(256, 256, k, "f32", "f32", True, True)[0], with_source=True)
    assert "rx_gemm_body_g<rx_el_f32, 64, 64, 2, 2, 1, 1, " not in text(512, "64,64,2,2,1,1")
    assert "rx_gemm_body_g<rx_el_f32, 64, 64, 2, 2, 1, 2, " in text(512, "64,64,2,2,1,2")
    assert "rx_gemm_body_g<rx_el_f32, 64, 64, 2, 2, 2, 1, " in text(64, "64,64,2,2,2,1")


@pytest.mark.parametrize("dt,m,n,k", [("f64", 576, 3456, 1024), ("f32", 576, 3456, 1024), ("f64", 704, 1152, 2048), ("bf16", 1344, 704, 1024), ("f64", 3904, 320, 1216),
                                      ("f64", 1600, 2496, 2944), ("f32", 664, 4096, 1024), ("f32", 1001, 777, 1531), ("f64", 2076, 2008, 1544), ("f32", 4096, 4096, 4096)])
def test_every_xcd_takes_its_share_of_the_tiles(dt, m, n, k):
    """The order in which workgroups (dealt to eight XCDs of 32 compute units in turn) walk the tiles: no XCD takes a tenth more
    rounds of tiles than an even share."""
    text = rx.compile_offline(dot_module(m, n, k, dt, dt, True, False)[0], with_source=True)
    args = re.search(r"rx_gemm_body_[gx]<(?:rx_el_\w+, )?([^>]*)>\(A, B, epi", text).group(1)
    x = re.match(r"(\d+), (\d+), [^a-z]*(?:(?:true|false), )+%d, %d, %d, (\d+), (\d+)," % (m, n, k), args)
    bm, bn, rb, cb = (int(v) for v in x.groups())
    gm, gn = -(-m // bm), -(-n // bn)
    load = [0] * 8
    if rb == 0:
        load = [len(range(x, gm * gn, 8)) for x in range(8)]
    else:
        for i, (r, c) in enumerate((r, c) for r in range(0, gm, rb) for c in range(0, gn, cb)):
            load[i % 8] += min(rb, gm - r) * min(cb, gn - c)
    even = -(-gm * gn // 8)
    assert sum(load) == gm * gn
    assert -(-max(load) // 32) <= 1.1 * -(-even // 32), (load, even)


@pytest.mark.parametrize("dt,m,n,k", [("f32", 276, 4096, 2048), ("f32", 615, 2048, 3000), ("f64", 1408, 1984, 3840), ("f64", 2432, 1472, 1920)])
def test_many_rounds_of_tiles_are_not_those_of_lone_wavefronts(dt, m, n, k):
    text = rx.compile_offline(dot_module(m, n, k, dt, dt, True, False)[0], with_source=True)
    wm, wn = re.search(r"rx_gemm_body_g<rx_el_\w+, \d+, \d+, (\d+), (\d+), ", text).groups()
    assert int(wm) * int(wn) > 2


# rows, columns, K and whether the matrix is stored [o][k]
@pytest.mark.parametrize("dt,m,n,k,kc,gemm", [("f32", 1, 1024, 8192, True, False), ("f32", 1, 8192, 1024, True, False), ("f32", 1, 2048, 4096, False, True), ("f32", 2, 1024, 8192, True, True),
                                              ("f64", 1, 512, 4096, False, False), ("f64", 1, 2048, 1024, False, True), ("f64", 1, 2048, 1024, True, False), ("f64", 2, 4096, 4096, False, False),
                                              ("f64", 2, 2048, 4096, True, True), ("f64", 2, 1024, 4096, True, False), ("f64", 3, 4096, 4096, False, True), ("f64", 3, 512, 8192, True, False),
                                              ("f64", 4, 512, 8192, False, False), ("f64", 4, 1024, 4096, False, True), ("bf16", 1, 1024, 8192, True, True), ("f8E4M3FN", 6, 4096, 4096, True, True)])
def test_few_rows_go_where_they_are_fast(dt, m, n, k, kc, gemm):
    out = "f32" if dt.startswith("f8") else dt
    assert ("kind=gemm" in rx.compile_offline(dot_module(m, n, k, dt, out, True, kc)[0])) == gemm


@pytest.mark.parametrize("dt,m,n,k,orders,slices", [("bf16", 32, 4096, 25088, (True, False), 8), ("bf16", 16, 2048, 8192, (True, False), 16), ("f16", 64, 4096, 18432, (True, True), 8),
                                                    ("bf16", 4096, 20, 8192, (False, True), 8), ("f8E4M3FN", 16, 4096, 8192, (True, False), 8), ("bf16", 32, 4096, 4096, (True, False), 8), ("bf16", 16, 4096, 4096, (True, False), 1), ("bf16", 40, 4096, 4096, (True, False), 1),
                                                    ("bf16", 32, 8192, 8192, (True, False), 1), ("bf16", 16, 1000, 25088, (True, False), 0), ("bf16", 32, 1000, 25088, (True, False), 0),
                                                    ("bf16", 32, 8192, 18432, (True, False), 0), ("bf16", 32, 4096, 18432, (True, True), 1)])
def test_long_matrices_against_few_rows_are_cut_on_the_ring_skeleton(dt, m, n, k, orders, slices):
    """0: cut, but not on that skeleton."""
    out = "f32" if dt.startswith("f8") else dt
    text, _, _ = dot_module(m, n, k, dt, out, *orders)
    text = text.replace("return %0", "%%1 = stablehlo.add %%0, %%0 : (T, T) -> T\n    return %%1".replace("%%", "%").replace("T", "tensor<%dx%dx%s>" % (m, n, out)))
    src = rx.compile_offline(text, with_source=True)
    cut = int(re.search(r"kind=gemm_\w+ grid=\d+x(\d+)x1", src).group(1))
    assert ("rx_gemm_body_dl<" in src) == (slices > 1)
    assert cut == slices if slices else cut > 1


@pytest.mark.parametrize("dt,m,n,k,cut", [("f32", 256, 256, 2048, True), ("bf16", 512, 1024, 4096, True), ("bf16", 512, 1024, 2048, False), ("f32", 512, 1024, 2048, False)])
def test_which_products_without_a_consumer_are_cut(dt, m, n, k, cut):
    rep = rx.compile_offline(dot_module(m, n, k, dt, dt, False, False)[0])
    assert (int(re.search(r"kind=gemm_\w+ grid=\d+x(\d+)x1", rep).group(1)) > 1) == cut


HELD = """module {
  func.func @main(%%arg0: tensor<%(m)dx2048x%(dt)s>, %%arg1: tensor<1024x2048x%(dt)s>, %%arg2: tensor<%(m)dx1024x%(dt)s>) -> (%(types)s) {
    %%0 = stablehlo.dot_general %%arg0, %%arg1, contracting_dims = [1] x [1], precision = [DEFAULT, DEFAULT] : (tensor<%(m)dx2048x%(dt)s>, tensor<1024x2048x%(dt)s>) -> T
%(body)s
  }
}
"""
D = "    %1 = stablehlo.subtract %0, %arg2 : T\n"
TWO = D + "    %2 = stablehlo.multiply %1, %1 : T\n    %3 = stablehlo.tanh %1 : T\n    return %2, %3 : T, T"
ONE = D + "    %2 = stablehlo.tanh %1 : T\n    return %2 : T"
JOINED = D + "    %2 = stablehlo.tanh %1 : T\n    %3 = stablehlo.multiply %1, %2 : T\n    return %3 : T"
LATE = D + "    %2 = stablehlo.tanh %1 : T\n    %3 = stablehlo.multiply %1, %2 : T\n    %4 = stablehlo.multiply %3, %3 : T\n    %5 = stablehlo.exponential %3 : T\n    return %4, %5 : T, T"
EXACT = D + "    %2 = stablehlo.abs %1 : T\n    %3 = stablehlo.negate %1 : T\n    return %2, %3 : T, T"


# what is computed from the product: several results of one value, one result, one result by two ways, one value by two ways that
# several results are computed from, several results without a rounding of their own
@pytest.mark.parametrize("dt,m,body,results,cut", [("bf16", 185, TWO, 2, True), ("f16", 64, TWO, 2, True), ("bf16", 185, ONE, 1, False), ("bf16", 185, JOINED, 1, False),
                                                   ("bf16", 185, LATE, 2, False), ("bf16", 185, EXACT, 2, False), ("bf16", 4096, TWO, 2, False)])
def test_products_that_several_results_are_computed_from_are_held_in_f32(dt, m, body, results, cut):
    ty = "tensor<%dx1024x%s>" % (m, dt)
    text = HELD % {"m": m, "dt": dt, "types": ", ".join([ty] * results), "body": body}
    rep = rx.compile_offline(re.sub(r"\bT\b", ty, text))
    assert (int(re.search(r"kind=gemm\w* grid=\d+x(\d+)x1", rep).group(1)) > 1) == cut
