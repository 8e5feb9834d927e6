"""The end of a full reduction in the map that reads its result: the smallest and largest number of partials, a result that later
launches read too, an initial value and element types of other sizes, and the sizes just outside."""
import numpy as np
import pytest

from _harness import gpu_run, oracle_run
from oracle import stablehlo_interp as I

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt,n,folded", [("f32", 64 * 4096, True), ("f32", 63 * 4096 + 4, True), ("f32", 63 * 4096, False), ("f32", 512 * 4096, True), ("f32", 512 * 4096 + 4, False),
                                         ("f64", 64 * 2048, True), ("bf16", 100 * 8192, True), ("i32", 100 * 4096, True)])
def test_results_and_launches(rx, client, dt, n, folded):
    """(max(x, i) - x, and its sum with max(x, i) on top)"""
    t, s = "tensor<%dx%s>" % (n, dt), "tensor<%s>" % dt
    text = ("module {\n  func.func @main(%%a: %s, %%i: %s) -> (%s, %s) {\n"
            "    %%0 = stablehlo.reduce(%%a init: %%i) applies stablehlo.maximum across dimensions = [0] : (%s, %s) -> %s\n"
            "    %%1 = stablehlo.broadcast_in_dim %%0, dims = [] : (%s) -> %s\n    %%2 = stablehlo.subtract %%1, %%a : %s\n"
            "    %%3 = stablehlo.reduce(%%2 init: %%i) applies stablehlo.maximum across dimensions = [0] : (%s, %s) -> %s\n"
            "    %%4 = stablehlo.add %%3, %%0 : %s\n    return %%2, %%4 : %s, %s\n  }\n}\n" % (t, s, t, s, t, s, s, s, t, t, t, s, s, s, t, s))
    rng = np.random.default_rng(n)
    args = [I.tensor(rng.integers(-40, 40, size=n), dt), I.tensor(np.asarray(-50), dt)]   # exact in every type
    got, exe = gpu_run(rx, client, text, args)
    kinds = [l["kind"] for l in exe.launches()]
    assert (kinds[:2] == ["reduce", "map"]) == folded, kinds
    for g, r in zip(got, oracle_run(text, args)):
        assert np.array_equal(np.asarray(g.a), np.asarray(r.a))
