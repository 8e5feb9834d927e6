"""Elementwise ops on the scalar of a full reduction run in its kernel."""
import numpy as np
import pytest

from _harness import gpu_run, oracle_run
from oracle import stablehlo_interp as I

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", ["f32", "f64", "bf16", "i32"])
@pytest.mark.parametrize("n", [1, 4099, 9001])     # one launch, one, two
def test_scalar_ops_of_a_reduction(rx, client, n, dt):
    """(max(x, i) * s - i), the init value and the scale arguments; the plain reduction where it is a result as well."""
    t, s = "tensor<%dx%s>" % (n, dt), "tensor<%s>" % dt
    head = "module {\n  func.func @main(%%a: %s, %%i: %s, %%s: %s) -> " % (t, s, s)
    body = ("    %%0 = stablehlo.reduce(%%a init: %%i) applies stablehlo.maximum across dimensions = [0] : (%s, %s) -> %s\n"
            "    %%1 = stablehlo.multiply %%0, %%s : %s\n    %%2 = stablehlo.subtract %%1, %%i : %s\n" % (t, s, s, s, s))
    rng = np.random.default_rng(n)
    args = [I.tensor(rng.integers(-9, 10, size=n), dt), I.tensor(np.asarray(-3), dt), I.tensor(np.asarray(5), dt)]   # exact in every type
    for res, kinds in (("%2", ["reduce"] if n <= 8192 else ["reduce", "reduce_final"]), ("%0, %2", (["reduce"] if n <= 8192 else ["reduce", "reduce_final"]) + ["map"])):
        types = ", ".join([s] * (res.count(",") + 1))
        text = head + "(%s) {\n" % types + body + "    return %s : %s\n  }\n}\n" % (res, types)
        got, exe = gpu_run(rx, client, text, args)
        assert [l["kind"] for l in exe.launches()] == kinds
        for g, r in zip(got, oracle_run(text, args)):
            assert np.array_equal(np.asarray(g.a), np.asarray(r.a))
