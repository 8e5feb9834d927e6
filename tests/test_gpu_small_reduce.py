"""Full reductions of few elements: one workgroup, one launch, for every reduction and element type, at the edges of a
wavefront, of the workgroup and of the rule's range, with an initial value that is an argument."""
import numpy as np
import pytest

from _harness import gpu_run, oracle_run
from oracle import stablehlo_interp as I

pytestmark = pytest.mark.gpu


def module(n, dt, op):
    t, s = "tensor<%dx%s>" % (n, dt), "tensor<%s>" % dt
    return ("module {\n  func.func @main(%%arg0: %s, %%arg1: %s) -> %s {\n"
            "    %%0 = stablehlo.reduce(%%arg0 init: %%arg1) applies stablehlo.%s across dimensions = [0] : (%s, %s) -> %s\n"
            "    return %%0 : %s\n  }\n}\n" % (t, s, s, op, t, s, s, s))


@pytest.mark.parametrize("dt", ["f32", "f64", "bf16", "i32", "i64"])
@pytest.mark.parametrize("n,op", [(1, "add"), (63, "maximum"), (65, "add"), (1023, "minimum"), (1025, "add"), (4096, "maximum"), (4099, "add"), (8191, "add"), (8192, "add"),
                                  (8193, "add")])
def test_one_launch(rx, client, n, op, dt):
    rng = np.random.default_rng(n)
    x = rng.integers(-9, 10, size=n) if dt[0] == "i" else rng.normal(size=n)
    if op != "add" and dt[0] != "i":
        x[n // 2] = {"maximum": -np.inf, "minimum": np.inf}[op]
    a, b = I.tensor(x, dt), I.tensor(np.asarray(3), dt)
    text = module(n, dt, op)
    got, exe = gpu_run(rx, client, text, [a, b])
    assert [l["kind"] for l in exe.launches()] == (["reduce"] if n <= 8192 else ["reduce", "reduce_final"])
    ref = oracle_run(text, [a, b], hifi=True)
    g, r = np.float64(got[0].a), np.float64(ref[0].a)
    # at most 11 additions in a thread, 6 in a wavefront, 16 across them and the initial value: 34 roundings of the sum of magnitudes
    bound = 0.0 if dt[0] == "i" or op != "add" else (np.abs(np.float64(a.a)).sum() + 3) * 34 * {"f32": 2.0 ** -24, "f64": 2.0 ** -53, "bf16": 2.0 ** -24}[dt]
    assert abs(g - r) <= bound + (abs(r) * 2.0 ** -8 if dt == "bf16" else 0.0)
