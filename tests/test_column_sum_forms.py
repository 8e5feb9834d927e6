"""Column sums in one launch or two: by the rows, by what an element costs, and by whether a product of the module can run beside
them; and the results of the loop's forms (whole batches of rows, rounds left over, rows left over, one round, none)."""
import numpy as np
import pytest

from _harness import gpu_run, oracle_run
from _loader import load_pkg
from oracle import stablehlo_interp as I

rx = load_pkg()


def column_sums(rows, cols, dt, ops=(), product=False):
    t, s, o, q = "tensor<%dx%dx%s>" % (rows, cols, dt), "tensor<%s>" % dt, "tensor<%dx%s>" % (cols, dt), "tensor<64x64x%s>" % dt
    v, lines = "%a", []
    for i, op in enumerate(ops):
        lines.append("%%m%d = stablehlo.%s %s : %s" % (i, op, v if op in ("tanh", "abs", "negate") else v + ", %a", t))
        v = "%%m%d" % i
    lines.append("%%r = stablehlo.reduce(%s init: %%i) applies stablehlo.add across dimensions = [0] : (%s, %s) -> %s" % (v, t, s, o))
    if product:
        lines.append("%%p = stablehlo.dot_general %%b, %%b, contracting_dims = [1] x [0] : (%s, %s) -> %s" % (q, q, q))
    ret = ("%r, %p", "%s, %s" % (o, q)) if product else ("%r", o)
    return ("module {\n  func.func @main(%%a: %s, %%i: %s%s) -> (%s) {\n    %s\n    return %s : %s\n  }\n}\n"
            % (t, s, ", %%b: %s" % q if product else "", ret[1], "\n    ".join(lines), ret[0], ret[1]))


@pytest.mark.parametrize("rows,dt,ops,product,launches,block", [
    (1024, "bf16", (), False, 1, 256), (1025, "bf16", (), False, 1, 1024), (4096, "f32", ("multiply",) * 12, False, 1, 1024), (4097, "f32", (), False, 2, None),
    (1024, "f32", ("tanh",), False, 1, 256), (1025, "f32", ("tanh",), False, 2, None), (1000, "bf16", ("divide",) * 3, False, 1, 256), (1000, "f32", ("divide",) * 4, False, 2, None),
    (768, "f32", ("divide",) * 4, False, 1, 256), (4096, "bf16", ("multiply",) * 2, True, 1, 256), (2048, "bf16", ("multiply",) * 3, True, 1, 256), (2049, "bf16", ("multiply",) * 3, True, 2, None)])
def test_launches(rows, dt, ops, product, launches, block):
    report = rx.compile_offline(column_sums(rows, 1024, dt, ops, product), True)
    assert ("combine partials" in report) == (launches == 2), report[:2000]
    assert block is None or " part[%d][" % (block // 4) in report, report[:2000]     # threads' sums, four vectors of outputs side by side


@pytest.mark.parametrize("n,launches", [(2, 2), (3, 1)])
def test_partial_results_stay_within_what_a_call_without_allocations_holds(n, launches):
    """1.9 MB of partial results per sum, 4 MiB for all"""
    t, o = "tensor<4096x2000xbf16>", "tensor<2000xbf16>"
    lines = ["%%m%d = stablehlo.tanh %%a%d : %s\n    %%r%d = stablehlo.reduce(%%m%d init: %%z) applies stablehlo.add across dimensions = [0] : (%s, tensor<bf16>) -> %s" % (i, i, t, i, i, t, o) for i in range(n)]
    text = ("module {\n  func.func @main(%s) -> (%s) {\n    %%z = stablehlo.constant dense<0.0> : tensor<bf16>\n    %s\n    return %s : %s\n  }\n}\n"
            % (", ".join("%%a%d: %s" % (i, t) for i in range(n)), ", ".join([o] * n), "\n    ".join(lines), ", ".join("%%r%d" % i for i in range(n)), ", ".join([o] * n)))
    assert ("combine partials" in rx.compile_offline(text)) == (launches == 2)


@pytest.mark.gpu
@pytest.mark.parametrize("dt", ["f32", "f64", "bf16", "i32"])
@pytest.mark.parametrize("rows", [65, 127, 640, 1021, 1024, 1025, 1279, 1280, 3333, 4095, 4096])
@pytest.mark.parametrize("cols,product", [(520, False), (1000, True)])
def test_results(rx, client, rows, cols, dt, product):
    text = column_sums(rows, cols, dt, ("negate",), product)
    rng = np.random.default_rng(rows)
    # whole numbers whose sums are exact in every accumulator, and in bf16 once rounded
    args = [I.tensor(rng.integers(-2, 3, size=(rows, cols)), dt), I.tensor(np.asarray(-3), dt)] + ([I.tensor(rng.integers(-1, 2, size=(64, 64)), dt)] if product else [])
    got, exe = gpu_run(rx, client, text, args)
    assert ("combine partials" in exe.report()) == (rows * cols * {"f32": 4, "f64": 8, "bf16": 2, "i32": 4}[dt] > 16 << 20)
    for g, r in zip(got, oracle_run(text, args, hifi=True)):
        assert np.array_equal(np.asarray(g.a), np.asarray(r.a))
