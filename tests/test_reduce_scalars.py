"""Reductions whose elements, initial value and scalar end read the same scalar: the end is code outside of the loop that read
it for the elements."""
import numpy as np
import pytest

from _harness import gpu_run, oracle_run
from _loader import load_pkg
from oracle import stablehlo_interp as I

rx = load_pkg()
BODIES = {
    "init": ["%m = stablehlo.multiply %a, %b : T", "%r = stablehlo.reduce(%m init: %s) applies stablehlo.add across dimensions = [0] : (T, S) -> S"],
    "tail": ["%m = stablehlo.subtract %a, %b : T", "%0 = stablehlo.reduce(%m init: %z) applies stablehlo.add across dimensions = [0] : (T, S) -> S", "%r = stablehlo.multiply %0, %s : S"],
    "both": ["%d = stablehlo.subtract %a, %b : T", "%m = stablehlo.multiply %d, %d : T",
             "%0 = stablehlo.reduce(%m init: %s) applies stablehlo.add across dimensions = [0] : (T, S) -> S", "%r = stablehlo.subtract %0, %s : S"],
}


def full(n, dt, form):
    lines = ["%z = stablehlo.constant dense<0.0> : S", "%b = stablehlo.broadcast_in_dim %s, dims = [] : (S) -> T"] + BODIES[form]
    text = "module {\n  func.func @main(%a: T, %s: S) -> S {\n    " + "\n    ".join(lines) + "\n    return %r : S\n  }\n}\n"
    return text.replace("T", "tensor<%dx%s>" % (n, dt)).replace("S", "tensor<%s>" % dt)


@pytest.mark.parametrize("form", sorted(BODIES))
@pytest.mark.parametrize("n", [1, 2, 4099, 8192, 8193])
def test_full_reductions_compile(n, form):
    report = rx.compile_offline(full(n, "f32", form))
    assert report.count("kind=") == (1 if n <= 8192 else 2), report


@pytest.mark.gpu
@pytest.mark.parametrize("dt", ["f32", "f64", "bf16"])
@pytest.mark.parametrize("form", sorted(BODIES))
@pytest.mark.parametrize("n", [1, 4099, 8192, 8193])
def test_full_reductions(rx, client, n, form, dt):
    text = full(n, dt, form)
    rng = np.random.default_rng(n)
    args = [I.tensor(rng.integers(-1, 2, size=n), dt), I.tensor(np.asarray(2), dt)]   # whole numbers: sums are exact in every accumulator
    got, _ = gpu_run(rx, client, text, args)
    assert np.array_equal(np.asarray(got[0].a), np.asarray(oracle_run(text, args, hifi=True)[0].a))


def some_dims(shape, dim, dt):
    """sum(a .* s; dims, init = s)"""
    text = ("module {\n  func.func @main(%a: T, %s: S) -> O {\n    %b = stablehlo.broadcast_in_dim %s, dims = [] : (S) -> T\n    %m = stablehlo.multiply %a, %b : T\n"
            "    %r = stablehlo.reduce(%m init: %s) applies stablehlo.add across dimensions = [DIM] : (T, S) -> O\n    return %r : O\n  }\n}\n")
    dims = ["".join("%dx" % d for k, d in enumerate(shape) if not drop or k != dim) for drop in (False, True)]
    return text.replace("DIM", str(dim)).replace("T", "tensor<%s%s>" % (dims[0], dt)).replace("S", "tensor<%s>" % dt).replace("O", "tensor<%s%s>" % (dims[1], dt))


# one launch by columns, two launches, one thread per output (eight and one at a time), two kept dimensions, a row kernel
FORMS = [((1024, 1024), 0), ((65, 1000), 0), ((4097, 512), 0), ((300, 7), 0), ((20, 4096), 0), ((3, 3), 1), ((3, 130, 1024), 1), ((16, 40, 300), 1), ((8, 640, 128), 0), ((70, 400), 1)]


@pytest.mark.parametrize("dt", ["f32", "bf16", "f64"])
@pytest.mark.parametrize("shape,dim", FORMS)
def test_reductions_of_some_dimensions_compile(shape, dim, dt):
    assert "code object" in rx.compile_offline(some_dims(shape, dim, dt))


@pytest.mark.gpu
@pytest.mark.parametrize("dt", ["f32", "bf16", "f64"])
@pytest.mark.parametrize("shape,dim", FORMS)
def test_reductions_of_some_dimensions(rx, client, shape, dim, dt):
    text = some_dims(shape, dim, dt)
    rng = np.random.default_rng(shape[0])
    args = [I.tensor(rng.integers(-1, 2, size=shape), dt), I.tensor(np.asarray(2), dt)]   # sums are exact in every accumulator
    got, _ = gpu_run(rx, client, text, args)
    assert np.array_equal(np.asarray(got[0].a), np.asarray(oracle_run(text, args, hifi=True)[0].a))


@pytest.mark.parametrize("op,n,dt,launches", [("tanh", 4096, "f64", 1), ("tanh", 4097, "f64", 2), ("log_plus_one", 8192, "f64", 2), ("sine", 8192, "f64", 1), ("tanh", 8192, "f32", 1), ("lgamma", 1024, "f64", 1), ("lgamma", 1025, "f64", 2), ("digamma", 4097, "f32", 2)])
def test_one_workgroup_or_two_launches(op, n, dt, launches):
    text = ("module {\n  func.func @main(%a: T) -> S {\n    %z = stablehlo.constant dense<0.0> : S\n    %m = OP\n"
            "    %r = stablehlo.reduce(%m init: %z) applies stablehlo.add across dimensions = [0] : (T, S) -> S\n    return %r : S\n  }\n}\n").replace("OP", "chlo.%s %%a : T -> T" % op if op in ("lgamma", "digamma") else "stablehlo.%s %%a : T" % op)
    report = rx.compile_offline(text.replace("T", "tensor<%dx%s>" % (n, dt)).replace("S", "tensor<%s>" % dt))
    assert report.count("kind=") == launches, report
