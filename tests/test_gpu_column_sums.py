"""Column reductions of small matrices in one launch: rows that are not a multiple of the threads' stride, ragged last workgroups,
every element size, an initial value that is an argument, a batch dimension, and the sizes from which two launches remain."""
import numpy as np
import pytest

from _harness import gpu_run, oracle_run
from oracle import stablehlo_interp as I

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", ["f32", "f64", "bf16", "f16", "i32", "i64"])
@pytest.mark.parametrize("shape,dim,op,launches", [([64, 520], 0, "add", 1), ([65, 1000], 0, "add", 1), ([1021, 528], 0, "add", 1), ([4096, 512], 0, "add", 1),
                                                   ([4097, 512], 0, "add", 2), ([300, 1032], 0, "maximum", 1), ([3, 130, 1024], 1, "add", 1)])
def test_columns(rx, client, shape, dim, op, launches, dt):
    t, s = "tensor<%s%s>" % ("".join("%dx" % d for d in shape), dt), "tensor<%s>" % dt
    out = "tensor<%s%s>" % ("".join("%dx" % d for k, d in enumerate(shape) if k != dim), dt)
    text = ("module {\n  func.func @main(%%a: %s, %%i: %s) -> %s {\n    %%0 = stablehlo.reduce(%%a init: %%i) applies stablehlo.%s across dimensions = [%d] : (%s, %s) -> %s\n"
            "    return %%0 : %s\n  }\n}\n" % (t, s, out, op, dim, t, s, out, out))
    rng = np.random.default_rng(shape[0])
    x = rng.integers(-9, 10, size=shape).astype(np.float64) if dt[0] == "i" else rng.normal(size=shape)
    if op == "maximum" and dt[0] != "i":
        x[7] = -np.inf
        x[:, 11] = -np.inf
    args = [I.tensor(x, dt), I.tensor(np.asarray(-3), dt)]
    got, exe = gpu_run(rx, client, text, args)
    assert len(exe.launches()) == launches, exe.report()
    g, r = np.asarray(got[0].a, dtype=np.float64), np.asarray(oracle_run(text, args, hifi=True)[0].a, dtype=np.float64)
    if dt[0] == "i" or op == "maximum":
        assert np.array_equal(g, r)
    else:
        # at most 64 additions in a thread, 64 of its workgroup's sums and the init value: 129 roundings of the sum of magnitudes
        eps = 2.0 ** -53 if dt == "f64" else 2.0 ** -24
        half = {"bf16": 2.0 ** -8, "f16": 2.0 ** -10}.get(dt, 0.0)   # the result's own rounding
        bound = 129 * eps * (np.abs(np.asarray(args[0].a, dtype=np.float64)).sum(axis=dim) + 3) + half * np.abs(r)
        assert np.all(np.abs(g - r) <= bound)
