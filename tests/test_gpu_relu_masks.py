"""A relu's mask is read off the relu: the product's kernel writes max(x, 0), and nothing else reads x."""
import numpy as np
import pytest

from _harness import contraction_err, gpu_run, oracle_run
from oracle import stablehlo_interp as I

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", ["f32", "bf16"])
@pytest.mark.parametrize("form", ["GT", "LT"])
def test_the_mask_of_a_relu(rx, client, dt, form):
    """h = max(x W, 0), dx = (x W > 0 ? d : 0): one launch writes h, one reads its sign; NaN, zeros of both signs and tiny sums."""
    m, k, n = 64, 64, 128
    X, W, H, B = ("tensor<%sx%s>" % (s, e) for s, e in (("64x64", dt), ("64x128", dt), ("64x128", dt), ("64x128", "i1")))
    cmp_ = ("%%c = stablehlo.compare GT, %%z, %%k, FLOAT : (%s, %s) -> %s" if form == "GT" else "%%c = stablehlo.compare LT, %%k, %%z, FLOAT : (%s, %s) -> %s") % (H, H, B)
    text = ("module {\n  func.func @main(%%x: %s, %%w: %s, %%d: %s, %%v: %s) -> (%s, %s) {\n"
            "    %%k = stablehlo.constant dense<0.0> : %s\n    %%z = stablehlo.dot_general %%x, %%w, contracting_dims = [1] x [0] : (%s, %s) -> %s\n"
            "    %%h = stablehlo.maximum %%z, %%k : %s\n    %s\n    %%g = stablehlo.dot_general %%d, %%v, contracting_dims = [1] x [0] : (%s, %s) -> %s\n"
            "    %%r = stablehlo.select %%c, %%g, %%k : %s, %s\n    return %%h, %%r : %s, %s\n  }\n}\n"
            % (X, W, X, W, H, H, H, X, W, H, H, cmp_, X, W, H, B, H, H, H))
    rng = np.random.default_rng(1)
    x, w, d, v = rng.normal(size=(m, k)), rng.normal(size=(k, n)), rng.normal(size=(m, k)), rng.normal(size=(k, n))
    x[3] = np.nan
    x[4] = 0.0
    x[5] = -0.0
    x[6] *= 2.0 ** -130
    args = [I.tensor(t, dt) for t in (x, w, d, v)]
    got, exe = gpu_run(rx, client, text, args)
    assert len(exe.launches()) == 2, exe.report()
    ref = oracle_run(text, args)
    for g, r, a, b in ((got[0], ref[0], x, w), (got[1], ref[1], d, v)):
        g, r = np.asarray(g.a, dtype=np.float64), np.asarray(r.a, dtype=np.float64)
        assert np.array_equal(np.isnan(g), np.isnan(r))
        sure = ~np.isnan(r)
        sure[6] = False                       # sums of 1e-39: whether one rounds to zero is the element type's affair
        bound = np.abs(np.asarray(I.tensor(a, dt).a, dtype=np.float64)) @ np.abs(np.asarray(I.tensor(b, dt).a, dtype=np.float64))
        assert contraction_err(g[sure], r[sure], bound[sure]) <= (4e-3 if dt == "bf16" else 1e-6)
    h, r = np.asarray(got[0].a, dtype=np.float64), np.asarray(got[1].a, dtype=np.float64)
    assert np.array_equal(r != 0, h > 0)
