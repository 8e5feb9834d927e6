"""The direct convolution on split operands (rx_conv_body_x): partial slabs of channels, features and tiles, strides,
dilations and layouts of the result's rows, on every grouping of the channels, and the inputs that do not split into three
bf16 numbers.  Bound per element: 1e-6 of |x| * |w|, as for f32 products (the terms left out are 2^-24 of it)."""
import numpy as np
import pytest

from _harness import contraction_err, dot_bound, gpu_run, oracle_run
from _loader import load_pkg
from oracle import stablehlo_interp as I
import _nn_modules as NN

TOL = 1e-6


def _run(rx, client, monkeypatch, xs, ws, kw, x, w, tile=None):
    monkeypatch.setenv("RX_CONV_SPLIT", "2")
    if tile:
        monkeypatch.setenv("RX_CONV_SPLIT_TILE", tile)
    text, _ = NN.convolution(xs, ws, "f32", **kw)
    args = [I.tensor(x, "f32"), I.tensor(w, "f32")]
    got, exe = gpu_run(rx, client, text, args)
    assert [l["kind"] for l in exe.launches()][0] == "filter_split" and exe.launches()[-1]["kind"].startswith("conv"), exe.report()
    return np.asarray(got[0].a), text, args


@pytest.mark.gpu
@pytest.mark.parametrize("xs,ws,kw,tile", [
    ([2, 64, 28, 28], [128, 64, 3, 3], dict(padding=[[1, 1], [1, 1]]), None),
    # 33 channels: one in the second slab; 65 features: one in the last group; columns that are no vectors
    ([1, 33, 9, 11], [65, 33, 3, 3], dict(padding=[[1, 1], [1, 1]]), "2,11,4,1"),
    ([3, 40, 17, 23], [100, 40, 3, 5], dict(strides=[2, 2], rhs_dil=[1, 2], padding=[[1, 0], [4, 4]]), "3,5,2,2"),
    ([2, 100, 13, 16], [130, 100, 1, 1], dict(), "5,16,1,4"),
    # more groups than slabs, tiles that are ragged in rows and columns
    ([1, 32, 20, 36], [96, 32, 5, 5], dict(padding=[[2, 2], [2, 2]]), "3,28,4,2"),
    ([2, 96, 10, 12], [72, 96, 3, 3], dict(padding=[[0, 2], [2, 0]]), "7,12,2,4"),
    ([1, 257, 7, 7], [128, 257, 3, 3], dict(padding=[[1, 1], [1, 1]]), "4,7,1,8"),
])
def test_sizes(rx, client, monkeypatch, xs, ws, kw, tile):
    rng = np.random.default_rng(3)
    got, text, args = _run(rx, client, monkeypatch, xs, ws, kw, rng.normal(size=xs), rng.normal(size=ws), tile)
    assert contraction_err(got, oracle_run(text, args)[0].a, dot_bound(text, args)) <= TOL


@pytest.mark.gpu
@pytest.mark.parametrize("tile", ["4,28,4,1", "4,14,1,8"])
@pytest.mark.parametrize("where", ["image", "filter"])
def test_numbers_that_do_not_split(rx, client, monkeypatch, tile, where):
    xs, ws, kw = [2, 256, 28, 28], [96, 256, 3, 3], dict(padding=[[1, 1], [1, 1]])
    rng = np.random.default_rng(4)
    x, w = rng.normal(size=xs).astype(np.float32), rng.normal(size=ws).astype(np.float32)
    # infinities, NaN, and a finite number that rounds to an infinite bf16
    big, at = (x, (1, 7)) if where == "image" else (w, (50, 7))
    big[at + (1, 1)], big[at + (1, 2)], big[at + (2, 0)] = np.inf, np.nan, -3.4e38
    other = w if where == "image" else x
    other *= np.float32(2.0 ** -8)   # -3.4e38 times it stays finite
    got, text, args = _run(rx, client, monkeypatch, xs, ws, kw, x, w, tile)
    ref = np.asarray(oracle_run(text, args)[0].a)
    assert np.array_equal(np.isnan(got), np.isnan(ref)) and np.array_equal(np.isposinf(got), np.isposinf(ref)) and np.array_equal(np.isneginf(got), np.isneginf(ref))
    fin = np.isfinite(ref)
    assert contraction_err(got[fin], ref[fin], np.asarray(dot_bound(text, args))[fin]) <= TOL
    # below 2^-102 the third part loses bits: sums that consist of such numbers are as exact as others
    x, w = rng.normal(size=xs).astype(np.float32), rng.normal(size=ws).astype(np.float32)
    (x if where == "image" else w)[...] *= np.float32(2.0 ** -116)
    got, text, args = _run(rx, client, monkeypatch, xs, ws, kw, x, w, tile)
    assert contraction_err(got, oracle_run(text, args)[0].a, dot_bound(text, args)) <= TOL


def test_plans(monkeypatch):
    rx = load_pkg()
    kinds = lambda text: [l.split("kind=")[1].split()[0] for l in rx.compile_offline(text).splitlines() if "kind=" in l]   # noqa: E731
    conv = lambda b, c, o, hw: NN.convolution([b, c, hw, hw], [o, c, 3, 3], "f32", padding=[[1, 1], [1, 1]])[0]           # noqa: E731
    assert kinds(conv(8, 64, 128, 56)) == ["filter_split", "conv"]
    assert kinds(conv(4, 128, 128, 28))[-1].startswith("conv")
    # a module whose temporaries fit RxExecuteNoAlloc's 4 MiB keeps doing so: 512 x 512 x 9 x 6 bytes would not
    assert kinds(conv(8, 512, 512, 14)) == ["conv"]
    monkeypatch.setenv("RX_CONV_SPLIT", "2")
    assert kinds(conv(8, 512, 512, 14)) == ["filter_split", "conv"]
    monkeypatch.setenv("RX_CONV_SPLIT", "0")
    assert kinds(conv(8, 64, 128, 56)) == ["conv"]


@pytest.mark.parametrize("xs,ws,stride,alone", [([4, 64, 41, 36], [192, 64, 3, 3], 2, False), ([4, 64, 18, 44], [384, 64, 1, 1], 1, False), ([16, 32, 50, 27], [128, 32, 3, 3], 1, False),
                                                ([2, 64, 28, 26], [72, 64, 5, 5], 2, True), ([4, 64, 36, 27], [128, 64, 1, 1], 1, True)])
def test_a_convolution_alone_pays_for_the_splitting_launch(xs, ws, stride, alone):
    """Several convolutions share the launch that splits their filters: those stay on split operands."""
    rx = load_pkg()
    pad = ws[2] // 2
    text, _ = NN.convolution(xs, ws, "f32", strides=[stride, stride], padding=[[pad, pad], [pad, pad]])
    assert ("filter_split" in rx.compile_offline(text)) == alone
    # the same operation twice, on other operands
    op = next(l for l in text.splitlines() if "stablehlo.convolution" in l)
    name, rest = op.split("=", 1)
    head, tail = text[text.index("@main(") + 6:].split(")", 1)
    xt, wt = [a.split(":", 1)[1].strip() for a in head.split("%")[1:]]
    out = tail[tail.index("->") + 2:tail.index("{")].strip()
    two = rest.replace("%arg0", "%arg2").replace("%arg1", "%arg3")
    assert two != rest
    text = ("module {\n  func.func @main(%%arg0: %s, %%arg1: %s, %%arg2: %s, %%arg3: %s) -> (%s, %s) {\n%s\n    %%second =%s\n    return %s, %%second : %s, %s\n  }\n}\n"
            % (xt.rstrip(","), wt, xt.rstrip(","), wt, out, out, op, two, name.strip(), out, out))
    assert "filter_split" in rx.compile_offline(text)
