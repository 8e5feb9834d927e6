"""Launches that run as one (folded reduction ends, joined launches): the texts and the local memory of such plans, and their results."""
import os
import re
import subprocess

import numpy as np

import pytest

from _harness import gpu_run, oracle_run
from _loader import load_pkg
from oracle import stablehlo_interp as I

rx = load_pkg()
READELF = "/opt/rocm/llvm/bin/llvm-readelf"


def two_quantizations(shape0, shape1, dt):
    """x / max|x| and y / max|y| of two tensors in one module."""
    lines, outs = [], []
    t = ["tensor<%dx%dx%s>" % (s[0], s[1], dt) for s in (shape0, shape1)]
    s = "tensor<%s>" % dt
    for k in range(2):
        lines += ["    %%%s0 = stablehlo.abs %%arg%d : %s" % ("xy"[k], k, t[k]),
                  "    %%%s1 = stablehlo.reduce(%%%s0 init: %%z) applies stablehlo.maximum across dimensions = [0, 1] : (%s, %s) -> %s" % ("xy"[k], "xy"[k], t[k], s, s),
                  "    %%%s2 = stablehlo.broadcast_in_dim %%%s1, dims = [] : (%s) -> %s" % ("xy"[k], "xy"[k], s, t[k]),
                  "    %%%s3 = stablehlo.divide %%arg%d, %%%s2 : %s" % ("xy"[k], k, "xy"[k], t[k])]
    return ("module {\n  func.func @main(%%arg0: %s, %%arg1: %s) -> (%s, %s) {\n    %%z = stablehlo.constant dense<0.0> : %s\n%s\n    return %%x3, %%y3 : %s, %s\n  }\n}\n"
            % (t[0], t[1], t[0], t[1], s, "\n".join(lines), t[0], t[1]))


def functions(report):
    """name -> text of the functions of a plan's source that are no kernels"""
    return {m.group(1): m.group(0) for m in re.finditer(r"^static __device__ \S+ void (\w+)\(.*?^}", report, re.M | re.S)}


def kinds(report):
    return [l.split("kind=")[1].split()[0] for l in report.splitlines() if "kind=" in l]


SHAPES = [((512, 1024), (2048, 1024), "bf16"), ((2048, 1024), (512, 1024), "bf16"), ((64, 4096), (70, 4096), "f32"), ((300, 1000), (300, 1000), "f32")]


@pytest.mark.parametrize("a,b,dt", SHAPES)
def test_a_folded_map_in_a_joined_launch_takes_its_own_workgroup_number(a, b, dt):
    report = rx.compile_offline(two_quantizations(a, b, dt), True)
    assert kinds(report) == ["reduce", "map"], report[:2000]
    parts = functions(report)
    assert len(parts) >= 4
    for name, text in parts.items():
        assert "blockIdx" not in text and "gridDim" not in text, text


@pytest.mark.gpu
@pytest.mark.parametrize("a,b,dt", SHAPES)
def test_two_quantizations(rx, client, a, b, dt):
    text = two_quantizations(a, b, dt)
    rng = np.random.default_rng(a[0])
    args = [I.tensor(rng.normal(size=s) * 3, dt) for s in (a, b)]
    got, exe = gpu_run(rx, client, text, args)
    assert len(exe.launches()) == 2
    for g, r in zip(got, oracle_run(text, args)):
        g, r = np.asarray(g.a, dtype=np.float64), np.asarray(r.a, dtype=np.float64)
        assert np.all(np.abs(g - r) <= {"bf16": 2.0 ** -8, "f32": 2.0 ** -23}[dt] * np.abs(r))      # a division, rounded: at most one unit in the last place


@pytest.mark.parametrize("dt,n,tail,folded", [("f32", 512 * 2048, "f64", True), ("f32", 1024 * 4096, "f16", False), ("f64", 32 * 2048, "f32", False), ("f64", 64 * 2048, "f32", True), ("f32", 32 * 4096, "f64", False)])
def test_partials_are_counted_whatever_the_type_of_the_end(dt, n, tail, folded):
    """x - s and y - s for s = sin(tanh(exp(sqrt(max(x))))) in a type of another width than its reduction: folded from 64 to 512 partials"""
    t, u, s, r, w = "tensor<%dx%s>" % (n, dt), "tensor<%dx%s>" % (n, tail), "tensor<%s>" % dt, "tensor<%s>" % tail, "tensor<77x%s>" % tail
    report = rx.compile_offline(
        "module {\n  func.func @main(%%a: %s, %%b: %s) -> (%s, %s) {\n    %%z = stablehlo.constant dense<0.0> : %s\n"
        "    %%0 = stablehlo.reduce(%%a init: %%z) applies stablehlo.maximum across dimensions = [0] : (%s, %s) -> %s\n    %%1 = stablehlo.sqrt %%0 : %s\n"
        "    %%2 = stablehlo.exponential %%1 : %s\n    %%t = stablehlo.tanh %%2 : %s\n    %%3 = stablehlo.sine %%t : %s\n    %%4 = stablehlo.convert %%3 : (%s) -> %s\n"
        "    %%5 = stablehlo.broadcast_in_dim %%4, dims = [] : (%s) -> %s\n    %%6 = stablehlo.convert %%a : (%s) -> %s\n    %%7 = stablehlo.subtract %%6, %%5 : %s\n"
        "    %%8 = stablehlo.broadcast_in_dim %%4, dims = [] : (%s) -> %s\n    %%9 = stablehlo.subtract %%b, %%8 : %s\n    return %%7, %%9 : %s, %s\n  }\n}\n"
        % (t, w, u, w, s, t, s, s, s, s, s, s, s, r, r, u, t, u, u, r, w, w, u, w))
    assert kinds(report)[:2] == (["reduce", "map"] if folded else ["reduce", "reduce_final"]), report[:2000]


def sums_beside(shapes, dt, product=None):
    """Column sums and a full sum of independent tensors, and a matrix product of others, in one module."""
    T = lambda *d: "tensor<%s%s>" % ("".join("%dx" % v for v in d), dt)   # noqa: E731
    lines, types, outs = ["    %%z = stablehlo.constant dense<0.0> : %s" % T()], [], []
    if product:
        m, n, k = product
        types += [T(m, k), T(k, n)]
        lines.append("    %%p = stablehlo.dot_general %%arg0, %%arg1, contracting_dims = [1] x [0] : (%s, %s) -> %s" % (T(m, k), T(k, n), T(m, n)))
        outs.append(("%p", T(m, n)))
    for r, c in shapes:
        i = len(types)
        types.append(T(r, c))
        for dims, out in (("0", T(c)), ("0, 1", T())):
            lines.append("    %%r%d_%d = stablehlo.reduce(%%arg%d init: %%z) applies stablehlo.add across dimensions = [%s] : (%s, %s) -> %s" % (i, len(dims), i, dims, T(r, c), T(), out))
            outs.append(("%%r%d_%d" % (i, len(dims)), out))
    rt = ", ".join(t for _, t in outs)
    return ("module {\n  func.func @main(%s) -> (%s) {\n%s\n    return %s : %s\n  }\n}\n"
            % (", ".join("%%arg%d: %s" % kv for kv in enumerate(types)), rt, "\n".join(lines), ", ".join(o for o, _ in outs), rt))


# a product whose tile takes all of the LDS; more differing sums than the LDS has room for one after the other; reductions of one
# workgroup of 1024 threads beside others
BESIDE = [(((512, 1024), (1024, 1000), (768, 1024)), "bf16", (2304, 2048, 2048)), (((64, 520), (65, 1000)), "f32", (512, 512, 256)),
          (tuple((512, 528 + 16 * i) for i in range(24)), "bf16", None), (((8, 1000), (100, 1032), (1000, 1024), (7, 33)), "f32", None)]


@pytest.mark.skipif(not os.path.exists(READELF), reason="no llvm-readelf")
@pytest.mark.parametrize("shapes,dt,product", BESIDE)
def test_joined_kernels_fit_the_local_memory(tmp_path, monkeypatch, shapes, dt, product):
    monkeypatch.setenv("RX_DUMP_CODE_OBJECT", str(tmp_path / "code"))
    report = rx.compile_offline(sums_beside(shapes, dt, product))
    notes = subprocess.run([READELF, "--notes", str(tmp_path / "code")], check=True, capture_output=True, text=True).stdout
    static = {m.group(2): int(m.group(1)) for m in re.finditer(r"\.group_segment_fixed_size: (\d+).*?\.symbol: +(\w+)\.kd", notes, re.S)}
    joined = [l.split() for l in report.splitlines() if "kind=" in l and "_joined" in l]
    assert joined
    for l in joined:
        lds = int(next(w for w in l if w.startswith("lds="))[4:])
        assert lds + static[l[1]] <= 160 * 1024 and (static[l[1]] == 0 if "gemm" in l[2] else lds == 0), l


@pytest.mark.gpu
@pytest.mark.parametrize("shapes,dt,product", BESIDE)
def test_sums_beside_a_product(rx, client, shapes, dt, product):
    text = sums_beside(shapes, dt, product)
    rng = np.random.default_rng(len(shapes))
    dims = ([(product[0], product[2]), (product[2], product[1])] if product else []) + list(shapes)
    x = [rng.integers(-1, 2, size=d).astype(np.float64) for d in dims]      # whole numbers: sums and products are exact in every accumulator
    got, exe = gpu_run(rx, client, text, [I.tensor(v, dt) for v in x])
    assert any("_joined" in l["kernel"] for l in exe.launches())
    want = ([x[0] @ x[1]] if product else []) + [s for v in x[2 if product else 0:] for s in (v.sum(axis=0), v.sum())]
    for g, w in zip(got, want):
        assert np.array_equal(np.asarray(g.a), np.asarray(I.tensor(w, dt).a))


def many_sums(n):
    """Sums of n short vectors of differing lengths."""
    args = ["%%a%d: tensor<%dxf32>" % (i, 3 + i) for i in range(n)]
    lines = ["    %%r%d = stablehlo.reduce(%%a%d init: %%z) applies stablehlo.add across dimensions = [0] : (tensor<%dxf32>, tensor<f32>) -> tensor<f32>" % (i, i, 3 + i) for i in range(n)]
    rt = ", ".join(["tensor<f32>"] * n)
    return ("module {\n  func.func @main(%s) -> (%s) {\n    %%z = stablehlo.constant dense<0.0> : tensor<f32>\n%s\n    return %s : %s\n  }\n}\n"
            % (", ".join(args), rt, "\n".join(lines), ", ".join("%%r%d" % i for i in range(n)), rt))


def test_a_joined_kernel_has_a_bounded_number_of_parts():
    report = rx.compile_offline(many_sums(130), True)
    assert kinds(report) == ["reduce"] * 3, report[:2000]
    for m in re.finditer(r"void \w+_joined\((.*?)\) \{\n", report):
        assert m.group(1).count(", ") < 256


@pytest.mark.gpu
def test_many_sums(rx, client):
    args = [I.tensor(np.arange(3 + i, dtype=np.float64) - i, "f32") for i in range(130)]      # exact
    got, _ = gpu_run(rx, client, many_sums(130), args)
    assert [float(np.asarray(g.a)) for g in got] == [float(np.asarray(a.a, dtype=np.float64).sum()) for a in args]
