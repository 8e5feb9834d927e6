"""Launches that run as one (folded reduction ends, joined launches): the plans' texts and resources, without a GPU."""
import re

import numpy as np

import pytest

from _harness import gpu_run, oracle_run
from _loader import load_pkg
from oracle import stablehlo_interp as I

rx = load_pkg()


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
