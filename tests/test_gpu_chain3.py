"""Runs of advection-diffusion steps on small 3-D arrays in chain kernels whose tile and length the planner chooses, the velocities
in registers: bit for bit what a map per step gives, on arrays smaller than a tile, cut by every edge, and around the sizes
at which the choice becomes maps."""
import numpy as np
import pytest

from _harness import gpu_run
from _loader import load_programs
from oracle import stablehlo_interp as I

pytestmark = pytest.mark.gpu
P = load_programs()


@pytest.mark.parametrize("dt", ["f64", "f32"])
@pytest.mark.parametrize("nx,ny,nz,steps", [(1, 1, 1, 4), (3, 2, 5, 5), (24, 24, 16, 9), (30, 17, 19, 6), (61, 47, 33, 10), (25, 120, 40, 7), (130, 7, 9, 4), (7, 9, 130, 11)])
def test_chosen_chains_equal_maps(rx, client, monkeypatch, nx, ny, nz, steps, dt):
    text = P.stencil(nx, ny, nz, steps=steps, elt=dt)
    rng = np.random.default_rng(nx)
    full = (nz + 6, ny + 6, nx + 6)
    c = np.zeros(full)
    c[3:-3, 3:-3, 3:-3] = rng.uniform(size=(nz, ny, nx))
    args = [I.tensor(c, dt)] + [I.tensor(rng.uniform(-1, 1, size=full), dt) for _ in range(3)]
    got, exe = gpu_run(rx, client, text, args)
    assert any(l["kind"] == "map_chain" for l in exe.launches()), exe.report()
    monkeypatch.setenv("RX_CHAIN_STEPS", "1")
    ref, plain = gpu_run(rx, client, text, args)
    assert all(l["kind"] != "map_chain" for l in plain.launches())
    assert np.array_equal(got[0].a, ref[0].a)


@pytest.mark.parametrize("nx,ny,nz,steps", [(255, 72, 99, 5), (90, 250, 100, 6), (24, 455, 205, 4)])
def test_chosen_chains_of_several_rounds_equal_maps(rx, client, monkeypatch, nx, ny, nz, steps):
    """More tiles than compute units, boxes of more than eight cells a thread."""
    test_chosen_chains_equal_maps(rx, client, monkeypatch, nx, ny, nz, steps, "f64")


def _two_fields(D, steps, dt):
    """Two arrays that step in turns, each around its own points and those of the other, scaled by a third."""
    tf, n = "tensor<%s%s>" % ("".join("%dx" % d for d in D), dt), [d - 2 for d in D]
    ti = "tensor<%s%s>" % ("".join("%dx" % d for d in n), dt)
    lines, cnt = [], [0]

    def new(s):
        cnt[0] += 1
        lines.append("    %%%d = %s" % (cnt[0], s))
        return "%%%d" % cnt[0]

    def sh(x, *off):
        return new("stablehlo.slice %s [%s] : (%s) -> %s" % (x, ", ".join("%d:%d" % (1 + o, 1 + o + m) for o, m in zip(off, n)), tf, ti))
    zero, eighth = new("stablehlo.constant dense<0.0> : tensor<%s>" % dt), new("stablehlo.constant dense<0.125> : %s" % ti)
    scale = sh("%arg2", 0, 0, 0)
    f = ["%arg0", "%arg1"]
    for i in range(2 * steps):
        a, b = f[i % 2], f[1 - i % 2]
        s = sh(a, -1, 0, 0)
        for x, off in ((a, (1, 0, 0)), (a, (0, -1, 0)), (a, (0, 1, 0)), (a, (0, 0, -1)), (b, (0, 0, 1))):
            s = new("stablehlo.add %s, %s : %s" % (s, sh(x, *off), ti))
        s = new("stablehlo.multiply %s, %s : %s" % (new("stablehlo.multiply %s, %s : %s" % (s, eighth, ti)), scale, ti))
        s = new("stablehlo.add %s, %s : %s" % (s, sh(a, 0, 0, 0), ti))
        f[i % 2] = new("stablehlo.pad %s, %s, low = [1, 1, 1], high = [1, 1, 1], interior = [0, 0, 0] : (%s, tensor<%s>) -> %s" % (s, zero, ti, dt, tf))
    return ("module {\n  func.func @main(%%arg0: %s, %%arg1: %s, %%arg2: %s) -> (%s, %s) {\n%s\n    return %s, %s : %s, %s\n  }\n}\n"
            % (tf, tf, tf, tf, tf, "\n".join(lines), f[0], f[1], tf, tf))


@pytest.mark.parametrize("dt", ["f64", "f32"])
@pytest.mark.parametrize("D,steps", [((20, 18, 22), 3), ((39, 53, 67), 5), ((64, 64, 64), 4)])
def test_steps_of_two_arrays_fit_the_local_memory(rx, client, monkeypatch, D, steps, dt):
    """The choice counts the tiles of one array; a chain over two, with twice as many, was refused by the device."""
    text = _two_fields(D, steps, dt)
    rng = np.random.default_rng(3)
    args = [I.tensor(rng.uniform(size=D), dt) for _ in range(3)]
    got, _ = gpu_run(rx, client, text, args)
    monkeypatch.setenv("RX_CHAIN_STEPS", "1")
    ref, plain = gpu_run(rx, client, text, args)
    assert all(l["kind"] != "map_chain" for l in plain.launches())
    assert np.array_equal(got[0].a, ref[0].a) and np.array_equal(got[1].a, ref[1].a)
