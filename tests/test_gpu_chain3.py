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
