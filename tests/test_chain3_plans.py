"""Which runs of 3-D steps are chain kernels: rows of odd length, over which maps are faster, from the sizes at which these win."""
import pytest

from _loader import load_pkg, load_programs

rx = load_pkg()
P = load_programs()


@pytest.mark.parametrize("nx,ny,nz,steps,dt,chained", [(105, 68, 54, 16, "f32", False), (87, 109, 59, 4, "f32", False), (65, 82, 39, 5, "f64", False), (93, 46, 63, 16, "f32", True),
                                                       (80, 77, 43, 10, "f32", True), (64, 82, 39, 5, "f64", True), (61, 47, 33, 10, "f64", True), (35, 25, 69, 4, "f64", True)])
def test_chains_or_maps(nx, ny, nz, steps, dt, chained):
    kinds = [l.split("kind=")[1].split()[0] for l in rx.compile_offline(P.stencil(nx, ny, nz, steps=steps, elt=dt)).splitlines() if "kind=" in l]
    assert ("map_chain" in kinds) == chained, kinds
