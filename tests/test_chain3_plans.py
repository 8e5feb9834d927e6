"""Which runs of 3-D steps are chain kernels: rows of odd length, over which maps are faster, from the sizes at which these win."""
import ctypes

import numpy as np
import pytest

from _loader import load_pkg, load_programs

rx = load_pkg()
P = load_programs()


@pytest.mark.parametrize("nx,ny,nz,steps,dt,chained", [(105, 68, 54, 16, "f32", False), (87, 109, 59, 4, "f32", False), (65, 82, 39, 5, "f64", False), (93, 46, 63, 16, "f32", True),
                                                       (80, 77, 43, 10, "f32", True), (64, 82, 39, 5, "f64", True), (61, 47, 33, 10, "f64", True), (35, 25, 69, 4, "f64", True)])
def test_chains_or_maps(nx, ny, nz, steps, dt, chained):
    kinds = [l.split("kind=")[1].split()[0] for l in rx.compile_offline(P.stencil(nx, ny, nz, steps=steps, elt=dt)).splitlines() if "kind=" in l]
    assert ("map_chain" in kinds) == chained, kinds


@pytest.mark.gpu
@pytest.mark.parametrize("nx,ny,nz,steps,dt", [(65, 82, 39, 5, "f64"), (87, 109, 59, 4, "f32")])
def test_steps_that_run_as_maps_run_without_allocations(rx, client, nx, ny, nz, steps, dt):
    """The maps' fields exceed the 4 MiB of RxExecuteNoAlloc, those of a chain do not: the same results either way."""
    text, full = P.stencil(nx, ny, nz, steps=steps, elt=dt), (nz + 6, ny + 6, nx + 6)
    exe = rx.xla_compile(client, text)
    assert all(l["kind"] != "map_chain" for l in exe.launches())
    rng = np.random.default_rng(nx)
    c = np.zeros(full)
    c[3:-3, 3:-3, 3:-3] = rng.uniform(size=(nz, ny, nx))
    bufs = [rx.Buffer.from_host(client, a.astype(rx._STORAGE[dt]), dt) for a in [c] + [rng.uniform(-1, 1, size=full) for _ in range(3)]]
    ref = exe.execute_sharded(bufs)[0].synced_buffer()
    out = rx.Buffer.uninitialized(client, ref.shape(), dt)
    before = client.default_device().allocator_stats()["num_allocs"]
    rx.lib.RxClearError()
    assert rx.lib.RxExecuteNoAlloc(exe.handle, 4, (ctypes.c_void_p * 4)(*[b.handle for b in bufs]), 1, (ctypes.c_void_p * 1)(out.handle)) == 0, rx.lib.RxLastError()
    client.default_device().synchronize()
    assert client.default_device().allocator_stats()["num_allocs"] == before
    assert np.array_equal(out.to_host(), ref.to_host())
