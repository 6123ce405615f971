"""Restoring and reading back records at the sizes where the two ways across the bus meet (9,830 records
are the last that the kernels carry themselves) and at remainders of a workgroup's 256 records; and
what the device's scan of the records decides: a force component other than +0 makes the next step start
from the records' forces, and masses unlike the first take the mesh off the tiled kernel and back."""
import numpy as np
import pytest

import feriphys_amd as fa
from feriphys_amd import workloads as wl
from gpu_common import announce

pytestmark = pytest.mark.gpu


def cloth(rows, cols):
    sim = wl.build_gpu(wl.config0(rows=rows, cols=cols, pins="edge"))
    return sim, sim.get_points(0)


@pytest.mark.parametrize("rows,cols", [(2, 2), (3, 85), (16, 16), (2, 257), (10, 983), (983, 10), (7, 1405), (64, 200)])
def test_records_round_trip(rows, cols):
    announce(f"records {rows}x{cols}")
    sim, rec = cloth(rows, cols)
    rng = np.random.default_rng(rows * cols)
    rec[:, 1:] = rng.normal(size=(rec.shape[0], 9)).astype(np.float32)
    sim.set_points(0, rec)
    assert np.array_equal(sim.get_points(0), rec)
    assert np.array_equal(sim.get_vertices(0)[0], rec[:, 1:4])


@pytest.mark.parametrize("n", [16, 120])
def test_forces_and_masses_are_noticed(n):
    """The last record alone carries the force or the other mass, so only a scan of all of them finds it."""
    announce(f"record scan {n}x{n}")
    sim, rec = cloth(n, n)
    sim.step(1)
    plain = sim.get_points(0)
    with_force = rec.copy()
    with_force[0, 9] = 0.5  # an unpinned vertex of the first row
    sim.set_points(0, with_force)
    sim.step(1)
    assert not np.array_equal(sim.get_points(0)[0], plain[0])
    assert np.array_equal(sim.get_points(0)[2 * n + 3:], plain[2 * n + 3:])
    assert sim.get_mesh_kernel(0) == fa.FP_STEP_TILED
    heavy = rec.copy()
    heavy[n * n - 1, 0] *= 2.0
    sim.set_points(0, heavy)
    assert sim.get_mesh_kernel(0) != fa.FP_STEP_TILED
    sim.set_points(0, rec)
    assert sim.get_mesh_kernel(0) == fa.FP_STEP_TILED
    sim.step(1)
    assert np.array_equal(sim.get_points(0), plain)
