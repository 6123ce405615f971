"""The rules that choose a cloth's launch form, on both sides of each line, bit for bit against the
one-thread-per-vertex grid kernel: 8x8 tiles with twelve waves up to 768 of them, a lane per vertex
beyond; and a batch whose meshes would have different tile shapes, which shares one while its tiles are
all resident."""
import numpy as np
import pytest

import feriphys_amd as fa
from feriphys_amd import workloads as wl
from gpu_common import announce, bits

pytestmark = pytest.mark.gpu


def scene(sizes, obstacle, seed=5):
    cloths = [wl.cloth_spec(r, c, pins=range((r - 1) * c, r * c)) for r, c in sizes]
    cfg = wl.config0().config
    obs = [wl.sphere_obstacle(0.6, (0.0, -0.603, 0.0), 2)] if obstacle else []
    return wl.Scene(cloths, cfg, obs, 1e-3, seed, 1, "rules")


def run(sc, kernel, integration, math, steps):
    sim = wl.build_gpu(sc)
    cfg = sim.config
    cfg.integration = fa.Integration(integration)
    sim.config = cfg
    sim.set_kernel(kernel, math)
    forces = []
    for k in range(len(sc.cloths)):  # forces and step both from the initial records
        rec = sim.get_points(k)
        sim.accumulate_forces(k)
        forces.append(sim.get_points(k)[:, 7:10])
        sim.set_points(k, rec)
    sim.step(steps)
    return [sim.get_points(k) for k in range(len(sc.cloths))], forces


@pytest.mark.parametrize("integration", [0, 1])
@pytest.mark.parametrize("rows,cols", [(8, 8), (9, 17), (100, 33), (192, 256), (192, 257), (250, 251)])
def test_exact_forms_equal_the_simple_kernel(rows, cols, integration):
    announce(f"launch rule {rows}x{cols}, integration {integration}")
    sc = scene([(rows, cols)], obstacle=True)
    a, fa_ = run(sc, fa.FP_KERNEL_GRID, integration, fa.FP_MATH_EXACT, 12)
    b, fb = run(sc, fa.FP_KERNEL_GRID_SIMPLE, integration, fa.FP_MATH_EXACT, 12)
    assert (bits(a[0]) == bits(b[0])).all() and (bits(fa_[0]) == bits(fb[0])).all()


@pytest.mark.parametrize("sizes", [[(12, 200), (40, 60)], [(12, 200), (10, 120), (130, 300), (60, 61)],
                                   [(13, 40), (300, 400), (400, 420), (9, 256)]])
def test_mixed_shapes_in_one_launch(sizes):
    """Exact: the same bits.  Fast: within 1e-5 of the exact step's forces and states, relative, as for
    any tile shape."""
    announce(f"mixed tile shapes {sizes}")
    sc = scene(sizes, obstacle=False)
    a, fx = run(sc, fa.FP_KERNEL_GRID, 1, fa.FP_MATH_EXACT, 1)
    b, fs = run(sc, fa.FP_KERNEL_GRID_SIMPLE, 1, fa.FP_MATH_EXACT, 1)
    c, ff = run(sc, fa.FP_KERNEL_GRID, 1, fa.FP_MATH_FAST, 1)
    for k in range(len(sizes)):
        assert (bits(a[k]) == bits(b[k])).all() and (bits(fx[k]) == bits(fs[k])).all()
        assert np.abs(c[k][:, 1:4] - a[k][:, 1:4]).max() <= 1e-5 * np.abs(a[k][:, 1:4]).max()
        assert np.abs(c[k][:, 4:7] - a[k][:, 4:7]).max() <= 1e-5 * np.abs(a[k][:, 4:7]).max()
        assert np.abs(ff[k] - fx[k]).max() <= 1e-5 * np.abs(fx[k]).max()
