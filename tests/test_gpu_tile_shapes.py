"""Tile shapes set by the caller: the shape that was set is the one that runs, and every exact form (15x15,
7x31 and 16x16 tiles with a lane per vertex) gives the bits of the one-thread-per-vertex grid kernel at sizes
around and between the tiles' edges."""
import numpy as np
import pytest

import feriphys_amd as fa
from feriphys_amd import workloads as wl
from gpu_common import announce, bits

pytestmark = pytest.mark.gpu
SHAPES = [fa.FP_TILE_15x15, fa.FP_TILE_7x31, fa.FP_TILE_16x16]


def scene(sizes, obstacle, pins="edge"):
    cloths = [wl.cloth_spec(r, c, pins=range((r - 1) * c, r * c) if pins == "edge" else [0, c - 1]) for r, c in sizes]
    obs = [wl.sphere_obstacle(0.6, (0.0, -0.603, 0.0), 2)] if obstacle else []
    return wl.Scene(cloths, wl.config0().config, obs, 1e-3, 7, 1, "shapes")


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("integration", [0, 1])
@pytest.mark.parametrize("rows,cols", [(2, 2), (7, 31), (15, 15), (16, 16), (17, 33), (31, 62), (61, 64), (250, 251)])
def test_exact_forms_equal_the_simple_kernel(shape, rows, cols, integration):
    announce(f"tile shape {shape}, {rows}x{cols}, integration {integration}")
    sc = scene([(rows, cols)], obstacle=True)
    out = []
    for kernel in (fa.FP_KERNEL_GRID, fa.FP_KERNEL_GRID_SIMPLE):
        sim = wl.build_gpu(sc)
        cfg = sim.config
        cfg.integration = fa.Integration(integration)
        sim.config = cfg
        sim.set_kernel(kernel, fa.FP_MATH_EXACT)
        sim.set_tile_shape(0, shape)
        rec = sim.get_points(0)
        sim.accumulate_forces(0)
        forces = sim.get_points(0)[:, 7:10]
        # a step from records with forces, then steps from clear ones
        rec[:, 7:10] = np.random.default_rng(3).normal(scale=0.01, size=forces.shape).astype(np.float32)
        sim.set_points(0, rec)
        sim.step(1)
        first = sim.get_points(0)
        sim.step(11)
        out.append((forces, first, sim.get_points(0)))
    for a, b in zip(*out):
        assert np.isfinite(b).all() and (bits(a) == bits(b)).all()


def test_shapes_side_by_side_and_switched():
    """Cloths of the three shapes and of the default in one step, switched between steps: the simple
    kernel's bits throughout."""
    sizes = [(33, 34), (29, 65), (48, 17), (40, 41)]
    sc = scene(sizes, obstacle=False, pins="corners")
    sim, ref = wl.build_gpu(sc), wl.build_gpu(sc)
    ref.set_kernel(fa.FP_KERNEL_GRID_SIMPLE, fa.FP_MATH_EXACT)
    announce("three set shapes and the default in one step")
    for turn in range(3):
        for k in range(3):
            sim.set_tile_shape(k, SHAPES[(k + turn) % 3])
            assert sim.get_tile_shape(k) == SHAPES[(k + turn) % 3]
        sim.step(10)
        sim.step_graph(10, 5)
        ref.step(20)
        for k in range(len(sizes)):
            assert (bits(sim.get_points(k)) == bits(ref.get_points(k))).all()


@pytest.mark.parametrize("shape", [fa.FP_TILE_15x15, fa.FP_TILE_7x31])
def test_a_set_shape_runs_whatever_the_other_meshes(shape):
    """The last bits of fast forces depend on the tile shape.  A cloth with a set shape has the same bits
    alone and beside cloths whose tiles outnumber its own, and the two shapes' bits differ."""
    def forces(sizes, which):
        sim = wl.build_gpu(scene(sizes, obstacle=False))
        sim.set_kernel(fa.FP_KERNEL_GRID, fa.FP_MATH_FAST)
        sim.set_tile_shape(0, which)
        sim.accumulate_forces(0)
        return sim.get_points(0)[:, 7:10]

    announce(f"fast, set shape {shape}, alone and in company")
    other = fa.FP_TILE_7x31 if shape == fa.FP_TILE_15x15 else fa.FP_TILE_15x15
    alone = forces([(40, 90)], shape)
    for company in ([(12, 600)], [(200, 200)], [(12, 600), (14, 900)]):
        assert (bits(forces([(40, 90)] + company, shape)) == bits(alone)).all()
    assert (bits(forces([(40, 90)], other)) != bits(alone)).any()


@pytest.mark.parametrize("math", [fa.FP_MATH_EXACT, fa.FP_MATH_FAST])
def test_autotune_reports_shapes_that_can_be_set(math):
    sc = scene([(12, 14), (20, 30), (48, 40), (70, 30)], obstacle=False)
    sim = wl.build_gpu(sc)
    sim.set_kernel(fa.FP_KERNEL_GRID, math)
    chosen = sim.autotune(3)
    announce(f"autotune, math {math}: {chosen}")
    for k, shape in enumerate(chosen):
        assert shape in SHAPES and sim.get_tile_shape(k) == shape


def test_fast_shapes_side_by_side_equal_each_alone():
    """Fast steps of cloths with set shapes, a launch per shape, and of default ones beside them (more tiles
    than are resident, so that they keep their own): each cloth's records are the bits of the cloth alone
    with the shape it runs in."""
    sizes = [(33, 34), (29, 65), (48, 17), (12, 200), (620, 640)]
    shapes = [fa.FP_TILE_15x15, fa.FP_TILE_7x31, fa.FP_TILE_16x16, None, None]
    alone = [fa.FP_TILE_15x15, fa.FP_TILE_7x31, fa.FP_TILE_15x15, fa.FP_TILE_7x31, fa.FP_TILE_15x15]
    sim = wl.build_gpu(scene(sizes, obstacle=True))
    sim.set_kernel(fa.FP_KERNEL_GRID, fa.FP_MATH_FAST)
    for k, shape in enumerate(shapes):
        if shape is not None:
            sim.set_tile_shape(k, shape)
    start = [sim.get_points(k) for k in range(len(sizes))]
    announce("fast, three launches a step")
    sim.step(7)
    sim.step_graph(10, 5)
    for k, size in enumerate(sizes):
        one = wl.build_gpu(scene([size], obstacle=True))
        one.set_kernel(fa.FP_KERNEL_GRID, fa.FP_MATH_FAST)
        one.set_tile_shape(0, alone[k])
        one.set_points(0, start[k])
        one.step(17)
        a, b = sim.get_points(k), one.get_points(0)
        assert np.isfinite(b).all() and (bits(a) == bits(b)).all(), size
