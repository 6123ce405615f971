"""The exact small-tile kernel's task split (feriphys_amd/csrc/grid_tile_core.hpp) run on the CPU against
the oracle, bit for bit: forces and one step, tiles inside the grid and at its border, grids smaller than a tile and not filling their last tiles, both integrators, corner and edge
pins, non-zero starting forces (tests/native/tile_emul.cpp: every staged index checked, the LDS filled
with NaN).  Integers equal or not: there is no tolerance."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

import pyoracle as orc
from feriphys_amd import workloads as wl
from test_fast_kernel_emulation import moving, oracle_cfg, run_emul

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
F32 = np.float32


@pytest.fixture(scope="module")
def emul(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("emul") / "tile_emul.so")
    subprocess.run(["/opt/rocm/bin/hipcc", "-x", "hip", "--cuda-host-only", "--offload-arch=gfx950", "-std=c++17",
                    "-O2", "-fPIC", "-shared", "-ffp-contract=off", "-fno-fast-math",
                    os.path.join(ROOT, "tests", "native", "tile_emul.cpp"), "-o", so], check=True)
    lib = C.CDLL(so)
    fp = C.POINTER(C.c_float)
    lib.emul_fast.argtypes = [C.c_uint32, C.c_uint32, C.c_float, fp, fp, fp, fp, fp, C.c_int32,
                              C.POINTER(C.c_uint32), C.c_int32, fp, C.c_int32, C.c_int32]
    lib.emul_fast.restype = C.c_int
    return lib


def bits(a):
    return np.ascontiguousarray(a, F32).view(np.uint32)


@pytest.mark.parametrize("rows,cols,pins,steps", [(2, 2, "edge", 3), (5, 3, "edge", 5), (8, 8, "edge", 5),
                                                  (17, 33, "corners", 5), (50, 70, "edge", 5), (9, 65, "corners", 5)])
def test_forces_and_step_equal_the_oracle(emul, rows, cols, pins, steps):
    for integration in (0, 1):
        sc = wl.config0(rows=rows, cols=cols, pins=pins)
        sc.config.integration = integration
        rec = moving(sc, steps)
        o = orc.build_scene(sc)
        o.mesh(0).set_points(rec)
        o.mesh(0).accumulate_forces(oracle_cfg(sc))
        assert (bits(run_emul(emul, sc, rec, 1, 0)[:, 7:10]) == bits(o.mesh(0).points()[:, 7:10])).all()
        rec[:, 7:10] = np.random.default_rng(3).normal(scale=0.01, size=(rec.shape[0], 3)).astype(F32)
        for force_init in (False, True):
            r = rec.copy()
            if not force_init:
                r[:, 7:10] = 0.0
            o = orc.build_scene(sc)
            o.mesh(0).set_points(r)
            o.step(1)
            got = run_emul(emul, sc, r, 0, 0, force_init=force_init)
            assert (bits(got[:, 1:7]) == bits(o.mesh(0).points()[:, 1:7])).all()
