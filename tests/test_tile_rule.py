"""The host's rule for the launch shapes of cloths (feriphys_amd/csrc/tile_rule.hpp): a shape that was set
is the one that runs, whatever else the simulation holds; the default gives way to 8x8 tiles in small exact
simulations and to one shape for all while the tiles are resident at once."""
import ctypes as C
import itertools
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
S15, S7, S16, S8 = 0, 1, 2, 3
DEFAULT = None


@pytest.fixture(scope="module")
def rule(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("rule") / "tile_rule.so")
    subprocess.run(["/opt/rocm/bin/hipcc", "-x", "hip", "--cuda-host-only", "--offload-arch=gfx950", "-std=c++17",
                    "-O1", "-fPIC", "-shared", os.path.join(ROOT, "tests", "native", "tile_rule_check.cpp"), "-o", so],
                   check=True)
    f = C.CDLL(so).rule
    f.restype = None

    def launch(cloths, fast):
        """cloths: (rows, cols, set shape or DEFAULT)"""
        n = len(cloths)
        shape = [s if s is not DEFAULT else (S7 if r < 15 and c >= 31 else S16) for r, c, s in cloths]
        out = (C.c_int32 * n)()
        f(n, (C.c_uint32 * n)(*(c[0] for c in cloths)), (C.c_uint32 * n)(*(c[1] for c in cloths)),
          (C.c_int32 * n)(*shape), (C.c_int32 * n)(*(c[2] is not DEFAULT for c in cloths)), int(fast), out)
        return list(out)

    return launch


def own(shape, fast):
    return S15 if fast and shape == S16 else shape


@pytest.mark.parametrize("fast", [False, True])
@pytest.mark.parametrize("others", [[], [(40, 40)], [(12, 200), (300, 300)], [(1024, 1024)]])
def test_a_set_shape_is_the_one_that_runs(rule, fast, others):
    for shape, (r, c) in itertools.product((S15, S7, S16), ((5, 5), (32, 32), (13, 400), (200, 200), (700, 900))):
        cloths = [(a, b, DEFAULT) for a, b in others] + [(r, c, shape)]
        assert rule(cloths, fast)[-1] == own(shape, fast)
        # three set shapes side by side stay three
        assert rule([(r, c, s) for s in (S15, S7, S16)], fast) == [own(s, fast) for s in (S15, S7, S16)]


def test_defaults_on_both_sides_of_the_lines(rule):
    assert rule([(192, 256, DEFAULT)], False) == [S8]        # 768 tiles of 8x8
    assert rule([(192, 257, DEFAULT)], False) == [S16]       # 792
    assert rule([(192, 256, DEFAULT)], True) == [S15]
    assert rule([(96, 256, DEFAULT), (12, 256, S7), (80, 256, DEFAULT)], False) == [S8, S7, S8]
    # all tiles resident: the commonest shape, 16x16 (15x15 in the fast form) for 1,200 of 1,300 tiles
    assert rule([(480, 640, DEFAULT), (7, 1600, DEFAULT)], False) == [S16, S16]
    assert rule([(480, 640, DEFAULT), (7, 1600, DEFAULT)], True) == [S15, S15]
    assert rule([(480, 640, DEFAULT), (7, 1600, S7)], True) == [S15, S7]
    # more than are resident: each its own
    assert rule([(1024, 1024, DEFAULT), (7, 1600, DEFAULT)], False) == [S16, S7]
    assert rule([(1024, 1024, DEFAULT), (7, 1600, DEFAULT)], True) == [S15, S7]
