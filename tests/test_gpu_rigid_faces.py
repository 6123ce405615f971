"""Rigid cubes over one to nine obstacle faces, against the CPU oracle bit for bit: the sides of the
corners are found two faces at a time (odd counts take the last one twice) and carried from step to
step, also over hits and over launches; nine faces take the grids, whose old corners are carried too."""
import numpy as np
import pytest

from gpu_common import announce, bits
from test_gpu_rigid_steps import both

pytestmark = pytest.mark.gpu


def faces(count):
    """`count` large triangles crossing under the cubes at different tilts, one obstacle each."""
    out = []
    for k in range(count):
        c, s = np.cos(0.7 * k), np.sin(0.7 * k)
        v = np.array([[-60, 0, 60], [60, 0, 60], [0, 0, -90]], np.float64)
        v = np.stack([c * v[:, 0] + s * v[:, 2], 0.01 * k * v[:, 0] - 0.2 * k, c * v[:, 2] - s * v[:, 0]], 1)
        out.append((v.astype(np.float32), np.array([0, 1, 2], np.uint64)))
    return out


@pytest.mark.parametrize("count", [1, 2, 3, 5, 8, 9])
@pytest.mark.parametrize("integration", [0, 1])
def test_face_counts_bit_exact(count, integration):
    g, o = both(130, integration, faces(count), 40 + count)
    for steps in (1, 64, 200, 130):
        announce(f"rigid 130 bodies, {count} faces, {steps} more steps")
        g.step(steps)
        o.step(steps)
        a, b = g.states(), o.states()
        assert np.isfinite(a).all()
        assert (bits(a) == bits(b)).all()
