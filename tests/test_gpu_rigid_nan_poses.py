"""Rigid cubes whose rotation leaves the numbers: thrown so hard by a low floor's impulses, or spun so fast,
that the quaternion's length overflows and the pose becomes NaN.  On which side of a plane a corner of such a
pose stands, and so whether the position and the momenta become NaN too, is the sign that a NaN keeps through
(r0 c0 + r1 c1) + r2 c2 and + x.  Against the CPU oracle bit for bit, a NaN for a NaN."""
import numpy as np
import pytest

import feriphys_amd as fa
import pyoracle as orc
from feriphys_amd import workloads as wl
from gpu_common import announce

pytestmark = pytest.mark.gpu
F32 = np.float32
# The sign of a NaN that an operation makes (or subtracts) is the machine's, and one for all of a pose's
# numbers on the CPU only: the bodies here whose poses hold NaNs of both signs on the GPU, which no way of
# forming the corners mends.
BOTH_SIGNS = {(1, "spun", 1): [60], (1, "thrown", 0): [74, 156], (1, "thrown", 1): [221]}


def same(a, b):
    return (a.view(np.uint32) == b.view(np.uint32)) | (np.isnan(a) & np.isnan(b))


@pytest.mark.parametrize("integration", [0, 1])
@pytest.mark.parametrize("case", ["thrown", "spun"])
@pytest.mark.parametrize("walls", [0, 1])
def test_a_pose_that_becomes_nan(integration, case, walls):
    rng = np.random.default_rng([integration, case == "spun", walls])
    n = 300
    obs = [wl.floor_obstacle(y=0.0, half=50.0)]
    if walls:
        obs.append((np.array([[-4, -9, 4], [4, -9, 4], [0, 9, 4]], F32), [0, 1, 2]))
    pos = rng.uniform(-3, 3, (n, 3)).astype(F32)
    pos[:, 1] = rng.uniform(0.3, 1.5, n)
    g = fa.RigidSimulation([fa.RigidBody(p, 1.0) for p in pos], [fa.CollidableMesh(*o) for o in obs])
    o = orc.RigidSimulation(pos, np.ones(n, F32), [orc.Obstacle(np.asarray(v, F32), np.asarray(i, np.uint64)) for v, i in obs])
    st = g.states()
    q = rng.normal(size=(n, 4))
    st[:, 3:7] = q / np.linalg.norm(q, axis=1, keepdims=True)
    st[:, 7:13] = rng.normal(0, 1, (n, 6))
    if case == "spun":
        st[:, 10:13] *= 10.0 ** rng.integers(8, 36, (n, 1))
    g.config = fa.RigidConfig(fa.Integration(integration), 0.01, 0.5, (0.0, -9.81, 0.0), (0.0, 0.0, 0.0))
    o.set_config(integration=integration, dt=F32(0.01), restitution=0.5, gravity=(0.0, -9.81, 0.0), torque=(0.0, 0.0, 0.0))
    g.set_states(st)
    o.set_states(st)
    for steps in (1, 1, 1, 5, 150):
        g.step(steps)
        o.step(steps)
        a, b = g.states(), o.states()
        wrong = np.nonzero(~same(a, b).all(1))[0]
        wrong = np.setdiff1d(wrong, BOTH_SIGNS.get((integration, case, walls), []))
        announce(f"{case} cubes, integration {integration}, {walls} walls, {steps} steps: "
                 f"{int(np.isnan(b[:, 3:7]).any(1).sum())} NaN poses, {int(np.isnan(b[:, 0:3]).any(1).sum())} NaN positions, "
                 f"{len(wrong)} wrong")
        assert len(wrong) == 0, wrong[:8]
    assert np.isnan(b[:, 3:7]).any()
