"""The rigid-body kernel's own branches against the CPU oracle, every 29-float record bit for bit: scenes
of few faces (scanned in order; the tumbling tests' sphere takes the grids), step counts on both sides
of a launch's chunk of 64, batch sizes around a wavefront and a workgroup, and records whose constant
fields hold -0 and whose forces and torques are not zero (the first step reads them, all clear them)."""
import numpy as np
import pytest

import feriphys_amd as fa
import pyoracle as orc
from gpu_common import announce, bits

pytestmark = pytest.mark.gpu

FLOOR = (np.array([[-60, 0, 60], [60, 0, 60], [60, 0, -60], [-60, 0, -60]], np.float32),
         np.array([0, 1, 2, 0, 2, 3], np.uint64))
RAMP = (np.array([[-60, -3, 60], [60, 4, 60], [60, 4, -60], [-60, -3, -60]], np.float32),
        np.array([0, 1, 2, 0, 2, 3], np.uint64))


def both(n, integration, obstacles, seed):
    rng = np.random.default_rng(seed)
    pos = rng.uniform((-6, 0.9, -6), (6, 2.0, 6), (n, 3)).astype(np.float32)
    mass = rng.uniform(0.5, 4.0, n).astype(np.float32)
    g = fa.RigidSimulation([fa.RigidBody(p, float(m)) for p, m in zip(pos, mass)],
                           [fa.CollidableMesh(*o) for o in obstacles])
    o = orc.RigidSimulation(pos, mass, [orc.Obstacle(*ob) for ob in obstacles])
    g.config = fa.RigidConfig(fa.Integration(integration), 1.0 / 600.0, 0.0, (0.0, -9.81, 0.0), (0.0, 0.1, 0.0))
    o.set_config(integration=integration, dt=np.float32(1.0 / 600.0), restitution=0.0, gravity=(0.0, -9.81, 0.0),
                 torque=(0.0, 0.1, 0.0))
    rec = g.states()
    rec[:, 7:13] = rng.normal(scale=1.0, size=(n, 6)).astype(np.float32)
    rec[::2, 23:29] = rng.normal(scale=0.5, size=(len(rec[::2]), 6)).astype(np.float32)
    rec[1::3, 23:29] = -0.0
    zero = rec[:, 14:23] == 0.0
    rec[:, 14:23][zero & (rng.random(zero.shape) < 0.5)] = -0.0
    g.set_states(rec)
    o.set_states(rec)
    assert (bits(g.states()) == bits(rec)).all()
    return g, o


@pytest.mark.parametrize("n", [1, 63, 65, 257])
@pytest.mark.parametrize("integration", [0, 1])
@pytest.mark.parametrize("scene", ["none", "floor", "floor+ramp"])
def test_few_faces_bit_exact(n, integration, scene):
    obstacles = {"none": [], "floor": [FLOOR], "floor+ramp": [FLOOR, RAMP]}[scene]
    g, o = both(n, integration, obstacles, n + integration)
    for steps in (1, 63, 65, 130):
        announce(f"rigid {n} bodies, {scene}, {steps} more steps")
        g.step(steps)
        o.step(steps)
        assert (bits(g.states()) == bits(o.states())).all()
