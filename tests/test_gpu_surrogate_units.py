"""The surrogate's shares of work: vertices dealt to workgroups in units of 32 or 64 (fewer units than
workgroups, one more than they have, last units not full), and the diagnostics per mesh of cloths of
one block and of many."""
import numpy as np
import pytest

import feriphys_amd as fa
from feriphys_amd import workloads as wl

pytestmark = pytest.mark.gpu


def bits(a):
    return np.ascontiguousarray(a, np.float32).view(np.uint32)


@pytest.mark.parametrize("rows,cols", [(3, 3), (31, 33), (64, 128), (91, 91), (130, 126)])
def test_every_vertex_once_whatever_the_units(rows, cols):
    """The network's output of a vertex does not depend on the unit that it falls in: units of 32 and of
    64 vertices give the same bits for every vertex, none of them left at zero."""
    sim = wl.build_gpu(wl.config0(steps=1, seed=rows, rows=rows, cols=cols, pins="edge"))
    rec = sim.get_points(0)
    rec[:, 4:7] = np.random.default_rng(cols).normal(0.0, 0.3, (len(rec), 3)).astype(np.float32)
    sim.set_points(0, rec)
    sim.set_surrogate(fa.Surrogate(seed=5))
    print(f"[gpu-test] units of a {rows}x{cols} cloth", flush=True)
    out = []
    for per_wave in (32, 64):
        sim.set_surrogate_shape(per_wave)
        out.append(sim.surrogate_accel(0))
    assert np.isfinite(out[0]).all() and (np.abs(out[0]).max(axis=1) > 0).all()
    assert (bits(out[0]) == bits(out[1])).all()


def test_diagnostics_are_the_largest_of_all_meshes():
    """The largest strain change of a big step over three cloths of one block, some and many blocks,
    against 64 bits from the records before and after.  A length is rounded to 2^-24 of itself and the
    strains here are below 1, so a change of strain is within 2 (1 + 1) 2^-24 and the reciprocal's ulp:
    1e-6."""
    parts = [wl.config0(steps=1, seed=s, rows=r, cols=c, pins="edge") for s, r, c in ((1, 9, 7), (2, 40, 50), (3, 200, 300))]
    sim = wl.build_gpu(wl.Scene([p.cloths[0] for p in parts], parts[0].config, [], 1e-3, 1, 1, "three cloths"))
    sim.set_surrogate(fa.Surrogate(fa.SurrogateConfig(strain_limit=1e30, energy_limit=1e30), seed=3))
    rng = np.random.default_rng(8)
    before = []
    for k in range(3):
        rec = sim.get_points(k)
        rec[:, 4:7] = rng.normal(0.0, 0.1 * (1 + k % 2), (len(rec), 3)).astype(np.float32)
        sim.set_points(k, rec)
        before.append(rec)
    print("[gpu-test] diagnostics of three cloths", flush=True)
    st = sim.step_surrogate(1)
    worst = 0.0
    for k in range(3):
        nbr, rest = sim.surrogate_slots(k)
        after = sim.get_points(k)
        v, j = np.nonzero(nbr >= 0)
        length = [np.linalg.norm(r[nbr[v, j], 1:4].astype(np.float64) - r[v, 1:4], axis=1) for r in (before[k], after)]
        worst = max(worst, float((np.abs(length[1] - length[0]) / rest[v, j]).max()))
    assert st.fallbacks == 0 and worst < 1.0
    assert abs(st.max_strain_residual - worst) <= 1e-6
