"""A device allocation that fails while a simulation's launch lists are rebuilt (records whose masses send a
cloth from the tiled kernel to the general one), or while the surrogate's slots are laid out.  The call reports
it; afterwards nothing is launched over half-built lists: the same records set again, other records, or a step
build them anew, and so does the surrogate set again.  The failure is injected on the host
(tests/native/failing_malloc.cpp), in a process of its own; no memory is exhausted."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

CHILD = r"""
import ctypes as C, sys
import numpy as np
shim = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)
sys.path.insert(0, sys.argv[2])
hip = C.CDLL("libamdhip64.so.7")
shim.failing_malloc_real.argtypes = [C.c_void_p]
shim.failing_malloc_real(C.cast(hip.hipMalloc, C.c_void_p))
shim.failing_host_malloc_real.argtypes = [C.c_void_p]
shim.failing_host_malloc_real(C.cast(hip.hipHostMalloc, C.c_void_p))
import feriphys_amd as fa
from feriphys_amd import workloads as wl

bits = lambda a: np.ascontiguousarray(a, np.float32).view(np.uint32)
sc = wl.config0(steps=1, seed=1, rows=20, cols=20)
ref = wl.build_gpu(sc)
assert shim.failing_malloc_calls() > 0  # the library's allocations pass through
rec = ref.get_points(0)
"""
LISTS = r"""
heavy = rec.copy()
heavy[::3, 0] *= 2.0

def result(sim, graph):
    if graph:
        sim.step_graph(6, 3)
    else:
        sim.step(6)
    return sim.get_points(0)

want = {}
for name, r in (("rec", rec), ("heavy", heavy)):
    ref.set_points(0, r)
    want[name] = result(ref, False)
ref.set_points(0, rec)
before = shim.failing_malloc_calls()
ref.set_points(0, heavy)
lists = shim.failing_malloc_calls() - before
print("allocations of the lists:", lists, flush=True)
assert lists >= 4
for nth in range(lists):
    for then in ("again", "back", "step", "graph", "forces"):
        sim = wl.build_gpu(sc)
        shim.failing_malloc_in(nth)
        try:
            sim.set_points(0, heavy)
            raise SystemExit("no failure")
        except fa.FpError as e:
            assert "out of memory" in str(e), e
        shim.failing_malloc_in(-1)
        print("allocation", nth, "failed, then", then, flush=True)
        if then == "again":
            sim.set_points(0, heavy)
        if then == "back":
            sim.set_points(0, rec)
        if then == "forces":
            sim.accumulate_forces(0)
            sim.set_points(0, heavy)
            sim.clear_forces(0)
        out = result(sim, then == "graph")
        assert sim.get_mesh_kernel(0) == (fa.FP_STEP_TILED if then == "back" else fa.FP_STEP_CSR)
        assert (bits(out) == bits(want["rec" if then == "back" else "heavy"])).all(), (nth, then)
print("ok", flush=True)
"""


SLOTS = r"""
net = fa.Surrogate(fa.SurrogateConfig(strain_limit=1e30, energy_limit=1e30), seed=3)
before = shim.failing_malloc_calls()
ref.set_surrogate(net)
made = shim.failing_malloc_calls() - before
print("allocations of the surrogate:", made, flush=True)
assert made >= 5
ref.step_surrogate(2)
want = ref.get_points(0)
for nth in range(made):
    sim = wl.build_gpu(sc)
    shim.failing_malloc_in(nth)
    try:
        sim.set_surrogate(net)
        raise SystemExit("no failure")
    except fa.FpError as e:
        assert "out of memory" in str(e), e
    shim.failing_malloc_in(-1)
    print("allocation", nth, "failed", flush=True)
    try:  # not set: refused, not launched
        sim.step_surrogate(1)
        raise SystemExit("stepped without a network")
    except fa.FpError:
        pass
    sim.set_surrogate(net)
    sim.step_surrogate(2)
    assert (bits(sim.get_points(0)) == bits(want)).all(), nth
print("ok", flush=True)
"""


# records in and out: one page-locked allocation for a simulation's life, reported when it fails
RECORDS = r"""
for size in (20, 120):
    sim = wl.build_gpu(wl.config0(steps=1, seed=1, rows=size, cols=size))
    before = shim.failing_host_malloc_calls()
    shim.failing_host_malloc_in(0)
    try:
        sim.set_points(0, np.ones((size * size, 10), np.float32))
        raise SystemExit("no failure")
    except fa.FpError as e:
        assert "out of memory" in str(e), e
    made = []
    r = rec if size == 20 else sim.get_points(0)
    for _ in range(2):
        sim.set_points(0, r)
        assert (bits(sim.get_points(0)) == bits(r)).all()
        made.append(shim.failing_host_malloc_calls() - before)
    print("page-locked allocations, the failed one among them:", made, flush=True)
    assert made == [2, 2]
print("ok", flush=True)
"""


@pytest.mark.parametrize("body", [LISTS, SLOTS, RECORDS], ids=["lists", "slots", "records"])
def test_lists_are_built_again_after_a_failed_allocation(tmp_path, body):
    shim = str(tmp_path / "failing_malloc.so")
    subprocess.run(["g++", "-O1", "-shared", "-fPIC", os.path.join(ROOT, "tests", "native", "failing_malloc.cpp"), "-o",
                    shim], check=True)
    p = subprocess.run([sys.executable, "-u", "-c", CHILD + body, shim, ROOT], capture_output=True, text=True, timeout=100)
    print(p.stdout[-3000:], p.stderr[-3000:], flush=True)
    assert p.returncode == 0 and p.stdout.rstrip().endswith("ok")
