"""The patch kernel's groups: vertices of one wavefront with different numbers of struts and faces (the
masked entries past the smallest), wavefronts and patches that are not full, and a strut whose squared
length leaves the range of the short square root.  In exact arithmetic the kernel equals the CSR kernel, which
shares neither its entries nor its groups, bit for bit."""
import numpy as np
import pytest

import feriphys_amd as fa

pytestmark = pytest.mark.gpu


def bits(a):
    return np.ascontiguousarray(a, np.float32).view(np.uint32)


def irregular(n, close):
    """n vertices of open fans of 1 to 16 triangles side by side (the last as large as fits), a few
    struts across each fan; with `close`, two more triangles whose first vertices are 1e-16 apart."""
    rng = np.random.default_rng(n)
    pos, tri, across = [], [], []
    while n - len(pos) >= 3:
        k = min(int(rng.integers(1, 17)), n - len(pos) - 2)
        if n - len(pos) - (k + 2) in (1, 2):  # leave room for a triangle or nothing
            k = n - len(pos) - 2
        hub, ang = len(pos), np.arange(k + 1) * 0.35
        pos.append((0.5 * hub, 0.56, 0.0))
        pos += [(0.5 * hub + 0.2 * np.cos(a), rng.uniform(0.5, 0.6), 0.2 * np.sin(a)) for a in ang]
        tri += [(hub, hub + 1 + j, hub + 2 + j) for j in range(k)]
        across += [(hub + 1 + j, hub + 1 + j + 2) for j in range(0, k - 1, int(rng.integers(1, 4)))]
    m = len(pos)
    if close:
        pos += [(0, 0, 0), (-0.1, 0, 0.1), (-0.1, 0, 0.2), (1e-16, 0, 0), (0.1, 0, -0.1), (0.1, 0, 0.2)]
        tri += [(m, m + 1, m + 2), (m + 3, m + 4, m + 5)]
    return np.array(pos, np.float32), np.array(tri, np.uint64).reshape(-1), across, m


@pytest.mark.parametrize("n", [3, 63, 65, 256, 257, 700])
@pytest.mark.parametrize("close", [False, True])
def test_irregular_meshes_match_the_csr_kernel(n, close):
    pos, idx, across, m = irregular(n, close)
    out = []
    for kernel, expect in ((fa.FP_KERNEL_AUTO, fa.FP_STEP_PATCH), (fa.FP_KERNEL_CSR, fa.FP_STEP_CSR)):
        mesh = fa.SpringyMesh(pos, idx, 0.02 * n, 3.0, 0.01)
        for pair in across:
            mesh.add_strut(pair, 0.5, 0.002)
        if close:
            mesh.add_strut((m, m + 3), 1e-20, 1e-20)
        floor = (np.array([[-9, 0.55, 9], [9, 0.55, 9], [9, 0.55, -9], [-9, 0.55, -9]], np.float32), [0, 1, 2, 0, 2, 3])
        sim = fa.Simulation([mesh], [fa.CollidableMesh(*floor)])
        sim.config = fa.Config(fa.Integration.Rk4, 1e-3, (0.0, -9.81, 0.0), (1.0, 0.5, 0.2), 0.2, 0.5, 0.3, 0.2)
        sim.set_kernel(kernel, fa.FP_MATH_EXACT)
        assert sim.get_mesh_kernel(0) == expect
        print(f"[gpu-test] irregular mesh of {n} vertices, close {close}, kernel {kernel}", flush=True)
        sim.step(1 if close else 20)
        out.append(sim.get_points(0))
    assert np.isfinite(out[0]).all() and np.isfinite(out[1]).all()
    assert (bits(out[0]) == bits(out[1])).all()
