"""The surrogate's features of a strut so short that the square of its length is subnormal (ends less than
1.1e-19 apart), where the inference kernel's short square root has no value: the direction and the strain are
still those of the strut, in the feature kernel and in the network's input."""
import numpy as np
import pytest

import feriphys_amd as fa
from feriphys_amd import workloads as wl

pytestmark = pytest.mark.gpu
A, B = 40, 42  # (4, 4) and (4, 6) of a 9 x 9 cloth: the ends of a bending strut


def bits(a):
    return np.ascontiguousarray(a, np.float32).view(np.uint32)


def close(apart):
    sim = wl.build_gpu(wl.config0(steps=1, seed=3, rows=9, cols=9, pins="corners"))
    rec = sim.get_points(0)
    rec[A, 1:4], rec[A + 1, 1:4], rec[B, 1:4] = 0.0, (0.0, 0.0, 0.04), (apart, 0.0, 0.0)
    sim.set_points(0, rec)
    sim.set_surrogate(fa.Surrogate(seed=5))
    return sim


@pytest.mark.parametrize("apart", [2e-19, 1e-19, 5e-20, 1e-20, 1e-21])
def test_features_of_a_strut_with_subnormal_squared_length(apart):
    """Against the same formula in 64 bits from the f32 square of the length.  Relative to it: the root,
    the strain's difference and four products round once each (2^-24), the two hardware reciprocals are
    within an ulp (2^-23): 10 x 2^-24 < 1e-6."""
    sim = close(apart)
    cfg = fa.SurrogateConfig()
    nbr, rest = sim.surrogate_slots(0)
    got = sim.surrogate_features(0)
    print(f"[gpu-test] features of a strut {apart} long", flush=True)
    assert np.isfinite(got).all()
    for v, other, sign in ((A, B, 1.0), (B, A, -1.0)):
        (j,) = np.nonzero(nbr[v] == other)[0]
        d = np.float32(apart)
        length = np.sqrt(np.float64(d * d))
        want = sign * cfg.strain_scale * (length - rest[v, j]) / rest[v, j] * (np.float64(d) / length)
        assert abs(got[v, 6 * j] - want) <= 1e-6 * abs(want)
        assert (got[v, 6 * j + 1:6 * j + 3] == 0.0).all()


@pytest.mark.parametrize("per_wave", [32, 64])
def test_the_network_sees_the_same_direction(per_wave):
    """A strut 1e-19 or 5e-20 long has the features of one 2e-19 long (whose square is normal) but for the
    last bits, which bf16 does not hold: the outputs are the same bits."""
    out = []
    for apart in (2e-19, 1e-19, 5e-20):
        sim = close(apart)
        sim.set_surrogate_shape(per_wave)
        out.append(sim.surrogate_accel(0))
    print(f"[gpu-test] network over a strut with subnormal squared length, {per_wave} vertices a wave", flush=True)
    assert np.isfinite(out[0]).all()
    for o in out[1:]:
        assert (bits(o) == bits(out[0])).all()
