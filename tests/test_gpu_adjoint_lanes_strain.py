"""The reverse P2G's four, two and one lanes per particle on a strained body:
a scene's gradients in a context of its own size against those of the same
scene at the head of a batch of more than 40,000 particles, one lane each.
Both contexts sum the grid in FP64 over the same parts of the same slots, so
the recorded forward does not differ, and a compression of 1.6% over the four
substeps keeps dL/dE0 far above rounding.  What is left
is the order of the gather's 64-term FP32 sums, below 64 * 2^-24 = 4e-6, which
is asked of every gradient."""
import numpy as np
import pytest

import mpm_amd as M
from mpm_amd import scenes

pytestmark = pytest.mark.gpu

DT, STEPS = 1e-4, 4


def _scene(seed, n):
    radius = (n / 8.0 * 3.0 / (4.0 * np.pi)) ** (1.0 / 3.0) / 64.0  # 8 particles a cell
    c = np.float32([0.5, 0.5, 0.5])
    sc = scenes.snowball(seed=seed, n=n, grid=64, radius=radius, centre=tuple(c), v0=(0.0, 0.0, 0.0), E=1.2e5)
    sc["v"] = (np.float32(-40.0) * (sc["x"] - c)).astype(np.float32)
    return sc


def _gradients(scs, a, b):
    sim = M.Simulation([M.default_params(s["dims"], s["h"], compose=M.COMPOSE_TEXTBOOK, bc_mode=M.BC_DOMAIN,
                                         theta_s=7.5e-3) for s in scs], [s["x"].shape[0] for s in scs])
    for i, s in enumerate(scs):
        sim.scene_set_particles(i, s["x"], s["v"], s["m"], s["E0"])
    sim.init_volumes()
    sim.adjoint_forward(DT, STEPS, 2)
    out = sim.adjoint_backward(a, b)
    sim.close()
    return out


@pytest.mark.parametrize("n", [63, 64, 65, 5003, 12000, 12001, 40000])
def test_lanes_agree(n):
    sc, filler = _scene(31, n), _scene(32, 40001)
    rng = np.random.default_rng(n)
    total = n + 40001
    a = rng.normal(size=(total, 3)).astype(np.float32)
    b = rng.normal(size=(total, 3)).astype(np.float32) * np.float32(1e-3)
    alone = _gradients([sc], a[:n], b[:n])
    batch = _gradients([sc, filler], a, b)
    for k, got, ref in zip(("x0", "v0", "E0"), alone, batch):
        ref = np.float64(ref[:n])
        err = np.linalg.norm(got - ref) / np.linalg.norm(ref)
        assert err < 64 * 2.0 ** -24, (k, err)
