"""The block passes' width of a context whose blocks are worked on in parts: as
for whole blocks, it starts as the number of the grid's blocks (2,048 at most),
and the autotuner tries no other where that is below 1,024.  Results do not
depend on it (reproducible mode)."""
import numpy as np
import pytest

import mpm_amd as M

pytestmark = pytest.mark.gpu


def test_width_of_a_crowded_grid():
    n = 20000  # 79 parts of 256 particles and more, in a grid of 27 blocks
    g = M.Simulation(M.default_params((12, 12, 12), 1 / 12, bc_mode=M.BC_DOMAIN), n)
    g.set_reproducible(True)
    rng = np.random.default_rng(1)
    x = rng.uniform(3.5 / 12, 8.5 / 12, (n, 3)).astype(np.float32)
    out = []
    for width in (None, 1, 26, 27, 5000):
        g.set_particles(x, np.zeros_like(x), np.full(n, 1e-3, np.float32))
        g.init_volumes()
        if width is None:
            assert g.tuning()[1] == 27
        else:
            g.set_tuning(16, width)
        g.substeps(1e-4, 40)
        g.sync()
        out.append(g.particles())
    for p in out[1:]:
        for k in p:
            np.testing.assert_array_equal(p[k], out[0][k])
    g.autotune(1e-4, steps=8)
    assert g.tuning()[1] == 27
    g.close()


def test_width_of_a_large_grid():
    g = M.Simulation(M.default_params((64, 64, 64), 1 / 64), 100)
    assert g.tuning()[1] == 2048
    g.close()
