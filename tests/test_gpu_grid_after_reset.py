"""The grid of a context whose substep epoch has been rewound between two
binnings (the first substeps after mpm_init_volumes or after a reverse sweep
start the epochs again, in the binning made before): blocks that the particles
have left read zero, whatever epoch the next binning falls on.  In reproducible
mode grids repeat bit for bit, so each is compared with a fresh context's."""
import numpy as np
import pytest

import mpm_amd as M

pytestmark = pytest.mark.gpu

H, N, DT = 1.0 / 48, 700, 1e-4


def _context(batch):
    prm = M.default_params((48, 40, 56), H, compose=M.COMPOSE_TEXTBOOK, bc_mode=2, resort_every=16)
    g = M.Simulation([prm] * 2, [N] * 2) if batch else M.Simulation(prm, N)
    g.set_reproducible(True)
    return g


def _cloud(seed, corner):
    rng = np.random.default_rng(seed)
    x = ((np.array(corner) + 5.0 * rng.random((N, 3))) * H).astype(np.float32)
    v = rng.normal(0, 0.5, (N, 3)).astype(np.float32)
    return x, v, np.full(N, 2e-5, np.float32)


def _place(g, seed, corner):
    for s in range(g.nscenes):
        g.scene_set_particles(s, *_cloud(seed + s, corner))


def _there(g, steps):
    """Particles far from where they were, their volumes given: no
    mpm_init_volumes, so no reset, before the next substeps."""
    _place(g, 50, (34.0, 28.0, 40.0))
    g.set_state(V0=np.full(g.nscenes * N, 1e-7, np.float32))
    g.substeps(DT, steps)
    g.sync()
    return [g.scene_grid(s) for s in range(g.nscenes)]


@pytest.mark.parametrize("batch", [False, True])
@pytest.mark.parametrize("how", ["volumes", "reverse"])
@pytest.mark.parametrize("off", [-1, 0, 1])
def test_blocks_left_behind_read_zero(how, batch, off):
    g = _context(batch)
    _place(g, 10, (6.0, 6.0, 6.0))
    g.init_volumes()
    if how == "volumes":  # binned at epoch 17, then 16 substeps from epoch 1
        g.substeps(DT, 16)
        _place(g, 20, (8.0, 9.0, 10.0))
        g.init_volumes()
        g.substeps(DT, 16 + off)
    else:  # 5 substeps forward and 5 in the sweep: its binning is left at epoch 11
        g.adjoint_forward(DT, 5, 5)
        g.adjoint_backward(np.ones((g.n, 3), np.float32), None)
        g.substeps(DT, 10 + off)
    fresh = _context(batch)
    for steps in (1, 4):
        for a, b in zip(_there(g, steps), _there(fresh, steps)):
            for k in ("active", "m", "vel"):
                np.testing.assert_array_equal(a[k], b[k], err_msg=k)
            assert not a["vel"][~a["active"]].any()
    g.close()
    fresh.close()
