"""Node sums of crowded home blocks.  A block is worked on in parts, and its
parts' sums meet in FP64: each node's sum is rounded to FP32 once, as if the
block were whole.  N = 2^k particles at one point, beside a scene of a single
particle there, make this exact: a node's sum is N times the single
particle's contribution, which FP64 holds (24 + k bits) and FP32 represents,
so masses scale by exactly N and velocities and dL/dv0 do not change by a bit.
(512 or more parts summed in FP32 round at almost every add.)"""
import numpy as np
import pytest

import mpm_amd as M

pytestmark = pytest.mark.gpu

H = 1.0 / 32
X = np.float32([0.4712, 0.5231, 0.4503])
V = np.float32([1.3, -0.7, 2.1])
G = np.float32([0.37, 1.9, -0.81])


def _pair(n, v, **kw):
    """Scene 0: one particle, scene 1: n, all alike and without stress."""
    prm = M.default_params((32, 32, 32), H, compose=M.COMPOSE_TEXTBOOK, bc_mode=M.BC_DOMAIN, gravity=(0, 0, 0), **kw)
    g = M.Simulation([prm, prm], [1, n])
    one = np.ones((n + 1, 1), np.float32)
    g.set_particles(X * one, v * one, np.full(n + 1, 1.7e-4, np.float32), np.zeros(n + 1, np.float32))
    return g


def _same_grids(g, n):
    a, b = g.scene_grid(0), g.scene_grid(1)
    assert a["active"].sum() == 64
    np.testing.assert_array_equal(b["m"], np.float32(n) * a["m"])
    np.testing.assert_array_equal(b["vel"], a["vel"])


# the three part sizes of 256, 512 and 768
SIZES = [131072, 262144, 524288]


@pytest.mark.parametrize("n", SIZES)
def test_node_sums_are_rounded_once(n):
    g = _pair(n, V)
    g.init_volumes()
    g.substeps(1e-4, 1)
    g.sync()
    _same_grids(g, n)
    g.close()


@pytest.mark.parametrize("n", SIZES)
def test_node_adjoints_are_rounded_once(n):
    g = _pair(n, V)
    g.adjoint_forward(1e-4, 1, 1)
    _, gv0, _ = g.adjoint_backward(None, G * np.ones((n + 1, 1), np.float32))
    np.testing.assert_array_equal(gv0[1:], np.broadcast_to(gv0[0], (n, 3)))
    g.close()


@pytest.mark.parametrize("n", [1, 95 * 256, 95 * 256 + 1])
def test_both_flushes(n):
    """At most 96 entries, and one more, where the flush changes its lanes: one
    rounding of N times the single particle's mass at every node; dL/dv0 within
    its gather's 64 terms."""
    g = _pair(n, V)
    g.init_volumes()
    g.substeps(1e-4, 1)
    g.sync()
    a, b = g.scene_grid(0), g.scene_grid(1)
    np.testing.assert_array_equal(b["m"], (np.float64(n) * a["m"].astype(np.float64)).astype(np.float32))
    np.testing.assert_array_equal(b["active"], a["active"])
    g.adjoint_forward(1e-4, 1, 1)
    _, gv0, _ = g.adjoint_backward(None, G * np.ones((n + 1, 1), np.float32))
    assert np.abs(gv0[1:] - gv0[0]).max() <= 64 * 2.0 ** -24 * np.abs(gv0[0]).max()
    g.close()


def test_particles_beyond_their_halo():
    """Six substeps of 0.64 cells without a binning: the last sums come from
    the scatter to global memory.  The reverse sweep's per-lane order of x
    gradients differs, by less than a 64-term FP32 sum a substep."""
    n, dt = 131072, 1e-3
    g = _pair(n, np.float32([20.0, 0.0, 0.0]), resort_every=64)
    g.init_volumes()
    g.substeps(dt, 6)
    g.sync()
    _same_grids(g, n)
    g.close()
    g = _pair(n, np.float32([20.0, 0.0, 0.0]), resort_every=64)
    g.adjoint_forward(dt, 6, 6)
    _, gv0, _ = g.adjoint_backward(None, G * np.ones((n + 1, 1), np.float32))
    err = np.abs(gv0[1:] - gv0[0]).max() / np.abs(gv0[0]).max()
    assert err < 6 * 64 * 2.0 ** -24
    g.close()
