"""Reads of growing size in one context: the pinned ring grows with them, and
smaller reads after a larger one use its head."""
import numpy as np
import pytest

import mpm_amd as M

pytestmark = pytest.mark.gpu


def test_ring_grows_with_the_reads():
    rng = np.random.default_rng(5)
    ns = (3, 40000, 200001)
    g = M.Simulation([M.default_params((64, 64, 64), 1 / 64)] * 3, ns)
    n = sum(ns)
    ref = dict(x=rng.uniform(0.2, 0.8, (n, 3)).astype(np.float32), v=rng.normal(size=(n, 3)).astype(np.float32))
    ref.update({k: rng.normal(size=(n, 9)).astype(np.float32) for k in ("B", "FE", "FP")})
    ref["V0"] = rng.random(n).astype(np.float32)
    g.set_particles(ref["x"], ref["v"], np.ones(n, np.float32))
    g.set_state(**{k: ref[k] for k in ("B", "FE", "FP", "V0")})
    g.debug_bin()
    for s in (0, 1, 2, None, 0, 2, 1):
        got = g.particles() if s is None else g.scene_particles(s)
        lo, hi = (0, n) if s is None else (g.offsets[s], g.offsets[s + 1])
        for k in ref:
            np.testing.assert_array_equal(got[k], ref[k][lo:hi], err_msg=f"{s} {k}")
    g.close()
